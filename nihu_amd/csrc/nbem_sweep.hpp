// nbem_sweep.hpp -- Burton-Miller matrices for many wavenumbers on one mesh.
//
// Regular pairs: one persistent launch.  A workgroup of 256 lanes (one test
// row per lane) takes work items (row tile, trial-column tile, batch of KB
// wavenumbers) with a fixed stride until none are left.  For each pair the
// wavenumber-independent geometry of every quadrature point (r, r - d, the
// weight over r, 1/r^2 and the test-normal projection) is computed once and
// kept in registers while the KB wavenumbers of the batch reuse it; per
// wavenumber only the phase, the hardware sin/cos and the kernel algebra
// remain.  The FP64 near-singular and diagonal passes compute their
// wavenumber-independent (Laplace static) parts once per pair into a buffer
// and add the dynamic part per (pair, wavenumber).

#pragma once

#include "nbem_kernels.hpp"

namespace nbk {

struct SweepArgs {
	int n, row_tiles, col_tiles, tile_cols, n_k, n_items;
	int nr, nc;                 // rows / columns processed (n, or a leading block when tuning)
	const double *c;            // centres [3][n]
	const float *nu;            // unit normals [3][n]
	const double *thr;          // [NTHR][n]
	const QPoint *qt;           // quadrature table of the fixed degree [n][Q]
	const double *k_rev;        // [n_k] k / (2 pi), FP64
	const float *kf;            // [n_k] k
	const float *krevf;         // [n_k] k / (2 pi)
	const float2 *alpha;        // [n_k], -i/k
	float2 *A, *B;
	long long ld, kstride;
};

template <int KB, int Q>
__global__ void __launch_bounds__(256) sweep_regular_kernel(SweepArgs a)
{
	const auto sc = uni(a.c);
	const auto snu = uni(a.nu);
	const auto thr = uni(a.thr);
	const auto k_rev = uni(a.k_rev);
	const auto kf = uni(a.kf);
	const auto krevf = uni(a.krevf);
	const auto alpha = uni((const float *)a.alpha);
	for (int item = blockIdx.x; item < a.n_items; item += gridDim.x) {
		const int rt = item % a.row_tiles;
		const int rest = item / a.row_tiles;
		const int ct = rest % a.col_tiles;
		const int f0 = (rest / a.col_tiles) * KB;
		const int i = rt * 256 + threadIdx.x;
		const bool row_ok = i < a.nr;
		const int ii = row_ok ? i : a.nr - 1;
		const double cix = a.c[ii], ciy = a.c[a.n + ii], ciz = a.c[2 * a.n + ii];
		const float nxx = a.nu[ii], nxy = a.nu[a.n + ii], nxz = a.nu[2 * a.n + ii];
		row_ready(cix, ciy, ciz, nxx, nxy, nxz, ii);
		const int j0 = ct * a.tile_cols;
		const int j1 = min(j0 + a.tile_cols, a.nc);
		for (int j = j0; j < j1; ++j) {
			const double cjx = sc[j], cjy = sc[a.n + j], cjz = sc[2 * a.n + j];
			const double d2 = d2_pair(cix, ciy, ciz, cjx, cjy, cjz);
			const bool act = row_ok && !(d2 < thr[THR_NEAR * a.n + j]) && i != j;
			if (__ballot(act) == 0) continue;
			const float dcx = (float)(cjx - cix), dcy = (float)(cjy - ciy), dcz = (float)(cjz - ciz);
			const float dcx2 = 2.0f * dcx, dcy2 = 2.0f * dcy, dcz2 = 2.0f * dcz;
			const float d2f = (float)d2;
			double y = __builtin_amdgcn_rsq(d2);
			y = y * (1.5 - 0.5 * d2 * y * y);
			const double d = d2 * y;
			const float df = (float)d;
			const float nyx = snu[j], nyy = snu[a.n + j], nyz = snu[2 * a.n + j];
			const float av = dcx * nyx + dcy * nyy + dcz * nyz;
			const float nn = nxx * nyx + nxy * nyy + nxz * nyz;
			const float b0 = dcx * nxx + dcy * nxy + dcz * nxz;
			// wavenumber-independent geometry of the points: the phase
			// correction and, with alpha = -i/k, the five real weights of the
			// entries (g = w / r^3, beta = nn - 3 a b / r^2; the formulas before
			// bm_add with a i = -1/k):
			//   A = sum [W1 - (i/k) W0 - i k W2] e^{-i th}
			//   B = sum [W3 - (i/k) W4] e^{-i th}
			// (seven weights, one per kernel sum, took 14 FMAs per point and
			// wavenumber instead of 10; 64 wavenumbers on 5120 triangles 10.0 -> 8.3
			// ms a call.  W3's w / r is taken from the root itself: as r g r it carried
			// the root's error five times, B's smaller entries 1/3 more error)
			float gdel[Q], W[5][Q];
			const auto qf = uni((const float *)(a.qt + (size_t)j * Q));
#pragma unroll
			for (int q = 0; q < Q; ++q) {
				const float ox = qf[8 * q], oy = qf[8 * q + 1], oz = qf[8 * q + 2], w = qf[8 * q + 3], oo = qf[8 * q + 4];
				const float u = __builtin_fmaf(dcx2, ox, __builtin_fmaf(dcy2, oy, __builtin_fmaf(dcz2, oz, oo)));
				const float r2 = d2f + u;
				const float rinv = __builtin_amdgcn_rsqf(r2);
				const float r = r2 * rinv;
				gdel[q] = u * __builtin_amdgcn_rcpf(r + df);
				const float ri2 = rinv * rinv;
				const float wr = w * rinv;
				const float g = wr * ri2;
				const float b = __builtin_fmaf(oz, nxz, __builtin_fmaf(oy, nxy, __builtin_fmaf(ox, nxx, b0)));
				const float beta = __builtin_fmaf(-3.0f * av, b * ri2, nn);
				const float gs = g * (b + r);
				W[0][q] = g * beta;
				W[1][q] = g * __builtin_fmaf(beta, r, -av);
				W[2][q] = av * gs;
				W[4][q] = g * b;
				W[3][q] = __builtin_fmaf(W[4][q], r, wr);
			}
			for (int fb = 0; fb < KB; ++fb) {
				const int f = f0 + fb;
				if (f >= a.n_k) break;
				double td = d * k_rev[f];
				td -= rint(td);
				const float t0 = (float)td;
				const float k = kf[f], kr = krevf[f];
				// A[m] = sum_q W[m][q] (cos t_q, sin t_q); e^{-i th} = (cos, -sin)
				float2 A[5];
#pragma unroll
				for (int m = 0; m < 5; ++m) A[m] = zero2();
#pragma unroll
				for (int q = 0; q < Q; ++q) {
					const float t = __builtin_fmaf(kr, gdel[q], t0);
					const float c = __builtin_amdgcn_cosf(t), sn = __builtin_amdgcn_sinf(t);
#pragma unroll
					for (int m = 0; m < 5; ++m) {
						A[m].x = __builtin_fmaf(W[m][q], c, A[m].x);
						A[m].y = __builtin_fmaf(W[m][q], sn, A[m].y);
					}
				}
				if (act) {
					const float al = alpha[2 * f + 1];      // -1/k
					const float ar = __builtin_fmaf(al, A[0].y, __builtin_fmaf(-k, A[2].y, A[1].x));
					const float ai = __builtin_fmaf(al, A[0].x, __builtin_fmaf(-k, A[2].x, -A[1].y));
					const float br = __builtin_fmaf(al, A[4].y, A[3].x);
					const float bi = __builtin_fmaf(al, A[4].x, -A[3].y);
					store_two(a.A, a.B, (long long)f * a.kstride + (long long)j * a.ld, (unsigned)i * 8u, 0,
						make_float2(ar, ai), make_float2(br, bi));
				}
			}
		}
	}
}

// NiHu's distance-driven policy over many wavenumbers in one persistent
// launch: per pair the FP64 distance, the near-singular test and the
// per-kernel degrees of the distance tables are found once; each wavenumber
// of the work item's batch then reduces its own phase of k d in FP64 and
// evaluates the pair as the single-wavenumber pass does (bm_regular_kernel's
// far, mid and close waves), so every wavenumber's matrices equal those of one
// Burton-Miller assembly at that wavenumber.
struct SweepNihuArgs {
	RegArgs r;                  // the mesh's tables, thresholds and records (its k, alpha, out unused)
	int n_k, n_items, col_tiles;
	const double *k_rev;        // [n_k] k / (2 pi), FP64
	const float *kf;            // [n_k] k
	const float *krevf;         // [n_k] k / (2 pi)
	const float2 *alpha;        // [n_k]
	float2 *A, *B;
	long long ld, kstride;
};

template <int KB>
__global__ void __launch_bounds__(256) sweep_nihu_kernel(SweepNihuArgs sa)
{
	const RegArgs &a = sa.r;
	const auto rec = uni(a.rec);
	const auto k_rev = uni(sa.k_rev);
	const auto kf = uni(sa.kf);
	const auto krevf = uni(sa.krevf);
	const auto alpha = uni((const float *)sa.alpha);
	for (int item = blockIdx.x; item < sa.n_items; item += gridDim.x) {
		const int rt = item % a.row_tiles;
		const int rest = item / a.row_tiles;
		const int ct = rest % sa.col_tiles;
		const int f0 = (rest / sa.col_tiles) * KB;
		const int i = rt * 256 + threadIdx.x;
		const bool row_ok = i < a.n_rows;
		const int ii = row_ok ? i : a.n_rows - 1;
		const double cix = a.tc[ii], ciy = a.tc[a.tn + ii], ciz = a.tc[2 * a.tn + ii];
		const float nxx = a.tnu[ii], nxy = a.tnu[a.tn + ii], nxz = a.tnu[2 * a.tn + ii];
		row_ready(cix, ciy, ciz, nxx, nxy, nxz, ii);
		const int j0 = ct * a.tile_cols;
		const int j1 = min(j0 + a.tile_cols, a.n_cols);
		for (int j = j0; j < j1; ++j) {
			const double dxd = rec[j].c[0] - cix, dyd = rec[j].c[1] - ciy, dzd = rec[j].c[2] - ciz;
			const double d2 = __fma_rn(dzd, dzd, __fma_rn(dyd, dyd, dxd * dxd));
			const bool act = row_ok & !(d2 < rec[j].thr[THR_NEAR]) & (i != j);
			if (!any_lane(act)) continue;
			const float w1 = rec[j].w1;
			BmPair p;
			double d;
			bm_geometry(dxd, dyd, dzd, d2, nxx, nxy, nxz, rec[j].nu[0], rec[j].nu[1], rec[j].nu[2], p, d);
			const bool allfar = !any_lane(act & (d2 < rec[j].thr[THR_22_3]));
			double t[NTHR];
			bool close = false;
			if (!allfar) {
#pragma unroll
				for (int q = 0; q < NTHR; ++q) t[q] = rec[j].thr[q];
				close = any_lane(act & (d2 < t[THR_3_6]));
			}
			const long long col = (long long)j * sa.ld;
			for (int fb = 0; fb < KB; ++fb) {
				const int f = f0 + fb;
				if (f >= sa.n_k) break;
				bm_wave(p, d, k_rev[f], kf[f], alpha[2 * f + 1]);
				BmEntry e = {-0.0f, -0.0f, -0.0f, -0.0f};
				if (allfar)
					bm_far(p, w1, e);
				else if (!close)
					bm_mid(p, nxx, nxy, nxz, a.qt[2] + (size_t)j * 3, w1, krevf[f], d2 < t[THR_9_1], d2 < t[THR_15_8],
						d2 < t[THR_22_3], e);
				else
					bm_close(a, j, act, d2, t, p, nxx, nxy, nxz, w1, krevf[f], e);
				if (act) {
					const long long at = (long long)f * sa.kstride + col;
					store_two(sa.A, sa.B, at, (unsigned)i * 8u, 0, make_float2(e.ar, e.ai), make_float2(e.br, e.bi));
				}
			}
		}
	}
}

// Wavenumber-independent parts of the FP64 pairs: near pairs (p < n_near)
// store the Laplace static integrals of SLP, DLP, DLPt, HSP; diagonal pairs
// (n_near <= p < n_near + n) store diag_static's four sums.
struct StaticArgs {
	int n, n_near;
	const int *pi, *pj;
	const double *c, *nu64, *X;
	const Rules *rules;
	double *st;                 // [(n_near + n) * 4]
};

__global__ void __launch_bounds__(64) fp64_static_kernel(StaticArgs a)
{
	const int p = blockIdx.x * blockDim.x + threadIdx.x;
	if (p >= a.n_near + a.n) return;
	const bool diag = p >= a.n_near;
	const int i = diag ? p - a.n_near : a.pi[p];
	const int j = diag ? i : a.pj[p];
	D3 V[3];
	for (int v = 0; v < 3; ++v)
		V[v] = {a.X[(3 * v) * a.n + j], a.X[(3 * v + 1) * a.n + j], a.X[(3 * v + 2) * a.n + j]};
	const D3 x0 = {a.c[i], a.c[a.n + i], a.c[2 * a.n + i]};
	double st[4];
	if (diag) {
		diag_static(V, x0, st);
	} else {
		const D3 nx = {a.nu64[i], a.nu64[a.n + i], a.nu64[2 * a.n + i]};
		near_static<ALL4>(V, x0, nx, *a.rules, st);
	}
	for (int t = 0; t < 4; ++t) a.st[(size_t)p * 4 + t] = st[t];
}

struct DynArgs {
	int n, n_near, n_k;
	int p0;                     // first pair of the launch (pairs p0 .. n_near + n - 1)
	const int *pi, *pj;
	const double *c, *nu64, *X, *J;
	const Rules *rules;
	const double *st;
	const double *k;            // [n_k]
	const double2 *alpha;       // [n_k]
	float2 *A, *B;
	long long ld, kstride;
};

// one lane per (FP64 pair, wavenumber): consecutive lanes take consecutive pairs
__global__ void __launch_bounds__(64) fp64_dynamic_kernel(DynArgs a)
{
	const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	const long long np = (long long)a.n_near + a.n - a.p0;
	if (t >= np * a.n_k) return;
	const int f = (int)(t / np);
	const int p = a.p0 + (int)(t % np);
	const bool diag = p >= a.n_near;
	const int i = diag ? p - a.n_near : a.pi[p];
	const int j = diag ? i : a.pj[p];
	const Rules &R = *a.rules;
	D3 V[3];
	for (int v = 0; v < 3; ++v)
		V[v] = {a.X[(3 * v) * a.n + j], a.X[(3 * v + 1) * a.n + j], a.X[(3 * v + 2) * a.n + j]};
	const D3 x0 = {a.c[i], a.c[a.n + i], a.c[2 * a.n + i]};
	const double k = a.k[f];
	const double J = a.J[j];
	double st[4];
	for (int q = 0; q < 4; ++q) st[q] = a.st[(size_t)p * 4 + q];
	double2 s[4] = {make_double2(0, 0), make_double2(0, 0), make_double2(0, 0), make_double2(0, 0)};
	const double2 al = a.alpha[f];
	double ar, ai, br, bi;
	if (diag) {
		double2 dyn[2];
		diag_dynamic<SLP | HSP>(V, x0, J, k, R, dyn);
		diag_combine<HELM, SLP | HSP>(st, dyn, k, s);
	} else {
		const D3 nx = {a.nu64[i], a.nu64[a.n + i], a.nu64[2 * a.n + i]};
		const D3 ny = {a.nu64[j], a.nu64[a.n + j], a.nu64[2 * a.n + j]};
		for (int q = 0; q < 4; ++q) s[q].x = st[q];
		near_dynamic<ALL4>(V, x0, nx, ny, J, k, R, s);
	}
	ar = al.x * s[3].x - al.y * s[3].y + s[1].x;
	ai = al.x * s[3].y + al.y * s[3].x + s[1].y;
	br = s[0].x + al.x * s[2].x - al.y * s[2].y;
	bi = s[0].y + al.x * s[2].y + al.y * s[2].x;
	if (diag) {
		ar += -0.5;
		br += al.x / 2.0;
		bi += al.y / 2.0;
	}
	const long long idx = (long long)f * a.kstride + (long long)j * a.ld + i;
	a.A[idx] = make_float2((float)ar, (float)ai);
	a.B[idx] = make_float2((float)br, (float)bi);
}

// Near pairs over uniformly spaced wavenumbers k_f = k_0 + f dk: one lane per
// (near pair, block of KBLK consecutive wavenumbers); at each of the 42 points
// e^{-i k r} comes from sincos once per block and is rotated by e^{-i dk r}
// (one FP64 complex product) from one wavenumber to the next; the other
// factors use the actual k_f.  Same terms as fp64_dynamic_kernel otherwise.
constexpr int KBLK = 4;

__global__ void __launch_bounds__(64) fp64_dynamic_rec_kernel(DynArgs a, double dk)
{
	const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
	const int nblk = (a.n_k + KBLK - 1) / KBLK;
	if (t >= (long long)a.n_near * nblk) return;
	const int fb = (int)(t / a.n_near);
	const int p = (int)(t % a.n_near);
	const int i = a.pi[p], j = a.pj[p];
	const Rules &R = *a.rules;
	D3 V[3];
	for (int v = 0; v < 3; ++v)
		V[v] = {a.X[(3 * v) * a.n + j], a.X[(3 * v + 1) * a.n + j], a.X[(3 * v + 2) * a.n + j]};
	const D3 x0 = {a.c[i], a.c[a.n + i], a.c[2 * a.n + i]};
	const D3 nx = {a.nu64[i], a.nu64[a.n + i], a.nu64[2 * a.n + i]};
	const D3 ny = {a.nu64[j], a.nu64[a.n + j], a.nu64[2 * a.n + j]};
	const double J = a.J[j];
	const int f0 = fb * KBLK;
	double kf[KBLK];
	double2 s[KBLK][4];
#pragma unroll
	for (int m = 0; m < KBLK; ++m) {
		kf[m] = a.k[min(f0 + m, a.n_k - 1)];
		for (int q = 0; q < 4; ++q) s[m][q] = make_double2(a.st[(size_t)p * 4 + q], 0.0);
	}
	const double nn = d3dot(nx, ny);
	for (int q = 0; q < 42; ++q) {
		const D3 y = tri_x(V, R.d14xi[q], R.d14eta[q]);
		const D3 rv = d3sub(y, x0);
		const double r2 = d3dot(rv, rv);
		const double rinv = rsqrt64(r2);
		const double r = r2 * rinv;
		const double g0 = rinv * (R.d14w[q] * J) * (1.0 / (4.0 * PI_D));
		const double rdny = d3dot(rv, ny) * rinv;
		const double rdnx = -d3dot(rv, nx) * rinv;
		double sn, cs, sd, cd;
		sincos64(kf[0] * r, &sn, &cs);
		sincos64(dk * r, &sd, &cd);
#pragma unroll
		for (int m = 0; m < KBLK; ++m) {
			dynamic_terms<ALL4>(cs, sn, kf[m] * r, g0, rinv, rdny, rdnx, nn, s[m]);
			// e^{-i (k + dk) r} = e^{-i k r} e^{-i dk r}
			const double c2 = cs * cd - sn * sd;
			sn = sn * cd + cs * sd;
			cs = c2;
		}
	}
#pragma unroll
	for (int m = 0; m < KBLK; ++m) {
		const int f = f0 + m;
		if (f >= a.n_k) break;
		const double2 al = a.alpha[f];
		const double ar = al.x * s[m][3].x - al.y * s[m][3].y + s[m][1].x;
		const double ai = al.x * s[m][3].y + al.y * s[m][3].x + s[m][1].y;
		const double br = s[m][0].x + al.x * s[m][2].x - al.y * s[m][2].y;
		const double bi = s[m][0].y + al.x * s[m][2].y + al.y * s[m][2].x;
		const long long idx = (long long)f * a.kstride + (long long)j * a.ld + i;
		a.A[idx] = make_float2((float)ar, (float)ai);
		a.B[idx] = make_float2((float)br, (float)bi);
	}
}

} // namespace nbk
