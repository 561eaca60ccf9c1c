// nbem_galquad.hpp -- Galerkin formalism on quadrilaterals (gfx950).
//
// Fields on quad_1 elements: constant (one dof per element, ND = 1) or
// isoparametric bilinear (one dof per mesh node, ND = 4 shape functions).
// Entry (dof_a, dof_b) = sum over element pairs (e, f) of
//   int_e N_a(x) int_f K(x, y) N_b(y) dy dx
// (nihu/core/double_integral.hpp:181-206 regular, :214-248 singular).
//
// Regular pairs (FP32): the organisation of the triangle kernel -- a wave
// holds a tile of up to 64 test elements (one per lane), the trial element is
// wave-uniform (scalar loads) -- with the N x N Gauss square rule of the
// pair's degree on both elements (degree = field complexity + the kernel's
// distance interval, or fixed; N = degree / 2 + 1).  Quadrilaterals are not
// flat, so every point row of the per-element tables carries its own unit
// normal: row = o (point - centre), |o|^2, n, o.n, w J N_b (b = 0..3), w J.
//   r = y - x = (c_f - c_e) + o_q - a_p,  r^2 = d^2 + u with
//   u = 2 (c_f - c_e - a_p).o_q + |o_q|^2 + |a_p|^2 - 2 (c_f - c_e).a_p;
//   r.n_q = (c_f - c_e - a_p).n_q + o_q.n_q;  r.n_p = (c_f - c_e - a_p).n_p + o_q.n_p;
// the phase as in the collocation kernels (FP64 fract(k d / 2 pi) per pair,
// k (r - d) = k u / (r + d) per point).  Nodal fields keep the lane-private
// LDS column slots of the triangle kernel (4 corners x GALQ_CS slots per lane)
// and add each evicted column with one global atomic per row node.
// Singular pairs (FP64, same mesh): coincident, edge- and corner-adjacent
// element pairs, one wave per pair over the 2048 / 1536 / 1280 points of the
// quad x quad rules, the element corners permuted to the rules' canonical
// configuration (nihu/core/singular_accelerator.hpp:283-325).

#pragma once

#include "nbem_galerkin.hpp"
#include "nbem_quad.hpp"

namespace nbk {

constexpr int GALQ_CS = 6;      // column-node slots per lane (nodal fields)
constexpr int GALQ_NMAX = 8;    // Gauss points per axis (degree <= 14)
constexpr int GALQ_ROW = 16;    // floats per point row

struct GalQArgs {
	int n_tiles, chunk;          // test wave tiles; trial sequence positions per chunk
	int tn, sn;                  // element counts of test / trial mesh (SoA strides)
	int same_mesh;
	const int *t_elem;           // nodal: [n_tiles][64] test element of each lane (-1: idle)
	const uint2 *t_contrib;      // nodal: [n_tiles][128] contributors lane * 4 + corner of local row r (lane r % 64)
	const int *t_rows;           // nodal: [n_tiles][128] node of each local row (-1: unused)
	const int *t_quad;           // test element nodes [4][tn]
	const GalRec *rec;           // trial sequence [sn] (constant fields: element order)
	const int *s_fin;            // nodal: [chunks][GALQ_CS] slot occupants at the end of a chunk
	const double *tc, *sc;       // centres x(0, 0) [3][n]
	const double *thr;           // trial distance thresholds [NTHR][sn]
	int split;                   // 1: the pairs below GalRec::near are left to galq_near_kernel
	const float *tq[GALQ_NMAX + 1], *sq[GALQ_NMAX + 1];   // point rows by points per axis
	int fixed_n;                 // > 0: the fixed rule's points per axis
	int complexity;              // field complexity: 1 constant, 2 nodal
	float k, k_revf;             // wavenumber, k / (2 pi)
	double k_rev;
	float ki;                    // imaginary part of a complex wavenumber (kernels with CK)
	float2 alpha;                // alpha / (4 pi)
	void *out;
	long long ld;
	int dtype, accumulate;
};

// trial point: offset o, |o|^2, unit normal n, o.n
struct GalqPoint { float ox, oy, oz, oo, nx, ny, nz, on; };

// test point of a pair: h = c_f - c_e - a_p, vp = |a_p|^2 - 2 (c_f - c_e).a_p, unit normal, h.n
struct GalqTest { float hx, hy, hz, vp, nx, ny, nz, rnx0; };

// from the first two quarters of a point row
template <int KM>
__device__ __forceinline__ GalqTest galq_test(float4 t0, float4 t1, const GalPair &P)
{
	GalqTest x;
	x.hx = __builtin_fmaf(0.5f, P.ex0, -t0.x);
	x.hy = __builtin_fmaf(0.5f, P.ey0, -t0.y);
	x.hz = __builtin_fmaf(0.5f, P.ez0, -t0.z);
	x.vp = t0.w - __builtin_fmaf(P.ex0, t0.x, __builtin_fmaf(P.ey0, t0.y, P.ez0 * t0.z));
	x.nx = t1.x; x.ny = t1.y; x.nz = t1.z;
	x.rnx0 = 0.0f;
	if (KM & (DLPT | HSP)) x.rnx0 = __builtin_fmaf(x.hx, x.nx, __builtin_fmaf(x.hy, x.ny, x.hz * x.nz));
	return x;
}

// One point pair's kernel value without 1 / (4 pi): SLP E, DLP -Q r.n_y, DLPt
// Q r.n_x, HSP n_x.n_y Q - (3Q - k^2 E r^2) r.n_x r.n_y / r^2 with
// E = e^{-i th}/r, G = E/r^2, Q = G (1 + i th), th = k r, th G = k e^{-i th}/r^2.
// CK: complex wavenumber k + i kim, the attenuation e^{kim r} on c and sn, Q
// gains -kim r G, k^2 becomes (k + i kim)^2.  w: a weight that multiplies the
// value.
template <int FAM, int KM, bool CK>
__device__ __forceinline__ float2 galq_point(const GalqPoint &y, const GalqTest &x, const GalPair &P, float k_revf,
	float k, float kim, float w = 1.0f)
{
	constexpr bool IM = FAM == HELM;
	const float u = __builtin_fmaf(2.0f * x.hx, y.ox, __builtin_fmaf(2.0f * x.hy, y.oy, __builtin_fmaf(2.0f * x.hz, y.oz, y.oo + x.vp)));
	const float r2 = P.d2f + u;
	const float rinv = __builtin_amdgcn_rsqf(r2);
	float c = 1.0f, sn = 0.0f;
	if (IM) {
		const float rd = u * __builtin_amdgcn_rcpf(__builtin_fmaf(r2, rinv, P.df));   // r - d
		const float tt = __builtin_fmaf(k_revf, rd, P.t0);
		c = __builtin_amdgcn_cosf(tt);
		sn = __builtin_amdgcn_sinf(tt);
		if (CK) {
			const float am = P.ad * __builtin_amdgcn_exp2f(kim * 1.4426950408889634f * rd);
			c *= am;
			sn *= am;
		}
	}
	float kr, ki = 0.0f;
	if (KM == SLP) {
		const float g = rinv * w;
		kr = g * c;
		if (IM) ki = -g * sn;
	} else {
		const float ri2 = rinv * rinv;
		const float g3 = rinv * ri2;
		const float Gr = g3 * c, Gi = IM ? -g3 * sn : 0.0f;
		const float kh = k * ri2;
		float Qr = IM ? __builtin_fmaf(kh, sn, Gr) : Gr;
		float Qi = IM ? __builtin_fmaf(kh, c, Gi) : 0.0f;
		if (CK) {
			const float kih = kim * ri2;
			Qr = __builtin_fmaf(-kih, c, Qr);
			Qi = __builtin_fmaf(kih, sn, Qi);
		}
		float rny = 0.0f;
		if (KM & (DLP | HSP)) rny = __builtin_fmaf(x.hx, y.nx, __builtin_fmaf(x.hy, y.ny, __builtin_fmaf(x.hz, y.nz, y.on)));
		if (KM == DLP) {
			const float rw = rny * w;
			kr = -Qr * rw; ki = -Qi * rw;
		} else {
			const float rnx = x.rnx0 + __builtin_fmaf(y.ox, x.nx, __builtin_fmaf(y.oy, x.ny, y.oz * x.nz));
			if (KM == DLPT) {
				const float rw = rnx * w;
				kr = Qr * rw; ki = Qi * rw;
			} else {
				const float nn = __builtin_fmaf(x.nx, y.nx, __builtin_fmaf(x.ny, y.ny, x.nz * y.nz));
				const float cf = rnx * rny * ri2;
				float hr, hi;
				if (CK) {
					const float kr2 = (k * k - kim * kim) * rinv, ki2 = 2.0f * k * kim * rinv;
					hr = 3.0f * Qr - (kr2 * c + ki2 * sn);
					hi = 3.0f * Qi - (ki2 * c - kr2 * sn);
				} else {
					const float kk = k * k * rinv;
					hr = __builtin_fmaf(3.0f, Qr, -kk * c);
					hi = __builtin_fmaf(3.0f, Qi, kk * sn);
				}
				kr = w * __builtin_fmaf(nn, Qr, -hr * cf);
				ki = w * __builtin_fmaf(nn, Qi, -hi * cf);
			}
		}
	}
	return make_float2(kr, ki);
}

// One pair over the diadic N x N rule: per test point p (lane's row) the
// trial sums S_b = sum_q K(x_p, y_q) w_q J_q N_b(q) (ND = 4) or w_q J_q
// (ND = 1), then blk[a][b] += w_p J_p N_a(p) S_b.
template <int FAM, int KM, int ND, bool CK = false>
__device__ __forceinline__ void galq_points(const float *tp, const float *sq_in, int nq, const GalPair &P,
	float k_revf, float k, float2 (&blk)[ND][ND], float kim)
{
	const auto sf = uni(sq_in);
	constexpr bool IM = FAM == HELM;
	for (int p = 0; p < nq; ++p) {
		const float4 t0 = *(const float4 *)(tp + GALQ_ROW * p);
		const float4 t1 = *(const float4 *)(tp + GALQ_ROW * p + 4);
		const float4 t2 = *(const float4 *)(tp + GALQ_ROW * p + 8);
		const float tw = tp[GALQ_ROW * p + 12];
		const GalqTest x = galq_test<KM>(t0, t1, P);
		float2 S[ND];
#pragma unroll
		for (int b = 0; b < ND; ++b) S[b] = zero2();
		for (int q = 0; q < nq; ++q) {
			const int o = GALQ_ROW * q;
			const float ox = sf[o], oy = sf[o + 1], oz = sf[o + 2];
			const GalqPoint y{ox, oy, oz, sf[o + 3], KM == SLP ? 0.0f : sf[o + 4], KM == SLP ? 0.0f : sf[o + 5],
				KM == SLP ? 0.0f : sf[o + 6], KM == SLP ? 0.0f : sf[o + 7]};
			const float2 K = galq_point<FAM, KM, CK>(y, x, P, k_revf, k, kim);
			const float kr = K.x, ki = K.y;
			if (ND == 1) {
				const float w = sf[o + 12];
				S[0].x = __builtin_fmaf(kr, w, S[0].x);
				if (IM || CK) S[0].y = __builtin_fmaf(ki, w, S[0].y);
			} else {
#pragma unroll
				for (int b = 0; b < ND; ++b) {
					const float w = sf[o + 8 + b];
					S[b].x = __builtin_fmaf(kr, w, S[b].x);
					if (IM || CK) S[b].y = __builtin_fmaf(ki, w, S[b].y);
				}
			}
		}
		// w J N_a of the test point (ND = 4), w J (ND = 1)
		const float w4[4] = {t2.x, t2.y, t2.z, t2.w};
		float wa[ND];
#pragma unroll
		for (int x = 0; x < ND; ++x) wa[x] = ND == 1 ? tw : w4[x];
#pragma unroll
		for (int x = 0; x < ND; ++x)
#pragma unroll
			for (int y = 0; y < ND; ++y) {
				blk[x][y].x = __builtin_fmaf(wa[x], S[y].x, blk[x][y].x);
				blk[x][y].y = __builtin_fmaf(wa[x], S[y].y, blk[x][y].y);
			}
	}
}

// The test element's points of the 2 x 2 rule in registers
struct GalqTest2 { float ax, ay, az, aa, nx, ny, nz, w; };

// The lowest rule of nodal fields, 2 x 2 Gauss points on both elements.  The
// shape functions at the points +-1/sqrt 3 are products of h+ = (1 + 1/sqrt 3)/2
// and h- = (1 - 1/sqrt 3)/2 per axis, so the sums with N_b over the points are
// two stages of h+ (v + rho v') and h+ (rho v + v'), rho = h-/h+ = 2 - sqrt 3:
// 8 FMAs instead of 16 for the four sums of a real part; the four factors h+
// ride on the test weights, which the point rows hold with them (column 13,
// formed in FP64 and rounded once: with an FP32 factor h+^4, 2.6e-8 too small
// for every entry, the matrices had 6 to 15 % more error).  Replaces blk.
template <int FAM, int KM, bool CK>
__device__ __forceinline__ void galq_two(const GalqTest2 (&t)[4], const float *sq_in, const GalPair &P, float k_revf, float k,
	float2 (&blk)[4][4], float kim)
{
	constexpr float RHO = 0.26794919243112270647f;
	const auto sf = uni(sq_in);
	// lo = v + rho u, hi = rho v + u
	auto stage = [](float2 v, float2 u, float2 &lo, float2 &hi) {
		lo = make_float2(__builtin_fmaf(RHO, u.x, v.x), __builtin_fmaf(RHO, u.y, v.y));
		hi = make_float2(__builtin_fmaf(RHO, v.x, u.x), __builtin_fmaf(RHO, v.y, u.y));
	};
	float2 W[2][2][4];      // [test xi point][test eta node][trial corner]
#pragma unroll
	for (int i = 0; i < 2; ++i) {
		float2 U[2][4];
#pragma unroll
		for (int j = 0; j < 2; ++j) {
			const GalqTest2 &p = t[2 * i + j];
			const GalqTest x = galq_test<KM>(make_float4(p.ax, p.ay, p.az, p.aa), make_float4(p.nx, p.ny, p.nz, 0.0f), P);
			float2 v[4];
#pragma unroll
			for (int q = 0; q < 4; ++q) {
				const int o = GALQ_ROW * q;
				const GalqPoint y{sf[o], sf[o + 1], sf[o + 2], sf[o + 3], KM == SLP ? 0.0f : sf[o + 4],
					KM == SLP ? 0.0f : sf[o + 5], KM == SLP ? 0.0f : sf[o + 6], KM == SLP ? 0.0f : sf[o + 7]};
				v[q] = galq_point<FAM, KM, CK>(y, x, P, k_revf, k, kim, sf[o + 12] * p.w);
			}
			// points xi outer, eta inner; corners (-,-), (+,-), (+,+), (-,+)
			float2 m0, m1, p0, p1;
			stage(v[0], v[1], m0, m1);
			stage(v[2], v[3], p0, p1);
			stage(m0, p0, U[j][0], U[j][1]);
			stage(m1, p1, U[j][3], U[j][2]);
		}
#pragma unroll
		for (int b = 0; b < 4; ++b) stage(U[0][b], U[1][b], W[i][0][b], W[i][1][b]);
	}
#pragma unroll
	for (int b = 0; b < 4; ++b) {
		stage(W[0][0][b], W[1][0][b], blk[0][b], blk[1][b]);
		stage(W[0][1][b], W[1][1][b], blk[3][b], blk[2][b]);
	}
}

// Grid: (test tiles / 4) x chunks, 256 lanes (4 waves, one test tile each).
// The lowest rule (nodal 2 x 2 points, constant one point at the centre) is
// what most pairs take: its test points stay in registers (a lane's rows of the
// tables are 64 different lines), its trial side comes through the scalar
// cache; see galerkin_regular_kernel for the rest.
template <int FAM, int KM, int ND, bool CK = false>
__global__ void __launch_bounds__(256) galq_regular_kernel(GalQArgs a)
{
	typedef GalSlots<4> Slots;
	__shared__ float2 acc_all[ND == 4 ? 4 * GALQ_CS * Slots::SLOT : 1];
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const int wg_tiles = (a.n_tiles + 3) >> 2;
	const int tile = (int)(blockIdx.x % wg_tiles) * 4 + wave;
	const int chunk = (int)(blockIdx.x / wg_tiles);
	if (tile >= a.n_tiles) return;     // no block-wide barriers below
	float2 *acc = acc_all + (ND == 4 ? wave * GALQ_CS * Slots::SLOT : 0);
	constexpr int ORDER = KM == SLP ? 1 : KM == HSP ? 3 : 2;

	int e;
	if (ND == 4) e = a.t_elem[tile * GAL_TILE + lane];
	else e = tile * GAL_TILE + lane < a.tn ? tile * GAL_TILE + lane : -1;
	const bool lane_ok = e >= 0;
	const int ee = lane_ok ? e : (ND == 4 ? a.t_elem[tile * GAL_TILE] : tile * GAL_TILE);
	const double cix = a.tc[ee], ciy = a.tc[a.tn + ee], ciz = a.tc[2 * a.tn + ee];
	int tv[4] = {-1, -1, -1, -1};
	if (a.same_mesh)
#pragma unroll
		for (int c = 0; c < 4; ++c) tv[c] = a.t_quad[c * a.tn + ee];
	GalRow<4> row[2];
	int node[4] = {-1, -1, -1, -1};
	int ncon = 0;
	if (ND == 4) {
#pragma unroll
		for (int r = 0; r < 2; ++r) row[r].set(a.t_contrib[(tile * 2 + r) * GAL_TILE + lane]);
#pragma unroll
		for (int t = 0; t < 4; ++t) node[t] = a.t_rows[tile * 2 * GAL_TILE + 32 * t + (lane >> 1)];
		ncon = max(row[0].used(), row[1].used());
#pragma unroll
		for (int s = 0; s < GALQ_CS; ++s) Slots::clear(acc, lane, s);
		if (lane < GALQ_CS) acc[lane * Slots::SLOT + 4 * GAL_TILE] = make_float2(0.0f, 0.0f);
	}
	GalPair P;
	P.nxx = P.nxy = P.nxz = 0.0f;
	P.nyx = P.nyy = P.nyz = 0.0f;
	P.dcny = P.dcnx = P.nn = 0.0f;
	P.ad = 1.0f;
	// the lowest rule's test side
	GalqTest2 tp2[ND == 4 ? 4 : 1];
	if (a.fixed_n <= 0) {
		const int nq = ND == 4 ? 4 : 1;
		const float *tp = a.tq[ND == 4 ? 2 : 1] + (size_t)ee * nq * GALQ_ROW;
#pragma unroll
		for (int p = 0; p < nq; ++p) {
			const float4 t0 = *(const float4 *)(tp + GALQ_ROW * p), t1 = *(const float4 *)(tp + GALQ_ROW * p + 4);
			tp2[p] = GalqTest2{t0.x, t0.y, t0.z, t0.w, t1.x, t1.y, t1.z, tp[GALQ_ROW * p + (ND == 4 ? 13 : 12)]};
		}
		if (ND == 1) { P.nxx = tp2[0].nx; P.nxy = tp2[0].ny; P.nxz = tp2[0].nz; }
	}
	const int i0 = chunk * a.chunk;
	const int i1 = min(i0 + a.chunk, a.sn);
	const auto rec = uni(a.rec);
	struct Head { double cx, cy, cz, share, near, far; float nx, ny, nz, w1; int v[4], ev[4], slots, f; };
	auto head = [&](int i) {
		const auto &r = rec[i];
		return Head{r.c[0], r.c[1], r.c[2], r.share, r.near[ORDER - 1], r.far[ORDER - 1], r.nu[0], r.nu[1], r.nu[2], r.w1,
			{r.node[0], r.node[1], r.node[2], r.node[3]}, {r.evict[0], r.evict[1], r.evict[2], r.evict[3]}, r.slots,
			r.elem};
	};
	Head nxt = head(i0);
	for (int i = i0; i < i1; ++i) {
		const Head h = nxt;
		nxt = head(i + 1 < i1 ? i + 1 : i);
		const int f = h.f;
		const int sl[4] = {h.slots & 31, (h.slots >> 5) & 31, (h.slots >> 10) & 31, (h.slots >> 15) & 31};
		if (ND == 4)
#pragma unroll
			for (int c = 0; c < 4; ++c)
				if (h.ev[c] >= 0) gal_flush<4, 2>(acc, lane, sl[c], h.ev[c], row, node, ncon, a);
		const double d2 = d2_pair(cix, ciy, ciz, h.cx, h.cy, h.cz);
		bool act = lane_ok && !(a.split && d2 < h.near);
		if (a.same_mesh && __ballot(d2 <= h.share) != 0) {
#pragma unroll
			for (int c = 0; c < 4; ++c)
				act = act && !(tv[c] == h.v[0] || tv[c] == h.v[1] || tv[c] == h.v[2] || tv[c] == h.v[3]);
		}
		float2 blk[ND][ND];
#pragma unroll
		for (int x = 0; x < ND; ++x)
#pragma unroll
			for (int y = 0; y < ND; ++y) blk[x][y] = zero2();
		if (__ballot(act) != 0) {
			const double dx = h.cx - cix, dy = h.cy - ciy, dz = h.cz - ciz;
			P.ex0 = (float)(2.0 * dx); P.ey0 = (float)(2.0 * dy); P.ez0 = (float)(2.0 * dz);
			P.d2f = (float)d2;
			double y = __builtin_amdgcn_rsq(d2);
			y = y * (1.5 - 0.5 * d2 * y * y);
			if (FAM == HELM) {
				const double d = d2 * y;
				double t = d * a.k_rev;
				t -= rint(t);
				P.df = (float)d;
				P.t0 = (float)t;
				if (CK) P.ad = __builtin_amdgcn_exp2f((float)(d * (a.ki * 1.4426950408889634)));
			} else {
				P.df = 0.0f; P.t0 = 0.0f;
			}
			const bool low = a.fixed_n <= 0 && act && !(d2 < h.far);
			if (low) {
				if (ND == 4) {
					galq_two<FAM, KM, CK>(reinterpret_cast<const GalqTest2 (&)[4]>(tp2), a.sq[2] + (size_t)f * 4 * GALQ_ROW, P,
						a.k_revf, a.k, reinterpret_cast<float2 (&)[4][4]>(blk), a.ki);
				} else {
					// the centres of both elements, with the normals there
					const float dcx = (float)dx, dcy = (float)dy, dcz = (float)dz;
					P.nyx = h.nx; P.nyy = h.ny; P.nyz = h.nz;
					if (KM & (DLP | HSP)) P.dcny = dcx * h.nx + dcy * h.ny + dcz * h.nz;
					if (KM & (DLPT | HSP)) P.dcnx = dcx * P.nxx + dcy * P.nxy + dcz * P.nxz;
					if (KM & HSP) P.nn = P.nxx * h.nx + P.nxy * h.ny + P.nxz * h.nz;
					const float2 K = gal_centres<FAM, KM, CK>(P, (float)y, a.k, a.ki);
					const float w = tp2[0].w * h.w1;
					blk[0][0] = make_float2(K.x * w, K.y * w);
				}
			}
			if (__ballot(act && !low) != 0) {
				// points per axis per lane; lanes are served one distinct rule at a time
				int nsel = -1;
				if (act && !low)
					nsel = a.fixed_n > 0 ? a.fixed_n : (a.complexity + table_degree<ORDER>(d2, uni(a.thr), a.sn, f)) / 2 + 1;
				for (;;) {
					const unsigned long long m = __ballot(nsel > 0);
					if (m == 0) break;
					const int N = __builtin_amdgcn_readlane(nsel, __ffsll((long long)m) - 1);
					const unsigned long long msel = __ballot(nsel == N);
					if ((msel >> __lane_id()) & 1ull) {
						const int nq = N * N;
						galq_points<FAM, KM, ND, CK>(a.tq[N] + (size_t)ee * nq * GALQ_ROW,
							a.sq[N] + (size_t)f * nq * GALQ_ROW, nq, P, a.k_revf, a.k, blk, a.ki);
						nsel = -1;
					}
				}
			}
		}
		if (ND == 1) {
			// singular entries and those of the close pairs: zero here, their passes add them
			if (lane_ok && (act || !a.accumulate)) {
				const float re = a.alpha.x * blk[0][0].x - a.alpha.y * blk[0][0].y;
				const float im = a.alpha.x * blk[0][0].y + a.alpha.y * blk[0][0].x;
				store_row(a.out, (long long)f * a.ld, e, a.dtype, a.accumulate, re, im);
			}
		} else if (act) {
#pragma unroll
			for (int y = 0; y < ND; ++y) Slots::add(acc, lane, sl[y], [&](int x) { return blk[ND > 1 ? x : 0][y]; });
		}
	}
	if (ND == 4) {
		const auto sfin = uni(a.s_fin);
		for (int s = 0; s < GALQ_CS; ++s) {
			const int v = sfin[chunk * GALQ_CS + s];
			if (v >= 0) gal_flush<4, 2>(acc, lane, s, v, row, node, ncon, a);
		}
	}
}

// The regular pairs of the higher distance-table degrees (4 x 4 points an
// element and more; close, not sharing a node): one wave per pair as in
// galerkin_near_kernel.
template <int FAM, int KM, int ND, bool CK = false>
__global__ void __launch_bounds__(256) galq_near_kernel(GalQArgs a, GalNear l)
{
	const int pair = (int)__builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
	if (pair >= l.n_pairs) return;
	const int lane = threadIdx.x & 63;
	const int e = uni(l.pi)[pair], f = uni(l.pj)[pair];
	constexpr int ORDER = KM == SLP ? 1 : KM == HSP ? 3 : 2;
	const auto tc = uni(a.tc), sc = uni(a.sc);
	const double dx = sc[f] - tc[e], dy = sc[a.sn + f] - tc[a.tn + e], dz = sc[2 * a.sn + f] - tc[2 * a.tn + e];
	const double d2 = __fma_rn(dz, dz, __fma_rn(dy, dy, dx * dx));
	const int N = __builtin_amdgcn_readfirstlane((a.complexity + table_degree<ORDER>(d2, uni(a.thr), a.sn, f)) / 2 + 1);
	const int nq = N * N;
	GalPair P;
	P.ex0 = (float)(2.0 * dx); P.ey0 = (float)(2.0 * dy); P.ez0 = (float)(2.0 * dz);
	P.d2f = (float)d2;
	P.df = P.t0 = 0.0f;
	P.ad = 1.0f;
	if (FAM == HELM) {
		double y = __builtin_amdgcn_rsq(d2);
		y = y * (1.5 - 0.5 * d2 * y * y);
		const double d = d2 * y;
		double t = d * a.k_rev;
		t -= rint(t);
		P.df = (float)d;
		P.t0 = (float)t;
		if (CK) P.ad = __builtin_amdgcn_exp2f((float)(d * (a.ki * 1.4426950408889634)));
	}
	const int groups = 64 / nq;
	const int g = lane / nq, q = lane - g * nq;
	float2 T[ND];
#pragma unroll
	for (int x = 0; x < ND; ++x) T[x] = zero2();
	const float4 *sr = (const float4 *)(a.sq[N] + ((size_t)f * nq + q) * GALQ_ROW);
	const float4 s0 = sr[0], s1 = sr[1], s2 = sr[2];
	const GalqPoint y{s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
	const float *tp = a.tq[N] + (size_t)e * nq * GALQ_ROW;
	for (int p = g < groups ? g : nq; p < nq; p += groups) {
		const float4 *tr = (const float4 *)(tp + GALQ_ROW * p);
		const GalqTest x = galq_test<KM>(tr[0], tr[1], P);
		const float4 t2 = tr[2];
		const float2 K = galq_point<FAM, KM, CK>(y, x, P, a.k_revf, a.k, a.ki);
		const float wa[4] = {ND == 1 ? tp[GALQ_ROW * p + 12] : t2.x, t2.y, t2.z, t2.w};
#pragma unroll
		for (int c = 0; c < ND; ++c) {
			T[c].x = __builtin_fmaf(wa[c], K.x, T[c].x);
			T[c].y = __builtin_fmaf(wa[c], K.y, T[c].y);
		}
	}
	// the trial weights w J N_b of the lane's point, then the sum over the
	// lanes (idle lanes hold zeros)
	const float wb[4] = {ND == 1 ? ((const float *)sr)[12] : s2.x, s2.y, s2.z, s2.w};
	auto entry = [&](int c, int b) {
		const float vr = wave_sum63(T[c].x * wb[b]);
		const float vi = FAM == HELM ? wave_sum63(T[c].y * wb[b]) : 0.0f;
		return make_float2(a.alpha.x * vr - a.alpha.y * vi, a.alpha.x * vi + a.alpha.y * vr);
	};
	if (ND == 1) {
		const float2 v = entry(0, 0);
		if (lane == 63) store_entry(a.out, (long long)f * a.ld + e, a.dtype, 1, v.x, v.y);
	} else {
		near_add<ND>(entry, l.t_dof, a.tn, e, l.s_dof, a.sn, f, a.out, a.ld, a.dtype);
	}
}

struct GalQSingArgs {
	int n_pairs;
	const int *pe, *pf, *pinfo;  // test / trial element, match | ind1 << 4 | ind2 << 8
	int n;                       // elements (SoA stride)
	const double *X;             // corners [12][n]
	const int *t_dof, *s_dof;    // row / column dof of each element corner [4][n] (nodes,
	                             // or the element at every corner for a constant field)
	const double *rule[3];       // canonical rules by match dimension: [points][5]
	int rule_n[3];
	double k;
	double ki;                   // imaginary part of a complex wavenumber (kernels with CK)
	double2 alpha;
	void *out;
	long long ld;
	int dtype;
};

// One wave per singular pair.  The rule's corner c of the test element is the
// element's corner (ind1 + c) % 4; of the trial element (ind2 + 1 - c) mod 4
// for a common edge (it runs the other way) and (ind2 + c) % 4 for a common
// corner.  The corner coordinates are permuted accordingly (a rotation or
// reflection of the reference square, |J| = 1), so that the shape function
// N_c at a rule point belongs to the permuted corner c; a reflection turns
// the cross product of the tangents around, and the unit normal is taken
// with the element's own orientation.
template <int FAM, int KM, int ND, bool CK = false>
__global__ void __launch_bounds__(64) galq_singular_kernel(GalQSingArgs a)
{
	const int p = blockIdx.x, lane = threadIdx.x;
	if (p >= a.n_pairs) return;
	const int e = a.pe[p], f = a.pf[p], info = a.pinfo[p];
	const int match = info & 15, i1 = (info >> 4) & 15, i2 = (info >> 8) & 15;
	int ct[4], cs[4];
	for (int c = 0; c < 4; ++c) {
		ct[c] = match == 2 ? c : (i1 + c) & 3;
		cs[c] = match == 2 ? c : match == 1 ? (i2 + 5 - c) & 3 : (i2 + c) & 3;
	}
	const int n = a.n;
	D3 Vt[4], Vs[4];
	for (int c = 0; c < 4; ++c) {
		Vt[c] = {a.X[(3 * ct[c]) * n + e], a.X[(3 * ct[c] + 1) * n + e], a.X[(3 * ct[c] + 2) * n + e]};
		Vs[c] = {a.X[(3 * cs[c]) * n + f], a.X[(3 * cs[c] + 1) * n + f], a.X[(3 * cs[c] + 2) * n + f]};
	}
	const Quad Qt = quad_from_corners(Vt), Qs = quad_from_corners(Vs);
	// a reflection of the corners (the trial element of an edge match)
	// reverses dx/dxi x dx/deta: the element's own normal is the opposite
	const double ot = ((ct[1] - ct[0]) & 3) == 1 ? 1.0 : -1.0;
	const double os = ((cs[1] - cs[0]) & 3) == 1 ? 1.0 : -1.0;
	const double *R = a.rule[match];
	const int nr = a.rule_n[match];
	double acc[ND * ND * 2];
	for (int q = 0; q < ND * ND * 2; ++q) acc[q] = 0.0;
	for (int q = lane; q < nr; q += 64) {
		const double txi = R[5 * q], teta = R[5 * q + 1], sxi = R[5 * q + 2], seta = R[5 * q + 3], w = R[5 * q + 4];
		D3 a1, b1, a2, b2;
		quad_dx(Qt, txi, teta, a1, b1);
		quad_dx(Qs, sxi, seta, a2, b2);
		const D3 n1 = d3cross(a1, b1), n2 = d3cross(a2, b2);
		const double s1 = d3dot(n1, n1), s2 = d3dot(n2, n2);
		const double i1 = rsqrt64(s1), i2 = rsqrt64(s2);
		const double J1 = s1 * i1, J2 = s2 * i2;
		const D3 x = quad_x(Qt, txi, teta), y = quad_x(Qs, sxi, seta);
		const D3 u1 = d3scale(n1, ot * i1), u2 = d3scale(n2, os * i2);
		const double2 K = CK ? kernel_value64_c<KM>(x, y, u1, u2, a.k, a.ki) : kernel_value64<FAM, KM>(x, y, u1, u2, a.k);
		const double wt = J1 * w, ws = J2;
		if (ND == 1) {
			acc[0] += wt * K.x * ws;
			acc[1] += wt * K.y * ws;
		} else {
			const double Nt[4] = {0.25 * (1 - txi) * (1 - teta), 0.25 * (1 + txi) * (1 - teta),
				0.25 * (1 + txi) * (1 + teta), 0.25 * (1 - txi) * (1 + teta)};
			const double Ns[4] = {0.25 * (1 - sxi) * (1 - seta), 0.25 * (1 + sxi) * (1 - seta),
				0.25 * (1 + sxi) * (1 + seta), 0.25 * (1 - sxi) * (1 + seta)};
			for (int x4 = 0; x4 < 4; ++x4)
				for (int y4 = 0; y4 < 4; ++y4) {
					const double ta = Nt[x4] * wt, sb = Ns[y4] * ws;
					acc[2 * (4 * x4 + y4)] += ta * K.x * sb;
					acc[2 * (4 * x4 + y4) + 1] += ta * K.y * sb;
				}
		}
	}
	for (int q = 0; q < ND * ND * 2; ++q)
		for (int off = 32; off >= 1; off >>= 1) acc[q] += __shfl_xor(acc[q], off);
	if (lane != 0) return;
	for (int x4 = 0; x4 < ND; ++x4)
		for (int y4 = 0; y4 < ND; ++y4) {
			const double vr = acc[2 * (ND * x4 + y4)], vi = acc[2 * (ND * x4 + y4) + 1];
			const double re = a.alpha.x * vr - a.alpha.y * vi, im = a.alpha.x * vi + a.alpha.y * vr;
			if (ND == 1) {
				store_entry64(a.out, (long long)f * a.ld + e, a.dtype, 1, re, im);
			} else {
				const int row = a.t_dof[ct[x4] * n + e], col = a.s_dof[cs[y4] * n + f];
				atomic_add_entry64(a.out, (long long)col * a.ld + row, a.dtype, re, im);
			}
		}
}

// identity (mass matrix) on quadrilaterals: the Gauss rule of degree
// shape orders + jacobian order 1 (nihu/core/single_integral.hpp:65-140):
// constant fields 4 J(0, 0) on the diagonal; nodal fields
// sum over the 2 x 2 points of N_a N_b J w per element, through the dof maps
// (a constant side names the element at every corner: the sums over its
// corners are the 2 x 2 rule of N_b J, NiHu's degree 2 for a constant test
// and a bilinear trial)
__global__ void galq_identity_kernel(void *out, long long ld, int n, const double *X, const int *t_map,
	const int *s_map, int nodal, int dtype, double ar, double ai)
{
	const int e = blockIdx.x * blockDim.x + threadIdx.x;
	if (e >= n) return;
	D3 V[4];
	for (int c = 0; c < 4; ++c) V[c] = {X[(3 * c) * n + e], X[(3 * c + 1) * n + e], X[(3 * c + 2) * n + e]};
	const Quad Q = quad_from_corners(V);
	if (!nodal) {
		D3 a, b;
		quad_dx(Q, 0.0, 0.0, a, b);
		const double m = 4.0 * d3norm(d3cross(a, b));
		store_entry64(out, (long long)e * ld + e, dtype, 1, ar * m, ai * m);
		return;
	}
	const double g = 0.57735026918962576451;   // 1 / sqrt 3, weights 1
	double M[4][4] = {};
	for (int q = 0; q < 4; ++q) {
		const double xi = (q & 2) ? g : -g, eta = (q & 1) ? g : -g;
		D3 a, b;
		quad_dx(Q, xi, eta, a, b);
		const double J = d3norm(d3cross(a, b));
		const double N[4] = {0.25 * (1 - xi) * (1 - eta), 0.25 * (1 + xi) * (1 - eta), 0.25 * (1 + xi) * (1 + eta),
			0.25 * (1 - xi) * (1 + eta)};
		for (int x = 0; x < 4; ++x)
			for (int y = 0; y < 4; ++y) M[x][y] += N[x] * N[y] * J;
	}
	for (int x = 0; x < 4; ++x)
		for (int y = 0; y < 4; ++y)
			atomic_add_entry64(out, (long long)s_map[y * n + e] * ld + t_map[x * n + e], dtype, ar * M[x][y], ai * M[x][y]);
}

} // namespace nbk
