"""The kept blocks of a field mesh, without a GPU: one per range and device, the
latest 32, built again when an array has changed."""

import threading
import time
from types import SimpleNamespace

import numpy as np
import pytest

from nihu_amd import nbem


def test_blocks(monkeypatch):
    mesh = object.__new__(nbem.Mesh)
    mesh.nodes, mesh.tris = np.arange(150.0).reshape(50, 3), np.arange(48).reshape(16, 3)
    monkeypatch.setattr(nbem, "Mesh", lambda nodes, tris: SimpleNamespace(nodes=nodes, tris=tris))
    a = mesh.block(0, 8, 0)
    assert a.tris.shape == (8, 3) and mesh.block(0, 8, 0) is a
    b = mesh.block(0, 8, 1)
    assert b is not a and mesh.block(0, 8, 0) is a and mesh.block(0, 8, 1) is b
    mesh.tris[3, 0] += 1
    assert mesh.block(0, 8, 0) is not a
    for r in range(40):
        mesh.block(r % 16, r % 16 + 1, 2 + r // 16)
    assert len(mesh._blocks) == 32


def bare(n=16):
    mesh = object.__new__(nbem.Mesh)
    mesh.nodes, mesh.tris = np.arange(9.0 * n).reshape(3 * n, 3), np.arange(3 * n).reshape(n, 3)
    return mesh


def test_block_holds_its_own_nodes(monkeypatch):
    # not the whole node array: a block stays when only nodes outside it change
    mesh = bare()
    monkeypatch.setattr(nbem, "Mesh", lambda nodes, tris: SimpleNamespace(nodes=nodes, tris=tris))
    a, b = mesh.block(0, 4), mesh.block(4, 16)
    assert len(a.nodes) == 12 and np.array_equal(a.nodes[a.tris], mesh.nodes[mesh.tris[:4]])
    mesh.nodes[30] += 1.0
    assert mesh.block(0, 4) is a and mesh.block(4, 16) is not b
    mesh.tris[5, 0] = 48
    with pytest.raises(ValueError):
        mesh.block(4, 16)


def test_latest_used_blocks_stay(monkeypatch):
    mesh = bare(64)
    monkeypatch.setattr(nbem, "Mesh", lambda nodes, tris: SimpleNamespace(nodes=nodes, tris=tris))
    first, second = mesh.block(0, 1), mesh.block(1, 2)
    for r in range(2, 33):
        mesh.block(r, r + 1)
        assert mesh.block(0, 1) is first
    assert mesh.block(1, 2) is not second
    monkeypatch.setattr(nbem, "KEPT_ELEMENTS", 40)
    mesh.block(0, 30)
    assert sum(k[2] - k[1] for k in mesh._blocks) <= 40
    large = mesh.block(0, 64)
    assert large.tris.shape == (64, 3) and (0, 0, 64) not in mesh._blocks


def test_threads_share_a_block(monkeypatch):
    mesh, built = bare(), []

    def slow(nodes, tris):
        built.append(tris)
        time.sleep(0.05)
        return SimpleNamespace(nodes=nodes, tris=tris)

    monkeypatch.setattr(nbem, "Mesh", slow)
    got = []
    threads = [threading.Thread(target=lambda: got.append(mesh.block(0, 8))) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(built) == 1 and all(g is got[0] for g in got)
