"""The kept blocks of a field mesh, without a GPU: one per range and device, the
latest 32, built again when an array has changed."""

from types import SimpleNamespace

import numpy as np

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
