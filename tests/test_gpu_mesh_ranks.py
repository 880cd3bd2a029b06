"""Meshes by edge ranks and by a field's own grid values equal the general path.

PSR_DENSE_INDEX_MAX_CELLS=0 takes the sorted edge keys (and, for the field, key
searches); wrapping the field in a plain callback takes points, evaluation and
subtraction.  Grids of one cell, of odd sides, of several slabs with a ragged
last one, surfaces through nodes (value exactly zero), empty and all-crossing
grids, and boxes that leave the cube (refused either way).
"""
import numpy as np
import pytest

from parity import fixture_arrays

pytestmark = pytest.mark.gpu

GRIDS = [(2, 2, 2), (3, 5, 4), (17, 16, 18), (33, 9, 31), (40, 40, 40)]


def sphere(torch):
    return lambda p: (p * p).sum(1) - 0.25


def checker(torch):
    return lambda p: torch.where(((p * 8).floor().long().sum(1) & 1) == 0, 1.0, -1.0).float()


def plane(torch):  # passes exactly through nodes of odd grids
    return lambda p: p[:, 0].contiguous()


def empty(torch):
    return lambda p: torch.ones_like(p[:, 0])


@pytest.mark.parametrize("shape", GRIDS, ids=str)
@pytest.mark.parametrize("field", [sphere, checker, plane, empty], ids=lambda f: f.__name__)
def test_ranks_equal_sorted_edges(cuda, monkeypatch, field, shape):
    import torch
    from warp_psr_amd.meshing import extract_isosurface
    print(f"mesh ranks: {field.__name__} {shape}", flush=True)
    kw = dict(resolution=shape, bounds=((-0.75, -0.75, -0.75), (0.75, 0.75, 0.75)), slab_size=7)
    a = extract_isosurface(field(torch), **kw)
    monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", "0")
    b = extract_isosurface(field(torch), **kw)
    assert torch.equal(a.vertices, b.vertices) and torch.equal(a.indices, b.indices)
    assert a.metadata == b.metadata


@pytest.mark.parametrize("cells", [None, "0"], ids=["words", "searches"])
@pytest.mark.parametrize("backend,slab", [("sparse", 16), ("sparse", 5), ("dense", 16)])
@pytest.mark.parametrize("shape", [(2, 3, 2), (37, 20, 33)], ids=str)
def test_field_values_equal_callback(cuda, monkeypatch, shape, backend, slab, cells):
    import torch
    from warp_psr_amd import reconstruct
    from warp_psr_amd.meshing import extract_isosurface, extract_mesh
    if cells is not None:
        monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", cells)
    p, n = fixture_arrays("torus", 3000, "float")
    r = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), depth=6, full_depth=3)
    kw = dict(resolution=shape, bounds=((-0.99, -0.99, -0.3), (0.99, 0.99, 0.3)), backend=backend, slab_size=slab)
    iso = torch.full((1,), r.iso_value, dtype=torch.float32, device=cuda)
    a = extract_mesh(r, **kw)
    b = extract_isosurface(lambda q: r.evaluate(q)[0] - iso, device=cuda, **kw)
    assert len(a.vertices) or min(shape) == 2  # the small grid's nodes all lie outside the torus
    assert torch.equal(a.vertices, b.vertices) and torch.equal(a.indices, b.indices)
    assert a.metadata == b.metadata
    c = extract_mesh(r.field, iso_value=iso, **kw)
    assert torch.equal(a.vertices, c.vertices) and torch.equal(a.indices, c.indices)
    with pytest.raises(ValueError, match="nonfinite"):
        extract_mesh(r, resolution=shape, bounds=((-2.0, -2.0, -2.0), (2.0, 2.0, 2.0)), backend=backend)
