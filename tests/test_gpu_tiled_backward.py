"""The tiled reverse sweeps against the launch-by-launch ones.

relax_tile chooses the form of the sweeps forwards and backwards: -1 reverses
launch by launch with scattered float64 atomics, a tile side gathers with the
transposed operator tile by tile.  The primal results are the same bits, so the
gradients differ only by the order of float64 sums: every entry is a sum of
some 1e5 products whose roundings (2^-53 each, growing like their square root)
stay under 1e-12 of the gradient's norm, and a float32 gradient adds one
rounding of the stored value (2^-24, twice for the accumulation onto zero).
"""
import numpy as np
import pytest

from parity import fixture_arrays

pytestmark = pytest.mark.gpu

CASES = [
    ("torus", 1500, "double", dict(depth=5, full_depth=2, iters=8)),
    ("torus", 2500, "double", dict(depth=6, full_depth=3, iters=7)),     # odd: the other buffer first
    ("sphere", 700, "double", dict(depth=5, full_depth=3, iters=1)),     # one visit
    ("torus", 2000, "double", dict(depth=6, full_depth=3, iters=16)),    # the tile tables' limit, two visit chunks
    ("torus", 1500, "float", dict(depth=6, full_depth=3, iters=8)),
    ("torus", 2000, "double", dict(depth=6, full_depth=3, iters=8, mixed=True)),
    ("sphere", 900, "double", dict(depth=5, full_depth=2, iters=9, point_weight=0.0)),
]


def gradients(torch, cuda, p, n, q, positions, **params):
    from warp_psr_amd import reconstruct_differentiable
    tp = torch.from_numpy(p).to(cuda).requires_grad_(positions)
    tn = torch.from_numpy(n).to(cuda).requires_grad_(True)
    r = reconstruct_differentiable(tp, tn, **params)
    v, g, _ = r.evaluate(torch.from_numpy(q).to(cuda), centered=True)
    ((v * v).sum() + 1e-3 * (g * g).sum()).backward()
    return [t.grad.cpu().numpy().astype(np.float64) for t in ([tp, tn] if positions else [tn])]


@pytest.mark.parametrize("tile", [8, 0, 40])
@pytest.mark.parametrize("positions", [False, True], ids=["normals", "positions"])
@pytest.mark.parametrize("shape,count,precision,params", CASES, ids=[f"{c[2]}-d{c[3]['depth']}-i{c[3]['iters']}" +
                                                                     ("-mixed" if c[3].get("mixed") else "") +
                                                                     ("-psr" if "point_weight" in c[3] else "") for c in CASES])
def test_tiled_equals_launched(cuda, shape, count, precision, params, positions, tile):
    import torch
    p, n = fixture_arrays(shape, count, precision)
    print(f"tiled backward: {shape} {count} {precision} {params} tile {tile} positions {positions}", flush=True)
    q = (p[::7] * p.dtype.type(1.02)).copy()
    want = gradients(torch, cuda, p, n, q, positions, relax_tile=-1, **params)
    got = gradients(torch, cuda, p, n, q, positions, relax_tile=tile, **params)
    bound = 2.0 ** -23 if precision == "float" else 1e-12
    for w, g in zip(want, got):
        assert np.isfinite(w).all() and np.linalg.norm(w) > 0
        assert np.linalg.norm(g - w) <= bound * np.linalg.norm(w)


@pytest.mark.parametrize("cells", ["0", "5000"])
def test_tiled_equals_launched_without_dense_index(cuda, monkeypatch, cells):
    """Tile tables built from sorted (tile, category) keys where a level has no dense index."""
    import torch
    monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", cells)
    p, n = fixture_arrays("torus", 2000, "double")
    params = dict(depth=6, full_depth=2)
    q = (p[::7] * 1.02).copy()
    want = gradients(torch, cuda, p, n, q, True, relax_tile=-1, **params)
    got = gradients(torch, cuda, p, n, q, True, **params)
    for w, g in zip(want, got):
        assert np.linalg.norm(g - w) <= 1e-12 * np.linalg.norm(w)
