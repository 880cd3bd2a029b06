"""Field lookups through node words: queries at the edges of cells, words and
levels give the oracle's bits, with words on every level, on some levels (the
deeper ones through column tables) and on none.

A level's column holds 2^d + 1 nodes in words of 32, so depths 5 and 6 have
cells whose two z nodes lie in different words (z = 31, 32 and 63, 64) and a
last word with a single node.  Queries are put on knots of every level (where
the left cell owns the point), just beside them, on the cube's faces and
outside it.
"""
import numpy as np
import pytest

import oracle
from parity import fixture_arrays, same

pytestmark = pytest.mark.gpu

CASES = [("sphere", 900, "float", dict(depth=5, full_depth=2)), ("torus", 3000, "double", dict(depth=6, full_depth=3)),
         ("plane", 300, "float", dict(depth=1, full_depth=1)), ("torus", 2000, "double", dict(depth=6, full_depth=5, mixed=True))]
# dense cells up to: every level, levels 0..4 (17^3 cells), no level
LIMITS = {"all": None, "to-depth-4": "5000", "none": "0"}


def edge_queries(inverse, depth, dtype, rng):
    """Model-space points whose cube coordinates are knots k / 2^d, knots one ulp to either side, faces and beyond."""
    axis = [np.array([0.0, 1.0, -1e-3, 1.0 + 1e-3])]
    for d in range(depth + 1):
        k = rng.integers(0, 2 ** d + 1, 12) / 2 ** d
        axis += [k, np.nextafter(k, -1), np.nextafter(k, 2)]
    axis += [rng.uniform(0, 1, 16)] + [np.array([31, 32, 33, 63, 64]) / 2 ** d for d in (5, 6)]
    axis = np.concatenate(axis)
    cube = rng.choice(axis, size=(6000, 3))
    m = np.asarray(inverse, dtype=np.float64).reshape(4, 4)
    return (cube @ m[:3, :3].T + m[:3, 3]).astype(dtype)


@pytest.mark.parametrize("limit", list(LIMITS))
@pytest.mark.parametrize("shape,count,precision,params", CASES, ids=[f"{c[0]}-d{c[3]['depth']}-{c[2]}" for c in CASES])
def test_edges_match_oracle(cuda, monkeypatch, limit, shape, count, precision, params):
    import torch
    from warp_psr_amd import reconstruct
    if LIMITS[limit] is not None:
        monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", LIMITS[limit])
    p, n = fixture_arrays(shape, count, precision)
    print(f"node words: {shape} depth {params['depth']} {precision}, {limit}", flush=True)
    gpu = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), **params)
    ref = oracle.reconstruct(p, n, **params)
    q = edge_queries(gpu.metadata["cube_to_model"], params["depth"], p.dtype, np.random.default_rng(7))
    values, grads, valid = gpu.evaluate(torch.from_numpy(q).to(cuda))
    rv, rg, rvalid = ref.evaluate(q)
    np.testing.assert_array_equal(valid.cpu().numpy(), rvalid)
    assert same(values.cpu().numpy(), rv)
    assert same(grads.cpu().numpy(), rg)
    assert gpu.iso_value == ref.iso_value
