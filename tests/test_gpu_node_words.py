"""Operators, transfers, loads and tile tables through node words, and beside
levels that have none.

With every level within the dense limit all lookups go through words; with the
limit between two levels, words and column tables meet in the prolongation,
restriction, cross operator and parent loads of the first level beyond it; with
no dense cells no level has words.  Stage arrays must equal the oracle's bit for
bit either way.  Depth 5 is the first level whose columns take two words (nodes
31 and 32 side by side), depth 7 has five; base depth 0 and 1, a plane of
points on a cell face and a cloud that leaves levels empty are the edges.
"""
import numpy as np
import pytest

import oracle
from parity import compare_stages, fixture_arrays

pytestmark = pytest.mark.gpu

# words for: every level, levels 0..5 (33^3 cells), levels 0..4, none
LIMITS = {"all": None, "to-depth-5": "36000", "to-depth-4": "5000", "none": "0"}
CASES = [
    ("torus", 3000, "float", dict(depth=5, full_depth=4)),
    ("sheets", 3000, "double", dict(depth=7, full_depth=2)),
    ("torus", 2500, "double", dict(depth=6, full_depth=5, base_depth=1, mixed=True)),
    ("plane", 400, "float", dict(depth=6, full_depth=1, base_depth=0)),
    ("plane", 16, "double", dict(depth=5, full_depth=1)),
    ("sphere", 200, "double", dict(depth=7, full_depth=2, samples_per_node=40.0)),
]


@pytest.mark.parametrize("limit", list(LIMITS))
@pytest.mark.parametrize("shape,count,precision,params", CASES, ids=[f"{c[0]}{c[1]}-d{c[3]['depth']}-{c[2]}" for c in CASES])
def test_stages_match_oracle(cuda, monkeypatch, limit, shape, count, precision, params):
    import torch
    from warp_psr_amd import reconstruct
    if LIMITS[limit] is not None:
        monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", LIMITS[limit])
    p, n = fixture_arrays(shape, count, precision)
    print(f"node words: {shape} {count} depth {params['depth']} {precision}, {limit}", flush=True)
    gpu = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), **params)
    ref = oracle.reconstruct(p, n, **params)
    mismatches = compare_stages(gpu.diagnostics, ref, ref.params)
    assert not mismatches, "\n".join(f"{s}[{lv}]: {m}" for s, lv, m in mismatches[:20])


@pytest.mark.parametrize("limit", list(LIMITS)[1:])
def test_gradients_match(cuda, monkeypatch, limit):
    """The reverse pass looks the same nodes up: sums of float64 products in another order of atomics (roundings of
    2^-53 each, some 1e5 of them, growing like their square root: under 1e-12 of the norm)."""
    import torch
    from warp_psr_amd import reconstruct_differentiable
    p, n = fixture_arrays("torus", 2000, "double")
    q = torch.from_numpy((p[::7] * 1.02).copy()).to(cuda)

    def gradient():
        tn = torch.from_numpy(n).to(cuda).requires_grad_(True)
        r = reconstruct_differentiable(torch.from_numpy(p).to(cuda), tn, depth=6, full_depth=3)
        v, g, _ = r.evaluate(q, centered=True)
        ((v * v).sum() + 1e-3 * (g * g).sum()).backward()
        return tn.grad.cpu().numpy()

    want = gradient()
    monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", LIMITS[limit])
    got = gradient()
    assert np.linalg.norm(want) > 0 and np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(want)
