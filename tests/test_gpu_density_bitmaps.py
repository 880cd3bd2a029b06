"""Aggregates, density nodes and densities from bitmaps equal those from sorts,
bit for bit.

PSR_DENSE_INDEX_MAX_CELLS=0 takes the sorts (parents by octant, splat records
by Morton order and node), the default the bitmaps, whose gathers add in the
same orders.  Kernel depths from 0 to the finest, rows of less than a word, one
word and several, clouds on the cube's faces (neighbours outside the grid), a
plane, a cluster whose nodes gather from all 27 cells, and a dense cloud on
both sides of the centre planes, where Morton order changes at the top bit.
"""
import numpy as np
import pytest

from parity import fixture_arrays, same

pytestmark = pytest.mark.gpu

DEPTHS = [dict(depth=1, full_depth=1, kernel_depth=1), dict(depth=4, full_depth=2, kernel_depth=0),
          dict(depth=5, full_depth=3, kernel_depth=5), dict(depth=6, full_depth=2), dict(depth=7, full_depth=3, kernel_depth=7),
          dict(depth=8, full_depth=3), dict(depth=10, full_depth=4)]
INPUTS = [("sphere", 900, "float"), ("plane", 250, "double"), ("cluster", 3000, "double"), ("disconnected", 40, "float"),
          ("block", 4000, "double")]


def cloud(shape, count, precision):
    if shape != "block":
        return fixture_arrays(shape, count, precision)
    rng = np.random.default_rng(3)
    p = rng.uniform(-1, 1, (count, 3)) * np.array([1.0, 0.2, 0.2])
    n = rng.normal(size=(count, 3))
    return p, n


def stages(torch, cuda, p, n, params):
    from warp_psr_amd import reconstruct
    r = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), point_weight=0.0, iters=1, **params)
    kd = params.get("kernel_depth", max(params["depth"] - 2, 0))
    out = {("densities", -1): r.diagnostics.array("densities"), ("depths_and_weights", -1): r.diagnostics.array("depths_and_weights")}
    for d in range(params["depth"] + 1):
        for name in ("aggregate_keys", "aggregate_values") + (("density_keys", "density_values") if d <= kd else ()):
            out[name, d] = r.diagnostics.array(name, d)
    return out


@pytest.mark.parametrize("params", DEPTHS, ids=["-".join(f"{k[0]}{v}" for k, v in d.items()) for d in DEPTHS])
@pytest.mark.parametrize("shape,count,precision", INPUTS, ids=[i[0] for i in INPUTS])
def test_same_bits(cuda, monkeypatch, shape, count, precision, params):
    import torch
    p, n = cloud(shape, count, precision)
    print(f"density bitmaps: {shape} {count} {params}", flush=True)
    bitmaps = stages(torch, cuda, p, n, params)
    monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", "0")
    sorted_ = stages(torch, cuda, p, n, params)
    for k in bitmaps:
        assert same(bitmaps[k], sorted_[k]), k
