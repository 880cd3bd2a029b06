"""The tree from bitmaps gives the keys of the tree from sorted candidates.

PSR_DENSE_INDEX_MAX_CELLS=0 takes the unique sort of every candidate brood,
the default the bitmap lattices.  Depth combinations cover the rule that picks
a level's requests (finer broods above the base level, moved-up requests from
it on): base level at, next to and far from the finest and at zero, complete
trees, one level, and levels whose lattice rows take one word, two words and
more; inputs cover the cube's faces, a handful of points and a plane.
"""
import numpy as np
import pytest

from parity import fixture_arrays

pytestmark = pytest.mark.gpu

DEPTHS = [dict(depth=1, full_depth=1), dict(depth=2, full_depth=0, base_depth=0), dict(depth=4, full_depth=4, base_depth=4),
          dict(depth=5, full_depth=4, base_depth=4), dict(depth=5, full_depth=5, base_depth=3), dict(depth=6, full_depth=2),
          dict(depth=7, full_depth=0, base_depth=0), dict(depth=7, full_depth=3, base_depth=1), dict(depth=8, full_depth=5, base_depth=2),
          dict(depth=10, full_depth=3, base_depth=3), dict(depth=11, full_depth=4, base_depth=2)]
INPUTS = [("sphere", 900, "float"), ("plane", 250, "double"), ("cluster", 1200, "double"), ("disconnected", 40, "float")]


def tree(torch, cuda, p, n, params):
    from warp_psr_amd import reconstruct
    r = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), point_weight=0.0, iters=1, **params)
    return [(r.diagnostics.array("tree_keys", d), r.diagnostics.array("basis_keys", d)) for d in range(params["depth"] + 1)]


@pytest.mark.parametrize("params", DEPTHS, ids=["-".join(f"{k[0]}{v}" for k, v in d.items()) for d in DEPTHS])
@pytest.mark.parametrize("shape,count,precision", INPUTS, ids=[i[0] for i in INPUTS])
def test_same_keys(cuda, monkeypatch, shape, count, precision, params):
    import torch
    p, n = fixture_arrays(shape, count, precision)
    print(f"tree bitmaps: {shape} {count} {params}", flush=True)
    bitmaps = tree(torch, cuda, p, n, params)
    monkeypatch.setenv("PSR_DENSE_INDEX_MAX_CELLS", "0")
    sorted_ = tree(torch, cuda, p, n, params)
    for d, ((ta, ba), (tb, bb)) in enumerate(zip(bitmaps, sorted_)):
        np.testing.assert_array_equal(ta, tb, err_msg=f"tree keys of level {d}")
        np.testing.assert_array_equal(ba, bb, err_msg=f"basis keys of level {d}")
