"""The base solve's one-workgroup V-cycle against the oracle, bit for bit.

Base depths 1 to 3 run every level in it (27, 125 and 729 rows in 1, 2 and 12
waves), depth 4 the levels below its 4,913 rows (a cycle then starts from zero
in the middle of the launches), depth 0 only the root solve.  Several cycles
start from the last one's solution; one sweep and an odd number; without
screening the root solve's conjugate gradient meets a singular operator.
"""
import numpy as np
import pytest

import oracle
from parity import compare_stages, fixture_arrays

pytestmark = pytest.mark.gpu

STAGES = [("point_load", "solve"), ("normal_load", "solve"), ("rhs", "solve"), ("matrix_values", "solve"), ("matrix_columns", "solve"),
          ("corrections", "solve"), ("coefficients", False), ("iso", False), ("cg_runs", False)]


@pytest.mark.parametrize("precision", ["float", "double"])
@pytest.mark.parametrize("weight", [0.0, 2.0])
@pytest.mark.parametrize("cycles,iters", [(1, 8), (3, 1), (2, 3)])
@pytest.mark.parametrize("base,full", [(0, 2), (1, 1), (2, 3), (3, 3), (4, 4)])
def test_base_solve_bit_exact(cuda, base, full, cycles, iters, weight, precision):
    import torch
    from warp_psr_amd import reconstruct
    p, n = fixture_arrays("torus", 1200, precision)
    params = dict(depth=5, full_depth=full, base_depth=base, point_weight=weight, base_v_cycles=cycles, iters=iters)
    print(f"base cycle: {params} {precision}", flush=True)
    gpu = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), **params)
    ref = oracle.reconstruct(p, n, **params)
    bad = compare_stages(gpu.diagnostics, ref, ref.params, STAGES)
    assert not bad, "; ".join(f"{s}[{lv}] {m}" for s, lv, m in bad[:5])
