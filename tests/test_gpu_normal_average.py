"""The normal average's chains, scanned in parallel, against the serial sum.

The result must be the serial chain's bits: chunks of 4,096 values (sizes on both
sides of one and several), binade crossings (every doubling of the sum, many in
the first chunk), halfway cases (float32 sums of short values), zeros in front
(skipped contributions longer than a chunk) and weights far apart (one cell with
many samples, whose value crosses binades by itself).
"""
import numpy as np
import pytest

import oracle
from parity import fixture_arrays, same

pytestmark = pytest.mark.gpu


def cloud(count, precision, zeros, heavy):
    p, n = fixture_arrays("sphere", count, precision)
    # cells whose normals cancel contribute nothing
    p, n = np.concatenate([p[:zeros], p]), np.concatenate([-n[:zeros], n])
    if heavy:
        p = np.concatenate([p, np.repeat(p[-count // 2:1 - count // 2], heavy, axis=0)])
        n = np.concatenate([n, np.repeat(n[-count // 2:1 - count // 2], heavy, axis=0)])
    return p, n


@pytest.mark.parametrize("precision", ["float", "double"])
@pytest.mark.parametrize("count,depth,zeros,heavy", [(8, 3, 0, 0), (600, 6, 3, 0), (4200, 8, 0, 0), (9000, 8, 5000, 0),
                                                     (9000, 8, 0, 3000), (40000, 8, 0, 0), (3000, 4, 2999, 0)])
def test_average_is_the_serial_sum(cuda, count, depth, zeros, heavy, precision):
    import torch
    from warp_psr_amd import reconstruct
    p, n = cloud(count, precision, zeros, heavy)
    print(f"normal average: {count} points depth {depth} {precision}, {zeros} cancelled normals, {heavy} in one cell", flush=True)
    params = dict(depth=depth, full_depth=2, iters=1)
    gpu = reconstruct(torch.from_numpy(p).to(cuda), torch.from_numpy(n).to(cuda), **params)
    ref = oracle.reconstruct(p, n, **params)
    assert same(gpu.diagnostics.array("normal_average"), ref.array("normal_average"))
