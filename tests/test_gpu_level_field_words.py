"""LevelField.evaluate through node words gives the bits of the searching
device_field().evaluate, over a caller's keys and coefficients: with and
without cumulative coefficients, levels of one word a column, two and more,
levels without nodes, one key, no keys (refused), the last key's pair at the array's
end, depths beyond the words, and keys that have no words (not ascending,
repeated, off the grid), which are searched as before."""
import numpy as np
import pytest

from parity import same

pytestmark = pytest.mark.gpu


def keys_of(depth, fill, rng, skip=()):
    out = []
    for d in range(depth + 1):
        n = 2 ** d + 1
        if d in skip:
            continue
        c = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), -1).reshape(-1, 3) if d <= 4 else rng.integers(0, n, (fill, 3))
        c = c[rng.uniform(size=len(c)) < 0.7] if d > 1 else c
        if d > 4:  # runs along z and both ends of the rows
            c = np.concatenate([c, c + [0, 0, 1], c + [0, 1, 0], c + [1, 0, 0], c * [1, 1, 0], c * [1, 1, 0] + [0, 0, n - 1]])
            c = c[(c < n).all(1)]
        out.append((np.int64(d) << 48) | (c[:, 0].astype(np.int64) << 32) | (c[:, 1] << 16) | c[:, 2])
    return np.unique(np.concatenate(out))


def compare(torch, cuda, keys, depth, dtype, cumulative, rng):
    from warp_psr_amd import LevelField
    K = len(keys)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(cuda)  # noqa: E731
    f = LevelField(t(keys), t(rng.normal(size=K).astype(dtype)), np.eye(3) * 0.5, [0.25, 0.125, 0.0], depth, 0.5,
                   cumulative=t(rng.normal(size=K).astype(dtype)) if cumulative else None)
    knots = np.concatenate([rng.integers(0, 2 ** d + 1, 6) / 2 ** d for d in range(depth + 1)])
    knots = np.concatenate([[0.0, 1.0, -0.01, 1.01, np.nan, np.inf], knots, np.nextafter(knots, -1), np.nextafter(knots, 2)])
    cube = np.concatenate([rng.uniform(0, 1, (3000, 3)), rng.choice(knots, (3000, 3))])
    q = t(((cube - [0.25, 0.125, 0.0]) * 2).astype(dtype))
    for a, b in zip(f.evaluate(q), f.device_field().evaluate(q)):
        assert same(a.cpu().numpy(), b.cpu().numpy())
    return f


@pytest.mark.parametrize("cumulative", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("depth", [0, 1, 4, 5, 6, 9, 10])
def test_same_bits(cuda, depth, dtype, cumulative):
    import torch
    rng = np.random.default_rng(depth)
    print(f"level field words: depth {depth} {dtype.__name__} cumulative {cumulative}", flush=True)
    f = compare(torch, cuda, keys_of(depth, 4000, rng), depth, dtype, cumulative, rng)
    assert (f._words is None) == (depth > 9)
    if depth == 6:
        compare(torch, cuda, keys_of(depth, 4000, rng, skip=(3, 6)), depth, dtype, cumulative, rng)
    if depth == 5:
        one = np.array([(5 << 48) | (32 << 32) | (32 << 16) | 32], dtype=np.int64)
        for keys in (one, one - (1 << 48) * 5):
            compare(torch, cuda, keys, depth, dtype, cumulative, rng)
        with pytest.raises(ValueError, match="field must be a psr_result_field view"):
            compare(torch, cuda, one[:0], depth, dtype, cumulative, rng)


@pytest.mark.parametrize("fault", ["swapped", "repeated", "off-grid", "too-deep"])
def test_keys_without_words_are_searched(cuda, fault):
    import torch
    rng = np.random.default_rng(3)
    keys = keys_of(6, 2000, rng)
    if fault == "swapped":
        keys[[40, 400]] = keys[[400, 40]]
    elif fault == "repeated":
        keys[50] = keys[51]
    elif fault == "off-grid":
        keys[-1] = (6 << 48) | (70 << 32) | (3 << 16) | 2
    else:
        keys[-1] = 7 << 48
    f = compare(torch, cuda, keys, 6, np.float64, True, rng)
    assert f._words is not None and int(f._words[1]) == 0
