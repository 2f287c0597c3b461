"""The bucket merge's shapes (three, four and five items per thread) and the sorts with nine-bit
digits, at the sizes where the choice between them changes."""
import numpy as np
import pytest

from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


def _chain_vector(M, N, n, rng):
    """n distinct addresses of M modes (N bosons thrown at random) with values in (1, 2), so that
    every entry makes one spawn attempt and a step has exactly n records."""
    occ = rng.multinomial(N, np.full(M, 1.0 / M), size=2 * n).astype(np.uint64)
    keys = np.zeros(len(occ), dtype=np.uint64)
    at = np.zeros(len(occ), dtype=np.uint64)
    one = np.uint64(1)
    for m in range(M):
        keys |= ((one << occ[:, m]) - one) << at
        at += occ[:, m] + one
    keys = np.unique(keys)
    keys = np.sort(rng.permutation(keys)[:n])
    assert len(keys) == n
    return keys, rng.uniform(1.01, 1.99, n) * rng.choice([-1.0, 1.0], n)


# 2n items in the fewest buckets of 2092 at most on average: up to 1188 take three items per
# thread, up to 1637 four, more five
@pytest.mark.parametrize("mean,buckets", [(1060, 16), (1180, 16), (1200, 16), (1630, 16), (1650, 16),
                                          (2080, 16), (1100, 256), (1100, 512), (2080, 512)])
def test_bucket_shapes_equal_merge_path(gpu, mean, buckets):
    M = N = 20
    n = mean * buckets // 2
    rng = np.random.default_rng(n)
    keys, vals = _chain_vector(M, N, n, rng)
    print(f"bucket shape mean={mean} buckets={buckets} n={n}", flush=True)
    out = []
    for mode in (2, 1):
        h = device_model(gpu, "real", M, N, 4.0, 1.0)
        e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 5, 4 * n, 4 * n)
        e.set_radix_mode(mode)
        e.set_timing(True)
        e.upload(keys, vals)
        st = [e.step(s, -2.0, 1e-3) for s in (1, 2)]
        out.append((e.download(), [(x.len, x.len_before, x.spawn_attempts) for x in st], set(e.kernel_times())))
        e.close()
    assert "bucket_merge" in out[0][2] and "bucket_fallback" not in out[0][2]
    assert "bucket_merge" not in out[1][2]
    assert out[0][1] == out[1][1] and out[0][1][0][2] == n
    assert np.array_equal(out[0][0][0], out[1][0][0])
    assert np.array_equal(out[0][0][1].view(np.uint64), out[1][0][1].view(np.uint64))


# 9, 17, 18, 27 and 36 bits are sorted in nine-bit digits, 16, 19 and 37 in eight-bit ones
@pytest.mark.parametrize("bits", [9, 16, 17, 18, 19, 27, 36, 37])
@pytest.mark.parametrize("n,noalloc", [(1, False), (4095, True), (4097, False), (70_001, True)])
def test_digit_widths_sort_stably(gpu, bits, n, noalloc):
    rng = np.random.default_rng(bits * n)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64)
    keys[rng.random(n) < 0.5] = keys[0]          # a long run of one key
    keys[-1] = (1 << bits) - 1
    vals = rng.normal(size=n) * 10.0 ** rng.integers(-8, 9, n)   # sums depend on their order
    k, v = gpu.annihilate(keys, vals, noalloc=noalloc)
    want = {}
    for key, val in zip(keys.tolist(), vals.tolist()):
        want[key] = want.get(key, 0.0) + val
    want = {a: b for a, b in sorted(want.items()) if b != 0.0}
    assert k.tolist() == list(want)
    assert v.tolist() == list(want.values())
