"""The bucket merge on two-word keys against the merge path, at the sizes where its shape and
the width of its packed words change."""
import numpy as np
import pytest

from test_gpu_parity import device_model
from test_gpu_reorder import _wide

pytestmark = pytest.mark.gpu


# bits below the bucket bits: 52 and fewer fit a packed word, more take the low word (at most
# 116, so 127 bits take 2^11 buckets or more); 2n items in the fewest buckets of 1637 at most: three items per thread up to 1188
@pytest.mark.parametrize("M,N", [(33, 33), (50, 50), (58, 58), (64, 64)])      # 65, 99, 115, 127 bits
@pytest.mark.parametrize("n", [1, 500, 800, 4400, 4900, 6400, 19_000])
@pytest.mark.parametrize("style,rule", [("dynamic", 0), ("dynamic", 1), ("integer", 0), ("integer", 2)])
def test_wide_buckets_equal_merge_path(gpu, M, N, n, style, rule):
    rng = np.random.default_rng(M * n)
    keys, m = _wide(M, N, n, rng)
    vals = rng.uniform(0.5, 3.0, m) * rng.choice([-1.0, 1.0], m)
    if style == "integer":
        vals = np.where(vals < 0, -1, 1) * rng.integers(1, 4, m)
    print(f"wide buckets {M}x{N} n={m} {style} rule={rule}", flush=True)
    st = {"dynamic": gpu.IsDynamicSemistochastic(), "integer": gpu.IsStochasticInteger()}[style]
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    out = []
    for mode in (2, 1):
        e = gpu._native.Engine(h.descriptor(), st.descriptor(), 5, 64 * m + 4096, 64 * m + 4096)
        e.set_radix_mode(mode)
        if rule:
            e.set_initiator(rule, 1.0)
        e.set_timing(True)
        e.upload(keys, vals)
        s = [e.step(i, -2.0, 1e-2) for i in range(1, 5)]
        out.append((e.download(), [(x.len, x.len_before, x.spawn_attempts, x.deaths) for x in s], set(e.kernel_times())))
        e.close()
    # (an integer population that grows tenfold in a step may outgrow its buckets and fall back)
    assert "bucket_merge" not in out[1][2] and "bucket_merge" in out[0][2]
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0][0], out[1][0][0])
    assert np.array_equal(out[0][0][1].view(np.uint64), out[1][0][1].view(np.uint64))


def test_addresses_that_agree_in_the_packed_word_fall_back(gpu):
    """127-bit stored keys that differ in their last 64 bits only: the packed words cannot tell
    them apart, the kernel notices and the step takes the merge path."""
    M = N = 64
    B, s = 127, 64
    mask = (1 << B) - 1
    c1 = 0x9E3779B97F4A7C15F39CC0605CEDC835 & mask          # the engine's storage order
    c2 = 0xD1B54A32D192ED03ABC98388FB8FAC03 & mask

    def mix(x):
        y = (x * c1) & mask
        y ^= y >> s
        y = (y * c2) & mask
        return y ^ (y >> s)

    def unmix(y):
        y ^= y >> s
        y = (y * pow(c2, -1, 1 << B)) & mask
        y ^= y >> s
        return (y * pow(c1, -1, 1 << B)) & mask

    rng = np.random.default_rng(12)
    base, m = _wide(M, N, 2000, rng)
    addr = {int(lo) | int(hi) << 64 for lo, hi in base.tolist()}
    for x in sorted(addr)[:5]:
        y = mix(x)
        assert unmix(y) == x
        for _ in range(10_000):
            z = unmix((y >> 64 << 64) | int.from_bytes(rng.bytes(8), "little"))
            if z != x and bin(z).count("1") == N:
                addr.add(z)
                break
        else:
            raise AssertionError("no second address found")
    keys = np.array([[k & (2 ** 64 - 1), k >> 64] for k in sorted(addr)], dtype=np.uint64)
    vals = rng.uniform(1.0, 3.0, len(keys))
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    out = []
    for mode in (2, 1):
        e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 5, 1 << 16, 1 << 16)
        e.set_radix_mode(mode)
        e.set_timing(True)
        e.upload(keys, vals)
        st = e.step(1, -2.0, 1e-3)
        out.append((e.download(), st.len_before, set(e.kernel_times())))
        e.close()
    assert "bucket_fallback" in out[0][2]
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0][0], out[1][0][0]) and np.array_equal(out[0][0][1], out[1][0][1])
