"""The rule that cuts a step's records into buckets: how many, and the items per thread of the
kernel that merges them, on both sides of each line."""
import numpy as np
import pytest

from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model
from test_gpu_reorder import _wide

pytestmark = pytest.mark.gpu


def _first_cut(gpu, M, N, items, style=None):
    """(bits, items per thread) of a step of `items` records and entries in equal parts."""
    n = items // 2
    rng = np.random.default_rng(items + M)
    if M + N - 1 > 64:
        keys, m = _wide(M, N, 2 * n, rng)
        keys = keys[np.sort(rng.permutation(m)[:n])]
        vals = rng.uniform(1.01, 1.99, n)
    else:
        keys, vals = _chain_vector(M, N, n, rng)
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), (style or gpu.IsDynamicSemistochastic()).descriptor(), 5, 64 * n + 64,
                           64 * n + 64)
    e.set_timing(True)
    e.upload(keys, vals)
    st = e.step(1, -2.0, 1e-3)
    cut, labels = e.last_cut(), set(e.kernel_times())
    if style is None:
        assert st.spawn_attempts == n
        e.set_radix_mode(1)
        e.step(2, -2.0, 1e-3)
        assert e.last_cut() == (-1, 0)
    e.close()
    assert not labels & {"bucket_retry", "bucket_fallback"}
    assert ("bucket_merge" in labels) == (cut[0] >= 0)
    return cut


# 39-bit keys.  A bucket of 512 k items holds (sqrt(512 k + 24.5) - sqrt(24.5))^2 on average at
# most: 1193.9 for k = 3, 1646.3 for 4; one bucket of everything up to 2105.7 with k = 5
@pytest.mark.parametrize("items,cut", [(2, (0, 3)), (1192, (0, 3)), (1196, (0, 4)), (1644, (0, 4)), (1648, (0, 5)),
                                       (2104, (0, 5)), (2108, (1, 3)), (1192 * 16, (4, 3)), (1196 * 16, (4, 4)),
                                       (1644 * 16, (4, 4)), (1648 * 16, (4, 5)), (2120 * 16, (5, 3))])
def test_one_word_keys(gpu, items, cut):
    assert _first_cut(gpu, 20, 20, items) == cut


# 19 bits: not mixed, so one bucket or none
@pytest.mark.parametrize("items,cut", [(2104, (0, 5)), (2108, (-1, 0))])
def test_short_keys(gpu, items, cut):
    assert _first_cut(gpu, 10, 10, items) == cut


# 55 bits: a packed word holds 48 key bits below the bucket bits
@pytest.mark.parametrize("items,cut", [(4000, (-1, 0)), (1100 * 128, (7, 3)), (1100 * 64, (-1, 0))])
def test_long_one_word_keys(gpu, items, cut):
    assert _first_cut(gpu, 28, 28, items) == cut


# 99 bits: four items per thread at most; 127 bits: the low word takes 116 key bits
@pytest.mark.parametrize("M,items,cut", [(50, 1192, (0, 3)), (50, 1196, (0, 4)), (50, 1644, (0, 4)), (50, 1648, (1, 3)),
                                         (50, 1196 * 4, (2, 4)), (64, 2000, (11, 3))])
def test_two_word_keys(gpu, M, items, cut):
    assert _first_cut(gpu, M, M, items) == cut


# exact steps: every hop is a record; one order of sums whatever the rule above says
@pytest.mark.parametrize("n,cut", [(50, (-1, 0)), (400, (3, 5))])
def test_exact_steps(gpu, n, cut):
    assert _first_cut(gpu, 20, 20, 2 * n, gpu.IsDeterministic()) == cut
