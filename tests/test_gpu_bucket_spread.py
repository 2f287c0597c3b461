"""Steps whose buckets vary more in size than the rule expects: after one that overfilled the
largest shape, smaller buckets hold the same records; and where the largest shape's mean lies."""
import numpy as np
import pytest

from test_gpu_bucket_rule import _first_cut
from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


def test_more_buckets_after_an_overflow(gpu):
    """Every address of 30 bosons on three modes (496) with 128 attempts each: 63,984 items, 2000 in
    each of 32 buckets on average, but as 15.5 addresses of 129, and 20 of those overfill a bucket.
    64 buckets would have to hold 20 where 7.75 come on average."""
    import oracle as O

    M, N = 3, 30
    keys = O.build_basis(M, N)
    assert len(keys) == 496
    vals = np.full(len(keys), 128.5)
    style = gpu.IsDynamicSemistochastic(rel_spawning_threshold=1e-9)
    h = device_model(gpu, "real", M, N, 0.0, 1.0)
    runs = []
    for mode in (2, 1):
        e = gpu._native.Engine(h.descriptor(), style.descriptor(), 5, 1 << 12, 1 << 17)
        e.set_radix_mode(mode)
        e.set_timing(True)
        cuts, states = [], []
        for s in range(1, 41):
            e.upload(keys, vals)
            st = e.step(s, 0.0, 1e-3)
            cuts.append(e.last_cut())
            states.append((st.spawn_attempts, st.len, *e.download()))
        runs.append((cuts, states, e.kernel_times().get("bucket_fallback", (0, 0))[1]))
        e.close()
    cuts, states, overflows = runs[0]
    print(cuts, overflows, states[0][:2], flush=True)
    assert states[0][0] == 128 * 496
    for x, y in zip(states, runs[1][1]):
        assert x[:2] == y[:2]
        assert np.array_equal(x[2], y[2]) and np.array_equal(x[3].view(np.uint64), y[3].view(np.uint64))
    assert cuts[:17] == [(-1, 0)] * 17          # the overflow, and 16 steps along the merge path
    assert cuts[17:] == [(6, 5)] * 23           # a mean of 999 instead of 1999; the smallest shape was overfilled once
    assert overflows == 1


# 39 bits: buckets of 2105 on average are the largest, 4.57 deviations of their count below the 2560
# items they hold; 99 bits: 1645 of 2048
@pytest.mark.parametrize("M,items,cut", [(20, 2101 * 16, (4, 5)), (20, 2109 * 16, (5, 3)),
                                         (50, 1642 * 4, (2, 4)), (50, 1649 * 4, (3, 3))])
def test_largest_mean(gpu, M, items, cut):
    assert _first_cut(gpu, M, M, items) == cut
