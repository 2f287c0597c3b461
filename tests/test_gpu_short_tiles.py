"""Steps around the sizes where the plan and the spawn change their tiles (131,072 entries; 262,144
attempts, of which a step sized by the one before it counts a quarter and 16,384 more), and around
one short tile of 256 attempts, bit for bit against the oracle."""
import numpy as np
import pytest

import oracle as O
from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model, oracle_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entries,attempts", [
    (1, 1), (3, 255), (3, 256), (3, 257), (257, 513), (1000, 196_600), (1000, 196_700), (1000, 262_143),
    (1000, 262_144), (1000, 262_145), (131_070, 131_070), (131_071, 196_000), (131_072, 262_000),
    (131_073, 262_500)])
@pytest.mark.parametrize("style", ["integer", "dynamic"])
def test_step_against_oracle(gpu, entries, attempts, style):
    M = N = 16
    rng = np.random.default_rng(entries + attempts)
    keys, _ = _chain_vector(M, N, entries, rng)
    vals = np.full(entries, attempts // entries, dtype=np.int64)
    vals[0] += attempts - int(vals.sum())
    vals *= rng.choice([-1, 1], entries)
    st = {"integer": gpu.IsStochasticInteger, "dynamic": gpu.IsDynamicSemistochastic}[style]()
    if style == "dynamic":
        vals = vals * rng.uniform(1.0, 1.0 + 1e-3 / (1 + attempts // entries), entries)
    h = device_model(gpu, "real", M, N, 6.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), st.descriptor(), 11, 1 << 20, 1 << 20)
    e.upload(keys, vals)
    om = oracle_model("real", M, N, 6.0, 1.0)
    k, v = keys, vals
    for step in (1, 2, 3):                          # the first step reads its counts back
        print(f"entries={entries} attempts={attempts} {style} step={step}", flush=True)
        got = e.step(step, -1.0, 1e-3)
        k, v, ost = O.step(om, O.style(style), k, v, seed=11, step=step, shift=-1.0, dtau=1e-3, order=1)
        gk, gv = e.download()
        assert np.array_equal(gk, k) and np.array_equal(gv, v)
        assert (got.spawn_attempts, got.len) == (ost["attempts"], len(k))
    e.close()
