"""GPU parity of the int8 matrix-core form of the Q8 mode (gemv_q8_mfma.hip),
forced on every case: the same bits as the oracle's Q8 restatement, at the
edges of its tiles (16 tokens, 64 rows, stages of 256 with a ring of three)."""
import numpy as np
import pytest

import oracle as O
import rce_amd
from rand_blocks import rand_blocks
from rce_amd import Mode
from test_gpu_gemv import bits, run_dev

pytestmark = pytest.mark.gpu
FORMATS = [O.Q4_0, O.Q8_0, O.Q5_0, O.Q4_1, O.Q4_K, O.Q5_K, O.Q6_K]
# (rows, columns, tokens): one row and one stage; ragged rows (scalar and
# vector stores) and tokens around one and two tiles; stage counts 1, 2, 3
# and 7; a row slice per XCD and one more
SHAPES = [(1, 256, 2), (63, 256, 15), (66, 512, 16), (130, 768, 17), (576, 1792, 33)]


@pytest.mark.parametrize("dt", FORMATS)
@pytest.mark.parametrize("n,k,t", SHAPES)
def test_bit_identical(ctx, monkeypatch, dt, n, k, t):
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "2")
    print(f"q8 mfma dtype={dt} n={n} k={k} t={t}", flush=True)
    rng = np.random.default_rng(dt * 1000 + n)
    if dt in (O.Q4_1, O.Q5_0):
        b = rand_blocks(rng, dt, n, k)
    else:
        b = O.quantize((rng.standard_normal((n, k)) * 0.02).astype(np.float32), dt)
    x = rng.standard_normal((t, k)).astype(np.float32)
    x[0, :32] = 0.0  # a block of zeros: scale 0
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, b, dt, n, k)
    got = run_dev(ctx, w, x, Mode.Q8)
    want = O.mm_batched_q8(x, b, dt, n, k)
    assert np.array_equal(bits(got), bits(want)), f"{np.sum(bits(got) != bits(want))} values differ"
    w.close()
