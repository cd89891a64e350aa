"""GPU parity of the Q6_K Q8 decode kernel (gemv_q6_k.hip): the same bits as the
oracle's Q8 restatement at the edges of its blocks (16 or 32 rows, one or two
tokens, passes of 16 or 8 super-blocks), on the longest row the mode takes and
in the decoder's fused forms."""
import numpy as np
import pytest

import oracle as O
import rce_amd
from llama_case import make_weights, tiny_cfg
from rce_amd import Mode
from test_gpu_gemv import bits, run_dev
from test_gpu_llama import TOKENS, run_pair
from test_gpu_moe_forms import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,t", [
    (1, 256, 1), (17, 512, 3), (64, 4096, 2),    # one row; ragged rows, an odd token; one whole pass of 16
    (33, 4352, 1), (79, 8448, 2),                # a second and a third pass of 16
    (16385, 256, 1), (609, 2304, 53),            # blocks of 32 rows: one super-block, passes of 8 and one more
    (20, 47616, 1), (20, 47616, 2),              # the longest row, past 64 KB of LDS
])
def test_bit_identical(ctx, monkeypatch, n, k, t):
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "0")
    print(f"q6_k q8 n={n} k={k} t={t}", flush=True)
    rng = np.random.default_rng(n + k)
    b = O.quantize((rng.standard_normal((n, k)) * 0.02).astype(np.float32), O.Q6_K)
    x = rng.standard_normal((t, k)).astype(np.float32)
    x[0, :32] = 0.0  # a block of zeros: scale 0
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, b, O.Q6_K, n, k)
    got = run_dev(ctx, w, x, Mode.Q8)
    want = O.mm_batched_q8(x, b, O.Q6_K, n, k)
    assert np.array_equal(bits(got), bits(want)), f"{np.sum(bits(got) != bits(want))} values differ"
    w.close()


@pytest.mark.parametrize("norm_kernel", [False, True])  # the forms with and without rms_norm inside
# gate/up and residual: whole blocks; a second pass of 16; a residual row past 64 KB of LDS
@pytest.mark.parametrize("d_ff", [512, 4352, 40448])
def test_fused_forms(ctx, monkeypatch, d_ff, norm_kernel):
    """A decoder whose linears are all Q6_K: q|k|v in one launch, the residual
    and gate/up forms and the head that ends the step, bit for bit against the
    device-order oracle."""
    print(f"q6_k fused forms d_ff={d_ff} norm_kernel={norm_kernel}", flush=True)
    if norm_kernel:
        monkeypatch.setenv("RCE_QMM_LLAMA_NORM_KERNEL", "1")
    W = make_weights(tiny_cfg(d_ff=d_ff), seed=41, lin_dtype=O.Q6_K, embd_dtype=O.Q6_K)
    run_pair(ctx, W, Mode.Q8, TOKENS[:4], 1e-3, separate_norms=norm_kernel).close()


def test_grouped_past_64_kb(ctx, monkeypatch):
    """Two slots per block of a 20480-long row: 65 KB of LDS."""
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "0")
    check(ctx, O.Q6_K, 2, 256, 20480, 3, 2, Mode.Q8)
