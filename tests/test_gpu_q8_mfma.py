"""GPU parity of the int8 matrix-core form of the Q8 mode (gemv_q8_mfma.hip),
forced on every case: the same bits as the oracle's Q8 restatement, at the
edges of its blocks (16 rows, tiles of 16 tokens; four waves taking chunks of
256 of K, 128 for blocks of 32, in turn, each through a ring of two or three)."""
import ctypes

import numpy as np
import pytest

import oracle as O
import rce_amd
from rand_blocks import rand_blocks
from rce_amd import Mode
from rce_amd._lib import check, lib
from test_gpu_gemm_wide import weight_bytes
from test_gpu_gemv import bits, run_dev

pytestmark = pytest.mark.gpu
FORMATS = [O.Q4_0, O.Q8_0, O.Q5_0, O.Q4_1, O.Q4_K, O.Q5_K, O.Q6_K]
# (rows, columns, tokens): one row, fewer chunks than waves; ragged rows and
# tokens around one and two tiles; a last round of one, two and three waves; a row slice
# per XCD and more; 9, 17 and 22 chunks of 256, where every slot of a ring is
# loaded again (from the 9th chunk on in a ring of two), up to twice
SHAPES = [(1, 256, 2), (63, 256, 15), (66, 512, 16), (130, 768, 17), (576, 1792, 33), (50, 2304, 18), (35, 4352, 33),
          (20, 5632, 17)]


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


def test_outputs_past_the_grid_limit(ctx, monkeypatch):
    """2^32 and more outputs: 65536 rows times 65552 tokens are 2^24 + 4096
    blocks of 256 threads, more threads than a grid dimension takes.  The first and last
    tokens have the bits of a call of their own."""
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "2")
    n, k, t = 65536, 256, 65552
    print(f"q8 mfma n={n} k={k} t={t}", flush=True)
    rng = np.random.default_rng(9)
    b = rand_blocks(rng, O.Q8_0, n, k)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, b, O.Q8_0, n, k)
    x = rng.standard_normal((t, k)).astype(np.float32)
    xa = rce_amd.DeviceBuffer.from_numpy(ctx, x)
    out = rce_amd.DeviceBuffer(ctx, 4 * n * t)
    rce_amd.mm_batched_dev(ctx, xa.ptr, rce_amd.GgufDtype.F32, t, w, out.ptr, Mode.Q8)
    ctx.synchronize()
    for t0 in (0, t - 32, t - 4):  # the first tokens, both sides of the second launch's first tile
        got = np.empty((4, n), np.float32)
        check(lib().rce_qmm_memcpy_d2h(ctx.handle, ctypes.c_void_p(got.ctypes.data), ctypes.c_void_p(out.ptr + 4 * n * t0), got.nbytes))
        assert np.array_equal(bits(got), bits(run_dev(ctx, w, x[t0:t0 + 4], Mode.Q8))), t0
    xa.free(); out.free(); w.close()


@pytest.mark.parametrize("dt", FORMATS)
@pytest.mark.parametrize("n,k,t", [(40, 512, 2), (40, 512, 48), (72, 4096, 13), (1030, 2048, 24), (24, 16640, 5)])
def test_the_rule_changes_no_bits(ctx, monkeypatch, dt, n, k, t):
    """The form the rule takes on both sides of its lines (short and long
    rows, rows of more than 256 units, few and many tokens), and either form forced."""
    print(f"q8 rule dtype={dt} n={n} k={k} t={t}", flush=True)
    rng = np.random.default_rng(dt * 1000 + n + t)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, weight_bytes(rng, dt, n, k), dt, n, k)
    x = rng.standard_normal((t, k)).astype(np.float32)
    got = []
    for form in (None, "0", "2"):
        if form is None:
            monkeypatch.delenv("RCE_QMM_Q8_MFMA", raising=False)
        else:
            monkeypatch.setenv("RCE_QMM_Q8_MFMA", form)
        got.append(bits(run_dev(ctx, w, x, Mode.Q8)))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    w.close()
