"""mm_batched_dev recorded into a HIP graph: forms that keep no growing
scratch stay valid on replay after larger calls on the same context, and equal
the eager call's bits on every replay."""
import numpy as np
import pytest

import oracle as O
import rce_amd
from bench import Hip
from rce_amd import GgufDtype as G
from rce_amd import Mode
from test_gpu_gemm_wide import weight_bytes

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


def weight(c, rng, dt, n, k):
    return rce_amd.QuantWeight.from_owned_bytes(c, weight_bytes(rng, dt, n, k), dt, n, k)


def replay_equals_eager(c, record, between, xa, act, t, w, mode):
    """Record the call (nothing eager before it unless record is "warm"),
    then check replays with `between` run before each."""
    n = w.n_rows
    hip = Hip()
    nan = np.full(t * n, np.nan, F32)
    out, eager = rce_amd.DeviceBuffer.from_numpy(c, nan), rce_amd.DeviceBuffer.from_numpy(c, nan)
    if record == "warm":
        rce_amd.mm_batched_dev(c, xa.ptr, act, t, w, eager.ptr, mode)
    c.synchronize()
    g, ex = hip.capture(c.stream, lambda: rce_amd.mm_batched_dev(c, xa.ptr, act, t, w, out.ptr, mode))
    rce_amd.mm_batched_dev(c, xa.ptr, act, t, w, eager.ptr, mode)
    c.synchronize()
    want = eager.download(F32, t * n)
    assert np.all(np.isfinite(want))
    for _ in range(3):
        between()
        out.upload(nan)
        hip.launch(ex, c.stream)
        c.synchronize()
        assert np.array_equal(out.download(F32, t * n).view(np.uint32), want.view(np.uint32))
    hip.destroy(g, ex)
    out.free(); eager.free()


@pytest.mark.parametrize("record", ["cold", "warm"])
def test_k_slices(record):
    """16 tokens in six slices (0.8 MB of sums) recorded; 77 in four (2.5 MB)
    and new allocations between the replays."""
    print(f"capture k slices {record}", flush=True)
    rng = np.random.default_rng(1)
    with rce_amd.Context(0) as c:
        w = weight(c, rng, O.Q6_K, 2048, 5632)
        xa = rce_amd.DeviceBuffer.from_numpy(c, rng.standard_normal((77, 5632)).astype(F16))
        big = rce_amd.DeviceBuffer(c, 77 * 2048 * 4)

        def between():
            rce_amd.mm_batched_dev(c, xa.ptr, G.F16, 77, w, big.ptr, Mode.F16_MFMA)
            c.synchronize()
            for nbytes in (786432, 1 << 20):
                rce_amd.DeviceBuffer.from_numpy(c, np.full(nbytes, 255, np.uint8)).free()

        replay_equals_eager(c, record, between, xa, G.F16, 16, w, Mode.F16_MFMA)
        xa.free(); big.free(); w.close()


@pytest.mark.parametrize("record", ["cold", "warm"])
@pytest.mark.parametrize("dt", [O.Q5_0, O.Q4_1, O.Q6_K])
def test_q8_formats_without_scratch(monkeypatch, dt, record):
    """32 tokens recorded for formats whose decode kernels quantize inside
    their blocks, 200 (a larger workspace of the matrix-core form) and new
    allocations between the replays."""
    print(f"capture q8 dtype={dt} {record}", flush=True)
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "2")
    rng = np.random.default_rng(2)
    with rce_amd.Context(0) as c:
        w = weight(c, rng, dt, 512, 2048)
        xa = rce_amd.DeviceBuffer.from_numpy(c, rng.standard_normal((200, 2048)).astype(F32))
        big = rce_amd.DeviceBuffer(c, 200 * 512 * 4)

        def between():
            rce_amd.mm_batched_dev(c, xa.ptr, G.F32, 200, w, big.ptr, Mode.Q8)
            c.synchronize()
            for nbytes in (81920, 1 << 17):
                rce_amd.DeviceBuffer.from_numpy(c, np.full(nbytes, 255, np.uint8)).free()

        replay_equals_eager(c, record, between, xa, G.F32, 32, w, Mode.Q8)
        xa.free(); big.free(); w.close()
