"""GPU checks of the prefill GEMM's K slices (gemm_f16.hip, short M): against
float64 products of the binary16 weights the kernel forms (f32 sums of at
most 8192 terms: 1e-5 normwise), run to run, and through the no-allocation
entry point next to a scratch that the activations nearly fill."""
import numpy as np
import pytest

import oracle as O
import rce_amd
from rce_amd import GgufDtype as G
from rce_amd import Mode
from test_gpu_gemm import normwise, run_gemm
from test_gpu_gemm_wide import weight_bytes
from test_gpu_moe import f16_weights

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32


# (M, N, K): one row tile and eight slices of unequal length (22 groups); rows
# and columns past a tile, sums not a multiple of four; two slices of 64- and
# 128-row tiles; the most slices (16 of two groups)
@pytest.mark.parametrize("dt", [O.Q4_K, O.Q4_0, O.Q5_K, O.Q4_1, O.Q5_0, O.Q8_0, O.Q6_K])
@pytest.mark.parametrize("m,n,k", [(16, 2048, 5632), (77, 1027, 4352), (1, 4096, 8192), (129, 2047, 6144), (9, 70, 8192)])
def test_slices(ctx, dt, m, n, k):
    print(f"gemm slices dtype={dt} M={m} N={n} K={k}", flush=True)
    rng = np.random.default_rng(m + n + dt)
    b = weight_bytes(rng, dt, n, k)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, b, dt, n, k)
    x = rng.standard_normal((m, k)).astype(F16)
    got, again = run_gemm(ctx, w, x, G.F16), run_gemm(ctx, w, x, G.F16)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32)), "not run-to-run deterministic"
    err = normwise(got, x.astype(np.float64) @ f16_weights(b, dt, n, k).T)
    assert err < 1e-5, err
    w.close()


def test_beside_a_full_scratch(ctx):
    m, n, k = 256, 1100, 24576  # 12.6 MB of binary16 activations and 4.5 MB of sums against 16 MiB
    rng = np.random.default_rng(3)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, weight_bytes(rng, O.Q4_0, n, k), O.Q4_0, n, k)
    xa = rce_amd.DeviceBuffer.from_numpy(ctx, rng.standard_normal((m, k)).astype(F32))
    out = rce_amd.DeviceBuffer(ctx, m * n * 4)
    got = []
    for call in (rce_amd.mm_batched_dev, rce_amd.mm_batched_dev_noalloc):
        call(ctx, xa.ptr, G.F32, m, w, out.ptr, Mode.F16_MFMA)
        ctx.synchronize()
        got.append(out.download(F32, m * n))
    assert np.all(np.isfinite(got[0]))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    xa.free(); out.free(); w.close()
