"""GPU tests of the large-tile prefill GEMM (gemm_wide.hip): each tile shape
its rule picks, for every weight format, at ragged row and column counts.

Quantized formats are compared with the small-tile kernel (gemm_f16.hip, the
route of calls of at most 64 rows here), which forms the same binary16 weights
and differs only in the order of the f32 sums: two orders of K <= 768 terms
differ by at most 2 K 2^-24 of the sum of the terms' magnitudes, about 1e-4 of
it in the worst case and 1e-6 of the largest output in practice; 1e-5
normwise catches any wrong weight, scale or fragment.  F16 weights are exact,
so they are compared with float64 products.
"""
import numpy as np
import pytest

import oracle as O
import rce_amd
from rand_blocks import rand_blocks
from rce_amd import GgufDtype as G, Mode
from test_gpu_gemm import normwise, run_gemm

pytestmark = pytest.mark.gpu
F16, F32 = np.float16, np.float32
QUANT = [O.Q4_K, O.Q5_K, O.Q4_0, O.Q4_1, O.Q5_0, O.Q8_0, O.Q6_K]
# (tokens, rows): one case per tile shape on a 256-CU chip
SHAPES = {"128x128": (1000, 4000), "256x128": (2000, 4040), "128x256": (600, 11000), "256x256": (1000, 11000),
          "256x256 then 128x256": (3000, 11000)}


def weight_bytes(rng, dt, n, k):
    if dt in (O.Q4_1, O.Q5_0):
        return rand_blocks(rng, dt, n, k)
    return rce_amd.quantize((rng.standard_normal((n, k)) * 0.02).astype(F32), dt)


# K: one super-block (two weight stages, none loaded into a slot twice), and
# an odd number of them (every slot of the rings refilled)
@pytest.mark.parametrize("k", [256, 768])
@pytest.mark.parametrize("dt", QUANT)
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_wide_tiles_match_the_small_tile_kernel(ctx, dt, shape, k):
    m, n = SHAPES[shape]
    print(f"wide tile {shape} dtype={dt} M={m} N={n} K={k}", flush=True)
    rng = np.random.default_rng(dt)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, weight_bytes(rng, dt, n, k), dt, n, k)
    x = rng.standard_normal((m, k)).astype(F16)
    got = run_gemm(ctx, w, x, G.F16)
    for r0 in (0, 100, 200, 448, m - 41):  # every 128- and 256-row piece of a tile, and the ragged end
        part = np.ascontiguousarray(x[r0:r0 + 64])
        want = run_gemm(ctx, w, part, G.F16)
        assert normwise(got[r0:r0 + len(part)], want) < 1e-5, f"rows {r0}.."
    again = run_gemm(ctx, w, x, G.F16)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    w.close()


@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (3, 65, 64), (129, 257, 192), (333, 700, 448), (200, 300, 2560),
                                   (1030, 4100, 320), (2050, 5000, 64)])
def test_f16_weights(ctx, m, n, k):
    """F16 weights at every tile shape the rule gives them, odd chunk counts
    included, against float64 products (the f32 sums of K terms in two chains:
    1e-5 normwise)."""
    print(f"wide f16 M={m} N={n} K={k}", flush=True)
    rng = np.random.default_rng(m + n)
    wf = (rng.standard_normal((n, k)) * 0.05).astype(F16)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, wf.view(np.uint8).reshape(-1), O.F16, n, k)
    x = rng.standard_normal((m, k)).astype(F16)
    got = run_gemm(ctx, w, x, G.F16)
    rows = np.unique(np.r_[0:min(m, 70), max(0, m - 70):m])
    want = x[rows].astype(np.float64) @ wf.astype(np.float64).T
    assert normwise(got[rows], want) < 1e-5
    w.close()


def test_f32_activations_are_rounded_to_binary16_first(ctx):
    n, k, m = 4000, 256, 1000
    rng = np.random.default_rng(5)
    w = rce_amd.QuantWeight.from_owned_bytes(ctx, weight_bytes(rng, O.Q4_K, n, k), O.Q4_K, n, k)
    x = rng.standard_normal((m, k)).astype(F32)
    a, b = run_gemm(ctx, w, x, G.F32), run_gemm(ctx, w, x.astype(F16), G.F16)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    w.close()


def test_supports_is_unchanged():
    for dt in QUANT + [O.F16]:
        assert rce_amd.supports(dt, 256, Mode.F16_MFMA)
        assert not rce_amd.supports(dt, 96, Mode.F16_MFMA)
