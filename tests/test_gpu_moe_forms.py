"""GPU parity of the grouped experts' EXACT and Q8 forms without a host
round trip: tiles of one and two slots on the decode kernels, tiles of 16 on
the int8 matrix cores, over every format, one and two slots per expert,
experts without slots, and the most experts whose table travels in the kernel
arguments (64) and one more.  Bit for bit with the oracle's device-order
restatement."""
import numpy as np
import pytest

import oracle as O
import rce_amd
from rand_blocks import rand_blocks
from rce_amd import Mode
from test_gpu_moe import bit_equal, run_moe

pytestmark = pytest.mark.gpu


def experts(rng, dt, count, n, k):
    if dt in (O.Q4_1, O.Q5_0, O.Q3_K):
        return [rand_blocks(rng, dt, n, k) for _ in range(count)]
    return [O.quantize((rng.standard_normal((n, k)) * 0.02).astype(np.float32), dt) for _ in range(count)]


def check(ctx, dt, E, dm, dff, t, k, mode):
    print(f"moe forms dtype={dt} E={E} d={dm} ff={dff} t={t} k={k} mode={mode}", flush=True)
    rng = np.random.default_rng(dt * 100 + E + t)
    w1, w2 = experts(rng, dt, E, dff, dm), experts(rng, dt, E, dm, dff)
    x = rng.standard_normal((t, dm)).astype(np.float32)
    ids, gw = rce_amd.moe_router(rng.standard_normal((t, E)).astype(np.float32), k)
    got = run_moe(ctx, w1, w2, dt, dm, dff, x, ids, gw, mode)
    want = O.moe_ffn(x, w1, w2, dt, dff, ids, gw, q8=mode == Mode.Q8, silu_dev=True)
    assert bit_equal(got, want)


@pytest.mark.parametrize("mode", [Mode.EXACT, Mode.Q8])
@pytest.mark.parametrize("dt", [O.Q4_0, O.Q8_0, O.Q5_0, O.Q4_1, O.Q3_K, O.Q4_K, O.Q5_K, O.Q6_K])
@pytest.mark.parametrize("E,t,k", [(4, 1, 1), (4, 5, 2), (2, 9, 2)])  # tiles of one, of two (ragged), several per expert
def test_formats(ctx, dt, E, t, k, mode):
    check(ctx, dt, E, 512, 768, t, k, mode)


@pytest.mark.parametrize("dt", [O.Q4_0, O.Q4_K, O.Q6_K])
def test_q8_on_the_matrix_cores(ctx, monkeypatch, dt):
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", "2")
    check(ctx, dt, 3, 512, 768, 37, 2, Mode.Q8)  # about 25 slots per expert: a full tile and a ragged one
    check(ctx, dt, 2, 2304, 2560, 20, 1, Mode.Q8)  # rows past 2048: a slot of every ring loaded again


@pytest.mark.parametrize("mode", [Mode.EXACT, Mode.Q8])
@pytest.mark.parametrize("E", [64, 65])
def test_expert_table_limits(ctx, E, mode):
    check(ctx, O.Q4_0, E, 256, 256, 40, 3, mode)


@pytest.mark.parametrize("E", [2, 64])
def test_mfma_expert_tables(ctx, E):
    """F16_MFMA: the same experts in another order, and with one more that no
    token takes (64: a table uploaded instead of written by the grouping
    launch), give the same bits, within the mode's 3e-3 of the EXACT result."""
    print(f"moe mfma tables E={E}", flush=True)
    rng = np.random.default_rng(E)
    dm, dff, t = 256, 512, 50
    w1, w2 = experts(rng, O.Q4_0, E + 1, dff, dm), experts(rng, O.Q4_0, E + 1, dm, dff)
    x = rng.standard_normal((t, dm)).astype(np.float32)
    ids, gw = rce_amd.moe_router(rng.standard_normal((t, E)).astype(np.float32), 2)
    got = [run_moe(ctx, w1[:E], w2[:E], O.Q4_0, dm, dff, x, ids, gw, Mode.F16_MFMA),
           run_moe(ctx, w1[:E][::-1], w2[:E][::-1], O.Q4_0, dm, dff, x, E - 1 - ids, gw, Mode.F16_MFMA),
           run_moe(ctx, w1, w2, O.Q4_0, dm, dff, x, ids, gw, Mode.F16_MFMA)]
    assert bit_equal(got[0], got[1]) and bit_equal(got[0], got[2])
    want = O.moe_ffn(x, w1, w2, O.Q4_0, dff, ids, gw)
    # binary16 activations, weights and h, 2^-11 each, f32 sums: the mode's budget for grouped experts
    assert np.linalg.norm(got[0].astype(np.float64) - want) < 3e-3 * np.linalg.norm(want)


@pytest.mark.parametrize("mode", [Mode.EXACT, Mode.Q8])
def test_experts_change_between_calls(ctx, mode):
    """Two expert sets alternately on one context (a model's layers)."""
    for seed in (1, 2, 1):
        rng = np.random.default_rng(seed)
        w1, w2 = experts(rng, O.Q4_K, 4, 512, 256), experts(rng, O.Q4_K, 4, 256, 512)
        x = rng.standard_normal((3, 256)).astype(np.float32)
        ids, gw = rce_amd.moe_router(rng.standard_normal((3, 4)).astype(np.float32), 2)
        got = run_moe(ctx, w1, w2, O.Q4_K, 256, 512, x, ids, gw, mode)
        assert bit_equal(got, O.moe_ffn(x, w1, w2, O.Q4_K, 512, ids, gw, q8=mode == Mode.Q8, silu_dev=True))


@pytest.mark.parametrize("mode", [Mode.EXACT, Mode.Q8])
def test_bad_id_is_an_error_and_the_next_call_is_clean(ctx, mode):
    rng = np.random.default_rng(3)
    w1, w2 = experts(rng, O.Q4_0, 4, 512, 256), experts(rng, O.Q4_0, 4, 256, 512)
    x = rng.standard_normal((4, 256)).astype(np.float32)
    ids, gw = rce_amd.moe_router(rng.standard_normal((4, 4)).astype(np.float32), 2)
    bad = ids.copy()
    bad[2, 1] = -1
    with pytest.raises(rce_amd.QmmError, match="out of range"):
        run_moe(ctx, w1, w2, O.Q4_0, 256, 512, x, bad, gw, mode)
    got = run_moe(ctx, w1, w2, O.Q4_0, 256, 512, x, ids, gw, mode)
    assert bit_equal(got, O.moe_ffn(x, w1, w2, O.Q4_0, 512, ids, gw, q8=mode == Mode.Q8, silu_dev=True))


@pytest.mark.parametrize("mma", ["0", "2"])
def test_many_experts_expert_by_expert_q8(ctx, monkeypatch, mma):
    """One expert past the kernel arguments' table, forty tokens on one of
    them: its products on the matrix cores and on the decode kernels."""
    monkeypatch.setenv("RCE_QMM_Q8_MFMA", mma)
    print(f"moe expert by expert mma={mma}", flush=True)
    rng = np.random.default_rng(6)
    E, dm, dff, t = 65, 256, 512, 40
    w1, w2 = experts(rng, O.Q4_0, E, dff, dm), experts(rng, O.Q4_0, E, dm, dff)
    x = rng.standard_normal((t, dm)).astype(np.float32)
    ids = np.stack([np.full(t, 64), np.arange(t) % 64], 1).astype(np.int32)
    gw = np.full((t, 2), 0.5, np.float32)
    got = run_moe(ctx, w1, w2, O.Q4_0, dm, dff, x, ids, gw, Mode.Q8)
    assert bit_equal(got, O.moe_ffn(x, w1, w2, O.Q4_0, dff, ids, gw, q8=True, silu_dev=True))


@pytest.mark.parametrize("dm,dff,t", [(512, 2048, 1300), (512, 2048, 1340), (256, 8448, 1340), (256, 8448, 1380)])
def test_exact_forms_on_both_sides_of_the_rule(ctx, dm, dff, t):
    """One Q8_0 expert: short rows, in tiles of two slots at any size, and rows
    of 264 blocks, 2898 and 2985 million multiply-adds, in tiles and as a
    product of its own."""
    print(f"moe exact rule d={dm} ff={dff} t={t}", flush=True)
    rng = np.random.default_rng(t)
    w1, w2 = experts(rng, O.Q8_0, 1, dff, dm), experts(rng, O.Q8_0, 1, dm, dff)
    x = rng.standard_normal((t, dm)).astype(np.float32)
    ids, gw = np.zeros((t, 1), np.int32), np.ones((t, 1), np.float32)
    got = run_moe(ctx, w1, w2, O.Q8_0, dm, dff, x, ids, gw, Mode.EXACT)
    assert bit_equal(got, O.moe_ffn(x, w1, w2, O.Q8_0, dff, ids, gw, silu_dev=True))


@pytest.mark.parametrize("dt", [O.Q4_0, O.Q8_0, O.Q5_0, O.Q4_1, O.Q3_K, O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("t", [34, 41])
def test_exact_sixteen_rows_per_lane(ctx, dt, t):
    """Both matrices at 16 rows per lane (at least 768 blocks; at 34 tokens
    the K-quants' first at 8), the last block of W2's rows part filled."""
    check(ctx, dt, 4, 4096, 1280, t, 2, Mode.EXACT)


@pytest.mark.parametrize("mode", [Mode.EXACT, Mode.Q8])
@pytest.mark.parametrize("E,dm", [(4, 256), (65, 256)])  # the grouped forms; expert by expert
def test_bad_id_leaves_the_output(ctx, mode, E, dm):
    print(f"bad id E={E} mode={mode}", flush=True)
    rng = np.random.default_rng(4)
    W1 = [rce_amd.QuantWeight.from_owned_bytes(ctx, b, O.Q4_0, 512, dm) for b in experts(rng, O.Q4_0, E, 512, dm)]
    W2 = [rce_amd.QuantWeight.from_owned_bytes(ctx, b, O.Q4_0, dm, 512) for b in experts(rng, O.Q4_0, E, dm, 512)]
    ids = np.array([[0, 1], [2, E]], np.int32)
    keep = rng.standard_normal(2 * dm).astype(np.float32)
    bufs = [rce_amd.DeviceBuffer.from_numpy(ctx, a) for a in (rng.standard_normal((2, dm)).astype(np.float32), ids,
                                                             np.full((2, 2), 0.5, np.float32), keep)]
    with pytest.raises(rce_amd.QmmError, match="out of range"):
        rce_amd.moe_ffn_dev(ctx, W1, W2, bufs[0].ptr, 2, bufs[1].ptr, bufs[2].ptr, 2, bufs[3].ptr, mode)
    ctx.synchronize()
    assert np.array_equal(bufs[3].download(np.float32, 2 * dm), keep)
    for x in bufs:
        x.free()
    for w in W1 + W2:
        w.close()
