"""The host-pointer entry points around the size of the pinned staging (256
KiB each way): the same bits as the device entry point on both sides of it,
for activation sizes that are no multiple of 16 bytes, for results that
change from call to call on reused staging, and from two threads with a
context each."""
import threading

import numpy as np
import pytest

import oracle as O
import rce_amd
from rand_blocks import float_bytes
from rce_amd import Mode
from test_gpu_gemv import bits, run_dev

pytestmark = pytest.mark.gpu


def weight(ctx, rng, dt, n, k):
    b = float_bytes(rng, dt, n, k) if dt == O.F32 else O.quantize((rng.standard_normal((n, k)) * 0.02).astype(np.float32), dt)
    return rce_amd.QuantWeight.from_owned_bytes(ctx, b, dt, n, k)


@pytest.mark.parametrize("dt,n,k,t", [
    (O.F32, 3, 5, 1), (O.F32, 7, 5, 3),            # 20 and 60 bytes of activations
    (O.Q8_0, 65536, 32, 1), (O.Q8_0, 65537, 32, 1),  # the output at the limit, one value past it
    (O.Q8_0, 64, 4096, 16), (O.Q8_0, 64, 4096, 17),  # the activations at the limit, one row past it
])
def test_same_bits_on_both_sides_of_the_staging(ctx, dt, n, k, t):
    print(f"host call dtype={dt} n={n} k={k} t={t}", flush=True)
    rng = np.random.default_rng(n + t)
    w = weight(ctx, rng, dt, n, k)
    for _ in range(3):
        x = rng.standard_normal((t, k)).astype(np.float32)
        got = rce_amd.mm_1d(x[0], w) if t == 1 else rce_amd.mm_batched(x, t, w)
        want = run_dev(ctx, w, x, Mode.EXACT)
        assert np.array_equal(bits(got).reshape(-1), bits(want).reshape(-1))
    w.close()


def test_two_threads_with_a_context_each():
    bad = []

    def work(seed):
        with rce_amd.Context(0) as c:
            rng = np.random.default_rng(seed)
            w = weight(c, rng, O.Q8_0, 200, 256)
            for _ in range(50):
                x = rng.standard_normal(256).astype(np.float32)
                if not np.array_equal(bits(rce_amd.mm_1d(x, w)), bits(run_dev(c, w, x.reshape(1, -1), Mode.EXACT)).reshape(-1)):
                    bad.append(seed)
            w.close()

    ts = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
