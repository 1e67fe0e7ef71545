"""Host-slice calls whose input and output are staged in pinned memory and whose end the host sees by a word that the
last kernel writes: the memory's kind, results that change from call to call, buffers that grow, and the sizes on both
sides of the staging limit (1 MB).  Results against the oracle's fused matvec on the oracle's Q8_0 bytes."""
import ctypes as C
import sys

import numpy as np
import pytest

import oracle as O
from oxillama_amd import capi, synth
from oxillama_amd import linear as L

pytestmark = pytest.mark.gpu
FP32_REL_TOL = 1e-5
HOST_PORTABLE, HOST_MAPPED, HOST_COHERENT = 0x1, 0x2, 0x40000000  # hip_runtime_api.h


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture
def cached(hip):
    lib = capi.load()
    lib.oxq_weight_cache_enable(1)
    yield lib
    lib.oxq_weight_cache_enable(0)
    lib.oxq_weight_cache_clear()


def make(hip, t, n, k, seed):
    w = synth.weights(t, seed, n, k)
    return w, L.QuantLinear(hip.QuantTensor(w, [n, k], t)), hip.KernelDispatcher().get_kernel(t)


def check(ref, t, w, x, y, n, k):
    want = ref.matvec_q8_fused_mt(t, w, ref.quantize_q8_0(x), n, k, 16)
    assert np.abs(y - want).max() <= FP32_REL_TOL * np.abs(want).max()
    return want


def test_staging_memory_is_coherent(hip, ref, cached):
    w, lin, kern = make(hip, O.Q8_0, 64, 256, 3)
    lin.forward(kern, synth.normal_f32(4, 256), np.zeros(64, np.float32))
    flags = (C.c_uint * 3)()
    assert cached.oxq_host_staging_flags(flags, 3) == capi.OK
    for f in flags:
        assert f & HOST_COHERENT and f & HOST_PORTABLE and f & HOST_MAPPED, [hex(f) for f in flags]


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_K], ids=lambda t: O.NAMES[t])
def test_small_cached_weights_with_changing_inputs(hip, ref, cached, t):
    """Two matrices in turn, a new input on every call: an input or output line left over from the call before, or a
    call that returns before its kernels are done, gives another vector's result."""
    say("changing inputs", O.NAMES[t])
    n, k = 96, 512
    mats = [make(hip, t, n, k, 10 + i) for i in range(2)]
    first = {}
    for call in range(200):
        w, lin, kern = mats[call % 2]
        seed = call % 50
        x, y = synth.normal_f32(100 + seed, k), np.full(n, 7.0, np.float32)
        lin.forward(kern, x, y)
        key = (call % 2, seed)
        if key not in first:
            check(ref, t, w, x, y, n, k)
            first[key] = y
        assert np.array_equal(y, first[key]), call


def test_larger_calls_after_smaller_ones(hip, ref, cached):
    """The staging buffers grow with the calls, and a smaller call after them uses their front."""
    for i, (n, k) in enumerate(((32, 256), (4096, 256), (64, 8192), (20000, 512), (32, 256), (33, 32))):
        say("growth", n, k)
        w, lin, kern = make(hip, O.Q8_0, n, k, 20 + i)
        x, y = synth.normal_f32(30 + i, k), np.full(n + 5, 7.0, np.float32)
        lin.forward(kern, x, y)
        check(ref, O.Q8_0, w, x, y[:n], n, k)
        assert np.all(y[n:] == 7.0)


LIMIT = (1 << 20) // 4  # floats


@pytest.mark.parametrize("n,k,m", [(32, 4096, LIMIT // 4096), (32, 4096, LIMIT // 4096 + 1), (4096, 256, LIMIT // 4096),
                                   (4096, 256, LIMIT // 4096 + 1), (33, 40, 7)])
def test_batches_on_both_sides_of_the_staging_limit(hip, ref, cached, n, k, m):
    """forward_batch: input and output of exactly 1 MB, of one row more, and rows that end inside a block."""
    say("limit, batch", n, k, m)
    t = O.Q8_0
    w, lin, kern = make(hip, t, n, k if k % 32 == 0 else (k + 31) // 32 * 32, 40 + m)
    if k % 32:
        lin = L.QuantLinear(hip.QuantTensor(w, [n, k], t))
    bias = synth.normal_f32(41, n)
    lin_b = L.QuantLinear(lin.weight, bias)
    k_pad = (k + 31) // 32 * 32
    for seed in (50, 51):
        x = synth.normal_f32(seed, m * k).reshape(m, k)
        y, yb = np.full((m, n), 7.0, np.float32), np.full((m, n), 7.0, np.float32)
        lin.forward_batch(kern, x, y.ravel(), m)
        lin_b.forward_batch(kern, x, yb.ravel(), m)
        for r in sorted({0, 1, m // 2, m - 1}):
            xp = np.zeros(k_pad, np.float32)
            xp[:k] = x[r]
            want = check(ref, t, w, xp, y[r], n, k_pad)
            assert np.abs(yb[r] - (want + bias)).max() <= FP32_REL_TOL * np.abs(want + bias).max()


@pytest.mark.parametrize("n", [LIMIT, LIMIT + 1])
def test_one_vector_on_both_sides_of_the_staging_limit(hip, ref, cached, n):
    say("limit, one vector", n)
    t, k = O.Q8_0, 32
    w, lin, kern = make(hip, t, n, k, 60)
    for seed in (61, 62):
        x, y = synth.normal_f32(seed, k), np.full(n, 7.0, np.float32)
        lin.forward(kern, x, y)
        check(ref, t, w, x, y, n, k)
