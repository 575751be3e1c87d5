"""hipStreamPerThread is one handle for as many streams as there are threads: what the library keeps beside a product (partial
sums, arrival counters) may not be shared between them."""
import ctypes as C
import threading

import numpy as np
import pytest

import trueno_amd as t
from oracle import kquant as kq
from trueno_amd import _ffi

pytestmark = pytest.mark.gpu
PER_THREAD = C.c_void_p(2)      # hipStreamPerThread


def _f32(k, n):
    def make(ctx, seed):
        rng = np.random.default_rng(seed)
        d = [t.GpuBuffer.from_host(ctx, rng.standard_normal(s).astype(np.float32)) for s in (k * n, k)]
        return d, n, lambda stream, y: _ffi.lib().trn_gemv_f32(stream, y, d[0].as_ptr(), d[1].as_ptr(), k, n)
    return make


def _gemm(m, n, k):
    def make(ctx, seed):
        d = [t.GpuBuffer.from_host(ctx, kq.gen_matrix("q4k", seed, n, k)), t.GpuBuffer.from_host(ctx, kq.gen_x(seed, m, k))]
        return d, m * n, lambda stream, y: _ffi.lib().trn_q4k_gemm(stream, d[1].as_ptr(), d[0].as_ptr(), y, m, n, k)
    return make


def _attention(heads, positions, dim):
    def make(ctx, seed):
        rng = np.random.default_rng(seed)
        d = [t.GpuBuffer.from_host(ctx, rng.standard_normal(s).astype(np.float32)) for s in (heads * dim, *[heads * positions * dim] * 2)]
        return d, heads * dim, lambda stream, y: _ffi.lib().trn_incremental_attention(
            stream, d[0].as_ptr(), d[1].as_ptr(), d[2].as_ptr(), y, positions, dim, heads, heads, positions, C.c_float(dim ** -0.5))
    return make


@pytest.mark.parametrize("make", [_f32(3000, 515), _f32(3000, 516), _gemm(16, 512, 4096), _attention(8, 900, 128)],
                         ids=["f32_odd_rows", "f32", "gemm", "attention"])
def test_two_threads_at_once(gpu, make):
    """Each thread's hundred products, queued without waiting, have the bits that the same product has on a stream of its own."""
    ctx, stream = gpu
    calls, rounds, bad = [make(ctx, 900 + i) for i in range(2)], 100, []
    want = []
    for held, size, issue in calls:
        dy = t.GpuBuffer.from_host(ctx, np.full(size, np.nan, np.float32))
        assert issue(stream.raw(), dy.as_ptr()) == 0
        stream.synchronize()
        want.append(dy.copy_to_host().view(np.uint32))
    out = [t.GpuBuffer.from_host(ctx, np.full(rounds * size, np.nan, np.float32)) for _, size, _ in calls]
    ready = threading.Barrier(2)

    def work(i):
        ctx.make_current()
        _, size, issue = calls[i]
        ready.wait()
        rc = [issue(PER_THREAD, out[i].as_ptr() + 4 * size * r) for r in range(rounds)]
        rc.append(_ffi.lib().trn_stream_synchronize(PER_THREAD))
        bad.extend(x for x in rc if x != 0)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for x in threads:
        x.start()
    for x in threads:
        x.join()
    assert not bad
    for dy, w in zip(out, want):
        assert np.all(dy.copy_to_host().view(np.uint32).reshape(rounds, -1) == w)


def test_threads_that_end_give_their_memory_back(gpu):
    """Twelve threads one after the other, 16 MiB of scratch each: at most two of them are held at a time."""
    ctx, _ = gpu
    _, size, issue = _gemm(16, 512, 4096)(ctx, 910)
    dy, free, rc = t.GpuBuffer.from_host(ctx, np.zeros(size, np.float32)), [], []

    def work():
        ctx.make_current()
        rc.append(issue(PER_THREAD, dy.as_ptr()))
        rc.append(_ffi.lib().trn_stream_synchronize(PER_THREAD))
        now, total = C.c_size_t(), C.c_size_t()
        rc.append(_ffi.lib().trn_mem_get_info(C.byref(now), C.byref(total)))
        free.append(now.value)

    for _ in range(12):
        x = threading.Thread(target=work)
        x.start()
        x.join()
    assert not any(rc) and free[1] - free[-1] < 48 << 20, free
