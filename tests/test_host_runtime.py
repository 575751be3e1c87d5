"""The library's host code (trn_runtime.cpp) over a stand-in for the HIP runtime (fake_hip.cpp): which kernel is launched with which scratch memory,
where that depends on threads, captures and failures that a GPU run cannot bring about or not every time."""
import ctypes as C
import os
import subprocess
import threading

import pytest

from tests.kq_helpers import FROM_THE_ENGINE, SHORT_ROWS_BESIDE, STREAMED_ALONE, STREAMED_IN_A_LIST
from trueno_amd._ffi import GemvDesc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
A, W, Y = 1 << 32, 1 << 40, 1 << 42


class Launch:
    def __init__(self, name, v):
        self.name, self.grid, self.block, self.stream, self.capture, self.args, self.lds = name, v[0], v[1], v[2], v[3], list(v[4:9]), v[9]


class Runtime:
    def __init__(self, path):
        self.lib = lib = C.CDLL(path)
        u64, u32 = C.c_uint64, C.c_uint32
        lib.fake_launch.restype, lib.fake_memory.restype = C.c_char_p, u64
        lib.fake_capture.argtypes = [u64, C.c_ulonglong]
        lib.fake_tuning_race.argtypes = [C.c_char_p, C.c_int, u32, u32, u32, C.c_int]
        lib.trn_q6k_gemv.argtypes = [u64, u64, u64, u64, u32, u32]
        lib.trn_gemv_f32.argtypes = [u64, u64, u64, u64, u32, u32]
        for fmt in ("q4k", "q5k", "q6k"):
            getattr(lib, f"trn_{fmt}_gemm").argtypes = [u64, u64, u64, u64, u32, u32, u32]
        lib.trn_incremental_attention.argtypes = [u64] * 5 + [u32] * 5 + [C.c_float]
        lib.trn_kquant_gemv_batch.argtypes = [u64, C.POINTER(GemvDesc), u32]
        lib.trn_stream_create.argtypes = [C.POINTER(u64), C.c_uint]
        lib.trn_stream_destroy.argtypes = [u64]

    def stream(self):
        s = C.c_uint64()
        assert self.lib.trn_stream_create(C.byref(s), 1) == 0
        return s.value

    def launched(self, issue):
        """(status, the launches) of one call."""
        before = self.lib.fake_launches()
        rc, v, out = issue(), (C.c_uint64 * 10)(), []
        for i in range(before, self.lib.fake_launches()):
            out.append(Launch(self.lib.fake_launch(i, v).decode(), v))
        return rc, out

    def f32(self, stream, k, n):
        return self.launched(lambda: self.lib.trn_gemv_f32(stream, Y, A, W, k, n))

    def gemm(self, fmt, stream, m, n, k):
        return self.launched(lambda: getattr(self.lib, f"trn_{fmt}_gemm")(stream, A, W, Y, m, n, k))

    def batch(self, stream, entries):
        """A list of products with one vector: (format code, k, n, offset of the weights) each."""
        descs = (GemvDesc * len(entries))()
        for i, (fmt, k, n, off) in enumerate(entries):
            descs[i] = GemvDesc(fmt=fmt, k=k, n=n, y=Y + (i << 32), w=W + (i << 34) + off, x=A)
        return self.launched(lambda: self.lib.trn_kquant_gemv_batch(stream, descs, len(entries)))


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    path = tmp_path_factory.mktemp("host") / "runtime.so"
    image = path.parent / "image"
    image.write_bytes(b"\x7fELF" + bytes(252))
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__", "-DKQ_U=2",
                    f"-I{os.environ.get('ROCM_PATH', '/opt/rocm')}/include", f'-DTRN_HSACO_PATH="{image}"', "-o", str(path),
                    os.path.join(ROOT, "trueno_amd", "csrc", "trn_runtime.cpp"), os.path.join(ROOT, "tests", "fake_hip.cpp"), "-pthread"], check=True)
    return Runtime(str(path))


@pytest.fixture
def rt(built):
    built.lib.fake_reset()
    yield built
    built.lib.fake_reset()


@pytest.mark.parametrize("n", [515, 516])
def test_threads_have_scratch_of_their_own_behind_the_handle_they_share(rt, n):
    counters, barrier = [], threading.Barrier(2)

    def work():
        barrier.wait()
        counters.append(rt.f32(2, 3000, n)[0])      # hipStreamPerThread
        barrier.wait()

    before = rt.lib.fake_launches()
    threads = [threading.Thread(target=work) for _ in range(2)]
    for x in threads:
        x.start()
    for x in threads:
        x.join()
    v, seen = (C.c_uint64 * 10)(), set()
    for i in range(before, rt.lib.fake_launches()):
        if rt.lib.fake_launch(i, v).decode().startswith("gemv_f32"):
            seen.add(v[8])
    assert counters == [0, 0] and len(seen) == 2


def test_scratch_of_threads_that_have_ended_is_freed(rt):
    held = []
    for _ in range(6):
        x = threading.Thread(target=lambda: rt.gemm("q4k", 2, 16, 512, 4096))
        x.start()
        x.join()
        held.append(rt.lib.fake_memory())
    assert held[1:] == held[:1] * 5      # (the one before is freed when the next is made)


@pytest.mark.parametrize("fmt,m,n,k", [("q4k", 121, 4192, 4096), ("q5k", 40, 2573, 5888)])
@pytest.mark.parametrize("warm", (False, True))
def test_captured_products_of_more_than_32_tokens_have_scratch_of_their_own(rt, fmt, m, n, k, warm):
    stream = rt.stream()
    if warm:
        rt.gemm(fmt, stream, m, n, k)
    rt.lib.fake_capture(stream, 7)
    rc, (fill, first) = rt.gemm(fmt, stream, m, n, k)
    rc2, (second,) = rt.gemm(fmt, stream, m, n, k)
    assert rc == rc2 == 0 and fill.name == "kq_fill_u32" and fill.capture == first.capture == 7
    assert fill.args[0] == first.args[3] == second.args[3]      # cleared in the graph, once
    rt.lib.fake_capture(stream, 0)
    rc, eager = rt.gemm(fmt, stream, m, n, k)
    assert rc == 0 and eager[-1].name == first.name and eager[-1].args[3] != first.args[3]
    assert [x.name for x in eager[:-1]] == ([] if warm else ["kq_fill_u32"])      # what the capture has cleared is not the stream's
    rt.lib.trn_stream_destroy(stream)


def test_a_buffer_whose_counters_could_not_be_cleared_is_not_kept(rt):
    stream, other = rt.stream(), rt.stream()
    rt.f32(other, 3000, 516)
    before = rt.lib.fake_memory()
    for n in (516, 515):
        rt.lib.fake_fail(b"kq_fill_u32")
        rc, launches = rt.f32(stream, 3000, n)
        assert rc != 0 and not launches and rt.lib.fake_memory() == before
        rt.lib.fake_capture(stream, 9)
        rc, launches = rt.f32(stream, 3000, n)
        assert rc != 0 and not launches and rt.lib.fake_memory() == before
        rt.lib.fake_capture(stream, 0)
    rt.lib.fake_fail(b"")
    for n in (515, 516):
        rc, launches = rt.f32(stream, 3000, n)
        assert rc == 0 and launches[-1].name == ("gemv_f32_ragged" if n == 515 else "gemv_f32_fast")
        assert [x.name for x in launches[:-1]] == (["kq_fill_u32"] if n == 515 else [])
    rt.lib.trn_stream_destroy(stream)
    assert rt.lib.fake_memory() == before
    rt.lib.trn_stream_destroy(other)


def test_eager_calls_make_their_scratch_while_another_stream_is_captured(rt):
    stream, captured = rt.stream(), rt.stream()
    rt.lib.fake_capture(captured, 11)
    for n in (515, 516):
        rc, launches = rt.f32(stream, 3000, n)
        assert rc == 0 and launches[-1].grid > (n + 255) // 256 and launches[-1].capture == 0      # parts of K


def test_captured_f32_products_of_odd_rows_are_cut_as_eager_ones(rt):
    """In the capture's own memory, whether or not the stream has some, and in one part, which needs none, where that cannot be had."""
    stream = rt.stream()
    for i, warm in enumerate((False, True)):
        rt.lib.fake_capture(stream, 20 + i)
        rc, (fill, product) = rt.f32(stream, 3000, 515)
        rt.lib.fake_capture(stream, 0)
        rc2, eager = rt.f32(stream, 3000, 515)
        assert rc == rc2 == 0 and fill.name == "kq_fill_u32" and product.capture == 20 + i
        assert (product.name, product.grid) == (eager[-1].name, eager[-1].grid) and product.grid > 3
        assert product.args[4] == fill.args[0] != eager[-1].args[4] and len(eager) == (1 if warm else 2)
    assert rt.lib.trn_set_tuning(b"gemm_workspace_none", 1) == 0
    rt.lib.fake_capture(stream, 30)
    rc, (product,) = rt.f32(stream, 3000, 515)
    assert rc == 0 and product.grid == 3
    assert rt.lib.trn_set_tuning(b"gemm_workspace_none", 0) == 0


def test_a_plan_is_not_older_than_the_tuning_call_before_it(rt):
    """A thread that plans a product while another changes a setting follows the change as soon as that call has returned."""
    assert rt.lib.fake_tuning_race(b"gemm_slices", 2, 64, 4096, 4096, 20000) == 0


@pytest.mark.parametrize("n", [0x7FFFFEFD, 0x7FFFFF00, 0x7FFFFF01, 0x7FFFFFFF, 0x80000001])
@pytest.mark.parametrize("shift", (0, 4))
def test_f32_products_of_two_thousand_million_columns_are_launched(rt, n, shift):
    """A launch has fewer than 2^32 threads (the stand-in refuses others, as HIP does), and the kernel with a thread per column takes what the tiled one cannot."""
    if n % 4 == 0 and shift == 0:
        n -= 2      # (the aligned form ends at 16384 column tiles)
    rc, (product,) = rt.launched(lambda: rt.lib.trn_gemv_f32(rt.stream(), Y, A + shift, W, 1, n))
    assert rc == 0 and product.grid * product.block >= n and (product.name == "gemv_f32_ragged") == (n <= 0x7FFFFF00)


def test_threads_behind_one_handle_do_not_share_the_resident_executor(rt):
    """Its tables and barrier counters belong to a stream; on hipStreamPerThread the list goes out in launches as with batch_mode 0."""
    entries, stream = [(4, 4096, 512, 0), (6, 2048, 300, 0)], rt.stream()
    plain = [x.name for x in rt.batch(stream, entries)[1]]
    assert rt.lib.trn_set_tuning(b"batch_mode", 1) == 0
    rc, own = rt.batch(stream, entries)
    rc2, shared = rt.batch(2, entries)
    assert rt.lib.trn_set_tuning(b"batch_mode", 0) == 0
    assert rc == rc2 == 0 and "kq_gemv_phases" in [x.name for x in own]
    assert [x.name for x in shared] == plain and all(x.stream == 2 for x in shared)
    rt.lib.trn_stream_destroy(stream)


@pytest.mark.parametrize("off", (0, 2, 6))
@pytest.mark.parametrize("n,k", STREAMED_ALONE + STREAMED_IN_A_LIST)
def test_the_shapes_tested_as_streamed_are(rt, n, k, off):
    """By the rings in LDS, which are larger with Q6_K's rows than with those of the Q4_K entry beside it; alone by the kernel's name as well."""
    if (n, k) in STREAMED_ALONE:
        issue = lambda: rt.launched(lambda: rt.lib.trn_q6k_gemv(0, Y, W + off, A, k, n))
    else:
        rows, cols = SHORT_ROWS_BESIDE
        issue = lambda: rt.batch(0, [(4, cols, rows, 0), (6, k, n, off)])
    seen = []
    try:
        for on in (0, 1):
            for key, value in ((b"gemv_stream_q6k", on), (b"gemv_stream_min_rows", 1), (b"group_stream_min_rows", 1)):
                assert rt.lib.trn_set_tuning(key, value) == 0
            rc, launches = issue()
            assert rc == 0 and len(launches) == 1
            seen.append(launches[0])
    finally:
        for key in (b"gemv_stream_q6k", b"gemv_stream_min_rows", b"group_stream_min_rows"):
            rt.lib.trn_set_tuning(key, 0)
    listed = (n, k) in STREAMED_IN_A_LIST or n == 32000      # (a large matrix alone is a list of one)
    assert [x.name for x in seen] == (["kq_gemv_group"] * 2 if listed else ["q6k_gemv_warp_reduce", "q6k_gemv_flags"])
    assert seen[1].lds > seen[0].lds


@pytest.mark.parametrize("fmt,m,n,k", FROM_THE_ENGINE)
def test_products_taken_from_the_engine(rt, fmt, m, n, k):
    rc, (product,) = rt.gemm(fmt, 0, m, n, k)
    assert rt.lib.trn_set_tuning(b"gemm_slices", 1) == 0
    rc2, (other,) = rt.gemm(fmt, 0, m, n, k)
    assert rt.lib.trn_set_tuning(b"gemm_slices", 0) == 0
    assert rc == rc2 == 0 and product.name.startswith(f"{fmt}_gemm_slices") and other.name == f"{fmt}_gemm_ggml"


@pytest.mark.parametrize("heads,kv_heads,dim,seq,kernel,workgroups", [
    (8, 8, 128, 128, "kq_attention_tiled_128", 8), (8, 8, 128, 129, "kq_attention_tiled_128", 24), (8, 8, 128, 512, "kq_attention_tiled_128", 64),
    (8, 8, 128, 513, "incremental_attention", 0), (1, 1, 128, 767, "incremental_attention", 0), (1, 1, 128, 768, "kq_attention_tiled_128", 12),
    (9, 9, 128, 513, "kq_attention_tiled_128", 81), (8, 4, 128, 513, "kq_attention_tiled_128", 36),
    (16, 16, 64, 128, "kq_attention_tiled_64", 16), (16, 16, 64, 129, "kq_attention_tiled_64", 48),
    (64, 8, 128, 1280, "kq_attention_tiled_128", 160), (64, 8, 128, 1281, "kq_attention_tiled_128", 88), (16, 16, 128, 1024, "kq_attention_tiled_128", 256),
    (8, 1, 128, 3840, "kq_attention_tiled_128", 60), (8, 1, 128, 3841, "kq_attention_tiled_128", 31), (1, 1, 128, 3841, "kq_attention_tiled_128", 61),
    (32, 32, 128, 4096, "kq_attention_tiled_128_w4", 256), (32, 32, 128, 3584, "kq_attention_tiled_128", 256), (32, 8, 128, 16000, "kq_attention_tiled_128", 256)])
def test_the_attention_kernels_and_their_cut(rt, heads, kv_heads, dim, seq, kernel, workgroups):
    """The lines of the rule, one position on either side: heads alone, one chunk of 128 positions, chunks of 128 instead of 64, four
    waves."""
    rc, launches = rt.launched(lambda: rt.lib.trn_incremental_attention(0, A, W, W << 1, Y, seq, dim, heads, kv_heads, seq, 0.1))
    assert rc == 0 and launches[-1].name == kernel and (workgroups == 0 or launches[-1].grid == workgroups)
