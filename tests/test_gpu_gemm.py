"""GPU parity, batched GEMM C = A . dequant(W)^T: within 1e-5 relative L2 of fp64 for M in {1, 4, 16, 64},
row-major C, m = 1 equal to the GEMV; typed launcher and launch-by-name."""
import ctypes as C

import numpy as np
import pytest

import trueno_amd as t
from oracle import kquant as kq
from trueno_amd import _ffi
from tests.kq_helpers import FROM_THE_ENGINE, REF_SLACK, gpu_gemm, gpu_gemv, record_ratio

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _c64(fmt, buf, a, n, k):
    return kq.gemm_fp64(a, kq.dequant_matrix(fmt, buf, n, k))


@pytest.mark.parametrize("m", (1, 4, 16, 64))
@pytest.mark.parametrize("fmt,n,k", [("q4k", 1024, 4096), ("q4k", 520, 14336), ("q5k", 300, 1024), ("q6k", 300, 2048)])
def test_gemm_against_fp64(gpu, fmt, n, k, m):
    buf, a = kq.gen_matrix(fmt, 200 + m, n, k), kq.gen_x(300 + m, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert c.shape == (m, n) and np.all(np.isfinite(c))
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


@pytest.mark.parametrize("m", (1, 5))
@pytest.mark.parametrize("fmt,n,k", [("q4k", 300, 1024), ("q5k", 300, 1024), ("q6k", 300, 2048), ("q4k", 64, 14336)])
def test_gemm_with_the_decode_as_written(gpu, fmt, n, k, m):
    """q*k_gemm_ggml with the GEMM family's own decode (policy 1; quantize.rs:445-514, :727-807, :1009-1064): against
    fp64 on the oracle's as-written weights, and really different from the canonical decode's product."""
    buf, a = kq.gen_matrix(fmt, 400 + m, n, k), kq.gen_x(500 + m, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k, as_written=True)
    want = kq.gemm_fp64(a, kq.dequant_matrix(fmt, buf, n, k, policy=1))
    assert c.shape == (m, n) and np.all(np.isfinite(c))
    assert kq.rel_l2(c, want) <= TOL
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) > 1e-2


@pytest.mark.parametrize("m", (1, 4, 16, 64))
def test_gemm_config_shape_w_14336x4096(gpu, m):
    n, k = 14336, 4096
    buf, a = kq.gen_matrix("q4k", 1234, n, k), kq.gen_x(4321, m, k)
    c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    assert kq.rel_l2(c, _c64("q4k", buf, a, n, k)) <= TOL


@pytest.mark.parametrize("m", (1, 4, 16, 64))
def test_gemm_config_shape_w_4096x14336(gpu, m):
    n, k = 4096, 14336
    buf, a = kq.gen_matrix("q4k", 1235, n, k), kq.gen_x(4322, m, k)
    c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    assert kq.rel_l2(c, _c64("q4k", buf, a, n, k)) <= TOL


@pytest.mark.parametrize("fmt", ("q4k", "q5k", "q6k"))
def test_gemm_m1_equals_gemv_and_by_name(gpu, fmt):
    ctx, _ = gpu
    n, k = 777, 1536
    buf, a = kq.gen_matrix(fmt, 7, n, k), kq.gen_x(8, 3, k)
    y = gpu_gemv(gpu, fmt, buf, a[0], k, n)
    c1 = gpu_gemm(gpu, fmt, buf, a[:1], 1, n, k)
    assert kq.rel_l2(c1[0], y.astype(np.float64)) <= 2e-7
    mod = t.CudaModule.from_builtin(ctx)
    c3 = gpu_gemm(gpu, fmt, buf, a, 3, n, k, by_name=mod)
    assert kq.rel_l2(c3, _c64(fmt, buf, a, n, k)) <= TOL
    assert kq.rel_l2(c3[0], y.astype(np.float64)) <= 2e-7


def test_gemm_edge_cases(gpu):
    ctx, stream = gpu
    a = t.GpuBuffer.from_host(ctx, np.ones(256, np.float32))
    w = t.GpuBuffer.from_host(ctx, np.zeros(144, np.uint8))
    c = t.GpuBuffer.from_host(ctx, np.full(4, 3.0, np.float32))
    t.QuantizeKernel.ggml(0, 1, 256).launch(stream, a, w, c)      # m = 0: nothing written
    t.QuantizeKernel.ggml(1, 0, 256).launch(stream, a, w, c)      # n = 0
    stream.synchronize()
    assert np.all(c.copy_to_host() == 3.0)
    with pytest.raises(t.GpuError):
        t.QuantizeKernel.ggml(1, 1, 300).launch(stream, a, w, c)  # k % 256 != 0


def _tune(key, value):
    from trueno_amd import _ffi
    assert _ffi.lib().trn_set_tuning(key.encode(), int(value)) == 0


MFMA_FORMATS = ("q4k", "q5k", "q6k")      # the formats whose GEMM runs on the matrix cores for m >= 2


@pytest.mark.parametrize("m", (4, 16, 64))
@pytest.mark.parametrize("fmt", ("q5k", "q6k"))
def test_gemm_4096x4096(gpu, fmt, m):
    n = k = 4096
    buf, a = kq.gen_matrix(fmt, 1239, n, k), kq.gen_x(4321, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


@pytest.mark.parametrize("m", (2, 9, 13, 33))
@pytest.mark.parametrize("n,k", [(100, 512), (1000, 2304)])
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_matrix_core_form_ragged(gpu, fmt, n, k, m):
    """Token counts that do not fill a tile of 16, row counts that do not fill a strip of 32 or a group of 8 strips."""
    buf, a = kq.gen_matrix(fmt, 50 + m, n, k), kq.gen_x(60 + m, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


@pytest.mark.parametrize("m", (17, 33, 40, 64))
@pytest.mark.parametrize("fmt", ("q4k", "q5k"))
def test_gemm_two_token_tiles_per_workgroup(gpu, fmt, m):
    """The kernels that take two tiles of 16 tokens per workgroup, forced on a small product: odd numbers of tiles
    (the second tile of the last pair does not exist), K in one part and in several, the same bits on every run;
    and one tile per workgroup gives the same bits for the same cut of K (a tile's sums do not depend on its
    company)."""
    n, k = 300, 1536
    buf, a = kq.gen_matrix(fmt, 70 + m, n, k), kq.gen_x(80 + m, m, k)
    c64 = _c64(fmt, buf, a, n, k)
    try:
        for parts in (1, 3):
            _tune("gemm_k_parts", parts)
            _tune("gemm_tiles", 2)
            two = gpu_gemm(gpu, fmt, buf, a, m, n, k)
            assert kq.rel_l2(two, c64) <= TOL
            again = gpu_gemm(gpu, fmt, buf, a, m, n, k)
            assert np.array_equal(again.view(np.uint32), two.view(np.uint32)), parts
            _tune("gemm_tiles", 1)
            one = gpu_gemm(gpu, fmt, buf, a, m, n, k)
            assert np.array_equal(one.view(np.uint32), two.view(np.uint32)), parts
    finally:
        _tune("gemm_k_parts", 0)
        _tune("gemm_tiles", 0)


@pytest.mark.parametrize("fmt", ("q4k", "q5k"))
def test_gemm_many_tokens(gpu, fmt):
    """512 tokens against 4096 x 2048: enough workgroups that the library itself takes two tiles per workgroup."""
    n, k, m = 4096, 2048, 512
    buf, a = kq.gen_matrix(fmt, 77, n, k), kq.gen_x(78, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


@pytest.mark.parametrize("m", (5, 20))
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_few_rows_long_k(gpu, fmt, m):
    """96 rows against K = 8192: one group of strips, so the library cuts K into as many parts as there are
    super-blocks (32) and the last workgroup adds them in two rounds of sixteen."""
    n, k = 96, 8192
    buf, a = kq.gen_matrix(fmt, 300 + m, n, k), kq.gen_x(310 + m, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL
    again = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert np.array_equal(again.view(np.uint32), c.view(np.uint32))


@pytest.mark.parametrize("m", (5, 24, 40))
def test_gemm_twelve_strips_per_workgroup(gpu, m):
    """The Q4_K kernel that takes twelve strips of 32 rows per workgroup (its last four waves convert no tokens), forced
    on a small product whose rows fill neither the last strip nor the last workgroup: within tolerance, and the same
    bits as eight strips per workgroup for the same cut of K (a strip's sums do not depend on its company)."""
    n, k = 777, 2048
    buf, a = kq.gen_matrix("q4k", 400 + m, n, k), kq.gen_x(410 + m, m, k)
    c64 = _c64("q4k", buf, a, n, k)
    try:
        for parts in (1, 3):
            _tune("gemm_k_parts", parts)
            _tune("gemm_waves", 12)
            twelve = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
            assert kq.rel_l2(twelve, c64) <= TOL
            _tune("gemm_waves", 8)
            _tune("gemm_tiles", 1)
            eight = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
            assert np.array_equal(eight.view(np.uint32), twelve.view(np.uint32)), parts
            _tune("gemm_tiles", 0)
    finally:
        _tune("gemm_k_parts", 0)
        _tune("gemm_waves", 0)
        _tune("gemm_tiles", 0)


@pytest.mark.parametrize("m", (4, 32))
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_ffn_shape_w_11008x4096(gpu, fmt, m):
    """The 7B gate/up shape: 43 groups of 8 strips do not divide the CUs well, so the library takes fewer parts of K than
    would fill them (and, for Q4_K with 32 tokens, twelve strips per workgroup)."""
    n, k = 11008, 4096
    buf, a = kq.gen_matrix(fmt, 500 + m, n, k), kq.gen_x(510 + m, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


def _random_shapes():
    rng = np.random.default_rng(20251125)
    for i in range(15):
        fmt = MFMA_FORMATS[i % 3]
        k = 256 * int(rng.integers(1, 33))
        n = int(rng.integers(1, 5000)) if i % 3 else 32 * int(rng.integers(1, 150))
        m = int(rng.choice([2, 3, 5, 9, 16, 17, 31, 33, 48, 64, 65, 100, 130, 257]))
        yield fmt, m, n, k, i


@pytest.mark.parametrize("fmt,m,n,k,i", list(_random_shapes()))
def test_gemm_random_shapes(gpu, fmt, m, n, k, i):
    """Shapes drawn at random (fixed seed): whatever cut of the product the library's estimate picks for them - strips per
    workgroup, token tiles per workgroup, parts of K of unequal length - the result is within tolerance."""
    buf, a = kq.gen_matrix(fmt, 1000 + i, n, k), kq.gen_x(2000 + i, m, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    assert np.all(np.isfinite(c))
    assert kq.rel_l2(c, _c64(fmt, buf, a, n, k)) <= TOL


@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_parts_of_k(gpu, fmt):
    """However K is cut into parts the result stays within tolerance, and the same cut gives the same bits on
    every run: the parts are added in part order by whichever workgroup arrives last."""
    n, k, m = 777, 2048, 24
    buf, a = kq.gen_matrix(fmt, 91, n, k), kq.gen_x(92, m, k)
    c64 = _c64(fmt, buf, a, n, k)
    try:
        for waves in (4, 8):
            _tune("gemm_waves", waves)
            for parts in (1, 2, 3, 8):
                _tune("gemm_k_parts", parts)
                first = gpu_gemm(gpu, fmt, buf, a, m, n, k)
                assert kq.rel_l2(first, c64) <= TOL
                for _ in range(3):
                    again = gpu_gemm(gpu, fmt, buf, a, m, n, k)
                    assert np.array_equal(again.view(np.uint32), first.view(np.uint32)), (waves, parts)
    finally:
        _tune("gemm_k_parts", 0)
        _tune("gemm_waves", 0)
    try:
        _tune("gemm_mfma_off", 1)
        valu = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    finally:
        _tune("gemm_mfma_off", 0)
    assert kq.rel_l2(valu, c64) <= TOL


# The matrix-core form against the reference's own f32 result, per format and cut: (shape, tokens).  4096 columns in one
# part, 14336 columns in parts of K; 16 tokens (one tile) and 64 (two tiles per workgroup for Q4_K / Q5_K).
@pytest.mark.parametrize("n,k,m", [(2048, 4096, 16), (1024, 14336, 16), (1024, 4096, 64)])
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_no_worse_than_reference_order_f32(gpu, coracle, fmt, n, k, m):
    """Per product, the error against fp64 is no larger than that of an f32 evaluation in the reference's summation
    order (quantize.rs:1412-1518), up to the sampling margin."""
    buf, a = kq.gen_matrix(fmt, 93, n, k), kq.gen_x(94, m, k)
    w = kq.dequant_matrix(fmt, buf, n, k)
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    c64 = kq.gemm_fp64(a, w)
    ref = np.stack([coracle.gemv_ref_order_f32(fmt, buf, a[i], k, n) for i in range(m)])
    err_ref, err_ours = kq.rel_l2(ref, c64), kq.rel_l2(c, c64)
    record_ratio("gemm", fmt, m, n, k, n, err_ours, err_ref)
    assert err_ours <= REF_SLACK * err_ref, (fmt, m, n, k, err_ours, err_ref, err_ours / err_ref)


@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_special_values(gpu, fmt):
    """An all-zero token, a huge and a tiny token, and a token with an infinity (its outputs are not finite,
    the other tokens are untouched)."""
    n, k, m = 64, 512, 5
    buf = kq.gen_matrix(fmt, 95, n, k)
    a = kq.gen_x(96, m, k)
    a[1] = 0.0
    a[2] *= 1e30
    a[3] *= 1e-30
    a[4, 17] = np.inf
    c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    w = kq.dequant_matrix(fmt, buf, n, k)
    c64 = kq.gemm_fp64(a[:4], w)
    assert np.all(c[1] == 0.0)
    for i in (0, 2, 3):
        assert kq.rel_l2(c[i], c64[i]) <= TOL
    assert not np.any(np.isfinite(c[4]))


def test_gemm_on_streams_that_come_and_go(gpu):
    """the scratch buffers a stream's products use (partial sums, arrival counters) go with the stream; a new stream,
    possibly with the old one's handle, starts from clean ones"""
    ctx, _ = gpu
    n, k, m = 1024, 4096, 4                       # K is cut in parts on this shape: partial sums and counters in use
    buf, a = kq.gen_matrix("q4k", 91, n, k), kq.gen_x(92, m, k)
    want = _c64("q4k", buf, a, n, k)
    first = None
    for _ in range(3):
        stream = t.CudaStream(ctx)
        c = gpu_gemm((ctx, stream), "q4k", buf, a, m, n, k)
        assert kq.rel_l2(c, want) <= TOL
        first = c if first is None else first
        assert np.array_equal(c.view(np.uint32), first.view(np.uint32))
        stream.destroy()


# ---- two to four tokens on the integer matrix cores (Q4_K, k <= 4096) --------------------------------------------------
FEW_SHAPES = [(64, 256), (100, 1024), (33, 2304), (1000, 4096), (8300, 4096), (14336, 4096)]


@pytest.mark.parametrize("m", (2, 3, 4))
@pytest.mark.parametrize("n,k", FEW_SHAPES)
def test_gemm_few_tokens_on_the_integer_cores(gpu, n, k, m):
    """One to 260 tiles of 32 rows (one or two per workgroup, the last one ragged), one to sixteen super-blocks per row,
    every token count the kernel takes: within the contract's distance of fp64, and not the result of another path."""
    buf, a = kq.gen_matrix("q4k", 600 + m, n, k), kq.gen_x(700 + m, m, k)
    want = _c64("q4k", buf, a, n, k)
    try:
        _tune("gemm_few", 1)
        c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
        _tune("gemm_few", 2)
        other = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    finally:
        _tune("gemm_few", 0)
    assert c.shape == (m, n) and np.all(np.isfinite(c))
    assert kq.rel_l2(c, want) <= TOL and kq.rel_l2(other, want) <= TOL
    assert not np.array_equal(c, other)                      # (two orders of summation: the same bits would mean one path ran twice)


@pytest.mark.parametrize("n,k,m", [(20000, 4096, 3), (40000, 4096, 2), (30000, 1024, 4), (70000, 256, 4)])
def test_gemm_few_tokens_several_tiles_per_workgroup(gpu, n, k, m):
    """Three to nine tiles per workgroup: the copies of the tile after next are issued between the products of the
    current one, and a tile's results leave while the next is multiplied (rows of 16, 4 and 1 super-blocks: four, two and
    one of the eight waves have products of their own)."""
    buf, a = kq.gen_matrix("q4k", 810 + m, n, k), kq.gen_x(820 + m, m, k)
    try:
        _tune("gemm_few", 1)
        c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    finally:
        _tune("gemm_few", 0)
    want = _c64("q4k", buf, a, n, k)
    assert np.all(np.isfinite(c)) and kq.rel_l2(c, want) <= TOL
    for i in range(m):                                       # every token, and the ends of the matrix on their own
        assert kq.rel_l2(c[i], want[i]) <= TOL
        assert kq.rel_l2(c[i, -40:], want[i, -40:]) <= TOL and kq.rel_l2(c[i, :40], want[i, :40]) <= TOL


@pytest.mark.parametrize("m", (2, 4))
def test_gemm_few_tokens_no_worse_than_reference_order_f32(gpu, coracle, m):
    n, k = 2048, 4096
    buf, a = kq.gen_matrix("q4k", 93, n, k), kq.gen_x(94, m, k)
    c64 = kq.gemm_fp64(a, kq.dequant_matrix("q4k", buf, n, k))
    try:
        _tune("gemm_few", 1)
        c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    finally:
        _tune("gemm_few", 0)
    ref = np.stack([coracle.gemv_ref_order_f32("q4k", buf, a[i], k, n) for i in range(m)])
    err_ref, err_ours = kq.rel_l2(ref, c64), kq.rel_l2(c, c64)
    record_ratio("gemm_few", "q4k", m, n, k, n, err_ours, err_ref)
    assert err_ours <= REF_SLACK * err_ref, (m, err_ours, err_ref, err_ours / err_ref)


def test_gemm_few_tokens_special_values(gpu):
    """Tokens of zeros, of huge and of tiny values; a token whose runs of 256 differ by 2^40 in size and one with a single
    large element among small ones (each run has its own power of two, so the small ones keep their bits); unit vectors
    (the product is then one weight, d * s * q - dmin * m, to a few ulps of its two terms); an infinity spoils its
    token and no other."""
    n, k = 96, 1024
    buf = kq.gen_matrix("q4k", 95, n, k)
    w = kq.dequant_matrix("q4k", buf, n, k)
    a = kq.gen_x(96, 4, k)
    a[1] = 0.0
    a[2] *= 1e30
    a[3, :256] *= 2.0 ** 40
    a[3, 700] = 3.0e4
    try:
        _tune("gemm_few", 1)
        c = gpu_gemm(gpu, "q4k", buf, a, 4, n, k)
        a2 = kq.gen_x(97, 3, k) * 1e-30
        a2[1] = 0.0
        a2[1, 517] = 1.0
        a2[2, 3] = np.inf
        c2 = gpu_gemm(gpu, "q4k", buf, a2.astype(np.float32), 3, n, k)
    finally:
        _tune("gemm_few", 0)
    c64 = kq.gemm_fp64(a, w)
    assert np.all(c[1] == 0.0)
    for i in (0, 2, 3):
        assert kq.rel_l2(c[i], c64[i]) <= TOL
    assert kq.rel_l2(c2[0], kq.gemm_fp64(a2[:1].astype(np.float32), w)[0]) <= TOL
    col = w[:, 517].astype(np.float64)
    assert np.all(np.abs(c2[1] - col) <= 2.0 ** -21 * np.abs(w).max())
    assert not np.any(np.isfinite(c2[2]))


def test_gemm_few_tokens_by_the_rule(gpu):
    """Left to itself the launcher takes the integer-core kernel where it is the fastest way (two tokens against 14336
    rows), and not for one token, for five, or for rows longer than a slab of 4096 columns."""
    for m, n, k, taken in [(2, 14336, 4096, True), (1, 2048, 4096, False), (5, 2048, 4096, False), (2, 256, 8192, False)]:
        buf, a = kq.gen_matrix("q4k", 31 + m, n, k), kq.gen_x(32 + m, m, k)
        c = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
        try:
            _tune("gemm_few", 2)
            other = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
        finally:
            _tune("gemm_few", 0)
        assert kq.rel_l2(c, _c64("q4k", buf, a, n, k)) <= TOL
        assert np.array_equal(c, other) != taken, (m, n, k)


@pytest.mark.parametrize("parts", (0, 1, 3))
@pytest.mark.parametrize("m,n,k", [(33, 1, 256), (64, 255, 512), (65, 257, 1280), (97, 700, 2304)])
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_many_tokens_kernel(gpu, fmt, m, n, k, parts):
    """The kernel for many tokens, forced: rows that fill neither a strip of 64 nor a group of 256, tokens that do not fill
    a tile of 32, one super-block, K in one part, three (of unequal length) and as many as the library takes: within
    tolerance and the same bits on every run, a token's values large against the others' of its tile, and a run with an
    infinity not finite - in its own token only."""
    buf, a = kq.gen_matrix(fmt, 600 + m, n, k), kq.gen_x(610 + m, m, k)
    a[1] *= np.float32(1e6)
    a[m - 1] *= np.float32(1e-6)
    c64 = _c64(fmt, buf, a, n, k)
    # a single result may cancel: each is held to 1e-5 of the sum of its terms' sizes (about forty roundings of 2^-24 in a
    # row at worst, the minimum's term on top), a whole token's results to the usual relative L2
    terms = np.abs(a).astype(np.float64) @ np.abs(kq.dequant_matrix(fmt, buf, n, k)).astype(np.float64).T
    try:
        _tune("gemm_tall", 2)
        _tune("gemm_k_parts", parts)
        c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert np.all(np.abs(c - c64) <= TOL * terms)
        for row in (slice(0, 1), slice(1, 2), slice(2, m - 1), slice(m - 1, m)):
            assert n < 255 or kq.rel_l2(c[row], c64[row]) <= TOL
        again = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert np.array_equal(again.view(np.uint32), c.view(np.uint32))
        a[3, 7] = np.inf
        c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert not np.any(np.isfinite(c[3])) and np.all(np.isfinite(np.delete(c, 3, axis=0)))
        assert np.array_equal(np.delete(c, 3, axis=0), np.delete(again, 3, axis=0))
    finally:
        _tune("gemm_tall", 0)
        _tune("gemm_k_parts", 0)


@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_many_tokens_no_less_exact_than_sixteen_at_a_time(gpu, fmt):
    """The rule's own choice for 200 tokens against 8192 x 2048, and the kernel that takes sixteen at a time: the error
    against fp64 is no larger (bound 1.02: what the seeds' scatter moves the ratio by)."""
    m, n, k = 200, 8192, 2048
    buf, a = kq.gen_matrix(fmt, 640, n, k), kq.gen_x(641, m, k)
    c64 = _c64(fmt, buf, a, n, k)
    err = {}
    try:
        for name, value in (("rule", 0), ("tall", 2), ("sixteen", 1)):
            _tune("gemm_tall", value)
            err[name] = kq.rel_l2(gpu_gemm(gpu, fmt, buf, a, m, n, k), c64)
    finally:
        _tune("gemm_tall", 0)
    assert err["rule"] == err["tall"] != err["sixteen"]
    assert err["tall"] <= 1.02 * err["sixteen"]


def test_gemm_many_tokens_under_capture_and_without_allocation(gpu):
    """Twice the same bits through a captured graph after a larger product has grown the workspace, and from
    trn_q4k_gemm_noalloc, whose workspace is the library's own."""
    import ctypes as C
    from trueno_amd import _ffi
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphExecDestroy.argtypes = [C.c_void_p]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    ctx, stream = gpu
    m, n, k = 700, 4096, 8192
    buf, a = kq.gen_matrix("q4k", 650, n, k), kq.gen_x(651, m, k)
    want = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
    dw, da = t.GpuBuffer.from_host(ctx, buf), t.GpuBuffer.from_host(ctx, a)
    dc = t.GpuBuffer.from_host(ctx, np.full(m * n, np.nan, np.float32))
    assert _ffi.lib().trn_q4k_gemm_noalloc(stream.raw(), da.as_ptr(), dw.as_ptr(), dc.as_ptr(), m, n, k) == 0
    stream.synchronize()
    assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), want.view(np.uint32))
    graph, gexec = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream.raw(), 0) == 0
    t.QuantizeKernel.ggml(m, n, k).launch(stream, da, dw, dc)
    assert hip.hipStreamEndCapture(stream.raw(), C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
    try:
        gpu_gemm(gpu, "q4k", buf, np.concatenate((a, a)), 2 * m, n, k)      # grows the workspace: the graph's stays
        for _ in range(3):
            dc.copy_from_host(np.full(m * n, np.nan, np.float32))
            assert hip.hipGraphLaunch(gexec, stream.raw()) == 0
            stream.synchronize()
            assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), want.view(np.uint32))
            again = gpu_gemm(gpu, "q4k", buf, a, m, n, k)
            assert np.array_equal(again.view(np.uint32), want.view(np.uint32))
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)


class _Dim3(C.Structure):
    _fields_ = [("x", C.c_uint), ("y", C.c_uint), ("z", C.c_uint)]


class _KernelNodeParams(C.Structure):
    _fields_ = [("block", _Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", _Dim3), ("args", C.POINTER(C.c_void_p)),
                ("lds", C.c_uint)]


def _hip():
    hip = C.CDLL("libamdhip64.so")
    hip.hipStreamBeginCapture.argtypes = [C.c_void_p, C.c_int]
    hip.hipStreamEndCapture.argtypes = [C.c_void_p, C.POINTER(C.c_void_p)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [C.c_void_p, C.c_void_p]
    hip.hipGraphGetRootNodes.argtypes = [C.c_void_p, C.POINTER(C.c_void_p), C.POINTER(C.c_size_t)]
    hip.hipGraphKernelNodeGetParams.argtypes = [C.c_void_p, C.POINTER(_KernelNodeParams)]
    hip.hipGraphExecDestroy.argtypes = [C.c_void_p]
    hip.hipGraphDestroy.argtypes = [C.c_void_p]
    return hip


class _Captured:
    """What `issue` puts on the stream, as a graph."""

    def __init__(self, stream, issue):
        self.hip, self.graph, self.instance = _hip(), C.c_void_p(), C.c_void_p()
        assert self.hip.hipStreamBeginCapture(stream.raw(), 0) == 0
        try:
            issue()
        finally:
            rc = self.hip.hipStreamEndCapture(stream.raw(), C.byref(self.graph))
        assert rc == 0 and self.hip.hipGraphInstantiate(C.byref(self.instance), self.graph, None, None, 0) == 0

    def replay(self, stream):
        assert self.hip.hipGraphLaunch(self.instance, stream.raw()) == 0

    def first_kernel(self):
        """(workgroups, the second argument as an address) of the kernel that the graph starts with."""
        node, count, p = C.c_void_p(), C.c_size_t(1), _KernelNodeParams()
        assert self.hip.hipGraphGetRootNodes(self.graph, C.byref(node), C.byref(count)) == 0 and count.value == 1
        assert self.hip.hipGraphKernelNodeGetParams(node, C.byref(p)) == 0
        return p.grid.x, C.cast(p.args[1], C.POINTER(C.c_uint64))[0]

    def close(self):
        assert self.hip.hipGraphExecDestroy(self.instance) == 0 and self.hip.hipGraphDestroy(self.graph) == 0


def test_gemm_many_tokens_captured_products_keep_to_themselves(gpu):
    """Two graphs captured on one stream, the first of them before that stream has seen any product: each has operand
    memory of its own, and both give the eager call's bits when they are replayed on other streams at once, beside eager
    products on the stream they were captured on, and after that stream is gone and its memory with it."""
    ctx, other = gpu
    shapes, stream, kernel = ((97, 1), (200, 2)), t.CudaStream(ctx), "q4k"
    n, k = 700, 2304
    buf = kq.gen_matrix(kernel, 660, n, k)
    dw, graphs, want, out, held = t.GpuBuffer.from_host(ctx, buf), [], [], [], []
    streams = [t.CudaStream(ctx) for _ in shapes]
    _tune("gemm_tall", 2)
    try:
        for m, seed in shapes:
            a = kq.gen_x(660 + seed, m, k)
            want.append(gpu_gemm(gpu, kernel, buf, a, m, n, k).view(np.uint32))
            da, dc = t.GpuBuffer.from_host(ctx, a), t.GpuBuffer.from_host(ctx, np.full(m * n, np.nan, np.float32))
            held.append(da)
            out.append(dc)
            graphs.append(_Captured(stream, lambda: t.QuantizeKernel.ggml(m, n, k).launch(stream, da, dw, dc)))
        first = [g.first_kernel() for g in graphs]
        assert [grid for grid, _ in first] == [(m + 31) // 32 * (k // 256) for m, _ in shapes]      # the kernel for many tokens
        assert first[0][1] != first[1][1]

        def replay_both():
            for dc in out:
                dc.copy_from_host(np.full(dc.len(), np.nan, np.float32))
            for _ in range(3):
                for g, s in zip(graphs, streams):
                    g.replay(s)

        def check():
            for dc, w, s in zip(out, want, streams):
                s.synchronize()
                assert np.array_equal(dc.copy_to_host().reshape(w.shape).view(np.uint32), w)

        big = kq.gen_x(669, 400, k)
        big_want = gpu_gemm(gpu, kernel, buf, big, 400, n, k).view(np.uint32)
        for _ in range(3):
            replay_both()
            assert np.array_equal(gpu_gemm((ctx, stream), kernel, buf, big, 400, n, k).view(np.uint32), big_want)
            check()
        stream.destroy()
        poison = [t.GpuBuffer.from_host(ctx, np.full(1 << 20, np.nan, np.float32)) for _ in range(8)]      # takes what was freed
        for _ in range(3):
            replay_both()
            check()
        assert all(np.all(np.isnan(p.copy_to_host())) for p in poison)
    finally:
        _tune("gemm_tall", 0)
        other.synchronize()
        for g in graphs:
            g.close()


def test_gemm_many_tokens_without_memory_for_a_workspace(gpu):
    """Where no workspace can be had the product goes to the kernel that takes sixteen tokens at a time: on a fresh stream, on
    one whose workspace is too small (which it keeps for smaller products), and under capture on a stream that has seen
    only products of many tokens."""
    ctx, _ = gpu
    n, k, (small, large) = 700, 2304, (64, 300)
    buf = kq.gen_matrix("q5k", 680, n, k)
    a = {m: kq.gen_x(681 + m, m, k) for m in (small, large)}
    bits, refused, used = {}, t.CudaStream(ctx), t.CudaStream(ctx)

    def run(stream, m):
        return gpu_gemm((ctx, stream), "q5k", buf, a[m], m, n, k).view(np.uint32)

    dw, da = t.GpuBuffer.from_host(ctx, buf), t.GpuBuffer.from_host(ctx, a[large])
    dc = t.GpuBuffer.from_host(ctx, np.full(large * n, np.nan, np.float32))
    try:
        for tall in (1, 2):
            _tune("gemm_tall", tall)
            bits[tall] = {m: run(gpu[1], m) for m in a}
        assert not any(np.array_equal(bits[1][m], bits[2][m]) for m in a)
        assert np.array_equal(run(used, small), bits[2][small])
        _tune("gemm_workspace_none", 1)
        for m in a:
            assert np.array_equal(run(refused, m), bits[1][m])
        assert np.array_equal(run(used, large), bits[1][large]) and np.array_equal(run(used, small), bits[2][small])
        _tune("gemm_workspace_none", 0)
        warm = t.CudaStream(ctx)
        assert np.array_equal(run(warm, large), bits[2][large])
        _tune("gemm_workspace_none", 1)
        graph = _Captured(warm, lambda: t.Q5KKernel(large, n, k).launch(warm, da, dw, dc))
        for _ in range(3):
            dc.copy_from_host(np.full(large * n, np.nan, np.float32))
            graph.replay(warm)
            warm.synchronize()
            assert np.array_equal(dc.copy_to_host().reshape(large, n).view(np.uint32), bits[1][large])
        graph.close()
    finally:
        _tune("gemm_tall", 0)
        _tune("gemm_workspace_none", 0)


def test_gemm_many_tokens_in_runs(gpu):
    """A workspace that holds three token tiles: the same bits in four runs as in one, from both entry points, and in as many
    runs of one tile.  The rule prices the runs: a product that it gives to the kernel for many tokens in one run goes sixteen
    tokens at a time in a workspace that would cut it into runs of a few tiles, from both entry points again."""
    ctx, stream = gpu
    L = _ffi.lib()

    def both(buf, a, n, k):
        m = a.shape[0]
        got = gpu_gemm(gpu, "q4k", buf, a, m, n, k).view(np.uint32)
        dw, da = t.GpuBuffer.from_host(ctx, buf), t.GpuBuffer.from_host(ctx, a)
        dc = t.GpuBuffer.from_host(ctx, np.full(m * n, np.nan, np.float32))
        assert L.trn_q4k_gemm_noalloc(stream.raw(), da.as_ptr(), dw.as_ptr(), dc.as_ptr(), m, n, k) == 0
        stream.synchronize()
        assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), got)
        return got

    try:
        n, k = 300, 2304                                  # a tile of 32 tokens: 9 x 34 KiB, in one part of K
        buf, a = kq.gen_matrix("q4k", 690, n, k), kq.gen_x(691, 321, k)
        _tune("gemm_tall", 2)
        for parts in (1, 3):
            _tune("gemm_k_parts", parts)
            _tune("gemm_workspace_mb", 0)
            whole = both(buf, a, n, k)
            for mb in (1, 2):
                _tune("gemm_workspace_mb", mb)
                assert np.array_equal(both(buf, a, n, k), whole), (parts, mb)
        _tune("gemm_tall", 0)
        _tune("gemm_k_parts", 0)
        n, k = 4096, 4096
        buf, a = kq.gen_matrix("q4k", 692, n, k), kq.gen_x(693, 512, k)
        bits = {}
        for name, tall, mb in (("tall", 2, 0), ("sixteen", 1, 0), ("rule", 0, 0), ("rule, small", 0, 2)):
            _tune("gemm_tall", tall)
            _tune("gemm_workspace_mb", mb)
            bits[name] = both(buf, a, n, k)
        assert np.array_equal(bits["rule"], bits["tall"]) and np.array_equal(bits["rule, small"], bits["sixteen"])
        assert not np.array_equal(bits["tall"], bits["sixteen"])
    finally:
        for key in ("gemm_tall", "gemm_k_parts", "gemm_workspace_mb"):
            _tune(key, 0)


@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_many_tokens_beside_one_value_much_larger(gpu, fmt):
    """One activation in every run of 256 is 2^12, 2^20, 2^24 times larger than the others, and the weights of its sub-block are
    zero: the others' pieces, scaled by the run's maximum, keep all their bits.  Two pieces of eleven bits hold a value to
    2^-23, the sums' rounding is about that much again (1.2e-7 in all without the large values): bound 2.5e-7."""
    m, n, k = 40, 300, 2048
    buf = kq.gen_matrix(fmt, 670, n, k).reshape(n * k // 256, -1).copy()
    if fmt == "q4k":
        buf[:, [4, 8]] &= 0xC0                      # scale and minimum of sub-block 0: the low six bits
    elif fmt == "q5k":
        buf[:, 4] = 0                               # the first of the 12-bit fields
        buf[:, 5] &= 0xF0
    else:
        buf[:, 192] = 0
    buf = buf.reshape(-1)
    w = kq.dequant_matrix(fmt, buf, n, k)
    assert not np.any(w[:, ::256]) and np.any(w[:, 32::256])
    try:
        _tune("gemm_tall", 2)
        for power in (12, 20, 24):
            a = kq.gen_x(671, m, k)
            a[:, 3::256] = np.float32(2.0 ** power)
            assert kq.rel_l2(gpu_gemm(gpu, fmt, buf, a, m, n, k), kq.gemm_fp64(a, w)) <= 2.5e-7, power
    finally:
        _tune("gemm_tall", 0)


@pytest.mark.parametrize("fmt,m,n,k,many", [("q4k", 425, 1314, 2048, False), ("q6k", 95, 1200, 3072, False), ("q5k", 117, 1148, 2304, False),
                                            ("q6k", 330, 6093, 2560, False), ("q4k", 84, 4506, 7936, False), ("q6k", 330, 11008, 2560, True)])
def test_gemm_many_tokens_by_the_rule(gpu, fmt, m, n, k, many):
    """Where the kernel for many tokens is slower (16.5 us sixteen tokens at a time and 22.0 with it, 12.2 and 19.1, 11.2 and 16.9), the one that takes sixteen at
    a time has the product; where the estimates lie within a few percent of each other as well, though it is 6-12 % slower there (74.9 and 66.0,
    33.8 and 31.6); the last is the former's (138 and 103)."""
    buf, a = kq.gen_matrix(fmt, 694, n, k), kq.gen_x(695, m, k)
    bits = {}
    try:
        for tall in (0, 1, 2):
            _tune("gemm_tall", tall)
            bits[tall] = gpu_gemm(gpu, fmt, buf, a, m, n, k).view(np.uint32)
    finally:
        _tune("gemm_tall", 0)
    assert np.array_equal(bits[0], bits[2 if many else 1]) and not np.array_equal(bits[1], bits[2])


@pytest.mark.parametrize("m,n,k,parts", [(2, 1, 256, 1), (16, 67, 2048, 1), (17, 95, 2304, 1), (33, 193, 4352, 3), (48, 64, 8192, 32), (5, 130, 1280, 5)])
@pytest.mark.parametrize("rows", (1, 2, 3, 4))
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_slices_kernel(gpu, fmt, rows, m, n, k, parts):
    """The kernel that deals the super-blocks of its rows to its waves, forced, with every height of a workgroup: one row, one super-block
    (seven waves idle), eight, nine (a second round for one wave) and seventeen in three parts, thirty-two parts, rows that fill no tile and
    are no multiple of four, tokens that fill no tile: within tolerance, the same bits on every run, a token's values large or small
    against the others', an infinity in its own token only."""
    if rows == 4 and fmt != "q4k":
        pytest.skip("64 rows are Q4_K's")
    buf, a = kq.gen_matrix(fmt, 700 + m, n, k), kq.gen_x(710 + m, m, k)
    a[0] *= np.float32(1e6)
    a[m - 1] *= np.float32(1e-6)
    w = kq.dequant_matrix(fmt, buf, n, k)
    c64, terms = _c64(fmt, buf, a, n, k), np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T
    try:
        _tune("gemm_slices", 2)
        _tune("gemm_slices_rows", rows)
        _tune("gemm_k_parts", parts)
        c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert np.all(np.abs(c - c64) <= TOL * terms)      # as above: 1e-5 of the sum of the terms' sizes
        again = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert np.array_equal(again.view(np.uint32), c.view(np.uint32))
        a[1, 7] = np.inf
        c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
        assert not np.any(np.isfinite(c[1])) and np.array_equal(np.delete(c, 1, axis=0), np.delete(again, 1, axis=0))
    finally:
        for key in ("gemm_slices", "gemm_slices_rows", "gemm_k_parts"):
            _tune(key, 0)


@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_slices_no_less_exact_than_sixteen_at_a_time(gpu, fmt):
    """By the rule, 16 tokens: against fp64 at most 1.03 times the error of the kernel that takes sixteen tokens at a time (0.95-0.98 over
    drawn products; the ratio of two error norms over 65536 results is stable to about 2 %)."""
    n, k, m = 4096, 4096, 16
    buf, a = kq.gen_matrix(fmt, 720, n, k), kq.gen_x(721, m, k)
    c64, err = _c64(fmt, buf, a, n, k), {}
    try:
        for slices in (0, 1):
            _tune("gemm_slices", slices)
            err[slices] = kq.rel_l2(gpu_gemm(gpu, fmt, buf, a, m, n, k), c64)
    finally:
        _tune("gemm_slices", 0)
    assert err[0] != err[1] and err[0] <= 1.03 * err[1], err


@pytest.mark.parametrize("fmt,m,n,k", FROM_THE_ENGINE)
def test_gemm_slices_no_less_exact_than_the_engine(gpu, fmt, m, n, k):
    """Two to eight tokens whose activations the GEMV engine multiplies as f32 and this kernel as two f16 pieces: against fp64 the error is not larger
    (0.57-0.92 of the engine's over 150 drawn products; a ratio over 6900 results and more is stable to about 2 %)."""
    buf, a = kq.gen_matrix(fmt, 722, n, k), kq.gen_x(723, m, k)
    c64, err = _c64(fmt, buf, a, n, k), {}
    try:
        for slices in (0, 1):
            _tune("gemm_slices", slices)
            err[slices] = kq.rel_l2(gpu_gemm(gpu, fmt, buf, a, m, n, k), c64)
    finally:
        _tune("gemm_slices", 0)
    assert err[0] != err[1] and err[0] <= err[1], err


def test_gemm_slices_captured_on_a_new_stream_and_without_allocation(gpu):
    """Four tokens against 6000 x 4096, which the integer cores took without scratch memory: captured on a stream that has seen no product.
    16 tokens against 512 x 4096, parts of K: the same bits from trn_q4k_gemm_noalloc."""
    ctx, stream = gpu
    for m, n, k, whole in ((4, 6000, 4096, True), (16, 512, 4096, False)):
        buf, a = kq.gen_matrix("q4k", 730 + m, n, k), kq.gen_x(731, m, k)
        want = gpu_gemm(gpu, "q4k", buf, a, m, n, k).view(np.uint32)
        dw, da = t.GpuBuffer.from_host(ctx, buf), t.GpuBuffer.from_host(ctx, a)
        dc = t.GpuBuffer.from_host(ctx, np.full(m * n, np.nan, np.float32))
        if whole:
            new = t.CudaStream(ctx)
            graph = _Captured(new, lambda: t.QuantizeKernel.ggml(m, n, k).launch(new, da, dw, dc))
            for _ in range(3):
                dc.copy_from_host(np.full(m * n, np.nan, np.float32))
                graph.replay(new)
                new.synchronize()
                assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), want)
            graph.close()
        else:
            for _ in range(2):
                assert _ffi.lib().trn_q4k_gemm_noalloc(stream.raw(), da.as_ptr(), dw.as_ptr(), dc.as_ptr(), m, n, k) == 0
                stream.synchronize()
                assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), want)


@pytest.mark.parametrize("m,n,k", [(33, 1, 256), (64, 255, 512), (65, 257, 1280), (97, 700, 2304)])
@pytest.mark.parametrize("fmt", ("q4k", "q5k"))
def test_gemm_many_tokens_either_shape_of_a_workgroup(gpu, fmt, m, n, k):
    """256 rows x 32 tokens and 128 x 64: the same sums in the same order, so the same bits for the same parts of K."""
    buf, a = kq.gen_matrix(fmt, 740 + m, n, k), kq.gen_x(741, m, k)
    try:
        _tune("gemm_tall", 2)
        for parts in (1, 2):
            _tune("gemm_k_parts", parts)
            bits = []
            for strips in (1, 2):
                _tune("gemm_tall_strips", strips)
                bits.append(gpu_gemm(gpu, fmt, buf, a, m, n, k).view(np.uint32))
            assert np.array_equal(*bits)
    finally:
        for key in ("gemm_tall", "gemm_k_parts", "gemm_tall_strips"):
            _tune(key, 0)


@pytest.mark.parametrize("fmt,m,n,k,warm", [("q4k", 121, 4192, 4096, False), ("q4k", 121, 4192, 4096, True), ("q5k", 40, 2573, 5888, False),
                                            ("q5k", 40, 2573, 5888, True), ("q4k", 16, 512, 4096, False)])
def test_gemm_captured_products_in_parts_keep_to_themselves(gpu, fmt, m, n, k, warm):
    """Products with K in parts that the kernels for up to sixteen and 48 tokens take by the rule, captured on a stream that has seen no product, or
    (33 tokens and more) one that has: their counters and partial sums are the capture's own, so three replays at once with the same and other
    products on the stream they were captured on, and after that stream is gone and its memory with it, give the eager call's bits."""
    ctx, other = gpu
    kernel = {"q4k": t.QuantizeKernel.ggml, "q5k": t.Q5KKernel}[fmt](m, n, k)
    stream, buf, a = t.CudaStream(ctx), kq.gen_matrix(fmt, 750, n, k), kq.gen_x(751, m, k)
    want = gpu_gemm(gpu, fmt, buf, a, m, n, k).view(np.uint32)
    dw, da = t.GpuBuffer.from_host(ctx, buf), t.GpuBuffer.from_host(ctx, a)
    dc, de = (t.GpuBuffer.from_host(ctx, np.full(m * n, np.nan, np.float32)) for _ in range(2))
    if warm:
        kernel.launch(stream, da, dw, de)
        stream.synchronize()
    graph = _Captured(stream, lambda: kernel.launch(stream, da, dw, dc))

    def replay(beside):
        dc.copy_from_host(np.full(m * n, np.nan, np.float32))
        for _ in range(4):
            graph.replay(other)
            beside()
        other.synchronize()
        assert np.array_equal(dc.copy_to_host().reshape(m, n).view(np.uint32), want)

    for _ in range(3):
        replay(lambda: kernel.launch(stream, da, dw, de))
        stream.synchronize()
        assert np.array_equal(de.copy_to_host().reshape(m, n).view(np.uint32), want)
    stream.destroy()
    poison = [t.GpuBuffer.from_host(ctx, np.full(1 << 20, np.nan, np.float32)) for _ in range(8)]      # takes what was freed
    for _ in range(3):
        replay(lambda: None)
    assert all(np.all(np.isnan(p.copy_to_host())) for p in poison)
    graph.close()


@pytest.mark.parametrize("tall", (1, 2))
@pytest.mark.parametrize("fmt", MFMA_FORMATS)
def test_gemm_sums_beyond_the_largest_float_are_infinite(gpu, fmt, tall):
    """Token r is finite, of one sign with row r's first 256 weights and so large that their sum is twice the largest float (every other term is
    of ordinary size): plus or minus infinity in that place, through eight further super-blocks, and a number wherever the terms' sizes add up
    to one."""
    m, n, k = 40, 64, 2304
    buf, a = kq.gen_matrix(fmt, 760, n, k), kq.gen_x(761, m, k)
    w = kq.dequant_matrix(fmt, buf, n, k)
    sign = np.where(np.arange(m) % 2 == 0, 1.0, -1.0)
    a[:, :256] = sign[:, None] * np.sign(w[:m, :256]) * (6.8e38 / np.abs(w[:m, :256]).astype(np.float64).sum(1))[:, None]
    assert np.all(np.isfinite(a))
    try:
        _tune("gemm_tall", tall)
        c = gpu_gemm(gpu, fmt, buf, a, m, n, k)
    finally:
        _tune("gemm_tall", 0)
    assert np.array_equal(c[np.arange(m), np.arange(m)], sign * np.inf)
    small = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T < 3e38
    assert np.all(np.isfinite(c[small]))
