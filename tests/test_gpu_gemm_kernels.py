"""Every GEMM kernel variant against the oracle: the 128x128 kernel and the
direct-to-LDS kernels (256x256 with one wave per SIMD, 256x128 and 128x128 four-wave),
forced through `omx_set_option`, on
shapes with ragged M and N (rows past the edge are fetched from a clamped
address and must never be stored), every operand layout, split-K, bf16 and f32
outputs and accumulation."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    backend = MiBackend(0)
    yield backend
    backend._lib.omx_set_option(backend._ctx, b"gemm_dma", C.c_int64(1))
    backend.close()


SHAPES = [(256, 64, 256), (300, 128, 520), (64, 192, 96), (513, 256, 257), (1024, 768, 768), (264, 1024, 136),
          (4160, 136, 264),  # a weight gradient over 4160 rows, split along K
          (520, 256, 400), (256, 1280, 192), (768, 384, 576)]  # one-wave tiles: ragged both ways, one exact 256 x 192 tile, six steps


@pytest.mark.parametrize("mode", [0, 1, 3, 4, 9, 10])
@pytest.mark.parametrize("rows,kin,nout", SHAPES)
def test_linear_bf16_under_each_kernel(be, mode, rows, kin, nout):
    from ojas_amd.backend import BF16, F32

    print(f"gemm mode {mode} {rows}x{kin}x{nout}", flush=True)
    assert be._lib.omx_set_option(be._ctx, b"gemm_dma", C.c_int64(mode)) == 0
    r = orc.SplitMix64(5000 + rows + mode)
    x = orc.round_bf16(r.vec(rows * kin, 0.5)).reshape(rows, kin)
    w = orc.round_bf16(r.vec(nout * kin, 0.5)).reshape(nout, kin)
    gy = orc.round_bf16(r.vec(rows * nout, 0.5)).reshape(rows, nout)
    orc.set_threads(8)
    oy = orc.linear_forward(x, w)
    ogx, ogw = orc.linear_backward(x, w, gy)
    dx, dw, dgy = be.upload(x, BF16), be.upload(w, BF16), be.upload(gy, BF16)

    def close(got, want, tol, what):
        err = float(np.max(np.abs(np.asarray(got, np.float64) - want)))
        assert err <= tol * max(1.0, float(np.max(np.abs(want)))), (what, err)

    close(be.download(be.linear_forward(dx, dw)), oy, 1e-5, "fwd f32 out")
    close(be.download_f32(be.linear_forward(dx, dw, out_dtype=BF16)), oy, 2e-2, "fwd bf16 out")
    gx, gw = be.linear_backward(dx, dw, dgy, gx_dtype=F32)
    close(be.download(gx), ogx, 1e-5, "gx")
    close(be.download(gw), ogw, 1e-5, "gw")
    # Accumulation into an f32 output continues the stored values.
    c0 = r.vec(rows * nout, 0.5).reshape(rows, nout)
    dc = be.upload(c0)
    be.gemm(dx, (kin, 1), dw, (1, kin), rows, kin, nout, c=dc)
    close(be.download(dc), oy.astype(np.float64) + c0, 1e-5, "accumulate")


@pytest.mark.parametrize("layout,m,k,n", [
    ("NN", 8192, 1024, 3072), ("NN", 8192, 8192, 2048), ("NN", 8192, 4096, 4096), ("NN", 4096, 768, 32000),
    ("NT", 8192, 8192, 2048), ("NT", 8192, 3072, 1024), ("NT", 8192, 16384, 4096), ("NT", 8192, 3072, 768),
    ("NT", 16384, 3072, 1536),
    ("TT", 4096, 8192, 1024), ("TT", 4096, 8192, 4096), ("TT", 1024, 8192, 1024), ("TT", 6144, 8192, 2048)])
def test_the_dispatcher_picks_a_tiling_within_a_tenth_of_the_best(be, layout, m, k, n):
    """Shapes of other models (d = 1024 / 2048 / 4096, 8192 tokens): the tiling the shape rule
    picks (`gemm_dma` 1) against every tiling forced in turn. The rule speaks of tiles per compute
    unit and K steps per tile; this holds it to within 10 % of the fastest one on shapes it was not
    tuned on. Timed as the best of three runs of ten launches each."""
    import time

    from ojas_amd.backend import BF16, F32

    print(f"gemm tiling choice {layout} {m}x{k}x{n}", flush=True)
    a = be.empty((m * k,), BF16)
    b = be.empty((k * n,), BF16)
    for t, seed in ((a, 1), (b, 2)):
        be._check(be._lib.omx_init_normal(be._ctx, be._p(t), C.c_int32(BF16), C.c_uint64(t.numel), C.c_uint64(seed),
                                          C.c_float(0.05)))
    out_dtype = F32 if layout == "TT" else BF16
    c = be.empty((m, n), out_dtype)
    a_strides = (1, m) if layout == "TT" else (k, 1)   # k-major A: element (i, p) at p * m + i
    b_strides = (1, k) if layout == "NN" else (n, 1)   # k-contiguous B: element (p, j) at j * k + p

    def launch():
        be._check(be._lib.omx_gemm(be._ctx, be._p(a), C.c_uint64(a_strides[0]), C.c_uint64(a_strides[1]), be._p(b),
                                   C.c_uint64(b_strides[0]), C.c_uint64(b_strides[1]), C.c_int32(BF16), be._p(c),
                                   C.c_int32(out_dtype), C.c_uint64(m), C.c_uint64(k), C.c_uint64(n), C.c_int32(0)))

    def seconds(mode):
        assert be._lib.omx_set_option(be._ctx, b"gemm_dma", C.c_int64(mode)) == 0
        best = float("inf")
        for _ in range(3):
            launch()
            be.sync()
            start = time.perf_counter()
            for _ in range(10):
                launch()
            be.sync()
            best = min(best, (time.perf_counter() - start) / 10)
        return best

    try:
        forced = {mode: seconds(mode) for mode in (3, 4, 9, 10)}
        chosen = seconds(1)
    finally:
        be.set_option("gemm_dma", 1)
    fastest = min(forced.values())
    print("  us: chosen %.1f, forced %s" % (chosen * 1e6, {mode: round(t * 1e6, 1) for mode, t in forced.items()}), flush=True)
    assert chosen <= 1.10 * fastest, (chosen, forced)


@pytest.mark.parametrize("m,tokens,n", [(768, 4096, 768), (1024, 8192, 1024), (512, 16384, 512), (1024, 16384, 1024),
                                        (2048, 16384, 512), (2048, 16384, 1024)])
def test_long_weight_gradients_take_a_tiling_within_a_tenth_of_the_best(be, m, tokens, n):
    """Weight gradients of one to four 128 x 128 tiles per eight compute units, where the tiling, its split and what shares
    a unit weigh against each other: the choice against the tilings below 256 x 256 forced in turn, the small ones unsplit.
    The kernels' own time, as the best of three runs of ten launches each."""
    from ojas_amd.backend import BF16

    print(f"gemm tiling choice, weight gradient {m}x{n} over {tokens}", flush=True)
    a, b, c = be.empty((tokens * m,), BF16), be.empty((tokens * n,), BF16), be.empty((m, n))
    for t, seed in ((a, 1), (b, 2)):
        be._check(be._lib.omx_init_normal(be._ctx, be._p(t), C.c_int32(BF16), C.c_uint64(t.numel), C.c_uint64(seed),
                                          C.c_float(0.05)))

    def us(mode):
        be.set_option("gemm_dma", mode)
        best = float("inf")
        for _ in range(3):
            be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(1)))
            for _ in range(10):
                be._check(be._lib.omx_gemm(be._ctx, be._p(a), C.c_uint64(1), C.c_uint64(m), be._p(b), C.c_uint64(n), C.c_uint64(1),
                                           C.c_int32(BF16), be._p(c), C.c_int32(0), C.c_uint64(m), C.c_uint64(tokens), C.c_uint64(n),
                                           C.c_int32(0)))
            ms = C.c_double()
            be._check(be._lib.omx_profile_gemm_report(be._ctx, None, C.byref(ms), None))
            be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
            best = min(best, ms.value * 100)
        return best

    try:
        us(1)  # clocks up
        forced = {mode: us(mode) for mode in (3, 4, 7, 8)}
        chosen = us(1)
    finally:
        be.set_option("gemm_dma", 1)
    print("  us: chosen %.1f, forced %s" % (chosen, {mode: round(t, 1) for mode, t in forced.items()}), flush=True)
    assert chosen <= 1.10 * min(forced.values()), (chosen, forced)


def test_tiles_that_do_not_divide_by_the_xcds_run_as_those_that_do(be):
    """684 rows by 5504 columns over 2048 are 11 x 86 tiles of 64 x 64, two more than a multiple of 8; 5632 columns are 11 x 88.
    An XCD takes a contiguous eighth of either, so the smaller product takes no longer (1.15 for the spread of two short
    runs; in index order 47.8 against some 25 us), and the choice for it is within a tenth of the tilings forced."""
    from ojas_amd.backend import BF16

    m, k = 684, 2048
    print("gemm tile order 684 x 2048 x 5504 / 5632", flush=True)
    a, b, c = be.empty((m * k,), BF16), be.empty((k * 5632,), BF16), be.empty((m * 5632,), BF16)
    for t, seed in ((a, 1), (b, 2)):
        be._check(be._lib.omx_init_normal(be._ctx, be._p(t), C.c_int32(BF16), C.c_uint64(t.numel), C.c_uint64(seed),
                                          C.c_float(0.05)))

    def us(mode, n):
        be.set_option("gemm_dma", mode)
        best = float("inf")
        for _ in range(3):
            be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(1)))
            for _ in range(10):
                be._check(be._lib.omx_gemm(be._ctx, be._p(a), C.c_uint64(k), C.c_uint64(1), be._p(b), C.c_uint64(1), C.c_uint64(k),
                                           C.c_int32(BF16), be._p(c), C.c_int32(BF16), C.c_uint64(m), C.c_uint64(k), C.c_uint64(n),
                                           C.c_int32(0)))
            ms = C.c_double()
            be._check(be._lib.omx_profile_gemm_report(be._ctx, None, C.byref(ms), None))
            be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
            best = min(best, ms.value * 100)
        return best

    try:
        us(1, 5504)  # clocks up
        even, odd = us(8, 5632), us(8, 5504)
        forced = {mode: us(mode, 5504) for mode in (3, 4, 7, 8)}
        chosen = us(1, 5504)
    finally:
        be.set_option("gemm_dma", 1)
    print("  us: 5632 columns %.1f, 5504 %.1f; chosen %.1f, forced %s" % (even, odd, chosen, forced), flush=True)
    assert odd <= 1.15 * even, (odd, even)
    assert chosen <= 1.10 * min(forced.values()), (chosen, forced)


def test_a_mostly_empty_last_round_is_cut_by_rows(be):
    """65 x 16 tiles of 256 x 256 are four rounds of the 256 compute units and 16 tiles more: the
    first 64 tile rows keep the tiling, the last goes to a launch of its own. Checked against the
    oracle (ragged M and N), and the rows of the first launch against the uncut product bit for bit."""
    from ojas_amd.backend import BF16

    m, k, n = 16616, 128, 4088
    print(f"gemm row split NT {m}x{k}x{n}", flush=True)
    r = orc.SplitMix64(77)
    a = orc.round_bf16(r.vec(m * k, 0.5)).reshape(m, k)
    b = orc.round_bf16(r.vec(k * n, 0.5)).reshape(k, n)
    orc.set_threads(8)
    want = orc.linear_forward(a, np.ascontiguousarray(b.T))
    da, db = be.upload(a, BF16), be.upload(b, BF16)
    be.set_option("gemm_dma", 1)
    try:
        cut = be.download(be.gemm(da, (k, 1), db, (n, 1), m, k, n))
        be.set_option("gemm_row_split", 0)
        whole = be.download(be.gemm(da, (k, 1), db, (n, 1), m, k, n))
    finally:
        be.set_option("gemm_row_split", 1)
    scale = max(1.0, float(np.max(np.abs(want))))
    assert float(np.max(np.abs(cut.astype(np.float64) - want))) <= 1e-5 * scale
    assert float(np.max(np.abs(whole.astype(np.float64) - want))) <= 1e-5 * scale
    assert np.array_equal(cut[:64 * 256], whole[:64 * 256])


def test_a_cut_weight_gradient_matches_the_uncut_one(be):
    """Both operands k-major over 4096 rows (a head's weight gradient in small): 86 x 3 tiles are one
    round and two tiles; the cut product accumulates into C like the uncut one."""
    from ojas_amd.backend import BF16, F32

    m, k, n = 22016, 4096, 768
    print(f"gemm row split TT {m}x{k}x{n}", flush=True)
    a = be.empty((k * m,), BF16)
    b = be.empty((k * n,), BF16)
    for t, seed in ((a, 3), (b, 4)):
        be._check(be._lib.omx_init_normal(be._ctx, be._p(t), C.c_int32(BF16), C.c_uint64(t.numel), C.c_uint64(seed),
                                          C.c_float(0.05)))
    c0 = np.full((m, n), 0.25, np.float32)
    be.set_option("gemm_dma", 1)
    try:
        cut = be.upload(c0)
        be.gemm(a, (1, m), b, (n, 1), m, k, n, c=cut)
        be.set_option("gemm_row_split", 0)
        whole = be.upload(c0)
        be.gemm(a, (1, m), b, (n, 1), m, k, n, c=whole)
    finally:
        be.set_option("gemm_row_split", 1)
    got, ref = be.download(cut), be.download(whole)
    assert np.array_equal(got[:85 * 256], ref[:85 * 256])
    # The last 256 rows take another tiling and split K: the same sums in another order.
    assert float(np.max(np.abs(got[85 * 256:] - ref[85 * 256:]))) <= 1e-5 * max(1.0, float(np.max(np.abs(ref))))
    assert float(np.max(np.abs(ref - 0.25))) > 0.1


@pytest.mark.parametrize("tiling", [9, 10])
@pytest.mark.parametrize("layout", ["NN", "NT", "TT"])
def test_one_wave_kernel_with_split_reduction_matches_the_register_staged_kernel(be, layout, tiling):
    """72 tiles of 256 x 256 (96 of 256 x 192) over K = 8192: the one-wave kernel splits K to fill the
    chip (partial sums, then the reduce pass). Against the 128 x 128 register-staged kernel, which the
    other tests hold to the oracle, on the same operands; f32 and bf16 outputs, and accumulation."""
    from ojas_amd.backend import BF16, F32

    m, k, n = 2048, 8192, 2304
    print(f"gemm one-wave split-K {layout} tiling {tiling} {m}x{k}x{n}", flush=True)
    a = be.empty((m * k,), BF16)
    b = be.empty((k * n,), BF16)
    for t, seed in ((a, 11), (b, 12)):
        be._check(be._lib.omx_init_normal(be._ctx, be._p(t), C.c_int32(BF16), C.c_uint64(t.numel), C.c_uint64(seed),
                                          C.c_float(0.05)))
    a_strides = (1, m) if layout == "TT" else (k, 1)
    b_strides = (1, k) if layout == "NN" else (n, 1)
    c0 = np.full((m, n), -0.5, np.float32)
    got = {}
    try:
        for mode in (tiling, 0):
            be.set_option("gemm_dma", mode)
            acc = be.upload(c0)
            be.gemm(a, a_strides, b, b_strides, m, k, n, c=acc)
            got[mode] = (be.download(be.gemm(a, a_strides, b, b_strides, m, k, n)),
                         be.download_f32(be.gemm(a, a_strides, b, b_strides, m, k, n, out_dtype=BF16)), be.download(acc))
    finally:
        be.set_option("gemm_dma", 1)
    scale = float(np.max(np.abs(got[0][0])))
    assert scale > 1.0
    assert float(np.max(np.abs(got[tiling][0] - got[0][0]))) <= 1e-5 * scale
    assert float(np.max(np.abs(got[tiling][1] - got[0][1]))) <= 8e-3 * scale  # one bf16 step
    assert float(np.max(np.abs(got[tiling][2] - got[0][2]))) <= 1e-5 * scale
    assert float(np.max(np.abs(got[0][2] - got[0][0] + 0.5))) <= 1e-5 * scale


def test_unknown_option_is_refused(be):
    assert be._lib.omx_set_option(be._ctx, b"no_such_knob", C.c_int64(1)) == 11
    assert be._lib.omx_set_option(be._ctx, b"gemm_dma", C.c_int64(5)) == 3


@pytest.mark.parametrize("mode", [0, 1, 3, 4, 9, 10])
@pytest.mark.parametrize("layers", [3, 4])  # tile counts that divide by the 8 XCDs evenly (4) and that do not (3)
@pytest.mark.parametrize("rows,kin,nout", [(1088, 136, 264), (2048, 768, 256), (2048, 200, 328)])
def test_strided_batch_of_weight_gradients(be, mode, rows, kin, nout, layers):
    """`omx_gemm_strided_batch` as the step driver uses it: gw[l] = gy[l]^T x[l] for three stacked
    layers in one launch, outputs at a padded stride; each equals the oracle's `linear_backward`
    weight gradient."""
    from ojas_amd.backend import BF16, F32

    print(f"gemm strided batch mode {mode} {rows}x{kin}x{nout} layers {layers}", flush=True)
    assert be._lib.omx_set_option(be._ctx, b"gemm_dma", C.c_int64(mode)) == 0
    pad = 64
    r = orc.SplitMix64(7100 + rows + mode + layers)
    x = orc.round_bf16(r.vec(layers * rows * kin, 0.5)).reshape(layers, rows, kin)
    gy = orc.round_bf16(r.vec(layers * rows * nout, 0.5)).reshape(layers, rows, nout)
    w = np.zeros((nout, kin), np.float32)
    orc.set_threads(8)
    stride_c = nout * kin + pad
    out = be.gemm_strided_batch(be.upload(gy, BF16), (1, nout), be.upload(x, BF16), (kin, 1), nout, rows, kin, layers,
                                (rows * nout, rows * kin, stride_c))
    got = be.download(out)
    for l in range(layers):
        _, ogw = orc.linear_backward(x[l], w, gy[l])
        mine = got[l * stride_c:l * stride_c + nout * kin].reshape(nout, kin).astype(np.float64)
        err = float(np.max(np.abs(mine - ogw)))
        assert err <= 1e-5 * max(1.0, float(np.max(np.abs(ogw)))), (l, err)


@pytest.mark.parametrize("mode", [1, 3, 4, 9, 10])
@pytest.mark.parametrize("tokens,m,n,pitch", [(65, 264, 256, 264), (127, 257, 192, 264), (191, 250, 384, 256), (1, 256, 256, 256),
                                              (3500, 512, 768, 512), (4161, 1000, 1152, 1000), (6300, 2048, 2304, 2048)])
def test_reductions_of_any_length_end_inside_a_step(be, mode, tokens, m, n, pitch):
    """Weight gradients over a number of tokens that no K step divides: the rows behind the last token (NaN here) are
    never multiplied, nor are the columns between a row's end and its pitch."""
    from ojas_amd.backend import BF16

    print(f"gemm ragged K mode {mode} {m}x{n} over {tokens}", flush=True)
    be.set_option("gemm_dma", mode)
    rng = np.random.default_rng(tokens + mode)
    gy = np.full((tokens + 256, pitch), np.nan, np.float32)
    x = np.full((tokens + 256, n), np.nan, np.float32)
    gy[:tokens, :m] = orc.round_bf16((rng.standard_normal((tokens, m)) * 0.5).astype(np.float32).ravel()).reshape(tokens, m)
    x[:tokens] = orc.round_bf16((rng.standard_normal((tokens, n)) * 0.5).astype(np.float32).ravel()).reshape(tokens, n)
    want = gy[:tokens, :m].T @ x[:tokens]
    got = be.download(be.gemm(be.upload(gy, BF16), (1, pitch), be.upload(x, BF16), (n, 1), m, tokens, n))
    be.set_option("gemm_dma", 1)
    assert float(np.max(np.abs(got - want))) <= 2e-5 * max(1.0, float(np.max(np.abs(want))))


@pytest.mark.parametrize("mode", [7, 8])
@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,k,n", [(64, 64, 64), (1, 128, 1), (65, 192, 63), (130, 256, 200), (333, 2048, 72)])
def test_small_direct_to_lds_tiles(be, mode, layout, m, k, n):
    """The 128 x 64 and 64 x 64 tiles: one tile, one row and column, a row and a column past a tile, fewer K steps than
    stages; f32, bf16 and accumulated outputs, and a batch. Against the f64 product of the same bf16 operands: every
    product is exact in f32, so what is left is f32 sums (1e-5 of the largest value) or one bf16 rounding (2^-8)."""
    from ojas_amd.backend import BF16

    print(f"gemm small tiles mode {mode} {layout} {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(m * k + n)
    lda, ldb = (m + 7) // 8 * 8, (n + 7) // 8 * 8
    ta, tb = layout[0] == "T", layout[1] == "T"
    a = orc.round_bf16((rng.standard_normal((2, k, lda) if ta else (2, m, k)) * 0.5).astype(np.float32).ravel()).reshape((2, k, lda) if ta else (2, m, k))
    b = orc.round_bf16((rng.standard_normal((2, k, ldb) if tb else (2, n, k)) * 0.5).astype(np.float32).ravel()).reshape((2, k, ldb) if tb else (2, n, k))
    fa = a.astype(np.float64)[:, :, :m].transpose(0, 2, 1) if ta else a.astype(np.float64)
    fb = b.astype(np.float64)[:, :, :n] if tb else b.astype(np.float64).transpose(0, 2, 1)
    want = fa @ fb
    sa, sb = ((1, lda) if ta else (k, 1)), ((ldb, 1) if tb else (1, k))
    c0 = rng.standard_normal((m, n)).astype(np.float32)
    da, db, dc = be.upload(a, BF16), be.upload(b, BF16), be.upload(c0)
    pad = (m * n + 3) // 4 * 4
    be.set_option("gemm_dma", mode)
    try:
        plain = be.download(be.gemm(da, sa, db, sb, m, k, n))
        short = be.download_f32(be.gemm(da, sa, db, sb, m, k, n, out_dtype=BF16))
        be.gemm(da, sa, db, sb, m, k, n, c=dc)
        both = be.download(be.gemm_strided_batch(da, sa, db, sb, m, k, n, 2, (a[0].size, b[0].size, pad)))
    finally:
        be.set_option("gemm_dma", 1)
    top = max(1.0, float(np.max(np.abs(want))))
    assert float(np.max(np.abs(plain - want[0]))) <= 1e-5 * top
    assert float(np.max(np.abs(short - want[0]))) <= 2.0 ** -8 * top
    assert float(np.max(np.abs(be.download(dc) - c0 - want[0]))) <= 1e-5 * top
    for j in range(2):
        assert float(np.max(np.abs(both[j * pad:j * pad + m * n].reshape(m, n) - want[j]))) <= 1e-5 * top


@pytest.mark.parametrize("mode", [7, 8])
@pytest.mark.parametrize("rows,kin,nout", [(64, 64, 64), (70, 192, 100), (300, 512, 520)])
def test_small_direct_to_lds_tiles_with_gelu(be, mode, rows, kin, nout):
    """The activation's store pass on the small tiles gives the bits of the 256 x 128 tiles' (one K order in both)."""
    from ojas_amd.backend import BF16

    rng = np.random.default_rng(rows)
    x = be.upload(orc.round_bf16((rng.standard_normal(rows * kin) * 0.5).astype(np.float32)).reshape(rows, kin), BF16)
    w = be.upload(orc.round_bf16((rng.standard_normal(nout * kin) * 0.2).astype(np.float32)).reshape(nout, kin), BF16)
    got = {}
    for m in (3, mode):
        be.set_option("gemm_dma", m)
        got[m] = [be.download(t) for t in be.linear_gelu_forward(x, w)]
    be.set_option("gemm_dma", 1)
    for mine, theirs in zip(got[mode], got[3]):
        assert np.array_equal(mine, theirs)


@pytest.mark.parametrize("mode", [7, 8])
@pytest.mark.parametrize("tokens,m,n,pitch", [(1, 64, 64, 64), (65, 72, 64, 72), (127, 57, 192, 64), (3500, 512, 512, 512)])
def test_small_tiles_end_a_reduction_inside_a_step(be, mode, tokens, m, n, pitch):
    test_reductions_of_any_length_end_inside_a_step(be, mode, tokens, m, n, pitch)


# More than one workgroup per compute unit of 256, where the small tiles keep three stages instead of five or six: 17 x 18 tiles
# of 128 x 64, 33 x 18 of 64 x 64.
@pytest.mark.parametrize("mode", [7, 8])
@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,k,n", [(2100, 64, 1100), (2100, 640, 1100)])
def test_small_tiles_that_share_a_compute_unit(be, mode, layout, m, k, n):
    test_small_direct_to_lds_tiles(be, mode, layout, m, k, n)


@pytest.mark.parametrize("mode", [7, 8])
def test_small_tiles_that_share_a_compute_unit_with_gelu(be, mode):
    test_small_direct_to_lds_tiles_with_gelu(be, mode, 2100, 320, 1100)


@pytest.mark.parametrize("mode", [7, 8])
def test_small_tiles_that_share_a_compute_unit_end_a_reduction_inside_a_step(be, mode):
    test_reductions_of_any_length_end_inside_a_step(be, mode, 333, 2100, 1104, 2104)


@pytest.mark.parametrize("rows,kin,nout,layers", [(4096, 16, 512, 6), (4096, 384, 48, 5), (2048, 8, 256, 16)])
def test_strided_batch_of_thin_weight_gradients_splits_the_reduction(be, rows, kin, nout, layers):
    """A batch of thin outputs over a long reduction (an adapter's rank x d gradients over the
    tokens of every layer): too few tiles to fill the chip, so each product's reduction is split
    and the partial sums of every product are added by one reduce launch. Outputs at a padded
    stride, untouched between them."""
    from ojas_amd.backend import BF16

    print(f"gemm strided batch thin {rows}x{kin}x{nout} layers {layers}", flush=True)
    be.set_option("gemm_dma", 1)
    pad = 32
    r = orc.SplitMix64(7300 + rows + kin + layers)
    x = orc.round_bf16(r.vec(layers * rows * kin, 0.5)).reshape(layers, rows, kin)
    gy = orc.round_bf16(r.vec(layers * rows * nout, 0.5)).reshape(layers, rows, nout)
    stride_c = nout * kin + pad
    out = be.gemm_strided_batch(be.upload(gy, BF16), (1, nout), be.upload(x, BF16), (kin, 1), nout, rows, kin, layers,
                                (rows * nout, rows * kin, stride_c))
    got = be.download(out)
    for l in range(layers):
        want = gy[l].astype(np.float64).T @ x[l].astype(np.float64)
        mine = got[l * stride_c:l * stride_c + nout * kin].reshape(nout, kin).astype(np.float64)
        err = float(np.max(np.abs(mine - want)))
        assert err <= 1e-5 * max(1.0, float(np.max(np.abs(want)))), (l, err)


@pytest.mark.parametrize("rows,d,r", [(2048, 256, 16), (8192, 2048, 16), (300, 128, 8)])
def test_pitched_strided_batch_writes_adjacent_column_blocks(be, rows, d, r):
    """Three thin products in one launch (an adapter's gh = gy B for the q, k and v sites): operand i
    is column block i of a [rows, 3 d] tensor, its B the i-th of three adjacent [d, r] matrices, its
    output column block i of a [rows, 4 r] tensor whose fourth block keeps what it held. The bits
    are those of three `gemm_pitched` calls."""
    import ctypes as C

    from ojas_amd.backend import BF16

    print(f"gemm pitched strided batch {rows} {d} {r}", flush=True)
    be.set_option("gemm_dma", 1)
    rng = orc.SplitMix64(8800 + rows + d)
    gy = orc.round_bf16(rng.vec(rows * 3 * d, 0.5)).reshape(rows, 3 * d)
    bm = orc.round_bf16(rng.vec(3 * d * r, 0.5)).reshape(3, d, r)
    held = orc.round_bf16(rng.vec(rows * 4 * r, 1.0)).reshape(rows, 4 * r)
    dgy, dbm = be.upload(gy, BF16), be.upload(bm, BF16)
    out = be.upload(held, BF16)
    be.gemm_pitched_strided_batch(dgy, (3 * d, 1), dbm, (r, 1), out, 4 * r, rows, d, r, 3, (d, d * r, r))
    got = be.download_f32(out).reshape(rows, 4 * r)
    assert np.array_equal(got[:, 3 * r:], held[:, 3 * r:])
    for j in range(3):
        want = gy[:, j * d:(j + 1) * d].astype(np.float64) @ bm[j].astype(np.float64)
        err = float(np.max(np.abs(got[:, j * r:(j + 1) * r] - want)))
        assert err <= 2e-2 * max(1.0, float(np.max(np.abs(want)))), (j, err)
    one = be.upload(held, BF16)
    for j in range(3):
        assert be._lib.omx_gemm_pitched(
            be._ctx, C.c_void_p(dgy.ptr + j * d * 2), C.c_uint64(3 * d), C.c_uint64(1), C.c_void_p(dbm.ptr + j * d * r * 2),
            C.c_uint64(r), C.c_uint64(1), C.c_int32(BF16), C.c_void_p(one.ptr + j * r * 2), C.c_int32(BF16),
            C.c_uint64(4 * r), C.c_uint64(rows), C.c_uint64(d), C.c_uint64(r), C.c_int32(0)) == 0
    assert np.array_equal(be.download(one), be.download(out))


@pytest.mark.parametrize("rows,k,n,b_km,f32_out", [
    (8192, 2048, 16, False, False), (8192, 2048, 48, False, False), (8192, 2048, 16, True, False),
    (16384, 768, 12, False, True), (1030, 128, 64, True, False), (4096, 384, 5, False, False), (2048, 256, 33, True, True)])
def test_thin_outputs_take_one_pass_over_a(be, rows, k, n, b_km, f32_out):
    """Outputs of at most 64 columns over many rows (an adapter's h = x A^T and gh = gy B, a gate's
    logits) take `gemm_thin_kernel`; held to the f64 product at the bf16-storage tolerance (1e-5 for an
    f32 output: bf16 products are exact and both sums are f32) and to the tiled kernels' result, with
    ragged rows and column counts that are not multiples of 16 or 4, into a pitched output whose
    other columns keep their values."""
    import ctypes as C

    from ojas_amd.backend import BF16, F32

    print(f"gemm thin {rows}x{k}x{n} b_km={b_km} f32_out={f32_out}", flush=True)
    be.set_option("gemm_dma", 1)
    rng = orc.SplitMix64(9900 + rows + k + n)
    a = orc.round_bf16(rng.vec(rows * k, 0.5)).reshape(rows, k)
    b = orc.round_bf16(rng.vec(k * n, 0.5)).reshape(k, n)  # B[k, n]
    ldc = n + 8
    held = orc.round_bf16(rng.vec(rows * ldc, 1.0)).reshape(rows, ldc)
    da = be.upload(a, BF16)
    db = be.upload(b if b_km else np.ascontiguousarray(b.T), BF16)
    b_rs, b_cs = (n, 1) if b_km else (1, k)
    od = F32 if f32_out else BF16
    outs = []
    for thin in (1, 0):
        be.set_option("gemm_thin", thin)
        out = be.upload(held, od)
        assert be._lib.omx_gemm_pitched(
            be._ctx, C.c_void_p(da.ptr), C.c_uint64(k), C.c_uint64(1), C.c_void_p(db.ptr), C.c_uint64(b_rs),
            C.c_uint64(b_cs), C.c_int32(BF16), C.c_void_p(out.ptr), C.c_int32(od), C.c_uint64(ldc), C.c_uint64(rows),
            C.c_uint64(k), C.c_uint64(n), C.c_int32(0)) == 0
        outs.append(be.download_f32(out).reshape(rows, ldc))
    be.set_option("gemm_thin", 1)
    want = a.astype(np.float64) @ b.astype(np.float64)
    scale = max(1.0, float(np.max(np.abs(want))))
    for got in outs:
        assert np.array_equal(got[:, n:], held[:, n:])
        assert float(np.max(np.abs(got[:, :n] - want))) <= (1e-5 if f32_out else 2e-2) * scale
    assert float(np.max(np.abs(outs[0][:, :n] - outs[1][:, :n]))) <= (2e-6 if f32_out else 8e-3) * scale


def test_strided_batch_refuses_bad_strides(be):
    from ojas_amd.backend import BF16, OjasError

    a, b = be.zeros((2, 64, 64), BF16), be.zeros((2, 64, 64), BF16)
    with pytest.raises(OjasError):  # a batch stride that is not a multiple of 16 bytes
        be.gemm_strided_batch(a, (1, 64), b, (64, 1), 64, 64, 64, 2, (64 * 64 + 2, 64 * 64, 64 * 64))
    with pytest.raises(OjasError):  # overlapping outputs
        be.gemm_strided_batch(a, (1, 64), b, (64, 1), 64, 64, 64, 2, (64 * 64, 64 * 64, 64))


@pytest.mark.parametrize("rows,k,n", [(1, 32, 1), (1, 768, 770), (3, 96, 17), (16, 2048, 33), (17, 320, 64), (31, 64, 5001),
                                      (32, 1312, 31), (65, 256, 300), (200, 768, 768), (1000, 224, 900)])
def test_few_rows_share_k_between_waves(be, rows, k, n):
    """gemm_skinny_kernel: every tile of its rule, rows and columns off the 16-block grid, steps that its eight
    waves share unevenly or not at all; f32 and bf16 outputs, accumulation, the activation's store pass."""
    from ojas_amd.backend import BF16

    print(f"skinny {rows}x{k}x{n}", flush=True)
    be.set_option("gemm_dma", 1)
    r = orc.SplitMix64(9100 + rows + n)
    x = orc.round_bf16(r.vec(rows * k, 0.5)).reshape(rows, k)
    w = orc.round_bf16(r.vec(n * k, 0.5)).reshape(n, k)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    scale = max(1.0, float(np.abs(want).max()))
    dx, dw = be.upload(x, BF16), be.upload(w, BF16)
    assert np.abs(be.download(be.linear_forward(dx, dw)) - want).max() <= 1e-5 * scale
    assert np.abs(be.download_f32(be.linear_forward(dx, dw, out_dtype=BF16)) - want).max() <= 5e-3 * scale
    c0 = r.vec(rows * n, 0.5).reshape(rows, n)
    dc = be.upload(c0)
    be.gemm(dx, (k, 1), dw, (1, k), rows, k, n, c=dc)
    assert np.abs(be.download(dc) - (want + c0)).max() <= 1e-5 * scale
    u, act = be.linear_gelu_forward(dx, dw)
    hu = be.download_f32(u)
    assert np.abs(hu - want).max() <= 5e-3 * scale
    ref = orc.gelu_erf_forward(hu.reshape(-1)).reshape(rows, n)
    assert np.abs(be.download_f32(act) - ref).max() <= 1e-2 * max(1.0, float(np.abs(ref).max()))


@pytest.mark.parametrize("rows,k,n", [(1, 128, 1), (4, 128, 4), (2, 768, 1023), (4, 1024, 1024), (3, 1152, 5), (1, 3072, 768), (4, 8192, 77),
                                      (2, 256, 1025), (5, 3072, 768)])
def test_few_rows_in_quarters_of_k(be, rows, k, n):
    """gemm_rows4_kernel (up to four rows, 1024 columns) at its edges: as above."""
    test_few_rows_share_k_between_waves(be, rows, k, n)


@pytest.mark.parametrize("rows,k,n", [(16, 16, 16), (16, 4, 16), (48, 20, 32), (100, 260, 36), (256, 256, 256), (130, 8, 62), (704, 256, 704),
                                      (1030, 72, 260), (52, 3000, 44), (2048, 256, 256), (31, 64, 29)])
def test_small_f32_outputs_share_k_between_waves(be, rows, k, n):
    """gemm_frag32_kernel: the tiles of its rule in all operand layouts, rows and columns off the tile, K off the
    16-column step (and shorter than one), more waves than steps, accumulation and a strided batch."""
    print(f"frag32 {rows}x{k}x{n}", flush=True)
    be.set_option("gemm_dma", 1)
    r = orc.SplitMix64(7700 + rows + n)
    a, b, c0 = (r.vec(x * y, 0.5).reshape(x, y) for x, y in ((rows, k), (k, n), (rows, n)))
    want = a.astype(np.float64) @ b.astype(np.float64)
    tol = 1e-5 * max(1.0, float(np.abs(want).max()))
    da, dat, db, dbt = (be.upload(np.ascontiguousarray(x)) for x in (a, a.T, b, b.T))
    for x, xs in ((da, (k, 1)), (dat, (1, rows))):
        for y, ys in ((db, (n, 1)), (dbt, (1, k))):
            got = be.download(be.gemm(x, xs, y, ys, rows, k, n))
            assert np.abs(got - want).max() <= tol, (xs, ys)
            c = be.upload(c0)
            be.gemm(x, xs, y, ys, rows, k, n, c=c)
            assert np.abs(be.download(c) - (want + c0)).max() <= tol, (xs, ys)
    if rows * k % 4 == 0 and k * n % 4 == 0 and rows * n % 4 == 0:
        many = be.gemm_strided_batch(be.upload(np.stack([a, -a, 2 * a])), (k, 1), be.upload(np.stack([b, b, b])), (n, 1), rows, k, n, 3,
                                     (rows * k, k * n, rows * n))
        got = be.download(many).reshape(3, rows, n)
        assert np.abs(got - np.stack([want, -want, 2 * want])).max() <= 2 * tol


@pytest.mark.parametrize("tile", [-1, 2, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("layout", ["NN", "NT", "TN", "TT"])
@pytest.mark.parametrize("m,k,n", [(1, 256, 4), (64, 256, 32), (68, 288, 100), (200, 320, 516), (300, 2048, 64), (33, 256, 129), (4, 261, 8),
                                   (132, 1000, 68), (2116, 256, 1028)])
def test_f32_tiles(be, tile, layout, m, k, n):
    """Every f32 tile, forced where it fits, in each operand layout: rows and columns that end inside a tile, fewer K steps
    than stages or wave groups, reductions that end inside a step, more tiles than compute units; plain, accumulated and
    batched outputs, against the f64 product. Rounding each of k products and k sums to f32 gives an error of at most
    (k + 1) 2^-24 sum |a||b| per output; a value accumulated onto is one term more of the sum."""
    from ojas_amd.backend import F32

    print(f"gemm f32 tile {tile} {layout} {m}x{k}x{n}", flush=True)
    rng = np.random.default_rng(m * 31 + k + n)
    a, b = rng.normal(size=(2, m, k)).astype(np.float32), rng.normal(size=(2, k, n)).astype(np.float32)
    a_km, b_km = layout[0] == "T", layout[1] == "T"
    if (m % 4 and a_km) or (n % 4 and b_km):
        pytest.skip("a batch's products start 16 bytes apart")
    pad = -k % 4  # rows 16-byte aligned
    da = be.upload(np.ascontiguousarray(a.transpose(0, 2, 1)) if a_km else np.pad(a, ((0, 0), (0, 0), (0, pad))))
    db = be.upload(b if b_km else np.pad(np.ascontiguousarray(b.transpose(0, 2, 1)), ((0, 0), (0, 0), (0, pad))))
    sa, sb = ((1, m) if a_km else (k + pad, 1)), ((n, 1) if b_km else (1, k + pad))
    want = a.astype(np.float64) @ b.astype(np.float64)
    bound = (k + 1) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)) + 1e-30
    be.set_option("gemm_f32", tile)
    try:
        one = be.download(be.gemm(da, sa, db, sb, m, k, n))
        assert (np.abs(one - want[0]) <= bound[0]).all()
        c0 = rng.normal(size=(m, n)).astype(np.float32)
        acc = be.upload(c0)
        be.gemm(da, sa, db, sb, m, k, n, c=acc)
        assert (np.abs(be.download(acc) - (want[0] + c0)) <= bound[0] * (k + 2) / (k + 1) + (k + 2) * 2.0 ** -24 * np.abs(c0)).all()
        if m * n % 4 == 0:
            size = lambda t: int(np.prod(t.shape)) // 2
            both = be.download(be.gemm_strided_batch(da, sa, db, sb, m, k, n, 2, (size(da), size(db), m * n))).reshape(2, m, n)
            assert np.array_equal(both[0], one) or tile < 0
            assert (np.abs(both - want) <= bound).all()
        if m > 1:
            bad = a[0].copy()
            bad[-1, -1] = np.inf
            dbad = be.upload(np.ascontiguousarray(bad.T) if a_km else np.pad(bad, ((0, 0), (0, pad))))
            from ojas_amd.backend import OjasError
            be.gemm(dbad, sa, db, sb, m, k, n)
            with pytest.raises(OjasError):
                be.sync()
    finally:
        be.set_option("gemm_f32", -1)


@pytest.mark.parametrize("tanh", [0, 1])
@pytest.mark.parametrize("rows,kin,nout", [(2048, 256, 1024), (70, 288, 36), (65, 256, 61), (513, 1024, 33), (3, 260, 20), (33, 64, 50), (300, 512, 512)])
def test_f32_activation_in_the_store_pass_carries_the_separate_passes_bits(be, rows, kin, nout, tanh):
    """`omx_linear_gelu_f32_forward` and `omx_linear_backward_input_gelu_f32` against product and pass: the kernel with the
    activation in its store pass at the edges of its tiles, and products that it does not take."""
    from ojas_amd.backend import F32

    print(f"f32 gelu products {rows}x{kin}x{nout} tanh={tanh}", flush=True)
    be.set_option("gemm_dma", 1)
    r = np.random.default_rng(rows + kin + nout)
    x, w, gy = ((r.standard_normal(s) * size).astype(np.float32) for s, size in (((rows, kin), 1.0), ((nout, kin), 0.1), ((rows, kin), 1.0)))
    dx, dw, u, act = be.upload(x), be.upload(w), be.empty((rows, nout), F32), be.empty((rows, nout), F32)
    n64 = lambda *v: tuple(C.c_uint64(i) for i in v)
    p = be._p
    be._check(be._lib.omx_linear_gelu_f32_forward(be._ctx, p(dx), p(dw), p(u), p(act), *n64(rows, kin, nout), C.c_int32(tanh)))
    forward, backward = (be.gelu_tanh_forward, be.gelu_tanh_backward) if tanh else (be.gelu_erf_forward, be.gelu_erf_backward)
    want = be.linear_forward(dx, dw)
    assert np.array_equal(be.download(u), be.download(want)) and np.array_equal(be.download(act), be.download(forward(want)))
    # gu [rows, nout] = (gy [rows, kin] . v [kin, nout]) gelu'(u)
    dv, dg, gu = be.upload(np.ascontiguousarray(w.T)), be.upload(gy), be.empty((rows, nout), F32)
    be._check(be._lib.omx_linear_backward_input_gelu_f32(be._ctx, p(dv), p(dg), p(u), p(gu), *n64(rows, nout, kin), C.c_int32(tanh)))
    assert np.array_equal(be.download(gu), be.download(backward(u, be.linear_backward_input(dv, dg))))


@pytest.mark.parametrize("tile", [5, 6, 7, 8, 9])  # gemm_dma32.hip's, whose store pass forms the activation; the kernel before a pass of its own
@pytest.mark.parametrize("tanh", [0, 1])
def test_f32_activation_in_the_store_pass_is_named_as_the_separate_pass_is(be, tile, tanh):
    """A product that is not finite carries the product's name, an activation that is not the activation's."""
    from ojas_amd.backend import OjasError

    print(f"f32 gelu products, fault names, tile {tile} tanh={tanh}", flush=True)
    r = np.random.default_rng(tile)
    rows, nin, nout = 70, 260, 256
    n64 = lambda *v: tuple(C.c_uint64(i) for i in v)
    p = be._p

    def backward(gy, w, u):
        gu = be.empty(u.shape)
        be._check(be._lib.omx_linear_backward_input_gelu_f32(be._ctx, p(w), p(gy), p(u), p(gu), *n64(rows, nin, nout), C.c_int32(tanh)))

    def forward(x, w):
        u, act = be.empty((rows, nin)), be.empty((rows, nin))
        be._check(be._lib.omx_linear_gelu_f32_forward(be._ctx, p(x), p(w), p(u), p(act), *n64(rows, nout, nin), C.c_int32(tanh)))

    w, gy, u = (r.standard_normal(s).astype(np.float32) for s in ((nout, nin), (rows, nout), (rows, nin)))
    bad_gy, bad_u, huge_gy, huge_w, peak_u = gy.copy(), u.copy(), np.zeros_like(gy), np.zeros_like(w), u.copy()
    bad_gy[-1, 4] = np.inf
    bad_u[69, 259] = np.nan
    huge_gy[3, 0], huge_w[0, 5], peak_u[3, 5] = 3.2e38, 1.0, 1.4  # a finite product, 1.13 times too large
    cases = [(backward, (bad_gy, w, u), "linear_backward"), (backward, (gy, w, bad_u), "gelu_backward"),
             (backward, (huge_gy, huge_w, peak_u), "gelu_backward"), (forward, (bad_gy, np.ascontiguousarray(w.T)), "linear_forward")]
    be.set_option("gemm_dma", 1)
    be.set_option("gemm_f32", tile)
    try:
        for op, args, name in cases:
            op(*[be.upload(a) for a in args])
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.detail == name, (tile, e.value.detail)
        backward(*[be.upload(a) for a in (gy, w, u)])
        be.sync()
    finally:
        be.set_option("gemm_f32", -1)


@pytest.mark.parametrize("pair", [1, 2, 3, 4, -1])
@pytest.mark.parametrize("rows,kin,nout", [(1, 4, 4), (16, 32, 16), (65, 34, 20), (130, 96, 36), (257, 70, 12), (1021, 66, 132), (300, 512, 260), (4100, 32, 64),
                                           (700, 900, 256), (900, 516, 320), (500, 380, 512)])  # last: gx on 1, 2 and 4 groups of waves
def test_both_gradients_in_one_launch(be, pair, rows, kin, nout):
    """Each pair of tiles, forced where it fits, and the rule's choice: outputs that end inside a tile, walks of one step, of fewer
    steps than waves and ending inside one, more tiles than compute units; against the f64 products, k products and k sums rounded
    to f32 each: (k + 1) 2^-24 sum |a||b|. A value that is not finite is named; outputs that overlap an operand take two launches.
    The weight gradient has an order of sums of its own there, no further from the f64 product than a call's for it alone."""
    from ojas_amd.backend import OjasError

    print(f"gradients together {pair} {rows}x{kin}x{nout}", flush=True)
    be.set_option("gemm_dma", 1)
    r = np.random.default_rng(rows + kin + nout)
    x, w, gy = (r.normal(size=s).astype(np.float32) for s in ((rows, kin), (nout, kin), (rows, nout)))
    x64, w64, g64 = (a.astype(np.float64) for a in (x, w, gy))
    bounds = [(nout + 1) * 2.0 ** -24 * (np.abs(g64) @ np.abs(w64)), (rows + 1) * 2.0 ** -24 * (np.abs(g64).T @ np.abs(x64))]
    dx, dw, dg = (be.upload(a) for a in (x, w, gy))
    be.set_option("gemm_f32_pair", pair)
    launches = C.c_uint64()

    def launched(call):
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(1)))
        result = call()
        be._check(be._lib.omx_profile_gemm_report(be._ctx, C.byref(launches), None, None))
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
        return launches.value, result

    try:
        count, grads = launched(lambda: be.linear_backward(dx, dw, dg))
        assert count == 1 or (pair < 0 and rows not in (700, 900, 500))
        for got, want, bound in zip(grads, (g64 @ w64, g64.T @ x64), bounds):
            assert (np.abs(be.download(got) - want) <= bound + 1e-30).all()
        if pair < 0:  # the input gradient's bits do not depend on who asks for it
            assert np.array_equal(be.download(be.linear_backward(dx, dw, dg)[0]), be.download(be.linear_backward_input(dw, dg)))
            off = [np.linalg.norm(be.download(g) - g64.T @ x64) for g in (grads[1], be.linear_backward(dx, dw, dg, need_gx=False)[1])]
            assert off[0] <= 1.05 * off[1], off
        before = r.normal(size=x.shape).astype(np.float32)
        onto, gw = be.linear_backward_onto(be.upload(before), dx, dw, dg)
        assert (np.abs(be.download(onto) - (g64 @ w64 + before)) <= bounds[0] * (nout + 2) / (nout + 1) + 2.0 ** -23 * np.abs(before)).all()
        assert (np.abs(be.download(gw) - g64.T @ x64) <= bounds[1] + 1e-30).all()
        n64 = tuple(C.c_uint64(v) for v in (rows, kin, nout))
        back = lambda gx: be._check(be._lib.omx_linear_backward(be._ctx, be._p(dx), be._p(dw), be._p(dg), C.c_int32(0), be._p(gx), C.c_int32(0),
                                                                be._p(gw), C.c_int32(0), *n64))
        be.set_option("gemm_f32_pair", 0)
        back(dx)  # over the layer's input, which the second product then reads
        apart = be.download(gw)
        dx = be.upload(x)
        be.set_option("gemm_f32_pair", pair)
        assert launched(lambda: back(dx))[0] == 2
        assert np.array_equal(be.download(gw), apart)
        gy[-1, -1] = np.inf
        be.linear_backward(be.upload(x), dw, be.upload(gy))
        with pytest.raises(OjasError) as e:
            be.sync()
        assert e.value.detail == "linear_backward"
    finally:
        be.set_option("gemm_f32_pair", -1)


def test_products_of_one_launch_are_in_the_profile(be):
    """Both gradients of a linear layer and the Newton-Schulz products of two shapes: one entry a launch with the products' operations,
    and the bits of a call that is not timed."""
    from ojas_amd.backend import MuonNs5Config

    print("profile of products together", flush=True)
    be.set_option("gemm_dma", 1)
    r = np.random.default_rng(3)
    x, w, gy = (be.upload(r.standard_normal(s, dtype=np.float32)) for s in ((1024, 256), (128, 256), (1024, 128)))
    dims = [(64, 48), (36, 100), (64, 48)]
    host = [[(r.standard_normal(d) * s).astype(np.float32) for d in dims] for s in (0.1, 0.05, 0.01)]

    def step():
        out = list(be.linear_backward(x, w, gy))
        p, g, m = ([be.upload(a) for a in xs] for xs in host)
        be.muon_ns5_step_shapes(p, g, m, MuonNs5Config(0.02, 0.95, 0.1, 1, 0))
        return [be.download(t) for t in out + p]

    want = step()
    try:
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(1)))
        got = step()
        launches, ms, flops = C.c_uint64(), C.c_double(), C.c_double()
        be._check(be._lib.omx_profile_gemm_report(be._ctx, C.byref(launches), C.byref(ms), C.byref(flops)))
    finally:
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    assert launches.value == 1 + 15 and ms.value > 0
    ns = sum(5 * 2.0 * (2 * min(d) ** 2 * max(d) + min(d) ** 3) for d in dims)
    assert flops.value == 4.0 * 1024 * 256 * 128 + ns


@pytest.mark.parametrize("rows,out,hidden,mode", [(300, 128, 128, 9), (256, 256, 384, 9), (1, 384, 128, 9), (513, 128, 640, 9), (300, 128, 72, 9),
                                                 (300, 192, 128, 1), (70, 64, 8, 1), (8192, 256, 1024, 1), (9000, 128, 3968, 1)])
def test_gradients_of_gates_and_ups_of_one_product_have_the_bits_of_two_calls(be, rows, out, hidden, mode):
    """linear_backward_input_swiglu, with the activation's gradient in the one-wave kernel's store pass (ragged rows, tiles half outside, a
    product cut by rows) and where it takes the pass: as linear_backward and swiglu_backward leave it; over int8 codes too; then a
    gradient, and a product, that is the first value that is not finite, named as its own op's."""
    from ojas_amd.backend import BF16, F32, OjasError, _native

    rng = np.random.default_rng(rows + hidden)
    gy = be.upload(rng.normal(size=(rows, out)).astype(np.float32), BF16)
    w = be.upload((0.2 * rng.normal(size=(out, hidden))).astype(np.float32), BF16)
    wide = rng.normal(size=(rows, 2 * hidden)).astype(np.float32)
    gu = be.upload(wide)
    be.set_option("gemm_dma", mode)
    try:
        gm, want, got, scratch = (be.empty((rows, c * hidden), BF16) for c in (1, 2, 2, 1))
        _native.omx_linear_backward(be._context, None, w, gy, BF16, gm, BF16, None, F32, rows, hidden, out)
        for side, dtype in ((gu, F32), (be.upload(wide, BF16), BF16)):
            _native.omx_swiglu_backward(be._context, side, gm, want, dtype, rows, hidden)
            _native.omx_linear_backward_input_swiglu(be._context, w, gy, BF16, side, dtype, scratch, got, rows, hidden, out)
            np.testing.assert_array_equal(be.download(got), be.download(want))
        if hidden % 32 == 0 and out % 32 == 0:
            codes, scales = rng.integers(-127, 128, (out, hidden)).astype(np.int8), rng.uniform(1e-3, 2e-3, (out, hidden // 32)).astype(np.float32)
            codes, scales = be.upload(codes), be.upload(scales)
            for widen in (0, 1):
                be.set_option("q8_widen", widen)
                _native.omx_linear_i8_group_backward_input(be._context, codes, scales, 32, 0, gy, BF16, None, None, gm, rows, hidden, out)
                _native.omx_swiglu_backward(be._context, gu, gm, want, F32, rows, hidden)
                _native.omx_linear_i8_group_backward_input_swiglu(be._context, codes, scales, 32, 0, gy, BF16, gu, scratch, got, rows, hidden, out)
                np.testing.assert_array_equal(be.download(got), be.download(want))
        large, steep = be.upload(np.full((rows, 2 * hidden), 2.0**100, np.float32)), be.upload(np.full((rows, out), 2.0**10, np.float32), BF16)
        for height, name in ((2.0**30, "mul_backward"), (2.0**120, "linear_backward")):
            _native.omx_linear_backward_input_swiglu(be._context, be.upload(np.full((out, hidden), height, np.float32), BF16), steep, BF16, large, F32, scratch,
                                                     got, rows, hidden, out)
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.detail == name
    finally:
        be.set_option("gemm_dma", 1)
        be.set_option("q8_widen", -1)


@pytest.mark.parametrize("rows,kin,hidden,mode", [(300, 128, 64, 9), (256, 256, 192, 9), (1, 384, 128, 9), (513, 128, 320, 9), (300, 128, 72, 9),
                                                 (300, 192, 64, 1), (70, 64, 8, 1), (8192, 256, 1024, 1), (9000, 128, 1984, 1)])
def test_gates_and_ups_of_one_product_have_the_bits_of_two_calls(be, rows, kin, hidden, mode):
    """linear_swiglu_forward, with the activation in the one-wave kernel's store pass (ragged rows, half tiles of units, a product cut by
    rows) and where it takes the pass: product and activation as linear_forward and swiglu_forward leave them; over int8 codes too; then
    an activation, and a product, that is the first value that is not finite, named as its own op's."""
    from ojas_amd.backend import BF16, F32, OjasError, _native

    rng = np.random.default_rng(rows + hidden)
    x = be.upload(rng.normal(size=(rows, kin)).astype(np.float32), BF16)
    w = be.upload((0.2 * rng.normal(size=(2 * hidden, kin))).astype(np.float32), BF16)
    be.set_option("gemm_dma", mode)
    try:
        gu = be.linear_forward(x, w, F32)
        act = be.swiglu_forward(gu)
        got_gu, got = be.empty((rows, 2 * hidden), F32), be.empty((rows, hidden), BF16)
        _native.omx_linear_swiglu_forward(be._context, x, w, BF16, got_gu, F32, got, rows, kin, hidden)
        np.testing.assert_array_equal(be.download(got_gu), be.download(gu))
        np.testing.assert_array_equal(be.download(got), be.download(act))
        gu16 = be.linear_forward(x, w, BF16)
        got16 = be.empty((rows, 2 * hidden), BF16)
        _native.omx_linear_swiglu_forward(be._context, x, w, BF16, got16, BF16, got, rows, kin, hidden)
        np.testing.assert_array_equal(be.download(got16), be.download(gu16))
        np.testing.assert_array_equal(be.download(got), be.download(be.swiglu_forward(gu16)))
        if kin % 128 == 0:
            codes, scales = rng.integers(-127, 128, (2 * hidden, kin)).astype(np.int8), rng.uniform(1e-3, 2e-3, (2 * hidden, kin // 32)).astype(np.float32)
            codes, scales = be.upload(codes), be.upload(scales)
            for widen in (0, 1):
                be.set_option("q8_widen", widen)
                _native.omx_linear_i8_group_forward(be._context, x, BF16, codes, scales, 32, 0, None, None, gu, F32, rows, kin, 2 * hidden)
                _native.omx_linear_i8_group_swiglu_forward(be._context, x, BF16, codes, scales, 32, 0, got_gu, got, rows, kin, hidden)
                np.testing.assert_array_equal(be.download(got_gu), be.download(gu))
                np.testing.assert_array_equal(be.download(got), be.download(be.swiglu_forward(gu)))
        big = be.upload(np.full((rows, kin), 2.0**60, np.float32), BF16)
        for height, name in ((2.0**10, "mul_forward"), (2.0**70, "linear_forward")):
            _native.omx_linear_swiglu_forward(be._context, big, be.upload(np.full((2 * hidden, kin), height, np.float32), BF16), BF16, got_gu, F32, got, rows,
                                              kin, hidden)
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.detail == name
    finally:
        be.set_option("gemm_dma", 1)
        be.set_option("q8_widen", -1)


@pytest.mark.parametrize("m,k,n,lda,count", [(1, 1, 8, 1, 1), (5, 31, 64, 5, 3), (10, 282, 640, 10, 2), (12, 33, 72, 12, 1), (16, 1023, 264, 17, 2), (13, 1024, 256, 13, 1),
                                             (12, 1025, 768, 12, 3), (3, 2049, 8, 9, 1), (12, 8200, 328, 12, 2), (15, 20000, 128, 15, 1)])
@pytest.mark.parametrize("bf16_out", [False, True])
def test_weight_gradients_of_a_few_heads(be, m, k, n, lda, count, bf16_out):
    """`gemm_heads_kernel`: at most 16 rows from two operands by rows of the reduction, A's pitch any; one share of the rows and several,
    partial last steps and column blocks. f32 sums of exact products: within k roundings of the terms' size."""
    from ojas_amd.backend import BF16, F32

    rng = np.random.default_rng(m + k + n)
    stride_a, stride_b = -(-k * lda // 8) * 8, k * n
    a = np.zeros((count, stride_a), np.float32)
    for i in range(count):
        a[i, :k * lda] = rng.normal(0, 1, k * lda)
    b = rng.normal(0, 1, (count, k, n)).astype(np.float32)
    da, db = be.upload(a, BF16), be.upload(b, BF16)
    if count == 1:
        got = be.gemm(da, (1, lda), db, (n, 1), m, k, n, BF16 if bf16_out else F32)
    else:
        stride_c = -(-m * n // 8) * 8
        got = be.gemm_strided_batch(da, (1, lda), db, (n, 1), m, k, n, count, (stride_a, stride_b, stride_c), BF16 if bf16_out else F32)
    got = be.download_f32(got).reshape(-1)
    ar, br = be.download_f32(da).astype(np.float64), be.download_f32(db).astype(np.float64).reshape(count, k, n)
    for i in range(count):
        ai = ar.reshape(count, stride_a)[i, :k * lda].reshape(k, lda)[:, :m]
        want, size = ai.T @ br[i], np.abs(ai).T @ np.abs(br[i])
        at = 0 if count == 1 else i * stride_c
        part = got[at:at + m * n].reshape(m, n)
        assert np.all(np.abs(part - want) <= size * k * 2.0**-24 + (np.abs(want) * 2.0**-8 if bf16_out else 0) + 1e-30)


@pytest.mark.parametrize("blocks", [1, 2])
@pytest.mark.parametrize("m,k,n,count", [(1, 32, 8, 1), (15, 64, 64, 1), (17, 288, 72, 2), (33, 1280, 200, 1), (64, 736, 640, 1), (282, 544, 136, 1), (100, 4096, 64, 3)])
@pytest.mark.parametrize("by_k", [False, True])
def test_few_rows_on_64_columns_a_workgroup(be, m, k, n, count, blocks, by_k):
    """`gemm_skinny64_km_kernel` and `_kc_kernel`, linear layers and their input gradients of few rows: f32 and bf16 outputs, accumulation, ragged rows and columns, waves without a
    step. f32 sums of exact products: within k roundings of the terms' size."""
    from ojas_amd.backend import BF16, F32

    rng = np.random.default_rng(m + k + n)
    a, b = rng.normal(0, 1, (count, m, k)).astype(np.float32), rng.normal(0, 1, (count, k, n)).astype(np.float32)
    da, db = be.upload(a, BF16), be.upload(b, BF16)
    ar, br = be.download_f32(da).astype(np.float64), be.download_f32(db).astype(np.float64)
    want, size = ar @ br, np.abs(ar) @ np.abs(br)
    bound = size * k * 2.0**-24
    strides = (1, k) if by_k else (n, 1)
    if by_k:
        db = be.upload(np.ascontiguousarray(b.transpose(0, 2, 1)), BF16)
    try:
        be.set_option("gemm_skinny64", blocks)
        for dtype in (F32, BF16):
            if count == 1:
                got = be.gemm(da, (k, 1), db, strides, m, k, n, dtype)
            else:
                got = be.gemm_strided_batch(da, (k, 1), db, strides, m, k, n, count, (m * k, k * n, m * n), dtype)
            got = be.download_f32(got).reshape(want.shape)
            assert np.all(np.abs(got - want) <= bound + (np.abs(want) * 2.0**-8 if dtype == BF16 else 0))
        if count == 1:
            start = rng.normal(0, 1, (m, n)).astype(np.float32)
            got = be.download(be.gemm(da, (k, 1), db, strides, m, k, n, F32, be.upload(start)))
            assert np.all(np.abs(got - (want[0] + start)) <= bound[0] + (np.abs(want[0]) + np.abs(start)) * 2.0**-23)
    finally:
        be.set_option("gemm_skinny64", -1)
