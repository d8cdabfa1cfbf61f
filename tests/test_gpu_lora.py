"""GPU parity of the LoRA fine-tune path (int8 group weights, head_dim 128 attention, the step)
against the oracle (oracle/lora_exact.cpp), through the C ABI."""
import ctypes as C

import numpy as np
import pytest

import oracle_api as orc

pytestmark = pytest.mark.gpu

BF16_TOL = 2e-2  # per element, relative to the tensor's largest value (the bf16 tier's gate)


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    b = MiBackend(0)
    yield b
    b.close()


def _close(got, want, tol=BF16_TOL):
    scale = max(float(np.max(np.abs(want))), 1e-12)
    err = float(np.max(np.abs(got - want)))
    assert err <= tol * scale, (err / scale, got.shape)


# (rows, k_in, n_out): tile-exact, ragged in every direction, one step, many steps.
Q8_SHAPES = [(256, 64, 128), (300, 96, 100), (77, 32, 36), (512, 2048, 256), (1024, 256, 416), (33, 704, 160)]


@pytest.mark.parametrize("rows,kin,nout", Q8_SHAPES)
@pytest.mark.parametrize("with_add", [False, True])
def test_linear_i8_group_forward(be, rows, kin, nout, with_add):
    from ojas_amd.backend import BF16

    print(f"q8 forward rows={rows} kin={kin} nout={nout} add={with_add}", flush=True)
    rng = np.random.default_rng(rows * 7 + kin)
    x = orc.round_bf16(rng.normal(0, 1, (rows, kin)).astype(np.float32))
    codes, scales = orc.quantize_i8_group(rng.normal(0, 0.05, (nout, kin)).astype(np.float32) *
                                          rng.uniform(0.2, 3.0, (nout, 1)).astype(np.float32), 32)
    add = orc.round_bf16(rng.normal(0, 0.3, (rows, nout)).astype(np.float32)) if with_add else None
    want = orc.linear_i8_group_forward(x, codes, scales, 32) + (add if with_add else 0)
    y = be.linear_i8_group_forward(be.upload(x, BF16), be.upload(codes), be.upload(scales),
                                   be.upload(add, BF16) if with_add else None)
    _close(be.download_f32(y), want)
    # The same product left in f32: what the bf16 output is the rounding of.
    from ojas_amd.backend import F32
    y32 = be.linear_i8_group_forward(be.upload(x, BF16), be.upload(codes), be.upload(scales),
                                     be.upload(add, BF16) if with_add else None, out_dtype=F32)
    assert y32.dtype == F32
    assert np.array_equal(orc.round_bf16(be.download(y32)), be.download_f32(y))


@pytest.mark.parametrize("rows,kin,nout", [(256, 128, 64), (300, 96, 160), (77, 32, 32), (512, 256, 2048),
                                           (1024, 416, 256), (33, 160, 704)])
@pytest.mark.parametrize("with_add", [False, True])
def test_linear_i8_group_backward_input(be, rows, kin, nout, with_add):
    from ojas_amd.backend import BF16

    print(f"q8 input gradient rows={rows} kin={kin} nout={nout} add={with_add}", flush=True)
    rng = np.random.default_rng(rows * 5 + nout)
    gy = orc.round_bf16(rng.normal(0, 1, (rows, nout)).astype(np.float32))
    codes, scales = orc.quantize_i8_group(rng.normal(0, 0.05, (nout, kin)).astype(np.float32) *
                                          rng.uniform(0.2, 3.0, (nout, 1)).astype(np.float32), 32)
    add = orc.round_bf16(rng.normal(0, 0.3, (rows, kin)).astype(np.float32)) if with_add else None
    want = orc.linear_i8_group_backward_input(codes, scales, gy, 32) + (add if with_add else 0)
    gx = be.linear_i8_group_backward_input(be.upload(codes), be.upload(scales), be.upload(gy, BF16),
                                           be.upload(add, BF16) if with_add else None)
    _close(be.download_f32(gx), want)


# Rows: under and around a tile; k_in and n_out: one step and ragged tiles; (rank, block_cols) of the low-rank term.
@pytest.mark.parametrize("backward", [False, True])
@pytest.mark.parametrize("rows,kin,nout,rank,block,blocked", [
    (33, 128, 64, 16, 0, True), (257, 128, 384, 16, 128, True), (1025, 512, 768, 32, 256, True), (300, 192, 320, 16, 0, False),
    (4100, 256, 512, 0, 0, True), (8193, 768, 2304, 16, 768, True)])
def test_linear_i8_group_over_a_widened_copy(be, rows, kin, nout, rank, block, blocked, backward):
    # A weight widened in scratch gives the bits of one widened on its way where K is not shared: the same bf16 values, the same order
    # of sums.
    from ojas_amd.backend import BF16, F32

    print(f"q8 widened rows={rows} kin={kin} nout={nout} rank={rank} backward={backward}", flush=True)
    rng = np.random.default_rng(rows + kin)
    codes = be.upload(rng.integers(-127, 128, (nout, kin)).astype(np.int8))
    scales = be.upload(rng.uniform(1e-4, 1e-3, (nout, kin // 32)).astype(np.float32))
    if blocked:
        codes, scales = be.pack_i8_group(codes, scales)
    cols = kin if backward else nout
    if backward:
        block = 0
    x = be.upload(rng.normal(0, 1, (rows, nout if backward else kin)).astype(np.float32), BF16)
    low_rank = None
    if rank:
        h = rng.normal(0, 1, (rows, rank * (cols // block if block else 1))).astype(np.float32)
        low_rank = (be.upload(h, BF16), be.upload(rng.normal(0, 0.1, (cols, rank)).astype(np.float32), BF16), block)
    got = []
    try:
        for widen in (0, 1):
            be.set_option("q8_widen", widen)
            y = (be.linear_i8_group_backward_input(codes, scales, x, blocked=blocked, low_rank=low_rank) if backward else
                 be.linear_i8_group_forward(x, codes, scales, blocked=blocked, low_rank=low_rank, out_dtype=F32))
            got.append(be.download_f32(y))
    finally:
        be.set_option("q8_widen", -1)
    assert np.array_equal(got[0], got[1])


# Few tiles over a long reduction, few rows and few columns: over the copy K is shared between launches or between waves.
@pytest.mark.parametrize("backward", [False, True])
@pytest.mark.parametrize("rows,kin,nout,rank", [(256, 8192, 2048, 16), (300, 4096, 1024, 32), (64, 2048, 6144, 0), (17, 4096, 256, 0),
                                                (1500, 2048, 64, 0), (1100, 128, 2048, 0)])
def test_linear_i8_group_over_a_widened_copy_that_shares_k(be, rows, kin, nout, rank, backward):
    """Both ways against the f64 product of the same bf16 operands: k exact products and as many f32 additions, (k + rank) 2^-23
    sum |a||b| with room for an accumulator that cuts off, an input gradient's store to bf16 on top; and the copy's error no larger."""
    from ojas_amd.backend import BF16, F32

    print(f"q8 widened, K shared: rows={rows} kin={kin} nout={nout} rank={rank} backward={backward}", flush=True)
    rng = np.random.default_rng(rows + nout)
    codes, scales = rng.integers(-127, 128, (nout, kin)).astype(np.int8), rng.uniform(1e-4, 1e-3, (nout, kin // 32)).astype(np.float32)
    w = orc.round_bf16(codes * np.repeat(scales, 32, 1)).astype(np.float64)
    w = w if backward else w.T
    x = orc.round_bf16(rng.normal(0, 1, (rows, len(w))).astype(np.float32))
    dx, low_rank = be.upload(x, BF16), None
    want, size = x.astype(np.float64) @ w, np.abs(x).astype(np.float64) @ np.abs(w)
    if rank:
        h, up = (orc.round_bf16(rng.normal(0, s, (n, rank)).astype(np.float32)) for s, n in ((1, rows), (0.1, w.shape[1])))
        low_rank = (be.upload(h, BF16), be.upload(up, BF16), 0)
        want, size = want + h.astype(np.float64) @ up.T, size + np.abs(h).astype(np.float64) @ np.abs(up.T)
    bound = (len(w) + rank) * 2.0 ** -23 * size
    dc, ds = be.pack_i8_group(be.upload(codes), be.upload(scales))
    errors = []
    try:
        for widen in (0, 1):
            be.set_option("q8_widen", widen)
            y = (be.linear_i8_group_backward_input(dc, ds, dx, blocked=True, low_rank=low_rank) if backward else
                 be.linear_i8_group_forward(dx, dc, ds, blocked=True, low_rank=low_rank, out_dtype=F32))
            off = np.abs(be.download_f32(y) - want)
            assert (off <= bound + (2.0 ** -8 * (np.abs(want) + bound) if backward else 0)).all()
            errors.append(np.linalg.norm(off))
    finally:
        be.set_option("q8_widen", -1)
    assert errors[1] <= 1.01 * errors[0], errors


def test_linear_i8_group_scale_per_group_is_exact(be):
    # One code per group set, powers of two as scales, a one-hot input: the product is exact in
    # bf16, so a scale taken from the wrong group or row, or a mis-signed code, shows bit for bit.
    from ojas_amd.backend import BF16

    nout, kin = 160, 128
    rng = np.random.default_rng(9)
    codes = rng.integers(-127, 128, (nout, kin)).astype(np.int8)
    codes[3, 5], codes[7, 64] = -127, 127
    scales = (2.0 ** rng.integers(-6, 3, (nout, kin // 32))).astype(np.float32)
    x = np.eye(kin, dtype=np.float32)  # row k picks column k of W
    y = be.download_f32(be.linear_i8_group_forward(be.upload(x, BF16), be.upload(codes), be.upload(scales)))
    want = orc.round_bf16(orc.dequant_i8_group(codes, scales, 32)).T
    assert np.array_equal(y, want)
    gy = np.eye(nout, dtype=np.float32)
    gx = be.download_f32(be.linear_i8_group_backward_input(be.upload(codes), be.upload(scales), be.upload(gy, BF16)))
    assert np.array_equal(gx, want.T)


@pytest.mark.parametrize("rows,kin,nout", [(300, 128, 104), (512, 2048, 256), (260, 384, 160)])
def test_blocked_layout_gives_the_same_products(be, rows, kin, nout):
    from ojas_amd.backend import BF16

    print(f"q8 blocked rows={rows} kin={kin} nout={nout}", flush=True)
    rng = np.random.default_rng(rows + kin + nout)
    x = be.upload(rng.normal(0, 1, (rows, kin)).astype(np.float32), BF16)
    gy = be.upload(rng.normal(0, 1, (rows, nout)).astype(np.float32), BF16)
    codes_h = rng.integers(-127, 128, (nout, kin)).astype(np.int8)
    scales_h = rng.uniform(1e-3, 2e-2, (nout, kin // 32)).astype(np.float32)
    codes, scales = be.upload(codes_h), be.upload(scales_h)
    bc, bs = be.pack_i8_group(codes, scales)
    # The blocked form is a permutation of the same bytes, spelled out here from its definition.
    r, c = np.meshgrid(np.arange(nout), np.arange(kin), indexing="ij")
    g = c // 32
    off = ((r // 8) * (kin // 128) + g // 4) * 1024 + (g % 4) * 256 + (r % 8) * 32 + c % 32
    want = np.empty(nout * kin, np.int8)
    want[off.reshape(-1)] = codes_h.reshape(-1)
    assert np.array_equal(be.download(bc).reshape(-1), want)
    rs, gs = np.meshgrid(np.arange(nout), np.arange(kin // 32), indexing="ij")
    soff = ((rs // 8) * (kin // 128) + gs // 4) * 32 + (gs % 4) * 8 + rs % 8
    swant = np.empty(scales_h.size, np.float32)
    swant[soff.reshape(-1)] = scales_h.reshape(-1)
    assert np.array_equal(be.download(bs).reshape(-1), swant)
    uc, us = be.unpack_i8_group(bc, bs)
    assert np.array_equal(be.download(uc), codes_h) and np.array_equal(be.download(us), scales_h)
    # Same arithmetic in the same order: bit-identical products.
    y0 = be.download(be.linear_i8_group_forward(x, codes, scales))
    y1 = be.download(be.linear_i8_group_forward(x, bc, bs, blocked=True))
    assert np.array_equal(y0, y1)
    if nout % 32 == 0:
        g0 = be.download(be.linear_i8_group_backward_input(codes, scales, gy))
        g1 = be.download(be.linear_i8_group_backward_input(bc, bs, gy, blocked=True))
        assert np.array_equal(g0, g1)


@pytest.mark.parametrize("rows,kin,time,heads,plain,dim,mode", [(300, 128, 70, 4, 2, 64, 9), (257, 256, 257, 2, 1, 128, 9), (513, 128, 3, 2, 3, 128, 9),
                                                               (40, 128, 1, 2, 2, 64, 9), (300, 128, 100, 2, 1, 64, 9), (300, 128, 100, 2, 1, 32, 9),
                                                               (300, 256, 150, 4, 2, 64, 1), (8192, 256, 512, 8, 4, 128, 1)])
@pytest.mark.parametrize("ranked", [True, False])
def test_turned_heads_of_one_product_have_the_bits_of_two_calls(be, rows, kin, time, heads, plain, dim, mode, ranked):
    """linear_i8_group_rope_forward, with the rotation in the one-wave kernel's store pass (both head widths, ragged rows, sequences that end
    inside a row block) and where it takes the pass, over the codes and over a widened copy; then a product that is not finite and one whose
    rotation is not, each named as its own op's."""
    from ojas_amd.backend import BF16, F32, OjasError, _native

    nout, rank = (heads + plain) * dim, 16
    rng = np.random.default_rng(rows + nout)
    x = be.upload(rng.normal(size=(rows, kin)).astype(np.float32), BF16)
    codes = be.upload(rng.integers(-127, 128, (nout, kin)).astype(np.int8))
    scales = be.upload(rng.uniform(1e-3, 2e-3, (nout, kin // 32)).astype(np.float32))
    cos, sin = (be.upload(f(np.outer(np.arange(time), rng.uniform(0.01, 1.0, dim))).astype(np.float32)) for f in (np.cos, np.sin))
    low_rank = (be.upload(rng.normal(size=(rows, rank)).astype(np.float32), BF16),
                be.upload(rng.normal(size=(nout, rank)).astype(np.float32), BF16), 0) if ranked else None
    tail, tail_at = be._low_rank(low_rank)
    be.set_option("gemm_dma", mode)
    try:
        for widen in (0, 1):
            be.set_option("q8_widen", widen)
            y = be.linear_i8_group_forward(x, codes, scales, low_rank=low_rank, out_dtype=F32)
            want, got, scratch = be.empty((rows, nout), BF16), be.empty((rows, nout), BF16), be.empty((rows, nout), F32)
            _native.omx_rope_half_split_pitched(be._context, y, F32, want, nout, cos, sin, rows, time, heads, plain, dim)
            call = lambda a, s: _native.omx_linear_i8_group_rope_forward(be._context, a, BF16, codes, s, 32, 0, tail_at, scratch, got, cos, sin, rows, kin, time,
                                                                         heads, plain, dim)
            call(x, scales)
            np.testing.assert_array_equal(be.download(got), be.download(want))
        def refused(a, s):
            call(a, s)
            with pytest.raises(OjasError) as e:
                be.sync()
            return e.value.detail

        assert refused(be.upload(np.full((rows, kin), 2.0**100, np.float32), BF16), be.upload(np.full((nout, kin // 32), 2.0**30, np.float32))) == "linear_forward"
        # A head's first half 2^127, its second -2^127: with cos = sin = 1 the turned ones are 2^128 and 0.
        half = np.where(np.arange(nout) % dim < dim // 2, 1, -1).astype(np.int8)
        row = np.zeros((rows, kin), np.float32)
        row[:, 0] = 2.0**60
        codes, cos, sin = be.upload(np.repeat(half[:, None], kin, axis=1)), be.upload(np.ones((time, dim), np.float32)), be.upload(np.ones((time, dim), np.float32))
        assert refused(be.upload(row, BF16), be.upload(np.full((nout, kin // 32), 2.0**67, np.float32))) == "rope_half_split_forward"
    finally:
        be.set_option("gemm_dma", 1)
        be.set_option("q8_widen", -1)


@pytest.mark.parametrize("rows,kin,nout,rank,blocks", [(300, 128, 256, 16, 1), (520, 256, 384, 16, 3),
                                                         (256, 64, 128, 48, 1)])
def test_low_rank_term_rides_in_the_accumulators(be, rows, kin, nout, rank, blocks):
    from ojas_amd.backend import BF16

    print(f"q8 low-rank rows={rows} kin={kin} nout={nout} rank={rank} blocks={blocks}", flush=True)
    rng = np.random.default_rng(rows + rank)
    bf = lambda a: orc.round_bf16(a.astype(np.float32))
    x = bf(rng.normal(0, 1, (rows, kin)))
    codes, scales = orc.quantize_i8_group(rng.normal(0, 0.05, (nout, kin)).astype(np.float32), 32)
    h = bf(rng.normal(0, 1, (rows, blocks * rank)))
    w = bf(rng.normal(0, 0.3, (nout, rank)))
    block_cols = nout // blocks
    want = orc.linear_i8_group_forward(x, codes, scales, 32)
    for j in range(blocks):
        cols = slice(j * block_cols, (j + 1) * block_cols)
        want[:, cols] += h[:, j * rank:(j + 1) * rank].astype(np.float64) @ w[cols].astype(np.float64).T
    y = be.linear_i8_group_forward(be.upload(x, BF16), be.upload(codes), be.upload(scales),
                                   low_rank=(be.upload(h, BF16), be.upload(w, BF16), block_cols if blocks > 1 else 0))
    _close(be.download_f32(y), want)
    # Input gradient: gx = gy W + gh A with A^T [kin, rank] as the term's second operand.
    gy = bf(rng.normal(0, 1, (rows, nout)))
    gh = bf(rng.normal(0, 1, (rows, rank)))
    at = bf(rng.normal(0, 0.3, (kin, rank)))
    if nout % 32 == 0:
        want = orc.linear_i8_group_backward_input(codes, scales, gy, 32) + gh.astype(np.float64) @ at.astype(np.float64).T
        gx = be.linear_i8_group_backward_input(be.upload(codes), be.upload(scales), be.upload(gy, BF16),
                                               low_rank=(be.upload(gh, BF16), be.upload(at, BF16), 0))
        _close(be.download_f32(gx), want)


def test_rope_in_place_and_swiglu(be):
    from ojas_amd.backend import BF16

    tokens, time, heads, dim, pitch = 48, 12, 6, 32, 6 * 32 + 64  # 4 query + 2 key heads, then 64 value columns
    rng = np.random.default_rng(21)
    x = orc.round_bf16(rng.normal(0, 1, (tokens, pitch)).astype(np.float32))
    cos, sin = orc.rope_tables(time, dim)
    rot = orc.rope_forward(np.ascontiguousarray(x[:, :heads * dim]).reshape(tokens // time, time, heads, dim), cos, sin)
    dx = be.upload(x, BF16)
    be.rope_half_split_inplace(dx, be.upload(cos), be.upload(sin), tokens, time, heads, dim)
    got = be.download_f32(dx)
    _close(got[:, :heads * dim], rot.reshape(tokens, heads * dim), 1e-2)
    assert np.array_equal(got[:, heads * dim:], x[:, heads * dim:])  # the value block is untouched
    # The backward is the inverse rotation: forward then backward returns the input (to bf16 rounding).
    be.rope_half_split_inplace(dx, be.upload(cos), be.upload(sin), tokens, time, heads, dim, backward=True)
    back = orc.rope_backward(rot, cos, sin).reshape(tokens, heads * dim)
    _close(be.download_f32(dx)[:, :heads * dim], back, 2e-2)
    # The rotation out of place from an f32 projection output: rotated heads and the value block in
    # one pass, one rounding each.
    from ojas_amd.backend import F32
    x32 = rng.normal(0, 1, (tokens, pitch)).astype(np.float32)
    rot32 = orc.rope_forward(np.ascontiguousarray(x32[:, :heads * dim]).reshape(tokens // time, time, heads, dim), cos, sin)
    for dtype, src in ((F32, x32), (BF16, x)):
        out = be.rope_half_split_pitched(be.upload(src, dtype), be.upload(cos), be.upload(sin), tokens, time, heads, 2, dim)
        got = be.download_f32(out)
        want = rot32 if dtype == F32 else rot
        _close(got[:, :heads * dim], want.reshape(tokens, heads * dim), 1e-2)
        assert np.array_equal(got[:, heads * dim:], orc.round_bf16(src[:, heads * dim:]))  # the value block: converted as it is
    # SwiGLU on a fused gate | up tensor.
    rows, hidden = 37, 72
    gu = orc.round_bf16(rng.normal(0, 1.5, (rows, 2 * hidden)).astype(np.float32))
    gm = orc.round_bf16(rng.normal(0, 1, (rows, hidden)).astype(np.float32))
    gate, up = np.ascontiguousarray(gu[:, :hidden]), np.ascontiguousarray(gu[:, hidden:])
    act = orc.silu_forward(gate)
    want = orc.mul_forward(act, up)
    dgu = be.upload(gu, BF16)
    _close(be.download_f32(be.swiglu_forward(dgu)), want)
    g_act, g_up = orc.mul_backward(act, up, gm)
    g_gate = orc.silu_backward(gate, g_act)
    got = be.download_f32(be.swiglu_backward(dgu, be.upload(gm, BF16)))
    _close(got[:, :hidden], g_gate)
    _close(got[:, hidden:], g_up)
    # The same on an unrounded f32 gate | up tensor (the projection's output kept in f32).
    from ojas_amd.backend import F32
    gu32 = rng.normal(0, 1.5, (rows, 2 * hidden)).astype(np.float32)
    gate, up = np.ascontiguousarray(gu32[:, :hidden]), np.ascontiguousarray(gu32[:, hidden:])
    act = orc.silu_forward(gate)
    dgu = be.upload(gu32, F32)
    out = be.swiglu_forward(dgu)
    assert out.dtype == BF16
    _close(be.download_f32(out), orc.mul_forward(act, up))
    g_act, g_up = orc.mul_backward(act, up, gm)
    got = be.download_f32(be.swiglu_backward(dgu, be.upload(gm, BF16)))
    _close(got[:, :hidden], orc.silu_backward(gate, g_act))
    _close(got[:, hidden:], g_up)


def test_linear_i8_group_refusals(be):
    from ojas_amd.backend import BF16, DTYPE, OUT_OF_RANGE, SHAPE, UNSUPPORTED, OjasError

    x = be.upload(np.zeros((8, 48), np.float32), BF16)
    codes = be.upload(np.zeros((32, 48), np.int8))
    scales = be.upload(np.zeros((32, 1), np.float32))
    with pytest.raises(OjasError) as e:  # k_in is not a multiple of the group
        be._check(be._lib.omx_linear_i8_group_forward(be._ctx, be._p(x), C.c_int32(1), be._p(codes), be._p(scales),
                                                      C.c_uint64(32), C.c_int32(0), None, None, be._p(x), C.c_int32(1), C.c_uint64(8), C.c_uint64(48),
                                                      C.c_uint64(32)))
    assert e.value.code == SHAPE
    with pytest.raises(OjasError) as e:
        be._check(be._lib.omx_linear_i8_group_forward(be._ctx, be._p(x), C.c_int32(1), be._p(codes), be._p(scales),
                                                      C.c_uint64(64), C.c_int32(0), None, None, be._p(x), C.c_int32(1), C.c_uint64(8), C.c_uint64(64),
                                                      C.c_uint64(32)))
    assert e.value.code == UNSUPPORTED
    with pytest.raises(OjasError) as e:
        be._check(be._lib.omx_linear_i8_group_forward(be._ctx, be._p(x), C.c_int32(0), be._p(codes), be._p(scales),
                                                      C.c_uint64(32), C.c_int32(0), None, None, be._p(x), C.c_int32(1), C.c_uint64(8), C.c_uint64(64),
                                                      C.c_uint64(32)))
    assert e.value.code == DTYPE
    # The kernel addresses a lane's bytes with 32 bits beside a 64-bit base: weights of 2 GiB or more and
    # k_in of 4 Mi or more are refused before anything is launched.
    for kin, nout in ((1 << 22, 32), (1 << 16, 1 << 15)):
        with pytest.raises(OjasError) as e:
            be._check(be._lib.omx_linear_i8_group_forward(be._ctx, be._p(x), C.c_int32(1), be._p(codes), be._p(scales),
                                                          C.c_uint64(32), C.c_int32(0), None, None, be._p(x), C.c_int32(1), C.c_uint64(8),
                                                          C.c_uint64(kin), C.c_uint64(nout)))
        assert e.value.code == OUT_OF_RANGE, (kin, nout)


# ---- the step: reduced shapes against the oracle ----
def _load_case(tr, cfg, frozen, quant):
    """Hands a seeded case (test_oracle_lora.make_lora_case) to the device trainer."""
    tr.set_embedding(frozen[0])
    for l in range(cfg.layers):
        base = 1 + 9 * l
        tr.set_norm(l, 0, frozen[base + 0])
        tr.set_norm(l, 1, frozen[base + 5])
        for which, idx in enumerate((1, 2, 3, 4, 6, 7, 8)):
            codes, scales = quant[base + idx]
            tr.set_matrix(l, which, codes, scales)
    tr.set_norm(cfg.layers, 0, frozen[-1])


# (layers, d, heads, head_dim, hidden, vocab, batch, seq, rank, scale)
LORA_STEP_SHAPES = [(2, 128, 2, 64, 256, 96, 2, 48, 16, 2.0), (1, 256, 2, 128, 384, 200, 1, 130, 16, 1.0),
                    (2, 128, 1, 128, 128, 64, 2, 64, 32, 0.5)]


@pytest.mark.parametrize("shape", LORA_STEP_SHAPES)
def test_lora_step_matches_the_oracle(be, shape):
    from test_oracle_lora import make_lora_case

    from ojas_amd.backend import AdamWConfig
    from ojas_amd.lora import LoraConfig, LoraTrainer

    print(f"lora step {shape}", flush=True)
    cfg = LoraConfig(*shape[:9], 1e-6, shape[9], 10000.0)
    ocfg = orc.LoraConfig(*shape[:9], 1e-6, shape[9], 10000.0)
    frozen, quant, adapters, ids, targets = make_lora_case(ocfg, 31 + shape[1])
    adapters = [orc.round_bf16(a) for a in adapters]  # bf16-exact operands on both sides
    tr = LoraTrainer(be, cfg)
    try:
        _load_case(tr, cfg, frozen, quant)
        tr.set_adapters(adapters)
        tr.set_batch(ids, targets)
        loss = tr.loss_and_grads()
        grads = tr.grads()
        oloss, ograds = orc.lora_loss_and_grads(ocfg, frozen, adapters, ids, targets)
        assert abs(loss - float(oloss)) <= 1e-3 * abs(float(oloss)), (loss, oloss)  # the bf16 tier's loss gate
        for i, (g, og) in enumerate(zip(grads, ograds)):
            scale = float(np.max(np.abs(og)))
            assert scale > 0, i
            err = float(np.max(np.abs(g - og)))
            assert err <= BF16_TOL * scale, (i, err / scale)
            assert np.linalg.norm(g - og) <= BF16_TOL * np.linalg.norm(og), i
        # One AdamW step moves every adapter element against its gradient's sign by about lr, and
        # nothing else: the update of an element with a solid gradient is lr to within 1 %.
        lr = 1e-3
        step_loss, norm = tr.step(AdamWConfig(lr, 0.9, 0.95, 1e-8, 0.0), 0.0)
        assert abs(step_loss - loss) <= 1e-6 * abs(loss)
        want_norm = float(np.sqrt(sum(float(np.sum(g.astype(np.float64) ** 2)) for g in grads)))
        assert abs(norm - want_norm) <= 1e-4 * want_norm
        after = tr.adapters()
        for a0, a1, g in zip(adapters, after, grads):
            solid = np.abs(g) > 1e-3 * np.max(np.abs(g))
            move = (a1 - a0.reshape(-1))[solid]
            assert np.all(np.abs(move + lr * np.sign(g[solid])) <= 1e-2 * lr + 4e-8 * np.abs(a0.reshape(-1)[solid]))
        assert tr.steps() == 1
    finally:
        tr.close()


def test_lora_adapter_starts_as_the_identity(be):
    # B = 0 (lora.rs:9-12): the loss is the base model's whatever A holds, dA is exactly zero and dB is not.
    from test_oracle_lora import make_lora_case

    from ojas_amd.lora import LoraConfig, LoraTrainer

    shape = (2, 128, 2, 64, 256, 96, 2, 48, 16)
    cfg = LoraConfig(*shape, 1e-6, 2.0, 10000.0)
    ocfg = orc.LoraConfig(*shape, 1e-6, 2.0, 10000.0)
    frozen, quant, adapters, ids, targets = make_lora_case(ocfg, 5)
    zero_b = [orc.round_bf16(a) if i % 2 == 0 else np.zeros_like(a) for i, a in enumerate(adapters)]
    tr = LoraTrainer(be, cfg)
    try:
        _load_case(tr, cfg, frozen, quant)
        tr.set_batch(ids, targets)
        tr.set_adapters(zero_b)
        loss0 = tr.loss_and_grads()
        grads = tr.grads()
        assert all(not np.any(g) for g in grads[0::2]) and all(np.any(g) for g in grads[1::2])
        tr.set_adapters([2 * a if i % 2 == 0 else a for i, a in enumerate(zero_b)])
        assert tr.loss_and_grads() == loss0
    finally:
        tr.close()


@pytest.mark.parametrize("rows,k,cols,rank,block", [(40, 1024, 192, 16, 0), (213, 1152, 384, 32, 128), (17, 2048, 64, 48, 0), (300, 1088, 136 * 8, 16, 0)])
@pytest.mark.parametrize("backward", [False, True])
def test_low_rank_term_of_few_rows_over_a_long_reduction(be, rows, k, cols, rank, block, backward):
    """The 64-column kernels of few rows with the low-rank term beside the waves' shares of K: within k + rank roundings of the f64 product's
    terms (exact products of bf16 values, f32 sums), and a bf16 output's own."""
    from ojas_amd.backend import BF16

    print(f"q8 low-rank few rows={rows} k={k} cols={cols} rank={rank} backward={backward}", flush=True)
    block = 0 if backward else block
    rng = np.random.default_rng(rows + k)
    nout, kin = (k, cols) if backward else (cols, k)
    codes, scales = rng.integers(-127, 128, (nout, kin)).astype(np.int8), np.full((nout, kin // 32), 2.0**-8, np.float32)
    bf = lambda a: orc.round_bf16(a.astype(np.float32))
    x, w = bf(rng.normal(0, 1, (rows, k))), bf(rng.normal(0, 0.3, (cols, rank)))
    blocks = cols // block if block else 1
    h = bf(rng.normal(0, 1, (rows, blocks * rank)))
    low_rank = (be.upload(h, BF16), be.upload(w, BF16), block)
    weight = bf(codes.astype(np.float32) * 2.0**-8).astype(np.float64)
    weight = weight if backward else weight.T
    want, size = x.astype(np.float64) @ weight, np.abs(x).astype(np.float64) @ np.abs(weight)
    for i in range(blocks):
        at = slice(i * block, (i + 1) * block) if block else slice(None)
        hi = h[:, i * rank:(i + 1) * rank].astype(np.float64)
        want[:, at] += hi @ w[at].T
        size[:, at] += np.abs(hi) @ np.abs(w[at]).T
    be.set_option("q8_widen", 1)
    try:
        args = (be.upload(codes), be.upload(scales), be.upload(x, BF16))
        y = be.linear_i8_group_backward_input(*args, low_rank=low_rank) if backward else be.linear_i8_group_forward(args[2], *args[:2], low_rank=low_rank)
    finally:
        be.set_option("q8_widen", -1)
    assert np.all(np.abs(be.download_f32(y) - want) <= size * (k + rank) * 2.0**-24 + np.abs(want) * 2.0**-8)
