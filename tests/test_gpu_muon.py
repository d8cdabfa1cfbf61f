"""Muon NS5 on the GPU against the CPU oracle (whose f32 path is pinned bit for
bit by the reference's muon_p / muon_m digests).

Gates: the momentum buffer is one f32 multiply-add per value and must carry the
oracle's bits; the parameter goes through five Newton-Schulz iterations of
re-ordered f32 sums, gated like the reference's device runs (1e-4 of the
largest value, ojas-wgpu/tests/common/mod.rs:11); the bf16 iteration is gated
at the reference's own bf16-NS5 parameter bound (5e-2 of the update's scale,
ojas-oracle/src/parity.rs:29-74)."""
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
    backend.close()


@pytest.mark.parametrize("rows,cols", [(64, 48), (48, 64), (130, 70), (97, 97), (768, 768), (768, 3072), (3072, 768)])
def test_muon_f32_matches_cpu_exact(be, rows, cols):
    from ojas_amd.backend import MuonNs5Config

    print(f"muon f32 {rows}x{cols}", flush=True)
    r = orc.SplitMix64(200 + rows)
    p = r.vec(rows * cols, 0.1).reshape(rows, cols)
    g = r.vec(rows * cols, 0.1).reshape(rows, cols)
    m = r.vec(rows * cols, 0.01).reshape(rows, cols)
    orc.set_threads(8)
    op, om = orc.muon_ns5_step(p, g, m)
    dp, dg, dm = be.upload(p), be.upload(g), be.upload(m)
    be.muon_ns5_step(dp, dg, dm, MuonNs5Config.nanolab_default())
    assert np.array_equal(be.download(dm), om), "momentum buffer bits"
    gp = be.download(dp)
    assert np.max(np.abs(gp - op)) <= 1e-4 * max(1.0, np.max(np.abs(op)))
    # The update itself (p_new - p * decay), relative to its own size.
    decay = np.float32(1.0 - 0.025 * 0.1)
    upd_gpu, upd_cpu = gp - p * decay, op - p * decay
    assert np.max(np.abs(upd_gpu - upd_cpu)) <= 2e-3 * np.max(np.abs(upd_cpu))


@pytest.mark.parametrize("rows,cols", [(64, 48), (130, 70), (768, 768), (3072, 768)])
def test_muon_bf16_iteration(be, rows, cols):
    from ojas_amd.backend import MuonNs5Config

    print(f"muon bf16 {rows}x{cols}", flush=True)
    r = orc.SplitMix64(300 + rows)
    p = r.vec(rows * cols, 0.1).reshape(rows, cols)
    g = r.vec(rows * cols, 0.1).reshape(rows, cols)
    m = r.vec(rows * cols, 0.01).reshape(rows, cols)
    orc.set_threads(8)
    op, om = orc.muon_ns5_step(p, g, m, lr=0.02, momentum=0.95, weight_decay=0.0, nesterov=True, bf16=True)
    dp, dg, dm = be.upload(p), be.upload(g), be.upload(m)
    be.muon_ns5_step(dp, dg, dm, MuonNs5Config(0.02, 0.95, 0.0, 1, 1))
    assert np.array_equal(be.download(dm), om)
    upd_gpu, upd_cpu = be.download(dp) - p, op - p
    assert np.max(np.abs(upd_gpu - upd_cpu)) <= 5e-2 * np.max(np.abs(upd_cpu))


def test_muon_is_all_or_nothing_and_refuses_bad_configs(be):
    from ojas_amd.backend import NON_FINITE, OUT_OF_RANGE, MuonNs5Config, OjasError

    rows, cols = 40, 24
    r = orc.SplitMix64(7)
    p, g, m = (r.vec(rows * cols, 0.1).reshape(rows, cols) for _ in range(3))
    g[3, 3] = np.nan
    dp, dg, dm = be.upload(p), be.upload(g), be.upload(m)
    be.muon_ns5_step(dp, dg, dm, MuonNs5Config.nanolab_default())
    with pytest.raises(OjasError) as e:
        be.sync()
    assert e.value.code == NON_FINITE and "muon_ns5_step" in e.value.detail
    assert np.array_equal(be.download(dp), p) and np.array_equal(be.download(dm), m)
    with pytest.raises(OjasError) as e:
        be.muon_ns5_step(dp, dg, dm, MuonNs5Config(-0.1, 0.9, 0.0, 1, 0))
    assert e.value.code == OUT_OF_RANGE
    assert be._lib.omx_muon_scratch_bytes(768, 3072) >= 4 * 768 * 3072 * 4


@pytest.mark.parametrize("rows,cols,count,bf16", [(64, 48, 5, 0), (48, 64, 3, 1), (130, 70, 2, 0), (256, 256, 7, 1),
                                                  (768, 768, 48, 1), (768, 3072, 12, 1), (3072, 768, 12, 0),
                                                  (32, 32, 70, 0)])
def test_batched_step_matches_the_oracle_per_tensor(be, rows, cols, count, bf16):
    """`omx_muon_ns5_step_batched` holds each tensor to the oracle at the single op's gates (momentum
    bit for bit; update 2e-3 of its largest element in f32, 5e-2 with the bf16 iteration). 70 tensors
    go through in two launches of at most 64."""
    from ojas_amd.backend import BF16, MuonNs5Config

    print(f"muon batched {count} x {rows}x{cols} bf16={bf16}", flush=True)
    r = np.random.default_rng(rows * 7 + cols + count)
    ps = [r.standard_normal((rows, cols)).astype(np.float32) * 0.1 for _ in range(count)]
    gs = [r.standard_normal((rows, cols)).astype(np.float32) * (0.02 + 0.05 * i / count) for i in range(count)]
    ms = [r.standard_normal((rows, cols)).astype(np.float32) * 0.01 for _ in range(count)]
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, bf16)
    dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in gs], [be.upload(x) for x in ms]
    mirrors = [be.upload(np.zeros((rows, cols), np.float32), BF16) if i % 2 == 0 else None for i in range(count)]
    be.muon_ns5_step_batched(dp, dg, dm, cfg, mirrors)
    be.sync()
    orc.set_threads(8)
    decay = np.float32(1.0 - 0.02 * 0.1)
    check = range(count) if rows * cols <= 1 << 17 else (0, count // 2, count - 1)  # the oracle is slow on big ones
    for i in check:
        op, om = orc.muon_ns5_step(ps[i], gs[i], ms[i], lr=0.02, momentum=0.95, weight_decay=0.1, nesterov=True,
                                   bf16=bool(bf16))
        assert np.array_equal(be.download(dm[i]), om), i
        got = be.download(dp[i])
        upd_gpu, upd_cpu = got - ps[i] * decay, op - ps[i] * decay
        assert np.max(np.abs(upd_gpu - upd_cpu)) <= (5e-2 if bf16 else 2e-3) * np.max(np.abs(upd_cpu)), i
        if mirrors[i] is not None:
            assert np.array_equal(be.download(mirrors[i]), orc.to_bf16(got)), i


def test_batched_step_refuses_the_whole_batch(be):
    from ojas_amd.backend import NON_FINITE, MuonNs5Config, OjasError

    print("muon batched refusal", flush=True)
    r = np.random.default_rng(1)
    ps = [r.standard_normal((64, 32)).astype(np.float32) for _ in range(4)]
    gs = [r.standard_normal((64, 32)).astype(np.float32) for _ in range(4)]
    gs[2][5, 7] = np.nan
    dp, dg = [be.upload(x) for x in ps], [be.upload(x) for x in gs]
    dm = [be.zeros((64, 32)) for _ in range(4)]
    be.muon_ns5_step_batched(dp, dg, dm, MuonNs5Config.nanolab_default())
    with pytest.raises(OjasError) as e:
        be.sync()
    assert e.value.code == NON_FINITE and "muon_ns5_step" in str(e.value)
    for i in range(4):
        assert np.array_equal(be.download(dp[i]), ps[i]) and not be.download(dm[i]).any()


@pytest.mark.parametrize("rows,cols,count", [(64, 48, 2), (130, 70, 3), (768, 768, 6), (768, 3072, 2), (3072, 768, 2),
                                             (2048, 2048, 2), (2048, 2048, 1)])
def test_bf16_iteration_sums_in_the_store_pass_carry_the_separate_kernels_bits(be, rows, cols, count):
    """The bf16 iteration forms b A + c A^2 and a X + B X in the store passes of the products that
    feed them (`muon_fused_sums`, the default, for calls on more than one tensor): same roundings in
    the same order as the separate kernels, so parameters, momenta and bf16 copies are the same bits; and a NaN gradient leaves
    every tensor of the call untouched under either setting."""
    from ojas_amd.backend import BF16, NON_FINITE, MuonNs5Config, OjasError

    print(f"muon fused sums {count} x {rows}x{cols}", flush=True)
    r = np.random.default_rng(rows + 3 * cols + count)
    ps = [r.standard_normal((rows, cols)).astype(np.float32) * 0.1 for _ in range(count)]
    gs = [r.standard_normal((rows, cols)).astype(np.float32) * 0.03 for _ in range(count)]
    ms = [r.standard_normal((rows, cols)).astype(np.float32) * 0.01 for _ in range(count)]
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, 1)
    got = {}
    try:
        for fused in (1, 0):
            be.set_option("muon_fused_sums", fused)
            dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in gs], [be.upload(x) for x in ms]
            mirrors = [be.upload(np.zeros((rows, cols), np.float32), BF16) for _ in range(count)]
            be.muon_ns5_step_batched(dp, dg, dm, cfg, mirrors)
            be.sync()
            got[fused] = [be.download(t) for t in dp + dm + mirrors]
            # all or nothing
            bad = [g.copy() for g in gs]
            bad[-1][rows // 2, cols // 3] = np.nan
            dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in bad], [be.upload(x) for x in ms]
            be.muon_ns5_step_batched(dp, dg, dm, cfg, None)
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.code == NON_FINITE and "muon" in e.value.detail
            for t, want in zip(dp + dm, ps + ms):
                assert np.array_equal(be.download(t), want)
    finally:
        be.set_option("muon_fused_sums", 1)
    for a, b in zip(got[1], got[0]):
        assert np.array_equal(a, b)
    assert any(np.any(a != p) for a, p in zip(got[1][:count], ps))


@pytest.mark.parametrize("rows,cols,count,room,bf16", [(256, 256, 5, 2, 0), (96, 512, 7, 1, 1), (512, 96, 70, 64, 0)])
def test_list_step_takes_the_scratch_there_is(be, rows, cols, count, room, bf16):
    """`muon_ns5_step_list` with room for the scratch of `room` matrices: as many at a time, each held to the oracle."""
    from ojas_amd.backend import CAPACITY_EXCEEDED, MiBackend, MuonNs5Config, OjasError

    print(f"muon list {count} x {rows}x{cols}, room for {room}", flush=True)
    r = np.random.default_rng(rows + count)
    ps, gs, ms = ([r.standard_normal((rows, cols)).astype(np.float32) * s for _ in range(count)] for s in (0.1, 0.05, 0.01))
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, bf16)
    each = int(be._lib.omx_muon_scratch_bytes(rows, cols))
    rounded = (each * room + (1 << 20) - 1) >> 20 << 20
    small = MiBackend(0, budget_bytes=3 * count * rows * cols * 4 + rounded)
    dp, dg, dm = [small.upload(x) for x in ps], [small.upload(x) for x in gs], [small.upload(x) for x in ms]
    if room < min(count, 64):
        with pytest.raises(OjasError) as e:  # all of them at once do not fit
            small.muon_ns5_step_batched(dp, dg, dm, cfg)
        assert e.value.code == CAPACITY_EXCEEDED
    small.muon_ns5_step_list(dp, dg, dm, cfg)
    decay = np.float32(1.0 - 0.02 * 0.1)
    for i in sorted({0, room - 1, room % count, count - 1}):
        op, om = orc.muon_ns5_step(ps[i], gs[i], ms[i], lr=0.02, momentum=0.95, weight_decay=0.1, nesterov=True, bf16=bool(bf16))
        assert np.array_equal(small.download(dm[i]), om), i
        upd_gpu, upd_cpu = small.download(dp[i]) - ps[i] * decay, op - ps[i] * decay
        assert np.max(np.abs(upd_gpu - upd_cpu)) <= (5e-2 if bf16 else 2e-3) * np.max(np.abs(upd_cpu)), i
    small.close()


@pytest.mark.parametrize("rows,cols,bf16", [(64, 48, 0), (130, 70, 1), (256, 256, 0), (256, 256, 1)])
def test_list_step_refuses_each_matrix_by_itself(be, rows, cols, bf16):
    """A gradient that is not finite, a momentum that is not, and a matrix whose norm overflows keep their own matrix as
    it was; the others step as they do without them."""
    from ojas_amd.backend import NON_FINITE, MuonNs5Config, OjasError

    print(f"muon list refusals {rows}x{cols} bf16={bf16}", flush=True)
    r = np.random.default_rng(rows)
    ps, gs, ms = ([r.standard_normal((rows, cols)).astype(np.float32) * s for _ in range(6)] for s in (0.1, 0.05, 0.01))
    bad_g, bad_m = [g.copy() for g in gs], [m.copy() for m in ms]
    bad_g[0][3, 5] = np.nan
    bad_m[2][-1, -1] = np.inf
    bad_g[4][:] = 3e38
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, bf16)
    out = []
    for g, m in ((gs, ms), (bad_g, bad_m)):
        dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in g], [be.upload(x) for x in m]
        be.muon_ns5_step_list(dp, dg, dm, cfg)
        if g is bad_g:
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.code == NON_FINITE and "muon_ns5_step" in str(e.value)
        out.append([(be.download(p), be.download(m)) for p, m in zip(dp, dm)])
    for i in range(6):
        if i in (0, 2, 4):
            assert np.array_equal(out[1][i][0], ps[i]) and np.array_equal(out[1][i][1], bad_m[i]), i
        else:
            assert np.array_equal(out[1][i][0], out[0][i][0]) and np.array_equal(out[1][i][1], out[0][i][1]), i


def test_a_model_of_many_matrices_steps_within_its_budget():
    """84 matrices of 512 x 512: 64 of them at once are 403 MB of scratch, one is 6.3."""
    from ojas_amd.backend import MiBackend
    from ojas_amd.nanolab import NanolabSpec, NanolabTrainer

    print("muon: 84 matrices under a budget", flush=True)
    be = MiBackend(0, budget_bytes=480 << 20)
    spec = NanolabSpec(n_layer=12, n_embd=512, n_head=8, n_kv_head=8, head_dim=64, hidden=512, vocab=256, window=None, max_seq=16)
    r = np.random.default_rng(2)
    host = {n: (r.standard_normal(s) * 0.02 if len(s) == 2 else np.ones(s)).astype(np.float32) for n, s in spec.param_shapes().items()}
    tr = NanolabTrainer(be, spec, host)
    ids = r.integers(0, 256, (1, 16)).astype(np.uint32)
    assert np.isfinite(tr.run([(ids, ids)], 0.1).loss)
    del tr
    be.close()


@pytest.mark.parametrize("rows,cols,count", [(1, 5, 1), (63, 48, 2), (130, 70, 3), (256, 704, 8), (704, 256, 4), (64, 256, 8), (768, 768, 1),
                                             (1024, 300, 1), (2000, 90, 1)])
def test_f32_iteration_sums_in_the_store_pass_carry_the_separate_kernels_bits(be, rows, cols, count):
    """The same of the f32 iteration, a single tensor's split reductions (whose last pass adds) and odd widths included."""
    from ojas_amd.backend import NON_FINITE, MuonNs5Config, OjasError

    print(f"muon f32 fused sums {count} x {rows}x{cols}", flush=True)
    r = np.random.default_rng(rows + 3 * cols + count)
    ps, gs, ms = ([(r.standard_normal((rows, cols)) * size).astype(np.float32) for _ in range(count)] for size in (0.1, 0.03, 0.01))
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, 0)
    got = {}
    try:
        for fused in (1, 0):
            be.set_option("muon_fused_sums", fused)
            dp, dg, dm = ([be.upload(x) for x in xs] for xs in (ps, gs, ms))
            be.muon_ns5_step_batched(dp, dg, dm, cfg, None)
            be.sync()
            got[fused] = [be.download(t) for t in dp + dm]
            bad = [g.copy() for g in gs]
            bad[-1][rows // 2, cols // 3] = np.inf
            dp, dg, dm = ([be.upload(x) for x in xs] for xs in (ps, bad, ms))
            be.muon_ns5_step_batched(dp, dg, dm, cfg, None)
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.code == NON_FINITE and "muon" in e.value.detail
            for t, want in zip(dp + dm, ps + ms):
                assert np.array_equal(be.download(t), want)
    finally:
        be.set_option("muon_fused_sums", 1)
    for a, b in zip(got[1], got[0]):
        assert np.array_equal(a, b)
    assert any(np.any(a != p) for a, p in zip(got[1][:count], ps))


# (rows, cols, tensors) of a call; widths off the 32 x 32 tile and off the 16-column step of K, more shapes than a launch takes products
# of, more tensors than a launch takes, and shapes that keep their own launches (130 x 70).
MIXES = [
    [(256, 256, 3), (128, 256, 2), (4, 256, 2), (704, 256, 2), (256, 704, 1)],
    [(64, 48, 2), (36, 100, 1), (100, 36, 1), (130, 70, 2), (4, 4, 1), (4, 32, 1), (32, 4, 1), (12, 20, 1), (8, 72, 1), (60, 60, 1), (68, 44, 1)],
    [(32, 32, 50), (32, 64, 30)],
]
# f32: third products of many shapes and tiles that are too short for 64 x 64 ones (LARGE_TILES), and on 64 x 64 tiles that end inside
# one, over six, seven and eight steps of K, beside some on 32 x 32 (LONG_TILES). (The bf16
# iteration has launches of its own for each shape. Its gate is not meant for these: a 96 x 100 matrix of random values has singular
# values from some 0.01 of its largest, which five iterations raise by up to 3.4 each with every operand rounded to 2^-9.)
LARGE_TILES = [(96, 100, 16), (100, 96, 12), (224, 32, 8), (32, 224, 2), (4, 100, 2), (60, 52, 3)]
LONG_TILES = [(192, 200, 10), (200, 192, 5), (224, 292, 2), (292, 256, 2), (160, 200, 3), (4, 100, 2)]


@pytest.mark.parametrize("mix,bf16", [(mix, bf16) for bf16 in (0, 1) for mix in MIXES] + [(LARGE_TILES, 0), (LONG_TILES, 0)])
def test_shapes_step_matches_the_oracle_per_tensor(be, mix, bf16):
    """`muon_ns5_step_shapes` at the single op's gates (momentum bit for bit; update 2e-3 of its largest element in f32,
    5e-2 with the bf16 iteration), tensors of one shape apart from each other in the call."""
    from ojas_amd.backend import BF16, MuonNs5Config

    print(f"muon shapes {mix} bf16={bf16}", flush=True)
    r = np.random.default_rng(len(mix))
    dims = [(rows, cols) for rows, cols, n in mix for _ in range(n)]
    dims = [dims[i] for i in r.permutation(len(dims))]
    ps, gs, ms = ([(r.standard_normal(d) * size).astype(np.float32) for d in dims] for size in (0.1, 0.05, 0.01))
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, bf16)
    dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in gs], [be.upload(x) for x in ms]
    mirrors = [be.upload(np.zeros(d, np.float32), BF16) if i % 2 == 0 else None for i, d in enumerate(dims)]
    be.muon_ns5_step_shapes(dp, dg, dm, cfg, mirrors)
    be.sync()
    orc.set_threads(8)
    decay = np.float32(1.0 - 0.02 * 0.1)
    for i in range(len(dims)):
        op, om = orc.muon_ns5_step(ps[i], gs[i], ms[i], lr=0.02, momentum=0.95, weight_decay=0.1, nesterov=True, bf16=bool(bf16))
        assert np.array_equal(be.download(dm[i]), om), dims[i]
        got = be.download(dp[i])
        upd_gpu, upd_cpu = got - ps[i] * decay, op - ps[i] * decay
        assert np.max(np.abs(upd_gpu - upd_cpu)) <= (5e-2 if bf16 else 2e-3) * np.max(np.abs(upd_cpu)), dims[i]
        if mirrors[i] is not None:
            assert np.array_equal(be.download(mirrors[i]), orc.to_bf16(got)), dims[i]


def test_shapes_step_refuses_each_matrix_by_itself(be):
    """As the list's test, across shapes; and a configuration or a shape that is refused steps nothing."""
    from ojas_amd.backend import NON_FINITE, OUT_OF_RANGE, SHAPE, MuonNs5Config, OjasError

    print("muon shapes refusals", flush=True)
    r = np.random.default_rng(8)
    dims = [(64, 48), (32, 96), (64, 48), (130, 70), (96, 32), (32, 96)]
    ps, gs, ms = ([(r.standard_normal(d) * s).astype(np.float32) for d in dims] for s in (0.1, 0.05, 0.01))
    bad_g, bad_m = [g.copy() for g in gs], [m.copy() for m in ms]
    bad_g[0][3, 5] = np.nan
    bad_m[3][-1, -1] = np.inf
    bad_g[5][:] = 3e38
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, 0)
    out = []
    for g, m in ((gs, ms), (bad_g, bad_m)):
        dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in g], [be.upload(x) for x in m]
        be.muon_ns5_step_shapes(dp, dg, dm, cfg)
        if g is bad_g:
            with pytest.raises(OjasError) as e:
                be.sync()
            assert e.value.code == NON_FINITE and "muon_ns5_step" in str(e.value)
        out.append([(be.download(p), be.download(m)) for p, m in zip(dp, dm)])
    for i in range(6):
        if i in (0, 3, 5):
            assert np.array_equal(out[1][i][0], ps[i]) and np.array_equal(out[1][i][1], bad_m[i]), i
        else:
            assert np.array_equal(out[1][i][0], out[0][i][0]) and np.array_equal(out[1][i][1], out[0][i][1]), i
    dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in gs], [be.upload(x) for x in ms]
    with pytest.raises(OjasError) as e:
        be.muon_ns5_step_shapes(dp, dg, dm, MuonNs5Config(-0.1, 0.9, 0.0, 1, 0))
    assert e.value.code == OUT_OF_RANGE
    with pytest.raises(OjasError) as e:
        be.muon_ns5_step_shapes(dp, [dg[1]] + dg[1:], dm, cfg)
    assert e.value.code == SHAPE
    be.sync()
    assert all(np.array_equal(be.download(d), p) for d, p in zip(dp + dm, ps + ms))


def test_shapes_step_takes_the_scratch_there_is():
    """Room for the scratch of the largest two tensors of seven: two or three at a time, each held to the oracle."""
    from ojas_amd.backend import MiBackend, MuonNs5Config

    print("muon shapes under a budget", flush=True)
    r = np.random.default_rng(3)
    dims = [(256, 512), (256, 256), (256, 512), (256, 256), (512, 256), (128, 512), (256, 256)]
    ps, gs, ms = ([(r.standard_normal(d) * s).astype(np.float32) for d in dims] for s in (0.1, 0.05, 0.01))
    small = MiBackend(0, budget_bytes=3 * 4 * sum(a * b for a, b in dims) + (6 << 20))
    dp, dg, dm = [small.upload(x) for x in ps], [small.upload(x) for x in gs], [small.upload(x) for x in ms]
    small.muon_ns5_step_shapes(dp, dg, dm, MuonNs5Config(0.02, 0.95, 0.1, 1, 0))
    decay = np.float32(1.0 - 0.02 * 0.1)
    for i in range(len(dims)):
        op, om = orc.muon_ns5_step(ps[i], gs[i], ms[i], lr=0.02, momentum=0.95, weight_decay=0.1, nesterov=True, bf16=False)
        assert np.array_equal(small.download(dm[i]), om), i
        upd_gpu, upd_cpu = small.download(dp[i]) - ps[i] * decay, op - ps[i] * decay
        assert np.max(np.abs(upd_gpu - upd_cpu)) <= 2e-3 * np.max(np.abs(upd_cpu)), i
    small.close()


@pytest.mark.parametrize("dim,same", [(128, True), (160, True), (192, False)])
def test_products_below_192_keep_their_tiles_whatever_the_count(be, dim, same):
    """64 x 64 tiles, whose sums over a short K are less exact than those of 32 x 32 ones, are for K >= 192: below, a matrix steps to
    the same bits among forty of its shape as among two."""
    from ojas_amd.backend import MuonNs5Config

    print(f"muon shapes {dim}", flush=True)
    r = np.random.default_rng(dim)
    cfg, got = MuonNs5Config(0.02, 0.95, 0.1, 1, 0), []
    many = [(dim, dim)] * 40 + [(32, 36)]
    ps, gs, ms = ([(r.standard_normal(d) * s).astype(np.float32) for d in many] for s in (0.1, 0.05, 0.01))
    for part in (slice(0, 41), slice(39, 41)):
        dp, dg, dm = ([be.upload(x) for x in xs[part]] for xs in (ps, gs, ms))
        be.muon_ns5_step_shapes(dp, dg, dm, cfg)
        got.append(be.download(dp[-2]))
    assert np.array_equal(*got) == same


@pytest.mark.parametrize("option,value", [("gemm_f32", 2), ("gemm_dma", 0)])
def test_a_forced_kernel_takes_the_products_of_several_shapes_too(be, option, value):
    """Under an option that forces a tile or the register-staged kernel, each shape's products go out as they do in a list of its own."""
    from ojas_amd.backend import MuonNs5Config

    print(f"muon shapes {option}={value}", flush=True)
    r = np.random.default_rng(value)
    dims = [(64, 48), (36, 100), (64, 48)]
    ps, gs, ms = ([(r.standard_normal(d) * s).astype(np.float32) for d in dims] for s in (0.1, 0.05, 0.01))
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, 0)
    launches = C.c_uint64()
    be.set_option(option, value)
    try:
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(1)))
        got = [[be.upload(x) for x in xs] for xs in (ps, gs, ms)]
        be.muon_ns5_step_shapes(*got, cfg)
        be._check(be._lib.omx_profile_gemm_report(be._ctx, C.byref(launches), None, None))
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
        for shape in ((0, 2), (1,)):
            want = [[be.upload(xs[i]) for i in shape] for xs in (ps, gs, ms)]
            be.muon_ns5_step_list(*want, cfg)
            assert all(np.array_equal(be.download(got[0][i]), be.download(p)) for i, p in zip(shape, want[0]))
    finally:
        be._check(be._lib.omx_profile_gemm(be._ctx, C.c_int32(0)))
        be.set_option(option, -1 if option == "gemm_f32" else 1)
    assert launches.value == 2 * 15


@pytest.mark.parametrize("tiling", [1, 3, 4, 7, 8])
@pytest.mark.parametrize("rows,cols,count", [(128, 128, 2), (192, 320, 3), (320, 192, 3), (448, 448, 2), (456, 576, 2), (64 * 11, 128, 4), (768, 1024, 2)])
def test_half_formed_symmetric_products_carry_the_whole_ones_bits(be, rows, cols, count, tiling):
    """X X^T and b A + c A^2 of a bf16 batch form one half and store it twice (`muon_symmetric`, the default): element (j, i) sums the
    products of element (i, j) in the same order, so every bit is that of products formed whole, on every tiling, at its edges."""
    from ojas_amd.backend import BF16, MuonNs5Config

    print(f"muon symmetric {count} x {rows}x{cols}, tiling {tiling}", flush=True)
    r = np.random.default_rng(rows + 5 * cols + count)
    ps = [r.standard_normal((rows, cols)).astype(np.float32) * 0.1 for _ in range(count)]
    gs = [r.standard_normal((rows, cols)).astype(np.float32) * 0.03 for _ in range(count)]
    ms = [r.standard_normal((rows, cols)).astype(np.float32) * 0.01 for _ in range(count)]
    got = {}
    try:
        be.set_option("gemm_dma", tiling)
        for symmetric in (1, 0):
            be.set_option("muon_symmetric", symmetric)
            dp, dg, dm = [be.upload(x) for x in ps], [be.upload(x) for x in gs], [be.upload(x) for x in ms]
            mirrors = [be.upload(np.zeros((rows, cols), np.float32), BF16) for _ in range(count)]
            be.muon_ns5_step_batched(dp, dg, dm, MuonNs5Config(0.02, 0.95, 0.1, 1, 1), mirrors)
            be.sync()
            got[symmetric] = [be.download(t) for t in dp + dm + mirrors]
    finally:
        be.set_option("muon_symmetric", 1)
        be.set_option("gemm_dma", 1)
    for a, b in zip(got[1], got[0]):
        assert np.array_equal(a, b)
    assert any(np.any(a != p) for a, p in zip(got[1][:count], ps))


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 3), (3, 5), (33, 50), (64, 48), (97, 97), (515, 1030)])
def test_tensors_off_16_bytes_carry_the_aligned_ones_bits(be, rows, cols, bf16):
    """The passes around the iteration take four elements a lane where the tensors lie on 16 bytes, else one, and the last elements of a
    count that is no multiple of four by themselves: the same bits, and nothing behind the tensors."""
    from ojas_amd.backend import BF16, F32, DeviceTensor, MuonNs5Config

    print(f"muon off 16 bytes {rows}x{cols} bf16 {bf16}", flush=True)
    r = np.random.default_rng(rows + 3 * cols)
    n = rows * cols
    p, g, m = (r.standard_normal(n).astype(np.float32) * k for k in (0.1, 0.03, 0.01))
    got = []
    for lead in (0, 1, 2):
        def at(x, dtype):
            whole = be.upload(np.concatenate([np.full(lead, 7.0, np.float32), x, np.full(9, 7.0, np.float32)]), dtype)
            return whole, DeviceTensor(be, whole.ptr + lead * (2 if dtype == BF16 else 4), (rows, cols), dtype, owns=False)

        held = [at(p, F32), at(g, F32), at(m, F32), at(np.zeros(n, np.float32), BF16)]
        tensors = [t for _, t in held]
        be.muon_ns5_step_batched([tensors[0]], [tensors[1]], [tensors[2]], MuonNs5Config(0.02, 0.95, 0.1, 1, bf16), [tensors[3]])
        be.sync()
        parts = [be.download_f32(whole) for whole, _ in held]
        assert all(np.all(x[:lead] == 7.0) and np.all(x[lead + n:] == 7.0) for x in parts)
        got.append([x[lead:lead + n] for x in parts])
    assert not np.array_equal(got[0][0], p)
    assert np.array_equal(got[0][1], g)
    for other in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got[0], other))
