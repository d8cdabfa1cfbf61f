"""Passes over tensors larger than the memory-side cache, which read (and some write) past the caches, against the same
op on pieces small enough not to: an element's arithmetic does not depend on how its tensor is loaded, so the bits are
the same (attention over a cache parts its keys by the number of rows, and is held to f32 rounding)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    backend = MiBackend(0)
    yield backend
    backend.close()


@pytest.mark.parametrize("n", [1 << 24, (1 << 24) + 3])  # the first size that is streamed; a tail that is not whole packs
def test_adamw_over_a_large_arena(be, n):
    from ojas_amd.backend import BF16, F32, AdamWConfig

    print(f"adamw {n}", flush=True)
    r = np.random.default_rng(n)
    cfg, cut = AdamWConfig(3e-4, 0.9, 0.95, 1e-8, 0.1), n // 8 * 4
    host = [r.standard_normal(n, dtype=np.float32) * s for s in (0.1, 0.01, 0.01)] + [r.random(n, dtype=np.float32) * 1e-3]
    whole = [be.upload(x) for x in host]
    copy = be.zeros((n,), BF16)
    be.adamw_step(*whole, 3, cfg, copy)
    parts = [[be.upload(x[a:b]) for x in host] for a, b in ((0, cut), (cut, n))]
    copies = [be.zeros((b - a,), BF16) for a, b in ((0, cut), (cut, n))]
    for p, c in zip(parts, copies):
        be.adamw_step(*p, 3, cfg, c)
    for i in (0, 2, 3):
        assert np.array_equal(be.download(whole[i]), np.concatenate([be.download(p[i]) for p in parts])), i
    assert np.array_equal(be.download(copy), np.concatenate([be.download(c) for c in copies]))
    assert whole[0].dtype == F32


@pytest.mark.parametrize("rows,hidden,bf16", [(8192, 6144, False), (8192, 6152, False), (12288, 8192, True), (8192, 4608, False),
                                              (8192, 4600, False)])  # last: the first size whose forward is streamed, and one under it
def test_swiglu_over_a_large_projection(be, rows, hidden, bf16):
    from ojas_amd.backend import BF16, F32

    print(f"swiglu {rows}x{hidden} bf16={bf16}", flush=True)
    r = np.random.default_rng(hidden)
    x = r.standard_normal((64, 2 * hidden), dtype=np.float32)
    x = np.concatenate([x * (0.1 + k / 40) for k in range(rows // 64)])
    gy = r.standard_normal((rows, hidden), dtype=np.float32)
    dtype, cut = BF16 if bf16 else F32, rows // 8
    dx, dg = be.upload(x, dtype), be.upload(gy, BF16)
    out, back = be.download(be.swiglu_forward(dx)), be.download(be.swiglu_backward(dx, dg))
    for a in range(0, rows, cut):
        px, pg = be.upload(x[a:a + cut], dtype), be.upload(gy[a:a + cut], BF16)
        assert np.array_equal(out[a:a + cut], be.download(be.swiglu_forward(px))), a
        assert np.array_equal(back[a:a + cut], be.download(be.swiglu_backward(px, pg))), a


@pytest.mark.parametrize("rows,vocab", [(4096, 50304), (4001, 50301)])
def test_loss_over_a_large_tile_of_logits(be, rows, vocab):
    """One tile of all rows against tiles of 512: the loss is summed over rows in one order, a row's gradient over the
    vocabulary in one order whatever the tile (the products choose their tilings by rows: f32 rounding)."""
    from ojas_amd.backend import BF16, U32

    print(f"loss {rows}x{vocab}", flush=True)
    r = np.random.default_rng(vocab)
    dim = 64
    x, w = be.upload(r.standard_normal((rows, dim), dtype=np.float32), BF16), be.upload(r.standard_normal((vocab, dim), dtype=np.float32) * 0.2, BF16)
    t = r.integers(0, vocab, rows).astype(np.uint32)
    t[5] = 7
    targets = be.upload(t, U32)
    got = be.linear_cross_entropy_mean(x, w, targets, ignore_index=7, chunk=(rows, vocab))
    want = be.linear_cross_entropy_mean(x, w, targets, ignore_index=7, chunk=(512, vocab))
    assert np.array_equal(be.download(got[0]), be.download(want[0]))
    for a, b in zip(got[1:], want[1:]):
        a, b = be.download(a), be.download(b)
        assert np.linalg.norm(a - b) <= 2e-6 * np.linalg.norm(b)
    assert not be.download(got[1])[5].any()


@pytest.mark.parametrize("b,heads,dim,kv_len,bf16", [(44, 12, 64, 512, False), (88, 12, 64, 511, True), (1200, 4, 64, 64, False), (24, 8, 128, 700, False),
                                                     (300, 16, 16, 900, False)])
def test_decoding_over_large_caches(be, b, heads, dim, kv_len, bf16):
    from ojas_amd.backend import BF16

    print(f"decode {b}x{heads}x{dim} {kv_len} bf16={bf16}", flush=True)
    r = np.random.default_rng(b)
    q = r.standard_normal((b, 1, heads, dim), dtype=np.float32)
    k, v = (r.standard_normal((b, kv_len, heads, dim), dtype=np.float32) for _ in range(2))
    up = lambda x: be.upload(x, BF16) if bf16 else be.upload(x)
    got = be.download(be.cached_attention_forward(be.upload(q), up(k), up(v), kv_len))
    for a in range(0, b, b // 4):
        part = be.download(be.cached_attention_forward(be.upload(q[a:a + b // 4]), up(k[a:a + b // 4]), up(v[a:a + b // 4]), kv_len))
        assert np.linalg.norm(got[a:a + b // 4] - part) <= 1e-6 * np.linalg.norm(part)
    if not bf16:
        v[-1, 3, -1, 5] = np.nan
        be.cached_attention_forward(be.upload(q), up(k), up(v), kv_len)
        from ojas_amd.backend import OjasError
        with pytest.raises(OjasError):
            be.sync()


def test_muon_over_large_batches(be):
    from ojas_amd.backend import MuonNs5Config

    print("muon 17 x 1024 x 1000", flush=True)
    r = np.random.default_rng(4)
    dims, n = (1024, 1000), 17
    ps, gs, ms = ([r.standard_normal(dims, dtype=np.float32) * s for _ in range(n)] for s in (0.1, 0.05, 0.01))
    cfg = MuonNs5Config(0.02, 0.95, 0.1, 1, 1)
    got, want = [], []
    for out, step in ((got, n), (want, 6)):
        dp, dg, dm = ([be.upload(x) for x in xs] for xs in (ps, gs, ms))
        for a in range(0, n, step):
            be.muon_ns5_step_batched(dp[a:a + step], dg[a:a + step], dm[a:a + step], cfg)
        be.sync()
        out.extend(be.download(x) for x in dp + dm)
    for i in range(n, 2 * n):
        assert np.array_equal(got[i], want[i]), i
    for i in range(n):  # the products' tilings go by the batch: bf16 roundings of the iterate differ
        assert np.linalg.norm(got[i] - want[i]) <= 2e-3 * np.linalg.norm(want[i] - ps[i]), i
