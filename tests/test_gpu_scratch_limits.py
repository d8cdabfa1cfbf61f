"""Ops at the limits of their scratch memory: a full device or budget, and inside a captured graph."""
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


def test_a_refused_allocation_leaves_the_next_op_alone(be):
    """More memory than the device has: the refusal is that call's own, and no later launch reports it."""
    from ojas_amd.backend import CAPACITY_EXCEEDED, OjasError

    print("allocation of 64 TiB", flush=True)
    x = be.upload(np.ones((4, 64), np.float32))
    with pytest.raises(OjasError) as e:
        be.empty((1 << 44,))
    assert e.value.code == CAPACITY_EXCEEDED
    assert np.array_equal(be.download(be.residual_add_forward(x, x)), np.full((4, 64), 2.0, np.float32))


class Graph:
    """What `record()` launches on a backend's stream, captured (relaxed, so that it may allocate its results, which it returns)."""

    def __init__(self, be, record):
        self.hip, self.stream = be._lib, C.c_void_p(be.stream())
        self.graph, self.program = C.c_void_p(), C.c_void_p()
        assert self.hip.hipStreamBeginCapture(self.stream, C.c_int(2)) == 0
        self.results = record()
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.program), self.graph, None, None, C.c_size_t(0)) == 0

    def launch(self):
        assert self.hip.hipGraphLaunch(self.program, self.stream) == 0

    def close(self):
        self.hip.hipGraphExecDestroy(self.program)
        self.hip.hipGraphDestroy(self.graph)


def test_what_a_capture_freed_is_for_captures_only():
    """A graph writes its temporaries whenever it is replayed: their blocks go to no eager allocation, not into the pool and, where the
    device refuses an allocation, not back to it. A later capture takes them, and what it keeps of them and is freed afterwards is held
    likewise."""
    from ojas_amd.backend import MiBackend, OjasError

    be = MiBackend(0)
    n, large = (1 << 16) + 64, (256 << 18) + 64  # the second above the largest block that is parked
    x, z = be.upload(np.full((n,), 1.5, np.float32)), be.zeros((large,))
    inner = []

    def record(t):
        a = be.residual_add_forward(t, t)
        inner.append(a.ptr)
        return be.residual_add_forward(a, t)

    for t, want in ((x, 4.5), (z, 0.0)):
        inner.clear()
        print(f"graph with a temporary of {t.nbytes} bytes", flush=True)
        pooled, live = be.budget()["pooled"], be.budget()["live"]
        graph = Graph(be, lambda: record(t))
        assert be.budget()["pooled"] == pooled and be.budget()["live"] == live + t.nbytes
        others = [be.empty(t.shape) for _ in range(2)]
        assert inner[0] not in [o.ptr for o in others], "the temporary's block went to an eager allocation"
        sevens = np.full(t.shape, 7.0, np.float32)
        for o in others:
            load(be, o, sevens)
        graph.launch()
        assert all(np.array_equal(be.download(o), sevens) for o in others)
        print("a refused allocation", flush=True)
        del others
        with pytest.raises(OjasError):
            be.empty((1 << 44,))
        assert be.budget()["pooled"] == 0
        for _ in range(3):
            load(be, graph.results, np.full(t.shape, np.nan, np.float32))
            graph.launch()
            assert np.array_equal(be.download(graph.results), np.full(t.shape, want, np.float32))
        print("a second graph", flush=True)
        second = Graph(be, lambda: be.residual_add_forward(t, t))  # its result is the first one's temporary
        assert second.results.ptr == inner[0]
        second.launch()
        assert np.array_equal(be.download(second.results), np.full(t.shape, 2.0 * want / 3.0, np.float32))
        second.close()
        second.results = None
        assert be.empty(t.shape).ptr != inner[0]
        graph.close()
        del graph
    be.close()


def load(be, tensor, values):
    be._check(be._lib.omx_upload(be._ctx, be._p(tensor), C.c_uint64(0), values.ctypes.data_as(C.c_void_p), C.c_uint64(values.nbytes)))


def test_a_captured_graph_keeps_the_scratch_it_was_recorded_with():
    """A later call that needs more takes a block of its own: the graph's stays where it was, and its replays stay right while
    that call's scratch is written in between."""
    from ojas_amd.backend import MiBackend

    print("captured argmax, then a norm with more scratch", flush=True)
    be = MiBackend(0)
    r = np.random.default_rng(1)
    x = be.zeros((2, 50257))
    rows = [be.upload(r.standard_normal((4096, 4096)).astype(np.float32)) for _ in range(2)]
    w = be.upload(np.ones(4096, np.float32))
    be.argmax_rows(x)  # grows the workspace: 1 MiB
    graph = Graph(be, lambda: be.argmax_rows(x))
    be.sync()
    live = be.budget()["live"]
    norm = be.rms_norm_backward(rows[0], w, rows[1])  # 288 rows of partial sums: 5 MiB
    assert be.budget()["live"] == live + sum(t.nbytes for t in norm) + (5 << 20)
    want = be.download(norm[1])
    for _ in range(4):
        values = r.standard_normal((2, 50257)).astype(np.float32)
        load(be, x, values)
        graph.launch()
        assert np.array_equal(be.download(graph.results), np.argmax(values, axis=1).astype(np.uint32))
        assert np.array_equal(be.download(be.rms_norm_backward(rows[0], w, rows[1])[1]), want)
    graph.close()
    be.close()


def test_scratch_that_grows_inside_a_capture_leaves_the_smaller_block():
    """An op that cannot do without: the capture ends well, the block from before it stays, and so does the new one after it."""
    from ojas_amd.backend import MiBackend

    print("norm backward captured over a smaller workspace", flush=True)
    be = MiBackend(0)
    r = np.random.default_rng(3)
    x, gy = (r.standard_normal((4096, 4096)).astype(np.float32) for _ in range(2))
    w = np.ones(4096, np.float32)
    held = [be.upload(a) for a in (x, w, gy)]
    be.argmax_rows(be.zeros((1, 20000)))  # 1 MiB
    live = be.budget()["live"]
    graph = Graph(be, lambda: be.rms_norm_backward(*held))
    assert be.budget()["live"] == live + sum(t.nbytes for t in graph.results) + (5 << 20)
    want = orc.rms_norm_backward(x, w, gy)
    for _ in range(3):
        for t in graph.results:
            load(be, t, np.full(t.shape, np.nan, np.float32))
        graph.launch()
        for a, b in zip(graph.results, want):
            assert np.max(np.abs(be.download(a) - b)) <= 1e-5 * max(1.0, float(np.max(np.abs(b))))
        be.argmax_rows(be.zeros((1, 20000)))
    graph.close()
    be.close()


def with_less(op, arrays, mib):
    """`op`'s results in a budget that lacks `mib` MiB of what it takes where nothing is scarce."""
    from ojas_amd.backend import MiBackend

    wide = MiBackend(0)
    results = op(wide, *[wide.upload(a) for a in arrays])
    peak = wide.budget()["peak"]
    del results
    wide.close()
    tight = MiBackend(0, budget_bytes=peak - (mib << 20))
    got = [tight.download(t) for t in op(tight, *[tight.upload(a) for a in arrays])]
    tight.close()
    return got


@pytest.mark.parametrize("rows,cols", [(1, 16384), (3, 20001), (16, 16384)])
def test_argmax_without_room_for_scratch(rows, cols):
    """Under a full budget, and first called in a capture (which takes nothing but the result)."""
    from ojas_amd.backend import MiBackend

    print(f"argmax {rows}x{cols} without scratch", flush=True)
    r = np.random.default_rng(cols)
    draw = lambda: r.integers(-1000, 1000, (rows, cols)).astype(np.float32)  # (ties)
    values = draw()
    (got,) = with_less(lambda be, x: (be.argmax_rows(x),), [values], 1)
    assert np.array_equal(got, np.argmax(values, axis=1).astype(np.uint32))
    be = MiBackend(0)
    x = be.upload(values)
    live = be.budget()["live"]
    graph = Graph(be, lambda: be.argmax_rows(x))
    assert be.budget()["live"] == live + graph.results.nbytes
    for _ in range(3):
        values = draw()
        load(be, x, values)
        graph.launch()
        want = np.argmax(values, axis=1).astype(np.uint32)
        assert np.array_equal(be.download(graph.results), want) and np.array_equal(be.download(be.argmax_rows(x)), want)
    graph.close()
    be.close()


def close(got, want):
    """Within the f32 tier's 1e-5 of the oracle."""
    assert np.max(np.abs(got - want)) <= 1e-5 * max(1.0, float(np.max(np.abs(want))))


@pytest.mark.parametrize("mib", [1, 2, 4])
def test_f32_attention_backward_with_room_for_fewer_parts(mib):
    """Sixteen parts of the rows are 4 MiB of scratch: with room for 3, for 2, for none."""
    print(f"f32 attention backward, {mib} MiB less", flush=True)
    r = np.random.default_rng(mib)
    q, k, v, gy = (r.standard_normal((1, heads, 512, 64)).astype(np.float32) for heads in (4, 1, 1, 4))
    orc.set_threads(8)
    out, lse = orc.causal_sdpa_forward(q, k, v)
    got = with_less(lambda be, *t: be.causal_sdpa_backward(*t), [q, k, v, out, lse, gy], mib)
    for a, b in zip(got, orc.causal_sdpa_backward(q, k, v, out, lse, gy)):
        close(a, b)


def test_f32_attention_backward_takes_no_scratch_for_parts_inside_a_capture():
    from ojas_amd.backend import MiBackend

    print("f32 attention backward, captured first", flush=True)
    r = np.random.default_rng(7)
    host = [r.standard_normal((1, heads, 512, 64)).astype(np.float32) for heads in (4, 1, 1, 4)]
    out, lse = orc.causal_sdpa_forward(*host[:3])
    want = orc.causal_sdpa_backward(*host[:3], out, lse, host[3])
    be = MiBackend(0)
    q, k, v, o, l, gy = (be.upload(a) for a in (*host[:3], out, lse, host[3]))
    small = [be.upload(a[:, :, :16]) for a in (*host[:3], out, lse, host[3])]
    be.causal_sdpa_backward(*small)  # the row term's scratch, 1 MiB
    live = be.budget()["live"]
    graph = Graph(be, lambda: be.causal_sdpa_backward(q, k, v, o, l, gy))
    assert be.budget()["live"] == live + sum(t.nbytes for t in graph.results)
    for _ in range(3):
        for t in graph.results:
            load(be, t, np.full(t.shape, np.nan, np.float32))
        graph.launch()
        for a, b in zip(graph.results, want):
            close(be.download(a), b)
        for a, b in zip(be.causal_sdpa_backward(q, k, v, o, l, gy), want):
            close(be.download(a), b)
    graph.close()
    be.close()


def test_attention_over_a_long_cache_takes_no_scratch_inside_a_capture():
    """16 new rows over 4096 positions: the keys' parts are left out where a capture would have to allocate them."""
    from ojas_amd.backend import MiBackend

    print("cached attention, captured first", flush=True)
    r = np.random.default_rng(8)
    q, k, v = (r.standard_normal(s).astype(np.float32) for s in ((1, 16, 2, 64), (1, 4096, 2, 64), (1, 4096, 2, 64)))
    want = orc.cached_attention_forward(q, k, v, 4096, 0)
    be = MiBackend(0)
    held = [be.upload(a) for a in (q, k, v)]
    live = be.budget()["live"]
    graph = Graph(be, lambda: be.cached_attention_forward(*held, 4096))
    assert be.budget()["live"] == live + graph.results.nbytes
    for _ in range(3):
        load(be, graph.results, np.full(q.shape, np.nan, np.float32))
        graph.launch()
        close(be.download(graph.results), want)
        close(be.download(be.cached_attention_forward(*held, 4096)), want)
    graph.close()
    be.close()


def test_norm_backward_with_room_for_fewer_partial_rows():
    """4000 x 2500: 250 partial rows are 3 MiB, 125 are 2."""
    print("norm backward 4000x2500, 1 MiB less", flush=True)
    r = np.random.default_rng(1)
    x, gy = (r.standard_normal((4000, 2500)).astype(np.float32) for _ in range(2))
    w = (1 + 0.1 * r.standard_normal(2500)).astype(np.float32)
    for a, b in zip(with_less(lambda be, *t: be.rms_norm_backward(*t), [x, w, gy], 1), orc.rms_norm_backward(x, w, gy)):
        close(a, b)


def test_gate_backward_with_room_for_fewer_partial_rows():
    """2800 rows of 256 heads: 7 MiB of scratch with 700 partial rows, 6 with 175."""
    print("gate backward 2800 x 256 heads, 1 MiB less", flush=True)
    r = np.random.default_rng(2)
    x, w, b = (0.3 * r.standard_normal(s).astype(np.float32) for s in ((2800, 32), (256, 32), (256,)))
    attn, gy = (r.standard_normal((2800, 256, 4)).astype(np.float32) for _ in range(2))
    got = with_less(lambda be, *t: be.per_head_sigmoid_gate_backward(*t), [x, w, b, attn, gy], 1)
    for a, c in zip(got, orc.gate_backward(x, w, b, attn, gy)):
        close(a, c)


def test_a_widened_weight_makes_room_for_what_is_allocated_next():
    # 2 MiB of bf16 weight in scratch; the budget then has room for the next tensor only without it.
    from ojas_amd.backend import BF16, F32, MiBackend

    rng = np.random.default_rng(3)
    x, codes = rng.normal(0, 1, (512, 1024)).astype(np.float32), rng.integers(-127, 128, (1024, 1024)).astype(np.int8)
    scales = rng.uniform(1e-4, 1e-3, (1024, 32)).astype(np.float32)
    be = MiBackend(0, budget_bytes=16 << 20)
    try:
        dx, dc, ds = be.upload(x, BF16), be.upload(codes), be.upload(scales)
        be.set_option("q8_widen", 0)
        want = be.download_f32(be.linear_i8_group_forward(dx, dc, ds))
        be.set_option("q8_widen", 1)
        held = be.budget()["live"]
        y = be.linear_i8_group_forward(dx, dc, ds)
        assert be.budget()["live"] - held >= 2 << 20
        rest = be.empty(((16 << 20) - be.budget()["live"] + (1 << 20)) // 4, F32)  # a MiB more than there is
        assert np.array_equal(be.download_f32(y), want)
        z = be.linear_i8_group_forward(dx, dc, ds)  # no room for the copy
        assert np.array_equal(be.download_f32(z), want)
        del rest
    finally:
        be.close()


def test_a_plan_does_not_depend_on_scratch_that_can_be_given_back():
    """A Muon list takes as many matrices at a time as the budget has room for, and as many after an int8 product has left its widened
    weight behind: the same scratch in the end, the same bits."""
    from ojas_amd.backend import BF16, MiBackend, MuonNs5Config

    print("muon list beside a widened weight", flush=True)
    r = np.random.default_rng(4)
    n, d = 8, (256, 512)
    ps, gs, ms = ([(r.standard_normal(d) * s).astype(np.float32) for _ in range(n)] for s in (0.1, 0.05, 0.01))
    x, codes = r.normal(0, 1, (64, 1024)).astype(np.float32), r.integers(-127, 128, (2048, 1024)).astype(np.int8)
    scales = r.uniform(1e-4, 1e-3, (2048, 32)).astype(np.float32)
    out = []
    for widened in (False, True):
        be = MiBackend(0, budget_bytes=3 * n * 4 * d[0] * d[1] + (14 << 20))  # five matrices' scratch
        try:
            if widened:
                be.set_option("q8_widen", 1)
                before = be.budget()["live"]
                be.linear_i8_group_forward(be.upload(x, BF16), be.upload(codes), be.upload(scales))
                be.sync()
                assert be.budget()["live"] - before == 4 << 20
            dp, dg, dm = ([be.upload(a) for a in xs] for xs in (ps, gs, ms))
            be.muon_ns5_step_list(dp, dg, dm, MuonNs5Config(0.02, 0.95, 0.1, 1, 0))
            out.append((be.budget()["live"], [be.download(t) for t in dp + dm]))
        finally:
            be.close()
    assert out[0][0] == out[1][0]
    assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))


def test_sums_that_wait_make_room_for_what_is_allocated_next():
    """The partial rows of a norm's weight gradient are scratch: an allocation that needs their room gets it, and the gradient is formed."""
    from ojas_amd.backend import F32, MiBackend

    print("an allocation while sums wait", flush=True)
    r = np.random.default_rng(5)
    be = MiBackend(0, budget_bytes=32 << 20)
    try:
        rows, dim = 2048, 512
        x, gy = (be.upload(r.standard_normal((rows, dim), dtype=np.float32)) for _ in range(2))
        w, gx, gw = be.upload(r.normal(1, 0.1, dim).astype(np.float32)), be.empty((rows, dim), F32), be.zeros((dim,))
        want = be.download(be.rms_norm_backward(x, w, gy, 1e-6)[1])
        held = be.budget()["live"]
        be._check(be._lib.omx_defer_weight_sums(be._ctx, C.c_uint32(64)))
        be._check(be._lib.omx_rms_norm_backward(
            be._ctx, be._p(x), C.c_int32(F32), be._p(w), be._p(gy), C.c_int32(F32), be._p(gx), C.c_int32(F32), be._p(gw), C.c_uint64(rows),
            C.c_uint64(dim), C.c_float(1e-6)))
        assert be.budget()["live"] - held >= 1 << 20
        rest = be.empty((((32 << 20) - be.budget()["live"] + (1 << 20)) // 4,), F32)  # a MiB more than there is
        be._check(be._lib.omx_form_weight_sums(be._ctx, C.c_int32(1)))
        assert np.array_equal(be.download(gw), want)
        del rest
    finally:
        be.close()


def test_a_full_pool_makes_room_for_a_size_that_comes_back():
    """Parked blocks of sizes no longer asked for go back to the device for one that is asked for again and again; the sizes of a
    round through more than the pool holds stay, and so does a block that a capture freed, which its graph still writes."""
    from ojas_amd.backend import MiBackend

    be = MiBackend(0)
    most = 4 << 30
    x = be.upload(np.full((1 << 16,), 1.5, np.float32))
    print("graph with a temporary", flush=True)
    graph = Graph(be, lambda: be.residual_add_forward(be.residual_add_forward(x, x), x))
    print("4 GiB parked", flush=True)
    held = [be.empty(((200 << 18) + 1024 * k,)) for k in range(21)]
    del held
    full = be.budget()["pooled"]
    assert most - (201 << 20) < full <= most
    held = [be.empty((n,)) for n in (1 << 25, 1 << 25)]  # up to less than 16 MiB below the limit, or nothing left to fill
    del held
    print("a size that comes back", flush=True)
    n = (200 << 18) - 1024
    seen = []
    for _ in range(4):
        t = be.empty((n,))
        seen.append(be.budget()["pooled"])
        del t
        assert be.budget()["pooled"] <= most
    assert seen[3] == be.budget()["pooled"] - 4 * n, "the fourth was not taken from the pool"
    for _ in range(3):
        graph.launch()
        assert np.array_equal(be.download(graph.results), np.full((1 << 16,), 4.5, np.float32))
    print("a size that went back to the device", flush=True)
    parked = be.budget()["pooled"]
    old = be.empty((200 << 18,))
    assert be.budget()["pooled"] == parked, "the pool still held the block that was asked for longest ago"
    del old
    print("a round through more than the pool holds", flush=True)
    sizes = [(160 << 18) + 1024 * k for k in range(32)]
    hits = 0
    for turn in range(3):
        held = []
        for m in sizes:
            before = be.budget()["pooled"]
            held.append(be.empty((m,)))
            hits += turn == 2 and be.budget()["pooled"] < before
        del held
    assert hits >= 20, "the pool gave up blocks that were about to be asked for"
    graph.close()
    be.close()


def test_attention_backward_without_room_for_shares_of_the_key_sums():
    """Scratch for the sums of a key block's workgroups that the budget refuses: one workgroup walks all tiles, to the same bits as
    where the option says so."""
    from ojas_amd.backend import BF16, MiBackend

    be = MiBackend(0, 16 << 20)
    rng = np.random.default_rng(5)
    q, k, v, gy = (be.upload(rng.normal(size=(1, n, 300, 64)).astype(np.float32), BF16) for n in (4, 1, 1, 4))
    out, lse = be.causal_sdpa_forward(q, k, v, None, BF16)
    be.set_option("flash_kv_parts", 1)
    whole = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
    be.set_option("flash_kv_parts", 5)  # 5 x 300 x 64 x 8 bytes
    grads = [be.empty(t.shape, BF16) for t in (q, k, v)]
    budget = be.budget()
    held = be.empty(((budget["limit"] - budget["live"] - (1 << 19)) // 4,))
    del grads
    split = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
    assert all(np.array_equal(a, e) for a, e in zip(split, whole))
    del held
    split = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
    assert not all(np.array_equal(a, e) for a, e in zip(split, whole))
    be.close()


def test_shares_of_the_key_sums_are_all_or_none():
    """Room for some of the shares only: the bits are those of one workgroup's walk, and not of as many shares as fit."""
    from ojas_amd.backend import BF16, MiBackend

    print("5 shares of 1.5 MiB, room for 4 MiB", flush=True)
    be = MiBackend(0, 64 << 20)
    rng = np.random.default_rng(6)
    q, k, v, gy = (be.upload(rng.normal(size=(1, n, 3072, 64)).astype(np.float32), BF16) for n in (4, 1, 1, 4))
    out, lse = be.causal_sdpa_forward(q, k, v, None, BF16)
    be.set_option("flash_schedule", 1)
    try:
        be.set_option("flash_kv_parts", 1)
        whole = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
        be.set_option("flash_kv_parts", 5)
        grads = [be.empty(t.shape, BF16) for t in (q, k, v)]
        budget = be.budget()
        held = be.empty(((budget["limit"] - budget["live"] - (4 << 20)) // 4,))
        del grads
        some = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
        assert all(np.array_equal(a, e) for a, e in zip(some, whole))
        del held
        split = [be.download_f32(g) for g in be.causal_sdpa_backward(q, k, v, out, lse, gy, None, BF16)]
        assert not all(np.array_equal(a, e) for a, e in zip(split, whole))
    finally:
        be.set_option("flash_schedule", 0)
        be.close()


@pytest.mark.parametrize("waits", [True, False])
def test_norm_backward_of_few_rows_asks_for_the_scratch_that_it_uses(waits):
    """768 x 1300: 192 partial rows that wait are a MiB, with the scratch of a sum that does not they are two. In a MiB the waiting sum has the
    bits it has where nothing is scarce, and the other goes without half of its rows."""
    from ojas_amd.backend import F32, MiBackend

    print(f"norm backward 768x1300, 1 MiB, waits {waits}", flush=True)
    r = np.random.default_rng(9)
    x, gy = (r.standard_normal((768, 1300)).astype(np.float32) for _ in range(2))
    w = r.normal(1, 0.1, 1300).astype(np.float32)
    got = []
    for mib in (0, 1):
        be = MiBackend(0, budget_bytes=64 << 20)
        try:
            dx, dgy, dw, gx, gw = be.upload(x), be.upload(gy), be.upload(w), be.empty(x.shape, F32), be.zeros((1300,))
            held = be.empty((((64 << 20) - be.budget()["live"] - (mib << 20)) // 4,)) if mib else None
            if waits:
                be._check(be._lib.omx_defer_weight_sums(be._ctx, C.c_uint32(1)))
            be._check(be._lib.omx_rms_norm_backward(
                be._ctx, be._p(dx), C.c_int32(F32), be._p(dw), be._p(dgy), C.c_int32(F32), be._p(gx), C.c_int32(F32), be._p(gw), C.c_uint64(768),
                C.c_uint64(1300), C.c_float(1e-6)))
            if waits:
                be._check(be._lib.omx_form_weight_sums(be._ctx, C.c_int32(1)))
            got.append((be.download(gx), be.download(gw)))
            del held
        finally:
            be.close()
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1]) == waits
    for gx, gw in got:
        want = orc.rms_norm_backward(x, w, gy)
        close(gx, want[0])
        close(gw, want[1])


@pytest.mark.parametrize("rows,kin,nout,rank", [(5, 256, 512, 0), (67, 1408, 1024, 16), (130, 1024, 1408, 0), (1042, 1280, 896, 16)])
def test_a_kept_copy_of_a_weight_gives_the_bits_of_a_copy_of_its_own(rows, kin, nout, rank):
    """`omx_i8_copy_next`: forward products leave their widened copies for the input gradients. The same bits as copies formed for each, with
    two weights in the scratch, after an allocation took it back (no copy is kept from then on), and with a mark that another block gave."""
    import ctypes as C

    from ojas_amd.backend import BF16, F32, MiBackend

    print(f"kept copies {rows} x {kin} -> {nout}, rank {rank}", flush=True)
    r = np.random.default_rng(rows + nout)
    weights = [(r.integers(-127, 128, (nout, kin)).astype(np.int8), r.uniform(1e-4, 1e-3, (nout, kin // 32)).astype(np.float32)) for _ in range(2)]
    xs, gs = (r.normal(0, 1, (rows, n)).astype(np.float32) for n in (kin, nout))
    size = (2 * nout * kin + 255) // 256 * 256
    budget = 96 << 20
    be = MiBackend(0, budget_bytes=budget)
    try:
        be.set_option("q8_widen", 1)
        ws = [tuple(be.upload(t) for t in w) for w in weights]
        x, g = be.upload(xs, BF16), be.upload(gs, BF16)
        tails = [None, None]
        if rank:
            tails = [tuple(be.upload(r.normal(0, 0.1, (n, rank)).astype(np.float32), BF16) for n in (rows, cols)) + (0,) for cols in (nout, kin)]

        def both(copies, formed=None):
            ys, left, first = [], [], [0, 0]
            if copies == "in one launch":
                marks, many = (C.c_uint64 * 2)(), lambda xs: (C.c_uint64 * 2)(*xs)
                be._check(be._lib.omx_i8_copies_form(
                    be._ctx, (C.c_void_p * 2)(*(w[0].ptr for w in ws)), (C.c_void_p * 2)(*(w[1].ptr for w in ws)), many([nout] * 2), many([kin] * 2),
                    many([0, size]), C.c_uint64(2), C.c_uint64(2 * size), C.c_uint64(32), C.c_int32(0), C.c_uint64(rows), marks))
                first = list(marks)
                assert all(first)
            for i, w in enumerate(ws):
                if copies:
                    be._check(be._lib.omx_i8_copy_next(be._ctx, C.c_uint64(i * size), C.c_uint64(2 * size), C.c_uint64(first[i])))
                ys.append(be.linear_i8_group_forward(x, *w, low_rank=tails[0]))
                left.append(formed or be._lib.omx_i8_copy_formed(be._ctx))
            yield left
            for i, w in enumerate(ws):
                if copies:
                    be._check(be._lib.omx_i8_copy_next(be._ctx, C.c_uint64(i * size), C.c_uint64(2 * size), C.c_uint64(left[i])))
                ys.append(be.linear_i8_group_backward_input(*w, g, low_rank=tails[1]))
            yield [be.download_f32(y) for y in ys]

        be._lib.omx_i8_copy_formed.restype = C.c_uint64
        left, want = both(False)
        assert left == [0, 0]
        left, got = both(True)
        assert left[0] != 0 and left[0] == left[1]
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert all(np.array_equal(a, b) for a, b in zip(list(both("in one launch"))[1], want))
        _, got = both(True, formed=left[0] + 7)  # not this block's: formed anew
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        pair = both(True)
        assert next(pair)[0] == left[0]
        rest = be.empty(((budget - be.budget()["live"] + (1 << 20)) // 4,), F32)
        del rest  # (a MiB more than there was: the scratch went back)
        assert all(np.array_equal(a, b) for a, b in zip(next(pair), want))
        left, got = both(True)
        assert left == [0, 0]
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
    finally:
        be.close()
