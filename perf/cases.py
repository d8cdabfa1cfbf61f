"""The work this framework is used for, as cases that can be timed and whose results can be compared.

A case is one pass through the public entry points, of one of these kinds:

  gpt        one optimizer step of the GPT-2-shaped model: `GptTrainer.set_batch` + `step` / `step_hybrid`
  nanolab    one optimizer step of the nanolab model through the native driver: `NativeNanolabTrainer.run`
  tape       the same step made op by op over the backend, as a generic tape does: `NanolabTrainer.run`
  lora       one LoRA step on a frozen int8 decoder: `LoraTrainer.set_batch` + `step`
  attention  causal attention, forward and backward, through `MiBackend.causal_sdpa_*`
  cached     a decoder pass over KV caches (`MiBackend`, op by op): tq = 1 decodes one token per sequence, a larger
             tq reads a prompt's chunk in

`listed` holds one model of each size and shape that the framework's configurations name, small and ragged ones beside
them; `draw` gives more of the same ranges. What a native driver hands its caller is the step's loss and gradient norm
(its parameters stay with the driver), and those are its outputs here; a norm over every gradient and, from the second
step on, a loss over every updated parameter. The op-by-op kinds hand back every tensor: updated parameters, attention
outputs and gradients, logits and caches.
"""
import numpy as np
import torch

from ojas_amd.backend import BF16, F32, U32, AdamWConfig, DeviceTensor, MiBackend, MuonNs5Config
from ojas_amd.lora import LoraConfig, LoraTrainer, adapter_params, base_params
from ojas_amd.lora import step_flops as lora_step_flops
from ojas_amd.nanolab import NanolabSpec, NanolabTrainer, NativeNanolabTrainer, nanolab_step_flops
from ojas_amd.trainer import GptConfig, GptTrainer, matmul_params
from ojas_amd.trainer import step_flops as gpt_step_flops


def listed():
    return [
        # The tiny f32 configuration: a step of some 150 small launches, where launch count and latency weigh most.
        {"name": "gpt_tiny_f32", "kind": "gpt", "layers": 4, "d_model": 256, "head_dim": 64, "ctx": 256, "vocab": 8192,
         "batch": 8, "bf16": False, "muon": False},
        # The headline: the 124M-parameter bf16 AdamW step on 16384 tokens.
        {"name": "gpt_124m_bf16", "kind": "gpt", "layers": 12, "d_model": 768, "head_dim": 64, "ctx": 1024,
         "vocab": 50304, "batch": 16, "bf16": True, "muon": False},
        # The same with Muon-NS5 on the hidden matrices.
        {"name": "gpt_124m_muon", "kind": "gpt", "layers": 12, "d_model": 768, "head_dim": 64, "ctx": 1024,
         "vocab": 50304, "batch": 16, "bf16": True, "muon": True},
        # A middle-sized model whose batch, context and vocabulary nobody padded: 3500 tokens, an odd vocabulary.
        {"name": "gpt_ragged_bf16", "kind": "gpt", "layers": 6, "d_model": 512, "head_dim": 64, "ctx": 500,
         "vocab": 32003, "batch": 7, "bf16": True, "muon": False},
        # The reference's own model at its 124M size, Muon and AdamW groups.
        {"name": "nanolab_124m_bf16", "kind": "nanolab", "layers": 12, "d_model": 768, "head_dim": 64, "kv_heads": 12,
         "hidden": 2048, "vocab": 50304, "batch": 16, "seq": 1024, "window": 0, "micro": 1, "bf16": True},
        # A tape over the backend: every op a call of its own, parameters and gradients the caller's tensors.
        {"name": "tape_small_f32", "kind": "tape", "layers": 4, "d_model": 256, "head_dim": 64, "kv_heads": 2,
         "hidden": 704, "vocab": 8192, "batch": 4, "seq": 256, "window": 0, "micro": 1, "autocast": False},
        # LoRA rank 16 on the frozen int8 1B decoder: the largest step.
        {"name": "lora_1b", "kind": "lora", "layers": 16, "d_model": 2048, "head_dim": 128, "hidden": 8192,
         "vocab": 32000, "batch": 4, "seq": 2048, "rank": 16},
        # Attention on its own at the isolated configuration.
        {"name": "attention_bf16", "kind": "attention", "batch": 8, "heads": 12, "kv_heads": 12, "time": 1024,
         "head_dim": 64, "window": 0, "bf16": True},
        # The f32 tier of the same op: grouped heads, a sliding window, a length that no tile divides.
        {"name": "attention_f32_window", "kind": "attention", "batch": 2, "heads": 8, "kv_heads": 2, "time": 777,
         "head_dim": 64, "window": 256, "bf16": False},
        # Decoding for one user: one token through twelve blocks, nothing but latency.
        {"name": "decode_one", "kind": "cached", "layers": 12, "d_model": 768, "head_dim": 64, "kv_heads": 12,
         "vocab": 50304, "batch": 1, "tq": 1, "kv_len": 301, "bf16_cache": True},
        # Decoding for 64 users at full context, f32 caches as the trait prescribes.
        {"name": "decode_batch", "kind": "cached", "layers": 12, "d_model": 768, "head_dim": 64, "kv_heads": 12,
         "vocab": 50304, "batch": 64, "tq": 1, "kv_len": 1024, "bf16_cache": False},
        # Reading a chunk of four prompts in.
        {"name": "prefill", "kind": "cached", "layers": 12, "d_model": 768, "head_dim": 64, "kv_heads": 12,
         "vocab": 50304, "batch": 4, "tq": 256, "kv_len": 700, "bf16_cache": True},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, evenly over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _divisor(rng, n):
    return rng.choice([k for k in range(1, n + 1) if n % k == 0])


def _draw_once(rng):
    kind = rng.choice(["gpt", "gpt", "nanolab", "tape", "lora", "attention", "attention", "cached", "cached", "cached"])
    head_dim = rng.choice([64, 64, 128])
    heads = rng.randint(2, 1024 // head_dim)
    model = {"layers": rng.randint(2, 12), "d_model": heads * head_dim, "head_dim": head_dim}
    vocab = _spread(rng, 1000, 50304)
    window = rng.choice([0, 0, _spread(rng, 32, 1024)])
    if kind == "gpt":
        bf16 = rng.random() < 0.7
        return dict(model, kind=kind, ctx=_spread(rng, 32, 1024), vocab=vocab, batch=_spread(rng, 1, 16), bf16=bf16,
                    muon=rng.random() < 0.3)
    if kind == "nanolab":
        return dict(model, kind=kind, kv_heads=_divisor(rng, heads), hidden=64 * _spread(rng, 4, 48), vocab=vocab,
                    batch=_spread(rng, 1, 16), seq=_spread(rng, 32, 1024), window=window, micro=rng.randint(1, 3),
                    bf16=rng.random() < 0.7)
    if kind == "tape":
        return dict(model, kind=kind, layers=rng.randint(1, 4), kv_heads=_divisor(rng, heads),
                    hidden=64 * _spread(rng, 2, 24), vocab=_spread(rng, 256, 16384), batch=_spread(rng, 1, 8),
                    seq=_spread(rng, 16, 512), window=window, micro=rng.randint(1, 2), autocast=rng.random() < 0.5)
    if kind == "lora":
        d_model = 128 * rng.randint(2, 16)
        return {"kind": kind, "layers": rng.randint(1, 16), "d_model": d_model, "head_dim": rng.choice([64, 128]),
                "hidden": 128 * _spread(rng, 4, 64), "vocab": _spread(rng, 1000, 32000), "batch": _spread(rng, 1, 4),
                "seq": _spread(rng, 64, 2048), "rank": rng.choice([16, 16, 32])}
    if kind == "attention":
        heads = rng.randint(1, 16)
        return {"kind": kind, "batch": _spread(rng, 1, 16), "heads": heads, "kv_heads": _divisor(rng, heads),
                "time": _spread(rng, 32, 4096), "head_dim": head_dim, "window": window, "bf16": rng.random() < 0.6}
    tq = rng.choice([1, 1, _spread(rng, 8, 512)])
    return dict(model, kind=kind, kv_heads=_divisor(rng, heads), vocab=vocab, batch=_spread(rng, 1, 64), tq=tq,
                kv_len=tq + _spread(rng, 1, 1024) - 1, bf16_cache=rng.random() < 0.5)


def draw(rng):
    # At most an eighth of the largest step's products (f32 products are some sixteen times as dear).
    while True:
        case = _draw_once(rng)
        w = work(case)
        f32 = case.get("bf16") is False or case["kind"] == "tape"
        if w["flops"] <= (2e11 if f32 else 5e12) and w["bytes"] <= 6e9:
            return case


# ---- what each kind needs ----
_BACKEND = None


def _backend():
    """One context for the process, as a program keeps it."""
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = MiBackend(0)
    return _BACKEND


_TORCH = {F32: ("<f4", None), BF16: ("<i2", torch.bfloat16), U32: ("<i4", None)}


class _Interface:
    """A device tensor of the framework's as torch takes one (it keeps the tensor alive)."""

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": _TORCH[t.dtype][0], "data": (t.ptr, False),
                                         "version": 2}


def _as_torch(t):
    x = torch.as_tensor(_Interface(t), device="cuda")
    return x.view(_TORCH[t.dtype][1]) if _TORCH[t.dtype][1] is not None else x


def _as_device(be, x):
    """A torch tensor as the framework takes one (the state keeps the torch tensor)."""
    dtype = {torch.float32: F32, torch.bfloat16: BF16, torch.int32: U32}[x.dtype]
    return DeviceTensor(be, x.data_ptr(), tuple(x.shape), dtype, owns=False)


class _Random:
    """Inputs from a seed, made on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, dtype=torch.float32):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return x.mul_(std).to(dtype)

    def ids(self, shape, vocab):
        return torch.randint(0, vocab, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def batch(self, batch, time, vocab):
        """A batch as a sampler hands it over, on the host: windows of time + 1 tokens, ids and the ids after them."""
        w = self.ids((batch, time + 1), vocab).cpu().numpy().astype(np.uint32)
        return np.ascontiguousarray(w[:, :-1]), np.ascontiguousarray(w[:, 1:])


class _State:
    """What a case keeps; a trainer's device memory goes back with it."""

    def __init__(self, **kw):
        self.trainer = None
        self.__dict__.update(kw)

    def __del__(self):
        if self.trainer is not None and hasattr(self.trainer, "close"):
            self.trainer.close()


def _gpt_config(c):
    return GptConfig(c["layers"], c["d_model"], c["d_model"] // c["head_dim"], c["head_dim"], 4 * c["d_model"],
                     c["ctx"], c["vocab"], c["batch"], 0, int(c["bf16"]))


def _gpt_params(c):
    return matmul_params(_gpt_config(c)) + (c["ctx"] + 2 * c["layers"] + 1) * c["d_model"]


def _spec(c):
    return NanolabSpec(n_layer=c["layers"], n_embd=c["d_model"], n_head=c["d_model"] // c["head_dim"],
                       n_kv_head=c["kv_heads"], head_dim=c["head_dim"], hidden=c["hidden"], vocab=c["vocab"],
                       window=c["window"] or None, max_seq=c["seq"])


def _lora_config(c):
    return LoraConfig(c["layers"], c["d_model"], c["d_model"] // c["head_dim"], c["head_dim"], c["hidden"], c["vocab"],
                      c["batch"], c["seq"], c["rank"], 1e-6, 1.0, 10000.0)


def _nanolab_params(spec, r):
    """N(0, 0.02) matrices and table, norm weights 1, gate bias 0, value blend 0.5: one device-to-host copy."""
    shapes = spec.param_shapes()
    matrices = [n for n in spec.param_names() if len(shapes[n]) == 2]
    sizes = [int(np.prod(shapes[n])) for n in matrices]
    flat = r.normal(sum(sizes), 0.02).cpu().numpy()
    out, at = {}, 0
    for n, size in zip(matrices, sizes):
        out[n] = flat[at:at + size].reshape(shapes[n])
        at += size
    for n, shape in shapes.items():
        if n not in out:
            value = 0.0 if n.endswith("bias") else 0.5 if n.endswith("lambda") else 1.0
            out[n] = np.full(shape, value, np.float32)
    return out


def _prepare_gpt(c, r):
    tr = GptTrainer(_backend(), _gpt_config(c))
    lens = tr.param_lens()
    flat, params, at = r.normal(sum(lens), 0.02).cpu().numpy(), [], 0
    for i, n in enumerate(lens):
        norm = i == len(lens) - 1 or (i >= 2 and (i - 2) % 8 in (0, 5))
        params.append(np.ones(n, np.float32) if norm else flat[at:at + n])
        at += n
    tr.set_params(params)
    return _State(trainer=tr, batch=r.batch(c["batch"], c["ctx"], c["vocab"]),
                  adamw=AdamWConfig(3e-4, 0.9, 0.95, 1e-8, 0.1),
                  muon=MuonNs5Config(0.02, 0.95, 0.1, 1, int(c["bf16"])) if c["muon"] else None)


def _run_gpt(s):
    s.trainer.set_batch(*s.batch)
    if s.muon is None:
        loss, norm = s.trainer.step(s.adamw, 1.0)
    else:
        loss, norm = s.trainer.step_hybrid(s.muon, s.adamw, 1.0)
    return {"loss": loss, "grad_norm": norm}


def _prepare_nanolab(c, r):
    spec = _spec(c)
    tr = NativeNanolabTrainer(_backend(), spec, c["batch"], c["seq"], _nanolab_params(spec, r), ns5_bf16=c["bf16"],
                              bf16=c["bf16"])
    return _State(trainer=tr, batches=[r.batch(c["batch"], c["seq"], c["vocab"]) for _ in range(c["micro"])])


def _run_nanolab(s):
    report = s.trainer.run(s.batches, 0.1)  # a tenth of the peak rates: the schedule's tail
    return {"loss": report.loss, "grad_norm": report.grad_norm}


def _prepare_tape(c, r):
    spec = _spec(c)
    tr = NanolabTrainer(_backend(), spec, _nanolab_params(spec, r), autocast=c["autocast"])
    return _State(trainer=tr, batches=[r.batch(c["batch"], c["seq"], c["vocab"]) for _ in range(c["micro"])],
                  params={n: _as_torch(t) for n, t in tr.params.items()})


def _run_tape(s):
    report = s.trainer.run(s.batches, 0.1)
    return {"loss": report.loss, "grad_norm": report.grad_norm, "params": s.params}


def _prepare_lora(c, r):
    tr = LoraTrainer(_backend(), _lora_config(c))
    tr.init_base(int(torch.randint(1 << 30, (1,), generator=r.g, device="cuda")), 0.02)
    lens = tr.adapter_lens()
    flat = r.normal(sum(lens), 0.02).cpu().numpy()  # B as well as A: the middle of a fine-tune
    tr.set_adapters(np.split(flat, np.cumsum(lens)[:-1]))
    return _State(trainer=tr, batch=r.batch(c["batch"], c["seq"], c["vocab"]),
                  adamw=AdamWConfig(1e-4, 0.9, 0.95, 1e-8, 0.0))


def _run_lora(s):
    s.trainer.set_batch(*s.batch)
    loss, norm = s.trainer.step(s.adamw, 1.0)
    return {"loss": loss, "grad_norm": norm}


def _prepare_attention(c, r):
    dtype = torch.bfloat16 if c["bf16"] else torch.float32
    q = (c["batch"], c["heads"], c["time"], c["head_dim"])
    kv = (c["batch"], c["kv_heads"], c["time"], c["head_dim"])
    keep = [r.normal(shape, 1.0, dtype) for shape in (q, kv, kv, q)]
    be = _backend()
    return _State(be=be, keep=keep, args=[_as_device(be, x) for x in keep], window=c["window"] or None,
                  dtype=BF16 if c["bf16"] else F32)


def _run_attention(s):
    q, k, v, gy = s.args
    out, lse = s.be.causal_sdpa_forward(q, k, v, s.window, s.dtype)
    grads = s.be.causal_sdpa_backward(q, k, v, out, lse, gy, s.window, s.dtype)
    return [_as_torch(t) for t in (out, lse) + tuple(grads)]


def _prepare_cached(c, r):
    """bf16 weights of a decoder, its KV caches filled up to the new positions, and the new tokens. The table is
    N(0, 1), so that the logits have a clear largest value, as a trained model's have."""
    be, d, hd, kv = _backend(), c["d_model"], c["head_dim"], c["kv_heads"]
    b, tq, kv_len, bf16 = c["batch"], c["tq"], c["kv_len"], torch.bfloat16
    keep = []

    def dev(x):
        keep.append(x)
        return _as_device(be, x)

    s = _State(be=be, keep=keep, shape=(b, tq, d // hd, kv, hd), at=kv_len - tq, kv_len=kv_len)
    s.table, s.positions = dev(r.normal((c["vocab"], d), 1.0, bf16)), dev(r.normal((kv_len, d), 0.02, bf16))
    s.blocks, s.caches = [], []
    for _ in range(c["layers"]):
        weights = [dev(r.normal(shape, 0.02, bf16)) for shape in
                   ((d, d), (kv * hd, d), (kv * hd, d), (d, d), (4 * d, d), (d, 4 * d))]
        s.blocks.append([dev(torch.ones(d, device="cuda")), dev(torch.ones(d, device="cuda"))] + weights)
        cache = [r.normal((b, kv_len, kv, hd), 0.5, bf16 if c["bf16_cache"] else torch.float32) for _ in range(2)]
        s.caches.append([dev(x) for x in cache])
    s.out_caches = [x for x in keep if x.dim() == 4]
    s.final_norm = dev(torch.ones(d, device="cuda"))
    s.ids = dev(r.ids((b * tq,), c["vocab"]))
    s.places = dev((torch.arange(b * tq, device="cuda") % tq + s.at).to(torch.int32))
    s.last = dev(((torch.arange(b, device="cuda") + 1) * tq - 1).to(torch.int32))
    return s


def _run_cached(s):
    be, (b, tq, h, kv, hd) = s.be, s.shape
    n = b * tq
    x = be.embedding_forward(s.table, s.ids)
    y = be.embedding_forward(s.positions, s.places)
    for (norm1, norm2, wq, wk, wv, wo, w1, w2), (k_cache, v_cache) in zip(s.blocks, s.caches):
        x, normed = be.residual_add_rms_norm_forward(x, y, norm1, out_dtype=BF16)
        q, k, v = (be.linear_forward(normed, w) for w in (wq, wk, wv))
        be.kv_cache_write(k_cache, k.reshape(b, tq, kv, hd), s.at)
        be.kv_cache_write(v_cache, v.reshape(b, tq, kv, hd), s.at)
        att = be.cached_attention_forward(q.reshape(b, tq, h, hd), k_cache, v_cache, s.kv_len)
        y = be.linear_forward(be.to_bf16(att).reshape(n, h * hd), wo, BF16)
        x, normed = be.residual_add_rms_norm_forward(x, y, norm2, out_dtype=BF16)
        _, act = be.linear_gelu_forward(normed, w1)
        y = be.linear_forward(act, w2, BF16)
    x, normed = be.residual_add_rms_norm_forward(x, y, s.final_norm, out_dtype=BF16)
    if tq > 1:  # only the last position of each prompt chunk goes through the head
        normed = be.embedding_forward(normed, s.last, BF16)
    logits = be.linear_forward(normed, s.table)
    return {"logits": _as_torch(logits), "next": _as_torch(be.argmax_rows(logits)), "caches": s.out_caches}


_KINDS = {"gpt": (_prepare_gpt, _run_gpt), "nanolab": (_prepare_nanolab, _run_nanolab),
          "tape": (_prepare_tape, _run_tape), "lora": (_prepare_lora, _run_lora),
          "attention": (_prepare_attention, _run_attention), "cached": (_prepare_cached, _run_cached)}


def prepare(case, seed):
    make, go = _KINDS[case["kind"]]
    state = make(case, _Random(seed))
    state.go = go
    return state


def run(state):
    return state.go(state)


# ---- what a pass cannot do without ----
def _pairs(time, window, before=0):
    """Query-key pairs that `time` queries after `before` earlier positions see."""
    w = window if window else time + before
    return float(sum(min(before + i + 1, w) for i in range(time)))


def _newton_schulz_flops(shapes):
    """Five iterations of three products each."""
    total = 0.0
    for rows, cols in shapes:
        r, c = min(rows, cols), max(rows, cols)
        total += 5 * (2.0 * r * r * c * 2 + 2.0 * r * r * r)
    return total


def work(case):
    c = case
    if c["kind"] == "gpt":
        # Parameters and both moments read and written (one momentum under Muon), the batch read.
        d, p = c["d_model"], _gpt_params(c)
        flops, nbytes = gpt_step_flops(_gpt_config(c)), 24.0 * p + 8.0 * c["batch"] * c["ctx"]
        if c["muon"]:
            flops += _newton_schulz_flops([(d, d)] * 4 * c["layers"] + [(4 * d, d)] * 2 * c["layers"])
            nbytes -= 8.0 * c["layers"] * 12 * d * d
        return {"bytes": nbytes, "flops": flops}
    if c["kind"] in ("nanolab", "tape"):
        spec = _spec(c)
        shapes = spec.param_shapes()
        hidden = [s for n, s in shapes.items() if len(s) == 2 and n != "tok_emb.weight"]
        p, m = sum(int(np.prod(s)) for s in shapes.values()), sum(int(np.prod(s)) for s in hidden)
        tokens = c["batch"] * c["seq"] * c["micro"]
        return {"bytes": 24.0 * p - 8.0 * m + 8.0 * tokens,
                "flops": c["micro"] * nanolab_step_flops(spec, c["batch"], c["seq"]) + _newton_schulz_flops(hidden)}
    if c["kind"] == "lora":
        cfg = _lora_config(c)
        table = c["vocab"] * c["d_model"]
        return {"bytes": 1.125 * (base_params(cfg) - table) + 2.0 * table + 24.0 * adapter_params(cfg),
                "flops": lora_step_flops(cfg)}
    if c["kind"] == "attention":
        # Forward: two products over every visible pair; backward: five. q, k, v, gy in; out, lse, three gradients out.
        pairs = c["batch"] * c["heads"] * _pairs(c["time"], c["window"])
        q, kv = (c["batch"] * n * c["time"] * c["head_dim"] for n in (c["heads"], c["kv_heads"]))
        return {"bytes": (4.0 * q + 4.0 * kv) * (2 if c["bf16"] else 4) + 4.0 * c["batch"] * c["heads"] * c["time"],
                "flops": 14.0 * pairs * c["head_dim"]}
    # A decoder pass: every weight and the visible caches once, the new keys and values and the logits written.
    d, n, kvd = c["d_model"], c["batch"] * c["tq"], c["kv_heads"] * c["head_dim"]
    weights, table = c["layers"] * (10.0 * d * d + 2.0 * d * kvd), c["vocab"] * d
    span = c["batch"] * c["kv_len"] * kvd * 2.0 * c["layers"] * (2 if c["bf16_cache"] else 4)
    pairs = c["batch"] * (d // c["head_dim"]) * _pairs(c["tq"], 0, c["kv_len"] - c["tq"])
    return {"bytes": 2.0 * (weights + table) + span + 4.0 * c["batch"] * c["vocab"],
            "flops": 2.0 * n * weights + 2.0 * c["batch"] * table + 4.0 * pairs * c["head_dim"] * c["layers"]}


def tolerance(case):
    if case["kind"] == "attention":
        # bf16 results and probabilities; f32 sums over the row.
        return {"rel": 1e-2} if case["bf16"] else {"rel": 2e-5}
    if case["kind"] == "cached":
        # bf16 operands through up to twelve blocks. A token differs where two logits tie within that.
        return {"rel": 1e-2, "differ": 0.01}
    if case["kind"] == "lora" or case.get("bf16") or case.get("autocast"):
        return {"rel": 1e-2}
    # f32 throughout, a model deep, and an optimizer step that divides by a gradient's own size.
    return {"rel": 1e-4}
