"""BASELINE.json configs[3] (Muon-NS5 + AdamW hybrid step at the GPT-124M shape) and configs[4] (LoRA
rank-16 step on the frozen int8 ~1B decoder) at their full sizes.

The oracle cannot run either whole configuration in test time, so each is tied to it in links and
held to what the mathematics fixes at full size:

the forward / backward of this step is configs[2]'s (tests/test_gpu_full_size.py); here
the optimizer runs at size. Newton-Schulz drives a matrix towards an orthogonal one, so every
Muon update is what the singular value decomposition of its gradient says it is (the iteration
acts on singular values alone: ojas-cpu/tests/numerical_invariants.rs T5 checks the same map on a
diagonal matrix); the f32 and bf16 tiers must agree; the tables and norms must move against their
gradients' signs by about lr (AdamW's first step).

(1) the model at full width (d 2048, 16 heads of 128, SwiGLU 8192, vocabulary 32000, rank
16) but 2 blocks and 1 x 512 tokens equals the oracle; (2) at the full configuration the quantised
products equal the bf16 products of the dequantised weights; (3) the adapter starts as the identity
(B = 0: the loss does not depend on A and dA is exactly zero); (4) the gradient predicts the change
of the loss along itself; (5) AdamW on the adapters lowers the loss on a fixed batch.

The nanolab graph at the 124M size: the bf16 tier against the f32 tier (which the oracle pins at
small sizes, tests/test_gpu_nanolab_native.py), the same derivative check, micro-batch accumulation
and the hybrid step.
"""
import numpy as np
import pytest

import oracle_api as orc

pytestmark = pytest.mark.gpu

GPT124M = (12, 768, 12, 64, 3072, 1024, 50304, 16, 0)
LORA1B = (16, 2048, 16, 128, 8192, 32000, 4, 2048, 16)


@pytest.fixture(scope="module")
def be():
    from ojas_amd.backend import MiBackend

    backend = MiBackend(0)
    yield backend
    backend.close()


# ------------------------------------------------------------------ configs[3]
def ns5_closed_form(g):
    """What five Newton-Schulz steps make of g, from its singular value decomposition: the iteration
    X <- a X + (b A + c A^2) X with A = X X^T keeps the singular vectors and sends every singular
    value s through s (a + b s^2 + c s^4), starting from s / ||g||_F (optim.rs:650-700)."""
    u, s, vt = np.linalg.svd(g.astype(np.float64), full_matrices=False)
    s = s / (np.sqrt(np.sum(s * s)) + 1e-7)
    for _ in range(5):
        s = s * (3.4445 + s * s * (-4.7750 + 2.0315 * s * s))
    return (u * s) @ vt, s


def test_hybrid_step_at_full_size(be):
    from ojas_amd.backend import AdamWConfig, MuonNs5Config
    from ojas_amd.trainer import GptConfig, GptTrainer, synthetic_batch

    layers, d, mlp = GPT124M[0], GPT124M[1], GPT124M[4]
    lr, mlr, wd = 3e-4, 0.02, 0.1
    adamw = AdamWConfig.nanolab(lr, 0.0)
    rng = np.random.default_rng(33)
    results = {}
    for bf16 in (0, 1):
        print(f"full-size hybrid step, bf16={bf16}", flush=True)
        cfg = GptConfig(*GPT124M, bf16)
        tr = GptTrainer(be, cfg)
        try:
            if bf16 == 0:
                params = [np.ones(n, np.float32) if n == d else rng.normal(0, 0.02, n).astype(np.float32)
                          for n in tr.param_lens()]
                ids, targets = synthetic_batch(cfg, 8)
            tr.set_params(params)
            tr.set_batch(ids, targets)
            loss0 = tr.loss_and_grads()
            grads = tr.grads()
            muon = MuonNs5Config(mlr, 0.95, wd, 1, bf16)
            loss, norm = tr.step_hybrid(muon, adamw, 1.0)
            assert loss == loss0
            after = tr.params()
            more = [tr.step_hybrid(muon, adamw, 1.0)[0] for _ in range(4)]
        finally:
            tr.close()
        print(f"  losses {loss:.4f} -> {more}", flush=True)
        assert more[-1] < more[0] < loss, (loss, more)
        results[bf16] = (loss, norm, grads, after)

    assert abs(results[1][0] - results[0][0]) <= 1e-3 * abs(results[0][0])
    assert abs(results[1][1] - results[0][1]) <= 2e-2 * results[0][1]
    decay = np.float32(1.0 - mlr * wd)
    worst = {0: 0.0, 1: 0.0, "tiers": 0.0}
    for bf16 in (0, 1):
        loss, norm, grads, after = results[bf16]
        want_norm = np.sqrt(sum(float(np.sum(g.astype(np.float64) ** 2)) for g in grads))
        assert abs(norm - want_norm) <= 1e-5 * want_norm
        clip = min(1.0, 1.0 / (want_norm + 1e-6))
        for i, p in enumerate(params):
            in_layer = 2 <= i < len(params) - 1
            which = (i - 2) % 8 if in_layer else -1
            layer = (i - 2) // 8
            if which in (1, 2, 3, 4, 6, 7):
                shape = (d, d) if which <= 4 else ((mlp, d) if which == 6 else (d, mlp))
                # new = old (1 - lr wd) - lr sqrt(max(rows / cols, 1)) O: what is left after the decay is O.
                scale = mlr * np.sqrt(max(shape[0] / shape[1], 1.0))
                got = -((after[i] - p * decay).reshape(shape).astype(np.float64)) / scale
                if bf16 == 1:
                    other = -((results[0][3][i] - p * decay).reshape(shape).astype(np.float64)) / scale
                    gap = np.linalg.norm(got - other) / np.linalg.norm(other)
                    worst["tiers"] = max(worst["tiers"], gap)
                    assert gap <= 0.17, (i, gap)
                    # The bf16 iteration's error is noise around the f32 update, not a change of its size: the
                    # component of one along the other is 1 (a wrong scale would show here at full size).
                    along = float(np.vdot(got, other) / np.vdot(other, other))
                    worst["along"] = max(worst.get("along", 0.0), abs(along - 1.0))
                    assert abs(along - 1.0) <= 1.5e-2, (i, along)
                if layer in (0, layers - 1):  # one decomposition per matrix: first and last block only
                    want, sv = ns5_closed_form(grads[i].reshape(shape))  # clip and Nesterov only rescale g
                    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
                    worst[bf16] = max(worst[bf16], rel)
                    assert rel <= (0.16 if bf16 else 1e-3), (bf16, i, rel)
                    along = float(np.vdot(got, want) / np.vdot(want, want))
                    worst["along"] = max(worst.get("along", 0.0), abs(along - 1.0))
                    assert abs(along - 1.0) <= (1.5e-2 if bf16 else 1e-3), (bf16, i, along)
                    assert sv.max() < 1.3  # no direction is amplified beyond the iteration's fixed band
            else:
                g = grads[i].astype(np.float64) * clip
                # first AdamW step, bias corrections applied: m / sqrt(v) = g / |g|, so -lr g / (|g| + eps)
                want = -lr * g / (np.abs(g) + 1e-8)
                off = float(np.max(np.abs((after[i] - p) - want) - 1.2e-7 * np.abs(p)))
                assert off <= 1e-2 * lr, (bf16, i, off / lr)
                assert np.mean(np.abs(after[i] - p) > 0.9 * lr) > 0.5, i  # and most elements do move by lr
    print(f"  Muon update against the closed form: f32 {worst[0]:.2e}, bf16 {worst[1]:.2e}; tiers apart {worst['tiers']:.2e}; "
          f"component along the other, worst |1 - c| {worst['along']:.2e}",
          flush=True)


# ------------------------------------------------------------------ configs[4]
def _frozen_case(cfg, seed):
    """Seeded frozen base at the given shape: (dequantised f32 tensors, codes + scales per matrix)."""
    rng = np.random.default_rng(seed)
    frozen, quant = [], []
    for shape in orc.lora_frozen_shapes(cfg):
        if len(shape) == 1:
            frozen.append((1.0 + 0.05 * rng.normal(size=shape)).astype(np.float32))
            quant.append(None)
        elif shape[0] == cfg.vocab:
            frozen.append(orc.round_bf16(rng.normal(0, 0.05, shape).astype(np.float32)))
            quant.append(None)
        else:
            codes, scales = orc.quantize_i8_group(rng.normal(0, 0.02, shape).astype(np.float32), 32)
            frozen.append(orc.dequant_i8_group(codes, scales, 32))
            quant.append((codes, scales))
    return frozen, quant


def _load(tr, cfg, frozen, quant):
    tr.set_embedding(frozen[0])
    for l in range(cfg.layers):
        base = 1 + 9 * l
        tr.set_norm(l, 0, frozen[base + 0])
        tr.set_norm(l, 1, frozen[base + 5])
        for which, idx in enumerate((1, 2, 3, 4, 6, 7, 8)):
            tr.set_matrix(l, which, *quant[base + idx])
    tr.set_norm(cfg.layers, 0, frozen[-1])


def test_lora_full_width_two_blocks_match_the_oracle(be):
    from ojas_amd.lora import LoraConfig, LoraTrainer

    shape = (2,) + LORA1B[1:6] + (1, 512, 16)
    print(f"lora full width {shape}", flush=True)
    cfg = LoraConfig(*shape, 1e-6, 1.0, 10000.0)
    ocfg = orc.LoraConfig(*shape, 1e-6, 1.0, 10000.0)
    frozen, quant = _frozen_case(ocfg, 3)
    rng = np.random.default_rng(4)
    adapters = [orc.round_bf16(rng.normal(0, 0.02, s).astype(np.float32)) for s in orc.lora_adapter_shapes(ocfg)]
    ids = rng.integers(0, ocfg.vocab, 512).astype(np.uint32)
    targets = rng.integers(0, ocfg.vocab, 512).astype(np.uint32)
    orc.set_threads(16)
    oloss, ograds = orc.lora_loss_and_grads(ocfg, frozen, adapters, ids, targets)
    tr = LoraTrainer(be, cfg)
    try:
        _load(tr, cfg, frozen, quant)
        tr.set_adapters(adapters)
        tr.set_batch(ids, targets)
        loss = tr.loss_and_grads()
        grads = tr.grads()
    finally:
        tr.close()
    assert abs(loss - float(oloss)) <= 1e-3 * abs(float(oloss)), (loss, oloss)
    elementwise = [float(np.max(np.abs(g - og)) / np.max(np.abs(og))) for g, og in zip(grads, ograds)]
    normwise = [float(np.linalg.norm(g - og) / np.linalg.norm(og)) for g, og in zip(grads, ograds)]
    print("  worst element / largest:", " ".join(f"{e:.4f}" for e in elementwise), flush=True)
    print("  normwise:", " ".join(f"{e:.4f}" for e in normwise), flush=True)
    # 2e-2 of each tensor's largest value per element, and normwise (measured at most 1.9e-2 on the
    # last block's query and key adapters and 0.9e-2 to 1.6e-2 elsewhere): the forward's product
    # outputs stay f32, so every activation is rounded to bf16 once.
    assert max(elementwise) <= 2e-2, elementwise
    assert max(normwise) <= 2e-2, normwise


@pytest.mark.parametrize("time,seed", [(705, 1), (768, 2), (1100, 3)])
def test_lora_over_longer_sequences_matches_the_oracle(be, time, seed):
    """Two blocks of eight heads of 128, where attention's row blocks are shared by groups of waves in the forward too, and
    without: the bounds of 512 positions."""
    from ojas_amd.lora import LoraConfig, LoraTrainer

    shape = (2, 1024, 8, 128, 2048, 1000, 1, time, 16)
    print(f"lora {shape}", flush=True)
    cfg, ocfg = LoraConfig(*shape, 1e-6, 1.0, 10000.0), orc.LoraConfig(*shape, 1e-6, 1.0, 10000.0)
    frozen, quant = _frozen_case(ocfg, seed)
    rng = np.random.default_rng(seed)
    adapters = [orc.round_bf16(rng.normal(0, 0.02, s).astype(np.float32)) for s in orc.lora_adapter_shapes(ocfg)]
    ids, targets = (rng.integers(0, ocfg.vocab, time).astype(np.uint32) for _ in range(2))
    orc.set_threads(16)
    oloss, ograds = orc.lora_loss_and_grads(ocfg, frozen, adapters, ids, targets)
    tr = LoraTrainer(be, cfg)
    try:
        _load(tr, cfg, frozen, quant)
        tr.set_adapters(adapters)
        tr.set_batch(ids, targets)
        for schedule in (0, 1):  # by the rule: two groups; one
            be.set_option("flash_schedule", schedule)
            loss, grads = tr.loss_and_grads(), tr.grads()
            assert abs(loss - float(oloss)) <= 1e-3 * abs(float(oloss)), (schedule, loss, oloss)
            elementwise = [float(np.max(np.abs(g - og)) / np.max(np.abs(og))) for g, og in zip(grads, ograds)]
            normwise = [float(np.linalg.norm(g - og) / np.linalg.norm(og)) for g, og in zip(grads, ograds)]
            print(f"  schedule {schedule}: worst element / largest {max(elementwise):.4f}, normwise {max(normwise):.4f}", flush=True)
            # (measured over 12 models of 768 and 1100 positions: at most 1.6e-2 and 1.4e-2 either way)
            assert max(elementwise) <= 2e-2, elementwise
            assert max(normwise) <= 2e-2, normwise
    finally:
        be.set_option("flash_schedule", 0)
        tr.close()


@pytest.mark.parametrize("kin,nout", [(2048, 6144), (2048, 16384), (8192, 2048)])
def test_quantised_products_at_full_size_equal_the_bf16_products_of_the_dequantised_weight(be, kin, nout):
    """8192 tokens against the fused q|k|v, gate|up and down matrices of configs[4], in the blocked
    layout the step uses: the same values reach the matrix units either way (the codes are widened
    to the bf16 the dense product reads), so the two differ by the order of f32 sums only."""
    from ojas_amd.backend import BF16

    print(f"q8 at full size {kin}x{nout}", flush=True)
    rows = 8192
    rng = np.random.default_rng(kin + nout)
    x = be.upload(rng.normal(0, 1, (rows, kin)).astype(np.float32), BF16)
    gy = be.upload(rng.normal(0, 1, (rows, nout)).astype(np.float32), BF16)
    codes_h = rng.integers(-127, 128, (nout, kin)).astype(np.int8)
    scales_h = rng.uniform(1e-4, 4e-4, (nout, kin // 32)).astype(np.float32)
    codes, scales = be.upload(codes_h), be.upload(scales_h)
    bc, bs = be.pack_i8_group(codes, scales)
    w16 = be.upload(codes_h.astype(np.float32) * np.repeat(scales_h, 32, axis=1), BF16)
    y_q = be.download_f32(be.linear_i8_group_forward(x, bc, bs, blocked=True))
    y_d = be.download_f32(be.linear_forward(x, w16, out_dtype=BF16))
    assert np.max(np.abs(y_q - y_d)) <= 1e-2 * np.max(np.abs(y_d))
    assert np.mean(y_q == y_d) > 0.9  # bf16 outputs: most values round to the same bits
    g_q = be.download_f32(be.linear_i8_group_backward_input(bc, bs, gy, blocked=True))
    g_d = be.download_f32(be.linear_backward_input(w16, gy, gx_dtype=BF16))
    assert np.max(np.abs(g_q - g_d)) <= 1e-2 * np.max(np.abs(g_d))
    assert np.mean(g_q == g_d) > 0.9


def test_lora_step_at_full_size(be):
    from ojas_amd.backend import AdamWConfig
    from ojas_amd.lora import LoraConfig, LoraTrainer

    cfg = LoraConfig(*LORA1B, 1e-6, 1.0, 10000.0)
    print("lora step at full size", flush=True)
    tr = LoraTrainer(be, cfg)
    try:
        tr.init_base(77, 0.02)
        tr.init_adapters(5, 0.02)  # B = 0
        rng = np.random.default_rng(6)
        window = rng.integers(0, cfg.vocab, (cfg.batch, cfg.seq + 1)).astype(np.uint32)
        tr.set_batch(window[:, :-1], window[:, 1:])
        # (3) the identity at B = 0.
        loss0 = tr.loss_and_grads()
        grads0 = tr.grads()
        assert abs(loss0 - np.log(cfg.vocab)) < 1.0  # an untrained model: about ln V
        assert all(not np.any(g) for g in grads0[0::2]) and all(np.any(g) for g in grads0[1::2])
        a0 = tr.adapters()
        tr.set_adapters([2 * a if i % 2 == 0 else a for i, a in enumerate(a0)])
        assert tr.loss_and_grads() == loss0
        # (4) along the gradient, from a point where both A and B carry weight.
        start = [a if i % 2 == 0 else rng.normal(0, 0.02, a.shape).astype(np.float32) for i, a in enumerate(a0)]
        tr.set_adapters(start)
        base = tr.loss_and_grads()
        grads = tr.grads()
        assert all(np.any(g) for g in grads)
        sq = sum(float(np.sum(g.astype(np.float64) ** 2)) for g in grads)
        eps = 0.02 / sq  # a first-order change of 0.02 each way
        losses = []
        for sign in (1.0, -1.0):
            tr.set_adapters([a + np.float32(sign * eps) * g for a, g in zip(start, grads)])
            losses.append(tr.loss_and_grads())
        measured = losses[0] - losses[1]
        print(f"loss {base:.5f}; along the gradient: measured {measured:.5f}, predicted {2 * eps * sq:.5f}", flush=True)
        assert losses[1] < base < losses[0]
        assert abs(measured - 2 * eps * sq) <= 0.1 * 2 * eps * sq, (measured, 2 * eps * sq)
        # (5) AdamW on the adapters only.
        tr.set_adapters(start)
        adamw = AdamWConfig(1e-3, 0.9, 0.95, 1e-8, 0.0)
        curve = [tr.step(adamw, 1.0)[0] for _ in range(6)]
        assert curve[0] == base and curve[-1] < curve[0] - 1e-3 and tr.steps() == 6, curve
    finally:
        tr.close()


# ------------------------------------------------------------------ the nanolab graph at the 124M size
def _nanolab_124m_params(spec, rng, bf16_exact=True):
    """N(0, 0.02) matrices and table (bf16-exact by default: both tiers then multiply the same
    weights), norm weights one, a gate that is not flat and value residuals that are not at their
    start."""
    params = {}
    for name, shape in spec.param_shapes().items():
        if len(shape) == 2:
            w = rng.normal(0, 0.02, shape).astype(np.float32)
            params[name] = orc.round_bf16(w) if bf16_exact else w
        elif name.endswith("vr_lambda"):
            params[name] = rng.uniform(0.2, 0.8, shape).astype(np.float32)
        elif name.endswith("gate.bias"):
            params[name] = rng.normal(0, 0.5, shape).astype(np.float32)
        else:
            params[name] = np.ones(shape, np.float32)
    return params


def _matrix_distances(got, want, shapes):
    """(worst normwise, worst element / largest) over the matrices and the table."""
    normwise = elementwise = 0.0
    for name, ref in want.items():
        if len(shapes[name]) != 2:
            continue
        ref = ref.reshape(-1).astype(np.float64)
        diff = got[name].reshape(-1).astype(np.float64) - ref
        normwise = max(normwise, float(np.linalg.norm(diff) / np.linalg.norm(ref)))
        elementwise = max(elementwise, float(np.max(np.abs(diff)) / np.max(np.abs(ref))))
    return normwise, elementwise


def test_nanolab_124m_against_the_oracle_at_full_depth_and_width(be):
    """`ModelSpec::nanolab_124m` (ojas-model/src/spec.rs:74-91: 12 blocks, 768 wide, 12 heads of 64,
    SwiGLU 2048, vocabulary 50304) on one 256-token sequence, which the oracle finishes in seconds.
    f32 tier: loss 1e-5 relative, every gradient 1e-4 normwise (the reference's gate for a device,
    ojas-oracle/src/parity.rs:28-40). bf16 tier: loss 1e-3 relative. Its gradients cannot be inside
    2e-2 at this depth: the oracle's own Exact arithmetic with nothing but the products' operands
    rounded to bf16 (`ROUND_OPERANDS`, the least rounding a tier with bf16 products can do) is
    about 3e-2 from its unrounded self here, normwise and per element (1e-2 per sqrt(block),
    tests/test_oracle_bf16_floor.py), and the reference's own rounding points (`ROUND_AUTOCAST`) 4e-2.
    The device's tier is held to that floor: within 1.25 x of it, and below the reference's tier."""
    from ojas_amd.nanolab import NativeNanolabTrainer, spec_nanolab_124m
    from test_gpu_nanolab_native import oracle_step

    spec = spec_nanolab_124m()
    shapes = spec.param_shapes()
    rng = np.random.default_rng(77)
    params = _nanolab_124m_params(spec, rng)
    window = rng.integers(0, spec.vocab, (1, 257)).astype(np.uint32)
    ids, targets = np.ascontiguousarray(window[:, :-1]), np.ascontiguousarray(window[:, 1:])
    print("nanolab 124M, 1 x 256 tokens: oracle (exact, operands-only, autocast points)", flush=True)
    orc.set_threads(16)
    o_loss, exact = oracle_step(spec, params, ids, targets, 1, 256)
    _, floor = oracle_step(spec, params, ids, targets, 1, 256, rounding=orc.ROUND_OPERANDS)
    _, autocast = oracle_step(spec, params, ids, targets, 1, 256, rounding=orc.ROUND_AUTOCAST)
    floor_n, floor_e = _matrix_distances(floor, exact, shapes)
    auto_n, auto_e = _matrix_distances(autocast, exact, shapes)
    print(f"  oracle operands-only: {floor_n:.4f} normwise, {floor_e:.4f} per element; autocast points: {auto_n:.4f}, {auto_e:.4f}",
          flush=True)
    assert 2e-2 < floor_n < auto_n < 6e-2
    for bf16 in (False, True):
        tr = NativeNanolabTrainer(be, spec, 1, 256, params, bf16=bf16)
        try:
            loss, grads = tr.loss_and_grads(ids, targets)
        finally:
            tr.close()
        normwise, elementwise = _matrix_distances(grads, exact, shapes)
        print(f"  device bf16={bf16}: loss {loss:.6f} (oracle {o_loss:.6f}), matrices {normwise:.2e} normwise, "
              f"{elementwise:.2e} per element", flush=True)
        if not bf16:
            assert abs(loss - o_loss) <= 1e-5 * abs(o_loss)
            for name, ref in exact.items():
                if np.any(ref):
                    got = grads[name].astype(np.float64)
                    assert np.linalg.norm(got - ref.reshape(-1)) <= 1e-4 * np.linalg.norm(ref), name
            continue
        assert abs(loss - o_loss) <= 1e-3 * abs(o_loss)
        assert normwise <= 1.25 * floor_n and elementwise <= 1.25 * floor_e, (normwise, floor_n, elementwise, floor_e)
        assert normwise < auto_n


def test_nanolab_124m_step_at_full_size(be):
    """The native nanolab driver at `ModelSpec::nanolab_124m` (ojas-model/src/spec.rs:74-91), 16 x 1024
    tokens, bf16 tier: the paths only this size takes (MFMA attention on the fused q | k | v output,
    the weight gradients as strided batches after the backward, one AdamW pass over the table and
    the vectors). The two tiers agree on the loss and, at 4 x 1024 tokens, on every matrix gradient
    as closely as 12 blocks of bf16 operands allow (the test above measures that floor against
    the oracle: about 3e-2; the gate here is 4e-2 normwise); the gradient predicts the change of the
    loss along itself; two half-weighted micro-batches add up to the whole one; six hybrid steps on
    one batch lower the loss."""
    from ojas_amd.nanolab import NativeNanolabTrainer, spec_nanolab_124m

    spec = spec_nanolab_124m()
    rng = np.random.default_rng(31)
    print("nanolab 124M: tiers at 4 x 1024", flush=True)
    small = rng.integers(0, spec.vocab, (4, 1025)).astype(np.uint32)
    params = _nanolab_124m_params(spec, rng)
    tier = {}
    for bf16 in (True, False):
        tr = NativeNanolabTrainer(be, spec, 4, 1024, params, bf16=bf16)
        try:
            tier[bf16] = tr.loss_and_grads(small[:, :-1], small[:, 1:])
        finally:
            tr.close()
    (loss16, g16), (loss32, g32) = tier[True], tier[False]
    print(f"loss bf16 {loss16:.5f} f32 {loss32:.5f}", flush=True)
    assert abs(loss32 - np.log(spec.vocab)) < 1.0 and abs(loss16 - loss32) <= 1e-3 * abs(loss32)
    assert not np.any(g32["blocks.0.mixer.vr_lambda"]) and not np.any(g16["blocks.0.mixer.vr_lambda"])
    normwise, elementwise = _matrix_distances(g16, g32, spec.param_shapes())
    print(f"tier distance over the matrices: {normwise:.4f} normwise, {elementwise:.4f} per element", flush=True)
    assert normwise <= 4e-2, normwise
    lam = [n for n in g32 if n.endswith("vr_lambda") and n != "blocks.0.mixer.vr_lambda"]
    want = np.array([g32[n][0] for n in lam], np.float64)
    got = np.array([g16[n][0] for n in lam], np.float64)
    # A lambda's gradient is one number, a sum over every value element with both signs: the eleven
    # are held as one vector.
    print("lambda gradients: distance", float(np.linalg.norm(got - want) / np.linalg.norm(want)), flush=True)
    assert np.linalg.norm(got - want) <= 8e-2 * np.linalg.norm(want), (got, want)
    print("nanolab 124M: 16 x 1024", flush=True)
    # Weights between bf16 values from here on: a step along the gradient is far smaller than the
    # spacing of bf16 numbers, and from bf16-exact weights the tier's operand copies would not move.
    params = _nanolab_124m_params(spec, rng, bf16_exact=False)
    window = rng.integers(0, spec.vocab, (16, 1025)).astype(np.uint32)
    ids, targets = window[:, :-1], window[:, 1:]
    tr = NativeNanolabTrainer(be, spec, 16, 1024, bf16=True, adam_lr=1e-3, matrix_lr=0.02)
    try:
        tr.set_params(params)
        base, grads = tr.loss_and_grads(ids, targets)
        # two micro-batches at half weight add up to the whole one
        tr._micro(ids, targets, 0.5, 0.5, True)
        tr._micro(ids, targets, 0.5, 0.5, False)
        twice = tr.grads()
        for name, g in grads.items():
            scale = float(np.max(np.abs(g)))
            assert float(np.max(np.abs(twice[name] - g))) <= 1e-6 * scale, name
        # along the gradient
        sq = sum(float(np.sum(g.astype(np.float64) ** 2)) for g in grads.values())
        eps = 0.02 / sq
        losses = []
        for sign in (1.0, -1.0):
            tr.set_params({n: params[n] + np.float32(sign * eps) * grads[n].reshape(params[n].shape) for n in params})
            losses.append(tr.loss_and_grads(ids, targets)[0])
        measured = losses[0] - losses[1]
        print(f"loss {base:.5f}; along the gradient: measured {measured:.5f}, predicted {2 * eps * sq:.5f}", flush=True)
        assert losses[1] < base < losses[0]
        assert abs(measured - 2 * eps * sq) <= 0.1 * 2 * eps * sq, (measured, 2 * eps * sq)
        # the hybrid step
        tr.set_params(params)
        curve = [tr.run([(ids, targets)], 1.0).loss for _ in range(6)]
        print("curve", curve, flush=True)
        assert abs(curve[0] - base) <= 1e-6 * base and curve[-1] < curve[0] - 0.1 and tr.step == 6, curve
        after = tr.download_params()
        assert np.array_equal(after["blocks.0.mixer.vr_lambda"], params["blocks.0.mixer.vr_lambda"])
        assert all(np.all(np.isfinite(a)) for a in after.values())
    finally:
        tr.close()
