"""The work that users of this package have it do, as measurable cases.

A case is a dict of plain values.  ``op`` names the public entry point:

* ``bitlinear``    one ``BitLinear`` on ``M`` rows (a projection on its own)
* ``ffn``          one ``FeedForward`` on ``B x L`` tokens
* ``siso``         one ``TESM_SISO`` prefill, ``window`` 0 being the global entanglement; with ``cache`` it also
                   fills the inference cache, as the prompt pass of a generation does
* ``siso_decode``  one decode step of a ``TESM_SISO`` over a filled cache
* ``mimo``         one ``TESMMIMO_Optimized`` prefill
* ``mimo_decode``  one decode step of a ``TESMMIMO_Optimized`` over a filled cache
* ``lm``           one ``TESMLMHeadModel`` forward to its logits

Sizes are those of the ``TESMConfig`` presets, ``bench.py`` and the tests.  ``exact`` restates each entry point in
plain torch with sums, scans, gates and norms in 64 bits; the int8 and ternary codes are part of what a BitLinear
is, so they are formed from values of the module's own dtype, with its own rounding.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from tesm_amd import BitLinear, FeedForward, TESM_SISO, TESMConfig, TESMLMHeadModel, TESMMIMO_Optimized

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

# Layer sizes of the presets: d_model, d_state, ent_rank, window, threshold, scale, decay bias, scan chunk, feed-forward.
PRESETS = {
    "tiny": (768, 384, 96, 16, 0.05, 0.25, 1.0, 16, 3072),
    "small": (512, 256, 48, 0, 0.08, 0.2, 1.0, 16, 1536),
    "base": (768, 384, 64, 32, 0.08, 0.2, 2.0, 16, 2048),
    "base_w16": (768, 256, 64, 16, 0.08, 0.2, 2.0, 16, 2048),
    "base_global": (768, 256, 64, 0, 0.08, 0.2, 2.0, 16, 2048),
    "medium": (1024, 512, 80, 32, 0.08, 0.25, 2.0, 16, 2816),
    "long_context": (256, 512, 32, 32, 0.08, 0.25, 6.0, 16, 512),
    "large_40b": (4096, 2048, 256, 64, 0.05, 0.2, 6.0, 32, 16384),
}


def _layer_case(op, preset, dtype, **sizes):
    dm, D, R, W, thr, scale, decay, chunk, inner = PRESETS[preset]
    case = dict(op=op, dtype=dtype, d_model=dm)
    if op == "ffn":
        case["d_inner"] = inner
    else:
        case.update(d_state=D, rank=R, window=W, threshold=thr, scale=scale, decay=decay, chunk=chunk)
    case.update(sizes)
    return case


def listed():
    return [
        # one projection of one token: the smallest call, launch and dispatch bound
        dict(name="bitlinear_gemv", op="bitlinear", dtype="bf16", M=1, K=4096, N=4096),
        # one projection of a prompt, in the parameters' default dtype
        dict(name="bitlinear_prefill", op="bitlinear", dtype="f32", M=2048, K=4096, N=4096),
        # one generated token for each of 32 sequences, a base layer
        dict(name="siso_decode", **_layer_case("siso_decode", "base_w16", "bf16", B=32, context=64)),
        # the headline: a base layer on a full batch of prompts
        dict(name="siso_base", **_layer_case("siso", "base_w16", "bf16", B=4, L=2048, cache=False)),
        # a medium layer on ragged prompts, filling the cache for the decode that follows
        dict(name="siso_medium", **_layer_case("siso", "medium", "bf16", B=3, L=1365, cache=True)),
        # a float32 layer on short, odd prompts
        dict(name="siso_tiny_f32", **_layer_case("siso", "tiny", "f32", B=2, L=333, cache=False)),
        # global entanglement (the small preset's kind) at base sizes: quadratic in the length
        dict(name="siso_global", **_layer_case("siso", "base_global", "bf16", B=4, L=2048, cache=False)),
        # one of the large single-head layers
        dict(name="siso_large", **_layer_case("siso", "large_40b", "bf16", B=1, L=4096, cache=False)),
        # the multi-head layer at large sizes on a long prompt: the largest call
        dict(name="mimo_large", **_layer_case("mimo", "large_40b", "bf16", heads=4, B=1, L=32768)),
        # one generated token for each of 32 sequences, the large multi-head layer
        dict(name="mimo_decode", **_layer_case("mimo_decode", "large_40b", "bf16", heads=4, B=32, context=64)),
        # the feed-forward of the medium block on ragged prompts
        dict(name="ffn_medium", **_layer_case("ffn", "medium", "bf16", B=3, L=1365)),
        # the whole tiny() model on two prompts of its training length, to logits
        dict(name="lm_tiny", op="lm", dtype="bf16", B=2, L=256),
    ]


def _log(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case of the listed ones' ranges: any entry point, preset sizes, batch and length spread over their logarithm."""
    op = rng.choice(["bitlinear", "bitlinear", "ffn", "siso", "siso", "siso", "global", "siso_decode", "mimo", "mimo_decode", "lm"])
    dtype = "f32" if rng.random() < 0.25 else "bf16"
    if op == "bitlinear":
        K, N = rng.choice([(4096, 4096), (4096, 11008), (11008, 4096), (768, 2432), (1024, 2816), (700, 1000), (2048, 4096)])
        return dict(op=op, dtype=dtype, M=_log(rng, 1, 8192), K=K, N=N)
    if op == "ffn":
        B = rng.randint(1, 4)
        return _layer_case(op, rng.choice(["tiny", "small", "base", "medium", "long_context"]), dtype, B=B, L=_log(rng, 1, 8192 // B))
    if op == "siso":
        preset = rng.choice(["tiny", "base", "base_w16", "medium", "long_context", "large_40b"])
        B = 1 if preset == "large_40b" else rng.randint(1, 8)
        return _layer_case(op, preset, dtype, B=B, L=_log(rng, 16, (4096 if preset == "large_40b" else 16384) // B), cache=rng.random() < 0.5)
    if op == "global":
        B = rng.randint(1, 8)
        return _layer_case("siso", rng.choice(["small", "base_global"]), dtype, B=B, L=_log(rng, 16, 8192 // B), cache=rng.random() < 0.5)
    if op == "siso_decode":
        return _layer_case(op, rng.choice(["tiny", "base", "base_w16", "medium", "long_context"]), dtype, B=_log(rng, 1, 128), context=_log(rng, 8, 256))
    if op == "mimo":
        preset = rng.choice(["base_w16", "medium", "large_40b"])
        return _layer_case(op, preset, dtype, heads=4, B=1, L=_log(rng, 64, 8192))
    if op == "mimo_decode":
        return _layer_case(op, rng.choice(["base_w16", "medium", "large_40b"]), dtype, heads=4, B=_log(rng, 1, 64), context=_log(rng, 64, 256))
    B = rng.randint(1, 4)
    return dict(op="lm", dtype=dtype, B=B, L=_log(rng, 16, 1024 // B))


def _tokens(case):
    return case["M"] if case["op"] == "bitlinear" else case["B"] * case.get("L", 1)


def _randn(case, seed, *shape):
    gen = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    return torch.randn(*shape, generator=gen, device="cuda").to(DTYPES[case["dtype"]])


def _module(case, seed):
    """The layer with its seeded initial weights, in eval, its packed weights laid out."""
    torch.manual_seed(int(seed))
    op = case["op"]
    with torch.device("cuda"):
        if op == "bitlinear":
            module = BitLinear(case["K"], case["N"])
        elif op == "ffn":
            module = FeedForward(TESMConfig(d_model=case["d_model"], d_intermediate=case["d_inner"]))
        elif op == "lm":
            module = TESMLMHeadModel(TESMConfig.tiny())
        else:
            kw = dict(d_model=case["d_model"], d_state=case["d_state"], ent_rank=case["rank"],
                      entanglement_window=case["window"], entanglement_threshold=case["threshold"],
                      entanglement_scale=case["scale"], decay_init_bias=case["decay"],
                      state_scan_chunk_size=case["chunk"], max_seq_len=max(2048, case.get("L", 0)))
            module = TESMMIMO_Optimized(n_heads=case["heads"], **kw) if op.startswith("mimo") else TESM_SISO(**kw)
    module = module.to(DTYPES[case["dtype"]]).eval()
    with torch.no_grad():
        for m in module.modules():
            if isinstance(m, BitLinear):
                m.packed_weight()
    return module


def prepare(case, seed):
    op = case["op"]
    module = _module(case, seed)
    state = {"op": op, "module": module}
    if op == "lm":
        gen = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
        vocab = module.tesm_config.vocab_size
        state["ids"] = torch.randint(0, vocab, (case["B"], case["L"]), generator=gen, device="cuda")
    elif op == "bitlinear":
        state["x"] = _randn(case, seed, case["M"], case["K"])
    elif op.endswith("_decode"):
        # a prompt of `context` tokens has filled the cache; u is the next token of each sequence
        x = _randn(case, seed, case["B"], case["context"] + 1, case["d_model"])
        cache = module.allocate_inference_cache(case["B"], case["context"] + 1)
        with torch.no_grad():
            module(x[:, :-1].contiguous(), inference_params={"state_cache": cache})
        state["cache"], state["x"] = cache, x[:, -1:].contiguous()
    else:
        state["x"] = _randn(case, seed, case["B"], case["L"], case["d_model"])
        state["fill"] = case.get("cache", False)
    return state


def run(state):
    op, module = state["op"], state["module"]
    with torch.no_grad():
        if op in ("bitlinear", "ffn"):
            return module(state["x"])
        if op == "lm":
            out, finals = module(state["ids"])
            return [out.logits, finals]
        if op.endswith("_decode"):
            # the step after the prompt, each time: it writes the same ring slot with the same values
            cache = dict(state["cache"])
            y, h = module(state["x"], inference_params={"state_cache": cache})
            return [y, h, cache["ent_k_cache"], cache["ent_v_cache"]]
        if state["fill"]:
            cache = module.allocate_inference_cache(state["x"].shape[0], module.max_seq_len)
            y, h = module(state["x"], inference_params={"state_cache": cache})
            return [y, h, cache["ent_k_cache"], cache["ent_v_cache"]]
        y, h = module(state["x"])
        return [y, h]


def _layer_work(case, M, rows_per_seq, weights_only=False):
    """(bytes, operations) of one layer on M tokens, `rows_per_seq` of them in a sequence (0: a decode step)."""
    dm, H = case["d_model"], case.get("heads", 1)
    HD, HR, W = case["d_state"] * H, case["rank"] * H, case["window"]
    n_in = 2 * dm + 3 * HD + 2 * HR
    el = 2 if case["dtype"] == "bf16" else 4
    weights = dm * n_in + 2 * HD * dm + dm * dm
    pairs = min(W, rows_per_seq or W) if W else (rows_per_seq + 1) / 2
    flops = 2 * M * weights + M * pairs * 2 * (HR + HD) + 4 * M * HD
    nbytes = weights / 4 + 2 * M * dm * el
    if rows_per_seq:
        nbytes += (M // rows_per_seq) * HD * 8
    else:  # a step reads and writes the state and reads the rings
        nbytes += M * HD * 16 + M * max(W, 1) * (HR + HD) * 4
    return nbytes, flops


def work(case):
    op, M = case["op"], _tokens(case)
    el = 2 if case["dtype"] == "bf16" else 4
    if op == "bitlinear":
        K, N = case["K"], case["N"]
        return {"bytes": N * K / 4 + M * (K + N) * el, "flops": 2 * M * N * K}
    if op == "ffn":
        dm, inner = case["d_model"], case["d_inner"]
        return {"bytes": 3 * dm * inner / 4 + 2 * M * dm * el, "flops": 6 * M * dm * inner}
    if op == "lm":
        cfg = TESMConfig.tiny()
        layer = _layer_case("siso", "tiny", case["dtype"])
        nbytes, flops = _layer_work(layer, M, case["L"])
        ffn = 3 * cfg.d_model * cfg.d_intermediate
        head = cfg.vocab_size * cfg.d_model
        return {"bytes": cfg.n_layer * (nbytes - 2 * M * cfg.d_model * el + ffn / 4) + head * el + M * cfg.vocab_size * el,
                "flops": cfg.n_layer * (flops + 2 * M * ffn) + 2 * M * head}
    nbytes, flops = _layer_work(case, M, 0 if op.endswith("_decode") else case["L"])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """A BitLinear's integer sums are exact, so only its rounding to the output dtype may move.  In a layer a rounding
    that falls the other way moves an int8 code or a ternary weight, and everything behind it: about 3e-4 of a float32
    layer's result and 1e-2 of a bf16 one's against 64 bits (3e-2 where long states decay slowly, or over 12 layers)."""
    f32 = case["dtype"] == "f32"
    if case["op"] == "bitlinear":
        return {"rel": 2e-6 if f32 else 8e-3}
    if case["op"] == "lm" or not f32:
        return {"rel": 0.03, "max": 0.99}
    return {"rel": 1e-3, "max": 0.3}


# ---------------------------------------------------------------------------------------------------------------
# 64-bit restatement
# ---------------------------------------------------------------------------------------------------------------
def _linear(module, x):
    """codes(x) / scale(x) times codes(w) / scale(w), summed in 64 bits; codes and scales in the module's dtype."""
    dt = module.weight.dtype
    x = x.to(dt)
    s = 127 / x.abs().amax(dim=-1, keepdim=True).clamp_min(module.bit_eps)
    qx = (x * s).round().clamp(-128, 127).double() / s.double()
    w = module.weight.detach()
    sw = 1.0 / w.abs().mean().clamp_min(module.bit_eps)
    codes = (w * sw).round().clamp(-1, 1)
    one = (torch.ones_like(sw) / sw).double()
    rows = qx.reshape(-1, qx.shape[-1])
    out = torch.empty(rows.shape[0], w.shape[0], dtype=torch.float64, device=x.device)
    cd = codes.double().t().contiguous()
    for r in range(0, rows.shape[0], 8192):
        out[r:r + 8192] = (rows[r:r + 8192] @ cd) * one
    return out.reshape(*x.shape[:-1], w.shape[0])


def _rope(x, base, first=0):
    """x (B, L, H, R): rotary positions, the table in 64 bits of the float32 angles."""
    half = x.shape[-1] // 2
    pos = torch.arange(first, first + x.shape[1], device=x.device, dtype=torch.float32)
    idx = torch.arange(half, device=x.device, dtype=torch.float32)
    theta = (pos[:, None] * (1.0 / base ** (2.0 * idx / x.shape[-1]))).double()[:, None]
    c, s = theta.cos(), theta.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


def _ternary(scores, threshold):
    return (scores > threshold).double() - (scores < -threshold).double()


def _global_bias(layer, L, dt, device):
    """The relative-position bias by distance: positions and frequencies of the layer's dtype, functions and sums in 64 bits."""
    n = layer.global_rel_pos_dim
    pos = torch.arange(L, device=device, dtype=dt)
    freq = torch.arange(1, n + 1, device=device, dtype=dt) * math.pi / 1000.0
    emb = layer.global_rel_pos_embed.detach().to(dt).double()
    values, where = torch.unique(pos[:, None] - pos[None, :], return_inverse=True)
    ang = (values[:, None] * freq[None, :]).double()
    bias = ((ang.sin() + ang.cos()) * emb).sum(-1)
    bias = bias * layer.global_rel_pos_scale.detach().to(dt).double() + layer.global_rel_pos_bias.detach().to(dt).double()
    return bias[where]


def _mix(layer, q, k, S, dt):
    """q, k (B, L, H, R) rotated, S (B, L, H, D): the ternary-weighted mean of the window (or of all earlier states)."""
    B, L, H, R = q.shape
    thr = layer.entanglement_threshold
    if layer.entanglement_window <= 0:
        qf, kf, Sf = q.reshape(B, L, -1), k.reshape(B, L, -1), S.reshape(B, L, -1)
        bias = _global_bias(layer, L, dt, q.device)
        out = torch.empty_like(Sf)
        for b in range(B):
            t = _ternary((qf[b] @ kf[b].t()) / math.sqrt(H * R) + bias, thr).tril_()
            out[b] = (t / t.abs().sum(-1, keepdim=True).clamp_min(1.0)) @ Sf[b]
        return out.reshape(S.shape)
    W = min(layer.entanglement_window, L)
    lb = layer.local_entanglement_bias.detach().to(dt).double()
    lb = (lb if lb.dim() == 2 else lb[None])[:, -W:]
    total, norm = torch.zeros_like(S), torch.zeros(B, L, H, 1, dtype=torch.float64, device=S.device)
    for w in range(W):
        back = W - 1 - w
        n = L - back
        t = _ternary((q[:, back:] * k[:, :n]).sum(-1) / math.sqrt(R) + lb[:, w], thr)[..., None]
        total[:, back:].addcmul_(t, S[:, :n])
        norm[:, back:] += t.abs()
    return total / norm.clamp_min(1.0)


def _split(layer, p, H, dt):
    dm, D, R = layer.d_model, layer.d_state, layer.ent_rank
    p = p.to(dt).double()  # in_proj's output is a tensor of the layer's dtype
    local, sv, decay, write, gate, q, k = torch.split(p, [dm, H * D, H * D, H * D, dm, H * R, H * R], dim=-1)
    B, L = p.shape[:2]
    shape = (B, L, H, D)
    decay = torch.sigmoid(decay.reshape(shape) + layer.decay_bias.detach().double().reshape(H, D))
    update = torch.sigmoid(write.reshape(shape)) * torch.tanh(sv.reshape(shape))
    return local, decay, update, torch.sigmoid(gate), q.reshape(B, L, H, R), k.reshape(B, L, H, R)


def _scan(decay, update):
    S = torch.empty_like(update)
    h = torch.zeros_like(update[:, 0])
    for t in range(update.shape[1]):
        h = torch.addcmul(update[:, t], decay[:, t], h)
        S[:, t] = h
    return S


def _output(layer, local, gate, te, change):
    sp, ep = _linear(layer.state_proj, te), _linear(layer.ent_proj, change)
    return _linear(layer.out_proj, local + gate * sp + ep)


def _prefill(layer, u, cross=None):
    """(y, final state, states, rotated keys) of a prefill."""
    H, dt = getattr(layer, "n_heads", 1), u.dtype if u.dtype != torch.float64 else layer.in_proj.weight.dtype
    B, L = u.shape[:2]
    local, decay, update, gate, q, k = _split(layer, _linear(layer.in_proj, u), H, dt)
    q, k = _rope(q, layer.rope_base), _rope(k, layer.rope_base)
    if cross is not None:
        q = q + _linear(layer.cross_layer_q_proj, cross).reshape(q.shape)
    S = _scan(decay, update)
    del decay, update
    A = _mix(layer, q, k, S, dt)
    if H == 1 and not hasattr(layer, "mimo_x"):
        A.sub_(S).mul_(layer.entanglement_scale)
        E, C, first = (S + A).reshape(B, L, -1), A.reshape(B, L, -1), S
    else:  # the ranks are scaled copies of one state, merged by mimo_o
        x, o = layer.mimo_x.detach().double(), layer.mimo_o.detach().double()
        coef = (x * x * o).sum(1)
        if layer.entanglement_window > 0:
            A.sub_(S).mul_(layer.entanglement_scale).add_(S)
        E, C, first = (A * coef).reshape(B, L, -1), ((A - S) * coef).reshape(B, L, -1), S * (x[:, 0] ** 2)
    y = _output(layer, local, gate, torch.tanh(E), C)
    h = first[:, -1].clone()
    return y, h.reshape(B, -1) if H == 1 else h, first, k


def _decode(layer, u, context):
    """The step after a prompt of `context` tokens: the rings hold the prompt's last states, the newest slot 0."""
    H, dt = getattr(layer, "n_heads", 1), u.dtype
    B, W = u.shape[0], max(layer.entanglement_window, 1)
    D, R = layer.d_state, layer.ent_rank
    _, h, S, k = _prefill(layer, u[:, :-1])
    rk = torch.zeros(B, W, H, R, dtype=torch.float64, device=u.device)
    rv = torch.zeros(B, W, H, D, dtype=torch.float64, device=u.device)
    n = min(W, context)
    rk[:, W - n:], rv[:, W - n:] = k[:, -n:], S[:, -n:]
    local, decay, update, gate, q, kn = _split(layer, _linear(layer.in_proj, u[:, -1:]), H, dt)
    q, kn = _rope(q, layer.rope_base, context), _rope(kn, layer.rope_base, context)
    new = decay[:, 0] * h.reshape(B, H, D) + update[:, 0]
    rk[:, 0], rv[:, 0] = kn[:, 0], new
    valid = min(context + 1, W)
    lb = layer.local_entanglement_bias
    scores = (q * rk[:, :valid]).sum(-1) / math.sqrt(R)
    if lb is not None:
        lb = lb.detach().to(dt).double()
        scores = scores + (lb if lb.dim() == 2 else lb[None]).t()[W - valid:]
    t = _ternary(scores, layer.entanglement_threshold)[..., None]
    A = (t * rv[:, :valid]).sum(1) / t.abs().sum(1).clamp_min(1.0)
    C = (layer.entanglement_scale * (A - new)).reshape(B, 1, -1)
    y = _output(layer, local, gate, torch.tanh(new.reshape(B, 1, -1) + C), C)
    state = new.reshape(B, -1) if H == 1 else new
    ring = (B, W, R) if H == 1 else (B, W, H, R)
    return [y, state, rk.reshape(ring), rv.reshape(*ring[:-1], D)]


def _ffn(module, x):
    return _linear(module.down_proj, F.silu(_linear(module.gate_proj, x)) * _linear(module.up_proj, x))


def _norm(module, x):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + module.eps) * module.weight.detach().double()


def _lm(model, ids):
    net = model.backbone
    hidden = (net.embedding(ids) + net.position_embedding(torch.arange(ids.shape[1], device=ids.device))).double()
    residual, cross, finals = 0.0, None, []
    for block in net.layers:
        residual = hidden + residual
        hidden, h, cross, _ = _prefill(block.mixer, _norm(block.norm, residual), cross)
        cross = cross.reshape(*ids.shape, -1)
        finals.append(h)
        residual = hidden + residual
        hidden = _ffn(block.mlp, _norm(block.norm2, residual))
    return [_norm(net.norm_f, hidden + residual) @ model.lm_head.weight.detach().double().t(), finals]


def exact(case, seed):
    op = case["op"]
    module = _module(case, seed)
    with torch.no_grad():
        if op == "lm":
            return _lm(module, prepare(case, seed)["ids"])
        if op.endswith("_decode"):
            return _decode(module, _randn(case, seed, case["B"], case["context"] + 1, case["d_model"]), case["context"])
        if op == "bitlinear":
            return _linear(module, _randn(case, seed, case["M"], case["K"]))
        x = _randn(case, seed, case["B"], case["L"], case["d_model"])
        if op == "ffn":
            return _ffn(module, x)
        y, h, S, k = _prefill(module, x)
        if not case.get("cache"):
            return [y, h]
        B, L, W = case["B"], case["L"], max(case["window"], 1)
        n = min(W, L)
        rk = torch.zeros(B, W, case["rank"], dtype=torch.float64, device="cuda")
        rv = torch.zeros(B, W, case["d_state"], dtype=torch.float64, device="cuda")
        rk[:, W - n:], rv[:, W - n:] = k[:, -n:].reshape(B, n, -1), S[:, -n:].reshape(B, n, -1)
        return [y, h, rk, rv]
