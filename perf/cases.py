"""The work that users of this package have it do, as cases that can be timed and checked.

A case is a plain dict: ``kind`` names the path, the rest its sizes and options.

* ``scan``      the recurrence itself: ``field_scan`` / ``field_scan_norm`` (prompt processing) and
                ``fused_field_read`` with its gradients (training), over raw of either type, packed
                or a column slice of the fused input projection, zero or continued state;
* ``block``     a FieldBlock: one decode token, a prefill, a training pass;
* ``refresh``   a RefreshBlock's prefill (latent attention over windows and landmarks);
* ``mamba``     a Mamba2ResidualBlock's prefill;
* ``softpatch`` a BoundaryStateMixer's forward (the boundary scan inside);
* ``model``     the promoted 24-block model: a prefill, and one decode token of a batch of streams as
                a generation loop runs it, replayed from a HIP graph with its argmax feedback.

``exact`` restates every path in float64 with plain torch ops.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import fields_lm_amd as fl
from fields_lm_amd import model as M

VOCAB, DIM, FF = 16_384, 1024, 2528          # the promoted model's sizes
LANDMARK = 256


# ======================================================================================
# the cases
# ======================================================================================

def listed():
    return [
        # a chat turn of a few dozen tokens appended to a running conversation: two streams, the
        # state carried in and out, raw read in place from the fused projection
        dict(name="scan_short_turn", kind="scan", op="norm", B=2, T=61, C=512, raw="bf16", out="bf16",
             packed=True, state=True),
        # a research run at a width that is no multiple of the tile, full fp32
        dict(name="scan_ragged_fp32", kind="scan", op="read", B=3, T=1531, C=331, raw="fp32", out="fp32",
             packed=False, state=False),
        # a book-length document prefilled in one call
        dict(name="scan_long_norm", kind="scan", op="norm", B=1, T=65536, C=512, raw="bf16", out="bf16",
             packed=True, state=True),
        # the recurrence of a training step: fp32 read out, then all gradients
        dict(name="scan_train", kind="scan", op="train", B=8, T=2048, C=512, raw="bf16", out="fp32",
             packed=False, state=False),
        # one token of 64 streams through one block, called eagerly
        dict(name="block_step", kind="block", op="step", B=64, T=1, dim=1024, ff=2528),
        # a batch of prompts through one block
        dict(name="block_prefill", kind="block", op="prefill", B=4, T=2048, dim=1024, ff=2528),
        # one block's share of a training step: bf16 autocast over fp32 weights
        dict(name="block_train", kind="block", op="train", B=4, T=1024, dim=1024, ff=2528),
        # an attention block of a prefill whose length is no multiple of the window
        dict(name="refresh_prefill", kind="refresh", B=4, T=1900, dim=1024, heads=16, kv=4, window=512, ff=2528),
        # the state-space blocks of the same prefill
        dict(name="mamba_prefill", kind="mamba", B=4, T=2048, dim=1024),
        # the boundary mixer of the same prefill
        dict(name="softpatch", kind="softpatch", B=4, T=2048, dim=1024),
        # a batch of prompts through the whole model, up to the first token's logits
        dict(name="model_prefill", kind="model", op="prefill", B=4, T=2048),
        # one token of 64 streams through the whole model, inside a generation loop
        dict(name="model_decode", kind="model", op="decode", B=64, T=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "block", "block", "block", "refresh", "mamba", "softpatch",
                       "model"])
    if kind == "scan":
        op = rng.choice(["norm", "norm", "read", "train"])
        C = rng.choice([512, 512, _log_int(rng, 32, 1024), 64 * rng.randint(1, 16)])
        B = _log_int(rng, 1, 16)
        T = max(1, min(_log_int(rng, 16, 65536), (1 << 25) // (B * C)))
        raw = rng.choice(["bf16", "bf16", "fp32"])
        return dict(kind=kind, op=op, B=B, T=min(T, 4096) if op == "train" else T, C=C, raw=raw,
                    out="fp32" if op == "train" else rng.choice(["bf16", "fp32"]),
                    packed=op != "train" and rng.random() < 0.5, state=op != "train" and rng.random() < 0.5)
    if kind == "block":
        op = rng.choice(["step", "prefill", "train"])
        dim = rng.choice([1024, 1024, 8 * _log_int(rng, 16, 160)])
        ff = rng.choice([2272, 2528, 2784]) if dim == 1024 else 32 * max(4, round(dim / 12))
        if op == "step":
            return dict(kind=kind, op=op, B=_log_int(rng, 1, 128), T=1, dim=dim, ff=ff)
        B = _log_int(rng, 1, 8)
        return dict(kind=kind, op=op, B=B, T=min(_log_int(rng, 32, 4096), 8192 // B), dim=dim, ff=ff)
    if kind == "refresh":
        heads = rng.choice([16, 16, 8, 12])
        B = _log_int(rng, 1, 8)
        return dict(kind=kind, B=B, T=min(_log_int(rng, 32, 4096), 8192 // B), dim=64 * heads, heads=heads,
                    kv=heads // 4, window=rng.choice([256, 512, 1024]), ff=2528)
    if kind == "mamba":
        B = _log_int(rng, 1, 8)
        return dict(kind=kind, B=B, T=min(_log_int(rng, 32, 4096), 8192 // B), dim=rng.choice([1024, 1024, 512, 768]))
    if kind == "softpatch":
        B = _log_int(rng, 1, 16)
        return dict(kind=kind, B=B, T=min(_log_int(rng, 32, 8192), 16384 // B), dim=rng.choice([1024, 1024, 512, 768]))
    if rng.random() < 0.5:
        B = _log_int(rng, 1, 4)
        return dict(kind=kind, op="prefill", B=B, T=_log_int(rng, 64, 8192 // B))
    return dict(kind=kind, op="decode", B=_log_int(rng, 1, 64), T=_log_int(rng, 64, 2048))


# ======================================================================================
# inputs
# ======================================================================================

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _dtype(name):
    return {"bf16": torch.bfloat16, "fp32": torch.float32}[name]


def _transition(C, g):
    """The parameters of a mixer that has moved a little from its initial ring."""
    ring = torch.linspace(0.85, 0.999, C, device="cuda")
    logit = torch.log(ring / (1.0 - ring)) + 0.1 * torch.randn(C, device="cuda", generator=g)
    radius = torch.sigmoid(logit).clamp(0.50, 0.99995)
    theta = torch.linspace(0.03, math.pi * 0.97, C, device="cuda") + 0.01 * torch.randn(C, device="cuda", generator=g)
    return (radius * torch.cos(theta)).contiguous(), (radius * torch.sin(theta)).contiguous(), \
        torch.sqrt((1.0 - radius.square()).clamp_min(1e-4)).contiguous()


def _scan_inputs(c, seed):
    g = _gen(seed)
    B, T, C = c["B"], c["T"], c["C"]
    dt = _dtype(c["raw"])
    width = 5 * C if c["packed"] else 3 * C  # [raw 3C | gate 2C], as the fused input projection writes it
    raw = (0.8 * torch.randn(B, T, width, device="cuda", generator=g)).to(dt)[..., :3 * C]
    tr, ti, gamma = _transition(C, g)
    state = 0.5 * torch.randn(B, 2 * C, device="cuda", generator=g) if c["state"] else None
    weight = 1.0 + 0.1 * torch.randn(4 * C, device="cuda", generator=g)
    grad = torch.randn(B, T, 4 * C, device="cuda", generator=g) if c["op"] == "train" else None
    return raw, tr, ti, gamma, state, weight, grad


def _perturb(module, g):
    """Parameters as training leaves them: the zero-initialised gates and projections and the unit
    norm weights moved off their initial values."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith(("residual_gate.weight", "softpatch.up.weight", "softpatch.score.weight")) or \
                    (isinstance(module, M.BoundaryStateMixer) and name in ("up.weight", "score.weight")):
                p.normal_(0.0, 0.02, generator=g)
            elif "norm" in name and name.endswith("weight"):
                p.add_(0.1 * torch.randn(p.shape, device=p.device, generator=g))
            elif name.endswith("global_mix_logit"):
                p.add_(0.3 * torch.randn(p.shape, device=p.device, generator=g))
    return module


def _make(build, seed, cast=True):
    torch.manual_seed(int(seed))
    with torch.device("cuda"):
        module = build()
    _perturb(module, _gen(seed + 1))
    return (M.cast_for_inference(module) if cast else module).eval()


def _build(c):
    kind = c["kind"]
    if kind == "block":
        return fl.FieldBlock(c["dim"], "triton", 32, 32, 64, c["ff"])
    if kind == "refresh":
        return M.RefreshBlock(c["dim"], c["heads"], c["kv"], M.LATENT_DIM, c["window"], LANDMARK, c["ff"])
    if kind == "mamba":
        return M.Mamba2ResidualBlock(c["dim"], **M.MAMBA)
    if kind == "softpatch":
        return M.BoundaryStateMixer(c["dim"], M.SOFTPATCH_RANK, vocab=VOCAB)
    core = M.FieldTokenSystem(vocab=VOCAB, dim=DIM, ff_hidden=FF)
    with torch.no_grad():
        core.emb.weight.normal_(0.0, 0.02)
    return core


def _module(c, seed):
    return _make(lambda: _build(c), seed, cast=c.get("op") != "train")


def _hidden(c, seed, dtype):
    """A residual stream: unit-scale activations."""
    return torch.randn(c["B"], c["T"], c["dim"], device="cuda", generator=_gen(seed + 2)).to(dtype)


def _tokens(c, seed):
    n = c["T"] + (1 if c["op"] == "decode" else 0)
    return torch.randint(0, VOCAB, (c["B"], n), device="cuda", generator=_gen(seed + 3))


def _max_len(c):
    return c["T"] + 2048


class _autocast:
    """Inference of the whole model: no gradients, bf16 autocast over bf16 weights."""

    def __enter__(self):
        self.a, self.b = torch.no_grad(), torch.autocast(device_type="cuda", dtype=torch.bfloat16)
        self.a.__enter__()
        self.b.__enter__()

    def __exit__(self, *e):
        self.b.__exit__(*e)
        self.a.__exit__(*e)


def prepare(case, seed):
    c = case
    if c["kind"] == "scan":
        raw, tr, ti, gamma, state, weight, grad = _scan_inputs(c, seed)
        if c["op"] == "train":
            raw, tr, ti, gamma = (t.requires_grad_() for t in (raw, tr, ti, gamma))
        return dict(c=c, raw=raw, tr=tr, ti=ti, gamma=gamma, state=state, weight=weight, grad=grad)
    m = _module(c, seed)
    if c["kind"] == "model":
        tokens = _tokens(c, seed)
        if c["op"] == "prefill":
            return dict(c=c, m=m, tokens=tokens)
        return _decode_loop(c, m, tokens)
    s = dict(c=c, m=m)
    if c["kind"] == "block" and c["op"] == "step":
        g = _gen(seed + 2)
        s["x"] = torch.randn(c["B"], c["dim"], device="cuda", generator=g).to(torch.bfloat16)
        s["state"] = 0.5 * torch.randn(c["B"], c["dim"], device="cuda", generator=g)
        s["params"] = m.mixer.decode_params()
    elif c["kind"] == "block" and c["op"] == "train":
        s["x"] = _hidden(c, seed, torch.float32).requires_grad_()
        s["grad"] = torch.randn(c["B"], c["T"], c["dim"], device="cuda", generator=_gen(seed + 4))
    else:
        s["x"] = _hidden(c, seed, torch.bfloat16)
        s["tokens"] = torch.randint(0, VOCAB, (c["B"], c["T"]), device="cuda", generator=_gen(seed + 3))
    return s


def _decode_loop(c, core, tokens):
    """A generation loop after its prompt: the step and its argmax feedback captured once, the cache
    and the token put back to where the prompt ended."""
    with _autocast():
        _, cache = core.prefill(tokens[:, :c["T"]], max_len=_max_len(c))
        kept = _cache_leaves(cache)
        saved = [t.clone() for t in kept]
        tok = tokens[:, c["T"]].clone()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            core.step(tok, cache)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            logits = core.step(tok, cache)
            tok.copy_(logits.argmax(-1))
        for t, v in zip(kept, saved):
            t.copy_(v)
        tok.copy_(tokens[:, c["T"]])
    return dict(c=c, m=core, cache=cache, tok=tok, graph=graph, logits=logits)


def _cache_leaves(cache):
    out = [cache["softpatch"], cache["pos"]]
    for st in cache["blocks"]:
        out.extend(st.values() if isinstance(st, dict) else [st])
    return out


# ======================================================================================
# one pass
# ======================================================================================

def run(s):
    c = s["c"]
    return {"scan": _run_scan, "block": _run_block, "refresh": _run_refresh, "mamba": _run_mamba,
            "softpatch": _run_softpatch, "model": _run_model}[c["kind"]](c, s)


def _run_scan(c, s):
    if c["op"] == "train":
        read = fl.fused_field_read(s["raw"], s["tr"], s["ti"], s["gamma"], 32, 64)
        grads = torch.autograd.grad(read, (s["raw"], s["tr"], s["ti"], s["gamma"]), s["grad"])
        return {"read": read, "grads": list(grads)}
    with torch.no_grad():
        if c["op"] == "norm":
            out = fl.field_scan_norm(s["raw"], s["tr"], s["ti"], s["gamma"], s["weight"], 1e-6,
                                     state_in=s["state"], return_state=c["state"], out_dtype=_dtype(c["out"]))
        else:
            out = fl.field_scan(s["raw"], s["tr"], s["ti"], s["gamma"], state_in=s["state"],
                                return_state=c["state"], read_dtype=_dtype(c["out"]))
    return list(out) if c["state"] else [out]


def _run_block(c, s):
    m = s["m"]
    if c["op"] == "train":
        with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = m(s["x"])
        params = list(m.parameters())
        return {"y": y, "grads": list(torch.autograd.grad(y, [s["x"], *params], s["grad"]))}
    with torch.no_grad():
        if c["op"] == "step":
            return {"y": m.step(s["x"], s["state"], s["params"]), "state": s["state"]}
        y, state = m.prefill(s["x"])
        return {"y": y, "state": state}


def _run_refresh(c, s):
    with torch.no_grad():
        y, st = s["m"].prefill(s["x"], c["T"] + 256)
    return {"y": y, **st}


def _run_mamba(c, s):
    with torch.no_grad():
        y, st = s["m"].prefill(s["x"], c["T"] + 256)
    return {"y": y, **st}


def _run_softpatch(c, s):
    with torch.no_grad():
        y, last = s["m"](s["x"], s["tokens"], return_state=True)
    return {"y": y, "last": last}


def _run_model(c, s):
    if c["op"] == "decode":
        s["graph"].replay()
        return {"logits": s["logits"], "states": s["cache"]["blocks"], "softpatch": s["cache"]["softpatch"]}
    with _autocast():
        logits, cache = s["m"].prefill(s["tokens"], _max_len(c))
    return {"logits": logits, "states": cache["blocks"], "softpatch": cache["softpatch"]}


# ======================================================================================
# what a pass cannot do without
# ======================================================================================

def _block_work(tokens, dim, ff, es=2):
    weights = 5 * dim * dim + dim * dim // 2 + 3 * dim * ff  # write, out, gate, FFN
    return weights * es + 2 * tokens * dim * es, 2 * tokens * weights + 40 * tokens * dim


def _refresh_work(B, T, dim, window, ff):
    weights = dim * (dim + 256) + 256 * dim // 2 + 2 * dim * dim + 3 * dim * ff
    w = min(window, T)
    pairs = B * T * ((w + 1) / 2 + 1 + T / (2 * LANDMARK))  # query-key pairs of every head
    return weights * 2 + 2 * B * T * dim * 2, 2 * B * T * weights + 4 * pairs * dim


def _mamba_work(B, T, dim):
    inner = 2 * dim
    weights = dim * (2 * inner + 256 + inner // 64) + inner * dim
    # the recurrence itself: state update and readout, 64 x 128 per head and token
    return weights * 2 + 2 * B * T * dim * 2, 2 * B * T * weights + 4 * B * T * inner * 128


def _softpatch_work(B, T, dim):
    weights = dim * 65 + 128 * dim
    return weights * 2 + 2 * B * T * dim * 2, 2 * B * T * weights


def work(case):
    c = case
    if c["kind"] == "scan":
        n = c["B"] * c["T"] * c["C"]
        e, o = (2 if c["raw"] == "bf16" else 4), (2 if c["out"] == "bf16" else 4)
        if c["op"] == "train":  # forward, then raw, read and its gradient in, raw's gradient out
            return {"bytes": n * (3 * e + 16) + n * (3 * e + 16 + 3 * e), "flops": n * 120}
        return {"bytes": n * (3 * e + 4 * o) + (16 * c["B"] * c["C"] if c["state"] else 0), "flops": n * 40}
    B, T = c["B"], c["T"]
    if c["kind"] == "block":
        b, f = _block_work(B * T, c["dim"], c["ff"], 4 if c["op"] == "train" else 2)
        if c["op"] == "train":
            b, f = 3 * b, 3 * f
        return {"bytes": b + 8 * B * c["dim"], "flops": f}
    if c["kind"] == "refresh":
        b, f = _refresh_work(B, T, c["dim"], c["window"], c["ff"])
    elif c["kind"] == "mamba":
        b, f = _mamba_work(B, T, c["dim"])
    elif c["kind"] == "softpatch":
        b, f = _softpatch_work(B, T, c["dim"])
    else:
        n = T if c["op"] == "prefill" else 1
        b, f = 2 * VOCAB * DIM, 2 * B * VOCAB * DIM
        parts = [_block_work(B * n, DIM, FF)] * 18 + [_mamba_work(B, n, DIM)] * 2 + [_softpatch_work(B, n, DIM)]
        parts += [_refresh_work(B, n, DIM, w, FF) for w in (256, 512, 1024, 1024)]
        b += sum(p[0] for p in parts)
        f += sum(p[1] for p in parts)
        if c["op"] == "decode":  # recurrent states in and out, window keys and values in
            b += B * (18 * 8 * DIM + 2 * 2 * 4 * 2 * DIM * 128 + 2 * 2 * 256 * (256 + 512 + 2 * 1024) // 2)
    return {"bytes": b, "flops": f}


def tolerance(case):
    c = case
    if c["kind"] == "scan":
        if "bf16" in (c["out"], c["raw"] if c["op"] == "train" else ""):
            return {"rel": 5e-3}  # one rounding to bf16 (1.7e-3 against float64)
        return {"rel": 4e-6}      # fp32 throughout (1e-7 to 2e-7)
    if c["kind"] == "block":      # 2.7e-3; the gradients 5.8e-3
        return {"rel": 2.5e-2 if c["op"] == "train" else 1e-2}
    if c["kind"] == "refresh":    # 4.4e-3
        return {"rel": 2e-2}
    if c["kind"] == "mamba":      # 2.7e-3
        return {"rel": 1.2e-2}
    if c["kind"] == "softpatch":  # 3.7e-3
        return {"rel": 1.5e-2}
    return {"rel": 8e-2}          # 24 layers in bf16: up to 2e-2


# ======================================================================================
# the same in float64
# ======================================================================================

def _lin(x, layer):
    y = x @ layer.weight.double().t()
    return y if layer.bias is None else y + layer.bias.double()


def _rms(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _recurrence(raw, tr, ti, gamma, s0=None):
    """read [B,T,4C] and the last state [B,2C] of the Field recurrence."""
    zr, zi, zv = raw.chunk(3, dim=-1)
    v = 0.9 * torch.sigmoid(zv)
    lam = torch.complex(tr, ti)
    a = ((1.0 - v) * lam).unbind(1)
    b = (gamma * v * torch.complex(torch.tanh(zr), torch.tanh(zi))).unbind(1)
    C = tr.numel()
    s = torch.zeros_like(b[0]) if s0 is None else torch.complex(s0[:, :C], s0[:, C:])
    states = [s]
    for at, bt in zip(a, b):
        s = torch.addcmul(bt, at, s)
        states.append(s)
    h = torch.stack(states, 1)
    disp = v * lam * h[:, :-1]
    h = h[:, 1:]
    return torch.cat((h.real, h.imag, disp.real, disp.imag), -1), torch.cat((s.real, s.imag), -1)


def _field64(blk, x, s0=None):
    m = blk.mixer
    radius = torch.sigmoid(m.radius_logit.double()).clamp(0.50, 0.99995)
    theta = m.theta.double()
    gamma = torch.sqrt((1.0 - radius.square()).clamp_min(1e-4))
    read, last = _recurrence(_lin(x, m.write_proj), radius * torch.cos(theta), radius * torch.sin(theta), gamma, s0)
    x = x + _lin(_rms(read, m.read_norm.weight, m.read_norm.eps), m.out_proj) * torch.sigmoid(_lin(x, m.gate_proj))
    h = _rms(x, blk.ff_norm.weight, blk.ff_norm.eps)
    first, second = (blk.ff.w12, blk.ff.w3) if hasattr(blk.ff, "w12") else (blk.ff.gate_up, blk.ff.down)
    gate, up = _lin(h, first).chunk(2, dim=-1)
    return x + _lin(F.silu(gate) * up, second), last


def _rope(x, pos):
    """x [..., T, hd] rotated at positions pos [T]."""
    hd = x.shape[-1]
    inv = 1.0 / (10000.0 ** (torch.arange(0, hd, 2, device=x.device, dtype=torch.float64) / hd))
    f = pos.double()[:, None] * inv
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * f.cos() - b * f.sin(), b * f.cos() + a * f.sin()), -1)


def _softmax_rows(q, k, v, allowed):
    s = (q @ k.transpose(-1, -2)) * q.shape[-1] ** -0.5
    return torch.softmax(s.masked_fill(~allowed, float("-inf")), -1) @ v


def _refresh64(blk, x, max_len=None):
    att = blk.attn
    B, T, dim = x.shape
    hq, hk, hd, c = att.q_heads, att.kv_heads, att.head_dim, att.landmark_chunk
    z = _rms(x, blk.norm1.weight, blk.norm1.eps)
    qraw, latent = _lin(z, att.q_latent_proj).split((hq * hd, att.latent_dim), -1)
    pos = torch.arange(T, device=x.device)

    def heads(t, n):
        return t.view(t.shape[0], -1, n, hd).transpose(1, 2)

    kr, vr = _lin(latent, att.kv_up).split(hk * hd, -1)
    q, k, v = _rope(heads(qraw, hq), pos), _rope(heads(kr, hk), pos), heads(vr, hk)
    full, w, rep = T // c, min(att.local_window, T), hq // hk
    mean = latent[:, :full * c].view(B, full, c, -1).mean(2)
    lk, lv = _lin(mean, att.kv_up).split(hk * hd, -1)
    lk, lv = heads(lk, hk), heads(lv, hk)
    if full:
        lk = _rope(lk, torch.arange(c - 1, full * c, c, device=x.device))
    mix = torch.sigmoid(att.global_mix_logit.double())
    y = torch.empty(B, hq, T, hd, device=x.device, dtype=torch.float64)
    chunk = torch.arange(T, device=x.device) // c
    see = torch.cat((torch.ones(T, 1, device=x.device, dtype=torch.bool),
                     torch.arange(full, device=x.device)[None] < chunk[:, None]), 1)
    zero = torch.zeros(hk, 1, hd, device=x.device, dtype=torch.float64)
    for b in range(B):
        for g in range(0, T, w):
            e = min(g + w, T)
            causal = torch.ones(e - g, e - g, device=x.device, dtype=torch.bool).tril()
            y[b, :, g:e] = _softmax_rows(q[b, :, g:e], k[b, :, g:e].repeat_interleave(rep, 0),
                                         v[b, :, g:e].repeat_interleave(rep, 0), causal)
        if full:
            gk = torch.cat((zero, lk[b]), 1).repeat_interleave(rep, 0)
            gv = torch.cat((zero, lv[b]), 1).repeat_interleave(rep, 0)
            y[b] += mix * _softmax_rows(q[b], gk, gv, see)
    a = _lin(y.transpose(1, 2).reshape(B, T, dim), att.out_proj)
    x = x + torch.sigmoid(_lin(z, blk.residual_gate)) * a
    gate, up = _lin(_rms(x, blk.norm2.weight, blk.norm2.eps), blk.ff.gate_up).chunk(2, -1)
    out = x + _lin(F.silu(gate) * up, blk.ff.down)
    if max_len is None:
        return out, None
    n_land, g0 = (max_len - 1) // c + 1, T // att.local_window * att.local_window
    st = {"kt": x.new_zeros(B, hk, hd, att.local_window), "v": x.new_zeros(B, hk, att.local_window, hd),
          "lkt": x.new_zeros(B, hk, hd, 1 + n_land), "lv": x.new_zeros(B, hk, 1 + n_land, hd),
          "lat_sum": latent[:, full * c:].sum(1)}
    st["kt"][..., :T - g0] = k[:, :, g0:].transpose(-1, -2)
    st["v"][:, :, :T - g0] = v[:, :, g0:]
    st["lkt"][..., 1:1 + full] = lk.transpose(-1, -2)
    st["lv"][:, :, 1:1 + full] = lv
    return out, st


def _mamba64(blk, x, states=False):
    m = blk.mixer
    B, T, _ = x.shape
    H, P, N, K = m.nheads, m.headdim, m.d_state, m.d_conv
    z, xbc_raw, dt = _lin(_rms(x, blk.norm.weight, blk.norm.eps), m.in_proj).split((m.d_inner, m.conv_dim, H), -1)
    pad = F.pad(xbc_raw, (0, 0, K - 1, 0))
    w = m.conv1d.weight.double()[:, 0]
    xbc = F.silu(sum(pad[:, k:k + T] * w[:, k] for k in range(K)) + m.conv1d.bias.double())
    xs, bm, cm = xbc.split((m.d_inner, N, N), -1)
    xh = xs.reshape(B, T, H, P)
    dt = F.softplus(dt + m.dt_bias.double())
    decay = torch.exp(dt * -torch.exp(m.A_log.double()))
    s = torch.zeros(B, H, P, N, device=x.device, dtype=torch.float64)
    y = torch.empty_like(xh)
    u = xh * dt[..., None]
    for t in range(T):
        s = torch.addcmul(s * decay[:, t, :, None, None], u[:, t, :, :, None], bm[:, t, None, None, :])
        y[:, t] = (s.view(B, H * P, N) @ cm[:, t, :, None]).view(B, H, P)
    y = (y + m.D.double()[:, None] * xh).reshape(B, T, m.d_inner) * F.silu(z)
    out = x + _lin(_rms(y, m.norm.weight, m.norm.eps), m.out_proj)
    if not states:
        return out, None
    conv = F.pad(xbc_raw.transpose(1, 2), (max(0, K - T), 0))[..., -K:]
    return out, {"conv": conv, "ssm": s}


def _softpatch64(m, x):
    h = _rms(x, m.norm.weight, m.norm.eps)
    z = _lin(h, m.down)
    p = torch.sigmoid(_lin(h, m.score)).clamp(0.01, 0.99)  # the lexical prior is zero at this vocabulary
    s = torch.zeros_like(z[:, 0])
    states = []
    for a, d in zip((1.0 - p).unbind(1), (p * z).unbind(1)):
        s = torch.addcmul(d, a, s)
        states.append(s)
    return x + _lin(torch.cat((z, torch.stack(states, 1)), -1), m.up), s


def _model64(core, tokens, max_len=None):
    """The last position's logits and every block's state (those of the attention blocks with
    ``max_len`` only: a decode cache also holds what earlier windows left in its slots)."""
    x = core.emb.weight.double()[tokens]
    states = []
    for i, blk in enumerate(core.blocks):
        if isinstance(blk, fl.FieldBlock):
            x, st = _field64(blk, x)
        elif isinstance(blk, M.RefreshBlock):
            x, st = _refresh64(blk, x, max_len)
        else:
            x, st = _mamba64(blk, x, states=True)
        states.append(st)
        if i == core.patch_position:
            x, soft = _softpatch64(core.softpatch, x)
    h = _rms(x[:, -1], core.final_norm.weight, core.final_norm.eps)
    return {"logits": h @ core.emb.weight.double().t(), "states": states, "softpatch": soft}


def exact(case, seed):
    c = case
    if c["kind"] == "scan":
        raw, tr, ti, gamma, state, weight, grad = _scan_inputs(c, seed)
        leaves = [t.double() for t in (raw, tr, ti, gamma)]
        if c["op"] == "train":
            leaves = [t.requires_grad_() for t in leaves]
            read, _ = _recurrence(*leaves)
            return {"read": read.detach(), "grads": list(torch.autograd.grad(read, leaves, grad.double()))}
        with torch.no_grad():
            read, last = _recurrence(*leaves, None if state is None else state.double())
            out = _rms(read, weight, 1e-6) if c["op"] == "norm" else read
        return [out, last] if c["state"] else [out]
    m = _module(c, seed)
    if c["kind"] == "block" and c["op"] == "train":
        x = _hidden(c, seed, torch.float32).double().requires_grad_()
        grad = torch.randn(c["B"], c["T"], c["dim"], device="cuda", generator=_gen(seed + 4)).double()
        m = m.double()
        y, _ = _field64(m, x)
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, [x, *m.parameters()], grad))}
    with torch.no_grad():
        if c["kind"] == "model":
            if c["B"] * c["T"] > 16_384:  # too long in float64; the smaller draws hold the path to it
                return None
            return _model64(m, _tokens(c, seed), _max_len(c) if c["op"] == "prefill" else None)
        if c["kind"] == "block" and c["op"] == "step":
            g = _gen(seed + 2)
            x = torch.randn(c["B"], c["dim"], device="cuda", generator=g).to(torch.bfloat16).double()
            state = 0.5 * torch.randn(c["B"], c["dim"], device="cuda", generator=g)
            y, last = _field64(m, x[:, None], state.double())
            return {"y": y[:, 0], "state": last}
        x = _hidden(c, seed, torch.bfloat16).double()
        if c["kind"] == "block":
            y, last = _field64(m, x)
            return {"y": y, "state": last}
        if c["kind"] == "refresh":
            y, st = _refresh64(m, x, c["T"] + 256)
            return {"y": y, **st}
        if c["kind"] == "mamba":
            y, st = _mamba64(m, x, states=True)
            return {"y": y, **st}
        y, last = _softpatch64(m, x)
        return {"y": y, "last": last}
