"""GPU: the refresh block's attention kernels at the edges of their query tiles, key steps, windows and
landmark chunks, against the stock ops in fp32 on the same bf16 weights.

Tolerances: no more than the stock bf16 ops are off (they round their scores too), and 2e-2 norm-wise:
the weights are scaled so that scores reach 5 to 6, q and k carry 2^-9 each into them, so the
probabilities move by up to 6 * 2^-8. States 1e-2.
"""
from __future__ import annotations

import copy

import pytest
import torch

from fields_lm_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    return torch.device("cuda:0")


def _norm(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


def _block(dev, heads, kv, window, chunk, latent=64, seed=0):
    torch.manual_seed(seed)
    blk = M.RefreshBlock(64 * heads, heads, kv, latent, window, chunk, 96).to(dev)
    with torch.no_grad():
        blk.residual_gate.weight.normal_(0, 0.05)
        blk.attn.global_mix_logit.fill_(0.7)
        blk.attn.q_latent_proj.weight.mul_(3.0)  # scores that spread the softmax
        blk.attn.kv_up.weight.mul_(3.0)
        blk.norm2.weight.add_(0.1 * torch.randn_like(blk.norm2.weight))
    return M.cast_for_inference(blk).eval()


CASES = [(16, 4, 256, 256, 1, 1), (16, 4, 256, 256, 2, 31), (8, 2, 64, 32, 1, 33), (8, 2, 64, 32, 2, 64), (8, 2, 64, 32, 3, 321),
         (4, 4, 128, 64, 2, 200), (4, 2, 192, 96, 1, 400), (8, 1, 64, 64, 1, 150), (16, 4, 512, 256, 1, 1300),
         (12, 3, 256, 32, 1, 2100), (16, 4, 1024, 256, 1, 1025)]


@pytest.mark.parametrize("heads,kv,window,chunk,B,T", CASES)
def test_attention_against_fp32(dev, heads, kv, window, chunk, B, T):
    print(f"[case] refresh attention heads={heads}/{kv} window={window} chunk={chunk} B={B} T={T}", flush=True)
    att = _block(dev, heads, kv, window, chunk, seed=T).attn
    ref = copy.deepcopy(att).float()
    x = torch.randn(B, T, 64 * heads, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    stock = att(x).detach()  # gradients enabled: the stock ops
    with torch.no_grad():
        y = att(x)
        exp, st_exp = ref.prefill(x.float(), T + 70)
        used = [torch.full(t.shape, float("nan"), device=dev, dtype=x.dtype) for t in st_exp.values()]
        del used  # what an unwritten slot would hold
        yp, st = att.prefill(x, T + 70)
    assert torch.equal(y, yp)
    e, e_stock = _norm(y, exp), _norm(stock, exp)
    print(f"[case] native {e:.2e} stock {e_stock:.2e}", flush=True)
    assert e <= 2e-2 and e <= e_stock + 1e-4
    assert set(st) == set(st_exp)
    for name in st:
        assert st[name].shape == st_exp[name].shape and st[name].dtype == (torch.float32 if name == "lat_sum" else x.dtype)
        assert _norm(st[name], st_exp[name]) <= 1e-2, name
    n, full = T % window, T // chunk  # slots in use: the open window's tokens; landmarks after the null slot
    for name, unused in (("kt", st["kt"][..., n:]), ("v", st["v"][:, :, n:]), ("null key", st["lkt"][..., :1]),
                         ("null value", st["lv"][:, :, :1]), ("lkt", st["lkt"][..., 1 + full:]),
                         ("lv", st["lv"][:, :, 1 + full:])):
        assert not unused.any(), name


@pytest.mark.parametrize("T", [40, 63, 130])
def test_block_forward_prefill_and_steps_agree(dev, T):
    print(f"[case] refresh block T={T}", flush=True)
    blk = _block(dev, 8, 2, 64, 32, seed=T)
    ref = copy.deepcopy(blk).float()
    x = torch.randn(2, T + 40, 512, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    keep = x.clone()
    with torch.no_grad():
        full = blk(x)
        y, st = blk.prefill(x[:, :T], T + 41)
        steps = torch.stack([blk.step(x[:, T + i], torch.tensor(T + i, device=dev), st) for i in range(40)], 1)
        exp = ref(x.float())
    assert torch.equal(x, keep)  # the residual product accumulates onto its own buffer
    assert _norm(full, exp) <= 2e-2
    assert _norm(y, exp[:, :T]) <= 2e-2
    assert _norm(steps, exp[:, T:]) <= 2e-2


@pytest.mark.parametrize("rows,dim", [(1, 8), (5, 1024), (4097, 520), (3, 2056), (2, 4096)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32], ids=["w16", "w32"])
def test_rms_norm_edges(dev, rows, dim, wdtype):
    print(f"[case] rms_norm {rows}x{dim} {wdtype}", flush=True)
    n = M.NativeRMSNorm(dim).to(dev)
    g = torch.Generator(device=dev).manual_seed(dim)
    n.weight.data = (1 + 0.2 * torch.randn(dim, device=dev, generator=g)).to(wdtype)
    x = (3 * torch.randn(rows, dim, device=dev, generator=g)).to(torch.bfloat16)
    with torch.no_grad():
        y = n(x)
        shifted = n(torch.cat((x.new_zeros(1), x.view(-1)))[1:].view(rows, dim))  # not 16-byte aligned
    xf = x.double()
    exp = xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + n.eps) * n.weight.double()
    assert torch.equal(y, shifted)
    assert bool(((y.double() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-6).all())  # one rounding: half a step


@pytest.mark.parametrize("dim,rank,B,T", [(64, 64, 1, 1), (128, 64, 2, 15), (512, 64, 3, 16), (128, 8, 2, 17), (1024, 64, 4, 1030),
                                          (128, 100, 1, 300), (2056, 64, 2, 130), (512, 64, 1, 4099)])
def test_softpatch_against_fp32(dev, dim, rank, B, T):
    print(f"[case] softpatch dim={dim} rank={rank} B={B} T={T}", flush=True)
    torch.manual_seed(T)
    sp = M.BoundaryStateMixer(dim, rank, vocab=50).to(dev)
    with torch.no_grad():
        sp.up.weight.normal_(0, 0.1)
        sp.score.weight.normal_(0, 0.2)
        sp.norm.weight.add_(0.1 * torch.randn_like(sp.norm.weight))
        sp._boundary_lut.copy_(torch.randn(50, device=dev))
    M.cast_for_inference(sp)
    ref = copy.deepcopy(sp).float()
    g = torch.Generator(device=dev).manual_seed(T)
    x = torch.randn(B, T, dim, device=dev, generator=g).to(torch.bfloat16)
    tok = torch.randint(0, 50, (B, T), device=dev, generator=g)
    keep = x.clone()
    with torch.no_grad():
        y, last = sp(x, tok, return_state=True)
        assert torch.equal(sp(x, tok), y)
        exp, last_exp = ref(x.float(), tok, return_state=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            stock = sp(x, tok)
    assert torch.equal(x, keep) and last.dtype == torch.float32
    e, e_stock = _norm(y, exp), _norm(stock, exp)
    print(f"[case] softpatch native {e:.2e} stock {e_stock:.2e}", flush=True)
    assert e <= 1.1 * e_stock + 1e-4 and e <= 1e-2
    assert _norm(last, last_exp) <= 2e-2  # z rounded to bf16, boundaries from a bf16 score


class _Stock(M.LandmarkAttention):
    """The same attention through the stock ops (the kernels take the class itself only)."""


@pytest.mark.parametrize("heads,kv,window,chunk,B,prompt", [(16, 4, 256, 256, 5, 250), (8, 2, 64, 32, 1, 60), (8, 8, 100, 16, 3, 95),
                                                            (4, 1, 33, 4, 2, 30)])
@pytest.mark.parametrize("autocast", [False, True], ids=["plain", "autocast"])
def test_attention_step_gives_the_stock_bits(dev, heads, kv, window, chunk, B, prompt, autocast):
    """Tokens across the end of a window and of a chunk, to the last position the state is sized for:
    outputs and every state equal the stock ops' bit for bit."""
    print(f"[case] refresh step bits heads={heads}/{kv} window={window} chunk={chunk} B={B}", flush=True)
    att = _block(dev, heads, kv, window, chunk, seed=window).attn
    stock = copy.deepcopy(att)
    stock.__class__ = _Stock
    n = 12
    x = torch.randn(B, prompt + n, 64 * heads, device=dev, generator=torch.Generator(device=dev).manual_seed(B)).to(torch.bfloat16)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        _, st = stock.prefill(x[:, :prompt], prompt + n)
        att._rope_len = stock._rope_len
        mine = {k: v.clone() for k, v in st.items()}
        for i in range(n):
            pos = torch.tensor(prompt + i, device=dev)
            assert att._native_step(att.q_latent_proj(x[:, prompt + i]), pos, mine)
            a, b = att.step(x[:, prompt + i], pos, mine), stock.step(x[:, prompt + i], pos, st)
            assert torch.equal(a, b), i
            for k in st:
                assert torch.equal(mine[k], st[k]), (i, k)


@pytest.mark.parametrize("B,T,window", [(2, 300, 64), (1, 77, 128), (3, 130, 256)])
def test_causal_scores_under_autocast_give_the_stock_bits(dev, B, T, window):
    """Prompts under autocast: the scaled, masked scores in one pass leave every bit as it was."""
    print(f"[case] masked scores B={B} T={T} window={window}", flush=True)
    att = _block(dev, 8, 2, window, 32, seed=T).attn
    x = torch.randn(B, T, 512, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock = att(x).detach()  # gradients enabled: the stock ops
        with torch.no_grad():
            assert torch.equal(att(x), stock)


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("lk", [1, 5, 16, 17, 32, 33, 63, 64, 65, 127, 128, 200, 257, 512, 777, 1023, 1024, 1025])
def test_masked_softmax_gives_the_stock_bits(dev, lk, mode):
    """Every unroll of the row at its edges, spread scores, equal scores, a row of -inf and one infinity."""
    if mode == 3 and lk > 1024:
        pytest.skip("longer landmark rows take the stock ops")
    print(f"[case] masked softmax lk={lk} mode={mode}", flush=True)
    lq = lk if mode == 0 else 7
    rows, period = 6 * lq, max(1, (lk + 1) // 2) if mode else 0
    g = torch.Generator(device=dev).manual_seed(lk)
    raw = (torch.randn(rows, lk, device=dev, generator=g) * 40).to(torch.bfloat16)
    raw[0] = 3.0
    raw[1] = raw[1] * 1e4
    raw[2] = float("-inf")
    raw[3, -1] = float("inf")
    pos = torch.tensor(period + lk // 3, device=dev, dtype=torch.int64)
    row = torch.arange(rows, device=dev) % lq
    limit = {0: row, 1: (pos % max(period, 1)).expand(rows), 2: (pos // max(period, 1)).expand(rows),
             3: row // max(period, 1)}[mode]
    scores = (raw.float() * 64 ** -0.5).masked_fill(torch.arange(lk, device=dev)[None] > limit[:, None], float("-inf"))
    stock = torch.softmax(scores, -1).to(torch.bfloat16)
    got = M.masked_softmax(raw, lq, mode, pos if mode in (1, 2) else None, period, 64)
    assert torch.equal(got.isnan(), stock.isnan())
    assert torch.equal(got.nan_to_num(7.0), stock.nan_to_num(7.0))


@pytest.mark.parametrize("T,window", [(1300, 512), (1100, 1024), (40, 64)])
def test_landmark_scores_under_autocast_give_the_stock_bits(dev, T, window):
    print(f"[case] landmark scores T={T} window={window}", flush=True)
    att = _block(dev, 8, 2, window, 32, seed=T).attn
    x = torch.randn(2, T, 512, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock = att(x).detach()  # gradients enabled: the stock ops
        with torch.no_grad():
            assert torch.equal(att(x), stock)


@pytest.mark.parametrize("heads,kv,B,T,window", [(8, 2, 2, 20, 64), (4, 4, 3, 130, 64), (6, 3, 1, 77, 20),
                                                 (8, 2, 2, 128, 64), (16, 4, 1, 1111, 512)])
def test_prompt_state_under_autocast_gives_the_stock_bits(dev, heads, kv, B, T, window):
    """Rotated, padded and transposed heads, no landmark yet, odd windows: output and decode state."""
    print(f"[case] prompt heads={heads}/{kv} B={B} T={T} window={window}", flush=True)
    att = _block(dev, heads, kv, window, 32, seed=T).attn
    x = torch.randn(B, T, 64 * heads, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock, st_stock = att.prefill(x, T + 9)  # gradients enabled: the stock ops
        with torch.no_grad():
            y, st = att.prefill(x, T + 9)
    assert torch.equal(y, stock)
    for k in st:
        assert torch.equal(st[k], st_stock[k]), k


@pytest.mark.parametrize("heads,ff,B,T", [(8, 96, 2, 70), (4, 44, 1, 33), (1, 8, 3, 1)])
def test_block_under_autocast_gives_the_stock_bits(dev, heads, ff, B, T):
    """The gated residual and the feed-forward's activation, rows that take 16 bytes and rows that do not."""
    print(f"[case] refresh block heads={heads} ff={ff} B={B} T={T}", flush=True)
    torch.manual_seed(T)
    blk = M.RefreshBlock(64 * heads, heads, 1, 64, 64, 32, ff).to(dev)
    with torch.no_grad():
        blk.residual_gate.weight.normal_(0, 2.0)  # sigmoids over their whole range
        blk.ff.gate_up.weight.mul_(20.0)
    blk = M.cast_for_inference(blk).eval()
    x = torch.randn(B, T, 64 * heads, device=dev, generator=torch.Generator(device=dev).manual_seed(T)).to(torch.bfloat16)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock, st_stock = blk.prefill(x, T + 9)  # gradients enabled: the stock ops
        step_stock = blk.step(x[:, 0], torch.tensor(T, device=dev), {k: v.detach().clone() for k, v in st_stock.items()})
        with torch.no_grad():
            y, st = blk.prefill(x, T + 9)
            step = blk.step(x[:, 0], torch.tensor(T, device=dev), st)
    assert torch.equal(y, stock) and torch.equal(step, step_stock)
