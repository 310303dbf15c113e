"""GPU: the Mamba-2 mixer's kernels against its stock ops (which run whenever a gradient is needed)
and the defining recurrence in float64, at the edges of the 64-token chunks and of both block splits.

Tolerances: fp32 states against float64 at 2e-6 norm-wise (64-term fp32 sums), outputs at 1e-5 (their
128-term dot products C B may cancel to a tenth of their terms: 128^0.5 2^-24 over that); bf16 against the stock ops at 1e-2 (both round the projection
to bf16 and the output once).
"""
from __future__ import annotations

import copy

import pytest
import torch
import torch.nn.functional as F

import oracle
from fields_lm_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    return torch.device("cuda:0")


def _mixer(dev, dim, seed=0):
    torch.manual_seed(seed)
    m = M.Mamba2Mixer(dim).to(dev)
    with torch.no_grad():
        m.norm.weight.add_(0.1 * torch.randn_like(m.norm.weight))
        m.D.add_(torch.randn_like(m.D))
        m.A_log[0] = 4.0       # decays of e^-5 a step: exponents far below the chunk's end
        m.dt_bias[1] = 25.0    # softplus above its threshold, with a slow decay
        m.A_log[1] = -6.0
    return m.eval()


def _f64(m, u):
    """The mixer in float64: projections, convolution, recurrence, gated norm."""
    m = copy.deepcopy(m).double()
    u = u.double()
    z, xbc, dt = m._split(m.in_proj(u))
    l = u.shape[1]
    conv = F.pad(xbc.transpose(1, 2)[..., -4:], (max(0, 4 - l), 0))
    pad = F.pad(xbc, (0, 0, 3, 0))
    w = m.conv1d.weight[:, 0]
    act = F.silu(m.conv1d.bias + sum(pad[:, k:k + l] * w[:, k] for k in range(4)))
    x, bm, cm = act.split((m.d_inner, m.d_state, m.d_state), -1)
    dt = F.softplus(dt + m.dt_bias)
    xh = x.reshape(*x.shape[:2], m.nheads, m.headdim)
    s = torch.zeros(u.shape[0], m.nheads, m.headdim, m.d_state, dtype=torch.float64, device=u.device)
    ys = []
    for t in range(l):
        s = s * torch.exp(-dt[:, t] * m.A_log.exp())[..., None, None] \
            + (xh[:, t] * dt[:, t, :, None])[..., None] * bm[:, t, None, None]
        ys.append((s * cm[:, t, None, None]).sum(-1) + m.D[:, None] * xh[:, t])
    y = torch.stack(ys, 1).reshape(*x.shape) * F.silu(z)
    y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + m.norm.eps) * m.norm.weight
    return m.out_proj(y), conv, s


@pytest.mark.parametrize("dim,B,L", [(64, 2, 1), (128, 1, 3), (512, 1, 64), (512, 2, 65), (128, 3, 63), (512, 9, 129),
                                     (1024, 4, 200), (192, 2, 128), (1024, 2, 70), (512, 5, 66)])
def test_mamba_prefill_fp32(dev, dim, B, L):
    print(f"[case] mamba prefill fp32 dim={dim} B={B} L={L}", flush=True)
    m = _mixer(dev, dim, seed=L)
    u = torch.randn(B, L, dim, device=dev, generator=torch.Generator(device=dev).manual_seed(dim + L))
    with torch.no_grad():
        y, st = m(u, return_state=True)
        only = m(u)
        exp, conv, ssm = _f64(m, u)
    assert torch.equal(only, y)
    stock, st_s = m(u, return_state=True)  # gradients enabled: the stock ops
    assert stock.requires_grad
    for name, got, want, other in (("y", y, exp, stock), ("conv", st["conv"], conv, st_s["conv"]),
                                   ("ssm", st["ssm"], ssm, st_s["ssm"])):
        e, e_stock = oracle.rel_err(got.cpu(), want.cpu()), oracle.rel_err(other.detach().cpu(), want.cpu())
        print(f"[case] {name}: {e:.2e} against float64, the stock ops {e_stock:.2e}", flush=True)
        assert e <= (1e-5 if name == "y" else 2e-6), name


@pytest.mark.parametrize("dim,B,L", [(512, 1, 70), (1024, 4, 130), (1024, 1, 257)])
def test_mamba_prefill_and_steps_bf16(dev, dim, B, L):
    """bf16 weights: the sequence kernel against the stock ops, and single tokens from its state
    against the sequence."""
    print(f"[case] mamba bf16 dim={dim} B={B} L={L}", flush=True)
    m = M.cast_for_inference(_mixer(dev, dim, seed=L))
    u = torch.randn(B, L + 6, dim, device=dev, generator=torch.Generator(device=dev).manual_seed(L)).to(torch.bfloat16)
    stock = m(u).detach()
    with torch.no_grad():
        full = m(u)
        y, st = m(u[:, :L], return_state=True)
        steps = torch.stack([m.step(u[:, L + i], st) for i in range(6)], 1)
    assert torch.equal(y, full[:, :L])
    assert oracle.rel_err(full.float().cpu(), stock.float().cpu()) <= 1e-2
    assert oracle.rel_err(steps.float().cpu(), full[:, L:].float().cpu()) <= 1e-2


@pytest.mark.parametrize("B", [1, 3, 64])
def test_mamba_step_fp32(dev, B):
    print(f"[case] mamba step fp32 B={B}", flush=True)
    m = _mixer(dev, 512, seed=B)
    g = torch.Generator(device=dev).manual_seed(B)
    st = {"conv": torch.randn(B, m.conv_dim, 4, device=dev, generator=g),
          "ssm": torch.randn(B, m.nheads, 64, 128, device=dev, generator=g)}
    st2 = {k: v.clone() for k, v in st.items()}
    u = torch.randn(B, 512, device=dev, generator=g)
    with torch.no_grad():
        y = m.step(u, st)
        st2["ssm"] = st2["ssm"].transpose(2, 3).contiguous().transpose(2, 3)  # not contiguous: the stock ops
        exp = m.step(u, st2)
    assert oracle.rel_err(y.cpu(), exp.cpu()) <= 1e-5
    assert torch.equal(st["conv"], st2["conv"])
    assert oracle.rel_err(st["ssm"].cpu(), st2["ssm"].cpu()) <= 1e-6


def test_mamba_other_geometries_and_modes_keep_the_stock_ops(dev):
    """A geometry the kernels do not have, forward-mode derivatives and vmap run as before."""
    print("[case] mamba stock routes", flush=True)
    torch.manual_seed(1)
    small = M.Mamba2Mixer(32, d_state=8, headdim=16, chunk_size=8).to(dev)
    u = torch.randn(2, 19, 32, device=dev)
    with torch.no_grad():
        assert oracle.rel_err(small(u).cpu(), small(u.double().float()).cpu()) == 0.0
    m = _mixer(dev, 64)
    x = torch.randn(1, 9, 64, device=dev)
    with torch.no_grad():
        y, tangent = torch.func.jvp(m, (x,), (torch.ones_like(x),))
        eps = 1e-2
        slope = (_f64(m, x + eps)[0] - _f64(m, x - eps)[0]) / (2 * eps)
        batched = torch.func.vmap(m)(torch.stack([x, 2 * x]))
        both = torch.stack([m(x), m(2 * x)])
    assert oracle.rel_err(tangent.cpu(), slope.cpu()) <= 1e-2
    assert oracle.rel_err(batched.cpu(), both.cpu()) <= 1e-5


@pytest.mark.parametrize("dim,B,L,weights", [(128, 2, 70, "bf16"), (512, 1, 300, "bf16"), (128, 1, 3, "fp32"), (1024, 2, 257, "fp32")])
def test_mamba_under_autocast_gives_the_stock_bits(dev, dim, B, L, weights):
    """Under autocast the convolution, the decayed products and the state update run in kernels that keep
    every bit of the stock ops (which run whenever a gradient is needed, and in a subclass's step)."""
    print(f"[case] mamba autocast bits dim={dim} B={B} L={L} {weights}", flush=True)
    m = _mixer(dev, dim, seed=L)
    if weights == "bf16":
        m = M.cast_for_inference(m)
    u = torch.randn(B, L + 3, dim, device=dev, generator=torch.Generator(device=dev).manual_seed(L))
    u = u.to(torch.bfloat16) if weights == "bf16" else u
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock, st_stock = m(u[:, :L], return_state=True)
        with torch.no_grad():
            y, st = m(u[:, :L], return_state=True)
            assert torch.equal(y, stock.detach())
            for k in st:
                assert torch.equal(st[k], st_stock[k].detach()), k
            other = {"conv": st["conv"].clone(), "ssm": st["ssm"].transpose(2, 3).contiguous().transpose(2, 3)}
            for i in range(3):  # a transposed state takes the stock ops
                a, b = m.step(u[:, L + i], st), m.step(u[:, L + i], other)
                assert torch.equal(a, b) and torch.equal(st["ssm"], other["ssm"]) and torch.equal(st["conv"], other["conv"])


@pytest.mark.parametrize("headdim,chunk,B,L", [(24, 24, 2, 50), (32, 72, 1, 72), (96, 136, 2, 300), (6, 16, 1, 33),
                                               (48, 20, 1, 45)])
def test_mamba_under_autocast_odd_geometry_gives_the_stock_bits(dev, headdim, chunk, B, L):
    """Tiles of the products' operands with remainders in tokens and dimensions, and what they do not take."""
    print(f"[case] mamba operands headdim={headdim} chunk={chunk} B={B} L={L}", flush=True)
    torch.manual_seed(L)
    m = M.Mamba2Mixer(headdim * 2, d_state=16, d_conv=4, expand=2, headdim=headdim, ngroups=1, chunk_size=chunk).to(dev)
    u = torch.randn(B, L, headdim * 2, device=dev, generator=torch.Generator(device=dev).manual_seed(L))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        stock, st_stock = m(u, return_state=True)
        with torch.no_grad():
            y, st = m(u, return_state=True)
    assert torch.equal(y, stock.detach())
    for k in st:
        assert torch.equal(st[k], st_stock[k].detach()), k
