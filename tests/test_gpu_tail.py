"""GPU: the Field block's elementwise kernels at the edges of their vector widths, and the transition
parameters, against the stock ops they replace.

Tolerances: a bf16 result may land one bf16 step away where an fp32 intermediate differs in its last
bit (2^-8 of its magnitude); the transition parameters are the stock ops' bits.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    return torch.device("cuda:0")


def _one_step(got, exp, scale):
    got, exp = got.float(), exp.float()
    assert bool(((got - exp).abs() <= 2.0 ** -7 * (exp.abs() + scale.float().abs()) + 1e-6).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("rows,hidden", [(1, 8), (3, 16), (257, 2528), (5, 12), (1, 1), (4100, 24)])
def test_swiglu_edges(dev, dtype, rows, hidden):
    from fields_lm_amd import swiglu

    print(f"[case] swiglu {dtype} {rows}x{hidden}", flush=True)
    g = torch.Generator().manual_seed(rows + hidden)
    gu = (torch.randn(rows, 2 * hidden, generator=g) * 4).to(dtype)
    gu.view(-1)[0] = float("-inf")           # silu(-inf) is NaN, as in the stock op
    gu.view(-1)[-1] = float("inf")
    gu = gu.to(dev)
    gate, up = gu.chunk(2, dim=-1)
    exp, got = F.silu(gate) * up, swiglu(gu)
    assert torch.equal(got.isnan(), exp.isnan())
    ok = exp.isfinite()
    assert torch.equal(got[~ok & ~exp.isnan()], exp[~ok & ~exp.isnan()])
    _one_step(got[ok], exp[ok], up[ok])
    shifted = torch.empty(gu.numel() + 1, device=dev, dtype=dtype)[1:].view_as(gu).copy_(gu)  # not 16-byte aligned
    assert torch.equal(swiglu(shifted).isnan(), exp.isnan())
    _one_step(swiglu(shifted)[ok], exp[ok], up[ok])


def _same_bits(got, exp):
    nan = exp.isnan()
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got[~nan].view(torch.int16), exp[~nan].view(torch.int16))


@pytest.mark.parametrize("cols", [256, 1], ids=["16-byte", "scalar"])
def test_activations_of_every_bf16_gate_have_the_stock_bits(dev, cols):
    """All 65,536 bf16 gates: the bits of the stock silu and sigmoid, subnormal results, zeros' signs and
    infinities included (generation under autocast runs these kernels in the stock ops' place)."""
    from fields_lm_amd import gate_residual_norm, swiglu

    print(f"[case] every bf16 gate, rows of {cols}", flush=True)
    gate = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).to(dev).view(-1, cols)
    one = torch.ones_like(gate)
    _same_bits(swiglu(torch.cat((gate, one), 1).contiguous()), F.silu(gate))
    x1, _ = gate_residual_norm(torch.zeros_like(gate), one, gate, torch.ones(cols, device=dev))
    _same_bits(x1, torch.sigmoid(gate))


@pytest.mark.parametrize("rows,dim", [(1, 8), (4097, 512), (5, 520), (4100, 1032), (2, 2048), (3, 2056), (7, 516), (6, 7)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32], ids=["w16", "w32"])
def test_gate_residual_norm_edges(dev, rows, dim, wdtype):
    from fields_lm_amd import gate_residual_norm

    print(f"[case] gate_residual_norm {rows}x{dim} {wdtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(rows * 3 + dim)
    x, out, gp = ((2 * torch.randn(rows, dim, device=dev, generator=g)).to(torch.bfloat16) for _ in range(3))
    w = (1.0 + 0.3 * torch.randn(dim, device=dev, generator=g)).to(wdtype)
    x1, h = gate_residual_norm(x, out, gp, w, 1e-6)
    exp_x = x + out * torch.sigmoid(gp)
    xf = exp_x.float()
    exp_h = (xf * torch.rsqrt(xf.square().mean(-1, keepdim=True) + 1e-6) * w.float()).to(x.dtype)
    _one_step(x1, exp_x, out)
    _one_step(h, exp_h, out.float() * (exp_h.float() / xf.abs().clamp_min(1e-3)))


@pytest.mark.parametrize("rows,dim,xt,gt", [(4034, 520, "bf16", "bf16"), (2050, 1024, "bf16", "f32"), (31776, 264, "f32", "bf16"),
                                            (16385, 40, "bf16", "bf16"), (16384, 256, "f32", "bf16"), (1021, 2056, "bf16", "bf16")])
def test_gate_residual_norm_routes_agree(dev, rows, dim, xt, gt):
    """Where the wave per row begins: the same bits as the block per row gives a part of the same rows (and
    as a misaligned copy gets), so that a row's result does not depend on its batch."""
    from fields_lm_amd import gate_residual_norm

    print(f"[case] gate_residual_norm routes {rows}x{dim} {xt}/{gt}", flush=True)
    types = {"bf16": torch.bfloat16, "f32": torch.float32}
    g = torch.Generator(device=dev).manual_seed(dim)
    x, out, gp = (2 * torch.randn(rows, dim, device=dev, generator=g) for _ in range(3))
    x, out, gp = x.to(types[xt]), out.to(types[gt]), gp.to(types[gt])
    w = 1.0 + 0.3 * torch.randn(dim, device=dev, generator=g)
    x1, h = gate_residual_norm(x, out, gp, w, 1e-6)
    for n in (1, 37):
        xp, hp = gate_residual_norm(x[-n:], out[-n:], gp[-n:], w, 1e-6)
        assert torch.equal(xp, x1[-n:]) and torch.equal(hp, h[-n:])
    shifted = torch.empty(x.numel() + 1, device=dev, dtype=x.dtype)[1:].view_as(x).copy_(x)
    xs, hs = gate_residual_norm(shifted, out, gp, w, 1e-6)
    assert torch.equal(xs, x1) and torch.equal(hs, h)


@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32], ids=["w16", "w32"])
@pytest.mark.parametrize("dim", [2, 256, 258, 1024, 2050])
def test_transition_parameters_match_stock_ops(dev, dim, wdtype):
    from fields_lm_amd import IndependentVacancyField

    print(f"[case] transition dim={dim} {wdtype}", flush=True)
    m = IndependentVacancyField(dim, "triton", 32, 32, 64).to(dev)
    g = torch.Generator(device=dev).manual_seed(dim)
    with torch.no_grad():
        m.radius_logit.add_(4 * torch.randn(dim // 2, device=dev, generator=g))
        m.radius_logit[0] = float("-inf")     # the clamp's lower end
        m.radius_logit[-1] = float("inf") if dim > 2 else 0.3  # its upper end
        m.read_norm.weight.add_(torch.randn(2 * dim, device=dev, generator=g))
    m.read_norm.weight.data = m.read_norm.weight.data.to(wdtype)
    exp = m.transition()                      # gradients enabled: the stock ops
    with torch.no_grad():
        got = m.decode_params()
    for a, b in zip(got, (*exp, m.read_norm.weight.float())):
        assert a.dtype == torch.float32 and a.is_contiguous()
        assert torch.equal(a, b.detach())


def test_block_residual_gemm_keeps_wrapped_layers(dev):
    """The FFN's output GEMM accumulates onto the residual only for a plain layer: a hook on it
    still fires and its change reaches the output."""
    from fields_lm_amd import FieldBlock

    print("[case] hooked FFN output layer", flush=True)
    torch.manual_seed(3)
    block = FieldBlock(128, "triton", 32, 32, 64, 256).to(dev).to(torch.bfloat16)
    block.mixer.radius_logit.data = block.mixer.radius_logit.data.float()
    block.mixer.theta.data = block.mixer.theta.data.float()
    x = torch.randn(2, 33, 128, device=dev).to(torch.bfloat16)
    with torch.no_grad():
        plain = block(x)
        handle = block.ff.w3.register_forward_hook(lambda mod, args, out: out * 0)
        off = block(x)
        handle.remove()
        block.ff.w3.weight.zero_()
        zero = block(x)
    assert torch.equal(off, zero)
    assert not torch.equal(off, plain)
