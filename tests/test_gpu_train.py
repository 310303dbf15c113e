"""GPU: the Field block's training kernels against the stock ops, in fp32 (where both are fp32 sums
of the same terms: 1e-5 norm-wise, 1e-4 for parameter gradients, which add over all tokens with
cancellation) and under bf16 autocast (no further from the fp32 gradients than the stock ops, 10 % for
their different roundings).
"""
from __future__ import annotations

import copy

import pytest
import torch

from fields_lm_amd import FieldBlock
from fields_lm_amd import model as M

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    return torch.device("cuda:0")


def _norm(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


def _block(dev, dim, hidden, seed=0):
    torch.manual_seed(seed)
    b = FieldBlock(dim, "triton", 32, 32, 64, hidden).to(dev)
    with torch.no_grad():
        for n in (b.mixer.read_norm, b.ff_norm):
            n.weight.add_(0.2 * torch.randn_like(n.weight))
        b.mixer.radius_logit[0] = -3.0   # below the lower clamp: no gradient
        b.mixer.radius_logit[-1] = 12.0  # above the upper one
    return b


def _grads(b, x, gy, native, autocast=False):
    b.fuse_tail = native
    x = x.clone().requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        assert bool(b._native_training(x)) == native
        y = b(x)
    names = ["x"] + [n for n, p in b.named_parameters() if p.requires_grad]
    params = [p for p in b.parameters() if p.requires_grad]
    return y.detach(), dict(zip(names, torch.autograd.grad(y, [x, *params], gy)))


@pytest.mark.parametrize("dim,hidden,B,T", [(1024, 2528, 2, 70), (16, 24, 1, 1), (136, 352, 3, 33), (1112, 2976, 1, 65),
                                            (2048, 96, 1, 40), (64, 40, 2, 1100), (256, 20, 1, 9)])
def test_training_kernels_fp32(dev, dim, hidden, B, T):
    print(f"[case] block training fp32 dim={dim} hidden={hidden} B={B} T={T}", flush=True)
    b = _block(dev, dim, hidden, seed=dim)
    if dim == 136:
        b.ff = M.GateUpSwiGLU(dim, hidden).to(dev)
        b.mixer.out_proj.weight.requires_grad_(False)
        b.ff_norm.weight.requires_grad_(False)
    g = torch.Generator(device=dev).manual_seed(T)
    x, gy = (torch.randn(B, T, dim, device=dev, generator=g) for _ in range(2))
    y, got = _grads(b, x, gy, True)
    ys, exp = _grads(b, x, gy, False)
    assert _norm(y, ys) <= 1e-5
    for n in exp:
        assert got[n].dtype == exp[n].dtype and got[n].shape == exp[n].shape
        assert _norm(got[n], exp[n]) <= (1e-5 if n == "x" else 1e-4), n
    assert float(got["mixer.radius_logit"][0]) == 0.0 == float(got["mixer.radius_logit"][-1])


@pytest.mark.parametrize("dim,hidden,B,T", [(1024, 2528, 2, 130), (136, 352, 2, 65)])
def test_training_kernels_autocast(dev, dim, hidden, B, T):
    print(f"[case] block training autocast dim={dim}", flush=True)
    b = _block(dev, dim, hidden, seed=dim)
    g = torch.Generator(device=dev).manual_seed(T)
    x, gy = (torch.randn(B, T, dim, device=dev, generator=g) for _ in range(2))
    y32, ref = _grads(b, x, gy, False)
    y, got = _grads(b, x, gy, True, autocast=True)
    ys, stock = _grads(b, x, gy, False, autocast=True)
    assert y.dtype == ys.dtype and _norm(y, y32) <= 1.1 * _norm(ys, y32) + 1e-5
    for n in ref:
        e, e_stock = _norm(got[n], ref[n]), _norm(stock[n], ref[n])
        assert got[n].dtype == stock[n].dtype
        assert e <= 1.1 * e_stock + 1e-4, (n, e, e_stock)


def test_training_partial_gradients_and_misaligned_input(dev):
    """Only some inputs need gradients; an input that is not 16-byte aligned is copied, not read past."""
    print("[case] block training, partial gradients", flush=True)
    b = _block(dev, 64, 40)
    for p in b.parameters():
        p.requires_grad_(False)
    x = torch.randn(2, 9, 64, device=dev)
    gy = torch.randn(2, 9, 64, device=dev)
    y, got = _grads(b, x, gy, True)
    ys, exp = _grads(b, x, gy, False)
    assert list(got) == ["x"] and _norm(got["x"], exp["x"]) <= 1e-5
    shifted = torch.empty(x.numel() + 1, device=dev)[1:].view_as(x).copy_(x).requires_grad_()
    b.fuse_tail = True
    assert _norm(torch.autograd.grad(b(shifted), shifted, gy)[0], exp["x"]) <= 1e-5
    b.ff_norm.weight.requires_grad_(True)
    b.fuse_tail = True
    native = torch.autograd.grad(b(x), b.ff_norm.weight, gy)[0]
    assert torch.equal(native, torch.autograd.grad(b(x), b.ff_norm.weight, gy)[0])
    b.fuse_tail = False
    assert _norm(native, torch.autograd.grad(b(x), b.ff_norm.weight, gy)[0]) <= 1e-4


def test_training_double_backward_matches_stock(dev):
    """create_graph: the elementwise parts differentiate a second time as the stock ops do (the scan's
    backward is not differentiable on either route)."""
    print("[case] block training, double backward", flush=True)
    b = _block(dev, 32, 24)
    x = torch.randn(2, 7, 32, device=dev)
    out = []
    for native in (True, False):
        b.fuse_tail = native
        xi = x.clone().requires_grad_()
        g, = torch.autograd.grad(b(xi).square().sum(), xi, create_graph=True)
        out.append(torch.autograd.grad(g.square().sum(), [xi, b.ff_norm.weight, b.ff.w12.weight, b.mixer.read_norm.weight,
                                                           b.mixer.gate_proj.weight]))
    for a, e in zip(*out):
        assert _norm(a, e) <= 1e-4


@pytest.mark.parametrize("wanted", [("ff_norm.weight",), ("mixer.theta", "ff_norm.weight")])
def test_training_double_backward_with_frozen_parameters(dev, wanted):
    print(f"[case] block training, double backward, only {wanted}", flush=True)
    b = _block(dev, 32, 24)
    for n, p in b.named_parameters():
        p.requires_grad_(n in wanted)
    params = [dict(b.named_parameters())[n] for n in wanted]
    x = torch.randn(2, 7, 32, device=dev)
    out = []
    for native in (True, False):
        b.fuse_tail = native
        grads = torch.autograd.grad(b(x).square().sum(), params, create_graph=True)
        out.append(torch.autograd.grad(sum(g.square().sum() for g in grads), params[-1:]))
    for a, e in zip(*out):
        assert _norm(a, e) <= 1e-4


def test_training_replaced_parts_keep_the_stock_ops(dev):
    print("[case] block training, replaced parts", flush=True)
    b = _block(dev, 64, 40)
    x = torch.randn(1, 5, 64, device=dev, requires_grad=True)
    assert b._native_training(x)
    for part in (b.mixer, b.ff, b.ff_norm, b.mixer.read_norm):
        handle = part.register_forward_hook(lambda mod, args, out: None)
        assert not b._native_training(x)
        handle.remove()
    assert not b._native_training(x.double())
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
        b(x)
    assert seen


def test_training_replaced_product_sees_fp32_under_autocast(dev):
    print("[case] block training, a product that computes in fp32", flush=True)

    class Fp32Linear(torch.nn.Linear):
        def forward(self, x):
            seen.append(x.dtype)
            with torch.autocast("cuda", enabled=False):
                return super().forward(x)

    for owner, name in (("mixer", "out_proj"), ("ff", "w12")):
        b = _block(dev, 64, 40)
        layer = getattr(getattr(b, owner), name)
        layer.__class__ = Fp32Linear
        x = torch.randn(1, 5, 64, device=dev, requires_grad=True)
        seen = []
        with torch.autocast("cuda", dtype=torch.bfloat16):
            b(x).sum().backward()
        assert seen == [torch.float32] and x.grad.isfinite().all()
