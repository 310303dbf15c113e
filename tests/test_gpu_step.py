"""GPU: a Field block's one-token kernels (few-row products with their epilogues) at the edges of their
row tiles, column tiles and depth splits, against the separate ops and the same block in fp32.

Tolerance: against fp32 on the same bf16 weights, no further off than the separate bf16 ops (10 %
for their different roundings) and 1e-2 norm-wise.
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


def _block(dev, dim, hidden, seed):
    torch.manual_seed(seed)
    b = FieldBlock(dim, "triton", 32, 32, 64, hidden).to(dev)
    with torch.no_grad():
        for n in (b.mixer.read_norm, b.ff_norm):
            n.weight.add_(0.2 * torch.randn_like(n.weight))
    return M.cast_for_inference(b).eval()


@pytest.mark.parametrize("dim,hidden,B", [(1024, 2528, 64), (1024, 2528, 1), (1024, 2784, 128), (136, 352, 16), (136, 352, 17),
                                          (1112, 2976, 33), (1280, 3424, 65), (2056, 96, 33), (1288, 96, 32), (256, 96, 65), (64, 8, 31), (16, 24, 2), (520, 264, 48)])
def test_block_step_kernels(dev, dim, hidden, B):
    print(f"[case] block step dim={dim} hidden={hidden} B={B}", flush=True)
    b = _block(dev, dim, hidden, seed=dim + B)
    if dim == 520:
        b.ff = M.cast_for_inference(M.GateUpSwiGLU(dim, hidden).to(dev))
        b.ff_norm.weight.data = b.ff_norm.weight.data.float()
    ref = copy.deepcopy(b).float()
    g = torch.Generator(device=dev).manual_seed(B)
    xs = torch.randn(3, B, dim, device=dev, generator=g).to(torch.bfloat16)
    s0 = torch.randn(B, dim, device=dev, generator=g)
    with torch.no_grad():
        params, rparams = b.mixer.decode_params(), ref.mixer.decode_params()
        assert b._native_step(xs[0], s0, params) is not None
        st, st_stock, st_ref = s0.clone(), s0.clone(), s0.clone()
        y = torch.stack([b.step(x, st, params) for x in xs])
        b.mixer.fuse_in_proj = False  # the separate ops
        stock = torch.stack([b.step(x, st_stock, params) for x in xs])
        exp = torch.stack([ref.step(x.float(), st_ref, rparams) for x in xs])
    e, e_stock = _norm(y, exp), _norm(stock, exp)
    print(f"[case] native {e:.2e} separate {e_stock:.2e}", flush=True)
    assert y.shape == (3, B, dim) and y.dtype == torch.bfloat16
    assert e <= 1.1 * e_stock + 1e-4 and e <= 1e-2
    assert _norm(st, st_ref) <= 1.1 * _norm(st_stock, st_ref) + 1e-4


def test_block_step_in_hip_graph_and_replaced_parts(dev):
    """The same bits from a graph's replays, and the separate ops whenever a part is replaced."""
    print("[case] block step graph, replaced parts", flush=True)
    b = _block(dev, 256, 96, seed=5)
    g = torch.Generator(device=dev).manual_seed(1)
    xs = torch.randn(4, 8, 256, device=dev, generator=g).to(torch.bfloat16)
    with torch.no_grad():
        params = b.mixer.decode_params()
        st, st2, x = torch.zeros(8, 256, device=dev), torch.zeros(8, 256, device=dev), xs[0].clone()
        eager = [b.step(v, st, params).clone() for v in xs]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            b.step(x, st2, params)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = b.step(x, st2, params)
        st2.zero_()
        for i in range(4):
            x.copy_(xs[i])
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager[i]), i
        calls = []
        for part in (b.mixer.out_proj, b.ff.w3, b.mixer.read_norm):
            handle = part.register_forward_pre_hook(lambda mod, args: calls.append(mod))
            assert b._native_step(x, st2, params) is None
            handle.remove()
        b.mixer.normed_step = b.mixer.normed_step
        assert b._native_step(x, st2, params) is None
        del b.mixer.normed_step
        assert b._native_step(x, st2, params) is not None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert b._native_step(x, st2, params) is None
    assert b._native_step(x, st2, params) is None  # gradients enabled
