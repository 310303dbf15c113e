"""Drop-in module surface on the CPU: constructor signatures, parameter names, seeded
initialisation and error behaviour of the reference's Field block API (canon:1131-1221)."""
from __future__ import annotations

import inspect

import numpy as np
import pytest
import torch

import fields_lm_amd as fl
from fields_lm_amd import FieldBlock, IndependentVacancyField, fused_field_read


def test_constructor_signatures_match_reference():
    # canon:1134-1141 and canon:1199-1207
    assert list(inspect.signature(IndependentVacancyField.__init__).parameters)[1:] == [
        "dim", "backend", "field_chunk", "triton_block_c", "triton_chunk_t"]
    assert list(inspect.signature(FieldBlock.__init__).parameters)[1:] == [
        "dim", "backend", "field_chunk", "triton_block_c", "triton_chunk_t", "ff_hidden"]
    params = inspect.signature(fused_field_read).parameters
    positional = [n for n, p in params.items() if p.kind != inspect.Parameter.KEYWORD_ONLY]
    assert positional == ["raw", "transition_r", "transition_i", "gamma", "block_c", "chunk_t"]
    # extensions are keyword-only, so every reference call site binds identically
    assert all(p.kind == inspect.Parameter.KEYWORD_ONLY for n, p in params.items() if n not in positional)


def test_seeded_construction_equals_reference_fixture(golden_dir):
    d = np.load(golden_dir / "selftest_block.npz")
    ref_sd = {k[len("param::"):]: d[k] for k in d.files if k.startswith("param::")}
    torch.manual_seed(7721)
    block = FieldBlock(64, "triton", 8, 8, 16, 192)
    sd = block.state_dict()
    assert list(sd) == list(ref_sd)  # same keys in the same registration order
    for k, v in sd.items():
        np.testing.assert_array_equal(v.numpy(), ref_sd[k], err_msg=k)
    block.load_state_dict({k: torch.from_numpy(v) for k, v in ref_sd.items()}, strict=True)


def test_parameter_count_promoted_geometry():
    mixer = IndependentVacancyField(1024, "triton", 32, 32, 64)
    assert sum(p.numel() for p in mixer.parameters()) == 4_725_248


def test_constructor_errors():
    with pytest.raises(ValueError):
        IndependentVacancyField(63, "triton", 32, 32, 64)
    with pytest.raises(ValueError):
        IndependentVacancyField(64, "cuda", 32, 32, 64)
    for backend in fl.BACKENDS:
        IndependentVacancyField(64, backend, 32, 32, 64)


def test_no_cpu_fallback():
    """The HIP path is the only path: CPU tensors raise like the reference's Triton path."""
    raw = torch.randn(1, 4, 24)
    p = torch.ones(8)
    with pytest.raises(RuntimeError):
        fused_field_read(raw, p, p, p, 32, 64)
    block = FieldBlock(16, "reference", 8, 8, 16, 64)
    with pytest.raises(RuntimeError):
        block(torch.randn(1, 4, 16))


def test_transition_params_match_oracle():
    from oracle import reference_path as ref

    mixer = IndependentVacancyField(256, "triton", 32, 32, 64)
    tr, ti, gamma = mixer.transition()
    etr, eti, egm = ref.transition_params(mixer.radius_logit.detach(), mixer.theta.detach())
    torch.testing.assert_close(tr, etr, rtol=0, atol=0)
    torch.testing.assert_close(ti, eti, rtol=0, atol=0)
    torch.testing.assert_close(gamma, egm, rtol=0, atol=0)
    assert float(gamma.min()) >= 0.01 - 1e-9 and float(tr.abs().max()) <= 0.99995


def test_forward_mode_through_the_fused_norm_is_refused(monkeypatch):
    """The fused scan has no forward-mode derivative: a dual read_norm.weight raises, it does not lose its
    tangent (the scan itself replaced by its shape: only the routing is under test)."""
    import torch.autograd.forward_ad as fwad

    from fields_lm_amd import field

    monkeypatch.setattr(field, "field_scan_norm", lambda raw, tr, ti, gamma, weight, eps, **kw:
                        torch.ones(*raw.shape[:2], 4 * tr.numel()) * weight.detach())
    m = field.IndependentVacancyField(16, "triton", 8, 8, 16)
    x = torch.randn(1, 3, 16)
    w = m.read_norm.weight.detach()
    del m.read_norm.weight
    with torch.no_grad(), fwad.dual_level():
        m.read_norm.weight = fwad.make_dual(w, torch.ones_like(w))
        with pytest.raises(NotImplementedError):
            m.normed_read(x)
        m.read_norm.weight = w
        assert m.normed_read(x).shape == (1, 3, 32)


def _host_eager(*tensors):
    """``eager`` without its device check, so that a route's other conditions decide on the CPU."""
    return all(type(t) in (torch.Tensor, torch.nn.Parameter)
               and not torch._C._functorch.is_functorch_wrapped_tensor(t) for t in tensors)


class _Call(torch.nn.Module):
    """A module's method as a forward, for functional_call."""

    def __init__(self, inner, fn):
        super().__init__()
        self.inner, self.fn = inner, fn

    def forward(self, *args):
        return self.fn(self.inner, *args)


def test_vmap_over_the_output_layer_of_a_residual(monkeypatch):
    """Only the layer's weight batched: the residual cannot take its product in place."""
    from fields_lm_amd import field

    monkeypatch.setattr(field, "eager", _host_eager)
    call = _Call(torch.nn.Linear(6, 4, bias=False), lambda layer, x, h: field._linear_residual(x, layer, h))
    x, h, ws = torch.randn(3, 4), torch.randn(3, 6), torch.randn(5, 4, 6)
    with torch.no_grad():
        got = torch.func.vmap(lambda w: torch.func.functional_call(call, {"inner.weight": w}, (x.clone(), h)))(ws)
    torch.testing.assert_close(got, x + torch.matmul(h, ws.transpose(1, 2)))


@pytest.mark.parametrize("name", ["ff.gate_up.weight", "residual_gate.weight", "residual_gate.bias", "norm2.weight"])
def test_vmap_over_refresh_block_weights_takes_the_stock_ops(monkeypatch, name):
    from fields_lm_amd import model as M

    def kernel(*args, **kw):
        raise AssertionError("a batched tensor on its way to a kernel")

    torch.manual_seed(2)
    blk = M.RefreshBlock(32, 4, 2, 16, 64, 32, 24).to(torch.bfloat16)
    call = _Call(blk, M.RefreshBlock._tail)
    x, z, a = (torch.randn(2, 3, 32).to(torch.bfloat16) for _ in range(3))
    ws = torch.stack([dict(blk.named_parameters())[name].detach() * k for k in (1, 2, 3)])
    with torch.no_grad():
        exp = torch.stack([torch.func.functional_call(call, {"inner." + name: w}, (x.clone(), z, a)) for w in ws])
        monkeypatch.setattr(M, "eager", _host_eager)
        monkeypatch.setattr(M, "gate_residual_norm", kernel)
        monkeypatch.setattr(M.RefreshBlock, "_gated", lambda self, x, z, a: x + self._gate(z) * a)
        got = torch.func.vmap(lambda w: torch.func.functional_call(call, {"inner." + name: w}, (x.clone(), z, a)))(ws)
    torch.testing.assert_close(got, exp, rtol=2e-2, atol=2e-2)


def test_refresh_block_replaced_layers_take_the_stock_ops(monkeypatch):
    """A gate or a packed projection that is not a plain layer may return any type or width (a gate of one
    column broadcasts): nothing that a kernel reads by address."""
    from fields_lm_amd import model as M

    def kernel(*args, **kw):
        raise AssertionError("a replaced layer's output on its way to a kernel")

    class Wide(torch.nn.Linear):
        def forward(self, x):
            return super().forward(x).float()

    monkeypatch.setattr(M, "eager", _host_eager)
    monkeypatch.setattr(M, "gate_residual_norm", kernel)
    monkeypatch.setattr(M.RefreshBlock, "_gated", lambda self, x, z, a: x + self._gate(z) * a)
    monkeypatch.setattr(M.GateUpSwiGLU, "forward", lambda self, x: self.down(torch.nn.functional.silu(
        self.gate_up(x).chunk(2, -1)[0].bfloat16())))
    x, z, a = (torch.randn(2, 3, 32).to(torch.bfloat16) for _ in range(3))
    parts = [("residual_gate", torch.nn.Linear(32, 1)), ("residual_gate", torch.nn.Sequential(torch.nn.Linear(32, 32))),
             ("gate_up", Wide(32, 48, bias=False)), ("gate_up", None)]
    for name, layer in parts:
        blk = M.RefreshBlock(32, 4, 2, 16, 64, 32, 24).to(torch.bfloat16)
        owner = blk if name == "residual_gate" else blk.ff
        if layer is None:  # the plain layer with a hook that changes its output's type
            owner.gate_up.register_forward_hook(lambda mod, args, out: out.float())
        else:
            setattr(owner, name, layer.to(torch.bfloat16))
        with torch.no_grad():
            assert blk._tail(x.clone(), z, a).shape == x.shape


def _training_block(monkeypatch):
    from fields_lm_amd import field

    monkeypatch.setattr(field, "eager", _host_eager)
    block = FieldBlock(16, "triton", 8, 8, 16, 24)
    return block, torch.randn(1, 3, 16)


def test_training_route_leaves_replaced_products_their_fp32_input(monkeypatch):
    """Under autocast the kernels write what a product reads in bf16; a layer that computes otherwise, or a
    hook that sees the input, gets the stock ops' fp32 values."""
    block, x = _training_block(monkeypatch)
    assert block._native_training(x)
    for owner, name in ((block.mixer, "out_proj"), (block.ff, "w12")):
        layer = getattr(owner, name)
        handle = layer.register_forward_pre_hook(lambda mod, args: None)
        assert not block._native_training(x)
        handle.remove()
        setattr(owner, name, torch.nn.Sequential(layer))
        assert not block._native_training(x)
        setattr(owner, name, layer)
    assert block._native_training(x)


@pytest.mark.parametrize("case", ["batched gate", "batched out", "batched up", "one gate column", "scalar norm"])
def test_training_route_checks_what_its_kernels_read(monkeypatch, case):
    """Outputs of batched or replaced layers, and weights of another shape that broadcast in the stock ops,
    stay with the stock ops."""
    from fields_lm_amd import field

    block, x = _training_block(monkeypatch)
    m = block.mixer

    def scan(raw, tr, ti, gamma, *args, **kw):
        return torch.cat((raw, raw[..., :raw.shape[-1] // 3]), -1)

    class Kernel:
        def __getattr__(self, name):
            raise AssertionError(name)

    def norm(t, w, eps, dtype):
        assert w.shape == t.shape[-1:] and _host_eager(t, w)
        return (t * torch.rsqrt(t.square().mean(-1, keepdim=True) + eps) * w).to(dtype)

    def gate_norm(t, out, gate, w, eps, dtype):
        assert out.shape == gate.shape == t.shape and _host_eager(t, out, gate)
        t = t + out * torch.sigmoid(gate)
        return t, norm(t, w, eps, dtype)

    monkeypatch.setattr(field, "fused_field_read", scan)
    monkeypatch.setattr(field.nat, "load", Kernel)
    for name, fn in (("Transition", lambda *a: field.train.transition_ops(*a)), ("Norm", norm), ("GateNorm", gate_norm)):
        monkeypatch.setattr(field.train, name, type(name, (), {"apply": staticmethod(fn)}))

    def swiglu(gu):
        assert _host_eager(gu)
        return field.train._swiglu_ops(gu)

    monkeypatch.setattr(field.train, "Swiglu", type("Swiglu", (), {"apply": staticmethod(swiglu)}))
    monkeypatch.setattr(field.IndependentVacancyField, "normed_read",
                        lambda self, t, raw=None: self.read_norm(scan(self.write_proj(t) if raw is None else raw, None, None, None)))
    if case == "one gate column":
        m.gate_proj = torch.nn.Linear(16, 1)
    elif case == "scalar norm":
        block.ff_norm.weight = torch.nn.Parameter(torch.ones(1))
    name = {"batched gate": "mixer.gate_proj.weight", "batched out": "mixer.out_proj.weight", "batched up": "ff.w12.weight"}.get(case)
    if name is None:
        block.fuse_tail = False
        exp = block(x)
        block.fuse_tail = True
        torch.testing.assert_close(block(x), exp)
        return
    ws = torch.stack([dict(block.named_parameters())[name].detach() * k for k in (1, 2)])
    got = torch.func.vmap(lambda w: torch.func.functional_call(block, {name: w}, (x,)))(ws)
    block.fuse_tail = False
    exp = torch.stack([torch.func.functional_call(block, {name: w}, (x,)) for w in ws])
    torch.testing.assert_close(got, exp)


def _step_call(monkeypatch):
    from fields_lm_amd import field
    from fields_lm_amd import model as M

    torch.manual_seed(4)
    block = M.cast_for_inference(FieldBlock(16, "triton", 8, 8, 16, 24))
    x, state = torch.randn(2, 16).to(torch.bfloat16), torch.zeros(2, 16)
    params = tuple(t.clone() for t in block.mixer.decode_params())  # the stock ops: no device here
    monkeypatch.setattr(field, "eager", _host_eager)
    return block, x, state, params


class _Gelu(torch.nn.Module):
    """A feed-forward with the packed layout's names and another activation."""

    def __init__(self):
        super().__init__()
        self.gate_up, self.down = torch.nn.Linear(16, 48, bias=False), torch.nn.Linear(24, 16, bias=False)

    def forward(self, x):
        gate, up = self.gate_up(x).chunk(2, -1)
        return self.down(torch.nn.functional.gelu(gate) * up)


def test_step_and_tail_ask_what_the_feed_forward_is(monkeypatch):
    """Only this package's SwiGLU classes, called without hooks, run as kernels; any other module is called."""
    block, x, state, params = _step_call(monkeypatch)
    with torch.no_grad():
        assert block._native_step(x, state, params) is not None and block._fused_tail(x)
        ff = block.ff
        handle = ff.register_forward_hook(lambda mod, args, out: out * 2)
        assert block._native_step(x, state, params) is None and not block._fused_tail(x)
        handle.remove()
        for other in (_Gelu(), torch.nn.Sequential(torch.nn.Linear(16, 16)), torch.nn.Identity()):
            block.ff = other.to(torch.bfloat16)
            assert block._native_step(x, state, params) is None and not block._fused_tail(x)
        block.ff = ff
        for owner, name in ((block, "ff_norm"), (block.mixer, "read_norm"), (block.mixer, "write_proj"),
                            (block.mixer, "gate_proj"), (block.mixer, "out_proj"), (ff, "w12"), (ff, "w3")):
            handle = getattr(owner, name).register_forward_pre_hook(lambda mod, args: None)
            assert block._native_step(x, state, params) is None, name
            handle.remove()
        assert block._native_step(x, state, params) is not None


@pytest.mark.parametrize("name,entries", [("write_proj.bias", 1), ("gate_proj.bias", 1), ("out_proj.bias", 1), ("ff_norm.weight", 1)])
def test_step_checks_the_length_of_vectors(monkeypatch, name, entries):
    """A bias or norm weight of one entry broadcasts in the stock ops; the kernels read whole vectors."""
    block, x, state, params = _step_call(monkeypatch)
    owner, attr = name.split(".")
    layer = block.ff_norm if owner == "ff_norm" else getattr(block.mixer, owner)
    setattr(layer, attr, torch.nn.Parameter(torch.ones(entries, dtype=torch.bfloat16)))
    with torch.no_grad():
        assert block._native_step(x, state, params) is None


def test_softpatch_route_asks_what_its_layers_are(monkeypatch):
    """A down projection, scorer or up projection that is wrapped, hooked or of another width stays with the
    stock ops: the kernels read bf16 rows of the rank's width by address."""
    from fields_lm_amd import field
    from fields_lm_amd import model as M

    monkeypatch.setattr(field, "eager", _host_eager)
    monkeypatch.setattr(M, "eager", _host_eager)
    x, tok = torch.randn(1, 3, 32).to(torch.bfloat16), torch.zeros(1, 3, dtype=torch.long)

    def mixer():
        sp = M.BoundaryStateMixer(32, 8, vocab=5)
        return M.cast_for_inference(sp)

    with torch.no_grad():
        assert mixer()._native(x, tok)
        for edit in (lambda sp: setattr(sp, "down", torch.nn.Sequential(sp.down)),
                     lambda sp: setattr(sp, "down", torch.nn.Identity()),
                     lambda sp: sp.down.register_forward_hook(lambda mod, args, out: out.float()),
                     lambda sp: setattr(sp, "down", torch.nn.Linear(32, 8).to(torch.bfloat16)),
                     lambda sp: setattr(sp, "down", torch.nn.Linear(32, 6, bias=False).to(torch.bfloat16)),
                     lambda sp: setattr(sp, "down", torch.nn.Linear(32, 8, bias=False)),
                     lambda sp: setattr(sp, "score", torch.nn.Linear(16, 1).to(torch.bfloat16)),
                     lambda sp: setattr(sp, "score", torch.nn.Linear(32, 2).to(torch.bfloat16)),
                     lambda sp: setattr(sp, "up", torch.nn.Linear(16, 16, bias=False).to(torch.bfloat16))):
            sp = mixer()
            edit(sp)
            assert not sp._native(x, tok)


def test_mamba_routes_check_what_their_kernels_read(monkeypatch):
    """Parameters that broadcast in the stock ops, a projection of another width, and an inner width that is
    no whole number of heads: the kernels read by the promoted shapes."""
    from fields_lm_amd import model as M

    monkeypatch.setattr(M, "eager", _host_eager)

    class Kernel:
        def __getattr__(self, name):
            raise AssertionError(name)

    monkeypatch.setattr(M.nat, "load", Kernel)
    one = lambda n=1: torch.nn.Parameter(torch.ones(n))  # noqa: E731
    with torch.no_grad():
        m = M.Mamba2Mixer(64)
        z = m.in_proj(torch.randn(1, 3, 64))
        assert m._native(z) and not m._native(z[..., :-2].contiguous()) and not m._native(torch.cat((z, z[..., :2]), -1))
        for name in ("A_log", "dt_bias", "D"):
            m = M.Mamba2Mixer(64)
            setattr(m, name, one())
            assert not m._native(z), name
        for owner, name, value in (("norm", "weight", one()), ("conv1d", "bias", one()),
                                   ("conv1d", "weight", torch.nn.Parameter(torch.ones(1, 1, 4)))):
            m = M.Mamba2Mixer(64)
            setattr(getattr(m, owner), name, value)
            assert not m._native(z), name
        m = M.Mamba2Mixer(48)  # 96 channels: one head and a half
        assert not m._native(m.in_proj(torch.randn(1, 3, 48)))
        m = M.Mamba2Mixer(64)
        rows = torch.randn(1, 3, m.conv_dim).to(torch.bfloat16)
        for name, value in (("bias", one()), ("weight", torch.nn.Parameter(torch.ones(1, 1, 4)))):
            m = M.Mamba2Mixer(64)
            setattr(m.conv1d, name, value)
            assert m._conv_silu(rows).shape == rows.shape  # the stock ops: no kernel was called
        monkeypatch.setattr(M, "_autocast_operands", lambda product, *others: product.dtype == torch.bfloat16)
        m = M.Mamba2Mixer(64)
        m.D = one()
        b, h, c, s, p, length = 1, 2, 1, 4, 64, 3
        y = torch.zeros(b, h, c, s, p, dtype=torch.bfloat16)
        acs, xh = torch.zeros(b, h, c, s), torch.zeros(b, length, h, p)
        zz = torch.zeros(b, length, h * p, dtype=torch.bfloat16)
        assert m._finish(y, y, acs, xh, zz) is None
        monkeypatch.setattr(M, "_autocast_operands",
                            lambda product, *others: len(others) == 3)  # only the operands' kernel
        y, _ = M.ssd_chunked(torch.randn(1, 8, 2, 4), torch.rand(1, 8, 1), -torch.ones(2), torch.randn(1, 8, 4),
                             torch.randn(1, 8, 4), 8)
        assert y.shape == (1, 8, 2, 4)


@pytest.mark.parametrize("shape", [(64,), (4, 1, 1)])
def test_refresh_attention_with_a_wider_mix_takes_the_stock_ops(monkeypatch, shape):
    """global_mix_logit per dimension or per head broadcasts in the stock ops; the kernels read one value."""
    from fields_lm_amd import model as M

    monkeypatch.setattr(M, "eager", _host_eager)
    att = M.cast_for_inference(M.LandmarkAttention(256, 4, 2, 16, 64, 32))
    x = torch.randn(2, 5, 256).to(torch.bfloat16)
    with torch.no_grad():
        st = att.new_state(2, 40, x.device, x.dtype)
        qlat, pos = att.q_latent_proj(x), torch.tensor(0)
        assert att._native(qlat) and att._exact(x, qlat) and att._native_step(qlat[:, 0].contiguous(), pos, st)
        att.global_mix_logit = torch.nn.Parameter(torch.zeros(shape, dtype=torch.bfloat16))
        assert not (att._native(qlat) or att._exact(x, qlat) or att._native_step(qlat[:, 0].contiguous(), pos, st))


def test_step_route_ends_where_its_products_lose(monkeypatch):
    """Wide blocks with many rows take the library's products; the line is weights x rows."""
    from fields_lm_amd import field

    block, x, state, params = _step_call(monkeypatch)
    work = 2 * (9 * 16 * 16 // 2 + 3 * 16 * 24)
    with torch.no_grad():
        for limit, native in ((work, True), (work - 1, False)):
            monkeypatch.setattr(field, "_STEP_WORK", limit)
            assert (block._native_step(x, state, params) is not None) == native


@pytest.mark.parametrize("attr", ["weight", "bias"])
def test_step_route_without_a_registered_parameter(monkeypatch, attr):
    """A weight or bias kept as a plain attribute (no longer a parameter) takes the separate launches."""
    block, x, state, params = _step_call(monkeypatch)
    layer = block.mixer.out_proj
    value = getattr(layer, attr).detach()
    delattr(layer, attr)
    setattr(layer, attr, value)
    with torch.no_grad():
        assert block._native_step(x, state, params) is None


def test_stock_gradients_with_frozen_inputs():
    """Differentiable gradients where some inputs, or some outputs with them, need none."""
    from fields_lm_amd import _train

    a, b, g = torch.randn(3), torch.randn(3), torch.randn(3)
    assert _train._stock_grads(lambda o, s: o * s, (a, b), (g,)) == [None, None]
    b.requires_grad_()
    ga, gb = _train._stock_grads(lambda o, s: (o * 2, s * s), (a, b), (g, g))  # the first output needs none
    assert ga is None
    torch.testing.assert_close(gb, 2 * b * g)
    assert _train._stock_grads(_train.transition_ops, (a, b), (g, g, g))[0] is None  # gamma depends on a alone
