"""The layer RMSNorm and SwiGLU's product on the kernels, against the same formulas
in 64 bits with the roundings between the steps that the data types give."""

import pytest
import torch
import torch.nn.functional as F

from nano_qwen_amd.model import LayerRMSNorm, ModelConfig, Qwen3Model, SwiGLU, TransformerBlock, _SwiGLUProduct
from nano_qwen_amd.norm import layer_rms_norm, rms_norm
from tests.helpers import randn, say

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, F32 = torch.bfloat16, torch.float32


def _close(got, want, dtype, terms, what):
    # 2-norm: a result passes at most two bf16 roundings of 2^-9 beside the ones
    # restated; fp32 sums of `terms` terms round by about sqrt(terms) 2^-24
    lim = 2.0 ** -8 if dtype == BF else 8 * terms ** 0.5 * 2.0 ** -24
    got, want = got.detach().double().cpu(), want.double()
    err = float((got - want).norm() / want.norm())
    assert err <= lim, (what, err, lim)


# one, some and all of a lane's chunks; rows below, at and above a workgroup's four and the grid's 2048
@pytest.mark.parametrize("rows,width", [(1, 8), (3, 256), (5, 512), (4, 520), (2049, 1024), (7, 2048), (2600, 2056),
                                        (2, 4096)])
@pytest.mark.parametrize("xdt,wdt", [(BF, BF), (BF, F32), (F32, F32), (F32, BF)])
def test_layer_rmsnorm(rows, width, xdt, wdt):
    say(f"layer RMSNorm {rows}x{width} {xdt} {wdt}")
    x = randn(rows, width, seed=11, dtype=xdt)
    w = (1 + 0.1 * randn(width, seed=12)).to(wdt)
    norm = LayerRMSNorm(width, input_kept=True).to(DEV, wdt)
    with torch.no_grad():
        norm.weight.copy_(w)
    xd = x.to(DEV).requires_grad_()
    y = norm(xd)
    ydt = torch.promote_types(xdt, wdt)
    assert y.dtype == ydt and y.grad_fn.name().startswith("LayerRMSNormFn")
    dy = randn(rows, width, seed=13, dtype=ydt)
    dx, dw = torch.autograd.grad(y, (xd, norm.weight), dy.to(DEV))
    with torch.no_grad():
        assert torch.equal(norm(xd), y)
    x6, w6, d6 = x.double(), w.double(), dy.double()
    r = torch.rsqrt(x6.square().mean(-1, keepdim=True) + 1e-6)
    n = x6 * r
    g = (d6 * w6).to(xdt).double()
    _close(y, (n.to(xdt).double() * w6), ydt, width, "y")
    _close(dx, r * (g - n * (g * n).mean(-1, keepdim=True)), xdt, width, "dx")
    # a bf16 n may round the other way: 2^-8 of a term now and then
    _close(dw, (d6 * n.to(xdt).double()).sum(0), BF if BF in (xdt, wdt) else F32, rows, "dw")
    assert dx.dtype == xdt and dw.dtype == wdt


@pytest.mark.parametrize("xdt", [BF, F32])
def test_one_row_of_a_wider_tensor(xdt):
    """A single row counts as contiguous whatever its stride, here no multiple of 16 bytes."""
    say(f"one row of a wider tensor {xdt}")
    big = randn(4, 71, seed=14, dtype=xdt)
    w = (1 + 0.1 * randn(64, seed=15)).to(xdt)
    norm = LayerRMSNorm(64).to(DEV, xdt)
    with torch.no_grad():
        norm.weight.copy_(w)
    x = big.to(DEV)[:1, :64]
    assert x.is_contiguous() and x.stride(0) == 71
    want = (big[:1, :64].double() * torch.rsqrt(big[:1, :64].double().square().mean(-1, keepdim=True) + 1e-6))
    want = want.to(xdt).double() * w.double()
    with torch.no_grad():
        _close(norm(x), want, xdt, 64, "y")
    _close(rms_norm(x, norm.weight.detach(), 1e-6), want, xdt, 64, "rms_norm")
    xg = x.detach().requires_grad_()
    y = norm(xg)
    _close(y, want, xdt, 64, "y with a gradient")
    (dx,) = torch.autograd.grad(y, xg, torch.ones_like(y))
    z = layer_rms_norm(xg, norm.weight, 1e-6)
    (want,) = torch.autograd.grad(z, xg, torch.ones_like(z))
    _close(dx, want.double().cpu(), xdt, 64, "dx")


def test_layer_rmsnorm_other_routes():
    """Calls the kernels do not take give what the tensor operations give."""
    norm = LayerRMSNorm(64, input_kept=True).to(DEV)
    x = randn(6, 64, seed=21).to(DEV).requires_grad_()
    # the gradient of the gradient
    y = norm(x)
    (gx,) = torch.autograd.grad(y.square().sum(), x, create_graph=True)
    (ggx,) = torch.autograd.grad(gx.square().sum(), x)
    z = layer_rms_norm(x, norm.weight, 1e-6)
    (hx,) = torch.autograd.grad(z.square().sum(), x, create_graph=True)
    (hhx,) = torch.autograd.grad(hx.square().sum(), x)
    torch.testing.assert_close(ggx, hhx, rtol=1e-3, atol=1e-5)
    # vmap, forward mode, a batch of gradients, a width and a layout the kernels do not take
    torch.testing.assert_close(torch.vmap(norm)(x[None])[0], z)
    torch.func.jvp(lambda t: layer_rms_norm(t, norm.weight, 1e-6), (x.detach(),), (x.detach(),))
    torch.func.jvp(norm, (x.detach(),), (x.detach(),))
    dys = torch.stack([torch.ones_like(y), 2 * torch.ones_like(y)])
    (b,) = torch.autograd.grad(norm(x), x, dys, is_grads_batched=True)
    torch.testing.assert_close(b[1], 2 * b[0])
    torch.testing.assert_close(torch.jit.script(norm)(x), z)
    odd = LayerRMSNorm(63).to(DEV)
    assert odd(x[:, :63]).shape == (6, 63) and norm(x[:0]).shape == (0, 64)
    xt = randn(64, 6, seed=22).to(DEV).t()
    assert norm(xt).stride() == layer_rms_norm(xt, norm.weight, 1e-6).stride()
    # without input_kept the input may change before the backward
    free = LayerRMSNorm(64).to(DEV, BF)
    h = randn(6, 64, seed=23, dtype=BF).to(DEV).requires_grad_() * 1
    out = free(h)
    h.add_(1)
    out.sum().backward()


def test_block_input_may_change_before_backward():
    """A block's caller may reuse its bf16 input's memory: gradients are those of the forward's input."""
    say("block input overwritten before the backward")
    cfg = ModelConfig(vocab_size=64, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                      num_attention_heads=4, num_key_value_heads=2, head_dim=32)
    block = TransformerBlock(cfg).to(DEV, BF)
    grads = []
    for overwrite in (False, True):
        x = randn(2, 9, 64, seed=24, dtype=BF).to(DEV).requires_grad_()
        h = x * 1
        y = block(h)
        y = y[0] if isinstance(y, tuple) else y
        if overwrite:
            h.zero_()
        grads.append(torch.autograd.grad(y.float().sum(), [x, *block.parameters()]))
    for a, b in zip(*grads):
        _close(b, a.double().cpu(), BF, 1, "gradient")


@pytest.mark.parametrize("name", ["norm", "layers.0.post_attention_layernorm", "layers.0.input_layernorm"])
def test_models_norms_let_their_input_change(name):
    """A program that calls one of a model's norms may write to its bf16 input before the backward."""
    say(f"input of {name} overwritten before the backward")
    cfg = ModelConfig(vocab_size=64, hidden_size=64, intermediate_size=128, num_hidden_layers=1,
                      num_attention_heads=4, num_key_value_heads=2, head_dim=32)
    norm = Qwen3Model(cfg).to(DEV, BF).get_submodule(name)
    grads = []
    for overwrite in (False, True):
        x = randn(5, 64, seed=25, dtype=BF).to(DEV).requires_grad_()
        h = x * 1
        y = norm(h)
        if overwrite:
            h.mul_(3)
        grads.append(torch.autograd.grad(y.float().square().sum(), [x, norm.weight]))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 8), (3, 683, 8), (2, 5, 6144)])
@pytest.mark.parametrize("dt", [BF, F32])
def test_swiglu_product(shape, dt):
    say(f"SwiGLU product {shape} {dt}")
    g, u, dy = (randn(*shape, seed=31 + i, dtype=dt) * (3 if i == 0 else 1) for i in range(3))
    gd, ud = g.to(DEV).requires_grad_(), u.to(DEV).requires_grad_()
    y = _SwiGLUProduct.apply(gd, ud)
    dg, du = torch.autograd.grad(y, (gd, ud), dy.to(DEV))
    g6, u6, d6 = g.double(), u.double(), dy.double()
    s = torch.sigmoid(g6)
    silu = (g6 * s).to(dt).double()
    _close(y, silu * u6, dt, 1, "y")
    _close(du, d6 * silu, dt, 1, "dup")
    _close(dg, (d6 * u6).to(dt).double() * s * (1 + g6 * (1 - s)), dt, 1, "dgate")


def test_swiglu_other_routes():
    ffn = SwiGLU(64, 128).to(DEV)
    x = randn(5, 64, seed=41).to(DEV)

    def plain(t):
        return ffn.down_proj(F.silu(ffn.gate_proj(t)) * ffn.up_proj(t))
    torch.testing.assert_close(ffn(x), plain(x))
    torch.testing.assert_close(torch.vmap(ffn)(x[None])[0], plain(x))
    torch.testing.assert_close(torch.jit.script(ffn)(x), plain(x))
    for f in (ffn, plain):
        torch.func.jvp(f, (x,), (x,))
    xs = x.clone().requires_grad_()
    res = []
    for f in (ffn, plain):
        (a,) = torch.autograd.grad(f(xs).square().sum(), xs, create_graph=True)
        (b,) = torch.autograd.grad(a.square().sum(), xs)
        res.append(b)
    torch.testing.assert_close(res[0], res[1], rtol=1e-3, atol=1e-5)
    gates = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -100.0, 100.0, 1e30, -1e30], device=DEV)
    torch.testing.assert_close(_SwiGLUProduct.apply(gates, torch.ones_like(gates)), F.silu(gates), equal_nan=True)


@pytest.mark.parametrize("rows,kernel", [(8191, False), (8192, True)])
def test_swiglu_route_by_size(rows, kernel):
    """A product with a gradient goes through the kernels from 2^23 elements on, one without always; the values agree."""
    say(f"SwiGLU of {rows} x 1024, with a gradient and without")
    ffn = SwiGLU(64, 1024).to(DEV, BF)
    seen = []
    ffn.down_proj.register_forward_pre_hook(lambda mod, args: seen.append(args[0]))
    x = randn(rows, 64, seed=42, dtype=BF).to(DEV).requires_grad_()
    y = ffn(x)
    assert seen[0].grad_fn.name().startswith("_SwiGLUProduct") == kernel
    with torch.no_grad():
        ffn(x)
    # one route rounds silu(gate) as the other does, which may fall the other way
    for p in seen:
        _close(p, (F.silu(ffn.gate_proj(x).double()).to(BF).double() * ffn.up_proj(x).double()).detach().cpu(), BF, 1, "product")
    (dx,) = torch.autograd.grad(y, x, torch.ones_like(y))
    g, u = ffn.gate_proj(x), ffn.up_proj(x)
    (want,) = torch.autograd.grad(ffn.down_proj(F.silu(g) * u), x, torch.ones_like(y))
    _close(dx, want.double().cpu(), BF, 1, "dx")
