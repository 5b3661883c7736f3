"""GEMM-GELU backward on the GPU: the fused gelu'(x @ w.T + b) * dout epilogue
and the autograd of strata_hip::gemm_bias_act / GemmGeluMlp, against torch's
own autograd of Linear + GELU(tanh) in fp32 on the same bf16 inputs
(relative L2 <= 1e-2)."""

import pytest
import torch
import torch.nn.functional as F

from strata_amd import _lib, ops
from strata_amd.modules import GemmGeluMlp

from .conftest import rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [(300, 512, 256), (4096, 1024, 1024), (77, 200, 64)]  # (M, N, K)


def _bf(shape, g, scale=1.0):
    return (torch.randn(shape, generator=g) * scale).bfloat16()


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_gelu_grad_epilogue(gpu, shape):
    M, N, K = shape
    g = torch.Generator().manual_seed(0)
    x, w, b, dout = _bf((M, K), g), _bf((N, K), g, K**-0.5), _bf((N,), g), _bf((M, N), g)
    got = ops.gemm_bias_act(x.to(gpu), w.to(gpu), b.to(gpu), dout.to(gpu), _lib.ACT_GELU_TANH_GRAD, _lib.RES_MUL)
    a = (x.double() @ w.double().T + b.double()).requires_grad_(True)
    (ga,) = torch.autograd.grad(F.gelu(a, approximate="tanh"), a, dout.double())
    assert rel_l2(got.float().cpu(), ga.float()) <= 1e-2


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("act", [_lib.ACT_GELU_TANH, _lib.ACT_NONE])
def test_gemm_autograd_vs_torch(gpu, shape, act):
    M, N, K = shape
    g = torch.Generator().manual_seed(1)
    x, w, b, r, dout = _bf((M, K), g), _bf((N, K), g, K**-0.5), _bf((N,), g), _bf((M, N), g), _bf((M, N), g)
    res = act == _lib.ACT_NONE  # the fc2 + residual shape; GELU runs without one (fc1)
    leaves = [t.to(gpu).requires_grad_(True) for t in ((x, w, b, r) if res else (x, w, b))]
    out = ops.gemm_bias_act(leaves[0], leaves[1], leaves[2], leaves[3] if res else None, act)
    out.backward(dout.to(gpu))
    ref_leaves = [t.float().requires_grad_(True) for t in ((x, w, b, r) if res else (x, w, b))]
    y = F.linear(ref_leaves[0], ref_leaves[1], ref_leaves[2])
    y = F.gelu(y, approximate="tanh") if act == _lib.ACT_GELU_TANH else y + ref_leaves[3]
    y.backward(dout.float())
    for name, a, bref in zip("xwbr", leaves, ref_leaves):
        assert rel_l2(a.grad.float().cpu(), bref.grad) <= 1e-2, name


@pytest.mark.parametrize("shape", [(300, 512, 256), (4096, 1024, 1024), (1000, 4104, 128)], ids=str)
def test_gemm_gelu_train(gpu, shape):
    """fc1 for training: its GELU output equals the inference launch's bit for bit, the
    saved derivative is gelu'(x @ w.T + b) within bf16 rounding, and its autograd (the
    derivative times the upstream gradient, then plain GEMMs and the bias gradient)
    matches torch's Linear + GELU(tanh) backward."""
    M, N, K = shape
    g = torch.Generator().manual_seed(3)
    x, w, b, dout = _bf((M, K), g), _bf((N, K), g, K**-0.5), _bf((N,), g), _bf((M, N), g)
    xg, wg, bg = (t.to(gpu).requires_grad_(True) for t in (x, w, b))
    out, dact = ops.gemm_gelu_train(xg, wg, bg)
    plain = ops.gemm_bias_act(x.to(gpu), w.to(gpu), b.to(gpu), None, _lib.ACT_GELU_TANH)
    assert torch.equal(out.detach(), plain)
    a = (x.double() @ w.double().T + b.double()).requires_grad_(True)
    (ga,) = torch.autograd.grad(F.gelu(a, approximate="tanh"), a, torch.ones_like(a))
    assert rel_l2(dact.float().cpu(), ga.float()) <= 1e-2
    out.backward(dout.to(gpu))
    ref = [t.float().requires_grad_(True) for t in (x, w, b)]
    F.gelu(F.linear(*ref), approximate="tanh").backward(dout.float())
    for name, got, r in zip("xwb", (xg, wg, bg), ref):
        assert rel_l2(got.grad.float().cpu(), r.grad) <= 1e-2, name


def test_mlp_module_backward(gpu):
    torch.manual_seed(0)
    mlp = GemmGeluMlp(256, 1024)
    g = torch.Generator().manual_seed(2)
    x, r, dout = _bf((2, 8, 16, 256), g), _bf((2, 8, 16, 256), g), _bf((2, 8, 16, 256), g)
    ref = GemmGeluMlp(256, 1024)
    ref.load_state_dict(mlp.state_dict())
    ref = ref.float()
    mlp = mlp.to(gpu).bfloat16()
    xg = x.to(gpu).requires_grad_(True)
    mlp(xg, r.to(gpu)).backward(dout.to(gpu))
    xr = x.float().requires_grad_(True)
    (ref.layers(xr) + r.float()).backward(dout.float())
    assert rel_l2(xg.grad.float().cpu(), xr.grad) <= 1e-2
    for (n1, p1), (n2, p2) in zip(mlp.named_parameters(), ref.named_parameters()):
        assert n1 == n2
        assert rel_l2(p1.grad.float().cpu(), p2.grad.bfloat16().float()) <= 1e-2, n1


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_gate_autograd_vs_torch(gpu, shape):
    """The attention gate sigmoid(x @ w.T + b) * a: gradients of x, w, b and a."""
    M, N, K = shape
    g = torch.Generator().manual_seed(3)
    x, w, b, a, dout = _bf((M, K), g), _bf((N, K), g, K**-0.5), _bf((N,), g), _bf((M, N), g), _bf((M, N), g)
    leaves = [t.to(gpu).requires_grad_(True) for t in (x, w, b, a)]
    ops.gemm_bias_act(*leaves, _lib.ACT_SIGMOID, _lib.RES_MUL).backward(dout.to(gpu))
    ref = [t.float().requires_grad_(True) for t in (x, w, b, a)]
    (torch.sigmoid(F.linear(ref[0], ref[1], ref[2])) * ref[3]).backward(dout.float())
    for name, got, want in zip("xwba", leaves, ref):
        assert rel_l2(got.grad.float().cpu(), want.grad) <= 1e-2, name


@pytest.mark.parametrize("shape", [(1, 8, 8), (63, 64, 72), (64, 256, 256), (65, 264, 248), (257, 8, 520),
                                   (1000, 384, 640), (20000, 200, 72), (70000, 264, 264)], ids=str)
def test_linear_grads(gpu, shape):
    """g.T @ x and the column sums of g at the edges of a 64-row stage, a 256-column tile and a row split, against float64
    (rounded once to bf16: 2^-9 of a value, 1.7e-3 of the norm; 3e-3 with the fp32 sums), from
    rows of wider tensors too, and bit for bit on a repeat."""
    M, N, K = shape
    g = torch.Generator().manual_seed(M + N + K)
    a, x = _bf((M, N + 8), g).to(gpu), _bf((M, K + 16), g).to(gpu)
    ref = a[:, :N].double().t() @ x[:, 16:].double()
    got, db = ops.linear_grads(a[:, :N], x[:, 16:], True)
    assert rel_l2(got.float().cpu(), ref.float().cpu()) <= 3e-3
    assert rel_l2(db.float().cpu(), a[:, :N].double().sum(0).float().cpu()) <= 3e-3
    again, none = ops.linear_grads(a[:, :N].contiguous(), x[:, 16:].contiguous(), False)
    assert torch.equal(got, again) and none.numel() == 0
    assert torch.equal(db, ops.linear_grads(a[:, :N], x[:, 16:], True)[1])


def test_linear_grads_second_derivative(gpu):
    """create_graph through a Linear's weight gradient, against torch's own."""
    g = torch.Generator().manual_seed(5)
    x, w, v = _bf((40, 24), g), _bf((16, 24), g), _bf((16, 24), g)

    def second(linear, dt):
        xi, wi = (t.to(gpu, dt).requires_grad_(True) for t in (x, w))
        (dw,) = torch.autograd.grad(linear(xi, wi).square().sum(), wi, create_graph=True)
        return torch.autograd.grad((dw * v.to(gpu, dt)).sum(), xi)[0]

    got = second(lambda a, b: ops.gemm_bias_act(a, b, None, None, _lib.ACT_NONE), torch.bfloat16)
    ref = second(lambda a, b: F.linear(a, b), torch.float64)
    assert rel_l2(got.double().cpu(), ref.cpu()) <= 2e-2


@pytest.mark.parametrize("shape", [(1, 8, 8, 8), (300, 64, 256, 72), (4096, 256, 1024, 256)], ids=str)
@pytest.mark.parametrize("frozen", [(), ("w2",), ("x", "w1", "b1")], ids=str)
def test_mlp_train_autograd(gpu, shape, frozen):
    """The MLP's one-op autograd against torch's in fp32 (1e-2, as the Mlp test above), with
    every gradient, without fc2's weight's, and with fc2's and the residual's alone."""
    M, K, H, N = shape
    g = torch.Generator().manual_seed(M + H)
    vals = dict(x=_bf((M, K), g), w1=_bf((H, K), g, K**-0.5), b1=_bf((H,), g), w2=_bf((N, H), g, H**-0.5),
                b2=_bf((N,), g), r=_bf((M, N), g))
    dout = _bf((M, N), g)
    grads = []
    for dt in (torch.bfloat16, torch.float32):
        t = {k: v.to(gpu, dt).requires_grad_(k not in frozen) for k, v in vals.items()}
        if dt == torch.bfloat16:
            out = ops.mlp_gelu_train(*t.values())[0]
        else:
            out = F.linear(F.gelu(F.linear(t["x"], t["w1"], t["b1"]), approximate="tanh"), t["w2"], t["b2"]) + t["r"]
        out.backward(dout.to(gpu, dt))
        grads.append({k: v.grad for k, v in t.items()})
    for k, a in grads[0].items():
        assert (a is None) == (k in frozen)
        if a is not None:
            assert rel_l2(a.float().cpu(), grads[1][k].cpu()) <= 1e-2, k


def test_mlp_second_derivative(gpu):
    """A penalty on the gradient of fc2's weight reaches x and fc1 through the hidden layer, on the
    kernels (2e-2: the roundings of the chain, as for the Linear above)."""
    g = torch.Generator().manual_seed(6)
    vals = dict(x=_bf((40, 24), g), w1=_bf((64, 24), g, 24**-0.5), b1=_bf((64,), g), w2=_bf((16, 64), g, 64**-0.5),
                b2=_bf((16,), g), r=_bf((40, 16), g))
    grads = []
    for dt in (torch.bfloat16, torch.float64):
        t = {k: v.to(gpu, dt).requires_grad_(True) for k, v in vals.items()}
        if dt == torch.bfloat16:
            out = ops.mlp_gelu_train(*t.values())[0]
        else:
            out = F.linear(F.gelu(F.linear(t["x"], t["w1"], t["b1"]), approximate="tanh"), t["w2"], t["b2"]) + t["r"]
        (dw2,) = torch.autograd.grad(out.square().sum(), t["w2"], create_graph=True)
        grads.append(torch.autograd.grad(dw2.square().sum(), [t[k] for k in ("x", "w1", "b1")]))
    for name, a, b in zip(("x", "w1", "b1"), *grads):
        assert rel_l2(a.double().cpu(), b.cpu()) <= 2e-2, name


def test_gelu_train_refusals_are_the_librarys_error(gpu):
    """K that is no multiple of 8: StrataHipError (a RuntimeError), from the op and the module."""
    x, w = torch.zeros(4, 12, dtype=torch.bfloat16, device=gpu), torch.zeros(16, 12, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(_lib.StrataHipError, match="multiple of 8"):
        ops.gemm_gelu_train(x, w, None)
    with pytest.raises(_lib.StrataHipError, match="multiple of 8"):
        GemmGeluMlp(12, 16, 8).to(gpu).bfloat16()(x.requires_grad_(True))
