"""Autograd of the one-op MLP (``mlp_gelu_train``) without a GPU: its launches are replaced by
torch products, so what is under test is the graph its backward builds."""

import pytest
import torch
import torch.nn.functional as F
from torch.fx.experimental.proxy_tensor import make_fx

from strata_amd import _lib, ops
from strata_amd.modules import GemmGeluMlp

from .conftest import rel_l2


def _gelu_and_grad(z):
    """gelu_tanh(z) and its derivative (an op's implementation runs below autograd: written out)."""
    k = (2.0 / torch.pi) ** 0.5
    t = torch.tanh(k * (z + 0.044715 * z**3))
    return 0.5 * z * (1 + t), 0.5 * (1 + t) + 0.5 * z * (1 - t * t) * k * (1 + 3 * 0.044715 * z * z)


@pytest.fixture
def torch_launches(monkeypatch):
    """The ops' launches on the CPU: fp32 products, each result rounded to bf16."""

    def linear(x, w, b):
        return F.linear(x.float(), w.float(), b.float() if b is not None else None)

    def gemm(x, w, b, residual, act, res_op):
        assert act == _lib.ACT_NONE
        z = linear(x, w, b).bfloat16()
        if residual is None:
            return z
        z = z.float() * residual.float() if res_op == _lib.RES_MUL else z.float() + residual.float()
        return z.bfloat16()

    def gelu_train(x, w, b):
        h, d = _gelu_and_grad(linear(x, w, b))
        return h.bfloat16(), d.bfloat16()

    def linear_grads(g, x, bias):
        return (g.float().t() @ x.float()).to(g.dtype), g.float().sum(0).to(g.dtype) if bias else g.new_empty(0)

    monkeypatch.setattr(ops, "_require_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_gemm_launch", gemm)
    monkeypatch.setattr(ops, "_gemm_gelu_train_launch", gelu_train)
    monkeypatch.setattr(ops, "linear_grads", linear_grads)


def _second(m, x, residual, wrt, fixed_upstream):
    """d |dW2|^2 / d(wrt): of loss = |out|^2, or with an upstream gradient that depends on nothing."""
    out = m(x, residual)
    up = None if not fixed_upstream else torch.ones_like(out)
    loss = out if fixed_upstream else out.square().sum()
    (dw2,) = torch.autograd.grad(loss, m.layers[2].weight, up, create_graph=True)
    return torch.autograd.grad(dw2.square().sum(), wrt)


class _Reference(torch.nn.Module):
    def __init__(self, layers):
        super().__init__()
        self.layers = layers

    def forward(self, x, residual):
        return self.layers(x) + residual


@pytest.mark.parametrize("fixed_upstream", [False, True])
def test_second_derivative_reaches_the_hidden_layer(torch_launches, fixed_upstream):
    """A penalty on fc2's weight gradient dY^T h reaches x, fc1's weight and bias through h, as in
    float64 (bf16 roundings of out, h and each gradient in the chain: six of 2^-9, so 1.2e-2; a
    path that is cut is off by a third or more)."""
    torch.manual_seed(0)
    m = GemmGeluMlp(24, 64, 16).bfloat16()
    x, r = torch.randn(40, 24).bfloat16().requires_grad_(True), torch.randn(40, 16).bfloat16()
    got = _second(m, x, r, [x, m.layers[0].weight, m.layers[0].bias], fixed_upstream)
    ref = _Reference(torch.nn.Sequential(torch.nn.Linear(24, 64), torch.nn.GELU(approximate="tanh"),
                                         torch.nn.Linear(64, 16))).double()
    ref.load_state_dict({k: v.double() for k, v in m.state_dict().items()})
    xd = x.detach().double().requires_grad_(True)
    want = _second(ref, xd, r.double(), [xd, ref.layers[0].weight, ref.layers[0].bias], fixed_upstream)
    for name, a, b in zip(("x", "w1", "b1"), got, want):
        assert rel_l2(a, b) <= 1.2e-2, name


@pytest.mark.parametrize("needs", [("x", "r", "layers.0.weight", "layers.0.bias", "layers.2.weight", "layers.2.bias"),
                                   ("layers.0.weight", "layers.0.bias"), ("x",)], ids=["all", "fc1", "x"])
def test_training_traces_without_data(needs):
    """Forward and backward in one trace (what torch.compile of a training step does): every launch
    in them is an op with a fake implementation, none asks a tensor without data for its pointer."""
    m = GemmGeluMlp(24, 64, 16).bfloat16()
    vals = dict(m.state_dict(), x=torch.randn(2, 20, 24).bfloat16(), r=torch.randn(2, 20, 16).bfloat16())

    def step(vals):
        vals = {k: t.detach().requires_grad_(k in needs) for k, t in vals.items()}
        params = {k: t for k, t in vals.items() if "." in k}
        out = torch.func.functional_call(m, params, (vals["x"], vals["r"]))
        return torch.autograd.grad(out, [vals[k] for k in needs], torch.ones_like(out))

    graph = make_fx(step, tracing_mode="fake")(vals)
    names = [str(n.target) for n in graph.graph.nodes if "strata_hip" in str(n.target)]
    assert "strata_hip.mlp_gelu_train.default" in names and "strata_hip.gemm_bias_act.default" in names
    (outs,) = (n.args[0] for n in graph.graph.nodes if n.op == "output")
    for k, n in zip(needs, outs):
        assert n.meta["val"].shape == vals[k].shape and n.meta["val"].dtype == vals[k].dtype, k


@pytest.mark.parametrize("M,N,K,bias,kernel", [
    (65536, 6144, 1536, True, False), (2048, 1536, 6144, True, False), (1000, 6144, 1536, True, True),
    (65536, 4608, 1536, True, True), (65536, 3584, 3584, True, True), (65536, 3072, 768, True, True),
    (1000, 4096, 1024, False, False), (1000, 4096, 1024, True, True), (256, 4096, 1024, False, True),
    (4096, 2048, 2048, False, False), (4096, 512, 128, False, True), (8192, 2048, 2048, False, True),
    (65536, 6144, 1536, False, False), (1000, 12, 64, True, False)])
def test_weight_gradient_route(monkeypatch, M, N, K, bias, kernel):
    """The weight gradient's kernel runs where it is the faster one, torch's product elsewhere
    (no data: the route alone)."""
    calls = []
    monkeypatch.setattr(ops, "linear_grads", lambda g, x, b: (calls.append("kernel"), (g.t() @ x, g.sum(0)))[1])
    monkeypatch.setattr(ops, "bias_grad", lambda g: g.sum(0))
    g, x = (torch.empty(s, device="meta", dtype=torch.bfloat16) for s in ((M, N), (M, K)))
    dw, db = ops._linear_param_grads(g, x, True, bias)
    assert bool(calls) == kernel
    assert tuple(dw.shape) == (N, K) and (db is not None) == bias
