"""Performance cases: the calls a user of this framework times, over their real range.

A case is a dict of plain values.  ``prepare`` makes what a program holds before the
call (inputs, weights, rotary tables) on the GPU, ``run`` is one pass through the
public entry points, ``exact`` the same outputs in float64 from plain torch.

Kinds:

``na3d``       ``strata_amd.natten.na3d`` (the drop-in attention call), or with ``halo`` the
               interior queries of a halo-padded tile (``torch.ops.strata_hip.na3d_fwd``);
               with ``train`` its forward and backward.
``attention``  one attention layer (``FusedNA3DAttention``): qkv, rotary pack, NA3D, gate, proj.
``mlp``        one ``GemmGeluMlp`` with the block's residual.
``block``      one ``StrataBlock``; with ``train`` the input's and every parameter's gradient.
``pixel``      one ``StrataPixelBlock`` conditioned on the semantic tokens.
``step``       one rollout step of ``TwoStageStrata`` on an fp32 state.
``halo``       the cube-sphere halo fill of a state and the crop back.
``step_io``    the step around the network: the dealiased patch embedding of the state and the
               state update from the head's tokens.
"""

import math

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from strata_amd import modules, natten, ops, rope
from strata_amd.model import TwoStageStrata
from strata_amd.pipeline import DealiasedPatchEmbed3D

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _na3d(batch, grid, heads, head_dim, kernel, dilation=1, dtype="bf16", halo=0, train=False):
    return dict(kind="na3d", batch=batch, z=grid[0], y=grid[1], x=grid[2], heads=heads, head_dim=head_dim,
                kz=kernel[0], ky=kernel[1], kx=kernel[2], dilation=dilation, dtype=dtype, halo=halo, train=train)


def _attention(batch, grid, dim, heads, kernel, dilation=1, gated=False, qk_norm=False, depthwise=False, base=10000.0,
               patch=1):
    return dict(kind="attention", batch=batch, z=grid[0], y=grid[1], x=grid[2], dim=dim, heads=heads, kz=kernel[0],
                ky=kernel[1], kx=kernel[2], dilation=dilation, gated=gated, qk_norm=qk_norm, depthwise=depthwise,
                base=base, patch=patch)


def _mlp(batch, grid, dim, hidden):
    return dict(kind="mlp", batch=batch, z=grid[0], y=grid[1], x=grid[2], dim=dim, hidden=hidden)


def _block(batch, grid, dim, heads, kernel, gated=False, qk_norm=False, train=False):
    return dict(kind="block", batch=batch, z=grid[0], y=grid[1], x=grid[2], dim=dim, heads=heads, kz=kernel[0],
                ky=kernel[1], kx=kernel[2], gated=gated, qk_norm=qk_norm, train=train)


def _pixel(batch, grid, dim, heads, kernel, cond_dim, factor):
    return dict(kind="pixel", batch=batch, z=grid[0], y=grid[1], x=grid[2], dim=dim, heads=heads, kz=kernel[0],
                ky=kernel[1], kx=kernel[2], cond_dim=cond_dim, factor=factor)


def _step(batch, grid, channels, dim1, heads1, depth1, k1, dim2, heads2, depth2, k2):
    return dict(kind="step", batch=batch, z=grid[0], y=grid[1], x=grid[2], channels=channels, dim1=dim1, heads1=heads1,
                depth1=depth1, k1=k1, dim2=dim2, heads2=heads2, depth2=depth2, k2=k2)


def _halo(lead, size, pad, dtype):
    return dict(kind="halo", lead=lead, size=size, pad=pad, dtype=dtype)


def _step_io(batch, channels, grid, patch, taps, embed_dim, cell):
    return dict(kind="step_io", batch=batch, channels=channels, z=grid[0], y=grid[1], x=grid[2], patch=patch,
                taps=taps, embed_dim=embed_dim, cell=cell)


def listed():
    return [
        # one small fp32 attention call: a notebook, a unit test, a regression check (latency)
        dict(name="na3d_fp32_small", **_na3d(1, (4, 16, 16), 4, 32, (3, 5, 5), dtype="fp32")),
        # the attention of one halo-padded tile per cube face, interior queries kept
        dict(name="na3d_halo_tiles", **_na3d(6, (16, 144, 144), 16, 64, (3, 13, 13), halo=8)),
        # the attention call in a training step
        dict(name="na3d_train", **_na3d(2, (8, 64, 64), 8, 64, (3, 7, 7), train=True)),
        # the production attention layer on one rollout tile (512 + 2 x 32 at patch 4)
        dict(name="attention_production",
             **_attention(1, (24, 144, 144), 1024, 16, (3, 3, 3), gated=True, qk_norm=True, base=100.0, patch=4)),
        # the MLP of a stage-1 block on an odd regional cut-out (10 125 tokens)
        dict(name="mlp_region", **_mlp(1, (5, 45, 45), 768, 3072)),
        # one block of a small model on a small tile (launches and host work)
        dict(name="block_small", **_block(1, (4, 16, 16), 256, 4, (3, 5, 5))),
        # one block at inference
        dict(name="block", **_block(4, (8, 64, 64), 1024, 16, (3, 7, 7))),
        # one stage-1 block in training, a tile per GPU
        dict(name="block_train", **_block(1, (16, 64, 64), 768, 12, (3, 7, 7), train=True)),
        # one pixel-stage block with its adaLN from the semantic tokens
        dict(name="pixel_block", **_pixel(6, (24, 64, 64), 128, 2, (9, 9, 9), 1024, 4)),
        # one step of the two-stage model on six face tiles
        dict(name="rollout_step", **_step(6, (16, 64, 64), 80, 768, 12, 12, 7, 1024, 16, 12, 9)),
        # the halo fill of a full state and the crop of the result
        dict(name="halo_fill", **_halo(80, 512, 32, "fp32")),
        # the rollout step around the network, with the shift-invariant embedding
        dict(name="step_io", **_step_io(6, 80, (16, 64, 64), 2, 5, 768, 2)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _windows(rng, grid, dilation=1):
    ks = [k for k in ((3, 3, 3), (3, 5, 5), (3, 7, 7), (3, 9, 9), (3, 13, 13), (5, 5, 5), (1, 7, 7))
          if all(a * dilation <= n for a, n in zip(k, grid))]
    return rng.choice(ks) if ks else (1, 1, 1)


def _draw_kind(rng, kind):
    if kind == "na3d":
        train = rng.random() < 0.4
        dtype = "fp32" if rng.random() < 0.25 else "bf16"
        dilation = 2 if rng.random() < 0.2 else 1
        grid = (_log(rng, 2, 24), _log(rng, 9, 144), _log(rng, 9, 144))
        head_dim = rng.choice((32, 64, 64, 64, 128))
        return _na3d(rng.randint(1, 4), grid, rng.randint(1, 16), head_dim, _windows(rng, grid, dilation), dilation,
                     dtype, 0, train)
    if kind == "na3d_halo":
        h = 8
        grid = (_log(rng, 3, 24), 2 * h + _log(rng, 8, 128), 2 * h + _log(rng, 8, 128))
        return _na3d(rng.randint(1, 6), grid, rng.randint(1, 16), 64, rng.choice(((3, 7, 7), (3, 9, 9), (3, 13, 13))),
                     halo=h)
    if kind == "attention":
        heads = rng.randint(2, 16)
        grid = (_log(rng, 4, 32), _log(rng, 9, 144), _log(rng, 9, 144))
        depthwise = rng.random() < 0.25
        dilation = 2 if not depthwise and rng.random() < 0.2 else 1
        return _attention(rng.randint(1, 2), grid, 64 * heads, heads, _windows(rng, grid, dilation), dilation,
                          rng.random() < 0.5, rng.random() < 0.5, depthwise, rng.choice((100.0, 10000.0)),
                          rng.choice((1, 2, 4)))
    if kind == "mlp":
        dim = 8 * _log(rng, 8, 128)
        return _mlp(rng.randint(1, 4), (_log(rng, 1, 24), _log(rng, 8, 144), _log(rng, 8, 144)), dim,
                    rng.choice((2, 4)) * dim)
    if kind == "block":
        heads = rng.randint(2, 16)
        grid = (_log(rng, 3, 16), _log(rng, 9, 96), _log(rng, 9, 96))
        gated = rng.random() < 0.4
        return _block(rng.randint(1, 4), grid, 64 * heads, heads, _windows(rng, grid), gated, rng.random() < 0.4,
                      rng.random() < 0.4)
    if kind == "pixel":
        heads = rng.choice((1, 2, 3, 4))
        factor = rng.choice((2, 4))
        grid = (_log(rng, 4, 24), factor * _log(rng, 4, 20), factor * _log(rng, 4, 20))
        k = min(9, 2 * ((min(grid) - 1) // 2) + 1)
        return _pixel(rng.randint(1, 6), grid, 64 * heads, heads, (k, k, k), 64 * rng.randint(2, 16), factor)
    if kind == "step":
        h1, h2 = rng.randint(2, 12), rng.randint(2, 16)
        grid = (2 * _log(rng, 3, 8), 2 * _log(rng, 9, 32), 2 * _log(rng, 9, 32))
        return _step(rng.randint(1, 6), grid, 8 * rng.randint(2, 10), 64 * h1, h1, rng.randint(1, 4),
                     rng.choice((5, 7)), 64 * h2, h2, rng.randint(1, 4), rng.choice((7, 9)))
    if kind == "halo":
        size = _log(rng, 48, 512)
        return _halo(_log(rng, 1, 80), size, rng.randint(1, min(32, size // 2)), rng.choice(("fp32", "fp32", "bf16")))
    patch = rng.choice((2, 4))
    cell = rng.choice((1, 2))
    grid = (2 * _log(rng, 2, 12), 4 * _log(rng, 3, 36), 4 * _log(rng, 3, 36))
    return _step_io(rng.randint(1, 6), rng.randint(5, 80), grid, patch, rng.choice((3, 4, 5)), 64 * rng.randint(2, 16),
                    cell)


def _cost(case):
    """A pass's rough cost in seconds on this card at a tenth of its rates."""
    w = work(case)
    rate = 5e12 if case.get("dtype") == "fp32" and case["kind"] == "na3d" else 2e14
    return w["flops"] / rate + w["bytes"] / 5e11


def draw(rng):
    kinds = ("na3d", "na3d", "na3d_halo", "attention", "attention", "mlp", "block", "block", "pixel", "step", "halo",
             "step_io")
    while True:
        case = _draw_kind(rng, rng.choice(kinds))
        if _cost(case) <= 0.1:
            return case


# ---------------------------------------------------------------------------
# Inputs and weights
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(shape, g, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _weights(module, g):
    """Xavier-uniform matrices and small biases, bf16, on the GPU."""
    module = module.to("cuda")
    with torch.no_grad():
        for name, p in module.named_parameters():
            if p.dim() == 1:
                p.normal_(0.0, 0.02, generator=g)
            else:
                fan_out, fan_in = p.shape[0], p[0].numel()
                bound = (6.0 / (fan_in + (fan_out if p.dim() == 2 else 0))) ** 0.5
                p.uniform_(-bound, bound, generator=g)
    return module.bfloat16()


def _grid(case):
    return case["z"], case["y"], case["x"]


def _kernel(case):
    return [case["kz"], case["ky"], case["kx"]]


def _tables(case, head_dim, base, patch, seed):
    scale = rope.default_rope_length_scale(patch)
    lat, lon = rope.synthetic_tile_latlon(case["batch"], case["y"], case["x"],
                                          torch.Generator().manual_seed(seed), spacing=scale)
    return rope.stereographic_rope_tables(lat.to("cuda"), lon.to("cuda"), head_dim, base, scale)


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "na3d":
        shape = (case["batch"], *_grid(case), case["heads"], case["head_dim"])
        # per-head scales as trained heads have them: some near uniform, some sharp
        s = (torch.rand(case["heads"], 1, generator=g, device="cuda") * 1.5 + 0.5)
        qkv = [(torch.randn(shape, generator=g, device="cuda") * s).to(_DTYPES[case["dtype"]]) for _ in range(3)]
        state = dict(case=case, qkv=qkv)
        if case["train"]:
            for t in qkv:
                t.requires_grad_(True)
            state["dout"] = _randn(shape, g, _DTYPES[case["dtype"]])
        return state
    if kind in ("attention", "mlp", "block"):
        shape = (case["batch"], *_grid(case), case["dim"])
        x = _randn(shape, g)
        state = dict(case=case, x=x)
        if kind == "mlp":
            state["module"] = _weights(modules.GemmGeluMlp(case["dim"], case["hidden"]), g).eval()
            state["residual"] = _randn(shape, g)
            return state
        d = case["dim"] // case["heads"]
        if kind == "attention":
            state["module"] = _weights(modules.FusedNA3DAttention(
                case["dim"], case["heads"], _kernel(case), case["dilation"], gated=case["gated"],
                qk_norm=case["qk_norm"], depthwise=case["depthwise"]), g).eval()
            state["rope"] = _tables(case, d, case["base"], case["patch"], seed)
            return state
        state["module"] = _weights(modules.StrataBlock(
            case["dim"], case["heads"], _kernel(case), gated=case["gated"], qk_norm=case["qk_norm"]), g)
        state["rope"] = _tables(case, d, 10000.0, 1, seed)
        if case["train"]:
            x.requires_grad_(True)
            state["dout"] = _randn(shape, g)
        else:
            state["module"].eval()
        return state
    if kind == "pixel":
        f = case["factor"]
        m = _weights(modules.StrataPixelBlock(case["dim"], case["heads"], _kernel(case), case["cond_dim"], f,
                                              qk_norm=True), g).eval()
        with torch.no_grad():
            m.adaln_bilinear_dw_proj.bias.normal_(0.0, 0.5, generator=g)
        return dict(case=case, module=m, x=_randn((case["batch"], *_grid(case), case["dim"]), g),
                    cond=_randn((case["batch"], case["z"], case["y"] // f, case["x"] // f, case["cond_dim"]), g))
    if kind == "step":
        with torch.device("cuda"):
            m = TwoStageStrata(case["channels"], case["dim1"], case["heads1"], case["depth1"],
                               (3, case["k1"], case["k1"]), case["dim2"], case["heads2"], case["depth2"],
                               (3, case["k2"], case["k2"]))
        m = _weights(m, g).eval()
        lat, lon = rope.synthetic_tile_latlon(case["batch"], case["y"], case["x"], torch.Generator().manual_seed(seed))
        t1, t2 = m.rope_tables(lat.to("cuda"), lon.to("cuda"))
        return dict(case=case, module=m, rope1=t1, rope2=t2,
                    state=_randn((case["batch"], case["channels"], *_grid(case)), g, torch.float32))
    if kind == "halo":
        n = case["size"]
        return dict(case=case, x=_randn((case["lead"], 6, n, n), g, _DTYPES[case["dtype"]]))
    c, p, e = case["channels"], case["patch"], case["cell"]
    taps = [math.comb(case["taps"] - 1, i) for i in range(case["taps"])]
    embed = _weights(DealiasedPatchEmbed3D(case["z"], case["y"], case["x"], (1, p, p), c, case["embed_dim"], taps),
                     g).eval()
    floor = torch.full((c,), float("nan"), device="cuda")
    floor[c // 2] = 0.0
    return dict(case=case, module=embed, state=_randn((case["batch"], c, *_grid(case)), g, torch.float32),
                pred=_randn((case["batch"], case["z"] // e, case["y"] // e, case["x"] // e, c * e ** 3), g),
                mean=torch.randn(c, generator=g, device="cuda"),
                std=torch.rand(c, generator=g, device="cuda") + 0.5,
                src=torch.arange(c, dtype=torch.int32, device="cuda"), floor=floor)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "na3d":
        q, k, v = state["qkv"]
        if case["halo"]:
            z, h = case["z"], case["halo"]
            return torch.ops.strata_hip.na3d_fwd(q, k, v, _kernel(case), [1, 1, 1], None, [0, h, h],
                                                 [z, case["y"] - 2 * h, case["x"] - 2 * h])
        out = natten.na3d(q, k, v, _kernel(case), dilation=case["dilation"])
        if not case["train"]:
            return out
        return [out.detach(), *torch.autograd.grad(out, (q, k, v), state["dout"])]
    m = state.get("module")
    if kind == "block" and case["train"]:
        x = state["x"]
        out = m(x, state["rope"])
        return [out.detach(), *torch.autograd.grad(out, [x, *m.parameters()], state["dout"])]
    with torch.no_grad():
        if kind in ("attention", "block"):
            return m(state["x"], state["rope"])
        if kind == "mlp":
            return m(state["x"], residual=state["residual"])
        if kind == "pixel":
            return m(state["x"], state["cond"])
        if kind == "step":
            return m.step(state["state"], state["rope1"], state["rope2"])
        if kind == "halo":
            y = ops.cube_pad_faces(state["x"], case["pad"])
            return [y, ops.cube_crop(y, case["pad"])]
        tokens = m(state["state"], state["mean"], state["std"])
        e = case["cell"]
        return [tokens, ops.state_update(state["pred"], state["state"], state["mean"], state["std"], state["src"],
                                         state["floor"], _grid(case), (e, e, e), 1)]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _block_work(tokens, dim, window, gated, weights_only=False):
    flops = 2.0 * tokens * dim * dim * (12 + (1 if gated else 0)) + 4.0 * tokens * window * dim
    weight_bytes = 2.0 * dim * dim * (12 + (1 if gated else 0))
    return flops, weight_bytes


def work(case):
    kind = case["kind"]
    if kind == "halo":
        n, p = case["size"], case["pad"]
        b = 4 if case["dtype"] == "fp32" else 2
        face, padded = n * n, (n + 2 * p) ** 2
        # state in, padded state out; padded state in, state out
        return {"bytes": 2.0 * case["lead"] * 6 * (face + padded) * b, "flops": 0.0}
    tokens = case["batch"] * case["z"] * case["y"] * case["x"]
    if kind == "na3d":
        c = case["heads"] * case["head_dim"]
        h, b = case["halo"], (4 if case["dtype"] == "fp32" else 2)
        queries = case["batch"] * case["z"] * (case["y"] - 2 * h) * (case["x"] - 2 * h)
        flops = 4.0 * queries * case["kz"] * case["ky"] * case["kx"] * c
        size = (2.0 * tokens + 2.0 * queries) * c * b
        if case["train"]:  # backward: scores and dP, then dq, dk, dv; dout in, three gradients out
            return {"bytes": size + 4.0 * tokens * c * b, "flops": 3.5 * flops}
        return {"bytes": size, "flops": flops}
    if kind == "step":
        dims = ((tokens, case["dim1"], case["depth1"], case["k1"]), (tokens // 8, case["dim2"], case["depth2"], case["k2"]))
        flops = 2.0 * tokens * case["dim1"] * case["channels"]  # embedding
        flops += 2.0 * (tokens // 8) * case["dim2"] * 8 * (case["dim1"] + case["channels"])  # merge, head
        size = 8.0 * tokens * case["channels"]
        for t, dim, depth, k in dims:
            f, w = _block_work(t, dim, 3 * k * k, False)
            flops, size = flops + depth * f, size + depth * w
        return {"bytes": size, "flops": flops}
    if kind == "step_io":
        c, p = case["channels"], case["patch"]
        values = tokens * c
        embed = tokens // (p * p) * case["embed_dim"]
        k = c * p * p
        # state in, tokens out; prediction and state in, state out
        return {"bytes": 4.0 * values + 2.0 * embed + 2.0 * k * case["embed_dim"] + (2 + 4 + 4) * float(values),
                "flops": 2.0 * embed * k}
    dim = case["dim"]
    if kind == "mlp":
        return {"bytes": 2.0 * (3 * tokens * dim + 2 * dim * case["hidden"]), "flops": 4.0 * tokens * dim * case["hidden"]}
    window = case["kz"] * case["ky"] * case["kx"]
    if kind == "attention":
        if case["depthwise"]:
            window = case["z"]
        g = 1 if case["gated"] else 0
        return {"bytes": 2.0 * (2 * tokens * dim + (4 + g) * dim * dim),
                "flops": 2.0 * tokens * dim * dim * (4 + g) + 4.0 * tokens * window * dim}
    if kind == "pixel":
        cond = tokens // case["factor"] ** 2 * case["cond_dim"]
        flops, w = _block_work(tokens, dim, window, False)
        flops += 12.0 * tokens * case["cond_dim"] * dim + 18.0 * tokens * case["cond_dim"]
        return {"bytes": 2.0 * (2 * tokens * dim + cond) + w + 12.0 * case["cond_dim"] * dim, "flops": flops}
    flops, w = _block_work(tokens, dim, window, case["gated"])
    size = 4.0 * tokens * dim + w
    if case["train"]:
        na = 4.0 * tokens * window * dim
        return {"bytes": size + 4.0 * tokens * dim + w, "flops": 3.0 * (flops - na) + 3.5 * na}
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times the largest error against ``exact`` that each kind showed."""
    kind = case["kind"]
    if kind == "halo":
        return "exact"  # copies, and the corners' two-value means in the state's own type
    if kind == "na3d":
        if case["dtype"] == "fp32":
            return {"rel": 1e-5}
        return {"rel": 2.4e-2 if case["train"] else 1.6e-2}  # measured 7.1e-3 (gradients), 4.6e-3
    if kind == "block":
        return {"rel": 2.5e-2 if case["train"] else 1.2e-2}  # 7.2e-3 (gradients), 2.8e-3
    if kind == "step":
        return {"rel": 3e-2}  # 8.2e-3: the roundings of 24 blocks
    # attention 5.0e-3, mlp 2.0e-3, pixel 3.3e-3, step_io 2.4e-3
    return {"rel": {"attention": 2e-2, "mlp": 8e-3, "pixel": 1.4e-2, "step_io": 1e-2}[kind]}


# ---------------------------------------------------------------------------
# The same outputs in float64
# ---------------------------------------------------------------------------
def _axis_keys(n, k, d, lo, ext):
    """Key index of each query of [lo, lo + ext) and each of the k window places: [ext, k]."""
    i = torch.arange(lo, lo + ext)
    g = i % d
    sub = (n - g + d - 1) // d
    start = torch.minimum((i // d - k // 2).clamp(min=0), sub - k)
    return ((start[:, None] + torch.arange(k)[None]) * d + g[:, None]).to("cuda")


def _attend(q, kk, vv, band, scale):
    """q [Y, H, X, D]; kk, vv [Y, H, rows * Xk, D]; band [X, rows * Xk]: False outside the window."""
    s = torch.matmul(q, kk.transpose(-1, -2)) * scale
    p = torch.softmax(s.masked_fill(~band, float("-inf")), dim=-1)
    return torch.matmul(p, vv)


def _slice(q, k, v, zk, yk, band, scale):
    """All queries of one z slice [Y, X, H, D] against the key slices zk of k, v [Z, Y, X, H, D]."""
    def rows(t):
        t = t[zk][:, yk]  # [kz, Yq, ky, Xk, H, D]
        return t.permute(1, 4, 0, 2, 3, 5).flatten(2, 4)
    return _attend(q.permute(0, 2, 1, 3), rows(k), rows(v), band, scale).permute(0, 2, 1, 3)


def _na3d64(q, k, v, kernel, dilation=1, halo=0):
    """q, k, v [B, Z, Y, X, H, D] float64; queries without the halo rows and columns."""
    B, Z, Y, X, H, D = q.shape
    d = [dilation] * 3 if isinstance(dilation, int) else dilation
    zi = _axis_keys(Z, kernel[0], d[0], 0, Z)
    yi = _axis_keys(Y, kernel[1], d[1], halo, Y - 2 * halo)
    xi = _axis_keys(X, kernel[2], d[2], halo, X - 2 * halo)
    band = torch.zeros(X - 2 * halo, X, dtype=torch.bool, device="cuda").scatter_(1, xi, True)
    band = band.repeat(1, kernel[0] * kernel[1])
    out = []
    for b in range(B):
        for z in range(Z):
            qz = q[b, z, halo:Y - halo, halo:X - halo]
            args = (qz, k[b], v[b], zi[z], yi, band, D ** -0.5)
            out.append(checkpoint(_slice, *args, use_reentrant=False) if torch.is_grad_enabled() else _slice(*args))
    return torch.stack(out).view(B, Z, Y - 2 * halo, X - 2 * halo, H, D)


def _norm64(t):
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6)


def _rotate64(t, tables):
    cos, sin = (a.double().unsqueeze(-2) for a in tables)
    a, b = t.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)


def _linear64(x, p, name):
    return F.linear(x, p[name + ".weight"], p[name + ".bias"])


def _attention64(x, p, prefix, heads, kernel, tables, dilation=1, qk_norm=False, gated=False):
    qkv = _linear64(x, p, prefix + "qkv").unflatten(-1, (3, heads, -1))
    q, k, v = qkv.unbind(-3)
    if qk_norm:
        q, k = _norm64(q), _norm64(k)
    if tables is not None:
        q, k = _rotate64(q, tables), _rotate64(k, tables)
    a = _na3d64(q, k, v, kernel, dilation).flatten(-2)
    if gated:
        a = a * torch.sigmoid(_linear64(x, p, prefix + "gate_proj"))
    return _linear64(a, p, prefix + "proj")


def _mlp64(x, p, prefix):
    return _linear64(F.gelu(_linear64(x, p, prefix + "layers.0"), approximate="tanh"), p, prefix + "layers.2")


def _ln64(x):
    return F.layer_norm(x, x.shape[-1:], eps=1e-6)


def _block64(x, p, prefix, heads, kernel, tables, qk_norm=False, gated=False):
    x = x + _attention64(_ln64(x), p, prefix + "attn.", heads, kernel, tables, 1, qk_norm, gated)
    return x + _mlp64(_ln64(x), p, prefix + "mlp.")


def _upsampled64(cond, weight, bias, f):
    B, Z, Y, X, C = cond.shape
    t = cond.reshape(B * Z, Y, X, C).permute(0, 3, 1, 2)
    t = F.interpolate(t, scale_factor=f, mode="bilinear", align_corners=False)
    w = weight.reshape(C, 3, 3)
    pad = F.pad(t, (1, 1, 1, 1))
    out = bias.view(1, C, 1, 1).expand_as(t).clone()
    for dy in range(3):
        for dx in range(3):
            out.addcmul_(pad[:, :, dy:dy + Y * f, dx:dx + X * f], w[:, dy, dx].view(1, C, 1, 1))
    return F.gelu(out, approximate="tanh").permute(0, 2, 3, 1).reshape(B, Z, Y * f, X * f, C)


def _dealiased64(x, axis, p, taps):
    """The axis' low-pass in front of the patches: out[i] = sum_t taps[t] x[clamp(p (i // p) - lo + t) + i % p]."""
    n = x.shape[axis]
    i = torch.arange(n, device=x.device)
    lo = (len(taps) - 1) // 2
    out = torch.zeros_like(x)
    for t, w in enumerate(taps):
        out += w * x.index_select(axis, (p * (i // p) - lo + t).clamp(0, n - p) + i % p)
    return out


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "na3d":
        leaves = [t.detach().double() for t in state["qkv"]]
        if not case["train"]:
            with torch.no_grad():
                return _na3d64(*leaves, _kernel(case), case["dilation"], case["halo"])
        for t in leaves:
            t.requires_grad_(True)
        out = _na3d64(*leaves, _kernel(case), case["dilation"])
        return [out.detach(), *torch.autograd.grad(out, leaves, state["dout"].double())]
    if kind == "halo":
        return [None, state["x"]]  # the padded state is copied bytes; the crop undoes the fill
    m = state["module"]
    p = {name: t.detach().double() for name, t in m.named_parameters()}
    if kind == "block" and case["train"]:
        x = state["x"].detach().double().requires_grad_(True)
        for t in p.values():
            t.requires_grad_(True)
        out = _block64(x, p, "", case["heads"], _kernel(case), state["rope"], case["qk_norm"], case["gated"])
        return [out.detach(), *torch.autograd.grad(out, [x, *p.values()], state["dout"].double())]
    with torch.no_grad():
        if kind == "mlp":
            return state["residual"].double() + _mlp64(state["x"].double(), p, "")
        if kind == "attention":
            kernel, dilation = ([case["z"], 1, 1], 1) if case["depthwise"] else (_kernel(case), case["dilation"])
            return _attention64(state["x"].double(), p, "", case["heads"], kernel, state["rope"], dilation,
                                case["qk_norm"], case["gated"])
        if kind == "block":
            return _block64(state["x"].double(), p, "", case["heads"], _kernel(case), state["rope"], case["qk_norm"],
                            case["gated"])
        if kind == "pixel":
            out = []
            for x, cond in zip(state["x"].double().split(1), state["cond"].double().split(1)):
                c = _upsampled64(cond, p["adaln_bilinear_dw_conv.weight"], p["adaln_bilinear_dw_conv.bias"],
                                 case["factor"])
                sh1, sc1, g1, sh2, sc2, g2 = _linear64(c, p, "adaln_bilinear_dw_proj").chunk(6, dim=-1)
                h = _ln64(x) * (1 + sc1) + sh1
                x = x + g1 * _attention64(h, p, "attn.", case["heads"], _kernel(case), None, qk_norm=True)
                out.append(x + g2 * _mlp64(_ln64(x) * (1 + sc2) + sh2, p, "mlp."))
            return torch.cat(out)
        if kind == "step":
            x = state["state"].double()
            h = _linear64(x.permute(0, 2, 3, 4, 1), p, "embed")
            for i in range(case["depth1"]):
                h = _block64(h, p, f"stage1.{i}.", case["heads1"], [3, case["k1"], case["k1"]], state["rope1"])
            B, Z, Y, X, C = h.shape
            h = h.view(B, Z // 2, 2, Y // 2, 2, X // 2, 2, C).permute(0, 1, 3, 5, 2, 4, 6, 7).flatten(4)
            h = _linear64(h, p, "merge")
            for i in range(case["depth2"]):
                h = _block64(h, p, f"stage2.{i}.", case["heads2"], [3, case["k2"], case["k2"]], state["rope2"])
            h = _linear64(_ln64(h), p, "head").view(B, Z // 2, Y // 2, X // 2, 2, 2, 2, -1)
            return x + h.permute(0, 7, 1, 4, 2, 5, 3, 6).reshape(x.shape)
        x = state["state"].double()
        c, pt, e = case["channels"], case["patch"], case["cell"]
        mean, std = (state[n].double().view(1, c, 1, 1, 1) for n in ("mean", "std"))
        taps = [math.comb(case["taps"] - 1, i) / 2.0 ** (case["taps"] - 1) for i in range(case["taps"])]
        t = (x - mean) / std
        for axis in (3, 4):
            t = _dealiased64(t, axis, pt, taps)
        B, _, Z, Y, X = x.shape
        t = t.view(B, c, Z, Y // pt, pt, X // pt, pt).permute(0, 2, 3, 5, 1, 4, 6).flatten(4)
        tokens = F.linear(t, p["proj.weight"].reshape(case["embed_dim"], -1), p["proj.bias"])
        d = state["pred"].double().view(B, Z // e, Y // e, X // e, e, e, e, c).permute(0, 7, 1, 4, 2, 5, 3, 6)
        nxt = x + d.reshape(x.shape) * std + mean
        nxt[:, c // 2].clamp_(min=0.0)
        return [tokens, nxt]
