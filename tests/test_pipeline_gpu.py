"""The rollout step's HIP kernels (state normalise + patchify, state update)
and the patch embeddings (plain and dealiased) against the CPU oracle:
bit-exact for the data movement and the fp32/bf16 element math, through the C
ABI; relative L2 <= 1e-2 for the bf16 embedding GEMMs."""

import ctypes

import pytest
import torch

from oracle import pipeline as O
from strata_amd import _lib, ops
from strata_amd.pipeline import DealiasedPatchEmbed3D, PatchEmbed3D, StepNorms

from .conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [  # (B, C, grid, patch)
    (2, 80, (4, 16, 16), (1, 1, 1)),
    (1, 5, (4, 8, 12), (1, 4, 4)),
    (2, 3, (4, 6, 8), (2, 2, 2)),
    (1, 3, (3, 4, 10), (3, 2, 5)),
    (1, 7, (2, 5, 130), (1, 1, 1)),  # odd C*P (2-byte path), x rows over several workgroups
]


def _state(shape, seed, gpu, nonfinite=True):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(shape, generator=g) * 3.0 + 0.5
    if nonfinite:
        x.view(-1)[:: 97] = float("nan")
        x.view(-1)[5 :: 211] = float("inf")
    return x, x.to(gpu)


@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("norm", [False, True])
def test_state_patchify_matches_oracle(gpu, case, norm):
    B, C, grid, patch = case
    x, xg = _state((B, C, *grid), 0, gpu)
    mean = std = None
    if norm:
        g = torch.Generator().manual_seed(1)
        mean = torch.randn(C, generator=g)
        std = O.norm_std(torch.rand(C, generator=g) * 4 + 0.1, 1e-9)
    got = ops.state_patchify(xg, mean.to(gpu) if norm else None, std.to(gpu) if norm else None, patch)
    ref = O.state_patchify(x, mean, std, patch)
    assert got.shape == ref.shape
    assert torch.equal(got.cpu(), ref)


@pytest.mark.parametrize("case", CASES, ids=str)
@pytest.mark.parametrize("order", [0, 1])
def test_state_update_matches_oracle(gpu, case, order):
    B, C, grid, patch = case
    P = patch[0] * patch[1] * patch[2]
    g = torch.Generator().manual_seed(2)
    T = tuple(n // p for n, p in zip(grid, patch))
    pred = (torch.randn(B, *T, C * P, generator=g) * 2).bfloat16()
    state, _ = _state((B, C + 2, *grid), 3, gpu, nonfinite=False)
    mean = torch.randn(C, generator=g)
    std = torch.rand(C, generator=g) * 3 + 0.2
    src = [(c + 2) % (C + 2) if c % 3 else -1 for c in range(C)]
    floor = torch.full((C,), float("nan"))
    floor[C // 2] = 0.25
    got = ops.state_update(pred.to(gpu), state.to(gpu), mean.to(gpu), std.to(gpu),
                           torch.tensor(src, dtype=torch.int32), floor.to(gpu), grid, patch, order)
    ref = O.state_update(pred, state, mean, std, src, floor, grid, patch, order)
    assert torch.equal(got.cpu(), ref)
    # identity tables: next = bf16(pred) + state
    got = ops.state_update(pred.to(gpu), state[:, :C].contiguous().to(gpu), None, None, None, None, grid, patch, order)
    assert torch.equal(got.cpu(), O.state_update(pred, state[:, :C], None, None, None, None, grid, patch, order))


def test_state_update_in_place_through_c_abi(gpu):
    """next may alias the state when every channel adds its own state channel."""
    B, C, grid, patch = 1, 6, (2, 8, 8), (1, 2, 2)
    g = torch.Generator().manual_seed(4)
    pred = (torch.randn(B, 2, 4, 4, C * 4, generator=g)).bfloat16().to(gpu)
    state = torch.randn(B, C, *grid, generator=g).to(gpu)
    ref = O.state_update(pred.cpu(), state.cpu(), None, None, None, None, grid, patch, 0)
    a = _lib.StateUpdateArgs()
    a.pred, a.state, a.next = pred.data_ptr(), state.data_ptr(), state.data_ptr()
    a.batch, a.channels, a.state_channels, a.order = B, C, C, 0
    a.grid[:] = list(grid)
    a.patch[:] = list(patch)
    _lib.call("strata_hip_state_update", a, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(state.cpu(), ref)


@pytest.mark.parametrize("patch,C", [((1, 1, 1), 80), ((1, 4, 4), 5), ((2, 2, 2), 9)])
def test_patch_embed_module_vs_conv3d(gpu, patch, C):
    torch.manual_seed(0)
    emb = PatchEmbed3D(patch, C, 64)
    g = torch.Generator().manual_seed(5)
    x = torch.randn(2, C, 4, 8, 16, generator=g)
    mean, std = torch.randn(C, generator=g), torch.rand(C, generator=g) + 0.5
    xn = O.normalize(x, mean, std).bfloat16().float()
    w = emb.proj.weight.detach().bfloat16().float()
    b = emb.proj.bias.detach().bfloat16().float()
    ref = torch.nn.functional.conv3d(xn, w, b, stride=patch).permute(0, 2, 3, 4, 1)
    with torch.no_grad():
        got = emb.to(gpu)(x.to(gpu), mean.to(gpu), std.to(gpu))
    assert got.shape == ref.shape
    assert rel_l2(got.float().cpu(), ref) <= 1e-2


def test_step_norms_from_running_norm_buffers(gpu):
    C = 4
    g = torch.Generator().manual_seed(6)
    mean, var = torch.randn(C, 1, 1, generator=g), torch.rand(C, 1, 1, generator=g) + 0.1
    n = StepNorms.from_running_norms(mean, var, mean * 2, var * 3, 1e-9, [0, 1, -1, 3], [float("nan")] * 3 + [0.0])
    assert torch.equal(n.in_std, (var.sqrt() + 1e-9).reshape(-1))
    assert n.src_channel.dtype == torch.int32 and n.src_channel.tolist() == [0, 1, -1, 3]
    n2 = n.to(gpu)
    assert n2.tgt_std.is_cuda and torch.equal(n2.tgt_mean.cpu(), (mean * 2).reshape(-1))


DEALIAS_CASES = [  # (B, C, grid, patch, resample_filter)
    (2, 5, (4, 16, 12), (1, 2, 2), (1, 4, 6, 4, 1)),
    (1, 3, (4, 8, 8), (2, 2, 2), (1, 1)),
    (1, 4, (2, 16, 8), (1, 4, 2), (1, 3, 3, 1)),
    (2, 80, (2, 8, 8), (1, 2, 2), (1, 4, 6, 4, 1)),
]


@pytest.mark.parametrize("case", DEALIAS_CASES, ids=str)
@pytest.mark.parametrize("normed", [False, True])
def test_dealiased_patch_embed_vs_oracle(gpu, case, normed):
    """DealiasedPatchEmbed3D (filter passes + patchify + GEMM) against the
    reference's stride-1 conv -> replicate pad -> strided low-pass
    (screamcast/dealias.py:111-143) in float64, on the normalised state
    rounded as the GPU path rounds its weights (bf16)."""
    B, C, grid, patch, filt = case
    torch.manual_seed(0)
    emb = DealiasedPatchEmbed3D(*grid, patch_size=patch, in_chans=C, embed_dim=48, resample_filter=filt)
    g = torch.Generator().manual_seed(8)
    x = torch.randn(B, C, *grid, generator=g) * 2 + 0.5
    mean, std = (torch.randn(C, generator=g), torch.rand(C, generator=g) + 0.5) if normed else (None, None)
    if normed:
        x[0, 0, 0, 0, 0] = float("nan")  # normalised to 0, as RunningNorm2d does
    w = emb.proj.weight.detach().bfloat16().double()
    b = emb.proj.bias.detach().bfloat16().double()
    ref = O.dealiased_patch_embed(O.normalize(x, mean, std), w, b, patch, filt)
    with torch.no_grad():
        got = emb.to(gpu)(x.to(gpu), None if mean is None else mean.to(gpu), None if std is None else std.to(gpu))
    assert got.shape == ref.shape
    assert torch.isfinite(got.float()).all()
    assert rel_l2(got.float().cpu(), ref.float()) <= 1e-2


def test_dealias_axis_pass_vs_fp64(gpu):
    """One filter pass per axis against the clamped-tap sum in float64."""
    g = torch.Generator().manual_seed(12)
    x = torch.randn(2, 3, 6, 10, 12, generator=g)
    taps = [0.0625, 0.25, 0.375, 0.25, 0.0625]
    for axis, p in ((0, 2), (1, 2), (2, 4), (2, 1)):
        got = ops.dealias_axis(x.to(gpu), None, None, axis, p, taps).cpu()
        S = x.shape[2 + axis]
        i = torch.arange(S)
        ref = torch.zeros_like(x, dtype=torch.float64)
        for t, f in enumerate(taps):
            src = (p * (i // p) - 2 + t).clamp(0, S - p) + i % p
            ref += f * x.double().index_select(2 + axis, src)
        assert (got.double() - ref).abs().max() <= 1e-6 * ref.abs().max(), (axis, p)


def test_dealiased_embed_is_state_dict_compatible(gpu):
    """The dealiased embedding loads a PatchEmbed3D checkpoint under strict=True
    (proj.weight / proj.bias; the filter buffer is not persistent), and a
    one-tap filter makes it the plain embedding."""
    plain = PatchEmbed3D((1, 2, 2), 4, 32)
    deal = DealiasedPatchEmbed3D(2, 8, 8, patch_size=(1, 2, 2), in_chans=4, embed_dim=32, resample_filter=(5.0,))
    deal.load_state_dict(plain.state_dict(), strict=True)
    assert "dealias_filter" not in deal.state_dict()
    x = torch.randn(1, 4, 2, 8, 8, generator=torch.Generator().manual_seed(13)).to(gpu)
    with torch.no_grad():
        assert torch.equal(deal.to(gpu)(x), plain.to(gpu)(x))


# (B, C, grid, patch): quads of the state over one, several and a ragged last workgroup, odd
# channel counts (2-byte token pieces), tokens of 1, 2 and 4 columns, more rows than one pass
WIDE_CASES = [(1, 1, (1, 1, 4), (1, 1, 1)), (2, 7, (2, 3, 132), (1, 1, 1)), (1, 33, (2, 6, 140), (1, 2, 2)),
              (1, 80, (4, 4, 72), (2, 2, 2)), (2, 19, (1, 8, 36), (1, 4, 4)), (1, 300, (1, 2, 20), (1, 1, 1))]


@pytest.mark.parametrize("case", WIDE_CASES, ids=str)
@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
def test_state_kernels_by_quads(gpu, case, offset):
    """Patchify and update bit-exact at the wide kernels' edges; a state that is only 4-byte
    aligned takes the element-wise kernels and gives the same bits; the update in place."""
    B, C, grid, patch = case
    x, _ = _state((B, C, *grid), 3, gpu)
    buf = torch.empty(x.numel() + offset, device=gpu)
    xg = buf[offset:].view(x.shape)
    xg.copy_(x)
    g = torch.Generator().manual_seed(4)
    mean, std = torch.randn(C, generator=g), torch.rand(C, generator=g) + 0.5
    got = ops.state_patchify(xg, mean.to(gpu), std.to(gpu), patch)
    assert torch.equal(got.cpu(), O.state_patchify(x, mean, std, patch))
    P = patch[0] * patch[1] * patch[2]
    pred = torch.randn(B, *(n // p for n, p in zip(grid, patch)), C * P, generator=g).bfloat16()
    src = torch.arange(C, dtype=torch.int32)
    src[0] = -1
    floor = torch.full((C,), float("nan"))
    floor[C // 2] = 0.0
    for order in (0, 1):
        args = [t.to(gpu) for t in (mean, std, src, floor)]
        ref = O.state_update(pred, x, mean, std, src.tolist(), floor, grid, patch, order)
        nxt = ops.state_update(pred.to(gpu), xg, *args, grid, patch, order)
        assert torch.equal(nxt.cpu().nan_to_num(7.0), ref.nan_to_num(7.0))
        a = _lib.StateUpdateArgs()  # next aliases state
        inp, pg = xg.clone() if offset == 0 else xg, pred.to(gpu)
        keep = inp.clone()
        a.pred, a.next, a.state = pg.data_ptr(), inp.data_ptr(), inp.data_ptr()
        a.mean, a.std, a.src_channel, a.clamp_min = (t.data_ptr() for t in args)
        a.batch, a.channels, a.state_channels, a.order = B, C, C, order
        a.grid[:], a.patch[:] = grid, patch
        _lib.call("strata_hip_state_update", a, torch.cuda.current_stream().cuda_stream)
        assert torch.equal(inp.nan_to_num(7.0), nxt.nan_to_num(7.0))
        inp.copy_(keep)


@pytest.mark.parametrize("case", [
    (1, 3, (1, 2, 4), (1, 2, 2), (3, 3)),       # every tap clamped
    (2, 5, (2, 6, 36), (1, 2, 2), (5, 5)),
    (1, 37, (1, 10, 132), (1, 2, 2), (4, 5)),   # columns over two workgroups, ragged row runs
    (1, 6, (2, 12, 40), (1, 4, 4), (5, 4)),
    (1, 9, (4, 8, 264), (2, 2, 2), (16, 16)),
    (1, 5, (1, 12, 16), (1, 4, 2), (1, 5)),     # one axis unfiltered
    (1, 5, (1, 12, 16), (1, 2, 4), (3, 1)),
    (1, 4, (1, 6, 12), (1, 3, 1), (5, 3)),      # a patch height that is no power of two
    (1, 4, (1, 6, 18), (1, 2, 2), (5, 5)),      # the three-launch chain: rows not in quads
], ids=str)
@pytest.mark.parametrize("norm", [False, True])
def test_dealias_patchify_equals_the_chain(gpu, case, norm):
    """The fused pass bit for bit against dealias_axis along y, then x, then the patchify,
    non-finite inputs included."""
    B, C, grid, patch, ntaps = case
    _, xg = _state((B, C, *grid), 5, gpu)
    g = torch.Generator().manual_seed(6)
    m, s = (torch.randn(C, generator=g).to(gpu), (torch.rand(C, generator=g) + 0.5).to(gpu)) if norm else (None, None)
    taps = [torch.softmax(torch.randn(n, generator=g), 0).tolist() for n in ntaps]
    got = ops.dealias_patchify(xg, m, s, patch, *taps)
    x = xg
    for axis, t in ((1, taps[0]), (2, taps[1])):
        if len(t) > 1:
            x, m, s = ops.dealias_axis(x, m, s, axis, patch[axis], t), None, None
    assert torch.equal(got, ops.state_patchify(x, m, s, patch))


@pytest.mark.parametrize("patch", [(1, 1, 1), (2, 2, 2), (1, 3, 4)], ids=str)
def test_dealias_patchify_without_filters_is_the_patchify(gpu, patch):
    """One tap on both axes filters nothing: the plain patchify's tokens, a normalised value past
    fp32's range (a vanishing std) kept as the patchify keeps it."""
    _, xg = _state((2, 3, 4, 6, 24), 7, gpu)
    m, s = torch.tensor([0.5, -1.0, 0.0], device=gpu), torch.tensor([0.7, 1e-38, 0.0], device=gpu)
    got = ops.dealias_patchify(xg, m, s, patch, [1.0], [1.0])
    ref = ops.state_patchify(xg, m, s, patch)
    assert torch.isinf(ref).any()
    assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), ref.nan_to_num(7.0, 8.0, 9.0))
