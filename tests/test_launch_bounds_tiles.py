"""The smaller GEMM tiles, the weight gradient and the rollout step I/O kernels touch exactly
their tensors and write every output once, by a CPU replay of their address arithmetic
(tests/launch_model.py) at the edges of tiles, stages, row ranges and workgroups."""

import pytest

from strata_amd import _lib

from . import launch_model as LM

GEMM_SHAPES = [(1, 8, 8), (63, 64, 64), (65, 72, 72), (127, 128, 136), (129, 136, 520), (300, 8, 64), (1350, 104, 208)]


@pytest.mark.parametrize("tile", list(LM.GEMM_TILES))
@pytest.mark.parametrize("M,N,K", GEMM_SHAPES)
def test_gemm_tile_kernel(tile, M, N, K):
    """Padded row strides, so a read past a row's end would not hide in the next row's start at
    the tensor's last row; every operand used to its last element."""
    ldx, ldw, ldo, ldr = K + 8, K + 16, N + 8, N + 24
    acc, written = LM.gemm_tile_launch(tile, M, N, K, ldx, ldw, ldo, ldr, bias=True, save=True)
    sizes = LM.gemm_sizes(M, N, K, ldx, ldw, ldo, ldr, bias=True, save=True)
    assert acc.check(sizes) == []
    assert (written == 1).all()
    for name in ("x", "w", "out", "out2", "res", "bias"):
        assert acc.lo[name] == 0 and acc.hi[name] == sizes[name], name


def test_gemm_choice_covers_every_tile():
    """The shapes named at the rule take the tile named there."""
    want = {(1024, 256, 1024): "64", (2000, 1024, 4096): "64", (3040, 888, 3552): "128 deep", (10125, 768, 3072): "128",
            (65536, 128, 128): "128", (49152, 1024, 4096): "256", (131072, 4096, 1024): "256", (100, 20, 64): "256"}
    assert {s: LM.gemm_choose(*s) for s in want} == want


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (63, 64, 72), (64, 256, 256), (65, 264, 248), (257, 8, 520), (300, 520, 16),
                                   (1000, 384, 640), (4133, 200, 72), (700, 2056, 1032)])
def test_weight_grad_kernels(M, N, K, bias):
    ldg, ldx = N + 8, K + 16
    acc, ws, written = LM.weight_grad_launch(M, N, K, ldg, ldx, bias)
    assert ws == _lib.load().strata_hip_weight_grad_workspace(M, N, K, int(bias))
    sizes = {"g": LM.span(M, N, ldg), "x": LM.span(M, K, ldx), "out": 2 * N * K, "ws": 4 * ws, "bias_out": 2 * N}
    assert acc.check(sizes) == []
    assert (written == 1).all()
    for name in ("g", "x", "out"):
        assert acc.lo[name] == 0 and acc.hi[name] == sizes[name], name


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("B,C,grid,patch", [(1, 1, (1, 1, 4), (1, 1, 1)), (2, 7, (2, 3, 132), (1, 1, 1)),
                                            (1, 33, (2, 6, 140), (1, 2, 2)), (1, 80, (4, 4, 72), (2, 2, 2)),
                                            (2, 19, (1, 8, 36), (1, 4, 4)), (1, 300, (1, 2, 20), (1, 1, 1)),
                                            (1, 5, (6, 9, 24), (3, 3, 2))])
def test_state_kernels_by_quads(B, C, grid, patch, order):
    acc, sizes = LM.state_quads_launch(B, C, grid, patch, order)
    assert acc.check(sizes) == []
    assert all(acc.lo[n] == 0 and acc.hi[n] == sizes[n] for n in sizes)


@pytest.mark.parametrize("B,C,grid,patch,ny,nx", [
    (1, 3, (1, 2, 4), (1, 2, 2), 3, 3), (2, 5, (2, 6, 36), (1, 2, 2), 5, 5), (1, 37, (1, 10, 132), (1, 2, 2), 4, 5),
    (1, 6, (2, 12, 40), (1, 4, 4), 5, 4), (1, 9, (4, 8, 264), (2, 2, 2), 16, 16), (1, 5, (1, 12, 16), (1, 4, 2), 1, 5),
    (1, 5, (1, 12, 16), (1, 2, 4), 3, 1), (1, 4, (1, 6, 12), (1, 3, 1), 5, 3), (1, 3, (1, 20, 300), (1, 1, 1), 7, 16)])
def test_dealias_patchify(B, C, grid, patch, ny, nx):
    acc, sizes = LM.dealias_patchify_launch(B, C, grid, patch, ny, nx)
    assert acc.check(sizes) == []
    assert all(acc.lo[n] == 0 and acc.hi[n] == sizes[n] for n in sizes)
