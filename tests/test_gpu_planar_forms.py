"""Planar (channel-first) features through every form of the transpose and the
planar gradient: planes of odd sizes, tiles and groups shifted back to a
camera's end, channels that no piece divides, one to several channel blocks,
fewer than 4 points or channels, storage that starts at any element, points
that are dropped (their rows are never read) and planes without a kept point.
Forward and backward bit-exact against the CPU oracle."""
from __future__ import annotations

import pytest
import torch

from oracle import torch_fallback as ref
from test_gpu_op import assert_bit_equal

pytestmark = pytest.mark.gpu

GRID = ((0.0, 24.0, 1.0), (0.0, 30.0, 1.0), (0.0, 2.0, 1.0))


def geometry(kind, shape, g):
    """Points at cell centres; x = -5 drops a point."""
    B, N, D, fH, fW = shape
    if kind == 'planes':  # every plane its own few cells
        cell = torch.arange(N * D).view(1, N, D, 1, 1) * 7 % (720 - 7)
        cell = cell + torch.randint(0, 7, shape, generator=g)
    elif kind == 'columns':  # a column one cell, shared by neighbouring bins and cameras
        cell = (torch.arange(D).view(1, 1, D, 1, 1) // 3 * 40 + torch.arange(fW)) % 720
        cell = cell.expand(shape)
    else:  # any point anywhere, 1 in 20 cells dense
        cell = torch.randint(0, 720, shape, generator=g)
        cell = torch.where(torch.rand(shape, generator=g) < 0.3, cell // 20 * 20, cell)
    x, y = (cell // 30).float() + 0.5, (cell % 30).float() + 0.5
    z = (torch.rand(shape, generator=g) < 0.3).float() + 0.5
    drop = torch.rand(shape, generator=g) < 0.1
    if D > 1:
        drop[:, :, D // 2] = True
    return torch.stack((torch.where(drop, torch.tensor(-5.0), x), y, z), -1)


@pytest.mark.parametrize('kind', ['planes', 'columns', 'any'])
@pytest.mark.parametrize('B,N,D,fH,fW,C', [
    (1, 2, 30, 32, 88, 8), (2, 1, 25, 29, 51, 67), (1, 3, 40, 15, 25, 130), (1, 2, 7, 53, 71, 97),
    (1, 1, 700, 9, 37, 21), (1, 2, 5, 5, 5, 129), (1, 2, 3, 3, 14, 260), (2, 3, 1, 1, 127, 5),
    (1, 2, 1, 1, 129, 4), (1, 2, 1, 3, 43, 6), (1, 3, 1, 1, 5, 9), (1, 3, 1, 2, 2, 4),
    (1, 2, 1, 1, 3, 8), (1, 2, 6, 7, 9, 3), (1, 2, 6, 7, 9, 2),
])
def test_planar_forward(pkg, cuda, kind, B, N, D, fH, fW, C):
    g = torch.Generator().manual_seed(D + C)
    geom = geometry(kind, (B, N, D, fH, fW), g)
    store = torch.randn(B * N, C + 1, D, fH, fW, generator=g)  # a slice of wider storage
    dx, bx, nx = ref.gen_dx_bx(*GRID)
    module = pkg.BevPoolTransform(*GRID).to(cuda)

    def view(t):
        return t[:, 1:].unflatten(0, (B, N)).permute(0, 1, 3, 4, 5, 2)

    xs = store.to(cuda).requires_grad_(True)
    out = module.bev_pool(geom.to(cuda), view(xs))
    want = ref.lss_bev_pool(geom, view(store), dx, bx, nx)
    assert_bit_equal(out, want, 'forward')
    up = torch.randn(out.shape, generator=g)
    grad, = torch.autograd.grad(out, xs, up.to(cuda))
    xc = store.clone().requires_grad_(True)
    want, = torch.autograd.grad(ref.lss_bev_pool(geom, view(xc), dx, bx, nx), xc, up)
    assert_bit_equal(grad, want, 'backward')


@pytest.mark.parametrize('C', [3969, 3971, 4097])
def test_planar_wide_rows(pkg, cuda, C):
    """Channel counts whose last block would hold fewer than 4 channels (and
    whose last transpose pass fewer than a 16-byte piece)."""
    test_planar_forward(pkg, cuda, 'any', 1, 2, 3, 5, 9, C)


@pytest.mark.parametrize('S', [4, 5, 8, 11, 12, 13, 24, 25, 100])
@pytest.mark.parametrize('C', [4, 16, 33, 36, 80])
def test_planar_small_planes(pkg, cuda, S, C):
    """Many planes of a few points, by elements and by tiles."""
    from bevfusion_triton_amd import _pipeline as P

    src = torch.randn(300, C, S, generator=torch.Generator().manual_seed(S + C))
    rows = P.planar_rows(src.to(cuda))
    assert_bit_equal(rows, src.transpose(1, 2).reshape(-1, C), 'rows')


def test_planar_most_planes(pkg, cuda):
    """More planes of 5 points than a launch has blocks (2^24 of 256 threads)."""
    from bevfusion_triton_amd import _pipeline as P

    src = torch.arange(((1 << 24) + 9) * 25, dtype=torch.int32, device=cuda).view(torch.float32)
    src = src.view(-1, 5, 5)
    rows = P.planar_rows(src)
    want = src.transpose(1, 2).reshape(-1, 5)
    assert torch.equal(rows.view(torch.int32), want.view(torch.int32))
