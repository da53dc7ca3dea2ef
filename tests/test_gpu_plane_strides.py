"""The transposes on grids of a few cells per plane under any strides of the
sample, channel and height axes: planes in another order, planes that a
gradient shares (an expanded axis, stride 0) and planes that overlap.  Every
cell's own element, bit for bit."""
from __future__ import annotations

import itertools

import pytest
import torch

from oracle import torch_fallback as ref
from test_gpu_op import assert_bit_equal

pytestmark = pytest.mark.gpu


def all_cells(P, cuda, B, D, n_xy):
    """Coordinates and index of one point per cell, in rank order."""
    b, z, y = torch.meshgrid(torch.arange(B), torch.arange(D), torch.arange(n_xy), indexing='ij')
    coords = torch.stack((y * 0, y, z, b), -1).reshape(-1, 4).to(torch.int32)
    return coords, P.index_from_coords(coords.to(cuda), B, D, 1, n_xy)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('n_xy', [1, 2, 3, 4, 5, 7])
def test_gradient_strides(pkg, cuda, n_xy, dtype):
    from bevfusion_triton_amd import _pipeline as P

    C = 9
    for B, D in [(1, 4), (2, 2), (3, 3), (5, 2), (70, 1)]:
        coords, idx = all_cells(P, cuda, B, D, n_xy)
        _, y, z, b = coords.long().unbind(1)
        store = torch.randn(8000, generator=torch.Generator().manual_seed(B + n_xy)).to(dtype)
        grad = store.to(cuda)
        steps = (0, 1, 2, 3, n_xy, n_xy + 1, D * n_xy)
        for sb, sz, sc in itertools.product(steps, steps, (1, n_xy, B * D * n_xy)):
            xg = torch.empty((coords.shape[0], C), dtype=dtype, device=cuda)
            P.backward(idx, grad, C, sb, sc, sz, xg)
            at = (b * sb + z * sz + y).unsqueeze(1) + torch.arange(C) * sc
            assert_bit_equal(xg, store[at], f'{B, D, n_xy} strides {sb, sc, sz}')


@pytest.mark.parametrize('n_xy', [1, 2, 3, 5])
def test_output_strides(pkg, cuda, n_xy):
    """The forward into every order of the sample, height and channel axes;
    half of the cells empty."""
    from bevfusion_triton_amd import _pipeline as P

    C = 5
    for B, D in [(1, 4), (2, 2), (3, 3), (2, 65)]:
        coords, _ = all_cells(P, cuda, B, D, n_xy)
        coords = coords[::2]
        idx = P.index_from_coords(coords.to(cuda), B, D, 1, n_xy)
        feats = torch.randn((coords.shape[0], C), generator=torch.Generator().manual_seed(n_xy))
        want = ref.bev_pool(feats, coords, B, D, 1, n_xy)[:, :, :, 0]  # (B, C, D, n_xy)
        for order in itertools.permutations((0, 1, 2)):
            shape = [(B, C, D)[a] for a in order] + [n_xy]
            out = torch.full(shape, 7.0, device=cuda)
            view = out.permute(order.index(0), order.index(1), order.index(2), 3)
            P.forward(idx, feats.to(cuda), out, view.stride(0), view.stride(1), view.stride(2))
            assert_bit_equal(view, want, f'{B, D, n_xy} order {order}')


def test_expanded_gradient(pkg, cuda):
    """A 1 x 1 grid summed over its height bins: the gradient's planes repeat."""
    B, D, C = 2, 2, 3
    coords = torch.tensor([[0, 0, z, b] for b in range(B) for z in range(D)], dtype=torch.int32)
    f = torch.randn(4, C, device=cuda).requires_grad_(True)
    up = torch.randn(B, C, 1, 1)
    out = pkg.bev_pool(f, coords.to(cuda), B, D, 1, 1).sum(2)
    grad, = torch.autograd.grad(out, f, up.to(cuda))
    assert_bit_equal(grad, up[coords[:, 3].long(), :, 0, 0], 'backward')
