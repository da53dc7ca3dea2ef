"""The grouped forward accumulation at the sizes where it can go wrong: rows
of one 16-byte piece up to two blocks of 64, pieces that overlap, cells
around the points per batch, per group and per long cell in each of its three
regimes, against the CPU oracle.  Forward bit-exact (16-bit: the fp32 sum
rounded once), backward a copy."""
from __future__ import annotations

import pytest
import torch

from oracle import torch_fallback as ref
from test_gpu_op import assert_bit_equal, run_op

pytestmark = pytest.mark.gpu

# points per cell, in rank order (0: an empty cell), around 4/8/16 points a
# batch, 16/64 a group and 64/128/256 a long cell
LENGTHS = [1, 2, 3, 4, 5, 7, 8, 9, 0, 15, 16, 17, 31, 32, 33, 0, 63, 64, 65, 1, 127, 128, 129, 255,
           256, 257, 0, 0, 300, 511, 512, 513, 1, 1500, 64, 64, 128, 256]

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize('C,dtype,N', [
    (3, F32, 9000), (4, F32, 9000), (5, F32, 9000), (12, F32, 9000), (16, F32, 9000),
    (80, F32, 20000), (97, F32, 9000), (100, F32, 9000), (255, F32, 9000), (257, F32, 9000),
    (7, BF16, 9000), (8, F16, 9000), (9, BF16, 9000), (90, F16, 9000), (513, BF16, 9000),
    (256, F32, 70000), (256, F32, 270000),  # 64 points a group, long cells from 128 and 256
])
def test_cell_lengths(pkg, cuda, C, dtype, N):
    g = torch.Generator().manual_seed(C + N)
    H, W = 40, 50
    lengths = torch.tensor(LENGTHS)
    spare = N - int(lengths.sum())
    rank = torch.cat((torch.arange(len(LENGTHS)).repeat_interleave(lengths),
                      torch.randint(len(LENGTHS), H * W, (spare,), generator=g)))
    rank = rank[torch.randperm(N, generator=g)]
    coords = torch.stack((rank // W, rank % W, rank * 0, rank * 0), 1).to(torch.int32)
    feats = torch.randn((N, C), generator=g).to(dtype)
    out, grad, up = run_op(pkg, feats, coords, (1, 1, H, W), cuda)
    assert_bit_equal(out, ref.bev_pool(feats.float(), coords, 1, 1, H, W).to(dtype), 'forward')
    want = up.to(dtype).permute(0, 2, 3, 4, 1).reshape(H * W, C)[rank]
    assert_bit_equal(grad, want, 'backward')


@pytest.mark.parametrize('offset', [1, 2, 3])
@pytest.mark.parametrize('C,dtype', [(80, F32), (64, F16), (33, BF16)])
def test_unaligned_rows(pkg, cuda, C, dtype, offset):
    """Feature rows that start at any element of a wider storage."""
    g = torch.Generator().manual_seed(offset)
    N, H, W = 3001, 13, 11
    store = torch.randn((N, C + 7), generator=g).to(dtype)
    feats = store[:, offset:offset + C]
    coords = torch.stack([torch.randint(0, n, (N,), generator=g) for n in (H, W, 1, 1)], 1)
    out = pkg.bev_pool(store.to(cuda)[:, offset:offset + C], coords.to(cuda), 1, 1, H, W)
    assert_bit_equal(out, ref.bev_pool(feats.float(), coords, 1, 1, H, W).to(dtype), 'forward')


@pytest.mark.parametrize('C', [4, 60, 100, 252, 256])
def test_depth_rows(pkg, cuda, C):
    from bevfusion_triton_amd import synthetic

    case = synthetic.make_case('tiny', features=False)
    B, N, D, fH, fW = case.geom.shape[:5]
    g = torch.Generator().manual_seed(C)
    depth = torch.randn(B * N, D, fH, fW, generator=g).softmax(1)
    context = torch.randn(B * N, C, fH, fW, generator=g)
    dx, bx, nx = ref.gen_dx_bx(case.xbound, case.ybound, case.zbound)
    module = pkg.BevPoolTransform(case.xbound, case.ybound, case.zbound).to(cuda)
    out = module.bev_pool_depth(case.geom.to(cuda), depth.to(cuda), context.to(cuda))
    assert_bit_equal(out, ref.lss_bev_pool_depth(case.geom, depth, context, dx, bx, nx), 'forward')


ROWS = [(3, F32), (4, F32), (5, F32), (7, F16), (8, F16), (9, BF16), (90, F16), (129, F32),
        (130, F32), (257, BF16)]


@pytest.mark.parametrize('grid,C,dtype', [
    (grid, C, dtype) for grid in [(2, 3, 5, 7), (1, 1, 1, 1), (1, 2, 9, 15), (2, 1, 331, 333)]
    for C, dtype in ROWS if grid[2] < 100 or C <= 90])
def test_odd_planes(pkg, cuda, grid, C, dtype):
    """Planes that no vector width divides (4 cells that straddle two planes or
    the grid's end; from 200,000 cells the occupancy is read first), rows that
    none divides, and a gradient whose planes start at any element."""
    B, D, H, W = grid
    g = torch.Generator().manual_seed(C)
    N = 4001
    coords = torch.stack([torch.randint(0, n, (N,), generator=g) for n in (H, W, D, B)], 1)
    feats = torch.randn((N, C), generator=g).to(dtype)
    up = torch.randn((B, C + 1, D, H * W + 3), generator=g).to(dtype)[:, 1:, :, 2:2 + H * W]
    up = up.unflatten(3, (H, W))
    f = feats.to(cuda).requires_grad_(True)
    out = pkg.bev_pool(f, coords.to(cuda), B, D, H, W)
    store = torch.empty((B, C + 1, D, H * W + 3), dtype=dtype, device=cuda)
    view = store[:, 1:, :, 2:2 + H * W].unflatten(3, (H, W))
    view.copy_(up)
    grad, = torch.autograd.grad(out, f, view)
    assert_bit_equal(out, ref.bev_pool(feats.float(), coords, B, D, H, W).to(dtype), 'forward')
    x, y, z, b = coords.unbind(1)
    assert_bit_equal(grad, up[b, :, z, x, y], 'backward')


@pytest.mark.parametrize('grid', [(2, 1, 13, 11), (2, 2, 8, 16)])
@pytest.mark.parametrize('C,dtype', [(1921, F32), (1923, F32), (2049, F32), (1921, F16),
                                     (1927, BF16), (2055, F16)])
def test_wide_rows(pkg, cuda, grid, C, dtype):
    """Rows whose last transpose pass would hold fewer channels than a 16-byte
    piece, every cell occupied (what one cell's row spills into is another's)."""
    B, D, H, W = grid
    cells = B * D * H * W
    g = torch.Generator().manual_seed(C)
    rank = torch.cat((torch.arange(cells), torch.randint(cells, (300,), generator=g)))
    rank = rank[torch.randperm(rank.numel(), generator=g)]
    b, z, x, y = (t for t in torch.unravel_index(rank, grid))
    coords = torch.stack((x, y, z, b), 1).to(torch.int32)
    feats = torch.randn((rank.numel(), C), generator=g).to(dtype)
    out, grad, up = run_op(pkg, feats, coords, grid, cuda)
    assert_bit_equal(out, ref.bev_pool(feats.float(), coords, *grid).to(dtype), 'forward')
    assert_bit_equal(grad, up.to(dtype)[b, :, z, x, y], 'backward')


@pytest.mark.parametrize('C,dtype,N,grid', [
    (68, F32, 30000, (7, 9)), (80, F32, 70000, (40, 50)), (80, F32, 130000, (6, 6)),
    (132, F32, 200000, (20, 30)), (256, F32, 60000, (1, 2)), (260, F32, 90000, (30, 40)),
    (39, F32, 30000, (5, 3)), (130, F16, 60000, (6, 8)), (520, BF16, 40000, (9, 5)),
    (1032, BF16, 20000, (20, 20)), (17, F32, 300000, (30, 30)),
    (80, F32, 147000, (350, 360)), (80, F32, 148000, (350, 360)), (27, F32, 1600000, (360, 360))])
def test_points_per_cell(pkg, cuda, C, dtype, N, grid):
    """Grids from a few points a cell to all of them in two cells: the points
    of a long cell from their floor to the chain's limit, rows of one to four
    blocks of long-cell pieces (the last of one piece or more) and of two and
    three channel blocks; sparse grids on both sides of the line to 64 points a
    group."""
    g = torch.Generator().manual_seed(N + C)
    H, W = grid
    hot = torch.randint(max(1, H * W // 9), (N,), generator=g)
    rank = torch.where(torch.rand(N, generator=g) < 0.3, hot, torch.randint(H * W, (N,), generator=g))
    coords = torch.stack((rank // W, rank % W, rank * 0, rank * 0), 1).to(torch.int32)
    feats = torch.randn((N, C), generator=g).to(dtype)
    out, grad, up = run_op(pkg, feats, coords, (1, 1, H, W), cuda)
    assert_bit_equal(out, ref.bev_pool(feats.float(), coords, 1, 1, H, W).to(dtype), 'forward')
    want = up.to(dtype).permute(0, 2, 3, 4, 1).reshape(H * W, C)[rank]
    assert_bit_equal(grad, want, 'backward')


@pytest.mark.parametrize('C', [16, 20, 28, 32, 92])
@pytest.mark.parametrize('D,fH,fW,half', [(59, 32, 90, 8), (59, 32, 90, 200), (20, 64, 176, 400)])
def test_depth_batches(pkg, cuda, C, D, fH, fW, half):
    """Context rows with enough waves for batches of 8 and 16 points, on dense
    and on sparse grids."""
    g = torch.Generator().manual_seed(C + half)
    shape = (1, 6, D, fH, fW)
    geom = torch.stack([(torch.rand(shape, generator=g) - 0.5) * 2.1 * half * s for s in (1, 1)]
                       + [torch.zeros(shape)], -1)
    depth = torch.randn(6, D, fH, fW, generator=g).softmax(1)
    context = torch.randn(6, C, fH, fW, generator=g)
    bounds = ((-half, half, 1.0), (-half, half, 1.0), (-1.0, 1.0, 2.0))
    module = pkg.BevPoolTransform(*bounds).to(cuda)
    out = module.bev_pool_depth(geom.to(cuda), depth.to(cuda), context.to(cuda))
    want = ref.lss_bev_pool_depth(geom, depth, context, *ref.gen_dx_bx(*bounds))
    assert_bit_equal(out, want, 'forward')


def test_more_rows_than_are_streamed(pkg, cuda):
    """Feature rows of more than 1 GiB take ordinary loads."""
    C, N, H, W = 257, 1_050_000, 60, 70
    g = torch.Generator().manual_seed(5)
    rank = torch.randint(H * W, (N,), generator=g)
    coords = torch.stack((rank // W, rank % W, rank * 0, rank * 0), 1).to(torch.int32)
    feats = torch.randn((N, C), generator=g)
    out = pkg.bev_pool(feats.to(cuda), coords.to(cuda), 1, 1, H, W)
    assert_bit_equal(out, ref.bev_pool(feats, coords, 1, 1, H, W), 'forward')
