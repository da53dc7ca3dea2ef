"""The depth-weighted backward at the sizes where it can go wrong: feature maps
around the 4 x 4 pixels of a block (and the 16 in a row of a map of fewer than
4 rows or columns), depth bins around the 4 in flight, channels around the 64
and 16 that a lane's loads cover, geometry from one cell per column and bin to
a cell of its own for every point.  Held to the rounding bound of an n-term
fp32 sum against float64, |err| <= (n + 2) 2^-24 sum|terms| (n = C for depth, D
for context; a term is rounded at most n + 1 times on its way).  Gradients with
infinities and NaN reach the points of their own cells and no others."""

import pytest
import torch

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
H, W = 12, 20


def geometry(kind, BN, D, fH, fW, g):
    """Cell-centre positions (x, y, z) of a 12 x 20 grid; x = -5 drops a point."""
    shape = (1, BN, D, fH, fW)
    cells = {'column': (1, BN, D, 1, fW), 'runs': (1, BN, D, (fH + 4) // 5, fW),
             'points': shape}[kind]
    cell = torch.randint(0, H * W, cells, generator=g)
    if kind == 'runs':
        cell = cell.repeat_interleave(5, 3)[:, :, :, :fH]
    cell = cell.expand(shape)
    x, y = (cell // W).float() + 0.5, (cell % W).float() + 0.5
    x = torch.where(torch.rand(shape, generator=g) < 0.1, torch.tensor(-5.0), x)
    return torch.stack((x, y, torch.zeros(shape)), -1)


def run(pkg, cuda, kind, D, fH, fW, C, seed, spoil=False):
    g = torch.Generator().manual_seed(seed)
    BN = 2
    geom = geometry(kind, BN, D, fH, fW, g)
    depth = torch.randn(BN, D, fH, fW, generator=g).softmax(1)
    context = torch.randn(BN, C, fH, fW, generator=g)
    up = torch.randn(1, C, H, W, generator=g)
    if spoil:
        up[0, 0, 3, 4], up[0, C - 1, 5, 6], up[0, C // 2, 7, 8] = float('inf'), float('nan'), -float('inf')
    module = pkg.BevPoolTransform((0.0, H, 1.0), (0.0, W, 1.0), (-1.0, 1.0, 2.0)).to(cuda)
    d, c = depth.to(cuda).requires_grad_(True), context.to(cuda).requires_grad_(True)
    out = module.bev_pool_depth(geom.to(cuda), d, c)
    gd, gc = torch.autograd.grad(out, (d, c), up.to(cuda))
    kept = geom[0, ..., 0] >= 0  # (BN, D, fH, fW)
    cell = (geom[0, ..., 0].long() * W + geom[0, ..., 1].long()).clamp_min(0)
    rows = up[0].reshape(C, H * W).t().double()[cell] * kept.unsqueeze(-1)
    rows = torch.where(kept.unsqueeze(-1), rows, torch.zeros((), dtype=torch.float64))
    ctx = context.double().permute(0, 2, 3, 1).unsqueeze(1)  # (BN, 1, fH, fW, C)
    terms = rows * ctx
    want_d, mag_d = terms.sum(-1), terms.abs().sum(-1)
    terms = rows * depth.double().unsqueeze(-1)
    terms = torch.where(kept.unsqueeze(-1), terms, torch.zeros((), dtype=torch.float64))
    want_c, mag_c = terms.sum(1).permute(0, 3, 1, 2), terms.abs().sum(1).permute(0, 3, 1, 2)
    return (gd.cpu().double(), want_d, mag_d, C), (gc.cpu().double(), want_c, mag_c, D)


@pytest.mark.parametrize('kind', ['column', 'runs', 'points'])
@pytest.mark.parametrize('D,fH,fW,C', [
    (1, 1, 4, 4), (15, 15, 5, 16), (16, 16, 8, 20), (17, 17, 7, 32), (33, 31, 6, 36),
    (40, 33, 13, 64), (31, 16, 4, 80), (16, 48, 9, 96), (18, 2, 10, 112), (17, 20, 11, 128),
    (9, 5, 3, 80), (9, 3, 21, 64), (3, 6, 8, 132), (5, 7, 5, 252)])
def test_sizes(pkg, cuda, kind, D, fH, fW, C):
    for got, want, mag, n in run(pkg, cuda, kind, D, fH, fW, C, D + fH + fW + C):
        assert ((got - want).abs() <= (n + 2) * U * mag).all()


@pytest.mark.parametrize('kind', ['column', 'runs', 'points'])
def test_not_finite(pkg, cuda, kind):
    for got, want, mag, n in run(pkg, cuda, kind, 20, 19, 9, 80, 5, spoil=True):
        fin = want.isfinite()
        assert not fin.all()
        assert torch.equal(got.isfinite(), fin)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got[got.isinf()], want[want.isinf()])
        assert ((got - want).abs()[fin] <= (n + 2) * U * mag[fin]).all()


@pytest.mark.parametrize('kind', ['column', 'points'])
@pytest.mark.parametrize('D,fH,fW,C', [
    (5, 70, 1, 8), (9, 70, 2, 80), (6, 41, 3, 64), (7, 5, 6, 80), (4, 5, 9, 36), (5, 8, 22, 80),
    (3, 33, 89, 4), (4, 29, 51, 16), (5, 7, 7, 128),
    (4, 2, 9, 20), (3, 3, 3, 64), (3, 1, 47, 32)])
def test_narrow_maps(pkg, cuda, kind, D, fH, fW, C):
    """Maps that 4 x 4 patches would leave half empty (taken 16 pixels in a
    row of the whole map) and those around what is worth patches."""
    test_sizes(pkg, cuda, kind, D, fH, fW, C)
