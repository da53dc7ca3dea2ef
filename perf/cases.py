"""The calls that this library is measured on: what a program that pools
camera features into a bird's-eye-view grid has it do, through its public
entry points, from the smallest rig to the largest.

A case is a dict of plain values:

  kind      the entry point
              'last'     lss_bev_pool, features stored channel-last
              'first'    lss_bev_pool on the channel-first view that the LSS
                         depth net's product is ('(b n) c d h w -> b n d h w c')
              'depth'    lss_bev_pool_depth (depth and context, no product)
              'cameras'  lss_index_cameras, then lss_bev_pool_depth on it
              'op'       bev_pool(feats, coords, B, D, H, W)
              'legacy'   legacy.QuickCumsumCuda on rows sorted by rank
  grad      True: a training step, forward and the gradients of its inputs;
            False: inference, forward alone
  batch     samples, of six cameras each
  fh, fw    feature map of one camera (the image is 8 times as large)
  focal     focal length in image pixels
  dstep     depth bins from 1 m to dmax in steps of dstep
  half, nx, ny  the grid covers [-half, half) in x with nx cells and, with
            the same cell size, ny cells in y, centred
  nz        height bins: 1 (the whole column, 20 m) or more over [-3, 3) m
  augment   image and lidar augmentation as in training (each image scaled
            and turned, each sample turned), else a level rig
  far       share of the points moved out of the grid
  channels, dtype; coords: type of the op level's coordinates

Inputs come from the seed alone: camera positions and angles differ a little
from seed to seed, as they do from vehicle to vehicle and from one augmented
sample to the next.
"""
from __future__ import annotations

import functools
import importlib
import math

import torch

from __graft_entry__ import load_package

DTYPES = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16,
          'i32': torch.int32, 'i64': torch.int64}

# 1 x 6 cameras of 32 x 88 pixels, 118 depth bins, 360 x 360 cells of 0.3 m
DET = {'kind': 'last', 'grad': True, 'batch': 1, 'fh': 32, 'fw': 88, 'focal': 560.0,
       'dmax': 60.0, 'dstep': 0.5, 'half': 54.0, 'nx': 360, 'ny': 360, 'nz': 1,
       'augment': False, 'far': 0.0, 'channels': 80, 'dtype': 'f32', 'coords': 'i64'}


def _package():
    return load_package()


def _synthetic():
    return importlib.import_module(_package().__name__ + '.synthetic')


def listed():
    cases = [
        # the smallest rig (31,680 points, 16 channels): launches and latency
        dict(DET, name='tiny_step', fh=8, fw=22, focal=140.0, dstep=2.0, nx=90, ny=90,
             channels=16),
        # a detection camera branch, one training step on channel-last
        # features: the headline configuration
        dict(DET, name='det_step'),
        # the segmentation grid, trained on the view that the reference's
        # depth net hands over, with augmentation
        dict(DET, name='seg_first_step', kind='first', half=51.2, nx=256, ny=256, augment=True),
        # a training batch of four on the fused depth (x) context path
        dict(DET, name='train_depth_step', kind='depth', batch=4, augment=True),
        # one frame on a vehicle: index from the calibration, fused pooling
        dict(DET, name='det_cameras_infer', kind='cameras', grad=False),
        # double resolution, two samples, a tenth of the points outside: the largest
        dict(DET, name='hires_step', batch=2, fh=64, fw=176, focal=1120.0, nx=720, ny=720,
             far=0.1),
        # inference with four height bins on the reference's view
        dict(DET, name='z4_first_infer', kind='first', grad=False, nz=4),
        # mixed-precision op level: eight samples' kept points, int64 coords
        dict(DET, name='op_bf16_step', kind='op', batch=8, dtype='bf16'),
        # op level with a channel count and a grid that fit no vector width
        dict(DET, name='op_f16_odd_step', kind='op', batch=3, fh=29, fw=50, focal=350.0,
             dstep=1.0, half=50.25, nx=201, ny=199, channels=90, dtype='f16', coords='i32',
             far=0.05),
        # a small rig whose feature map has an odd number of pixels
        dict(DET, name='odd_depth_step', kind='depth', fh=15, fw=25, focal=180.0, dmax=45.0,
             dstep=1.0, half=50.0, nx=200, ny=200, channels=64),
        # the reference's view again, with an odd map, grid and batch
        dict(DET, name='odd_first_step', kind='first', batch=2, fh=29, fw=51, focal=350.0,
             dmax=45.0, dstep=1.0, half=50.25, nx=201, ny=201, channels=64, augment=True),
        # a program that still calls the legacy function on its sorted rows
        dict(DET, name='legacy_step', kind='legacy', half=51.2, nx=256, ny=256),
    ]
    return cases


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        case = dict(DET)
        case['kind'] = rng.choice(['last', 'first', 'depth', 'cameras', 'op', 'legacy'])
        case['grad'] = rng.random() < 0.7 if case['kind'] != 'cameras' else False
        case['batch'] = log_int(1, 8)
        case['fh'], case['fw'] = log_int(8, 64), log_int(22, 176)
        case['focal'] = 6.4 * case['fw']
        case['dmax'] = rng.choice([45.0, 60.0])
        case['dstep'] = rng.choice([0.5, 0.8, 1.0, 2.0])
        case['half'] = rng.choice([40.0, 50.0, 51.2, 54.0])
        case['nx'] = log_int(90, 720)
        case['ny'] = case['nx'] if rng.random() < 0.5 else max(90, case['nx'] - rng.randint(1, 40))
        case['nz'] = 4 if rng.random() < 0.15 and case['nx'] <= 400 else 1
        case['augment'] = rng.random() < 0.5
        # (a rig given by its cameras has its points where the cameras put them)
        case['far'] = rng.choice([0.0, 0.0, 0.1]) if case['kind'] != 'cameras' else 0.0
        if case['kind'] in ('depth', 'cameras'):
            case['channels'] = 4 * rng.randint(4, 32)
        else:
            case['channels'] = rng.choice([16, 32, 64, 80, 96, 128, rng.randint(16, 128)])
        if case['kind'] == 'op':
            case['dtype'] = rng.choice(['f32', 'f16', 'bf16'])
            case['coords'] = rng.choice(['i32', 'i64'])
        big = dict(DET, batch=2, fh=64, fw=176, nx=720, ny=720)
        if (_points(case) * case['channels'] <= 0.6 * _points(big) * 80
                and _cells(case) * case['channels'] <= _cells(big) * 80):
            return case


# ---- sizes -----------------------------------------------------------------

def _dbound(case):
    return 1.0, case['dmax'], case['dstep']


def _bins(case):
    return torch.arange(*_dbound(case), dtype=torch.float).numel()


def _points(case):
    return case['batch'] * 6 * _bins(case) * case['fh'] * case['fw']


@functools.lru_cache(maxsize=None)
def _grid_key(half, nx, ny, nz):
    """x, y and z bounds, and dx, bx, nx as the package derives them."""
    step = 2.0 * half / nx
    z = (-10.0, 10.0, 20.0) if nz == 1 else (-3.0, 3.0, 6.0 / nz)
    bounds = ((-half, half, step), (-0.5 * ny * step, 0.5 * ny * step, step), z)
    return bounds, _package().gen_dx_bx(*bounds)


def _grid(case):
    return _grid_key(case['half'], case['nx'], case['ny'], case['nz'])


def _cells(case):
    x, y, z = (int(v) for v in _grid(case)[1][2])
    return case['batch'] * x * y * z


# ---- the rig ---------------------------------------------------------------

def _cameras(case, seed):
    """Frustum and camera matrices (on the host): get_geometry's arguments."""
    s = _synthetic()
    spec = s.RigSpec(batch=case['batch'], image=(8 * case['fh'], 8 * case['fw']),
                     feature=(case['fh'], case['fw']), focal=case['focal'],
                     dbound=_dbound(case), yaw_jitter_deg=2.0, trans_jitter_m=0.1)
    return s.camera_inputs(spec, seed=seed, augment=case['augment'])


def _geometry(case, cam, seed, device):
    """(B, 6, D, fH, fW, 3) fp32 points, each operation rounded to fp32: the
    frustum point less post_trans, by post_rots^T, unprojected, by
    combine = rots inv(intrins), plus trans; then the lidar augmentation."""
    def mat(name):
        m = cam[name].to(device)
        return m.reshape(m.shape + (1,) * 3)  # (B, 6, 3[, 3], 1, 1, 1)

    fr = cam['frustum'].to(device)
    pr, pt, tr = mat('post_rots'), mat('post_trans'), mat('camera2lidar_trans')
    inv = torch.linalg.inv(cam['intrins'].double())
    comb = (cam['camera2lidar_rots'].double() @ inv).float().to(device)
    comb = comb.reshape(comb.shape + (1,) * 3)
    a = [fr[..., i] - pt[:, :, i] for i in range(3)]
    b = [(pr[:, :, 0, i] * a[0] + pr[:, :, 1, i] * a[1]) + pr[:, :, 2, i] * a[2]
         for i in range(3)]
    c = [b[0] * b[2], b[1] * b[2], b[2]]
    g = [((comb[:, :, i, 0] * c[0] + comb[:, :, i, 1] * c[1]) + comb[:, :, i, 2] * c[2])
         + tr[:, :, i] for i in range(3)]
    if cam['extra_rots'] is not None:
        er = cam['extra_rots'].to(device).reshape(-1, 3, 3, 1, 1, 1, 1)
        et = cam['extra_trans'].to(device).reshape(-1, 3, 1, 1, 1, 1)
        g = [((er[:, i, 0] * g[0] + er[:, i, 1] * g[1]) + er[:, i, 2] * g[2]) + et[:, i]
             for i in range(3)]
    geom = torch.stack(g, -1)
    if case['far']:
        gen = torch.Generator(device=device).manual_seed(seed + 77)
        away = torch.rand(geom.shape[:-1], generator=gen, device=device) < case['far']
        geom[..., 0] += away * (60.0 + 140.0 * torch.rand(away.shape, generator=gen,
                                                          device=device))
    return geom


def _cell_coords(case, geom):
    """int64 (n, 4) coordinates (x, y, z, b) of all points and the kept mask,
    as the vtransform forms them."""
    dx, bx, nx = (t.to(geom.device) for t in _grid(case)[1])
    b = torch.arange(case['batch'], device=geom.device).repeat_interleave(
        _points(case) // case['batch'])
    q = ((geom.reshape(-1, 3) - (bx - dx / 2.0)) / dx).long()
    kept = ((q >= 0) & (q < nx)).all(1)
    return torch.cat((q, b.unsqueeze(1)), 1), kept


def _ranks(case, coords):
    x, y, z = (int(v) for v in _grid(case)[1][2])
    return ((coords[:, 3] * z + coords[:, 2]) * x + coords[:, 0]) * y + coords[:, 1]


def _op_points(case):
    """Points of an op-level call: nine in ten of those that a rig keeps, the
    same number for every seed."""
    return _kept_key(case)[0] * 9 // 10


def _op_rows(kept, n, gen):
    """n of the kept points, in point order (some twice where too few are kept)."""
    order = torch.randperm(kept.numel(), generator=gen, device=kept.device)
    return kept[order.repeat(-(-n // kept.numel()))[:n].sort().values]


# ---- what a program has in hand before the call ------------------------------

def prepare(case, seed):
    dev = torch.device('cuda')
    pkg = _package()
    bounds, (dx, bx, nx) = _grid(case)
    X, Y, Z = (int(v) for v in nx)
    B, D, fH, fW, C = case['batch'], _bins(case), case['fh'], case['fw'], case['channels']
    cam = _cameras(case, seed)
    gen = torch.Generator(device=dev).manual_seed(seed)
    state = {'kind': case['kind'], 'grad': case['grad'], 'size': (B, Z, X, Y)}
    # softmax over the depth bins, and the context of each pixel
    depth = torch.randn(B * 6, D, fH, fW, generator=gen, device=dev).softmax(1)
    context = torch.randn(B * 6, C, fH, fW, generator=gen, device=dev)
    state['module'] = pkg.BevPoolTransform(*bounds).to(dev)
    if case['kind'] == 'cameras':
        state['cam'] = {k: None if v is None else v.to(dev) for k, v in cam.items()}
    else:
        geom = _geometry(case, cam, seed, dev)
    if case['kind'] in ('depth', 'cameras'):
        if case['kind'] == 'depth':
            state['geom'] = geom
        state['depth'], state['context'] = depth, context
        leaves = [depth, context]
    elif case['kind'] == 'first':
        # (B*N, C, D, fH, fW) storage, handed over as a view
        x = torch.empty(B, 6, C, D, fH, fW, device=dev)
        torch.mul(depth.view(B, 6, 1, D, fH, fW), context.view(B, 6, C, 1, fH, fW), out=x)
        state['geom'], state['x'] = geom, x
        leaves = [x]
    else:
        x = torch.empty(B, 6, D, fH, fW, C, device=dev)
        torch.mul(depth.view(B, 6, D, fH, fW, 1),
                  context.permute(0, 2, 3, 1).reshape(B, 6, 1, fH, fW, C), out=x)
        if case['kind'] == 'last':
            state['geom'], state['x'] = geom, x
        else:
            coords, kept = _cell_coords(case, geom)
            rows = _op_rows(kept.nonzero().view(-1), _op_points(case), gen)
            coords, x = coords[rows], x.view(-1, C)[rows]
            if case['kind'] == 'legacy':  # rows sorted by rank, as the caller sorts them
                ranks, order = _ranks(case, coords).sort(stable=True)
                x, coords = x[order], coords[order]
                state['ranks'] = ranks
            x = x.to(DTYPES[case['dtype']])
            state['x'], state['coords'] = x, coords.to(DTYPES[case['coords']])
        leaves = [x]
    if case['grad']:
        for t in leaves:
            t.requires_grad_(True)
        state['leaves'] = leaves
        shape = {'op': (B, C, Z, X, Y), 'legacy': (B, Z, X, Y, C)}.get(case['kind'],
                                                                      (B, Z * C, X, Y))
        state['g'] = torch.randn(shape, generator=gen, device=dev).to(leaves[0].dtype)
    return state


# ---- one pass --------------------------------------------------------------

def run(state):
    pkg = _package()
    kind, module = state['kind'], state['module']
    if kind == 'last':
        out = module.bev_pool(state['geom'], state['x'])
    elif kind == 'first':
        out = module.bev_pool(state['geom'], state['x'].permute(0, 1, 3, 4, 5, 2))
    elif kind == 'depth':
        out = module.bev_pool_depth(state['geom'], state['depth'], state['context'])
    elif kind == 'cameras':
        index = module.index_cameras(**state['cam'])
        out = module.bev_pool_depth(index, state['depth'], state['context'])
    elif kind == 'op':
        out = pkg.bev_pool(state['x'], state['coords'], *state['size'])
    else:
        out = pkg.legacy.QuickCumsumCuda.apply(state['x'], state['coords'], state['ranks'],
                                               *state['size'])
    if not state['grad']:
        return (out,)
    return (out.detach(),) + torch.autograd.grad(out, state['leaves'], state['g'])


# ---- the least work of one pass ----------------------------------------------

@functools.lru_cache(maxsize=None)
def _kept(key):
    """Kept points and occupied cells (of the first sample times the batch)."""
    case = dict(key)
    one = dict(case, batch=1)
    geom = _geometry(one, _cameras(one, 1), 1, torch.device('cpu'))
    coords, kept = _cell_coords(one, geom)
    ranks = _ranks(one, coords[kept])
    return case['batch'] * int(kept.sum()), case['batch'] * int(ranks.unique().numel())


def _kept_key(case):
    return _kept(tuple(sorted((k, v) for k, v in case.items() if k != 'name')))


def work(case):
    n, cells, C = _points(case), _cells(case), case['channels']
    kept, occ = _kept_key(case)
    if case['kind'] in ('op', 'legacy'):
        kept = _op_points(case)
    es = DTYPES[case['dtype']].itemsize
    pixels = n // _bins(case)
    out = es * C * cells
    if case['kind'] in ('depth', 'cameras'):
        geom = 12 * (n if case['kind'] == 'depth' else n // (6 * case['batch']))
        inputs = 4 * (n + C * pixels)  # depth and context
        total = geom + inputs + out
        flops = 2 * kept * C
        if case['grad']:
            total += 4 * C * occ + 2 * inputs  # gradient rows; inputs again, their gradients
            flops += 4 * kept * C
        return {'bytes': total, 'flops': flops}
    if case['kind'] in ('last', 'first'):
        points, rows = 12 * n, n
    elif case['kind'] == 'op':
        points, rows = 4 * DTYPES[case['coords']].itemsize * kept, kept
    else:
        points, rows = (8 + 4 * DTYPES[case['coords']].itemsize) * kept, kept
    total = points + es * C * kept + out
    if case['grad']:
        total += es * C * (occ + rows)
    return {'bytes': total, 'flops': kept * C}


# ---- how far from the exact sums ----------------------------------------------

def tolerance(case):
    """Four times the largest relative error seen against exact() over the
    listed cases and some dozens of drawn ones: 5e-7 where a cell's thousands
    of points are summed in fp32, 1.7e-3 and 2.1e-4 where the sum is then
    rounded to bfloat16 or half.  Gradients of the features are copies."""
    if case['dtype'] == 'bf16':
        return {'rel': 7e-3}
    if case['dtype'] == 'f16':
        return {'rel': 1e-3}
    return {'rel': 2e-6}


def exact(case, seed):
    """run()'s outputs in 64 bits from plain torch: the cell of each point as
    the vtransform forms it in fp32, then sums in double."""
    state = prepare(dict(case, grad=True), seed)
    dev = state['g'].device
    B, D, fH, fW, C = case['batch'], _bins(case), case['fh'], case['fw'], case['channels']
    _, Z, X, Y = state['size']
    cells, hw = B * Z * X * Y, fH * fW
    if case['kind'] in ('op', 'legacy'):
        rank = _ranks(case, state['coords'].long())
        rows = state['x'].detach()
        g = state['g']
        g = g.permute(0, 2, 3, 4, 1).reshape(cells, C) if case['kind'] == 'op' else g.view(cells, C)
    else:
        # on the host, where every fp32 operation is rounded by IEEE 754
        if case['kind'] == 'cameras':
            geom = _geometry(case, _cameras(case, seed), seed, torch.device('cpu'))
        else:
            geom = state['geom'].cpu()
        coords, kept = _cell_coords(case, geom)
        rank = torch.where(kept, _ranks(case, coords), cells).to(dev)  # dropped: past the cells
        g = state['g'].view(B, Z, C, X, Y).permute(0, 1, 3, 4, 2).reshape(cells, C)
        g = torch.cat((g, g.new_zeros(1, C)))
    total = torch.zeros(cells, C, dtype=torch.float64, device=dev)
    if case['kind'] in ('depth', 'cameras'):
        rank = rank.view(B * 6, D, hw)
        depth = state['depth'].detach().double().view(B * 6, D, hw)
        ctx = state['context'].detach().double().view(B * 6, C, hw).transpose(1, 2)
        gd, gc = torch.empty_like(depth), torch.zeros_like(ctx)
        for d in range(D):
            r, w = rank[:, d].reshape(-1), depth[:, d].unsqueeze(-1)
            inside = (r < cells).nonzero().view(-1)
            total.index_add_(0, r[inside], (w * ctx).reshape(-1, C)[inside])
            gr = g[r].double().view(B * 6, hw, C)
            gd[:, d] = (gr * ctx).sum(-1)
            gc += w * gr
        grads = (gd.view(B * 6, D, fH, fW), gc.transpose(1, 2).reshape(B * 6, C, fH, fW))
    else:
        if case['kind'] in ('last', 'first'):
            rows = state['x'].detach()
        if case['kind'] == 'first':
            rows = rows.permute(0, 1, 3, 4, 5, 2)
        rows = rows.reshape(-1, C)
        for i in range(0, rows.shape[0], 1 << 20):
            r = rank[i:i + (1 << 20)]
            inside = (r < cells).nonzero().view(-1)
            total.index_add_(0, r[inside], rows[i:i + (1 << 20)][inside].double())
        xg = g[rank]
        if case['kind'] == 'first':
            xg = xg.view(B, 6, D, fH, fW, C).permute(0, 1, 5, 2, 3, 4).contiguous()
        elif case['kind'] == 'last':
            xg = xg.view(B, 6, D, fH, fW, C)
        grads = (xg.double(),)
    total = total.view(B, Z, X, Y, C)
    if case['kind'] == 'op':
        out = total.permute(0, 4, 1, 2, 3).contiguous()
    elif case['kind'] == 'legacy':
        out = total
    else:
        out = total.permute(0, 1, 4, 2, 3).reshape(B, Z * C, X, Y)
    return (out,) + grads if case['grad'] else (out,)
