"""Workloads of the sparse-convolution library, one pass each through its
public operators: single layers forward and with their gradients, an int8
encoder, a decoder's upsampling, pooling and the point <-> voxel maps.

A case is a dict of plain values; ``prepare`` makes its inputs on the GPU from
a seed, ``run`` makes one pass, ``exact`` computes the same outputs in float64
with plain torch.  Fields of a layer case:

* ``op``: ``subm`` (submanifold), ``down`` (strided forward conv), ``up``
  (transposed conv, rows are the coarse rows);
* ``dtype``, ``c_in``, ``c_out``, ``kernel``, ``stride``, ``padding``,
  ``dilation``; ``bits``: 0 for a dense weight, 4 or 8 for a packed one;
* ``cloud``: ``uniform`` (voxels drawn from a cube), ``shells`` (surfaces of
  spheres) or ``lidar`` (a ground disc of density 1/r and box surfaces);
  ``order``: ``shuffled`` or ``scan`` (sorted by batch, x, y, z, as a cloud
  deduplicated by a sort comes);
* ``maps``: ``fresh`` (a new cloud: the pass builds the coordinate hash and
  kernel map, as the first layer of a level does) or ``kept`` (a further
  layer of the level, whose kernel map an earlier layer built);
* ``grad``: also the gradients of the features and the weight.
"""

from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE = Path(__file__).resolve().parent.parent / 'mlx-lattice_amd'
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

_DTYPES = {'f32': torch.float32, 'f16': torch.float16, 'bf16': torch.bfloat16}
_ENCODER_WIDTHS = (32, 64, 128, 256)


def _layer(name, op, dtype, c_in, c_out, rows, cloud, *, batches=1, kernel=3,
           stride=1, padding=0, dilation=1, bits=0, order='shuffled',
           maps='fresh', grad=False, bias=False):
    case = {'kind': 'layer', 'op': op, 'dtype': dtype, 'c_in': c_in,
            'c_out': c_out, 'rows': rows, 'cloud': cloud, 'batches': batches,
            'kernel': kernel, 'stride': stride, 'padding': padding,
            'dilation': dilation, 'bits': bits, 'order': order, 'maps': maps,
            'grad': grad, 'bias': bias}
    return {'name': name, **case} if name else case


def listed():
    return [
        # The smallest call: one layer over a small grid in the default
        # dtype, kernel map included; launches and host work dominate.
        _layer('small_f32', 'subm', 'f32', 16, 32, 20000, 'uniform', bias=True),
        # The headline layer: kernel map and matrix-core conv of 400k rows.
        _layer('layer_f16', 'subm', 'f16', 128, 128, 400000, 'shells'),
        # A further layer of a level at a width between the powers of two,
        # with bias and ReLU, over a cloud in scan order.
        _layer('conv_bf16_96', 'subm', 'bf16', 96, 96, 150001, 'lidar',
               batches=2, order='scan', maps='kept', bias=True),
        # An encoder's downsampling layer: new coordinates and their map.
        _layer('down_bf16', 'down', 'bf16', 64, 128, 199884, 'lidar',
               batches=2, kernel=2, stride=2, bias=True),
        # A packed int4 layer of a served model on a kept map.
        _layer('conv_int4', 'subm', 'f16', 64, 64, 200000, 'shells', bits=4,
               maps='kept'),
        # Half-precision training of one layer on a new cloud.
        _layer('train_f16', 'subm', 'f16', 64, 64, 200000, 'shells', grad=True),
        # Training in the default dtype: a layer on a kept map ...
        _layer('train_f32', 'subm', 'f32', 64, 64, 60001, 'lidar',
               order='scan', maps='kept', grad=True),
        # ... and a downsampling layer on a new cloud.
        _layer('train_down_f32', 'down', 'f32', 32, 64, 100003, 'lidar',
               batches=2, kernel=2, stride=2, grad=True),
        # A decoder's upsampling layer: every coarse row expands to eight.
        _layer('up_f16', 'up', 'f16', 128, 128, 124523, 'shells', kernel=2,
               stride=2),
        # A whole served model: an int8 encoder over four scans, maps of all
        # its levels included.
        {'name': 'encoder_int8', 'kind': 'encoder', 'rows': 479627,
         'batches': 4, 'bits': 8},
        # Max pooling and its gradient on a kept relation.
        {'name': 'pool_f32', 'kind': 'pool', 'mode': 'max', 'channels': 64,
         'rows': 400000, 'cloud': 'shells', 'batches': 1, 'kernel': 2,
         'stride': 2, 'order': 'shuffled'},
        # Points to voxels and back with the gradient of the point features
        # (the point branch of a point-voxel network).
        {'name': 'points_f32', 'kind': 'points', 'channels': 64,
         'points': 1000000, 'voxels': 400000},
    ]


def draw(rng):
    """A case of the ranges above; sizes are log-uniform and mostly odd."""
    def rows(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    cloud = rng.choice(('shells', 'lidar', 'shells', 'uniform'))
    batches = rng.choice((1, 1, 2, 4))
    order = rng.choice(('shuffled', 'scan'))
    kind = rng.choice(('subm', 'subm', 'subm', 'stem', 'down', 'down', 'up',
                       'train', 'train', 'pool', 'points', 'encoder'))
    if kind == 'encoder':
        return {'kind': 'encoder', 'rows': rows(8000, 400000),
                'batches': batches, 'bits': rng.choice((4, 8))}
    if kind == 'pool':
        return {'kind': 'pool', 'mode': rng.choice(('max', 'avg', 'sum')),
                'channels': rng.choice((16, 30, 32, 64, 96)),
                'rows': rows(4000, 250000), 'cloud': cloud,
                'batches': batches, 'kernel': rng.choice((2, 2, 3)),
                'stride': 2, 'order': order}
    if kind == 'points':
        points = rows(10000, 900000)
        return {'kind': 'points', 'channels': rng.choice((3, 4, 16, 32, 64)),
                'points': points,
                'voxels': max(2000, int(points * rng.uniform(0.2, 0.6)))}
    dtype = rng.choice(('f16', 'bf16', 'f32'))
    common = {'batches': batches, 'order': order,
              'maps': rng.choice(('fresh', 'kept')),
              'bias': rng.random() < 0.5}
    if kind == 'stem':
        return _layer(None, 'subm', dtype, rng.choice((3, 4, 5, 8)),
                      rng.choice((16, 32)), rows(4000, 200000), cloud,
                      kernel=rng.choice((3, 3, 5)), **common)
    widths = (16, 24, 32, 48, 64, 80, 96, 128)
    c_in, c_out = rng.choice(widths), rng.choice(widths)
    bits = 0
    if kind == 'subm':
        if dtype != 'f32':
            c_in, c_out = rng.choice((c_in, 256)), rng.choice((c_out, 256))
            bits = rng.choice((0, 0, 4, 8))
            if bits:
                c_in = max(32, c_in // 32 * 32)
        if rng.random() < 0.6:
            c_out = c_in
    grad = kind == 'train'
    if grad:
        common['bias'] = False
        if rng.random() < 0.6:
            c_out = c_in
    # No costlier than the listed cases: float32 layers stay under the
    # listed training layer, 16-bit ones under the headline layer.
    budget = 60001 * 64 * 64 if dtype == 'f32' else 400000 * 128 * 128 // 3
    if dtype == 'f32' and not grad:
        budget *= 2
    most = max(3000, min(300000, budget // (c_in * c_out)))
    n = rows(2000, most)
    if kind == 'up':
        if rng.random() < 0.3:
            return _layer(None, 'up', dtype, c_in, c_out, max(1000, n // 8),
                          cloud, kernel=3, stride=2, **common)
        return _layer(None, 'up', dtype, c_in, c_out, max(1000, n // 4),
                      cloud, kernel=2, stride=2, **common)
    if kind == 'down' or (grad and rng.random() < 0.3):
        kernel = rng.choice((2, 2, 3))
        return _layer(None, 'down', dtype, c_in, c_out, n, cloud,
                      kernel=kernel, stride=2, padding=kernel // 3, grad=grad,
                      **common)
    dilation = rng.choice((1, 1, 1, 1, 2))
    return _layer(None, 'subm', dtype, c_in, c_out, n, cloud, bits=bits,
                  dilation=dilation, grad=grad, **common)


# ------------------------------------------------------------------ clouds --


def _device():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


_AXIS = 2048  # axis span of every cloud made here (coordinates are >= 0)


def _keys(coords):
    """Scalar keys of (b, x, y, z) rows; offsets may leave the span by a few
    voxels, which the margin of 16 per axis keeps distinct."""
    c = coords.long() + 16
    span = _AXIS + 32
    return ((c[:, 0] * span + c[:, 1]) * span + c[:, 2]) * span + c[:, 3]


def _distinct(points):
    """Distinct (x, y, z) rows, sorted."""
    keys = torch.unique((points[:, 0] * _AXIS + points[:, 1]) * _AXIS
                        + points[:, 2])
    return torch.stack([keys // (_AXIS * _AXIS), keys // _AXIS % _AXIS,
                        keys % _AXIS], 1)


def _uniform(rows, gen):
    side = max(8, round((rows * 13) ** (1 / 3)))
    pick = torch.randperm(side ** 3, generator=gen, device=gen.device)[:rows]
    return torch.stack([pick // (side * side), pick // side % side,
                        pick % side], 1)


def _shells(rows, gen, seed):
    """Complete one-voxel-thick shells of random spheres, in seeded order
    until ``rows`` distinct voxels are there; the last one is cut."""
    host = np.random.default_rng(seed)
    grid = 512 if rows > 250000 else 256
    high = min(60.0, grid / 6)
    have = torch.zeros((0, 3), dtype=torch.long, device=gen.device)
    while True:
        parts, area = [have], 0.0
        while area < 1.2 * (rows - have.shape[0]) + 500:
            r = host.uniform(8.0, high)
            c = torch.tensor(host.uniform(r + 2, grid - r - 2, 3),
                             device=gen.device)
            lo = (c - r - 1).floor().long()
            axis = torch.arange(int(2 * r) + 4, device=gen.device)
            d = [((axis + lo[a]) + 0.5 - c[a]) ** 2 for a in range(3)]
            dist = (d[0][:, None, None] + d[1][None, :, None]
                    + d[2][None, None, :]).sqrt()
            parts.append(((dist - r).abs() < 0.5).nonzero() + lo)
            area += 4 * math.pi * r * r
        have = _distinct(torch.cat(parts))
        if have.shape[0] >= rows:
            keep = have.shape[0] - rows  # whole shells, one end cut
            return have[keep:]


def _lidar(rows, gen, seed):
    """A 1440 x 1440 x 40 extent: 60% ground (radius uniform, so density
    1/r, three voxels deep), the rest whole surfaces of boxes, one cut."""
    host = np.random.default_rng(seed)
    want = rows - int(rows * 0.6)
    boxes = torch.zeros((0, 3), dtype=torch.long, device=gen.device)
    while boxes.shape[0] < want:
        size = host.integers(10, 81, 3)
        size[2] = min(size[2], 38)
        low = [host.integers(0, e - s) for e, s in zip((1440, 1440, 40), size)]
        axes = [torch.arange(int(s), device=gen.device) for s in size]
        box = torch.cartesian_prod(*axes)
        last = torch.tensor(size - 1, device=gen.device)
        face = ((box == 0) | (box == last)).any(1)
        boxes = torch.cat([boxes, box[face]
                           + torch.tensor(low, device=gen.device)])
    boxes = boxes[:want]
    both = boxes[:0]
    draws = 2 * rows
    while both.shape[0] < rows:
        u = torch.rand((3, draws), generator=gen, device=gen.device)
        r, a = 719 * u[0], 2 * math.pi * u[1]
        ground = torch.stack([(720 + r * a.cos()).floor(),
                              (720 + r * a.sin()).floor(),
                              (3 * u[2]).floor().clamp_max(2)], 1).long()
        # box voxels first, then the ground voxels that no box holds
        both = torch.cat([boxes, ground])
        keys = (both[:, 0] * _AXIS + both[:, 1]) * _AXIS + both[:, 2]
        both = both[_first_seen(keys)[0]]
        draws *= 2
    return both[:rows]


def _first_seen(keys):
    """(first positions of the distinct keys in first-seen order, group of
    every key in that order)."""
    unique, inverse = torch.unique(keys, return_inverse=True)
    first = torch.full((unique.shape[0],), keys.shape[0],
                       dtype=torch.long, device=keys.device)
    first.scatter_reduce_(0, inverse, torch.arange(
        keys.shape[0], device=keys.device), 'amin')
    order = torch.argsort(first)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(order.shape[0], device=keys.device)
    return first[order], rank[inverse]


def _cloud(kind, rows, batches, order, seed):
    """(rows, 4) int32 distinct coordinates (batch, x, y, z)."""
    gen = _generator(seed)
    parts = []
    for b in range(batches):
        n = rows // batches + (1 if b < rows % batches else 0)
        points = (_uniform(n, gen) if kind == 'uniform'
                  else _shells(n, gen, 31 * seed + b) if kind == 'shells'
                  else _lidar(n, gen, 31 * seed + b))
        parts.append(torch.cat([torch.full_like(points[:, :1], b), points], 1))
    coords = torch.cat(parts)
    if order == 'scan':
        coords = coords[torch.argsort(_keys(coords))]
    else:
        coords = coords[torch.randperm(coords.shape[0], generator=gen,
                                       device=gen.device)]
    return coords.to(torch.int32).contiguous()


# ------------------------------------------------------------------ inputs --


def _normal(shape, gen, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device=gen.device)
            * scale).to(dtype)


def _layer_inputs(case, seed):
    """Coordinates, features, dense weight (C_out, Kx, Ky, Kz, C_in), bias
    and the cotangent of the output."""
    dtype, k = _DTYPES[case['dtype']], case['kernel']
    coords = _cloud(case['cloud'], case['rows'], case['batches'],
                    case['order'], seed)
    gen = _generator(seed + 1)
    n, c_in, c_out = coords.shape[0], case['c_in'], case['c_out']
    feats = _normal((n, c_in), gen, dtype)
    weight = _normal((c_out, k, k, k, c_in), gen, dtype,
                     math.sqrt(2.0 / (k ** 3 * c_in)))
    bias = _normal((c_out,), gen, dtype, 0.1) if case['bias'] else None
    out_rows = n * k ** 3 if case['op'] == 'up' else n
    cot = _normal((out_rows, c_out), gen, dtype) if case['grad'] else None
    return coords, feats, weight, bias, cot


def _packed(case, weight):
    from mlx_lattice_amd import quantize_weight

    return quantize_weight(weight, group_size=32, bits=case['bits'])


def _encoder_inputs(case, seed):
    """Coordinates, features and the layers [(op, weight, bias)]."""
    coords = _cloud('lidar', case['rows'], case['batches'], 'shuffled', seed)
    gen = _generator(seed + 1)
    feats = torch.rand((coords.shape[0], 4), generator=gen,
                       device=gen.device).to(torch.float16)
    layers = []

    def add(op, k, c_in, c_out):
        layers.append((op, _normal((c_out, k, k, k, c_in), gen, torch.float16,
                                   math.sqrt(2.0 / (k ** 3 * c_in))),
                       _normal((c_out,), gen, torch.float16, 0.1)))

    add('subm', 3, 4, _ENCODER_WIDTHS[0])
    for c_in, c_out in zip(_ENCODER_WIDTHS[:-1], _ENCODER_WIDTHS[1:]):
        add('down', 2, c_in, c_out)
        add('subm', 3, c_out, c_out)
        add('subm', 3, c_out, c_out)
    return coords, feats, layers


def _encoder_module(op, weight, bias, bits):
    from mlx_lattice_amd import nn

    c_out, k, _, _, c_in = weight.shape
    if op == 'subm':
        dense = nn.SubmConv3d(c_in, c_out, kernel_size=k, device=weight.device,
                              dtype=weight.dtype)
        cls = nn.QuantizedSubmConv3d
    else:
        dense = nn.Conv3d(c_in, c_out, kernel_size=k, stride=2,
                          device=weight.device, dtype=weight.dtype)
        cls = nn.QuantizedConv3d
    dense.weight.data.copy_(weight)
    dense.bias.data.copy_(bias)
    return cls.from_conv(dense, group_size=32, bits=bits)


def _pool_inputs(case, seed):
    coords = _cloud(case['cloud'], case['rows'], case['batches'],
                    case['order'], seed)
    gen = _generator(seed + 1)
    shape = (coords.shape[0], case['channels'])
    return (coords, _normal(shape, gen, torch.float32),
            _normal(shape, gen, torch.float32))


def _points_inputs(case, seed):
    """Points inside the voxels of a shell cloud (unit voxels), their batch
    indices and features, and the cotangent of the sampled features."""
    voxels = _cloud('shells', case['voxels'], 1, 'shuffled', seed)
    gen = _generator(seed + 1)
    n = case['points']
    base = voxels[torch.randint(0, voxels.shape[0], (n,), generator=gen,
                                device=gen.device)]
    points = base[:, 1:].float() + torch.rand((n, 3), generator=gen,
                                              device=gen.device)
    shape = (n, case['channels'])
    return (points.contiguous(), base[:, 0].contiguous(),
            _normal(shape, gen, torch.float32),
            _normal(shape, gen, torch.float32))


def _call(case, x, weight, bias):
    from mlx_lattice_amd import ops

    act = 'relu' if case['bias'] else None
    if case['op'] == 'subm':
        return ops.subm_conv3d(x, weight, bias, kernel_size=case['kernel'],
                               dilation=case['dilation'], activation=act)
    conv = ops.conv3d if case['op'] == 'down' else ops.conv_transpose3d
    return conv(x, weight, bias, kernel_size=case['kernel'],
                stride=case['stride'], padding=case['padding'],
                dilation=case['dilation'], activation=act)


def prepare(case, seed):
    from mlx_lattice_amd import SparseTensor, ops

    state = {'case': case}
    if case['kind'] == 'layer':
        coords, feats, weight, bias, cot = _layer_inputs(case, seed)
        stride = case['stride'] if case['op'] == 'up' else 1
        if case['bits']:
            weight = _packed(case, weight)
        if case['grad']:
            feats.requires_grad_()
            weight.requires_grad_()
        state.update(coords=coords, feats=feats, weight=weight, bias=bias,
                     cot=cot, stride=stride)
        if case['maps'] == 'kept':
            # an earlier layer of the level has run over these coordinates
            state['x'] = SparseTensor(coords, feats, stride=stride)
            run(state)
    elif case['kind'] == 'encoder':
        coords, feats, layers = _encoder_inputs(case, seed)
        state.update(coords=coords, feats=feats, modules=[
            _encoder_module(*layer, case['bits']) for layer in layers])
    elif case['kind'] == 'pool':
        coords, feats, cot = _pool_inputs(case, seed)
        x = SparseTensor(coords, feats.requires_grad_())
        state.update(x=x, cot=cot)
        ops.pool3d(x, mode=case['mode'], kernel_size=case['kernel'],
                   stride=case['stride'])
    else:
        points, batches, feats, cot = _points_inputs(case, seed)
        state.update(points=points, batches=batches,
                     feats=feats.requires_grad_(), cot=cot)
    return state


def run(state):
    from mlx_lattice_amd import SparseTensor, ops

    case = state['case']
    if case['kind'] == 'layer':
        x = state.get('x')
        if x is None:
            x = SparseTensor(state['coords'], state['feats'],
                             stride=state['stride'])
        y = _call(case, x, state['weight'], state['bias'])
        out = {'feats': y.feats}
        if case['op'] != 'subm':
            out['coords'] = y.coords
        if case['grad']:
            grads = torch.autograd.grad(
                y.feats, (state['feats'], state['weight']), state['cot'])
            out['feats'] = y.feats.detach()
            out['grad_feats'], out['grad_weight'] = grads
        return out
    if case['kind'] == 'encoder':
        x = SparseTensor(state['coords'], state['feats'])
        for module in state['modules']:
            x = module(x, activation='relu')
        return {'feats': x.feats, 'coords': x.coords}
    if case['kind'] == 'pool':
        x = state['x']
        y = ops.pool3d(x, mode=case['mode'], kernel_size=case['kernel'],
                       stride=case['stride'])
        grad, = torch.autograd.grad(y.feats, (x.feats,), state['cot'])
        return {'feats': y.feats.detach(), 'grad_feats': grad}
    q = ops.sparse_quantize(state['points'], 1.0,
                            batch_indices=state['batches'])
    voxels = ops.voxelize_with_quantization(q, state['feats'],
                                            reduction='mean')
    sampled = ops.devoxelize(state['points'], voxels, 1.0,
                             batch_indices=state['batches'])
    grad, = torch.autograd.grad(sampled, (state['feats'],), state['cot'])
    return {'coords': q.coords, 'inverse': q.inverse_rows, 'counts': q.counts,
            'voxels': voxels.feats.detach(), 'sampled': sampled.detach(),
            'grad_feats': grad}


# --------------------------------------------------------------- reference --


def _offsets(kernel, dilation):
    """Kernel offsets, x outer and z inner; odd extents are centred."""
    axis = [dilation * (i - (kernel // 2 if kernel % 2 else 0))
            for i in range(kernel)]
    return [(x, y, z) for x in axis for y in axis for z in axis]


class _Lookup:
    """Row of a coordinate, or -1."""

    def __init__(self, coords):
        self.sorted, self.order = torch.sort(_keys(coords))

    def rows(self, coords):
        keys = _keys(coords)
        at = torch.searchsorted(self.sorted, keys).clamp_max(
            self.sorted.shape[0] - 1)
        return torch.where(self.sorted[at] == keys, self.order[at],
                           torch.full_like(at, -1))


def _shift(coords, delta):
    return coords + torch.tensor((0, *delta), device=coords.device)


def _map(op, coords, kernel, stride, padding, dilation):
    """(output coordinates of the active rows, per offset the input row of
    every output row or -1), from the definition of the relations: a strided
    conv's outputs are the floor-divided cells in first-seen order, a
    transposed conv's are coord * stride + offset - padding, one per (row,
    offset) when the stride exceeds the offsets' extent and distinct in
    first-seen order otherwise."""
    offsets = _offsets(kernel, dilation)
    c = coords.long()
    if op == 'subm':
        look = _Lookup(c)
        return c, [look.rows(_shift(c, o)) for o in offsets]
    scale = torch.tensor((1, stride, stride, stride), device=c.device)
    if op == 'down':
        cells = torch.div(c, scale, rounding_mode='floor')
        cells = cells[_first_seen(_keys(cells))[0]]
        look = _Lookup(c)
        return cells, [look.rows(_shift(cells * scale, tuple(
            v - padding for v in o))) for o in offsets]
    n, k = c.shape[0], len(offsets)
    out = torch.stack([_shift(c * scale, tuple(v - padding for v in o))
                       for o in offsets], 1).reshape(n * k, 4)
    if stride > max(o[0] for o in offsets) - min(o[0] for o in offsets):
        first, group = torch.arange(n * k, device=c.device), torch.arange(
            n * k, device=c.device)
    else:
        first, group = _first_seen(_keys(out))
    maps = []
    for j in range(k):
        m = torch.full((first.shape[0],), -1, dtype=torch.long,
                       device=c.device)
        m[group[j::k]] = torch.arange(n, device=c.device)
        maps.append(m)
    return out[first], maps


def _conv(feats, weight, maps, rows, bias, relu):
    """Float64 conv over a map; rows past the active ones hold the bias."""
    c_out = weight.shape[0]
    w = weight.reshape(c_out, -1, weight.shape[4])
    out = torch.zeros((rows, c_out), dtype=torch.float64, device=feats.device)
    for k, m in enumerate(maps):
        o = (m >= 0).nonzero()[:, 0]
        out[o] += feats[m[o]] @ w[:, k].T
    if bias is not None:
        out += bias
    return out.clamp_min(0.0) if relu else out


def _conv_grads(feats, weight, maps, cot):
    c_out = weight.shape[0]
    w = weight.reshape(c_out, -1, weight.shape[4])
    grad_feats = torch.zeros_like(feats)
    grad_weight = torch.zeros_like(w)
    for k, m in enumerate(maps):
        o = (m >= 0).nonzero()[:, 0]
        grad_feats.index_add_(0, m[o], cot[o] @ w[:, k])
        grad_weight[:, k] = cot[o].T @ feats[m[o]]
    return grad_feats, grad_weight.reshape(weight.shape)


def _unpacked(q):
    """The float64 weight scale * code + bias of a packed spatial weight:
    codes LSB first along C_in in 32-bit words (K, words, C_out)."""
    words = q.weight.to(torch.int64) & 0xffffffff
    shifts = torch.arange(0, 32, q.bits, device=words.device)
    codes = (words[:, :, None, :] >> shifts[None, None, :, None]) & (
        2 ** q.bits - 1)
    k, _, _, c_out = codes.shape
    codes = codes.reshape(k, -1, c_out).double()
    group = q.group_size
    w = (codes * q.scales.double().repeat_interleave(group, 1)
         + q.biases.double().repeat_interleave(group, 1))
    w = w[:, :q.in_channels]
    return w.permute(2, 0, 1).reshape(c_out, *q.kernel_size, q.in_channels)


def _padded(coords, rows):
    out = torch.zeros((rows, 4), dtype=torch.int32, device=coords.device)
    out[:coords.shape[0]] = coords
    return out


def _exact_layer(case, seed):
    coords, feats, weight, bias, cot = _layer_inputs(case, seed)
    active, maps = _map(case['op'], coords, case['kernel'], case['stride'],
                        case['padding'], case['dilation'])
    n = coords.shape[0]
    rows = n * case['kernel'] ** 3 if case['op'] == 'up' else n
    f, w = feats.double(), (_unpacked(_packed(case, weight)) if case['bits']
                            else weight.double())
    b = None if bias is None else bias.double()
    out = {'feats': _conv(f, w, maps, rows, b, case['bias'])}
    if case['op'] != 'subm':
        out['coords'] = _padded(active, rows)
    if case['grad']:
        out['grad_feats'], out['grad_weight'] = _conv_grads(f, w, maps,
                                                            cot.double())
    return out


def _exact_encoder(case, seed):
    coords, feats, layers = _encoder_inputs(case, seed)
    rows, active, x = coords.shape[0], coords.long(), feats.double()
    subm = None
    for op, weight, bias in layers:
        k = weight.shape[1]
        w = _unpacked(_packed(case, weight))
        if op == 'down':
            active, maps = _map('down', active, k, 2, 0, 1)
            subm = None
        else:
            if subm is None:
                subm = _map('subm', active, k, 1, 0, 1)[1]
            maps = subm
        x = _conv(x, w, maps, rows, bias.double(), True)
    return {'feats': x, 'coords': _padded(active, rows)}


def _exact_pool(case, seed):
    coords, feats, cot = _pool_inputs(case, seed)
    n, c = feats.shape
    _, maps = _map('down', coords, case['kernel'], case['stride'], 0, 1)
    f, g = feats.double(), cot.double()
    worst = -math.inf if case['mode'] == 'max' else 0.0
    out = torch.full((n, c), worst, dtype=torch.float64, device=f.device)
    degree = torch.zeros((n, 1), dtype=torch.float64, device=f.device)
    ties = torch.zeros((n, c), dtype=torch.float64, device=f.device)
    edges = [((m >= 0).nonzero()[:, 0], m) for m in maps]
    for o, m in edges:
        if case['mode'] == 'max':
            out[o] = torch.maximum(out[o], f[m[o]])
        else:
            out[o] += f[m[o]]
        degree[o] += 1
    if case['mode'] == 'avg':
        out /= degree.clamp_min(1)
    if case['mode'] == 'max':
        for o, m in edges:
            ties[o] += (f[m[o]] == out[o]).double()
    grad = torch.zeros_like(f)
    for o, m in edges:
        if case['mode'] == 'max':
            part = torch.where(f[m[o]] == out[o], g[o] / ties[o],
                               torch.zeros_like(g[o]))
        else:
            part = g[o] / (degree[o] if case['mode'] == 'avg' else 1.0)
        grad.index_add_(0, m[o], part)
    return {'feats': out, 'grad_feats': grad}


def _exact_points(case, seed):
    points, batches, feats, cot = _points_inputs(case, seed)
    n = points.shape[0]
    cells = torch.cat([batches[:, None].long(), points.floor().long()], 1)
    first, inverse = _first_seen(_keys(cells))
    counts = torch.bincount(inverse, minlength=n)
    f = feats.double()
    scale = 1.0 / counts.clamp_min(1).double()[:, None]
    voxels = torch.zeros_like(f).index_add_(0, inverse, f) * scale
    look = _Lookup(cells[first])
    frac = (points - points.floor()).double()
    sampled = torch.zeros_like(f)
    grad_voxels = torch.zeros_like(f)
    for corner in range(8):
        d = ((corner >> 2) & 1, (corner >> 1) & 1, corner & 1)
        w = torch.ones((n,), dtype=torch.float64, device=f.device)
        for a in range(3):
            w = w * (frac[:, a] if d[a] else 1.0 - frac[:, a])
        row = look.rows(_shift(cells, d))
        hit = (row >= 0).nonzero()[:, 0]
        sampled[hit] += voxels[row[hit]] * w[hit, None]
        grad_voxels.index_add_(0, row[hit], cot[hit].double() * w[hit, None])
    grad = (grad_voxels * scale)[inverse]
    return {'coords': _padded(cells[first], n),
            'inverse': inverse.to(torch.int32),
            'counts': counts.to(torch.int32), 'voxels': voxels,
            'sampled': sampled, 'grad_feats': grad}


def exact(case, seed):
    return {'layer': _exact_layer, 'encoder': _exact_encoder,
            'pool': _exact_pool, 'points': _exact_points}[case['kind']](
                case, seed)


# ------------------------------------------------- work and error of a pass --


@functools.lru_cache(maxsize=None)
def _edges(op, cloud, rows, batches, kernel, stride, padding, dilation):
    """Relation edges of the cloud of seed 0 (other seeds' are close)."""
    coords = _cloud(cloud, rows, batches, 'scan', 0)
    _, maps = _map(op, coords, kernel, stride, padding, dilation)
    return int(sum(int((m >= 0).sum()) for m in maps))


def work(case):
    """Inputs read once, outputs written once: coordinates (fresh maps) or
    the map's row index per edge (kept maps), features, weight, output; a
    training pass also reads the cotangent, the features and the weight and
    writes both gradients.  Two operations per edge and channel pair in each
    of the products."""
    if case['kind'] == 'points':
        n, c = case['points'], case['channels']
        # points and batches; inverse, counts, voxel coordinates; point
        # features, voxel features, samples; cotangent and gradient
        return {'bytes': n * 16.0 + n * 24.0 + 5 * n * c * 4.0,
                'flops': n * c * (8 * 4 + 4.0)}
    if case['kind'] == 'pool':
        n, c = case['rows'], case['channels']
        e = _edges('down', case['cloud'], n, case['batches'], case['kernel'],
                   case['stride'], 0, 1)
        return {'bytes': 4.0 * n * c * 4 + 8.0 * e, 'flops': 2.0 * e * c}
    if case['kind'] == 'encoder':
        n, b, flops = case['rows'], case['batches'], 0.0
        coords = _cloud('lidar', n, b, 'scan', 0).long()
        weights = 0.0
        for level, c in enumerate(_ENCODER_WIDTHS):
            below = _ENCODER_WIDTHS[level - 1]
            if level:
                coords, maps = _map('down', coords, 2, 2, 0, 1)
                flops += 2.0 * below * c * sum(int((m >= 0).sum())
                                               for m in maps)
                weights += 8 * below * c
            maps = _map('subm', coords, 3, 1, 0, 1)[1]
            e = sum(int((m >= 0).sum()) for m in maps)
            flops += 2.0 * e * (4 * c if level == 0 else 2 * c * c)
            weights += 27 * (4 * c if level == 0 else 2 * c * c)
        return {'bytes': n * (16 + 8 + 16 + 2.0 * _ENCODER_WIDTHS[-1])
                + weights * case['bits'] / 8, 'flops': flops}
    size = 4 if case['dtype'] == 'f32' else 2
    n, c_in, c_out, k = (case['rows'], case['c_in'], case['c_out'],
                         case['kernel'] ** 3)
    out_rows = n * k if case['op'] == 'up' else n
    e = (n * k if case['op'] == 'up' else
         _edges(case['op'], case['cloud'], n, case['batches'], case['kernel'],
                case['stride'], case['padding'], case['dilation']))
    weight = k * c_in * c_out * (case['bits'] / 8 if case['bits'] else size)
    nbytes = (16.0 * n if case['maps'] == 'fresh' else 4.0 * e)
    if case['op'] != 'subm' and case['maps'] == 'fresh':
        nbytes += 16.0 * out_rows
    nbytes += n * c_in * size + out_rows * c_out * size + weight
    flops = 2.0 * e * c_in * c_out
    if case['grad']:
        nbytes += out_rows * c_out * size + 2 * n * c_in * size + 2 * weight
        flops *= 3
    return {'bytes': nbytes, 'flops': flops}


def tolerance(case):
    """About four times the distance to ``exact`` that the pass shows:
    float32 sums in another order (conv outputs 4e-7, weight gradients over
    1e5 edges 3e-6, pooling and point maps 1e-7), one rounding to float16
    (2e-4, also at the end of the encoder) or bfloat16, with a second one
    after the bias (2.4e-3)."""
    if case['kind'] in ('pool', 'points'):
        return {'rel': 1e-6}
    if case['kind'] == 'encoder':
        return {'rel': 2e-3}
    return {'rel': {'f32': 1e-5, 'f16': 1e-3, 'bf16': 1e-2}[case['dtype']]}
