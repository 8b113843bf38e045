"""The streamed conv's padded instances: float32, and channel counts that do
not fill the tiles, against the fp64 edge sum over the oracle's relation.

Bounds: a sum of L products in binary32, in any order, is off by at most
(L + 1) 2^-24 sum|f w|; a 16-bit result then rounds once (2^-11 or 2^-8 of
its value), and once more after the bias."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from helpers import to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'
HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11,
            torch.bfloat16: 2.0 ** -8}


def _cloud(rows, seed):
    """Distinct voxels on the faces of a box and scattered around it, so
    that rows use one to all of the 27 offsets."""
    rng = np.random.default_rng(seed)
    side = max(3, int(np.ceil((rows / 2) ** (1 / 3))))
    dense = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing='ij'),
                     -1).reshape(-1, 3)[:(rows + 1) // 2]
    far = rng.integers(100, 100 + 4 * side, (8 * rows + 8, 3))
    pts = np.concatenate([dense, np.unique(far, axis=0)])
    pts = np.concatenate([pts[:len(dense)],
                          rng.permutation(pts[len(dense):])])[:rows]
    pts = pts[rng.permutation(len(pts))]
    return np.concatenate([np.zeros((len(pts), 1), np.int64), pts],
                          1).astype(np.int32), rng


def _bound(feats, weight, rel, ref, dtype, c_in, bias):
    mag = O.conv_features_fp64(np.abs(feats), O.mapped_weight(np.abs(weight)),
                               rel)
    terms = 27 * c_in + 1
    out = terms * 2.0 ** -24 * mag
    if dtype != torch.float32 or bias:
        out = out + 2 * HALF_ULP[dtype] * (np.abs(ref) + 0.5 * bias) + 1e-7
    return out + 1e-30


def _check(actual, ref, bound, what):
    err = np.abs(actual - ref)
    assert np.isfinite(actual).all(), what
    assert (err <= bound).all(), (what, float((err / bound).max()))


@pytest.mark.parametrize('dtype,c_in,c_out,rows', [
    (torch.float32, 4, 1, 1),          # one row, one column
    (torch.float32, 20, 33, 63),       # partial chunk; one column past 32
    (torch.float32, 32, 32, 64),       # whole chunk, whole column group
    (torch.float32, 36, 64, 65),       # a row past the 64-row tile
    (torch.float32, 64, 130, 129),     # two column tiles, odd columns
    (torch.float32, 96, 96, 3001),
    (torch.float16, 8, 24, 127),
    (torch.float16, 40, 65, 129),      # columns with no 16-byte rows
    (torch.float16, 96, 96, 3001),
    (torch.bfloat16, 72, 200, 1000),   # two column tiles, the last partial
    (torch.bfloat16, 320, 48, 500),    # five chunks
])
def test_padded_conv_matches_fp64(dtype, c_in, c_out, rows):
    from mlx_lattice_amd import SparseTensor, ops
    from mlx_lattice_amd._native import ext

    coords, rng = _cloud(rows, 3 * c_in + c_out)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    b = torch.as_tensor(rng.standard_normal(c_out)).to(DEV, dtype)
    print(f'padded {dtype} {c_in}->{c_out} rows={rows}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    rel = x.coord_manager.submanifold_kernel_relation(x.coord_key,
                                                      kernel_size=3)
    view = rel.require_sorted_implicit_gemm()
    plain = ext.sparse_conv_features_padded(
        f, ext.conv_padded_fragments(w, 0), 0, c_out,
        view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks, rows,
        27)
    orel = O.kernel_relation(coords, kernel_size=3)
    fd, wd = to_np(f.double()), to_np(w.double())
    ref = O.conv_features_fp64(fd, O.mapped_weight(wd), orel)
    _check(to_np(plain.double()), ref,
           _bound(fd, wd, orel, ref, dtype, c_in, 0.0), 'plain')
    # the operator takes this route (bit for bit), bias and ReLU included;
    # a mapped weight is the same weight
    for weight in (w, w.permute(1, 2, 3, 4, 0).reshape(27, c_in, c_out)):
        y = ops.subm_conv3d(x, weight.contiguous(), kernel_size=3)
        assert torch.equal(y.feats, plain)
    y = ops.subm_conv3d(x, w, b, kernel_size=3, activation='relu')
    assert torch.equal(y.feats, torch.relu(plain + b))
    # a strided view of the features gives the same; rows that do not start
    # at 16 bytes are refused here and run on the CSR route
    wide = torch.cat([f, f], 1)
    assert torch.equal(
        ops.subm_conv3d(x.replace(feats=wide[:, :c_in]), w).feats, plain)
    flat = torch.empty(rows * c_in + 1, dtype=dtype, device=DEV)
    off = flat[1:].view(rows, c_in)
    off.copy_(f)
    assert not ext.conv_padded_supported(off, c_out, 27, rows)
    y = ops.subm_conv3d(x.replace(feats=off), w)
    _check(to_np(y.feats.double()), ref,
           _bound(fd, wd, orel, ref, dtype, c_in, 0.0), 'misaligned')
    torch.cuda.synchronize()


@pytest.mark.parametrize('dtype,bits,c_in,c_out', [
    (torch.float16, 4, 96, 96), (torch.float16, 8, 40, 24),
    (torch.bfloat16, 4, 288, 48), (torch.bfloat16, 8, 64, 96)])
def test_padded_quantized_conv_matches_the_unpacked_weight(dtype, bits, c_in,
                                                           c_out):
    from mlx_lattice_amd import SparseTensor, dequantize_weight, ops
    from mlx_lattice_amd import quantize_weight

    rows = 777
    coords, rng = _cloud(rows, bits + c_in)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    q = quantize_weight(torch.as_tensor(
        rng.standard_normal((c_out, 3, 3, 3, c_in)) / np.sqrt(9 * c_in)).to(
            DEV, dtype), group_size=32, bits=bits)
    print(f'padded int{bits} {dtype} {c_in}->{c_out}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    y = ops.subm_conv3d(x, q, kernel_size=3)
    torch.cuda.synchronize()
    # codes * scale + bias unrounded: the kernel contracts a weight as two
    # fragments, the second holding what the first's rounding leaves
    wd = to_np(dequantize_weight(dataclasses.replace(
        q, scales=q.scales.float(), biases=q.biases.float())).double())
    orel = O.kernel_relation(coords, kernel_size=3)
    fd = to_np(f.double())
    ref = O.conv_features_fp64(fd, O.mapped_weight(wd), orel)
    mag = O.conv_features_fp64(np.abs(fd), O.mapped_weight(np.abs(wd)), orel)
    bound = _bound(fd, wd, orel, ref, dtype, c_in, 0.0)
    _check(to_np(y.feats.double()), ref,
           bound + 4 * HALF_ULP[dtype] ** 2 * mag, f'int{bits}')


@pytest.mark.parametrize('dtype,c_in,c_out,rows', [
    (torch.float32, 48, 72, 33001),    # an order of four 32-row tiles each
    (torch.float32, 16, 32, 33001),    # two 64-row tiles
    (torch.bfloat16, 96, 96, 40001),
    (torch.float16, 24, 40, 66001),    # 128-row tiles of one column tile
    (torch.bfloat16, 72, 200, 33001),  # and of two
])
def test_padded_conv_with_a_tile_order(dtype, c_in, c_out, rows):
    """Enough rows for the longest-first order of the 128-row tiles, the last
    tile ragged: the same bits in any order of the tiles."""
    from mlx_lattice_amd import SparseTensor, ops
    from mlx_lattice_amd._native import ext

    coords, rng = _cloud(rows, c_in + c_out)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    print(f'tile order {dtype} {c_in}->{c_out} rows={rows}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    y = ops.subm_conv3d(x, w, kernel_size=3).feats
    rel = x.coord_manager.submanifold_kernel_relation(x.coord_key)
    view = rel.sorted_implicit_gemm
    order = view.tile_order()
    tiles = (rows + 127) // 128
    assert order is not None
    listed = order.view(torch.int32)[:tiles]
    assert torch.equal(listed.sort().values.cpu(),
                       torch.arange(tiles, dtype=torch.int32))
    # as they come, and shortest first
    for other in (torch.arange(tiles, dtype=torch.int32, device=DEV),
                  listed.flip(0)):
        given = order.clone()
        given.view(torch.int32)[:tiles] = other
        z = ext.sparse_conv_features_padded(
            f, ext.conv_padded_fragments(w, 0), 0, c_out,
            view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
            rows, 27, tile_order=given)
        assert torch.equal(y, z)
    torch.cuda.synchronize()
    orel = O.kernel_relation(coords, kernel_size=3)
    fd, wd = to_np(f.double()), to_np(w.double())
    ref = O.conv_features_fp64(fd, O.mapped_weight(wd), orel)
    _check(to_np(y.double()), ref,
           _bound(fd, wd, orel, ref, dtype, c_in, 0.0), 'tile order')


@pytest.mark.parametrize('dtype,bits,c_out', [
    (torch.float16, 8, 96), (torch.float16, 4, 40), (torch.bfloat16, 8, 48),
    (torch.bfloat16, 4, 96)])
def test_padded_quantized_weight_is_not_rounded(dtype, bits, c_out):
    """Rows with one edge whose features have the sign of what the rounding
    of column 0's weight leaves, so that it adds up over the channels: within
    the bound of two fragments, which a rounded weight exceeds."""
    from mlx_lattice_amd import SparseTensor, dequantize_weight, ops
    from mlx_lattice_amd import quantize_weight

    rows, c_in = 65, 256
    rng = np.random.default_rng(bits + c_out)
    coords = np.zeros((rows, 4), np.int32)
    coords[:, 1] = 4 * rng.permutation(rows)
    q = quantize_weight(torch.as_tensor(
        rng.standard_normal((c_out, 3, 3, 3, c_in)) / 32).to(DEV, dtype),
        group_size=32, bits=bits)
    exact = dequantize_weight(dataclasses.replace(
        q, scales=q.scales.float(), biases=q.biases.float()))
    w = to_np(exact.double()).reshape(c_out, 27, c_in)[:, 13]
    left = w - to_np(exact.to(dtype).double()).reshape(c_out, 27, c_in)[:, 13]
    f = np.sign(left[0]) * 2.0 ** rng.integers(-1, 2, (rows, 1))
    print(f'unrounded int{bits} {dtype} {c_in}->{c_out}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV),
                     torch.as_tensor(f).to(DEV, dtype))
    y = to_np(ops.subm_conv3d(x, q, kernel_size=3).feats.double())
    ref, mag = f @ w.T, np.abs(f) @ np.abs(w).T
    u = HALF_ULP[dtype]
    # a weight's two fragments are off by u^2 of it, or, where the second is
    # a subnormal float16, by half of the smallest one; fp32 sums of the two
    # products of each channel; one rounding of the result
    split = np.maximum(u * u * np.abs(w), 2.0 ** -25
                       if dtype == torch.float16 else 0.0)
    bound = (np.abs(f) @ split.T + (2 * c_in + 1) * 2.0 ** -24 * mag
             + u * np.abs(ref) * (1 + u) + 2.0 ** -25)
    _check(y, ref, bound, f'int{bits}')
    rounded = np.abs(f @ left.T)[:, 0]
    assert (rounded > 2 * bound[:, 0]).all()


@pytest.mark.parametrize('dtype,c_in,c_out', [
    (torch.float32, 64, 64), (torch.float32, 12, 20),
    (torch.bfloat16, 96, 96)])
@pytest.mark.parametrize('op', ['subm', 'down', 'up'])
def test_padded_input_grad_matches_fp64(op, dtype, c_in, c_out):
    """Over the forward view with the mirrored weight (submanifold), and the
    transposed view (strided and transposed convs)."""
    from mlx_lattice_amd import SparseTensor, ops

    rows = 900 if op != 'up' else 150
    coords, rng = _cloud(rows, 7 + c_in)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(
        DEV, dtype).requires_grad_()
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f,
                     stride=2 if op == 'up' else 1)
    print(f'padded input grad {op} {dtype} {c_in}->{c_out}', flush=True)
    if op == 'subm':
        y = ops.subm_conv3d(x, w, kernel_size=3)
        rel = O.kernel_relation(coords, kernel_size=3)
    elif op == 'down':
        y = ops.conv3d(x, w, kernel_size=3, stride=2, padding=1)
        rel = O.kernel_relation(coords, kernel_size=3, stride=2, padding=1)
    else:
        y = ops.conv_transpose3d(x, w, kernel_size=3, stride=2)
        rel = O.transposed_kernel_relation(coords, kernel_size=3, stride=2)
    cot = torch.as_tensor(rng.standard_normal(tuple(y.feats.shape))).to(
        DEV, dtype)
    grad, = torch.autograd.grad(y.feats, f, cot)
    torch.cuda.synchronize()
    e = int(rel['counts'][0])
    i, o, k = (rel[n][:e] for n in ('in_rows', 'out_rows', 'kernel_ids'))
    wk = to_np(w.double()).reshape(c_out, 27, c_in)
    cd = to_np(cot.double())
    ref = np.zeros((rows, c_in))
    mag = np.zeros((rows, c_in))
    for j in range(27):
        at = k == j
        np.add.at(ref, i[at], cd[o[at]] @ wk[:, j])
        np.add.at(mag, i[at], np.abs(cd[o[at]]) @ np.abs(wk[:, j]))
    bound = (27 * c_out + 1) * 2.0 ** -24 * mag + 1e-30
    if dtype != torch.float32:
        bound = bound + 2 * HALF_ULP[dtype] * np.abs(ref) + 1e-7
    _check(to_np(grad.double()), ref, bound, op)


@pytest.mark.parametrize('dtype,c_in,c_out,rows', [
    (torch.float32, 64, 64, 3001),     # whole tiles
    (torch.float32, 32, 64, 700),      # a narrow and a wide tile
    (torch.float32, 4, 16, 65),        # most of a tile is padding
    (torch.float32, 100, 72, 500),     # several tiles, the last partial
    (torch.float32, 5, 3, 64),         # rows of no whole 16-byte piece
    (torch.float32, 33, 64, 1),        # one edge
    (torch.float16, 20, 96, 700),      # 40-byte rows
    (torch.bfloat16, 130, 5, 300),
])
def test_weight_grad_matches_fp64(dtype, c_in, c_out, rows):
    """The matrix-core weight gradient of float32 and of rows that are not
    whole 16-byte pieces; also on features that start off a 16-byte border,
    and with a mapped weight."""
    from mlx_lattice_amd import SparseTensor
    from mlx_lattice_amd.ops._relation_exec import (
        sparse_conv_weight_grad_from_relation,
    )

    coords, rng = _cloud(rows, 11 + c_in)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    cot = torch.as_tensor(rng.standard_normal((rows, c_out))).to(DEV, dtype)
    w = torch.zeros((c_out, 3, 3, 3, c_in), dtype=dtype, device=DEV)
    print(f'weight grad {dtype} {c_in}->{c_out} rows={rows}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    rel = x.coord_manager.submanifold_kernel_relation(x.coord_key,
                                                      kernel_size=3)
    grad = sparse_conv_weight_grad_from_relation(f, cot, w, rel)
    flat = torch.empty(rows * c_in + 1, dtype=dtype, device=DEV)
    off = flat[1:].view(rows, c_in)
    off.copy_(f)
    shifted = sparse_conv_weight_grad_from_relation(off, cot, w, rel)
    mapped = sparse_conv_weight_grad_from_relation(
        f, cot, torch.zeros((27, c_in, c_out), dtype=dtype, device=DEV), rel)
    torch.cuda.synchronize()
    orel = O.kernel_relation(coords, kernel_size=3)
    e = int(orel['counts'][0])
    i, o, k = (orel[n][:e] for n in ('in_rows', 'out_rows', 'kernel_ids'))
    fd, cd = to_np(f.double()), to_np(cot.double())
    ref = np.zeros((27, c_out, c_in))
    mag = np.zeros((27, c_out, c_in))
    for j in range(27):
        at = k == j
        ref[j] = cd[o[at]].T @ fd[i[at]]
        mag[j] = (at.sum() + 1) * 2.0 ** -24 * (
            np.abs(cd[o[at]]).T @ np.abs(fd[i[at]]))
    bound = mag + 1e-30
    if dtype != torch.float32:
        bound = bound + 2 * HALF_ULP[dtype] * np.abs(ref) + 1e-7
    for got, what in ((grad, '5D'), (shifted, 'off a 16-byte border')):
        got = to_np(got.double()).reshape(c_out, 27, c_in).transpose(1, 0, 2)
        _check(got, ref, bound, what)
    _check(to_np(mapped.double()).transpose(0, 2, 1), ref, bound, 'mapped')


@pytest.mark.parametrize('dtype,c_in,c_out,rows,edges', [
    (torch.float32, 4, 16, 32768, True), (torch.float32, 4, 17, 32768, False),
    (torch.float32, 8, 8, 3000, True), (torch.float32, 8, 9, 3000, False),
    (torch.float32, 8, 16, 32769, True), (torch.float32, 4, 32, 32769, True),
    (torch.float32, 8, 32, 32769, False), (torch.float32, 12, 4, 3000, False),
    (torch.float32, 12, 4, 32769, True), (torch.float32, 12, 5, 32769, False),
    (torch.float16, 8, 12, 3000, True), (torch.float16, 8, 16, 3000, False),
])
def test_narrow_convs_of_new_relations_run_over_the_edges(dtype, c_in, c_out,
                                                          rows, edges):
    """At the borders of the rule; either route gives the sum, and a relation
    that holds a sorted view keeps to the padded instances."""
    from mlx_lattice_amd import SparseTensor, ops
    from mlx_lattice_amd._native import ext

    coords, rng = _cloud(rows, c_in + c_out)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    print(f'narrow {dtype} {c_in}->{c_out} rows={rows}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    y = ops.subm_conv3d(x, w, kernel_size=3).feats
    rel = x.coord_manager.submanifold_kernel_relation(x.coord_key)
    assert rel.holds_edges == edges
    dense_map = dtype == torch.float16 and c_out == 16
    viewed = rel._tiled is not None or rel.sorted_implicit_gemm is not None
    assert viewed == (not edges and not dense_map)
    orel = O.kernel_relation(coords, kernel_size=3)
    fd, wd = to_np(f.double()), to_np(w.double())
    ref = O.conv_features_fp64(fd, O.mapped_weight(wd), orel)
    bound = _bound(fd, wd, orel, ref, dtype, c_in, 0.0)
    _check(to_np(y.double()), ref, bound, 'new')
    view = rel.require_sorted_implicit_gemm()
    z = ops.subm_conv3d(x, w, kernel_size=3).feats
    _check(to_np(z.double()), ref, bound, 'sorted')
    if not dense_map:
        assert torch.equal(z, ext.sparse_conv_features_padded(
            f, ext.conv_padded_fragments(w, 0), 0, c_out,
            view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
            rows, 27))
    torch.cuda.synchronize()
