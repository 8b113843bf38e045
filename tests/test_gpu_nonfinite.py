"""Infinities and NaN in the padded streamed conv: an output is the sum over
its own edges, whatever the weight of an offset that the row has no neighbour
at holds, as on the edge kernel.  Against the fp64 edge sum over the oracle's
relation: the same NaN and infinities, and the finite values within the bound
of a float32 sum."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from helpers import to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'
INF, NAN = float('inf'), float('nan')
HALF_ULP = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11,
            torch.bfloat16: 2.0 ** -8}


def _cloud(rows, rng):
    flat = rng.choice(14 ** 3, rows, replace=False)
    return np.stack([np.zeros_like(flat), flat // 196, flat // 14 % 14,
                     flat % 14], 1).astype(np.int32)


def _edge_sum(feats, weight, rel, rows):
    """(rows, C_out) over weight (K, C_in, C_out) and the sum of the
    magnitudes, float64, edge by edge: nothing is multiplied by a zero that
    stands for a missing neighbour."""
    e = int(rel['counts'][0])
    out = np.zeros((rows, weight.shape[2]))
    mag = np.zeros_like(out)
    with np.errstate(invalid='ignore', over='ignore'):
        for i, o, k in zip(rel['in_rows'][:e], rel['out_rows'][:e],
                           rel['kernel_ids'][:e]):
            out[o] += feats[i] @ weight[k]
            mag[o] += np.abs(feats[i]) @ np.abs(weight[k])
    return out, mag


def _check(got, ref, mag, terms, dtype):
    got = to_np(got.double())
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(ref))
    at = np.isinf(ref)
    np.testing.assert_array_equal(got[at], ref[at])
    at = np.isfinite(ref)
    bound = (terms * 2.0 ** -24 * mag[at]
             + 2 * HALF_ULP[dtype] * np.abs(ref[at]) + 1e-7)
    assert (np.abs(got[at] - ref[at]) <= bound).all()
    # the case is one: some values are not finite and most are
    assert 0 < (~at).sum() < at.sum()


@pytest.mark.parametrize('dtype,c_in,c_out,rows', [
    (torch.float32, 12, 24, 500), (torch.float32, 48, 40, 500),
    (torch.float32, 36, 130, 129), (torch.float16, 24, 40, 500),
    (torch.float16, 72, 65, 500), (torch.bfloat16, 72, 200, 300)])
@pytest.mark.parametrize('where', ['weight', 'weight nan', 'feats'])
def test_padded_conv_sums_its_own_edges(dtype, c_in, c_out, rows, where):
    from mlx_lattice_amd import SparseTensor, ops

    rng = np.random.default_rng(c_in + c_out)
    coords = _cloud(rows, rng)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    if where == 'feats':
        f[7, 3], f[11, c_in - 1], f[20, 0] = INF, -INF, NAN
    else:
        w[c_out - 1, 0, 0, 0, 2] = INF if where == 'weight' else NAN
        w[3, 2, 2, 1, c_in - 1] = -INF
    print(f'{where} {dtype} {c_in}->{c_out}', flush=True)
    y = ops.subm_conv3d(SparseTensor(torch.as_tensor(coords).to(DEV), f), w)
    b = torch.full((c_out,), 0.5, dtype=dtype, device=DEV)
    z = ops.subm_conv3d(SparseTensor(torch.as_tensor(coords).to(DEV), f), w, b,
                        activation='relu')
    torch.cuda.synchronize()
    rel = O.kernel_relation(coords, kernel_size=3)
    wk = to_np(w.double()).reshape(c_out, 27, c_in).transpose(1, 2, 0)
    ref, mag = _edge_sum(to_np(f.double()), wk, rel, rows)
    _check(y.feats, ref, mag, 27 * c_in + 1, dtype)
    # torch.equal takes no NaN for itself
    assert torch.equal(torch.nan_to_num(z.feats, 7.0),
                       torch.nan_to_num(torch.relu(y.feats + b), 7.0))


@pytest.mark.parametrize('dtype,c_in,c_out', [
    (torch.float32, 48, 40), (torch.float16, 24, 72)])
@pytest.mark.parametrize('op', ['subm', 'down'])
def test_padded_input_grad_sums_its_own_edges(op, dtype, c_in, c_out):
    from mlx_lattice_amd import SparseTensor, ops

    rows = 400
    rng = np.random.default_rng(c_in)
    coords = _cloud(rows, rng)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(
        DEV, dtype).requires_grad_()
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    w[5, 0, 1, 2, 1] = INF
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f)
    print(f'input grad {op} {dtype} {c_in}->{c_out}', flush=True)
    args = dict(kernel_size=3) if op == 'subm' else dict(
        kernel_size=3, stride=2, padding=1)
    y = (ops.subm_conv3d if op == 'subm' else ops.conv3d)(x, w, **args)
    rel = O.kernel_relation(coords, **args)
    cot = torch.as_tensor(rng.standard_normal(tuple(y.feats.shape))).to(
        DEV, dtype)
    cot[2, 4] = -INF
    grad, = torch.autograd.grad(y.feats, f, cot)
    torch.cuda.synchronize()
    back = dict(rel, in_rows=rel['out_rows'], out_rows=rel['in_rows'])
    wk = to_np(w.double()).reshape(c_out, 27, c_in).transpose(1, 0, 2)
    ref, mag = _edge_sum(to_np(cot.double()), wk, back, rows)
    _check(grad, ref, mag, 27 * c_out + 1, dtype)


@pytest.mark.parametrize('dtype,bits,c_in,c_out', [
    (torch.float16, 4, 96, 96), (torch.float16, 8, 40, 24),
    (torch.bfloat16, 4, 64, 96), (torch.float16, 4, 64, 40)])
@pytest.mark.parametrize('where', ['feats', 'scale', 'past fp16'])
def test_padded_packed_conv_sums_its_own_edges(dtype, bits, c_in, c_out,
                                               where):
    """An infinite feature, an infinite scale, and a weight code * scale +
    bias that is finite in float32 and not in float16."""
    from mlx_lattice_amd import SparseTensor, dequantize_weight, ops
    from mlx_lattice_amd import quantize_weight

    rows = 500
    rng = np.random.default_rng(bits + c_out)
    coords = _cloud(rows, rng)
    f = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    w = torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                        / np.sqrt(9 * c_in)).to(DEV, dtype)
    if where == 'past fp16':
        f = f / 4096
    q = quantize_weight(w, group_size=32, bits=bits)
    if where == 'feats':
        f[7, 3], f[11, c_in - 1] = INF, -INF
    elif where == 'scale':
        q.scales[3, 0, 5] = INF
    else:
        q.scales[0, 0, 3] = 60000.0 / (2 ** bits - 1)
        q.biases[0, 0, 3] = 30000.0
    print(f'{where} int{bits} {dtype} {c_in}->{c_out}', flush=True)
    y = ops.subm_conv3d(SparseTensor(torch.as_tensor(coords).to(DEV), f), q)
    torch.cuda.synchronize()
    with np.errstate(invalid='ignore'):
        wd = dequantize_weight(dataclasses.replace(
            q, scales=q.scales.float(), biases=q.biases.float()))
    wk = to_np(wd.double()).reshape(c_out, 27, c_in).transpose(1, 2, 0)
    ref, mag = _edge_sum(to_np(f.double()), wk,
                         O.kernel_relation(coords, kernel_size=3), rows)
    if where == 'past fp16':
        got = to_np(y.feats.double())
        assert np.isfinite(got).all() and np.abs(wk).max() > 65504
        bound = ((27 * c_in + 1) * 2.0 ** -24 + 2 * HALF_ULP[dtype] ** 2) * mag
        bound = bound + 2 * HALF_ULP[dtype] * np.abs(ref) + 1e-7
        assert (np.abs(got - ref) <= bound).all()
    else:
        _check(y.feats, ref, mag * (1 + 4 * HALF_ULP[dtype] ** 2 * 2 ** 24
                                    / (27 * c_in + 1)), 27 * c_in + 1, dtype)
