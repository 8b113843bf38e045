"""The pooling gradient of relations whose input rows feed at most one output
row (written from the output rows) against the input-grouped form, bit for
bit: with inactive rows, repeated coordinates (no edge: zero gradient),
strides that skip voxels, ties, NaN and infinities."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_np

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.mark.parametrize('mode', ['sum', 'max', 'avg'])
@pytest.mark.parametrize('ks,stride,channels,rows,active', [
    (2, 2, 64, 4000, 4000),     # every row covered
    (2, 2, 30, 1500, 1400),     # inactive rows; channels one by one
    (2, 3, 4, 900, 900),        # voxels between the cells have no edge
    (1, 2, 8, 1, 1),
    (3, 3, 12, 5000, 5000),     # rows with more edges than stay in registers
    (2, 2, 16, 300, 0),
])
def test_exclusive_gradient_equals_the_input_grouped_one(mode, ks, stride,
                                                         channels, rows,
                                                         active):
    from mlx_lattice_amd import SparseTensor, ops
    from mlx_lattice_amd._native import ext

    rng = np.random.default_rng(rows + ks)
    side = max(4, int(np.ceil((1.3 * rows) ** (1 / 3))))
    flat = rng.choice(side ** 3, rows, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // side ** 2,
                       flat // side % side, flat % side], 1).astype(np.int32)
    if rows > 100:
        coords[rows // 2] = coords[1]
    values = rng.integers(-3, 4, (rows, channels)).astype(np.float32)
    values[rows // 3] = np.nan
    values[rows // 4, ::2] = np.inf
    values[rows // 5, 1::2] = -np.inf
    f = torch.as_tensor(values).to(DEV).requires_grad_()
    a = torch.tensor([active], dtype=torch.int32, device=DEV)
    print(f'pool grad {mode} k{ks}s{stride} C={channels}', flush=True)
    x = SparseTensor(torch.as_tensor(coords).to(DEV), f, active_rows=a)
    y = ops.pool3d(x, mode=mode, kernel_size=ks, stride=stride)
    cot = torch.as_tensor(rng.standard_normal(tuple(y.feats.shape)).astype(
        np.float32)).to(DEV)
    grad, = torch.autograd.grad(y.feats, f, cot)
    rel = x.coord_manager.kernel_relation(x.coord_key, kernel_size=ks,
                                          stride=stride)
    csr = rel.input_csr
    for off in (0, 1):      # and an array that starts off a 16-byte border
        flat_cot = torch.empty(cot.numel() + 1, device=DEV)
        shifted = flat_cot[off:off + cot.numel()].view(cot.shape)
        shifted.copy_(cot)
        ref = ext.sparse_pool_features_grad(
            shifted, f.detach(), y.feats.detach(), rel.edges.in_rows,
            rel.edges.out_rows, rel.output_csr.row_offsets, rel.counts,
            csr.row_offsets, csr.edge_ids, mode)
        got = ext.sparse_pool_features_grad_exclusive(
            shifted, f.detach(), y.feats.detach(), rel.edges.in_rows,
            rel.output_csr.row_offsets, rel.counts, a, mode)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(to_np(got), to_np(ref))
    np.testing.assert_array_equal(to_np(grad), to_np(ref))
