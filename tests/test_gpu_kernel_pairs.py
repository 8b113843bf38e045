"""Edges grouped by kernel offset from the row masks, against the oracle's
stable grouping (bit for bit), at the edges of the 64-row waves and 1024-row
blocks, with inactive rows and with all 32 mask bits in use."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.mark.parametrize('kind,size,rows,active', [
    ('submanifold', 3, 1, 1), ('submanifold', 3, 64, 64),
    ('submanifold', 3, 1023, 1000), ('submanifold', 3, 1025, 1025),
    ('submanifold', 3, 40000, 39001), ('submanifold', 1, 70, 0),
    ('forward', 2, 3000, 3000), ('forward', 3, 5000, 4999),
    ('forward', (4, 4, 2), 2000, 2000),      # K = 32: the sign bit of a mask
    ('target', 3, 2500, 2500),
])
def test_kernel_groups_match_the_oracle(kind, size, rows, active):
    from mlx_lattice_amd.core.coords import builders

    rng = np.random.default_rng(rows + active)
    side = max(6, int(np.ceil((4 * rows) ** (1 / 3))))
    flat = rng.choice(side ** 3, rows, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // side ** 2,
                       flat // side % side, flat % side], 1).astype(np.int32)
    c = torch.as_tensor(coords).to(DEV)
    a = torch.tensor([active], dtype=torch.int32, device=DEV)
    print(f'kernel groups {kind} {size} {rows}/{active}', flush=True)
    if kind == 'submanifold':
        rel = builders.build_submanifold_kernel_relation(c, a, size)
    elif kind == 'forward':
        rel = builders.build_kernel_relation(c, a, size, stride=2)
    else:
        target = torch.as_tensor(coords[::2].copy()).to(DEV)
        rel = builders.build_target_kernel_relation(c, target, kernel_size=3)
    offsets, pairs = rel.kernel_pairs()
    csr = rel.kernel_csr
    torch.cuda.synchronize()
    e = int(rel.counts[0].item())
    k = to_np(rel.edges.kernel_ids)[:e]
    ids = np.argsort(k, kind='stable')
    starts = np.searchsorted(k[ids], np.arange(rel.n_kernels + 1))
    np.testing.assert_array_equal(to_np(offsets), starts)
    np.testing.assert_array_equal(to_np(csr.row_offsets), starts)
    np.testing.assert_array_equal(to_np(csr.edge_ids)[:e], ids)
    np.testing.assert_array_equal(
        to_np(pairs)[:e], np.stack([to_np(rel.edges.in_rows)[:e][ids],
                                    to_np(rel.edges.out_rows)[:e][ids]], 1))
    if kind == 'submanifold' and active == rows:
        orel = O.kernel_relation(coords, kernel_size=size)
        np.testing.assert_array_equal(to_np(offsets),
                                      orel['kernel_row_offsets'])
        np.testing.assert_array_equal(to_np(csr.edge_ids)[:e],
                                      orel['kernel_edge_ids'][:e])


def test_weight_grad_over_pairs_equals_the_csr_route():
    from mlx_lattice_amd import SparseTensor
    from mlx_lattice_amd._native import ext

    rng = np.random.default_rng(5)
    flat = rng.choice(40 ** 3, 20000, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // 1600, flat // 40 % 40,
                       flat % 40], 1).astype(np.int32)
    x = SparseTensor(torch.as_tensor(coords).to(DEV),
                     torch.zeros((len(coords), 1), device=DEV))
    rel = x.coord_manager.submanifold_kernel_relation(x.coord_key)
    offsets, pairs = rel.kernel_pairs()
    csr = rel.kernel_csr
    for dtype, c_in, c_out in ((torch.float32, 48, 80),
                               (torch.float16, 128, 64)):
        f = torch.as_tensor(rng.standard_normal((len(coords), c_in))).to(
            DEV, dtype)
        g = torch.as_tensor(rng.standard_normal((len(coords), c_out))).to(
            DEV, dtype)
        w = torch.zeros((c_out, 3, 3, 3, c_in), dtype=dtype, device=DEV)
        a = ext.sparse_conv_weight_grad_pairs(f, g, w, pairs, offsets, 27)
        b = ext.sparse_conv_weight_grad(
            f, g, w, rel.edges.in_rows, rel.edges.out_rows, rel.counts,
            csr.row_offsets, csr.edge_ids, 27)
        torch.cuda.synchronize()
        assert torch.equal(a, b)
