"""Convs over the unsorted view of small relations: the same results, bit for
bit, as over the mask-sorted view, at the edges of the 16-row masks and
64-row tiles, with inactive rows, for every conv that takes a view."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_np

pytestmark = pytest.mark.gpu

DEV = 'cuda'


def _tensor(rows, active, channels, dtype, rng):
    from mlx_lattice_amd import SparseTensor

    side = max(6, int(np.ceil((4 * rows) ** (1 / 3))))
    flat = rng.choice(side ** 3, rows, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // side ** 2,
                       flat // side % side, flat % side], 1).astype(np.int32)
    return SparseTensor(
        torch.as_tensor(coords).to(DEV),
        torch.as_tensor(rng.standard_normal((rows, channels))).to(DEV, dtype),
        active_rows=torch.tensor([active], dtype=torch.int32, device=DEV))


@pytest.mark.parametrize('op,dtype,bits,c_in,c_out,rows,active', [
    ('subm', torch.float16, 0, 64, 64, 1, 1),
    ('subm', torch.float16, 0, 64, 64, 1000, 903),
    ('subm', torch.float16, 4, 64, 64, 129, 129),
    ('subm', torch.float16, 8, 32, 32, 500, 500),     # register-staged kernel
    ('subm', torch.float32, 0, 16, 32, 2049, 2000),
    ('down', torch.bfloat16, 0, 32, 64, 3000, 2999),
    ('down', torch.float32, 0, 24, 40, 777, 777),
])
def test_conv_over_the_tiled_view_equals_the_sorted_one(op, dtype, bits, c_in,
                                                        c_out, rows, active):
    from mlx_lattice_amd import ops, quantize_weight

    rng = np.random.default_rng(rows + c_in)
    k = 3 if op == 'subm' else 2
    x = _tensor(rows, active, c_in, dtype, rng)
    w = torch.as_tensor(rng.standard_normal((c_out, k, k, k, c_in)) / 8).to(
        DEV, dtype)
    weight = quantize_weight(w, group_size=32, bits=bits) if bits else w
    print(f'tiled {op} {dtype} int{bits} {c_in}->{c_out} {rows}', flush=True)

    def run(t):
        if op == 'subm':
            return ops.subm_conv3d(t, weight, kernel_size=3)
        return ops.conv3d(t, weight, kernel_size=2, stride=2)

    def relation(t):
        if op == 'subm':
            return t.coord_manager.submanifold_kernel_relation(t.coord_key)
        return t.coord_manager.kernel_relation(t.coord_key, kernel_size=2,
                                               stride=2)

    grads = not bits
    feats = x.feats.requires_grad_(grads)
    y = run(x)
    rel = relation(x)
    assert rel._tiled is not None and rel.sorted_implicit_gemm is None
    cot = torch.as_tensor(rng.standard_normal(tuple(y.feats.shape))).to(
        DEV, dtype)
    g = torch.autograd.grad(y.feats, feats, cot)[0] if grads else None
    rel.require_sorted_implicit_gemm()
    if op == 'down':
        rel.require_transposed_sorted_implicit_gemm()
    z = run(x)
    assert torch.equal(y.feats, z.feats)
    if grads:
        assert torch.equal(g, torch.autograd.grad(z.feats, feats, cot)[0])
    # the view itself: the map transposed, its rows' masks by sixteens
    view = rel._tiled
    dense = rel.require_implicit_gemm()
    torch.cuda.synchronize()
    n = int(view.reorder_rows.shape[0])
    np.testing.assert_array_equal(to_np(view.reorder_rows), np.arange(n))
    np.testing.assert_array_equal(to_np(view.sorted_kv_out_in_map),
                                  to_np(dense.out_in_map).T)
    masks = np.zeros((n + 63) // 64 * 64, np.int64)
    masks[:n] = to_np(dense.row_masks)[:, 0]
    np.testing.assert_array_equal(
        to_np(view.tile_masks),
        np.bitwise_or.reduce(masks.reshape(-1, 16), axis=1))


def test_wide_convs_and_large_relations_sort():
    from mlx_lattice_amd.core.relations.views import _tiled_pays

    assert _tiled_pays(16384, 16384) and _tiled_pays(32768, 8192)
    assert not _tiled_pays(16385, 16384)
    assert not _tiled_pays(32769, 1)
    assert not _tiled_pays(1, 16385)
