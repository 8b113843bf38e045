"""Views, groupings and tile orders that a relation makes on their first use:
a first use under graph capture leaves nothing behind that an eager call
would read before the graph runs, and one on a side stream is waited for by
the others."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


def _data(rows, dtype, c_in, c_out, kernel, seed):
    rng = np.random.default_rng(seed)
    side = int(np.ceil((4 * rows) ** (1 / 3)))
    flat = rng.choice(side ** 3, rows, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // side ** 2,
                       flat // side % side, flat % side], 1).astype(np.int32)
    feats = torch.as_tensor(rng.standard_normal((rows, c_in))).to(DEV, dtype)
    weight = torch.as_tensor(
        rng.standard_normal((c_out, kernel, kernel, kernel, c_in))
        / np.sqrt(9 * c_in)).to(DEV, dtype).requires_grad_()
    return torch.as_tensor(coords).to(DEV), feats, weight


def _relation(x, op):
    manager = x.coord_manager
    if op == 'subm':
        return manager.submanifold_kernel_relation(x.coord_key, map_only=True)
    return manager.kernel_relation(x.coord_key, kernel_size=2, stride=2,
                                   map_only=True)


def _step(x, feats, weight, cot, op):
    from mlx_lattice_amd import ops

    y = x.replace(feats=feats)
    y = (ops.subm_conv3d(y, weight) if op == 'subm' else
         ops.conv3d(y, weight, kernel_size=2, stride=2)).feats
    return (y.detach(), *torch.autograd.grad(y, (feats, weight), cot))


CASES = [
    ('subm', torch.float32, 32, 40, 3000),     # rows in their own order
    ('subm', torch.float32, 64, 64, 33001),    # sorted, with a tile order
    ('subm', torch.float16, 64, 64, 33001),
    ('subm', torch.bfloat16, 96, 96, 3000),
    ('down', torch.float32, 32, 64, 3000),     # transposed views
    ('down', torch.float16, 32, 64, 40000),
]


@pytest.mark.parametrize('op,dtype,c_in,c_out,rows', CASES)
def test_first_use_under_capture(op, dtype, c_in, c_out, rows):
    from mlx_lattice_amd import SparseTensor

    coords, f, weight = _data(rows, dtype, c_in, c_out,
                              3 if op == 'subm' else 2, rows + c_out)
    feats = f.clone().requires_grad_()
    cot = torch.randn((rows, c_out), device=DEV).to(dtype)
    print(f'capture first {op} {dtype} {c_in}->{c_out} {rows}', flush=True)
    want = _step(SparseTensor(coords, f), feats, weight, cot, op)
    # (autograd and the allocator warm, the relation built but not used)
    x = SparseTensor(coords, f)
    relation = _relation(x, op)
    relation.expect_backward()
    assert relation.transposed_map_exact
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        captured = _step(x, feats, weight, cot, op)
    for name in ('_kernel_pairs', '_tiled', '_transposed_tiled',
                 'sorted_implicit_gemm', 'transposed_sorted_implicit_gemm',
                 '_grouped', '_kernel_grouped'):
        assert getattr(relation, name) is None, name
    eager = _step(x, feats, weight, cot, op)       # before any replay
    torch.cuda.synchronize()
    for got, ref in zip(eager, want):
        assert torch.equal(got, ref)
    for _ in range(3):
        for t in captured:
            t.zero_()
        graph.replay()
        again = _step(x, feats, weight, cot, op)
        torch.cuda.synchronize()
        for got, ref in zip(captured, want):
            assert torch.equal(got, ref)
        for got, ref in zip(again, want):
            assert torch.equal(got, ref)


@pytest.mark.parametrize('op,dtype,c_in,c_out,rows', CASES)
def test_first_use_on_a_side_stream(op, dtype, c_in, c_out, rows):
    from mlx_lattice_amd import SparseTensor

    coords, f, weight = _data(rows, dtype, c_in, c_out,
                              3 if op == 'subm' else 2, rows + c_in)
    feats = f.clone().requires_grad_()
    cot = torch.randn((rows, c_out), device=DEV).to(dtype)
    busy = torch.randn((4096, 4096), device=DEV)
    print(f'side stream first {op} {dtype} {c_in}->{c_out} {rows}',
          flush=True)
    want = _step(SparseTensor(coords, f), feats, weight, cot, op)
    x = SparseTensor(coords, f)
    relation = _relation(x, op)
    relation.expect_backward()
    assert relation.transposed_map_exact
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):                        # milliseconds ahead of it
            busy = busy @ busy * 2.0 ** -7
        first = _step(x, feats, weight, cot, op)
    with torch.cuda.stream(other):
        second = _step(x, feats, weight, cot, op)
    third = _step(x, feats, weight, cot, op)
    torch.cuda.synchronize()
    for results in (first, second, third):
        for got, ref in zip(results, want):
            assert torch.equal(got, ref)
    written = relation._written['_kernel_pairs']
    assert written[0] == side.cuda_stream and len(written) == 3
