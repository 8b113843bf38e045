"""Relations built as a dense map alone: edges, row offsets, counts, groupings
and the transposed map made later from the map equal those of the build that
emits the edges (bit for bit), at the edges of the 64-row blocks, with
inactive rows and with all 32 mask bits in use; a use on another stream waits
for them, and one under graph capture keeps nothing."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


def _coords(rows, seed):
    rng = np.random.default_rng(seed)
    side = max(6, int(np.ceil((4 * rows) ** (1 / 3))))
    flat = rng.choice(side ** 3, rows, replace=False)
    c = np.stack([np.zeros_like(flat), flat // side ** 2,
                  flat // side % side, flat % side], 1).astype(np.int32)
    return torch.as_tensor(c).to(DEV)


@pytest.mark.parametrize('kind,size,rows,active', [
    ('submanifold', 3, 0, 0), ('submanifold', 3, 1, 1),
    ('submanifold', 3, 64, 64), ('submanifold', 3, 1025, 1000),
    ('submanifold', 3, 40000, 39001), ('submanifold', 1, 70, 0),
    ('submanifold', (5, 3, 1), 3000, 3000),
    ('forward', 2, 3000, 2999), ('forward', 3, 5000, 4999),
    ('forward', (4, 4, 2), 2000, 2000), ('forward', 4, 500, 500),
    ('target', 3, 2500, 2500),
])
def test_edges_of_a_map_equal_the_emitted_ones(kind, size, rows, active):
    from mlx_lattice_amd._native import ext
    from mlx_lattice_amd.core.coords import builders

    c = _coords(max(rows, 1), rows + active)[:rows].contiguous()
    a = torch.tensor([active], dtype=torch.int32, device=DEV)
    print(f'map edges {kind} {size} {rows}/{active}', flush=True)

    def build(map_only):
        if kind == 'submanifold':
            return builders.build_submanifold_kernel_relation(
                c, a, size, map_only=map_only)
        if kind == 'forward':
            return builders.build_kernel_relation(c, a, size, stride=2,
                                                  map_only=map_only)
        return builders.build_target_kernel_relation(
            c, c[::2].contiguous(), kernel_size=size, map_only=map_only)

    lazy, full = build(True), build(False)
    assert lazy.edge_capacity == full.edge_capacity
    assert (lazy._map_edges is not None) == (full.n_kernels <= 32)
    if full.n_kernels <= 32 and kind != 'target' and rows:
        # before any use of the edges
        got = lazy._transposed_map()
        want = ext.build_transposed_implicit_gemm_map(
            full.edges.in_rows, full.edges.out_rows, full.edges.kernel_ids,
            full.counts, full.n_in_capacity, full.n_kernels)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert int(lazy.out_count.item()) == int(full.out_count.item())
    e = int(full.edge_count.item())
    assert lazy.counts.tolist() == full.counts.tolist()
    assert int(lazy.contract.edge_count.item()) == e
    assert torch.equal(lazy.row_offsets, full.row_offsets)
    for name in ('in_rows', 'out_rows', 'kernel_ids'):
        assert torch.equal(getattr(lazy.edges, name)[:e],
                           getattr(full.edges, name)[:e])
    n = int(full.out_count.item())
    assert torch.equal(lazy.out_coords[:n], full.out_coords[:n])
    for view in ('input_csr', 'kernel_csr'):
        got, want = getattr(lazy, view), getattr(full, view)
        assert torch.equal(got.row_offsets, want.row_offsets)
        assert torch.equal(got.edge_ids[:e], want.edge_ids[:e])


def test_edges_used_on_another_stream_and_under_capture():
    from mlx_lattice_amd.core.coords import builders

    c = _coords(30000, 3)
    full = builders.build_submanifold_kernel_relation(c)
    lazy = builders.build_submanifold_kernel_relation(c, map_only=True)
    e = int(full.counts[0].item())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        out = torch.zeros(e, dtype=torch.int32, device=DEV)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            out.copy_(lazy.edges.in_rows[:e])
    assert lazy._map_edges._made is None
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, full.edges.in_rows[:e])
        assert lazy._map_edges._made is None
    with torch.cuda.stream(side):
        first = lazy.edges.in_rows[:e].clone()
    second = lazy.edges.out_rows[:e].clone()
    torch.cuda.synchronize()
    assert torch.equal(first, full.edges.in_rows[:e])
    assert torch.equal(second, full.edges.out_rows[:e])


@pytest.mark.parametrize('repeat', [False, True])
def test_repeat_flag_is_read_after_a_forward_without_gradients(repeat):
    """The status word of a submanifold relation is copied when something
    asks for it; a relation first used without gradients, then with them,
    and under capture before any copy, takes a route that holds every edge."""
    from mlx_lattice_amd import SparseTensor, ops

    c = _coords(3000, 11)
    if repeat:
        c[17] = c[5]
    rng = np.random.default_rng(4)
    f = torch.as_tensor(rng.standard_normal((3000, 32)).astype(np.float32))
    w = torch.as_tensor((rng.standard_normal((32, 3, 3, 3, 32)) / 17).astype(
        np.float32)).to(DEV)
    g = torch.as_tensor(rng.standard_normal((3000, 32)).astype(
        np.float32)).to(DEV)

    def grad(x, feats):
        y = ops.subm_conv3d(x.replace(feats=feats), w)
        return torch.autograd.grad(y.feats, feats, g)[0]

    feats = f.to(DEV).requires_grad_()
    want = grad(SparseTensor(c, f.to(DEV)), feats)
    x = SparseTensor(c, f.to(DEV))
    ops.subm_conv3d(x, w)                       # no gradient: no copy yet
    relation = x.coord_manager.submanifold_kernel_relation(x.coord_key)
    assert relation.repeated_coords.unreadable is False
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        captured = grad(x, feats)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        # fp32 sums of up to 27 * 32 products in another order
        assert torch.allclose(captured, want, rtol=1e-5, atol=1e-4)
    fresh = SparseTensor(c, f.to(DEV))
    ops.subm_conv3d(fresh, w)
    assert torch.equal(grad(fresh, feats), want)
    relation = fresh.coord_manager.submanifold_kernel_relation(
        fresh.coord_key)
    assert relation.transposed_map_exact is not repeat


@pytest.mark.parametrize('trained', ['weight', 'feats'])
def test_a_forward_without_grad_mode_prepares_a_captured_backward(trained):
    """A trainable layer evaluated under ``no_grad`` first: a step captured
    afterwards takes the input gradient that an eager one takes."""
    from mlx_lattice_amd import SparseTensor, ops

    c = _coords(3000, 12)
    rng = np.random.default_rng(5)
    f = torch.as_tensor(rng.standard_normal((3000, 64))).to(
        DEV, torch.float16)
    w = torch.as_tensor(rng.standard_normal((64, 3, 3, 3, 64)) / 24).to(
        DEV, torch.float16)
    g = torch.as_tensor(rng.standard_normal((3000, 64))).to(
        DEV, torch.float16)

    def grad(x, feats):
        y = ops.subm_conv3d(x.replace(feats=feats), w)
        return torch.autograd.grad(y.feats, feats, g)[0]

    feats = f.clone().requires_grad_()
    want = grad(SparseTensor(c, f), feats)
    x = SparseTensor(c, f)
    with torch.no_grad():
        if trained == 'weight':
            ops.subm_conv3d(x, w.clone().requires_grad_())
        else:
            ops.subm_conv3d(x.replace(feats=feats), w)
    relation = x.coord_manager.submanifold_kernel_relation(x.coord_key)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        assert not relation.repeated_coords.unreadable
        captured = grad(x, feats)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, want)
