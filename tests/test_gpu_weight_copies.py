"""Convs read the weight as it is when they run: float32 and widths that do
not fill the tiles, whose kernel takes the weight in another order, see
writes that the version counter does not count (through ``.data``, by a graph
replay), and a captured conv sees the weight of each replay."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


def _tensor(rows, channels, dtype, seed):
    from mlx_lattice_amd import SparseTensor

    rng = np.random.default_rng(seed)
    flat = rng.choice(14 ** 3, rows, replace=False)
    coords = np.stack([np.zeros_like(flat), flat // 196, flat // 14 % 14,
                       flat % 14], 1).astype(np.int32)
    x = SparseTensor(
        torch.as_tensor(coords).to(DEV),
        torch.as_tensor(rng.standard_normal((rows, channels))).to(DEV, dtype))
    return x, rng


def _weight(rng, c_out, c_in, dtype):
    return torch.as_tensor(rng.standard_normal((c_out, 3, 3, 3, c_in))
                           / np.sqrt(9 * c_in)).to(DEV, dtype)


def _both(x, w, cot):
    from mlx_lattice_amd import ops

    f = x.feats.detach().requires_grad_()
    y = ops.subm_conv3d(x.replace(feats=f), w).feats
    return y.detach(), torch.autograd.grad(y, f, cot)[0]


@pytest.mark.parametrize('dtype,c_in,c_out', [
    (torch.float32, 48, 40), (torch.float32, 64, 64), (torch.float16, 24, 40),
    (torch.bfloat16, 96, 96)])
def test_writes_through_data_are_seen(dtype, c_in, c_out):
    x, rng = _tensor(600, c_in, dtype, c_in)
    w = _weight(rng, c_out, c_in, dtype).requires_grad_()
    cot = torch.as_tensor(rng.standard_normal((600, c_out))).to(DEV, dtype)
    print(f'.data {dtype} {c_in}->{c_out}', flush=True)
    twice = 2 * w.detach()
    y, g = _both(x, w, cot)
    w.data.mul_(2)
    y2, g2 = _both(x, w, cot)
    y1, g1 = _both(x, twice, cot)
    other = _weight(rng, c_out, c_in, dtype)
    w.data = other.clone()
    y3, g3 = _both(x, w, cot)
    y4, g4 = _both(x, other, cot)
    torch.cuda.synchronize()
    assert torch.equal(y2, y1) and torch.equal(g2, g1)
    assert not torch.equal(y2, y) and not torch.equal(g2, g)
    assert torch.equal(y3, y4) and torch.equal(g3, g4)


@pytest.mark.parametrize('dtype,bits', [(torch.float16, 4),
                                        (torch.bfloat16, 8)])
def test_writes_to_packed_data_are_seen(dtype, bits):
    from mlx_lattice_amd import ops, quantize_weight

    x, rng = _tensor(600, 64, dtype, bits)
    q = quantize_weight(_weight(rng, 96, 64, dtype), group_size=32, bits=bits)
    other = quantize_weight(_weight(rng, 96, 64, dtype), group_size=32,
                            bits=bits)
    ops.subm_conv3d(x, q)
    print(f'packed .data {dtype} int{bits}', flush=True)
    for name in ('weight', 'scales', 'biases'):
        getattr(q, name).data.copy_(getattr(other, name))
    a, b = ops.subm_conv3d(x, q), ops.subm_conv3d(x, other)
    torch.cuda.synchronize()
    assert torch.equal(a.feats, b.feats)


@pytest.mark.parametrize('dtype,c_in,c_out', [
    (torch.float32, 48, 40), (torch.float16, 24, 40)])
def test_a_captured_step_and_eager_calls_between_replays(dtype, c_in, c_out):
    """The graph holds forward, gradients and the update of the weight."""
    from mlx_lattice_amd import ops

    x, rng = _tensor(600, c_in, dtype, 3)
    w = _weight(rng, c_out, c_in, dtype).requires_grad_()
    cot = torch.as_tensor(rng.standard_normal((600, c_out))).to(DEV, dtype)
    f = x.feats.detach().requires_grad_()

    def step():
        y = ops.subm_conv3d(x.replace(feats=f), w).feats
        gf, gw = torch.autograd.grad(y, (f, w), cot)
        with torch.no_grad():
            w.add_(gw, alpha=-2.0 ** -10)
        return y.detach(), gf

    print(f'captured step {dtype} {c_in}->{c_out}', flush=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        y, gf = step()
    for _ in range(3):
        y0, g0 = _both(x, w.detach().clone(), cot)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, y0) and torch.equal(gf, g0)
        now = _both(x, w, cot)               # the weight of the last replay
        fresh = _both(x, w.detach().clone(), cot)
        torch.cuda.synchronize()
        assert torch.equal(now[0], fresh[0]) and torch.equal(now[1], fresh[1])
        assert not torch.equal(now[0], y)


@pytest.mark.parametrize('mapped', [False, True])
def test_kept_copies_follow_a_new_storage(mapped):
    """The tuned 16-bit widths keep a copy of the weight in the kernel's
    order; one made of other storage (an assignment to ``.data``) is not
    taken for it."""
    from mlx_lattice_amd import ops, quantize_weight

    dtype = torch.float16
    x, rng = _tensor(600, 64, dtype, 5)
    w, other = (_weight(rng, 64, 64, dtype) for _ in range(2))
    if mapped:
        w, other = (v.permute(1, 2, 3, 4, 0).reshape(27, 64, 64).contiguous()
                    for v in (w, other))
    cot = torch.as_tensor(rng.standard_normal((600, 64))).to(DEV, dtype)
    print(f'kept copies mapped={mapped}', flush=True)
    w.requires_grad_()
    _both(x, w, cot)
    w.data = other.clone()
    now, want = _both(x, w, cot), _both(x, other, cot)
    q, r = (quantize_weight(_weight(rng, 64, 64, dtype), group_size=32,
                            bits=4) for _ in range(2))
    ops.subm_conv3d(x, q)
    for name in ('weight', 'scales', 'biases'):
        getattr(q, name).data = getattr(r, name).clone()
    a, b = ops.subm_conv3d(x, q), ops.subm_conv3d(x, r)
    torch.cuda.synchronize()
    assert torch.equal(now[0], want[0]) and torch.equal(now[1], want[1])
    assert torch.equal(a.feats, b.feats)
