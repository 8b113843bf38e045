"""A packed conv's arithmetic does not depend on the number of rows: the same
rows convolved alone and in a tensor whose capacity takes the kernel's large
tiles (the other rows inactive) give the same bits."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.mark.parametrize('dtype,bits,c_in,c_out,capacity', [
    (torch.float16, 4, 64, 64, 65537),     # one column tile: 65536 rows
    (torch.float16, 8, 96, 128, 65537),    # a partial last chunk
    (torch.bfloat16, 4, 64, 256, 16385),   # two column tiles: 16384 rows
    (torch.bfloat16, 8, 128, 64, 65537),
])
def test_packed_conv_of_few_rows_equals_that_of_many(dtype, bits, c_in, c_out,
                                                     capacity):
    from mlx_lattice_amd import SparseTensor, ops, quantize_weight

    rows = 1500
    rng = np.random.default_rng(bits + c_in)
    flat = rng.choice(18 ** 3, rows, replace=False)
    coords = np.zeros((capacity, 4), np.int32)
    coords[:rows, 1:] = np.stack([flat // 324, flat // 18 % 18, flat % 18], 1)
    c = torch.as_tensor(coords).to(DEV)
    f = torch.as_tensor(rng.standard_normal((capacity, c_in))).to(DEV, dtype)
    q = quantize_weight(torch.as_tensor(
        rng.standard_normal((c_out, 3, 3, 3, c_in)) / np.sqrt(9 * c_in)).to(
            DEV, dtype), group_size=32, bits=bits)
    print(f'int{bits} {dtype} {c_in}->{c_out}', flush=True)
    few = ops.subm_conv3d(SparseTensor(c[:rows], f[:rows]), q)
    many = ops.subm_conv3d(SparseTensor(
        c, f, active_rows=torch.tensor([rows], dtype=torch.int32, device=DEV)),
        q)
    torch.cuda.synchronize()
    assert torch.equal(few.feats, many.feats[:rows])
