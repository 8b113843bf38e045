"""Groupings of half a million and more edges (tiles of 4096 and 8192 items
ordered in LDS) against numpy's stable sort, at the edges of the rule, with a
ragged last tile, one digit row, 10- and 11-bit digits, and inactive edges."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import to_np

pytestmark = pytest.mark.gpu

DEV = 'cuda'


@pytest.mark.parametrize('n,active,groups', [
    ((1 << 19) - 1, (1 << 19) - 1, 300000),   # below the rule
    (1 << 19, 1 << 19, 300000),
    ((1 << 21) - 1, (1 << 21) - 1, 900000),
    (1 << 21, 1 << 21, 900000),
    (1300001, 1299990, 1),
    (1300001, 1300001, 2000),
    (2500001, 1000003, 900000),
    (600003, 600003, 2200000),                # 11-bit digits
    (2100003, 2100003, 2200000),
])
def test_large_groupings_are_stable_sorts(n, active, groups):
    from mlx_lattice_amd._native import ext

    rng = np.random.default_rng(n + groups)
    rows = rng.integers(0, groups, n).astype(np.int32)
    kernels = rng.integers(0, 27, n).astype(np.int32)
    counts = torch.tensor([active, 0], dtype=torch.int32, device=DEV)
    print(f'large grouping {n}/{active} over {groups}', flush=True)
    got = ext.build_relation_grouped_views(
        torch.as_tensor(rows).to(DEV), torch.as_tensor(kernels).to(DEV),
        counts, groups, 27)
    torch.cuda.synchronize()
    for keys, bins, offsets, ids in ((rows, groups, got[0], got[1]),
                                     (kernels, 27, got[2], got[3])):
        keys = keys[:active]
        want = np.argsort(keys, kind='stable')
        np.testing.assert_array_equal(to_np(ids)[:active], want)
        np.testing.assert_array_equal(
            to_np(offsets), np.searchsorted(keys[want], np.arange(bins + 1)))
