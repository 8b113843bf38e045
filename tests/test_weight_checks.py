"""A weight that does not fit the relation or the features is refused on the
routes of every type, with the error of the entry that checks it (on the CPU:
the checks come before anything that needs a device)."""

from __future__ import annotations

import pytest
import torch


def _relation(n_kernels):
    from mlx_lattice_amd.core.relations import KernelRelation

    rows = torch.zeros(3, dtype=torch.int32)
    return KernelRelation(
        rows, rows.clone(), rows.clone(),
        row_offsets=torch.zeros(4, dtype=torch.int32), n_in_capacity=3,
        n_out_capacity=3, n_kernels=n_kernels)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('shape,match', [
    ((27, 24, 40), 'kernel rows must match'),
    ((40, 3, 3, 3, 24), 'kernel rows must match'),
    ((24, 40), 'must have shape'),
    ((8, 16, 40), 'input channels'),
])
def test_forward_refuses_a_weight_of_another_relation(dtype, shape, match):
    from mlx_lattice_amd.ops import _relation_exec as ex

    feats = torch.zeros((3, 24), dtype=dtype)
    with pytest.raises(ValueError, match=match):
        ex.sparse_conv_features_from_relation(
            feats, torch.zeros(shape, dtype=dtype), _relation(8))


@pytest.mark.parametrize('dtype,channels', [
    (torch.float32, 36), (torch.float16, 32)])
def test_input_grad_refuses_a_cotangent_of_other_channels(dtype, channels):
    """Both channel counts fill the same number of fragments."""
    from mlx_lattice_amd.ops import _relation_exec as ex

    with pytest.raises(ValueError, match='cotangent channels'):
        ex.sparse_conv_input_grad_from_relation(
            torch.zeros((3, channels), dtype=dtype),
            torch.zeros((8, 24, 40 if channels == 36 else 24), dtype=dtype),
            _relation(8), 3)
