"""Dispatch of a prebuilt relation to the native conv kernels
(mlx_lattice/ops/_relation_exec.py:19-250).

Route policy (this build's, the reference routes by Metal capability):
features with at most 32 kernel offsets run a matrix-core implicit GEMM over
the mask-sorted view, for every relation kind whose edges fit the dense
(out_row, offset) map: fp16/bf16 with ``C_in % 32 == 0`` and ``C_out`` in
{16, 32, 64, 128, 256} on the kernels tuned for those, other channel counts
and fp32 on the streamed kernel's padded instances (rows of whole 16-byte
pieces); everything else, and the narrow rows of ``edges_pay``, runs the CSR
bandwidth kernel.  All routes compute the same sum with an fp32 accumulator.
Copies of a weight in a kernel's order are kept with it for the tuned widths
alone, by its identity, storage and version counter; the padded instances make theirs
in the call.
"""

from __future__ import annotations

import weakref

import torch

from mlx_lattice_amd._native import ext
from mlx_lattice_amd.core.quantized import QuantizedWeight
from mlx_lattice_amd.core.relations import KernelRelation

_MATRIX_CORE_C_OUT = (16, 32, 64, 128, 256)
# (id(weight), kind) -> (weak reference, (storage, shape, dtype, version),
# value)
_WEIGHT_CACHE: dict[tuple[int, str], tuple[weakref.ReferenceType, tuple,
                                           torch.Tensor]] = {}


def _empty_i32(device) -> torch.Tensor:
    return torch.empty(0, dtype=torch.int32, device=device)


def _require_static(relation: KernelRelation) -> None:
    if relation.n_out_capacity is None or relation.n_kernels is None:
        raise ValueError('kernel relation is missing static shape metadata.')


def _matrix_core_eligible(dtype: torch.dtype, c_in: int, c_out: int,
                          relation: KernelRelation, n_in: int = 0) -> bool:
    """Shapes the matrix-core kernel takes; its 32-bit gather offsets need
    the feature table under 2 GiB.  The relation must fit the dense
    (out_row, offset) map: a transposed relation with a repeated input
    coordinate runs the CSR route."""
    return (relation.dense_map_exact
            and dtype in (torch.float16, torch.bfloat16)
            and c_in % 32 == 0 and c_in <= 512
            and c_out in _MATRIX_CORE_C_OUT
            and relation.n_kernels is not None and relation.n_kernels <= 32
            and n_in * c_in * 2 < 2 ** 31)


def _small_dense_map(dtype: torch.dtype, c_in: int, c_out: int,
                     relation: KernelRelation) -> torch.Tensor | None:
    """The relation's dense map for the dense-map conv of few input
    channels (C_in 4 or 8, C_out 16 or 32, fp16/bf16), when the relation
    already holds it: the native CSR entry then contracts a row's whole
    neighbourhood on the matrix cores instead of walking its edges."""
    if (relation.implicit_gemm is None
            or dtype not in (torch.float16, torch.bfloat16)
            or c_in not in (4, 8) or c_out not in (16, 32)
            or relation.n_kernels is None or relation.n_kernels * c_in > 256):
        return None
    view = relation.require_implicit_gemm()
    if (view.out_in_map.dtype != torch.int32
            or tuple(view.out_in_map.shape) != (relation.n_out_capacity,
                                                relation.n_kernels)
            or not relation.dense_map_exact):
        return None
    return view.out_in_map


def _dense_without_edges(feats: torch.Tensor,
                         dense: torch.Tensor | None) -> bool:
    """Whether the native entry, given this dense map, runs the dense-map
    conv and so needs no edges (rows to write, feature rows aligned to their
    size)."""
    return (dense is not None and dense.numel() > 0
            and (not feats.is_contiguous()
                 or feats.data_ptr()
                 % (int(feats.shape[1]) * feats.element_size()) == 0))


# lattice_fragment_role: the weight of a padded conv
_FORWARD, _TRANSPOSED, _MIRRORED = 0, 1, 2


def _padded_eligible(feats: torch.Tensor, c_out: int,
                     relation: KernelRelation, rows: int) -> bool:
    """Whether a conv of ``feats`` with ``c_out`` output channels and
    ``rows`` output rows takes the streamed kernel's padded instances: types
    and channel counts the sorted entries refuse, in rows of whole 16-byte
    pieces (``ext.conv_padded_supported``: sizes and alignment)."""
    return (relation.n_kernels is not None and relation.n_kernels <= 32
            and feats.ndim == 2
            and ext.conv_padded_supported(feats, c_out, relation.n_kernels,
                                          rows))


def edges_pay(c_in: int, c_out: int, element_size: int, rows: int) -> bool:
    """Whether a conv over a new relation runs faster over its edges than in
    the padded instances: the edge kernels' time grows with rows and input
    channels, while the view costs a launch up to 32,768 rows and a sort
    above, and few outputs leave most of a 32-column group empty.  Map build
    and 3^3 fp32 conv, edges / padded us:

    rows     4 -> 3    4 -> 16   4 -> 24   4 -> 32   8 -> 8    8 -> 16
    4,000    53 / 59   54 / 58   55 / 59   55 / 58   53 / 58   56 / 57
    32,000   54 / 58   59 / 57             70 / 58             73 / 59
    65,000   66 / 116  70 / 117  95 / 115  80 / 116  76 / 116  83 / 115
    130,000  89 / 142  93 / 141  141 / 142 100 / 143 114 / 140 120 / 140
    400,000  257 / 290 293 / 287           303 / 291           514 / 288

    (8 -> 24 over 65,000 rows 154 / 116, 12 -> 3 91 / 117, 16 -> 16
    109 / 114; 16 -> 32 over 20,000 117 / 58.)  Over a sorted view that is
    there the padded instances are as fast or faster from 32,768 rows on
    (130,000 rows, 4 -> 16 35 / 36, 8 -> 16 63 / 36).  Packed weights gain
    more (int8 8 -> 8 over 32,000 rows 60 / 66, over 130,000 rows
    124 / 158)."""
    if rows <= 32768:
        return c_in <= 8 and c_out <= (16 if c_in * element_size <= 16 else 8)
    return rows * c_in <= 1 << 20 and (
        c_out <= 16 and c_in <= 8 or c_out <= 4 and c_in <= 16
        or c_out == 32 and c_in <= 4)


def _expanded_edges_pay(n_kernels: int, c_in: int, c_out: int) -> bool:
    """``edges_pay`` of transposed and generative relations, whose rows hold
    one edge or few.  fp16 over the edges / padded + its view, us, from 30,000
    rows: k2s2 16 -> 16 11 / 20 + 68, 16 -> 24 40 / 21 + 68, 16 -> 32
    22 / 20 + 68, 24 -> 24 53 / 20 + 68, 8 -> 64 89 / 23 + 68; k3s2 16 -> 16
    67 / 36 + 207, 16 -> 32 169 / 38 + 207, 24 -> 16 335 / 37 + 207; packed
    weights the same to 1.4 times as long on either side.  The last four of
    these gain little from the edges, or lose much to a view that is there."""
    rows_kernel = c_in <= 16 and c_out in (16, 32)
    return n_kernels * c_in * c_out <= (8192 if rows_kernel else 3072)


def _padded_forward(feats: torch.Tensor, c_in: int, c_out: int,
                    relation: KernelRelation) -> bool:
    """The forward conv's use of the padded instances: where they are
    eligible and the edges do not run faster.  Expanded relations keep the
    CSR route in fp32: k2s2 from 30,000 rows, 16 -> 32 channels take 27 us
    over the edges, and 24 over a view that takes 61 to build; from 32
    channels on the padded instances would be faster with the view too
    (64 -> 64: 2871 against 47 + 61)."""
    if not relation.dense_map_exact:
        return False
    if relation.kind in ('transposed', 'generative'):
        if (feats.dtype == torch.float32
                or _expanded_edges_pay(int(relation.n_kernels), c_in, c_out)):
            return False
    elif (relation.holds_edges and relation.sorted_implicit_gemm is None
            and edges_pay(c_in, c_out, feats.element_size(),
                          relation.n_out_capacity)):
        return False
    return _padded_eligible(feats, c_out, relation, relation.n_out_capacity)


def _weight_fits(weight: torch.Tensor, dtype: torch.dtype, c_in: int,
                 c_out: int, relation: KernelRelation) -> bool:
    """Whether the weight is that of a conv of these channels over the
    relation.  The padded conv takes the weight as fragments, whose size does
    not tell: any other weight goes to the entry that says what is wrong."""
    if weight.ndim not in (3, 5) or weight.dtype != dtype:
        return False
    shape = tuple(weight.shape)
    if weight.ndim == 3:
        return shape == (relation.n_kernels, c_in, c_out)
    return (shape[0] == c_out and shape[4] == c_in
            and shape[1] * shape[2] * shape[3] == relation.n_kernels)


def _offset_bytes(weight: torch.Tensor) -> int:
    """Bytes of the weight of one offset."""
    c_in = weight.shape[1] if weight.ndim == 3 else weight.shape[4]
    c_out = weight.shape[2] if weight.ndim == 3 else weight.shape[0]
    return int(c_in) * int(c_out) * weight.element_size()


def _padded_conv(feats, weight, role, view, rows, relation, bias=None,
                 relu=False) -> torch.Tensor:
    """The padded conv over ``weight`` as it is now, or (``role``) over its
    input gradient's weight: the kernel's order of it is made in the call."""
    return ext.sparse_conv_padded(
        feats, weight, role, view.sorted_kv_out_in_map, view.reorder_rows,
        view.tile_masks, rows, relation.n_kernels, bias=bias,
        tile_order=view.tile_order(), relu=relu)


_EXPAND_CHANNELS = (32, 64, 128, 256)


def _expand_eligible(feats: torch.Tensor, c_out: int,
                     relation: KernelRelation) -> bool:
    """A direct expanded relation (output row in * K + k = the single edge
    (in, k)) runs as a dense matrix-core GEMM without gathers."""
    return (relation.direct_expansion
            and relation.source_active_rows is not None
            and feats.dtype in (torch.float16, torch.bfloat16)
            and int(feats.shape[1]) in _EXPAND_CHANNELS
            and c_out in _EXPAND_CHANNELS
            and int(feats.shape[1]) * c_out <= 16384
            and relation.n_in_capacity == int(feats.shape[0])
            and relation.n_out_capacity
            == int(feats.shape[0]) * int(relation.n_kernels))


def sparse_conv_features_from_relation(feats: torch.Tensor,
                                       weight: torch.Tensor,
                                       relation: KernelRelation,
                                       bias: torch.Tensor | None = None,
                                       relu: bool = False,
                                       ) -> torch.Tensor:
    """Execute sparse convolution over a prebuilt relation
    (_relation_exec.py:84-116).  Differentiable in ``feats`` and ``weight``:
    the backward pass is the reference primitive's vjp
    (native/features/convolution/primitive.cpp:137-176).  ``relu`` fuses a
    ReLU after the bias into the store (the operators pass it only when
    autograd does not need the activation)."""
    _require_static(relation)
    if feats.requires_grad or weight.requires_grad:
        # (an evaluation of trainable layers too: a graph captured later
        # cannot read what was not copied before)
        relation.expect_backward()
    if torch.is_grad_enabled() and (feats.requires_grad
                                    or weight.requires_grad
                                    or (bias is not None
                                        and bias.requires_grad)):
        if relu:
            raise ValueError('a fused ReLU is not differentiable; apply it '
                             'separately when gradients are needed.')
        out = _SparseConvFeatures.apply(feats, weight, relation)
        return out if bias is None else _add_bias(out, bias)
    return _conv_features(feats, weight, relation, bias, relu)


def _add_bias(feats: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    if bias.ndim != 1:
        raise ValueError('bias must have shape (C_out,).')
    if bias.shape[0] != feats.shape[1]:
        raise ValueError('bias channels must match output channels.')
    if bias.dtype != feats.dtype:
        raise ValueError('bias dtype must match output features.')
    return feats + bias


class _SparseConvFeatures(torch.autograd.Function):
    """Sparse conv features with the reference's gradients
    (cpu/algorithms.cpp:355-481): the input gradient over the transposed or
    mirrored relation or the input-grouped CSR, the weight gradient over the
    edges grouped by offset."""

    @staticmethod
    def forward(ctx, feats, weight, relation):
        ctx.relation = relation
        ctx.save_for_backward(feats, weight)
        return _conv_features(feats, weight, relation)

    @staticmethod
    def backward(ctx, grad_out):
        feats, weight = ctx.saved_tensors
        relation = ctx.relation
        grad_out = grad_out.contiguous()
        grad_feats = grad_weight = None
        if ctx.needs_input_grad[0]:
            grad_feats = sparse_conv_input_grad_from_relation(
                grad_out, weight, relation, int(feats.shape[0]))
        if ctx.needs_input_grad[1]:
            grad_weight = sparse_conv_weight_grad_from_relation(
                feats, grad_out, weight, relation)
        return grad_feats, grad_weight, None


def _input_grad_matrix_core_eligible(cot: torch.Tensor, weight: torch.Tensor,
                                     relation: KernelRelation) -> bool:
    """The input gradient is the forward's implicit GEMM over the
    transposed relation: its contraction runs over C_out and it writes C_in
    columns."""
    c_in = int(weight.shape[1] if weight.ndim == 3 else weight.shape[4])
    c_out = int(cot.shape[1])
    return (relation.kind != 'target'
            and cot.dtype in (torch.float16, torch.bfloat16)
            and c_out % 32 == 0 and c_out <= 512
            and c_in in _MATRIX_CORE_C_OUT
            and relation.n_kernels is not None and relation.n_kernels <= 32
            and int(cot.shape[0]) * c_out * 2 < 2 ** 31
            # a repeated coordinate gives an input row several output rows
            # at one offset, which the dense transposed map cannot hold
            and relation.transposed_map_exact)


def _transposed_weight(weight: torch.Tensor) -> torch.Tensor:
    """(C_out, Kx, Ky, Kz, C_in) or (K, C_in, C_out) -> the 5D weight of the
    transposed conv, (C_in, Kx, Ky, Kz, C_out) (cached)."""
    def make(w):
        if w.ndim == 5:
            return w.permute(4, 1, 2, 3, 0).contiguous()
        k, c_in, c_out = w.shape
        return w.permute(1, 0, 2).contiguous().reshape(c_in, k, 1, 1, c_out)

    return _cached_weight(weight, 'transposed', make)


def _mirrored_weight(weight: torch.Tensor) -> torch.Tensor:
    """The transposed weight with its offsets reversed, W'[j] = W[K-1-j]^T,
    as a 5D (C_in, Kx, Ky, Kz, C_out) weight (cached)."""
    def make(w):
        if w.ndim == 5:
            return w.flip(1, 2, 3).permute(4, 1, 2, 3, 0).contiguous()
        k, c_in, c_out = w.shape
        return w.flip(0).permute(1, 0, 2).contiguous().reshape(
            c_in, k, 1, 1, c_out)

    return _cached_weight(weight, 'mirrored', make)


def _mirror_symmetric(relation: KernelRelation) -> bool:
    """A submanifold relation whose offsets come in opposite pairs,
    offset[K-1-k] = -offset[k] (odd kernels), and whose coordinates do not
    repeat: input row i then meets output row o at offset k exactly when
    o = out_in_map[i][K-1-k], so the transposed map is the forward map with
    its offsets reversed."""
    if relation.kind != 'submanifold':
        return False
    offs = relation.kernel_offsets
    k = len(offs)
    return k > 0 and all(
        tuple(-v for v in offs[k - 1 - j]) == tuple(offs[j]) for j in range(k))


def sparse_conv_input_grad_from_relation(cot: torch.Tensor,
                                         weight: torch.Tensor,
                                         relation: KernelRelation,
                                         in_capacity: int) -> torch.Tensor:
    """Input gradient ``(in_capacity, C_in)`` (make_sparse_conv_features_
    input_grad, primitive.cpp:597-639): on the matrix cores when the shapes
    allow, otherwise over the input-grouped CSR.  A submanifold relation
    over distinct coordinates runs the forward's own sorted view with the
    mirrored transposed weight (grad[i] = sum_j cot[out_in_map[i][j]] @
    W[K-1-j]^T); other relations run their transposed sorted view."""
    _require_static(relation)
    if _input_grad_matrix_core_eligible(cot, weight, relation):
        if _mirror_symmetric(relation):
            view = relation.conv_view(_offset_bytes(weight))
            mirrored = _mirrored_weight(weight)
            return ext.sparse_conv_features_sorted_implicit_gemm(
                cot, mirrored, view.sorted_out_in_map,
                view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
                None, None, None, None, None, None, None, None, None,
                in_capacity, relation.n_kernels, tile_order=view.tile_order(),
                weight_fragments=_weight_fragments(mirrored))
        view = relation.transposed_conv_view(_offset_bytes(weight))
        transposed = _transposed_weight(weight)
        return ext.sparse_conv_features_sorted_implicit_gemm(
            cot, transposed, view.sorted_out_in_map,
            view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
            None, None, None, None, None, None, None, None, None,
            in_capacity, relation.n_kernels, tile_order=view.tile_order(),
            weight_fragments=_weight_fragments(transposed))
    c_in = int(weight.shape[1] if weight.ndim == 3 else weight.shape[4])
    if (relation.kind != 'target'
            and _weight_fits(weight, cot.dtype, c_in, int(cot.shape[1]),
                             relation)
            and relation.transposed_map_exact
            and _padded_eligible(cot, c_in, relation, in_capacity)):
        mirrored = _mirror_symmetric(relation)
        size = _offset_bytes(weight)
        view = (relation.conv_view(size) if mirrored
                else relation.transposed_conv_view(size))
        return _padded_conv(cot, weight,
                            _MIRRORED if mirrored else _TRANSPOSED, view,
                            in_capacity, relation)
    input_csr = relation.input_csr
    return ext.sparse_conv_input_grad(
        cot, weight, relation.edges.out_rows, relation.edges.kernel_ids,
        relation.counts, input_csr.row_offsets, input_csr.edge_ids,
        in_capacity, relation.n_kernels)


def sparse_conv_weight_grad_from_relation(feats: torch.Tensor,
                                          cot: torch.Tensor,
                                          weight: torch.Tensor,
                                          relation: KernelRelation,
                                          ) -> torch.Tensor:
    """Weight gradient in ``weight``'s shape (make_sparse_conv_features_
    weight_grad, primitive.cpp:641-680) over the edges grouped by offset
    (pairs where the relation groups without a sort, else the CSR)."""
    _require_static(relation)
    pairs = relation.kernel_pairs()
    if pairs is not None:
        return ext.sparse_conv_weight_grad_pairs(
            feats, cot, weight, pairs[1], pairs[0], relation.n_kernels)
    kernel_csr = relation.kernel_csr
    return ext.sparse_conv_weight_grad(
        feats, cot, weight, relation.edges.in_rows, relation.edges.out_rows,
        relation.counts, kernel_csr.row_offsets, kernel_csr.edge_ids,
        relation.n_kernels)


def _conv_features(feats: torch.Tensor, weight: torch.Tensor,
                   relation: KernelRelation,
                   bias: torch.Tensor | None = None,
                   relu: bool = False) -> torch.Tensor:
    """Forward features on the matrix-core or the CSR route; ``bias``
    (optional) is added in the kernels' store, after the conv result is
    rounded, exactly as a separate ``feats + bias``; ``relu`` then applies
    ``maximum(v, 0)`` in the same store."""
    c_out = int(weight.shape[2] if weight.ndim == 3 else weight.shape[0])
    if feats.ndim == 2 and _expand_eligible(feats, c_out, relation):
        return ext.sparse_conv_features_expand(
            feats, weight, relation.source_active_rows,
            relation.n_kernels, bias=bias, relu=relu)
    if feats.ndim == 2 and _matrix_core_eligible(
            feats.dtype, int(feats.shape[1]), c_out, relation,
            int(feats.shape[0])):
        return sparse_conv_features_sorted_from_relation(feats, weight,
                                                         relation, bias=bias,
                                                         relu=relu)
    dense = (_small_dense_map(feats.dtype, int(feats.shape[1]), c_out,
                              relation) if feats.ndim == 2 else None)
    if (dense is None and feats.ndim == 2
            and _weight_fits(weight, feats.dtype, int(feats.shape[1]), c_out,
                             relation)
            and _padded_forward(feats, int(feats.shape[1]), c_out, relation)):
        return _padded_conv(feats, weight, _FORWARD,
                            relation.conv_view(_offset_bytes(weight)),
                            relation.n_out_capacity, relation, bias, relu)
    if _dense_without_edges(feats, dense):
        in_rows = kernel_ids = row_offsets = None
    else:
        edges = relation.edges
        in_rows, kernel_ids = edges.in_rows, edges.kernel_ids
        row_offsets = relation.output_csr.row_offsets
    return ext.sparse_conv_features_csr(
        feats, weight, in_rows, kernel_ids, relation._contract.counts,
        row_offsets, relation.n_out_capacity, relation.n_kernels, bias=bias,
        relu=relu, out_in_map=dense)


def sparse_conv_features_sorted_from_relation(feats: torch.Tensor,
                                              weight: torch.Tensor,
                                              relation: KernelRelation, *,
                                              store_sorted: bool = False,
                                              bias: torch.Tensor | None = None,
                                              relu: bool = False,
                                              ) -> torch.Tensor:
    """Matrix-core implicit GEMM over the sorted view
    (_relation_exec.py:119-156)."""
    _require_static(relation)
    c_out = int(weight.shape[2] if weight.ndim == 3 else weight.shape[0])
    if not _matrix_core_eligible(feats.dtype, int(feats.shape[1]), c_out,
                                 relation, int(feats.shape[0])):
        raise ValueError(
            'sorted implicit GEMM is not supported for this relation, '
            'feature tensor, or weight tensor.')
    # rows stored in sorted order need the sorted view
    view = (relation.require_sorted_implicit_gemm() if store_sorted
            else relation.conv_view(_offset_bytes(weight)))
    w5 = _matrix_core_weight(weight)
    return ext.sparse_conv_features_sorted_implicit_gemm(
        feats, w5, view.sorted_out_in_map,
        view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
        None, None, None, None, None, None, None, None, None,
        relation.n_out_capacity, relation.n_kernels,
        store_sorted=store_sorted, bias=bias, tile_order=view.tile_order(),
        relu=relu, weight_fragments=_weight_fragments(w5))


def sparse_quantized_conv_features_from_relation(
        feats: torch.Tensor, weight: QuantizedWeight,
        relation: KernelRelation,
        bias: torch.Tensor | None = None,
        relu: bool = False) -> torch.Tensor:
    """Quantized sparse convolution over a prebuilt relation
    (_relation_exec.py:19-61); the sorted plan is passed when the matrix-core
    route applies.  ``bias`` and ``relu`` are fused into the store."""
    _require_static(relation)
    if relation.n_kernels != weight.weight.shape[0]:
        raise ValueError('quantized weight kernel rows must match the relation.')
    device = feats.device
    kv = reorder = tiles = _empty_i32(device)
    order = fragments = None
    dense = None
    mapped = False
    if _matrix_core_eligible(feats.dtype, weight.in_channels,
                             weight.out_channels, relation,
                             int(feats.shape[0])):
        view = relation.conv_view(
            weight.in_channels * weight.out_channels * 2)
        kv = view.sorted_kv_out_in_map
        reorder = view.reorder_rows
        tiles = view.tile_masks
        order = view.tile_order()
        fragments = _quantized_fragments(weight)
        # an empty view (no rows) is no plan, and a shape without fragments
        # runs the entry that takes the edges
        mapped = relation.n_out_capacity > 0 and fragments.numel() > 0
    else:
        dense = _small_dense_map(feats.dtype, weight.in_channels,
                                 weight.out_channels, relation)
        if (dense is None and feats.dtype != torch.float32
                and feats.ndim == 2
                and int(feats.shape[1]) == weight.in_channels
                and feats.dtype == weight.scales.dtype
                and _padded_forward(feats, weight.in_channels,
                                    weight.out_channels, relation)):
            view = relation.conv_view(
                weight.in_channels * weight.out_channels * 2)
            return ext.sparse_quantized_conv_padded(
                feats, weight.weight, weight.scales, weight.biases,
                weight.in_channels, weight.out_channels,
                weight.storage_in_channels, weight.group_size, weight.bits,
                view.sorted_kv_out_in_map, view.reorder_rows, view.tile_masks,
                relation.n_out_capacity, relation.n_kernels, bias=bias,
                tile_order=view.tile_order(), relu=relu)
        mapped = _dense_without_edges(feats, dense)
    if mapped:
        in_rows = out_rows = kernel_ids = row_offsets = None
    else:
        edges = relation.edges
        in_rows, out_rows, kernel_ids = (edges.in_rows, edges.out_rows,
                                         edges.kernel_ids)
        row_offsets = relation.output_csr.row_offsets
    return ext.sparse_quantized_conv_features(
        feats, weight.weight, weight.scales, weight.biases, in_rows,
        out_rows, kernel_ids, relation._contract.counts, row_offsets, kv,
        reorder, tiles,
        relation.n_out_capacity, relation.n_kernels, weight.in_channels,
        weight.out_channels, weight.storage_in_channels, weight.group_size,
        weight.bits, bias=bias, tile_order=order, relu=relu,
        weight_fragments=fragments,
        out_in_map=dense)


def sparse_pool_features_from_relation(feats: torch.Tensor,
                                       relation: KernelRelation, *,
                                       input_exclusive: bool,
                                       mode: str) -> torch.Tensor:
    """Sparse pooling over a prebuilt kernel relation
    (_relation_exec.py:253-276), differentiable in ``feats``."""
    _require_static(relation)
    if torch.is_grad_enabled() and feats.requires_grad:
        return _SparsePoolFeatures.apply(feats, relation, input_exclusive,
                                         mode)
    return _pool_features(feats, relation, input_exclusive, mode)


def _pool_features(feats, relation, input_exclusive, mode):
    return ext.sparse_pool_features(
        feats, relation.edges.in_rows, relation.edges.out_rows,
        relation.edges.kernel_ids, relation.output_csr.row_offsets,
        relation.counts, input_exclusive, mode, relation.n_out_capacity,
        relation.n_kernels)


class _SparsePoolFeatures(torch.autograd.Function):
    """Pooling with the reference's vjp (pooling/primitive.cpp:109-160):
    max routes the cotangent to the inputs equal to the pooled value, split
    over ties.  A relation whose inputs feed at most one output each writes
    it from the output rows; others walk the input-grouped CSR."""

    @staticmethod
    def forward(ctx, feats, relation, input_exclusive, mode):
        pooled = _pool_features(feats, relation, input_exclusive, mode)
        ctx.relation = relation
        ctx.mode = mode
        ctx.input_exclusive = input_exclusive
        ctx.save_for_backward(feats, pooled)
        return pooled

    @staticmethod
    def backward(ctx, grad_out):
        feats, pooled = ctx.saved_tensors
        relation = ctx.relation
        active = relation.source_active_rows
        if ctx.input_exclusive and active is not None:
            grad = ext.sparse_pool_features_grad_exclusive(
                grad_out.contiguous(), feats, pooled, relation.edges.in_rows,
                relation.output_csr.row_offsets, relation.counts, active,
                ctx.mode)
            return grad, None, None, None
        input_csr = relation.input_csr
        grad = ext.sparse_pool_features_grad(
            grad_out.contiguous(), feats, pooled, relation.edges.in_rows,
            relation.edges.out_rows, relation.output_csr.row_offsets,
            relation.counts, input_csr.row_offsets, input_csr.edge_ids,
            ctx.mode)
        return grad, None, None, None


def _cached_weight(weight: torch.Tensor, kind: str, make) -> torch.Tensor:
    """``make(weight)``, cached by the weight's identity, storage, shape,
    dtype and version counter (so an in-place update, as an optimizer step
    makes, and an assignment to ``.data`` rebuild it; a write through
    ``.data`` is not seen), like the reference's ``_mapped_weight``
    (_relation_exec.py:217-250)."""
    key = (id(weight), kind)
    state = (weight.data_ptr(), tuple(weight.shape), weight.dtype,
             weight._version)
    cached = _WEIGHT_CACHE.get(key)
    if cached is not None and cached[0]() is weight and cached[1] == state:
        return cached[2]
    value = make(weight)

    def _drop(ref, key=key):
        entry = _WEIGHT_CACHE.get(key)
        if entry is not None and entry[0] is ref:
            _WEIGHT_CACHE.pop(key, None)

    _WEIGHT_CACHE[key] = (weakref.ref(weight, _drop), state, value)
    return value


def _weight_fragments(weight5d: torch.Tensor) -> torch.Tensor:
    """The streamed matrix-core conv's fragment-ordered copy of a 5D
    fp16/bf16 weight (``ext.conv_weight_fragments``; empty when the shape
    takes the other matrix-core kernel), cached with the weight."""
    return _cached_weight(weight5d, 'fragments', ext.conv_weight_fragments)


def _quantized_fragments(weight: QuantizedWeight) -> torch.Tensor:
    """The streamed matrix-core conv's fragment-ordered packed copy of a
    quantized weight (``ext.quantized_weight_fragments``: codes, scale and
    bias per 16-byte piece, dequantised in the kernel; empty when the shape
    takes the other matrix-core kernel), cached with the packed words and
    rebuilt when they, the scales or the biases change."""
    kind = ('quantized fragments',
            *((id(t), t.data_ptr(), t._version)
              for t in (weight.scales, weight.biases)))

    def make(words):
        return ext.quantized_weight_fragments(
            words, weight.scales, weight.biases, weight.in_channels,
            weight.out_channels, weight.storage_in_channels,
            weight.group_size, weight.bits)

    return _cached_weight(weight.weight, kind, make)


def _matrix_core_weight(weight: torch.Tensor) -> torch.Tensor:
    """5D weights go to the kernels as they are (C_in contiguous per
    (C_out, k)); a mapped ``(K, C_in, C_out)`` weight is transposed once to
    ``(C_out, K, 1, 1, C_in)`` and cached."""
    if weight.ndim == 5:
        return weight

    def make(w):
        k, c_in, c_out = w.shape
        return w.permute(2, 0, 1).contiguous().reshape(c_out, k, 1, 1, c_in)

    return _cached_weight(weight, 'mapped', make)
