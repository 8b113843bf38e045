"""Kernel relation contract and its execution views over torch tensors.

Mirrors mlx_lattice/core/relations/views.py (RelationEdges :19-45,
RelationCSRView :48-62, RelationImplicitGemmView :68-101,
RelationSortedImplicitGemmView :104-146, SparseRelationContract :149-236,
KernelRelation :259-525).  Every array is an int32 torch tensor on the
relation's device; counts stay on the device.
"""

from __future__ import annotations

import threading
from collections.abc import Callable
from dataclasses import dataclass, field, fields, is_dataclass
from typing import Literal

import torch

from mlx_lattice_amd import _native
from mlx_lattice_amd.core.types import Triple

RelationKind = Literal['forward', 'target', 'submanifold', 'transposed',
                       'generative']

_INDEX_DTYPES = (torch.int32, torch.int64)
# Rows whose 128-row tiles all start at once, one per CU.
_ONE_ROUND_ROWS = 256 * 128
# Rows, weight bytes per offset and their product up to which convs take the
# rows in their own order (conv_view).
_TILED_ROWS = 32768
_TILED_WEIGHT_BYTES = 16384
_TILED_WORK = 16384 * 16384
_KEEP_LOCK = threading.RLock()


def _arrays(value) -> list[torch.Tensor]:
    """The tensors of a tensor, view or tuple of them."""
    if isinstance(value, torch.Tensor):
        return [value]
    if isinstance(value, tuple):
        return [t for item in value for t in _arrays(item)]
    if is_dataclass(value):
        return [t for f in fields(value)
                for t in _arrays(getattr(value, f.name))]
    return []


def _kept(holder, name: str, device: torch.device, make: Callable):
    """``holder.name``, device arrays that ``make`` builds on their first
    use.  They are kept with the stream that wrote them, and another stream's
    first use of them waits for it.  Under graph capture nothing is kept (the
    arrays hold values only once the graph runs) but for the rest of that
    capture's work on the stream; arrays made before a capture are used as
    they are.  ``holder._written`` holds the streams ordered after each
    array's writes, the writer first; a value given at construction is not in
    it."""
    value = getattr(holder, name)
    if device.type != 'cuda':
        if value is None:
            value = make()
            object.__setattr__(holder, name, value)
        return value
    ext = _native.ext
    written = holder._written
    if value is not None:
        streams = written.get(name)
        if streams is None or ext.current_stream(device.index) in streams:
            return value
        stream, capture = ext.stream_state(device.index)
        if capture:
            return value
        if not ext.join_stream(device.index, streams[0]):
            return make()   # the writer is being captured: nothing to wait for
        current = torch.cuda.current_stream(device)
        for array in _arrays(value):
            array.record_stream(current)
        written[name] = (*streams, stream)
        return value
    stream, capture = ext.stream_state(device.index)
    if capture:
        captured = written.get((name, 'captured'))
        if captured is None or captured[:2] != (stream, capture):
            captured = (stream, capture, make())
            written[name, 'captured'] = captured
        return captured[2]
    with _KEEP_LOCK:
        if getattr(holder, name) is None:
            value = make()
            written[name] = (stream,)
            object.__setattr__(holder, name, value)
            return value
    return _kept(holder, name, device, make)   # another thread made it


@dataclass(frozen=True, slots=True)
class RelationEdges:
    """Edge arrays ``(in_row, out_row, kernel_id)`` at the same index."""

    in_rows: torch.Tensor
    out_rows: torch.Tensor
    kernel_ids: torch.Tensor

    def __post_init__(self) -> None:
        _validate_row_array(self.in_rows, name='in_rows')
        _validate_row_array(self.out_rows, name='out_rows')
        _validate_row_array(self.kernel_ids, name='kernel_ids')
        _require_same_rows(self.in_rows, self.out_rows, self.kernel_ids,
                           names=('in_rows', 'out_rows', 'kernel_ids'))

    @property
    def capacity(self) -> int:
        return int(self.in_rows.shape[0])


@dataclass(frozen=True, slots=True)
class RelationCSRView:
    """CSR view: ``row_offsets`` ``(rows + 1,)`` int32 and optional
    ``edge_ids`` remapping CSR order to the canonical edge arrays."""

    row_offsets: torch.Tensor
    edge_ids: torch.Tensor | None = None

    def __post_init__(self) -> None:
        _validate_row_offsets(self.row_offsets)
        if self.edge_ids is not None:
            _validate_row_array(self.edge_ids, name='edge_ids')


RelationView = RelationCSRView


@dataclass(frozen=True, slots=True)
class RelationImplicitGemmView:
    """Dense ``out_in_map[o, k]`` (input row or -1) plus ``row_masks``
    (bit k%32 of word k/32 set when offset k contributes)."""

    out_in_map: torch.Tensor
    row_masks: torch.Tensor

    def __post_init__(self) -> None:
        if self.out_in_map.ndim != 2:
            raise ValueError('out_in_map must have shape (Nout, K).')
        if self.out_in_map.dtype not in _INDEX_DTYPES:
            raise ValueError('out_in_map must be int32 or int64.')
        if self.row_masks.ndim != 2:
            raise ValueError('row_masks must have shape (Nout, M).')
        if self.row_masks.dtype not in _INDEX_DTYPES:
            raise ValueError('row_masks must be int32 or int64.')
        if int(self.row_masks.shape[0]) != int(self.out_in_map.shape[0]):
            raise ValueError('row_masks must have one row per out_in_map row.')
        expected = (int(self.out_in_map.shape[1]) + 31) // 32
        if int(self.row_masks.shape[1]) != expected:
            raise ValueError(
                'row_masks must have ceil(K / 32) words per output row.')


@dataclass(frozen=True, slots=True)
class RelationSortedImplicitGemmView:
    """Mask-sorted implicit-GEMM view consumed by the matrix-core route."""

    sorted_out_in_map: torch.Tensor
    sorted_kv_out_in_map: torch.Tensor
    reorder_rows: torch.Tensor
    tile_masks: torch.Tensor
    _tile_order: torch.Tensor | None = field(default=None, compare=False,
                                             repr=False)
    _written: dict = field(default_factory=dict, init=False, compare=False,
                           repr=False)

    def __post_init__(self) -> None:
        if self.sorted_out_in_map.ndim != 2:
            raise ValueError('sorted_out_in_map must have shape (Nout, K).')
        if self.sorted_kv_out_in_map.ndim != 2:
            raise ValueError('sorted_kv_out_in_map must have shape (K, Nout).')
        if (int(self.sorted_kv_out_in_map.shape[0])
                != int(self.sorted_out_in_map.shape[1])
                or int(self.sorted_kv_out_in_map.shape[1])
                != int(self.sorted_out_in_map.shape[0])):
            raise ValueError('sorted_kv_out_in_map must be the K-major view '
                             'of sorted_out_in_map.')
        _validate_row_array(self.reorder_rows, name='reorder_rows')
        _validate_row_array(self.tile_masks, name='tile_masks')
        if int(self.reorder_rows.shape[0]) != int(
                self.sorted_out_in_map.shape[0]):
            raise ValueError(
                'reorder_rows must have one row per sorted_out_in_map row.')

    def tile_order(self) -> torch.Tensor | None:
        """Longest-first order of the view's 128-row tiles for the
        matrix-core conv, computed on first use and kept with the view so
        repeated convs over it skip their per-call schedule; None when the
        tiles all start at once."""
        if int(self.reorder_rows.shape[0]) <= _ONE_ROUND_ROWS:
            return None
        return _kept(self, '_tile_order', self.tile_masks.device,
                     self._order_tiles)

    def _order_tiles(self) -> torch.Tensor:
        from mlx_lattice_amd._native import ext

        return ext.conv_tile_order(self.tile_masks,
                                   int(self.reorder_rows.shape[0]))


class _StatusWord:
    """A device status word copied to pinned host memory when the relation
    is built, or by queue() (``deferred``) once something is known to ask
    for it: the copy is queued on the current stream and never waited for
    there; read() waits only for the copy's event (usually long complete by
    the time a backward pass asks)."""

    __slots__ = ('_device', '_word')

    def __init__(self, word: torch.Tensor, deferred: bool = False) -> None:
        self._device = word
        self._word = None
        if not deferred:
            self.queue()

    @property
    def unreadable(self) -> bool:
        """Not queued, and under a graph capture, where nothing can be read."""
        return (self._word is None and self._device.is_cuda
                and torch.cuda.is_current_stream_capturing())

    def queue(self) -> None:
        if self._word is not None:
            return
        if self._device.is_cuda:
            from mlx_lattice_amd._native import ext

            self._word = ext.StatusWord(self._device)
        else:
            self._word = self._device.clone()

    def read(self) -> int:
        """The word's value.  Raises RuntimeError when the builder's
        coordinate table overflowed (lattice_relation_flags bit 16): the
        table is sized above its key count, so this marks a sizing error
        and the relation's contents are void."""
        self.queue()
        value = (int(self._word[0]) if isinstance(self._word, torch.Tensor)
                 else self._word.read())
        if value & 16:
            raise RuntimeError('relation build: the coordinate table '
                               'overflowed (status word bit 16); the '
                               'relation is invalid.')
        return value


class _MapEdges:
    """The edges and their row offsets of a relation built as a dense map
    alone, made from the map and its masks on first use (``_kept``)."""

    __slots__ = ('_view', '_counts', '_made', '_written')

    def __init__(self, view: RelationImplicitGemmView,
                 counts: torch.Tensor) -> None:
        self._view = view
        self._counts = counts
        self._made = None
        self._written = {}

    @property
    def capacity(self) -> int:
        return int(self._view.out_in_map.numel())

    def get(self) -> tuple[RelationEdges, RelationCSRView]:
        return _kept(self, '_made', self._counts.device, self._make)

    def _make(self) -> tuple[RelationEdges, RelationCSRView]:
        from mlx_lattice_amd._native import ext

        *edges, row_offsets = ext.build_map_edges(
            self._view.out_in_map, self._view.row_masks, self._counts)
        return RelationEdges(*edges), RelationCSRView(row_offsets)


@dataclass(frozen=True, slots=True)
class SparseRelationContract:
    """Counts, capacities, coordinate context and geometry of a relation."""

    counts: torch.Tensor
    kernel_offsets: tuple[Triple, ...]
    out_coords: torch.Tensor | None = None
    n_in_capacity: int | None = None
    n_out_capacity: int | None = None
    n_kernels: int | None = None
    source_coords: torch.Tensor | None = None
    source_active_rows: torch.Tensor | None = None
    target_coords: torch.Tensor | None = None
    target_active_rows: torch.Tensor | None = None
    stride: Triple = (1, 1, 1)
    padding: Triple = (0, 0, 0)
    kind: RelationKind = 'forward'
    # One view object per count: a strided output tensor is keyed in its
    # coordinate manager by the identity of its active-row array, so handing
    # out the same view lets repeated calls reuse the output's relations.
    _edge_count: torch.Tensor = field(init=False, repr=False, compare=False)
    _out_count: torch.Tensor = field(init=False, repr=False, compare=False)

    def __post_init__(self) -> None:
        _validate_counts(self.counts)
        object.__setattr__(self, '_edge_count', self.counts[:1])
        object.__setattr__(self, '_out_count', self.counts[1:2])
        for name in ('out_coords', 'source_coords', 'target_coords'):
            value = getattr(self, name)
            if value is not None:
                _validate_coords(value, name=name)
        for name in ('source_active_rows', 'target_active_rows'):
            value = getattr(self, name)
            if value is not None:
                _validate_active_rows(value, name=name)
        if self.kind not in ('forward', 'target', 'submanifold',
                             'transposed', 'generative'):
            raise ValueError(
                "relation kind must be 'forward', 'target', "
                "'submanifold', 'transposed', or 'generative'.")
        offsets = _int_offsets(self.kernel_offsets)
        object.__setattr__(self, 'kernel_offsets', offsets)
        object.__setattr__(self, 'stride', tuple(map(int, self.stride)))
        object.__setattr__(self, 'padding', tuple(map(int, self.padding)))
        n_in = _optional_count(self.n_in_capacity, 'n_in_capacity')
        n_out = _optional_count(self.n_out_capacity, 'n_out_capacity')
        n_kernels = _optional_count(self.n_kernels, 'n_kernels')
        if offsets:
            if n_kernels is not None and n_kernels != len(offsets):
                raise ValueError('n_kernels must match kernel_offsets.')
            n_kernels = len(offsets)
        if self.out_coords is not None:
            out_capacity = int(self.out_coords.shape[0])
            if n_out is not None and n_out != out_capacity:
                raise ValueError(
                    'n_out_capacity must match out_coords capacity.')
            n_out = out_capacity
        object.__setattr__(self, 'n_in_capacity', n_in)
        object.__setattr__(self, 'n_out_capacity', n_out)
        object.__setattr__(self, 'n_kernels', n_kernels)

    @property
    def edge_count(self) -> torch.Tensor:
        return self._edge_count

    @property
    def out_count(self) -> torch.Tensor:
        return self._out_count


@dataclass(frozen=True, slots=True, init=False)
class KernelRelation:
    """Sparse kernel relation with edge, CSR and implicit-GEMM views."""

    _contract: SparseRelationContract
    _edges: RelationEdges | None
    _output_csr: RelationCSRView | None
    # Relations built as a dense map alone: makes the edges, the row offsets
    # and the edge count on their first use.
    _map_edges: _MapEdges | None
    _input_csr: RelationCSRView | None
    _kernel_csr: RelationCSRView | None
    # The (input, kernel) CSR views when `_grouped_views` makes them.
    _grouped: tuple[RelationCSRView, RelationCSRView] | None
    _grouped_views: Callable[..., tuple] | None
    # Builds the edges grouped by offset without a sort (dense-map relations
    # of at most 32 offsets): the edge ids when called with the row offsets,
    # else the (input row, output row) pairs.
    _kernel_groups: Callable[[torch.Tensor | None], tuple] | None
    _kernel_grouped: RelationCSRView | None
    _kernel_pairs: tuple[torch.Tensor, torch.Tensor] | None
    _written: dict = field(compare=False, repr=False)
    implicit_gemm: RelationImplicitGemmView | None = None
    sorted_implicit_gemm: RelationSortedImplicitGemmView | None = None
    transposed_sorted_implicit_gemm: RelationSortedImplicitGemmView | None = None
    # The unsorted views of small relations (conv_view).
    _tiled: RelationSortedImplicitGemmView | None = None
    _transposed_tiled: RelationSortedImplicitGemmView | None = None
    # Transposed relations only: whether two edges share (out_row, kernel_id)
    # (a repeated input coordinate).  The builder hands over its device
    # status word, copied to pinned memory at build time (a _StatusWord) and
    # read on the first question (dense_map_exact), so building the relation
    # never waits for the device.  None: unknown.
    repeated_edges: bool | _StatusWord | None = None
    # Generative, and transposed relations whose stride exceeds the offsets'
    # extent: output row in * K + k holds the single edge (in, k).
    direct_expansion: bool = False
    # Submanifold relations, and forward ones of unit stride without padding:
    # whether an active row repeats an earlier row's coordinate (each copy is an output row with the same neighbours, so
    # an input row can have several output rows at one offset).  Held as a
    # _StatusWord copied to pinned memory when a conv of trainable features
    # or weights runs (expect_backward) and read on the first question
    # (transposed_map_exact).  None: no repeats possible.
    repeated_coords: bool | _StatusWord | None = None
    # Submanifold relations built with their workspace: it starts with the
    # block table of the coordinates (the coordinate manager hands it to
    # the next forward relation over the same key).
    block_table: torch.Tensor | None = None

    def __init__(
        self,
        in_rows: torch.Tensor | None,
        out_rows: torch.Tensor | None,
        kernel_ids: torch.Tensor | None,
        *,
        row_offsets: torch.Tensor | None = None,
        counts: torch.Tensor | None = None,
        in_row_offsets: torch.Tensor | None = None,
        in_edge_ids: torch.Tensor | None = None,
        kernel_row_offsets: torch.Tensor | None = None,
        kernel_edge_ids: torch.Tensor | None = None,
        kernel_offsets: tuple[Triple, ...] = (),
        out_coords: torch.Tensor | None = None,
        n_in_capacity: int | None = None,
        n_out_capacity: int | None = None,
        n_kernels: int | None = None,
        source_coords: torch.Tensor | None = None,
        source_active_rows: torch.Tensor | None = None,
        target_coords: torch.Tensor | None = None,
        target_active_rows: torch.Tensor | None = None,
        stride: Triple = (1, 1, 1),
        padding: Triple = (0, 0, 0),
        kind: RelationKind = 'forward',
        implicit_gemm: RelationImplicitGemmView | None = None,
        sorted_implicit_gemm: RelationSortedImplicitGemmView | None = None,
        grouped_views: Callable[..., tuple] | None = None,
        kernel_groups: Callable[[torch.Tensor | None], tuple] | None = None,
        repeated_edges: bool | torch.Tensor | None = None,
        direct_expansion: bool = False,
        repeated_coords: torch.Tensor | None = None,
        block_table: torch.Tensor | None = None,
    ) -> None:
        """``grouped_views``, when given and the input/kernel CSR arrays are
        not, is called on first access of ``input_csr`` / ``kernel_csr`` and
        returns ``(in_row_offsets, in_edge_ids, kernel_row_offsets,
        kernel_edge_ids)``; the forward convolution never reads those
        views, so they are only built for consumers that do.
        ``kernel_groups`` likewise builds the grouping by offset alone.
        The builders pass no edges (None, with ``counts``, ``implicit_gemm``
        and ``grouped_views``) for a relation built as a dense map."""
        map_edges = None
        if in_rows is None:
            if counts is None or implicit_gemm is None:
                raise ValueError('a relation without edges needs its dense '
                                 'map and counts.')
            map_edges = _MapEdges(implicit_gemm, counts)
            device = counts.device
        else:
            device = in_rows.device
        if counts is None:
            counts = torch.tensor(
                [in_rows.shape[0],
                 0 if out_coords is None else out_coords.shape[0]],
                dtype=torch.int32, device=device)
        _validate_counts(counts)
        contract = SparseRelationContract(
            counts=counts, kernel_offsets=kernel_offsets,
            out_coords=out_coords, n_in_capacity=n_in_capacity,
            n_out_capacity=n_out_capacity, n_kernels=n_kernels,
            source_coords=source_coords,
            source_active_rows=source_active_rows,
            target_coords=target_coords,
            target_active_rows=target_active_rows, stride=stride,
            padding=padding, kind=kind)
        edges = csr = None
        if map_edges is None:
            if row_offsets is None:
                cap = int(contract.n_out_capacity or 0)
                row_offsets = torch.zeros(cap + 1, dtype=torch.int32,
                                          device=device)
            _validate_row_offsets(row_offsets)
            edges = RelationEdges(in_rows, out_rows, kernel_ids)
        lazy_views = grouped_views is not None and in_row_offsets is None
        if lazy_views:
            pass
        elif in_row_offsets is None:
            cap = int(contract.n_in_capacity or 0)
            in_row_offsets = torch.zeros(cap + 1, dtype=torch.int32,
                                         device=device)
        if not lazy_views:
            if in_edge_ids is None:
                in_edge_ids = torch.zeros(edges.capacity, dtype=torch.int32,
                                          device=device)
            if kernel_row_offsets is None:
                cap = int(contract.n_kernels or 0)
                kernel_row_offsets = torch.zeros(cap + 1, dtype=torch.int32,
                                                 device=device)
            if kernel_edge_ids is None:
                kernel_edge_ids = torch.zeros(edges.capacity,
                                              dtype=torch.int32, device=device)
        if map_edges is None:
            if (contract.n_out_capacity is not None
                    and int(row_offsets.shape[0])
                    != int(contract.n_out_capacity) + 1):
                raise ValueError(
                    'row_offsets must have length n_out_capacity + 1.')
            csr = RelationCSRView(row_offsets)
        object.__setattr__(self, '_contract', contract)
        object.__setattr__(self, '_edges', edges)
        object.__setattr__(self, '_output_csr', csr)
        object.__setattr__(self, '_map_edges', map_edges)
        object.__setattr__(
            self, '_input_csr', None if lazy_views
            else RelationCSRView(in_row_offsets, in_edge_ids))
        object.__setattr__(
            self, '_kernel_csr', None if lazy_views
            else RelationCSRView(kernel_row_offsets, kernel_edge_ids))
        object.__setattr__(self, '_grouped_views',
                           grouped_views if lazy_views else None)
        object.__setattr__(self, '_kernel_groups',
                           kernel_groups if lazy_views else None)
        object.__setattr__(self, '_grouped', None)
        object.__setattr__(self, '_kernel_grouped', None)
        object.__setattr__(self, '_kernel_pairs', None)
        object.__setattr__(self, '_written', {})
        object.__setattr__(self, 'implicit_gemm', implicit_gemm)
        object.__setattr__(self, 'sorted_implicit_gemm', sorted_implicit_gemm)
        object.__setattr__(self, 'transposed_sorted_implicit_gemm', None)
        object.__setattr__(self, '_tiled', None)
        object.__setattr__(self, '_transposed_tiled', None)
        object.__setattr__(
            self, 'repeated_edges',
            _StatusWord(repeated_edges)
            if isinstance(repeated_edges, torch.Tensor) else repeated_edges)
        object.__setattr__(
            self, 'repeated_coords',
            _StatusWord(repeated_coords, deferred=True)
            if repeated_coords is not None else None)
        object.__setattr__(self, 'block_table', block_table)
        object.__setattr__(self, 'direct_expansion', bool(direct_expansion))

    @property
    def edges(self) -> RelationEdges:
        if self._map_edges is not None:
            return self._map_edges.get()[0]
        return self._edges

    @property
    def holds_edges(self) -> bool:
        """Whether the edges were emitted by the build (or made since)."""
        return self._map_edges is None or self._map_edges._made is not None

    @property
    def output_csr(self) -> RelationCSRView:
        if self._map_edges is not None:
            return self._map_edges.get()[1]
        return self._output_csr

    @property
    def contract(self) -> SparseRelationContract:
        """The contract, its edge count written."""
        if self._map_edges is not None:
            self._map_edges.get()
        return self._contract

    @property
    def kind(self) -> RelationKind:
        return self._contract.kind

    @property
    def source_active_rows(self) -> torch.Tensor | None:
        return self._contract.source_active_rows

    def _keep(self, name: str, make: Callable):
        return _kept(self, name, self._contract.counts.device, make)

    @property
    def input_csr(self) -> RelationCSRView:
        """Edges grouped by input row (stable in edge order)."""
        if self._input_csr is not None:
            return self._input_csr
        return self._keep('_grouped', self._group)[0]

    @property
    def kernel_csr(self) -> RelationCSRView:
        """Edges grouped by kernel offset (stable in edge order)."""
        if self._kernel_csr is not None:
            return self._kernel_csr
        if self._kernel_groups is not None:
            return self._keep('_kernel_grouped', self._group_by_kernel)
        return self._keep('_grouped', self._group)[1]

    def kernel_pairs(self) -> tuple[torch.Tensor, torch.Tensor] | None:
        """(offsets (K + 1,), pairs (E, 2)): the (input row, output row) of
        every edge, grouped by kernel offset in the order of ``kernel_csr``,
        built on first use; None for relations that group by a sort."""
        if self._kernel_groups is None:
            return None
        return self._keep('_kernel_pairs',
                          lambda: self._kernel_groups(None)[:2])

    def _group_by_kernel(self) -> RelationCSRView:
        offsets, _, ids = self._kernel_groups(self.output_csr.row_offsets)
        return RelationCSRView(offsets, ids)

    def _group(self) -> tuple[RelationCSRView, RelationCSRView]:
        in_offsets, in_ids, k_offsets, k_ids = (
            self._grouped_views() if self._map_edges is None
            else self._grouped_views(self.edges))
        return (RelationCSRView(in_offsets, in_ids),
                RelationCSRView(k_offsets, k_ids))

    @property
    def edge_capacity(self) -> int:
        if self._map_edges is not None:
            return self._map_edges.capacity
        return self._edges.capacity

    @property
    def counts(self) -> torch.Tensor:
        """Native counts array ``[edge_count, out_count]`` (device)."""
        return self.contract.counts

    @property
    def edge_count(self) -> torch.Tensor:
        return self.contract.edge_count

    @property
    def out_count(self) -> torch.Tensor:
        return self._contract.out_count

    @property
    def kernel_offsets(self) -> tuple[Triple, ...]:
        return self._contract.kernel_offsets

    @property
    def out_coords(self) -> torch.Tensor | None:
        return self._contract.out_coords

    @property
    def n_in_capacity(self) -> int | None:
        return self._contract.n_in_capacity

    @property
    def n_out_capacity(self) -> int | None:
        return self._contract.n_out_capacity

    @property
    def n_kernels(self) -> int | None:
        return self._contract.n_kernels

    @property
    def row_offsets(self) -> torch.Tensor:
        return self.output_csr.row_offsets

    @property
    def in_row_offsets(self) -> torch.Tensor:
        return self.input_csr.row_offsets

    @property
    def in_edge_ids(self) -> torch.Tensor:
        if self.input_csr.edge_ids is None:
            raise ValueError('input CSR view is missing edge ids.')
        return self.input_csr.edge_ids

    @property
    def kernel_row_offsets(self) -> torch.Tensor:
        return self.kernel_csr.row_offsets

    @property
    def kernel_edge_ids(self) -> torch.Tensor:
        if self.kernel_csr.edge_ids is None:
            raise ValueError('kernel CSR view is missing edge ids.')
        return self.kernel_csr.edge_ids

    @property
    def out_view(self) -> RelationCSRView:
        return self.output_csr

    @property
    def in_view(self) -> RelationCSRView:
        return self.input_csr

    @property
    def kernel_view(self) -> RelationCSRView:
        return self.kernel_csr

    def require_implicit_gemm(self) -> RelationImplicitGemmView:
        """Return or lazily build the implicit-GEMM view (views.py:452-465)."""
        return self._keep('implicit_gemm', self._implicit_gemm)

    def _implicit_gemm(self) -> RelationImplicitGemmView:
        if self._contract.kind in ('transposed', 'generative'):
            return self._expanded_implicit_gemm()
        from mlx_lattice_amd.core.coords.builders import (
            build_relation_implicit_gemm_view,
        )

        return build_relation_implicit_gemm_view(self)

    @property
    def dense_map_exact(self) -> bool:
        """Whether the dense (out_row, offset) -> in_row map holds every edge:
        at most one edge per (out_row, kernel_id).  Forward, submanifold and
        generative relations hold it by construction (a target relation
        too: each (target row, offset) has one candidate input, its first
        row); a transposed relation does unless an input coordinate repeats."""
        if self._contract.kind != 'transposed':
            return True
        if isinstance(self.repeated_edges, _StatusWord):
            # lattice_relation_flags: bit 2 = repeated (out_row, kernel_id)
            flags = self.repeated_edges.read()
            object.__setattr__(self, 'repeated_edges', bool(flags & 2))
        if self.repeated_edges is None:
            return False
        return not self.repeated_edges

    @property
    def transposed_map_exact(self) -> bool:
        """Whether the dense transposed (in_row, offset) -> out_row map holds
        every edge: at most one edge per (in_row, kernel_id).  Forward,
        generative and transposed relations hold it by construction (their
        output coordinates are distinct, or each output row has one edge); a
        submanifold relation, and a forward one of unit stride without
        padding, whose output rows are the input rows too, does unless a
        coordinate repeats.  The first
        question reads the build's status word from pinned memory (copied
        when a conv of trainable features or weights ran), so it waits for
        that copy only; under graph capture a word that was not copied before
        counts as a repeat."""
        if self._contract.kind == 'target':
            return False
        if isinstance(self.repeated_coords, _StatusWord):
            if self.repeated_coords.unreadable:
                return False
            # lattice_relation_flags: bit 8 = repeated coordinate
            flags = self.repeated_coords.read()
            object.__setattr__(self, 'repeated_coords', bool(flags & 8))
        return not self.repeated_coords

    def expect_backward(self) -> None:
        """Queue the copy that ``transposed_map_exact`` reads."""
        if (isinstance(self.repeated_coords, _StatusWord)
                and not self.repeated_coords.unreadable):
            self.repeated_coords.queue()

    def _expanded_implicit_gemm(self) -> RelationImplicitGemmView:
        """Dense map of a generative or transposed relation, scattered from
        its edges: out_in_map[out][k] = in (the expanded relations carry no
        source table to query)."""
        if not self.dense_map_exact:
            raise ValueError('the dense implicit-GEMM map cannot hold a '
                             'relation with repeated (out_row, kernel_id) '
                             'edges.')
        from mlx_lattice_amd._native import ext

        out_in_map, row_masks, _ = ext.build_transposed_implicit_gemm_map(
            self.edges.out_rows, self.edges.in_rows, self.edges.kernel_ids,
            self.counts, int(self.n_out_capacity), int(self.n_kernels))
        return RelationImplicitGemmView(out_in_map, row_masks=row_masks)

    def require_sorted_implicit_gemm(self) -> RelationSortedImplicitGemmView:
        """Return or lazily build the mask-sorted view (views.py:467-510):
        ``reorder_rows`` is the stable argsort of the row masks, the maps are
        gathered in that order and ``tile_masks`` ORs each 16-row quarter of
        every 64-row tile."""
        return self._keep('sorted_implicit_gemm', self._sorted_implicit_gemm)

    def _sorted_implicit_gemm(self) -> RelationSortedImplicitGemmView:
        view = self.require_implicit_gemm()
        if view.row_masks.shape[1] != 1:
            raise ValueError(
                'sorted implicit GEMM view currently supports K <= 32.')
        return _sorted_view(view.out_in_map, view.row_masks)

    def conv_view(self, weight_bytes: int) -> RelationSortedImplicitGemmView:
        """The view a matrix-core conv whose weight has ``weight_bytes`` per
        offset reads: the mask-sorted one, or, for few rows and channels, the
        rows in their own order (one launch instead of a sort; the result is
        the same).  Such a launch lasts as long as its longest tile, which
        sorting hardly shortens: the sorted view takes 44 us to build and the
        other 9, and a conv over it runs 1 us longer for 64 -> 64 fp16 at
        16,000 rows and 3 at 32,000, 6 for 16 -> 32 fp32 at 32,000 and 7 for
        64 -> 64 fp32 at 16,000, but 30 for 128 -> 128 fp32."""
        if (self.sorted_implicit_gemm is not None
                or self._contract.kind not in ('forward', 'submanifold',
                                              'target')
                or not _tiled_pays(self.n_out_capacity, weight_bytes)):
            return self.require_sorted_implicit_gemm()
        return self._keep('_tiled', self._tile)

    def _tile(self) -> RelationSortedImplicitGemmView:
        view = self.require_implicit_gemm()
        return _tiled_view(view.out_in_map, view.row_masks)

    def transposed_conv_view(self, weight_bytes: int,
                             ) -> RelationSortedImplicitGemmView:
        """``conv_view`` of the transposed relation."""
        if (self.transposed_sorted_implicit_gemm is not None
                or self._contract.kind not in ('forward', 'submanifold')
                or self.n_in_capacity is None
                or not _tiled_pays(self.n_in_capacity, weight_bytes)
                or self.n_kernels is None or self.n_kernels > 32):
            return self.require_transposed_sorted_implicit_gemm()
        return self._keep('_transposed_tiled',
                          lambda: _tiled_view(*self._transposed_map()))

    def _transposed_map(self) -> tuple[torch.Tensor, torch.Tensor]:
        """(in_out_map, row_masks) of the transposed relation."""
        from mlx_lattice_amd._native import ext

        if self._map_edges is not None:
            return ext.build_transposed_map_from_dense(
                self.implicit_gemm.out_in_map, int(self.n_in_capacity))
        in_out_map, row_masks, _ = ext.build_transposed_implicit_gemm_map(
            self.edges.in_rows, self.edges.out_rows, self.edges.kernel_ids,
            self.counts, int(self.n_in_capacity), int(self.n_kernels))
        return in_out_map, row_masks

    def require_transposed_sorted_implicit_gemm(
            self) -> RelationSortedImplicitGemmView:
        """Mask-sorted view of the transposed relation (input row -> output
        row per offset), built on first use and cached: the matrix-core
        route of the input gradient runs the forward's implicit GEMM over
        it.  Strided forward relations have at most one output row per (input
        row, offset), generative and transposed relations exactly one, and
        relations whose output rows are their input rows too unless a
        coordinate repeats (``transposed_map_exact``, which the input
        gradient checks first);
        target relations (whose target may repeat a coordinate) are
        refused."""
        if (self.transposed_sorted_implicit_gemm is None
                and self._contract.kind not in ('forward', 'submanifold',
                                                'transposed', 'generative')):
            raise ValueError('the transposed implicit-GEMM view needs a '
                             'forward, submanifold, transposed or generative '
                             'relation.')
        return self._keep('transposed_sorted_implicit_gemm',
                          self._transposed_sorted_implicit_gemm)

    def _transposed_sorted_implicit_gemm(
            self) -> RelationSortedImplicitGemmView:
        if self.n_in_capacity is None or self.n_kernels is None:
            raise ValueError('kernel relation is missing static shape metadata.')
        if self.n_kernels > 32:
            raise ValueError(
                'sorted implicit GEMM view currently supports K <= 32.')
        return _sorted_view(*self._transposed_map())


# ---------------------------------------------------------------- helpers --


def _int_offsets(offsets) -> tuple[Triple, ...]:
    """The offsets as a tuple of int triples."""
    return (_int_offset_tuple(offsets) if type(offsets) is tuple
            else tuple((int(x), int(y), int(z)) for x, y, z in offsets))


def _int_offset_tuple(offsets: tuple) -> tuple[Triple, ...]:
    for offset in offsets:
        if type(offset) is not tuple or len(offset) != 3:
            break
        x, y, z = offset
        if type(x) is not int or type(y) is not int or type(z) is not int:
            break
    else:
        return offsets
    return tuple((int(x), int(y), int(z)) for x, y, z in offsets)


def _tiled_pays(rows: int, weight_bytes: int) -> bool:
    return (rows <= _TILED_ROWS and weight_bytes <= _TILED_WEIGHT_BYTES
            and rows * weight_bytes <= _TILED_WORK)


def _sorted_view(out_in_map: torch.Tensor, row_masks: torch.Tensor,
                 ) -> RelationSortedImplicitGemmView:
    from mlx_lattice_amd._native import ext

    reorder, sorted_map, kv_map, tiles = ext.build_sorted_implicit_gemm_view(
        out_in_map, row_masks)
    return RelationSortedImplicitGemmView(
        sorted_out_in_map=sorted_map, sorted_kv_out_in_map=kv_map,
        reorder_rows=reorder, tile_masks=tiles)


def _tiled_view(out_in_map: torch.Tensor, row_masks: torch.Tensor,
                ) -> RelationSortedImplicitGemmView:
    from mlx_lattice_amd._native import ext

    order, rows, kv_map, tiles = ext.build_tiled_view(out_in_map, row_masks)
    return RelationSortedImplicitGemmView(
        sorted_out_in_map=rows, sorted_kv_out_in_map=kv_map,
        reorder_rows=order, tile_masks=tiles)


def _validate_row_array(value: torch.Tensor, *, name: str) -> None:
    if value.ndim != 1:
        raise ValueError(f'{name} must have shape (E,).')
    if value.dtype not in _INDEX_DTYPES:
        raise ValueError(f'{name} must be int32 or int64.')


def _validate_coords(value: torch.Tensor, *, name: str) -> None:
    if value.ndim != 2 or value.shape[1] != 4:
        raise ValueError(f'{name} must have shape (N, 4).')
    if value.dtype not in _INDEX_DTYPES:
        raise ValueError(f'{name} must be int32 or int64.')


def _validate_counts(value: torch.Tensor) -> None:
    if tuple(value.shape) != (2,) or value.dtype != torch.int32:
        raise ValueError(
            'relation counts must have shape (2,) and int32 dtype.')


def _validate_active_rows(value: torch.Tensor, *, name: str) -> None:
    if tuple(value.shape) != (1,) or value.dtype != torch.int32:
        raise ValueError(f'{name} must have shape (1,) and int32 dtype.')


def _validate_row_offsets(value: torch.Tensor) -> None:
    if value.ndim != 1 or value.dtype != torch.int32:
        raise ValueError(
            'row_offsets must have shape (N + 1,) and int32 dtype.')


def _require_same_rows(first: torch.Tensor, *rest: torch.Tensor,
                       names: tuple[str, ...]) -> None:
    rows = int(first.shape[0])
    for name, value in zip(names[1:], rest, strict=True):
        if int(value.shape[0]) != rows:
            raise ValueError(
                f'{names[0]} and {name} must have the same row count.')


def _optional_count(value: int | None, name: str) -> int | None:
    if value is None:
        return None
    normalized = int(value)
    if normalized < 0:
        raise ValueError(f'{name} must be non-negative.')
    return normalized
