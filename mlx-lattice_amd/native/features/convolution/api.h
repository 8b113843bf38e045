// Sparse convolution feature entry points over torch device tensors.
// Mirrors native/features/convolution/api.cpp:119-313 and quantized.cpp:
// 57-268 of the reference: same argument order, validation messages and
// static output capacity (out_capacity, C_out).
#pragma once

#include <torch/extension.h>

#include <optional>

namespace lattice_native {

at::Tensor sparse_conv_features(const at::Tensor& feats, const at::Tensor& weights, const at::Tensor& in_rows,
                                const at::Tensor& out_rows, const at::Tensor& kernel_ids, const at::Tensor& counts,
                                const at::Tensor& row_offsets, const at::Tensor& in_row_offsets,
                                const at::Tensor& in_edge_ids, const at::Tensor& kernel_row_offsets,
                                const at::Tensor& kernel_edge_ids, int out_capacity, int n_kernels,
                                const std::optional<at::Tensor>& bias = std::nullopt, bool relu = false);

// The CSR conv without the grouped plan views the reference signature
// carries for its gradient (the forward reads only the output CSR).  With
// the relation's dense map (out_in_map, (out_capacity, n_kernels)) and a
// shape the dense-map conv takes (C_in 4 or 8), it runs that instead and
// does not need the edges.
at::Tensor sparse_conv_features_csr(const at::Tensor& feats, const at::Tensor& weights,
                                    const std::optional<at::Tensor>& in_rows,
                                    const std::optional<at::Tensor>& kernel_ids, const at::Tensor& counts,
                                    const std::optional<at::Tensor>& row_offsets, int out_capacity, int n_kernels,
                                    const std::optional<at::Tensor>& bias = std::nullopt, bool relu = false,
                                    const std::optional<at::Tensor>& out_in_map = std::nullopt);

// Dense expansion conv over a direct generative / transposed relation:
// (rows * K, C_out), output row in * K + k = feats[in] @ W[k].
at::Tensor sparse_conv_features_expand(const at::Tensor& feats, const at::Tensor& weights,
                                       const at::Tensor& active_rows, int n_kernels,
                                       const std::optional<at::Tensor>& bias = std::nullopt, bool relu = false);

at::Tensor sparse_conv_features_sorted_implicit_gemm(const at::Tensor& feats, const at::Tensor& weights,
                                                     const at::Tensor& sorted_out_in_map,
                                                     const at::Tensor& sorted_kv_out_in_map,
                                                     const at::Tensor& reorder_rows, const at::Tensor& tile_masks,
                                                     int out_capacity, int n_kernels, bool store_sorted,
                                                     const std::optional<at::Tensor>& bias = std::nullopt,
                                                     const std::optional<at::Tensor>& tile_order = std::nullopt,
                                                     bool relu = false,
                                                     const std::optional<at::Tensor>& weight_fragments = std::nullopt);

// The fragment-ordered copy of a 5D fp16/bf16 weight that the streamed
// matrix-core conv reads (lattice_hip_conv_weight_fragments), kept with the
// weight and passed back as `weight_fragments`; an empty tensor when the
// weight's shape does not take that route.
at::Tensor conv_weight_fragments(const at::Tensor& weights);

// Edges of a dense-map relation grouped by offset without a sort
// (lattice_hip_build_kernel_pairs): (kernel_row_offsets, pairs (E, 2) or
// none, kernel_edge_ids (E,) or none; the ids when row_offsets is given,
// else the pairs), and the weight gradient over the pairs.
std::tuple<at::Tensor, std::optional<at::Tensor>, std::optional<at::Tensor>> build_kernel_pairs(
    const at::Tensor& row_masks, const at::Tensor& out_in_map, const std::optional<at::Tensor>& row_offsets);
// (in_out_map (in_capacity, K), row_masks) of a relation with a dense map.
std::tuple<at::Tensor, at::Tensor> build_transposed_map_from_dense(const at::Tensor& out_in_map, int in_capacity);
at::Tensor sparse_conv_weight_grad_pairs(const at::Tensor& feats, const at::Tensor& cotangent,
                                         const at::Tensor& weights, const at::Tensor& pairs,
                                         const at::Tensor& kernel_row_offsets, int n_kernels);

// The streamed conv for the types and channel counts the sorted entry does
// not take (lattice_hip_sparse_conv_features_padded): whether a contiguous
// `feats` and the shape qualify; the fragments of a float weight (role:
// lattice_fragment_role) or of a packed one; the conv over a sorted view.
bool conv_padded_supported(const at::Tensor& feats, int out_channels, int n_kernels, int out_capacity);
at::Tensor conv_padded_fragments(const at::Tensor& weights, int role);
at::Tensor quantized_padded_fragments(const at::Tensor& weights, const at::Tensor& scales, const at::Tensor& biases,
                                      int in_channels, int out_channels, int storage_in_channels, int group_size,
                                      int bits);
at::Tensor sparse_conv_features_padded(const at::Tensor& feats, const at::Tensor& fragments, int bits,
                                       int out_channels, const at::Tensor& sorted_kv_out_in_map,
                                       const at::Tensor& reorder_rows, const at::Tensor& tile_masks,
                                       int out_capacity, int n_kernels,
                                       const std::optional<at::Tensor>& bias = std::nullopt,
                                       const std::optional<at::Tensor>& tile_order = std::nullopt,
                                       bool relu = false);
// The same with the fragments made in the call, from the weight as it is
// (one more launch, the size of the weight): what the operators run, since
// no counter sees every write to a weight (through .data, by a graph replay)
// and the edge kernels, which these stand in for, read the weight itself.
at::Tensor sparse_conv_padded(const at::Tensor& feats, const at::Tensor& weights, int role,
                              const at::Tensor& sorted_kv_out_in_map, const at::Tensor& reorder_rows,
                              const at::Tensor& tile_masks, int out_capacity, int n_kernels,
                              const std::optional<at::Tensor>& bias = std::nullopt,
                              const std::optional<at::Tensor>& tile_order = std::nullopt, bool relu = false);
at::Tensor sparse_quantized_conv_padded(const at::Tensor& feats, const at::Tensor& weights, const at::Tensor& scales,
                                        const at::Tensor& biases, int in_channels, int out_channels,
                                        int storage_in_channels, int group_size, int bits,
                                        const at::Tensor& sorted_kv_out_in_map, const at::Tensor& reorder_rows,
                                        const at::Tensor& tile_masks, int out_capacity, int n_kernels,
                                        const std::optional<at::Tensor>& bias = std::nullopt,
                                        const std::optional<at::Tensor>& tile_order = std::nullopt,
                                        bool relu = false);

at::Tensor sparse_quantized_conv_features(const at::Tensor& feats, const at::Tensor& weights,
                                          const at::Tensor& scales, const at::Tensor& biases,
                                          const std::optional<at::Tensor>& in_rows,
                                          const std::optional<at::Tensor>& out_rows,
                                          const std::optional<at::Tensor>& kernel_ids, const at::Tensor& counts,
                                          const std::optional<at::Tensor>& row_offsets,
                                          const at::Tensor& sorted_kv_out_in_map,
                                          const at::Tensor& reorder_rows, const at::Tensor& tile_masks,
                                          int out_capacity, int n_kernels, int in_channels, int out_channels,
                                          int storage_in_channels, int group_size, int bits,
                                          const std::optional<at::Tensor>& bias = std::nullopt,
                                          const std::optional<at::Tensor>& tile_order = std::nullopt,
                                          bool relu = false,
                                          const std::optional<at::Tensor>& weight_fragments = std::nullopt,
                                          const std::optional<at::Tensor>& out_in_map = std::nullopt);

// The fragment-ordered packed copy of a quantized weight that the streamed
// matrix-core conv reads (lattice_hip_quantized_weight_fragments: codes,
// scale and bias of each lane's 8 input channels in one 16-byte piece),
// kept with the weight and passed back as `weight_fragments`; an empty
// tensor when the shape does not take that route.
at::Tensor quantized_weight_fragments(const at::Tensor& weights, const at::Tensor& scales,
                                      const at::Tensor& biases, int in_channels, int out_channels,
                                      int storage_in_channels, int group_size, int bits);

// Longest-first order of the 128-row tiles of a sorted view
// (lattice_hip_conv_tile_order), kept with the view and passed back as
// `tile_order` so the conv skips its per-call schedule.
at::Tensor conv_tile_order(const at::Tensor& tile_masks, int out_capacity);

// Gradients (the reference conv primitive's vjp, primitive.cpp:137-176):
// input gradient over the input-grouped CSR, (in_capacity, C_in) in the
// cotangent dtype.
at::Tensor sparse_conv_input_grad(const at::Tensor& cot, const at::Tensor& weights, const at::Tensor& out_rows,
                                  const at::Tensor& kernel_ids, const at::Tensor& counts,
                                  const at::Tensor& in_row_offsets, const at::Tensor& in_edge_ids, int in_capacity,
                                  int n_kernels);

// Transposed dense map (in_out_map (in_capacity, K), row_masks, status) of
// a forward or submanifold relation, for the matrix-core input gradient;
// status (1,) gets LATTICE_STATUS_REPEATED_PAIR when the map is incomplete.
std::tuple<at::Tensor, at::Tensor, at::Tensor> build_transposed_implicit_gemm_map(const at::Tensor& in_rows,
                                                                      const at::Tensor& out_rows,
                                                                      const at::Tensor& kernel_ids,
                                                                      const at::Tensor& counts, int in_capacity,
                                                                      int n_kernels);

// Weight gradient over the kernel-grouped CSR, in the shape and layout of
// `weights` (5D or mapped) and the cotangent dtype.
at::Tensor sparse_conv_weight_grad(const at::Tensor& feats, const at::Tensor& cot, const at::Tensor& weights,
                                   const at::Tensor& in_rows, const at::Tensor& out_rows, const at::Tensor& counts,
                                   const at::Tensor& kernel_row_offsets, const at::Tensor& kernel_edge_ids,
                                   int n_kernels);

}  // namespace lattice_native
