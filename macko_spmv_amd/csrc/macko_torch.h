// The operators' kernels for the GPU, as macko_torch.cpp registers them: what macko_eager.cpp knows of them.
#pragma once

#include <ATen/ATen.h>

#include <optional>
#include <tuple>
#include <vector>

namespace macko_torch {

typedef std::tuple<at::Tensor, at::Tensor, at::Tensor, int64_t, int64_t> Compressed;  // values, deltas, row_indices, rows, cols

// plan: where the product's cuts go if they are wanted (fp16).  go_on: asked while the count pass runs; if it says no, that
// pass is all that is done, and undefined tensors are returned.
Compressed compress_on_device(const at::Tensor &M, at::Tensor *plan = nullptr, bool (*go_on)() noexcept = nullptr);

at::Tensor multiply_hip(const at::Tensor &M_values, const at::Tensor &M_deltas, const at::Tensor &M_row_indices,
                        int64_t M_rows, int64_t M_cols, const at::Tensor &V);
at::Tensor multiply_planned_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols, const at::Tensor &V,
                                const at::Tensor &plan);
void multiply_axpby_hip(const at::Tensor &M_values, const at::Tensor &M_deltas, const at::Tensor &M_row_indices,
                        int64_t M_rows, int64_t M_cols, const at::Tensor &V, at::Tensor C, double alpha, double beta);
void multiply_axpby_planned_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols, const at::Tensor &V,
                                at::Tensor C, double alpha, double beta, const at::Tensor &plan);
Compressed compress_hip(const at::Tensor &M);
at::Tensor plan_hip(const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols, int64_t padded_entries);
at::Tensor multiply_batched_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols, const at::Tensor &X);
at::Tensor multiply_int8_hip(const at::Tensor &M_values, const at::Tensor &M_deltas, const at::Tensor &M_row_indices,
                             int64_t M_rows, int64_t M_cols, const at::Tensor &V);
void multiply_int8_axpby_hip(const at::Tensor &M_values, const at::Tensor &M_deltas, const at::Tensor &M_row_indices,
                             int64_t M_rows, int64_t M_cols, const at::Tensor &V, at::Tensor C, double alpha,
                             double beta);
at::Tensor multiply_rmsnorm_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols, const at::Tensor &V,
                                const at::Tensor &norm_weight, double eps);
void multiply_silu_mul_axpby_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                 const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols,
                                 const at::Tensor &gate, const at::Tensor &up, at::Tensor C, double alpha,
                                 double beta);
void multiply_attention_axpby_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                                  const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols,
                                  const at::Tensor &parts, int64_t head_dim, at::Tensor C, double alpha, double beta);
at::Tensor decode_rmsnorm_hip(const at::Tensor &x, const at::Tensor &weight, double eps);
at::Tensor decode_norm_matvec_hip(const at::Tensor &W, const at::Tensor &x, const at::Tensor &norm_weight,
                                  double eps);
at::Tensor decode_rope_append_hip(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                                  const at::Tensor &cos_table, const at::Tensor &sin_table,
                                  const at::Tensor &position, at::Tensor k_cache, at::Tensor v_cache);
at::Tensor decode_attention_hip(const at::Tensor &q, const at::Tensor &k_cache, const at::Tensor &v_cache,
                                const at::Tensor &position, double scale);
at::Tensor decode_silu_mul_hip(const at::Tensor &gate, const at::Tensor &up);
at::Tensor decode_rope_attention_hip(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                                     const at::Tensor &cos_table, const at::Tensor &sin_table,
                                     const at::Tensor &position, at::Tensor k_cache, at::Tensor v_cache,
                                     double scale);
at::Tensor decode_rope_attention_parts_hip(const at::Tensor &q, const at::Tensor &k, const at::Tensor &v,
                                           const at::Tensor &cos_table, const at::Tensor &sin_table,
                                           const at::Tensor &position, at::Tensor k_cache, at::Tensor v_cache,
                                           double scale);
at::Tensor pack_rmsnorm_hip(const at::Tensor &x, const at::Tensor &weight, double eps);
at::Tensor rmsnorm_rows_hip(const at::Tensor &x, const at::Tensor &weight, double eps);
at::Tensor pack_silu_mul_hip(const at::Tensor &gate, const at::Tensor &up);
at::Tensor multiply_packed_hip(const at::Tensor &M_values, const at::Tensor &M_deltas,
                               const at::Tensor &M_row_indices, int64_t M_rows, int64_t M_cols,
                               const at::Tensor &packed, int64_t batch, const std::optional<at::Tensor> &residual);
std::vector<at::Tensor> multiply_packed_several_hip(at::TensorList M_values, at::TensorList M_deltas,
                                                    at::TensorList M_row_indices, at::IntArrayRef M_rows,
                                                    int64_t M_cols, const at::Tensor &packed, int64_t batch);
at::Tensor multiply_packed_silu_hip(at::TensorList M_values, at::TensorList M_deltas, at::TensorList M_row_indices, int64_t M_rows,
                                    int64_t M_cols, const at::Tensor &packed, int64_t batch);
void prefill_rope_append_hip(at::Tensor q, const at::Tensor &k, const at::Tensor &v, const at::Tensor &cos_rows,
                             const at::Tensor &sin_rows, const at::Tensor &positions, at::Tensor k_cache,
                             at::Tensor v_cache);
at::Tensor prefill_attention_hip(const at::Tensor &q, const at::Tensor &k_cache, const at::Tensor &v_cache,
                                 const at::Tensor &positions, double scale);

}  // namespace macko_torch
