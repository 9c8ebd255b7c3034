// Internal interface between the pieces of the unfiltered backward.
#pragma once

#include "cce_common.h"

namespace cce {

// The 16 x 16 x 32 kernels address rows by 32-bit byte offsets and stream at least two stages per tile.
inline bool dense_k16(int64_t n_rows, int64_t d, int64_t stride_e, int64_t stride_cv) {
  return d > kDmaBK && n_rows * stride_e * 2 < (int64_t(1) << 32) && 256 * stride_cv * 2 < (int64_t(1) << 32);
}
// Widths the logits of the unfiltered backward can be streamed at: whole stages, or (16 x 16 x 32 kernel only) whole
// 16-byte pieces.  The products take any multiple of 8.
inline bool dense_width_ok(int64_t n_rows, int64_t d, int64_t stride_e, int64_t stride_cv) {
  return d % kDmaBK == 0 || (d % 8 == 0 && dense_k16(n_rows, d, stride_e, stride_cv));
}

// dz of one vocabulary chunk (cce_dense_dz.hip); the arguments of cce_backward_dz plus `pad_store`: also store
// the zero gradients of the columns between v and ldz.
int dense_dz_launch(const void* e, const void* c, const void* bias,
                    const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                    const int32_t* valids, const int64_t* targets,
                    void* dz, int64_t ldz, int dz_is_fp32, int pad_store,
                    int64_t n_rows, int64_t b, int64_t v, int64_t d,
                    int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                    float grad_scale, int64_t shift, int64_t target_offset,
                    float softcap, int dtype, hipStream_t stream);

// ---- fp32 operands as 16-bit parts (cce_fp32.hip) ---------------------------------------------------------------
// A row of e_parts / c_parts holds its parts [hi | mid | lo] side by side, part_d (a multiple of 64) columns each;
// ld_e / ld_c elements from row to row, a multiple of 8.  terms: 6 cross terms of three parts, or 3 of two.
// Logits are formed from rows [hi | lo] of fp16 instead, packed, where the device finds *wide == 0: their products are 1 /
// halves_scale times what they stand for (a power of two).  lse_terms_launch finds these halves in the place of the parts.

// Spans per row block that lse_terms_launch makes of v classes: the float2 partials [spans][b] it writes.
int lse_terms_splits(int64_t b, int64_t v);
int lse_terms_launch(const uint16_t* e_parts, int64_t ld_e, const uint16_t* c_parts, int64_t ld_c, const float* bias,
                     float2* partial, int64_t b, int64_t v, int64_t part_d, int terms, const int* wide, float halves_scale,
                     float softcap, hipStream_t stream);

// dz of v classes as bf16 parts [b_store][parts][ldz], ldz = v rounded up to 64; columns past v and rows b .. b_store
// (b rounded up to 64) are zeros.  valids: the rows of the batch that the (compact) rows of e_parts are.
int dz_terms_launch(const uint16_t* e_parts, int64_t ld_e, const uint16_t* c_parts, int64_t ld_c, const uint16_t* e_halves,
                    const uint16_t* c_halves, const int* wide, float halves_scale, const float* bias,
                    const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                    const int32_t* valids, const int64_t* targets, uint16_t* dz_parts, int64_t ldz,
                    int64_t n_rows, int64_t b, int64_t b_store, int64_t v, int64_t part_d, int terms, int parts,
                    float grad_scale, int64_t shift, int64_t target_offset, float softcap, hipStream_t stream);

// Chunks of classes and cuts of the reductions of dE and dC for terms_products_launch.
struct TermsPlan {
  int64_t unit;
  int de_splits, dc_splits;
};
TermsPlan terms_plan(int64_t b, int64_t v, int64_t d, int terms, int64_t dz_bytes_per_class, int64_t c_bytes_per_class,
                     int64_t most_bytes);

// dE (+)= dz . C and dC (+)= dz^T . E of one chunk, fp32 results.  dz_parts as written by dz_terms_launch, c_parts and
// e_parts with zero rows up to cls_pad and b_pad (multiples of 64).  Range s of a reduction (de_len classes, dc_len rows,
// multiples of 64) goes to d_e + s * de_slot / d_c + s * dc_slot.  d_e is indexed by row number, or through valids.
int terms_products_launch(const uint16_t* dz_parts, int64_t ldz, const uint16_t* c_parts, int64_t ld_c, const uint16_t* e_parts,
                          int64_t ld_e, const int32_t* valids, float* d_e, int64_t ld_de, bool de_by_number, bool de_init,
                          int64_t de_slot, int de_len, float* d_c, int64_t ld_dc, bool dc_add, int64_t dc_slot, int dc_len,
                          bool out_vec, int64_t b, int64_t b_pad, int64_t cls, int64_t cls_pad, int64_t d, int64_t part_d, int terms,
                          int parts, hipStream_t stream);
// d_bias[class] += column sums of dz [b][parts][ldz] in dtype; dz is used up
int dz_colsum_launch(uint16_t* dz, int64_t ldz, int parts, int64_t b, int64_t n_cls, float* d_bias, int dtype, hipStream_t stream);
// out[row(i)][0 .. d) (+)= sum over the slots [count][rows][ld_slot]
int split_sum_launch(const float* slots, int count, int64_t rows, int64_t d, int64_t ld_slot, const int32_t* ids, float* out,
                     int64_t ld, bool add, bool out_vec, hipStream_t stream);

// ---- the loss of every valid row (cce_rows.hip) -------------------------------------------------------------------
constexpr int kLossRowsFp32 = -1;  // beside CCE_DTYPE_*
struct LossRowsParams {
  const void* e;
  const void* c;
  const void* bias;
  const int32_t* valids;
  const int64_t* targets;
  const float2* partial;  // [nsplit][b]
  float* lse;
  float* nll;
  int nsplit;
  int64_t n_rows, b, v, d, stride_e, stride_cv, stride_cd, shift, target_offset;
  float softcap;
};
int loss_rows_launch(const LossRowsParams& p, int dtype, hipStream_t stream);
// *out = the sum or mean of values[n] (n == 0: 0 or NaN), added up in fp64
int64_t row_total_workspace_bytes(int64_t n);
int row_total_launch(const float* values, int64_t n, bool mean, float* out, void* workspace, hipStream_t stream);

}  // namespace cce
