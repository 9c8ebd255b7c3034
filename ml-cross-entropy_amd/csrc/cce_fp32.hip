// fp32 inputs on matrix cores that multiply 16-bit numbers.
//
// gfx950 has no fast fp32 matrix path (the reference leans on Triton's tf32x3 / ieee dot for fp32 inputs,
// cut_cross_entropy/cce_lse_forward.py:81).  An fp32 value is split into three bf16 parts, x = hi + mid + lo (8 + 8 + 8
// significant bits), and a product of two of them is taken as its six leading cross terms
//     hi lo, lo hi, mid mid, hi mid, mid hi, hi hi      (what is left is below 2^-24 relative)
// summed in ONE reduction by the 16-bit kernels, whose stages walk the terms one after the other, smallest first (kTermsFirst
// / kTermsSecond in cce_common.h).  The parts of a matrix are stored once, side by side: [hi | mid | lo], 6 bytes per value
// where an operand widened by its terms takes 12, and the same copy of C serves the logits and dE = dz . C.  The gradient
// of the logits leaves its kernel as parts as well, so both products read it as it lies, all terms of a product in one
// launch: accumulators stay in registers from the first term to the last.
//
// The classes are walked in chunks (bounded copies of C and of dz), e is copied whole, rows of the batch only.  What bounds
// it: six bf16 products per fp32 product.  Splitting C moves 10 bytes per value and pass, 0.2 ms for [32064, 3072].
// Measured at E [2046, 3072] x C [32064, 3072], forward and backward: 15.4 ms with operands widened by library
// element-wise kernels and one launch of the products per term, 8.0 ms so on four-wave tiles, 7.3 on the eight-wave ones.
#include "cce_dense.h"

#include <algorithm>

namespace cce {

constexpr int64_t kForwardChunkBytes = int64_t(512) << 20;   // copy of a chunk of C
constexpr int64_t kBackwardChunkBytes = int64_t(384) << 20;  // copy of a chunk of C, dz of it, and the slots of cut reductions
constexpr int64_t kRowBlockBytes = (int64_t(1) << 32) - 1;   // the kernels reach the rows of e by 32-bit offsets

static int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }
static int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }
static int parts_of(int terms) { return terms == 6 ? 3 : 2; }

// x[row] -> [hi | mid (| lo)], part_d columns each: columns past d and rows past n are zeros.  Eight columns per thread.
template <bool VEC>
__global__ __launch_bounds__(256) void split_parts_kernel(const float* x, int64_t stride, const int32_t* ids, int64_t n, int64_t n_pad,
                                                          int d, int part_d, int parts, uint16_t* out) {
  const int per_row = part_d / 8;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (item >= n_pad * per_row) return;
  const int64_t i = item / per_row;
  const int col = static_cast<int>(item - i * per_row) * 8;
  float v[8] = {};
  if (i < n) {
    const float* row = x + (ids != nullptr ? static_cast<int64_t>(ids[i]) : i) * stride;
    if (VEC && col + 8 <= d) {
      const float4 a = *reinterpret_cast<const float4*>(row + col), b = *reinterpret_cast<const float4*>(row + col + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (col + k < d) ? row[col + k] : 0.0f;
    }
  }
  uint16_t* dst = out + i * parts * part_d + col;
#pragma unroll
  for (int part = 0; part < 3; ++part) {
    if (part >= parts) break;
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[k] = Elem<BF16>::pack2(v[2 * k], v[2 * k + 1]);
      v[2 * k] -= Elem<BF16>::to_float(static_cast<uint16_t>(w[k]));
      v[2 * k + 1] -= Elem<BF16>::to_float(static_cast<uint16_t>(w[k] >> 16));
    }
    *reinterpret_cast<uint4*>(dst + part * part_d) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

static int split_parts(const float* x, int64_t stride, const int32_t* ids, int64_t n, int64_t n_pad, int64_t d, int64_t part_d,
                       int parts, uint16_t* out, hipStream_t stream) {
  const bool vec = aligned16(x) && stride % 4 == 0;
  const dim3 grid(static_cast<unsigned>((n_pad * (part_d / 8) + 255) / 256));
  if (vec)
    hipLaunchKernelGGL(split_parts_kernel<true>, grid, dim3(256), 0, stream, x, stride, ids, n, n_pad, static_cast<int>(d),
                       static_cast<int>(part_d), parts, out);
  else
    hipLaunchKernelGGL(split_parts_kernel<false>, grid, dim3(256), 0, stream, x, stride, ids, n, n_pad, static_cast<int>(d),
                       static_cast<int>(part_d), parts, out);
  return status_from_hip(hipGetLastError());
}

// Rows of e per pass: all of them, or as many as 32-bit offsets reach.
static int64_t row_block(int64_t b, int64_t part_d, int parts) {
  const int64_t most = kRowBlockBytes / (parts * part_d * 2) / 256 * 256;
  return std::min(b, most);
}

// ---- forward
struct Fp32Forward {
  int parts;
  int64_t part_d, rows, unit;     // rows per block, classes per chunk
  int64_t e_bytes, c_bytes, partial_bytes;
};
static Fp32Forward plan_forward(int64_t b, int64_t v, int64_t d, int terms) {
  Fp32Forward f;
  f.parts = parts_of(terms);
  f.part_d = round_up(d, 64);
  f.rows = row_block(b, f.part_d, f.parts);
  const int64_t row_bytes = f.parts * f.part_d * 2;
  const int64_t v_pad = round_up(v, 256);
  const int64_t most = std::max<int64_t>(256, kForwardChunkBytes / row_bytes / 256 * 256);
  const int64_t chunks = (v_pad + most - 1) / most;
  f.unit = round_up((v_pad + chunks - 1) / chunks, 256);
  auto partials = [&](int64_t rows) {  // of all spans of all chunks
    int64_t splits = 0;
    for (int64_t v0 = 0; v0 < v; v0 += f.unit) splits += lse_terms_splits(rows, std::min(f.unit, v - v0));
    return splits * rows * static_cast<int64_t>(sizeof(float2));
  };
  const int64_t last = b - (b - 1) / f.rows * f.rows;
  f.e_bytes = align256(f.rows * row_bytes);
  f.c_bytes = align256(f.unit * row_bytes);
  f.partial_bytes = align256(std::max(partials(f.rows), partials(last)));
  return f;
}

// ---- backward
// dz is stored in the parts that its products read; all three of them where its column sums are wanted, whatever `terms`
// says, since those are sums of fp32 values and no products.  The workspace has room for that.
constexpr int kAllParts = 3;
struct Fp32Backward {
  int parts;
  int64_t part_d, rows, rows_pad, unit;
  TermsPlan cut;
  int de_len, dc_len, de_slots, dc_slots;
  int64_t e_bytes, c_bytes, dz_bytes, de_slot_bytes, dc_slot_bytes;
};
static Fp32Backward plan_backward(int64_t b, int64_t v, int64_t d, int terms) {
  Fp32Backward f;
  f.parts = parts_of(terms);
  f.part_d = round_up(d, 64);
  f.rows = row_block(b, f.part_d, f.parts);
  f.rows_pad = round_up(f.rows, 64);
  const int64_t row_bytes = f.parts * f.part_d * 2;
  f.cut = terms_plan(f.rows, v, f.part_d, terms, f.rows_pad * f.parts * 2, row_bytes, kBackwardChunkBytes, f.rows == b);
  f.unit = f.cut.unit;
  const int64_t cls = round_up(std::min(f.unit, v), 64);
  f.de_len = static_cast<int>((cls / 64 + f.cut.de_splits - 1) / f.cut.de_splits * 64);
  f.dc_len = static_cast<int>((f.rows_pad / 64 + f.cut.dc_splits - 1) / f.cut.dc_splits * 64);
  f.de_slots = static_cast<int>((cls + f.de_len - 1) / f.de_len);
  f.dc_slots = static_cast<int>((f.rows_pad + f.dc_len - 1) / f.dc_len);
  f.e_bytes = align256(f.rows_pad * row_bytes);
  f.c_bytes = align256(round_up(std::min(f.unit, v), 256) * row_bytes);
  f.dz_bytes = align256(f.rows_pad * kAllParts * cls * 2);
  f.de_slot_bytes = f.de_slots > 1 ? align256(f.de_slots * f.rows * f.part_d * 4) : 0;
  f.dc_slot_bytes = f.dc_slots > 1 ? align256(f.dc_slots * std::min(f.unit, v) * f.part_d * 4) : 0;
  return f;
}

static int check(const void* e, const void* c, const void* targets, int64_t n_rows, int64_t b, int64_t v, int64_t d,
                 const int32_t* valids, int64_t stride_cd, int64_t shift, int terms) {
  if (b < 0 || v <= 0 || d <= 0 || n_rows < 0 || shift < 0 || (terms != 3 && terms != 6)) return CCE_ERR_INVALID_ARGUMENT;
  if (b == 0) return CCE_OK;
  if (e == nullptr || c == nullptr || targets == nullptr) return CCE_ERR_INVALID_ARGUMENT;
  if (valids == nullptr && b > n_rows) return CCE_ERR_INVALID_ARGUMENT;
  if (n_rows >= (int64_t(1) << 31) || b >= (int64_t(1) << 31) - 512 || v >= (int64_t(1) << 31) - 512 || d > (1 << 20))
    return CCE_ERR_INVALID_ARGUMENT;
  if (stride_cd != 1) return CCE_ERR_MISALIGNED;
  return CCE_OK;
}

}  // namespace cce

using namespace cce;

extern "C" int64_t cce_fp32_forward_workspace_bytes(int64_t b, int64_t v, int64_t d, int terms) {
  if (b <= 0 || v <= 0 || d <= 0 || (terms != 3 && terms != 6)) return 0;
  const Fp32Forward f = plan_forward(b, v, d, terms);
  return f.e_bytes + f.c_bytes + f.partial_bytes;
}

extern "C" int cce_fp32_forward(const float* e, const float* c, const float* bias, const int32_t* valids, const int64_t* targets,
                                float* lse, float* nll, void* workspace, int64_t workspace_bytes,
                                int64_t n_rows, int64_t b, int64_t v, int64_t d,
                                int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                                int64_t shift, int64_t target_offset, float softcap, int terms, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  int st = check(e, c, targets, n_rows, b, v, d, valids, stride_cd, shift, terms);
  if (st != CCE_OK || b == 0) return st;
  if (lse == nullptr || nll == nullptr) return CCE_ERR_INVALID_ARGUMENT;
  const Fp32Forward f = plan_forward(b, v, d, terms);
  if (workspace == nullptr || workspace_bytes < f.e_bytes + f.c_bytes + f.partial_bytes) return CCE_ERR_WORKSPACE_TOO_SMALL;
  if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return CCE_ERR_MISALIGNED;
  unsigned char* const ws = static_cast<unsigned char*>(workspace);
  uint16_t* const e_parts = reinterpret_cast<uint16_t*>(ws);
  uint16_t* const c_parts = reinterpret_cast<uint16_t*>(ws + f.e_bytes);
  float2* const partial = reinterpret_cast<float2*>(ws + f.e_bytes + f.c_bytes);
  const int64_t ld = f.parts * f.part_d;

  for (int64_t r0 = 0; r0 < b; r0 += f.rows) {
    const int64_t rows = std::min(f.rows, b - r0);
    const int32_t* ids = valids != nullptr ? valids + r0 : nullptr;
    st = split_parts(valids != nullptr ? e : e + r0 * stride_e, stride_e, ids, rows, rows, d, f.part_d, f.parts, e_parts, stream);
    if (st != CCE_OK) return st;
    int nsplit = 0;
    for (int64_t v0 = 0; v0 < v; v0 += f.unit) {
      const int64_t cls = std::min(f.unit, v - v0);
      st = split_parts(c + v0 * stride_cv, stride_cv, nullptr, cls, round_up(cls, 256), d, f.part_d, f.parts, c_parts, stream);
      if (st != CCE_OK) return st;
      st = lse_terms_launch(e_parts, ld, c_parts, ld, bias != nullptr ? bias + v0 : nullptr, partial + nsplit * rows, rows, cls,
                            f.part_d, terms, softcap, stream);
      if (st != CCE_OK) return st;
      nsplit += lse_terms_splits(rows, cls);
    }
    const int64_t moved = valids == nullptr ? r0 : 0;
    const LossRowsParams p = {e + moved * stride_e, c, bias, ids, targets + moved, partial, lse + r0, nll + r0, nsplit, n_rows - moved,
                              rows, v, d, stride_e, stride_cv, stride_cd, shift, target_offset, softcap};
    st = loss_rows_launch(p, kLossRowsFp32, stream);
    if (st != CCE_OK) return st;
  }
  return CCE_OK;
}

extern "C" int64_t cce_fp32_backward_workspace_bytes(int64_t b, int64_t v, int64_t d, int terms) {
  if (b <= 0 || v <= 0 || d <= 0 || (terms != 3 && terms != 6)) return 0;
  const Fp32Backward f = plan_backward(b, v, d, terms);
  return f.e_bytes + f.c_bytes + f.dz_bytes + f.de_slot_bytes + f.dc_slot_bytes;
}

extern "C" int cce_fp32_backward(const float* e, const float* c, const float* bias, const float* lse, const float* d_out,
                                 int d_out_is_scalar, const float* d_lse, const int32_t* valids, const int64_t* targets,
                                 float* d_e, float* d_c, float* d_bias, void* workspace, int64_t workspace_bytes,
                                 int64_t n_rows, int64_t b, int64_t v, int64_t d,
                                 int64_t stride_e, int64_t stride_cv, int64_t stride_cd, int64_t ld_de, int64_t ld_dc,
                                 float grad_scale, int64_t shift, int64_t target_offset, float softcap, int terms, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  int st = check(e, c, targets, n_rows, b, v, d, valids, stride_cd, shift, terms);
  if (st != CCE_OK || b == 0) return st;
  if (lse == nullptr || d_out == nullptr) return CCE_ERR_INVALID_ARGUMENT;
  if (d_e == nullptr && d_c == nullptr && d_bias == nullptr) return CCE_OK;
  if ((d_e != nullptr && ld_de < d) || (d_c != nullptr && ld_dc < d)) return CCE_ERR_INVALID_ARGUMENT;
  const Fp32Backward f = plan_backward(b, v, d, terms);
  if (workspace == nullptr || workspace_bytes < f.e_bytes + f.c_bytes + f.dz_bytes + f.de_slot_bytes + f.dc_slot_bytes)
    return CCE_ERR_WORKSPACE_TOO_SMALL;
  if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return CCE_ERR_MISALIGNED;
  unsigned char* at = static_cast<unsigned char*>(workspace);
  auto take = [&](int64_t bytes) {
    unsigned char* const p = at;
    at += bytes;
    return p;
  };
  uint16_t* const e_parts = reinterpret_cast<uint16_t*>(take(f.e_bytes));
  uint16_t* const c_parts = reinterpret_cast<uint16_t*>(take(f.c_bytes));
  uint16_t* const dz_parts = reinterpret_cast<uint16_t*>(take(f.dz_bytes));
  float* const de_slots = reinterpret_cast<float*>(take(f.de_slot_bytes));
  float* const dc_slots = reinterpret_cast<float*>(take(f.dc_slot_bytes));
  const int64_t ld = f.parts * f.part_d;
  const int stored = d_bias != nullptr ? kAllParts : f.parts;
  const bool de_cut = d_e != nullptr && f.de_slots > 1, dc_cut = d_c != nullptr && f.dc_slots > 1;
  const bool out_vec = d % 8 == 0 && (d_e == nullptr || (aligned16(d_e) && ld_de % 4 == 0)) &&
                       (d_c == nullptr || (aligned16(d_c) && ld_dc % 4 == 0));
  const int de_len = de_cut ? f.de_len : static_cast<int>(round_up(std::min(f.unit, v), 64));
  const int dc_len = dc_cut ? f.dc_len : static_cast<int>(f.rows_pad);

  for (int64_t r0 = 0; r0 < b; r0 += f.rows) {
    const int64_t rows = std::min(f.rows, b - r0), rows_pad = round_up(rows, 64);
    const int64_t moved = valids == nullptr ? r0 : 0;  // without valids everything that is indexed by row moves with the block
    const int32_t* ids = valids != nullptr ? valids + r0 : nullptr;
    st = split_parts(e + moved * stride_e, stride_e, ids, rows, rows_pad, d, f.part_d, f.parts, e_parts, stream);
    if (st != CCE_OK) return st;
    for (int64_t v0 = 0; v0 < v; v0 += f.unit) {
      const int64_t cls = std::min(f.unit, v - v0), cls_pad = round_up(cls, 64);
      st = split_parts(c + v0 * stride_cv, stride_cv, nullptr, cls, round_up(cls, 256), d, f.part_d, f.parts, c_parts, stream);
      if (st != CCE_OK) return st;
      st = dz_terms_launch(e_parts, ld, c_parts, ld, bias != nullptr ? bias + v0 : nullptr, lse + r0,
                           d_out_is_scalar ? d_out : d_out + moved, d_out_is_scalar, d_lse != nullptr ? d_lse + moved : nullptr, ids,
                           targets + moved, dz_parts, cls_pad, n_rows - moved, rows, rows_pad, cls, f.part_d, terms, stored,
                           grad_scale, shift, target_offset + v0, softcap, stream);
      if (st != CCE_OK) return st;
      float* const de = d_e == nullptr ? nullptr : (de_cut ? de_slots : d_e + moved * ld_de);
      float* const dc = d_c == nullptr ? nullptr : (dc_cut ? dc_slots : d_c + v0 * ld_dc);
      st = terms_products_launch(dz_parts, cls_pad, c_parts, ld, e_parts, ld, de_cut ? nullptr : ids, de, de_cut ? f.part_d : ld_de,
                                 de_cut, de_cut && v0 == 0, rows * f.part_d, de_len, dc, dc_cut ? f.part_d : ld_dc, r0 > 0,
                                 cls * f.part_d, dc_len, out_vec, rows, rows_pad, cls, cls_pad, d, f.part_d, terms, stored, stream);
      if (st != CCE_OK) return st;
      if (dc_cut) {
        const int ranges = static_cast<int>((rows_pad + dc_len - 1) / dc_len);
        st = split_sum_launch(dc_slots, ranges, cls, d, f.part_d, nullptr, d_c + v0 * ld_dc, ld_dc, false, out_vec, stream);
        if (st != CCE_OK) return st;
      }
      if (d_bias != nullptr) {
        st = dz_colsum_launch(dz_parts, cls_pad, stored, rows, cls, d_bias + v0, CCE_DTYPE_BF16, stream);
        if (st != CCE_OK) return st;
      }
    }
    if (de_cut) {
      st = split_sum_launch(de_slots, f.de_slots, rows, d, f.part_d, ids, d_e + moved * ld_de, ld_de, true, out_vec, stream);
      if (st != CCE_OK) return st;
    }
  }
  return CCE_OK;
}
