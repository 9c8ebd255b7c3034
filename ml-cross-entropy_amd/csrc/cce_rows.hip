// The per-row work around the two big kernels: which rows of a batch count (cce_valid_rows), the loss of a row from the
// forward's partial sums (loss_rows_kernel), per-row values at their places in the batch and back, and the z-loss.  All are
// small and come with every call, so what they cost is launches: each replaces a chain of library kernels or of kernels of ours.
#include "cce_dense.h"

namespace cce {

// rows[0 .. count) = the positions p, in increasing order, whose label labels[p + shift] lies in the same sequence of
// `steps` labels and is not `ignored`.  One workgroup: 8192 positions per trip, eight independent loads per thread, a
// ballot per wave and load, one scan of the 128 counts.  (The library's boolean select takes seven launches for this and
// as many gaps: 45 us of host time per call, 31 us on the device for 4096 labels; this one is a single launch.)
// The count goes to host memory that the device can reach: the caller needs it to size everything else.
constexpr int kRowThreads = 1024, kRowLoads = 8;
__global__ __launch_bounds__(kRowThreads) void valid_rows_kernel(const int64_t* labels, int n, int steps, int shift, int64_t ignored,
                                                                 int32_t* rows, int64_t* count) {
  __shared__ int s_count[kRowLoads * 16];
  __shared__ int s_total;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0;
  for (int first = 0; first < n; first += kRowThreads * kRowLoads) {
    unsigned long long ballot[kRowLoads];
#pragma unroll
    for (int k = 0; k < kRowLoads; ++k) {
      const int p = first + k * kRowThreads + tid;
      bool keep = false;
      if (p < n && (shift == 0 || p % steps + shift < steps)) keep = labels[p + shift] != ignored;
      ballot[k] = __ballot(keep);
      if (lane == 0) s_count[k * 16 + wave] = __popcll(ballot[k]);
    }
    __syncthreads();
    if (wave == 0) {  // exclusive prefix sums of the 128 counts, two per lane
      const int a = s_count[2 * lane], b = s_count[2 * lane + 1];
      int incl = a + b;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
      }
      s_count[2 * lane] = incl - a - b;
      s_count[2 * lane + 1] = incl - b;
      if (lane == 63) s_total = incl;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kRowLoads; ++k) {
      if ((ballot[k] >> lane) & 1ull)
        rows[base + s_count[k * 16 + wave] + __popcll(ballot[k] & ((1ull << lane) - 1ull))] = first + k * kRowThreads + tid;
    }
    base += s_total;
    __syncthreads();  // the counts are read before the next trip writes them
  }
  // (a store that the host sees when it is made, not when the kernel has ended: cce_loss_call looks for it)
  if (tid == 0) __hip_atomic_store(count, static_cast<int64_t>(base), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[p] = values[r] where rows[r] + shift == p, 0 where there is no such r: the values of the valid rows (rows as
// valid_rows_kernel leaves them, in increasing order) at their places in the batch.  A search per position, all of it in
// cache; one launch in place of a fill, a widening, an addition and a scatter.
__global__ __launch_bounds__(256) void rows_to_batch_kernel(const float* values, const int32_t* rows, int count, int n, int shift,
                                                            float* out) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  int lo = 0, hi = count;  // the first r with rows[r] >= p - shift
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (rows[mid] < p - shift) lo = mid + 1;
    else hi = mid;
  }
  out[p] = (lo < count && rows[lo] == p - shift) ? values[lo] : 0.0f;
}

// Up to two sets of values at once, and the first `shift` steps of every sequence left out: out[s][j] of [n / steps][steps -
// shift] is the value of row s * steps + j.  With the z-loss's log-sum-exp beside a loss per token this is one launch of four (two
// searches, and autograd's zeros and copy for either slice on the way back, which steps_to_batch_kernel does in one).
struct TwoSets {
  const float* in[2];
  float* out[2];
};
__global__ __launch_bounds__(256) void rows_to_steps_kernel(TwoSets sets, const int32_t* rows, int count, int n_out, int steps, int kept) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= n_out) return;
  const int row = q / kept * steps + q % kept;
  int lo = 0, hi = count;  // the first r with rows[r] >= row
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (rows[mid] < row) lo = mid + 1;
    else hi = mid;
  }
  const bool found = lo < count && rows[lo] == row;
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (sets.out[k] != nullptr) sets.out[k][q] = found ? sets.in[k][lo] : 0.0f;
}

// The way back: out[s][j + shift] of [n / steps][steps] = in[s][j], zeros in the first `shift` steps.
__global__ __launch_bounds__(256) void steps_to_batch_kernel(TwoSets sets, int n, int steps, int shift) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= n) return;
  const int s = p / steps, j = p - s * steps - shift;
#pragma unroll
  for (int k = 0; k < 2; ++k)
    if (sets.out[k] != nullptr) sets.out[k][p] = j >= 0 ? sets.in[k][s * (steps - shift) + j] : 0.0f;
}

// The squares of log-sum-exps, zero where a label is ignored; as they are, or their sum or mean over what counts.  `rows`
// sequences of `cols` steps, either operand with a stride of its own from sequence to sequence (a slice of longer ones).
// Sums in fp64: one workgroup up to 16384 values, else partial sums of one workgroup each and another launch for them
// (fixed order, no atomics).  Launches are what it costs: with its gradient two of them, where the library's chain takes
// twelve (square, comparison, copy, fill, sum, count and division, and the same backwards).
struct ZLossParams {
  const float* lse;
  const int64_t* labels;  // nullptr: everything counts
  int64_t lse_stride, label_stride, ignored;
  int n, cols;
  uint8_t* kept;  // one byte per position, dense: the forward says which positions counted (nullptr: not wanted), the backward reads it
};
__device__ __forceinline__ bool z_loss_counts(const ZLossParams& p, int r, int c) {
  return p.labels == nullptr || p.labels[r * p.label_stride + c] != p.ignored;
}

constexpr int kZThreads = 1024, kZPerBlock = 16384, kZBlocks = 256;
struct ZPartial {
  double sum;
  int64_t count;
};
__device__ __forceinline__ ZPartial z_block_sum(ZPartial mine, ZPartial* s_part) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    mine.sum += __shfl_xor(mine.sum, off, 64);
    mine.count += __shfl_xor(static_cast<long long>(mine.count), off, 64);
  }
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = mine;
  __syncthreads();
  ZPartial all = {0.0, 0};
  if (threadIdx.x == 0) {
    for (int w = 0; w < kZThreads / 64; ++w) {
      all.sum += s_part[w].sum;
      all.count += s_part[w].count;
    }
  }
  return all;  // in thread 0
}
__device__ __forceinline__ void z_loss_result(const ZPartial& all, bool mean, float* out, float* count) {
  const float total = static_cast<float>(all.sum);
  *out = mean ? total / static_cast<float>(all.count) : total;
  if (count != nullptr) *count = static_cast<float>(all.count);
}

// SQUARE: the z-loss; else plain values, all of which count (the reduction of the loss itself)
template <bool SQUARE>
__global__ __launch_bounds__(kZThreads) void z_loss_sum_kernel(ZLossParams p, bool mean, ZPartial* partial, float* out, float* count) {
  __shared__ ZPartial s_part[kZThreads / 64];
  ZPartial mine = {0.0, 0};
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kZThreads + threadIdx.x; i < p.n; i += static_cast<int64_t>(gridDim.x) * kZThreads) {
    const int r = static_cast<int>(i) / p.cols, c = static_cast<int>(i) - r * p.cols;
    const bool counts = z_loss_counts(p, r, c);
    if (SQUARE && p.kept != nullptr) p.kept[i] = counts ? 1 : 0;
    if (counts) {
      const float x = p.lse[r * p.lse_stride + c];
      mine.sum += static_cast<double>(SQUARE ? x * x : x);
      ++mine.count;
    }
  }
  const ZPartial all = z_block_sum(mine, s_part);
  if (threadIdx.x != 0) return;
  if (gridDim.x == 1) z_loss_result(all, mean, out, count);
  else partial[blockIdx.x] = all;
}
__global__ __launch_bounds__(kZThreads) void z_loss_total_kernel(const ZPartial* partial, int blocks, bool mean, float* out, float* count) {
  __shared__ ZPartial s_part[kZThreads / 64];
  ZPartial mine = {0.0, 0};
  if (static_cast<int>(threadIdx.x) < blocks) mine = partial[threadIdx.x];
  const ZPartial all = z_block_sum(mine, s_part);
  if (threadIdx.x == 0) z_loss_result(all, mean, out, count);
}

// GRAD: the gradient of either, g the upstream value (one for a sum or mean, which divides by its count, or one per position)
template <bool GRAD>
__global__ __launch_bounds__(256) void z_loss_map_kernel(ZLossParams p, const float* grad, bool one_grad, const float* count, float* out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= p.n) return;
  const int r = static_cast<int>(i) / p.cols, c = static_cast<int>(i) - r * p.cols;
  const float x = p.lse[r * p.lse_stride + c];
  if (!GRAD) {
    const bool counts = z_loss_counts(p, r, c);
    if (p.kept != nullptr) p.kept[i] = counts ? 1 : 0;
    out[i] = counts ? x * x : 0.0f;
    return;
  }
  const bool counts = p.kept == nullptr || p.kept[i] != 0;
  float g = one_grad ? grad[0] : grad[i];
  if (count != nullptr) g /= count[0];
  out[i] = (counts ? g : 0.0f) * (2.0f * x);
}

// The loss of one valid row per wave: its log-sum-exp from the partial (max, sum) pairs of the vocabulary spans, and minus
// the soft-capped logit of its target, by a dot product of the two rows (0 where the target is no class of c), added up.
// Bound by the rows it reads; one launch in place of a merge, a dot product and an addition (12 - 25 us of a short call).
template <typename T, bool ALIGNED>
struct RowDot;
template <typename T>
struct RowDot<T, true> {
  static __device__ __forceinline__ float run(const uint16_t* a, const uint16_t* b, int64_t, int64_t d, int lane) {
    float acc = 0.0f;
    for (int64_t k = lane * 8; k < d; k += 512) {
      const uint4 x = *reinterpret_cast<const uint4*>(a + k), y = *reinterpret_cast<const uint4*>(b + k);
      const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, yw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc += Elem<T>::to_float(static_cast<uint16_t>(xw[j])) * Elem<T>::to_float(static_cast<uint16_t>(yw[j]));
        acc += Elem<T>::to_float(static_cast<uint16_t>(xw[j] >> 16)) * Elem<T>::to_float(static_cast<uint16_t>(yw[j] >> 16));
      }
    }
    return acc;
  }
};
template <typename T>
struct RowDot<T, false> {
  static __device__ __forceinline__ float run(const uint16_t* a, const uint16_t* b, int64_t stride_b, int64_t d, int lane) {
    float acc = 0.0f;
    for (int64_t k = lane; k < d; k += 64) acc += Elem<T>::to_float(a[k]) * Elem<T>::to_float(b[k * stride_b]);
    return acc;
  }
};
template <>
struct RowDot<float, true> {
  static __device__ __forceinline__ float run(const float* a, const float* b, int64_t, int64_t d, int lane) {
    float acc = 0.0f;
    for (int64_t k = lane * 4; k < d; k += 256) {
      const float4 x = *reinterpret_cast<const float4*>(a + k), y = *reinterpret_cast<const float4*>(b + k);
      acc = fmaf(x.x, y.x, acc);
      acc = fmaf(x.y, y.y, acc);
      acc = fmaf(x.z, y.z, acc);
      acc = fmaf(x.w, y.w, acc);
    }
    return acc;
  }
};
template <>
struct RowDot<float, false> {
  static __device__ __forceinline__ float run(const float* a, const float* b, int64_t stride_b, int64_t d, int lane) {
    float acc = 0.0f;
    for (int64_t k = lane; k < d; k += 64) acc = fmaf(a[k], b[k * stride_b], acc);
    return acc;
  }
};
template <typename T>
struct Stored {
  using type = uint16_t;
  static __device__ __forceinline__ float value(uint16_t x) { return Elem<T>::to_float(x); }
};
template <>
struct Stored<float> {
  using type = float;
  static __device__ __forceinline__ float value(float x) { return x; }
};

template <typename T, bool ALIGNED>
__global__ __launch_bounds__(256) void loss_rows_kernel(LossRowsParams p) {
  using S = typename Stored<T>::type;
  const int lane = threadIdx.x & 63;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (i >= p.b) return;
  const int64_t row = p.valids ? static_cast<int64_t>(p.valids[i]) : i;
  const int64_t at = row + p.shift;
  int64_t t = -1;
  if (at < p.n_rows) t = p.targets[at] - p.target_offset;
  const bool held = t >= 0 && t < p.v;  // wave-uniform

  float m = -INFINITY, sum = 0.0f;
  for (int s = lane; s < p.nsplit; s += 64) {
    const float2 x = p.partial[static_cast<int64_t>(s) * p.b + i];
    const float mn = fmaxf(m, x.x);
    const float ms = (mn == -INFINITY) ? 0.0f : mn;
    sum = sum * exp2f(m - ms) + x.y * exp2f(x.x - ms);
    m = mn;
  }
  float acc = 0.0f;
  if (held)
    acc = RowDot<T, ALIGNED>::run(static_cast<const S*>(p.e) + row * p.stride_e, static_cast<const S*>(p.c) + t * p.stride_cv,
                                  p.stride_cd, p.d, lane);
  // (a NaN row leaves (-inf, NaN) in its spans: the sum is scaled and never replaced, from a finite reference)
  const float top = wave_max(m);
  {
#pragma clang fp contract(off)  // rounded like the sums of the other lanes that it is added to
    sum = sum * exp2f(m - (top == -INFINITY ? 0.0f : top));
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    sum += __shfl_xor(sum, off, 64);
    acc += __shfl_xor(acc, off, 64);
  }
  if (lane == 0) {
    const float lse = (top + log2f(sum)) * kLn2;
    float r = 0.0f;
    if (held) {
      r = -acc;
      if (p.bias != nullptr) r -= Stored<T>::value(static_cast<const S*>(p.bias)[t]);
      if (p.softcap > 0.0f) r = tanhf(r / p.softcap) * p.softcap;
    }
    p.lse[i] = lse;
    p.nll[i] = r + lse;
  }
}

template <typename T>
static void launch_loss_rows(const LossRowsParams& p, bool aligned, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((p.b + 3) / 4));
  if (aligned) hipLaunchKernelGGL((loss_rows_kernel<T, true>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((loss_rows_kernel<T, false>), grid, dim3(256), 0, stream, p);
}

int loss_rows_launch(const LossRowsParams& p, int dtype, hipStream_t stream) {
  const int per16 = dtype == kLossRowsFp32 ? 4 : 8;
  const bool aligned = aligned16(p.e) && aligned16(p.c) && p.d % per16 == 0 && p.stride_e % per16 == 0 && p.stride_cv % per16 == 0 &&
                       p.stride_cd == 1;
  if (dtype == CCE_DTYPE_BF16) launch_loss_rows<BF16>(p, aligned, stream);
  else if (dtype == CCE_DTYPE_F16) launch_loss_rows<F16>(p, aligned, stream);
  else launch_loss_rows<float>(p, aligned, stream);
  return status_from_hip(hipGetLastError());
}

static int sum_blocks(int64_t n) {
  const int64_t wanted = (n + kZPerBlock - 1) / kZPerBlock;
  return static_cast<int>(wanted < 1 ? 1 : wanted > kZBlocks ? kZBlocks : wanted);
}
template <bool SQUARE>
static int sum_launch(const ZLossParams& p, int blocks, bool mean, ZPartial* partial, float* out, float* count, hipStream_t stream) {
  hipLaunchKernelGGL(z_loss_sum_kernel<SQUARE>, dim3(blocks), dim3(kZThreads), 0, stream, p, mean, partial, out, count);
  if (blocks > 1)
    hipLaunchKernelGGL(z_loss_total_kernel, dim3(1), dim3(kZThreads), 0, stream, partial, blocks, mean, out, count);
  return status_from_hip(hipGetLastError());
}

int64_t row_total_workspace_bytes(int64_t n) { return sum_blocks(n) > 1 ? kZBlocks * static_cast<int64_t>(sizeof(ZPartial)) : 0; }
int row_total_launch(const float* values, int64_t n, bool mean, float* out, void* workspace, hipStream_t stream) {
  const ZLossParams p = {values, nullptr, n, 0, 0, static_cast<int>(n), static_cast<int>(n > 0 ? n : 1), nullptr};
  return sum_launch<false>(p, sum_blocks(n), mean, static_cast<ZPartial*>(workspace), out, nullptr, stream);
}

}  // namespace cce

using namespace cce;

extern "C" int cce_valid_rows(const int64_t* labels, int64_t n, int64_t steps, int64_t shift, int64_t ignored, int32_t* rows,
                              int64_t* count, void* stream) {
  if (n < 0 || n >= (int64_t(1) << 31) - 8192 || steps <= 0 || shift < 0 || count == nullptr) return CCE_ERR_INVALID_ARGUMENT;
  if (n > 0 && (labels == nullptr || rows == nullptr || n % steps != 0)) return CCE_ERR_INVALID_ARGUMENT;
  if (shift >= steps && n > 0) shift = steps;  // no position has a label that far on
  hipLaunchKernelGGL(valid_rows_kernel, dim3(1), dim3(kRowThreads), 0, static_cast<hipStream_t>(stream), labels, static_cast<int>(n),
                     static_cast<int>(steps), static_cast<int>(shift), ignored, rows, count);
  return status_from_hip(hipGetLastError());
}

extern "C" int cce_rows_to_batch(const float* values, const int32_t* rows, int64_t count, int64_t n, int64_t shift, float* out,
                                 void* stream) {
  if (n < 0 || n >= (int64_t(1) << 31) - 8192 || count < 0 || count > n || shift < 0) return CCE_ERR_INVALID_ARGUMENT;
  if (n == 0) return CCE_OK;
  if (out == nullptr || (count > 0 && (values == nullptr || rows == nullptr))) return CCE_ERR_INVALID_ARGUMENT;
  if (shift > n) count = 0;  // no position is that far on
  hipLaunchKernelGGL(rows_to_batch_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), values, rows, static_cast<int>(count), static_cast<int>(n),
                     static_cast<int>(shift > n ? 0 : shift), out);
  return status_from_hip(hipGetLastError());
}

extern "C" int cce_rows_to_steps(const float* first, const float* second, const int32_t* rows, int64_t count, int64_t n, int64_t steps,
                                 int64_t shift, float* out_first, float* out_second, void* stream) {
  if (n < 0 || n >= (int64_t(1) << 31) - 8192 || count < 0 || count > n || shift < 0) return CCE_ERR_INVALID_ARGUMENT;
  if (n == 0) return CCE_OK;  // (sequences of no steps among them)
  if (steps <= 0) return CCE_ERR_INVALID_ARGUMENT;
  if (shift >= steps) return CCE_OK;
  if (n % steps != 0 || (count > 0 && rows == nullptr)) return CCE_ERR_INVALID_ARGUMENT;
  if (count > 0 && ((out_first != nullptr && first == nullptr) || (out_second != nullptr && second == nullptr)))
    return CCE_ERR_INVALID_ARGUMENT;
  const int n_out = static_cast<int>(n / steps * (steps - shift));
  const TwoSets sets = {{first, second}, {out_first, out_second}};
  hipLaunchKernelGGL(rows_to_steps_kernel, dim3((n_out + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), sets, rows,
                     static_cast<int>(count), n_out, static_cast<int>(steps), static_cast<int>(steps - shift));
  return status_from_hip(hipGetLastError());
}

extern "C" int cce_steps_to_batch(const float* first, const float* second, int64_t n, int64_t steps, int64_t shift, float* out_first,
                                  float* out_second, void* stream) {
  if (n < 0 || n >= (int64_t(1) << 31) - 8192 || shift < 0) return CCE_ERR_INVALID_ARGUMENT;
  if (n == 0) return CCE_OK;
  if (steps <= 0 || shift > steps) return CCE_ERR_INVALID_ARGUMENT;
  if (n % steps != 0 || (out_first != nullptr && first == nullptr) || (out_second != nullptr && second == nullptr))
    return CCE_ERR_INVALID_ARGUMENT;
  const TwoSets sets = {{first, second}, {out_first, out_second}};
  hipLaunchKernelGGL(steps_to_batch_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), sets, static_cast<int>(n), static_cast<int>(steps), static_cast<int>(shift));
  return status_from_hip(hipGetLastError());
}

static int z_loss_check(const float* lse, int64_t rows, int64_t cols, int64_t* n) {
  if (rows < 0 || cols < 0) return CCE_ERR_INVALID_ARGUMENT;
  if (cols > 0 && rows > ((int64_t(1) << 31) - 8192) / cols) return CCE_ERR_INVALID_ARGUMENT;
  *n = rows * cols;
  return (*n > 0 && lse == nullptr) ? CCE_ERR_INVALID_ARGUMENT : CCE_OK;
}

extern "C" int64_t cce_z_loss_workspace_bytes(int64_t rows, int64_t cols) {
  return rows > 0 && cols > 0 && rows * cols > kZPerBlock ? kZBlocks * static_cast<int64_t>(sizeof(ZPartial)) : 0;
}

extern "C" int cce_z_loss_forward(const float* lse, int64_t lse_stride, const int64_t* labels, int64_t label_stride, int64_t rows,
                                  int64_t cols, int64_t ignored, int reduction, float* out, float* count, uint8_t* kept,
                                  void* workspace, int64_t workspace_bytes, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  int64_t n = 0;
  const int st = z_loss_check(lse, rows, cols, &n);
  if (st != CCE_OK) return st;
  if (reduction < CCE_REDUCTION_NONE || reduction > CCE_REDUCTION_MEAN) return CCE_ERR_INVALID_ARGUMENT;
  if (out == nullptr && (n > 0 || reduction != CCE_REDUCTION_NONE)) return CCE_ERR_INVALID_ARGUMENT;
  const ZLossParams p = {lse, labels, lse_stride, label_stride, ignored, static_cast<int>(n), static_cast<int>(cols > 0 ? cols : 1), kept};
  if (reduction == CCE_REDUCTION_NONE) {
    if (n == 0) return CCE_OK;
    hipLaunchKernelGGL(z_loss_map_kernel<false>, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream, p, nullptr, false,
                       nullptr, out);
    return status_from_hip(hipGetLastError());
  }
  const bool mean = reduction == CCE_REDUCTION_MEAN;
  const int blocks = sum_blocks(n);
  if (blocks > 1 && (workspace == nullptr || workspace_bytes < cce_z_loss_workspace_bytes(rows, cols)))
    return CCE_ERR_WORKSPACE_TOO_SMALL;
  if ((reinterpret_cast<uintptr_t>(workspace) & 7u) != 0) return CCE_ERR_MISALIGNED;
  ZPartial* const partial = static_cast<ZPartial*>(workspace);
  return sum_launch<true>(p, blocks, mean, partial, out, count, stream);
}

extern "C" int cce_z_loss_backward(const float* lse, int64_t lse_stride, const uint8_t* kept, int64_t rows, int64_t cols,
                                   const float* grad, int grad_is_scalar, const float* count, float* d_lse, void* stream) {
  int64_t n = 0;
  const int st = z_loss_check(lse, rows, cols, &n);
  if (st != CCE_OK || n == 0) return st;
  if (grad == nullptr || d_lse == nullptr) return CCE_ERR_INVALID_ARGUMENT;
  const ZLossParams p = {lse, nullptr, lse_stride, 0, 0, static_cast<int>(n), static_cast<int>(cols), const_cast<uint8_t*>(kept)};
  hipLaunchKernelGGL(z_loss_map_kernel<true>, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), p, grad, grad_is_scalar != 0, count, d_lse);
  return status_from_hip(hipGetLastError());
}
