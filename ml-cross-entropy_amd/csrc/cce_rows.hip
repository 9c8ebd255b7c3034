// The per-row work around the two big kernels: which rows of a batch count (cce_valid_rows), and the loss of a row from
// the forward's partial sums (loss_rows_kernel).  Both are small and come with every call, so what they cost is launches:
// each replaces a chain of library kernels or of kernels of ours.
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
  if (tid == 0) *count = base;
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
