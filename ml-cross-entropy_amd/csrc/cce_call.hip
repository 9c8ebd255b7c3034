// The forward of one call of the operator: which rows count, how many they are, and everything that is sized by that number.
//
// The number is known on the device first, and the launches behind it are planned from it (row blocks, vocabulary spans),
// so the host has to read it.  With the wait in the caller the device idled from the end of the first kernel until the caller had woken
// up, allocated, and reached the next launch: 70 - 110 us of every call, whatever its size.  Here the caller has prepared
// everything before the first launch (buffers sized by all rows), the wait is a look at a word of pinned memory, and the next launch
// follows from C++: some 10 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>

#include "cce_dense.h"

namespace cce {

static int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Fewer rows may be cut into more spans than all of them would be.  The room for that: two rounds of workgroups' partial sums.
constexpr int64_t kSpareBytes = int64_t(1) << 20;

static int64_t partial_bytes(int64_t n, int64_t v, int64_t d, int dtype, int terms) {
  const int64_t need = dtype == CCE_DTYPE_F32 ? cce_fp32_forward_workspace_bytes(n, v, d, terms) : cce_lse_forward_workspace_bytes(n, v, d);
  return align256(need + kSpareBytes);
}

// The count that a kernel enqueued on `stream` stores to *word, which held -1 before.  The store is seen a microsecond after it is made;
// a wait that takes longer (a stream with much before it) is left to the runtime, which also knows of errors.
static int wait_for_count(const int64_t* word, hipStream_t stream, int64_t* count) {
  const auto start = std::chrono::steady_clock::now();
  for (;;) {
    for (int i = 0; i < 64; ++i) {
      *count = __atomic_load_n(word, __ATOMIC_ACQUIRE);
      if (*count >= 0) return CCE_OK;
      __builtin_ia32_pause();
    }
    if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(1)) break;
  }
  const hipError_t err = hipStreamSynchronize(stream);
  if (err != hipSuccess) return status_from_hip(err);
  *count = __atomic_load_n(word, __ATOMIC_ACQUIRE);
  return *count >= 0 ? CCE_OK : status_from_hip(hipErrorUnknown);
}

}  // namespace cce

using namespace cce;

extern "C" int64_t cce_loss_call_workspace_bytes(int64_t n, int64_t v, int64_t d, int dtype, int terms) {
  if (n <= 0 || v <= 0 || d <= 0) return 0;
  return partial_bytes(n, v, d, dtype, terms) + align256(n * 4) + align256(row_total_workspace_bytes(n));
}

extern "C" int cce_loss_call(const void* e, const void* c, const void* bias, const int64_t* labels, int32_t* rows, int64_t* count,
                             float* lse, float* tile_max, float* loss, float* lse_out, void* workspace, int64_t workspace_bytes,
                             int64_t n, int64_t steps, int64_t v, int64_t d, int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                             int64_t shift, int64_t ignored, int64_t target_offset, float softcap, int reduction, int dtype, int terms,
                             void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  // before anything is refused: a caller that keeps the word from call to call can tell a refusal from rows that are written
  if (count != nullptr) __atomic_store_n(count, int64_t(-1), __ATOMIC_RELEASE);
  if (n <= 0 || steps <= 0 || n % steps != 0 || shift < 0 || shift >= steps || v <= 0 || d <= 0) return CCE_ERR_INVALID_ARGUMENT;
  if (reduction < CCE_REDUCTION_NONE || reduction > CCE_REDUCTION_MEAN) return CCE_ERR_INVALID_ARGUMENT;
  if (dtype != CCE_DTYPE_BF16 && dtype != CCE_DTYPE_F16 && dtype != CCE_DTYPE_F32) return CCE_ERR_UNSUPPORTED_DTYPE;
  if (e == nullptr || c == nullptr || labels == nullptr || rows == nullptr || count == nullptr || lse == nullptr || loss == nullptr)
    return CCE_ERR_INVALID_ARGUMENT;
  if (workspace == nullptr || workspace_bytes < cce_loss_call_workspace_bytes(n, v, d, dtype, terms)) return CCE_ERR_WORKSPACE_TOO_SMALL;
  if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return CCE_ERR_MISALIGNED;
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  hipError_t err = hipStreamIsCapturing(stream, &capturing);
  if (err != hipSuccess) return status_from_hip(err);
  if (capturing != hipStreamCaptureStatusNone) return status_from_hip(hipErrorStreamCaptureUnsupported);  // nothing would run

  int st = cce_valid_rows(labels, n, steps, shift, ignored, rows, count, stream_);
  if (st != CCE_OK) return st;
  int64_t b = 0;
  st = wait_for_count(count, stream, &b);
  if (st != CCE_OK) return st;

  unsigned char* const ws = static_cast<unsigned char*>(workspace);
  const int64_t room = partial_bytes(n, v, d, dtype, terms);
  void* const totals = ws + room + align256(n * 4);
  const bool all = shift == 0 && b == n;  // rows as they lie need no list, and their values have their places
  const int32_t* const valids = all ? nullptr : rows;
  float* const nll = (all && reduction == CCE_REDUCTION_NONE) ? loss : reinterpret_cast<float*>(ws + room);
  if (b > 0) {
    if (dtype == CCE_DTYPE_F32)
      st = cce_fp32_forward(static_cast<const float*>(e), static_cast<const float*>(c), static_cast<const float*>(bias), valids, labels,
                            lse, nll, ws, room, n, b, v, d, stride_e, stride_cv, stride_cd, shift, target_offset, softcap, terms,
                            stream_);
    else
      st = cce_loss_forward(e, c, bias, valids, labels, lse, nll, tile_max, ws, room, n, b, v, d, stride_e, stride_cv, stride_cd, shift,
                            target_offset, softcap, dtype, stream_);
    if (st != CCE_OK) return st;  // (CCE_ERR_WORKSPACE_TOO_SMALL: rows and *count are there all the same)
  }
  if (!all && (reduction == CCE_REDUCTION_NONE || lse_out != nullptr)) {
    st = cce_rows_to_steps(nll, lse, rows, b, n, steps, shift, reduction == CCE_REDUCTION_NONE ? loss : nullptr, lse_out, stream_);
    if (st != CCE_OK) return st;
  }
  if (reduction != CCE_REDUCTION_NONE) st = row_total_launch(nll, b, reduction == CCE_REDUCTION_MEAN, loss, totals, stream);
  return st;
}
