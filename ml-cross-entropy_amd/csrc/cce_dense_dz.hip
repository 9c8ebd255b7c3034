// cce_backward_dz: the gradient of the loss with respect to the logits of one vocabulary chunk,
//     dz[i, j] = (p_ij (g_i + h_i) - [j == target_i] g_i) (1 - tanh^2)      p_ij = exp(s_ij - lse_i)
// written to memory in the input type (or as fp32), for the unfiltered ("exact") backward: with every entry of
// the gradient in play the two products dE = dz . C and dC = dz^T . E are dense matrix products over the chunk,
// which the kernels of cce_backward_dense.hip run.  The kernel is the forward kernel with another epilogue: same work
// items, same direct-to-LDS main loop, logits never leave the registers; only dz does, as row pieces of 128
// contiguous bytes (8 rows per wave instruction) after a transposition through LDS, while the first stages of the
// next tile are already arriving.
#include <type_traits>

#include "cce_dense.h"

namespace cce {

struct DzParams {
  const uint16_t* e;
  const uint16_t* c;
  const uint16_t* bias;
  const int32_t* valids;
  const float* lse;
  const float* d_out;
  const float* d_lse;
  const int64_t* targets;
  void* dz;
  int64_t ldz;
  int64_t n_rows, b, v, d;
  int64_t stride_e, stride_cv;
  int64_t shift, target_offset;
  float grad_scale;
  int d_out_is_scalar;
  int pad_store;  // also store the (zero) gradients of the classes between v and the end of their 16-byte piece,
                  // up to column ldz: the product kernels read dz in whole 64-class stages
  int nrb, nvt, nsplit, nitems, items_per_xcd;
  int block_rows, block_spans;  // the order of the items (item_place)
  Softcap sc;
  // operands and dz in 16-bit parts (kDzParts): d is the width of a part, rows of e are compact (valids only says which
  // targets and upstream gradients they belong to), dz is [b_store][parts][ldz], rows past b zeros
  const float* bias32;
  int terms, parts;
  int64_t b_store;
  // *wide == 0: the logits from halves, two to a row and packed, whose product is 1 / halves_scale times the logit
  const int* wide;
  const uint16_t* e_halves;
  const uint16_t* c_halves;
  float halves_scale;
};

// How dz leaves: in the input type, as fp32, or as an fp32 value in two or three bf16 parts
enum DzOut { kDz16Bit, kDzFp32, kDzParts };

constexpr int kDzWV = 4, kDzWT = 2, kDzNWV = 2, kDzNWT = 4;  // the forward kernel's wave tiling
constexpr int kDzThreads = 64 * kDzNWV * kDzNWT;
constexpr int kDzTile = 256;
constexpr int kDzStageRow = 128;                  // bytes of one row of a wave's staged block (64 x 16-bit or 32 x fp32)
constexpr int kDzStageBytes = 32 * kDzStageRow;   // 32 rows

// OUT32: dz leaves as fp32 (for inputs that are fp32 values split into 16-bit parts along D, whose
// gradients are wanted at fp32 accuracy): a staged block is then 32 rows x 32 classes.
template <typename T, bool GENERAL, bool OUT32>
__global__ __launch_bounds__(kDzThreads, 1) void dense_dz_kernel(DzParams p) {
  using Fast = DmaLogitTile<T, kDzWV, kDzWT, kDzNWV, kDzNWT>;
  static_assert(kDzStageBytes * kDzNWV * kDzNWT <= Fast::TILE_T * kDmaRowBytes, "the staging blocks fit the token half of a stage");
  extern __shared__ __align__(16) unsigned char smem[];
  float* s_addend = reinterpret_cast<float*>(smem + Fast::LDS_BYTES);  // [2][256]

  const int xcd = blockIdx.x & 7;
  const int slot = blockIdx.x >> 3;
  if (slot >= p.items_per_xcd) return;
  const int item = xcd * p.items_per_xcd + slot;
  if (item >= p.nitems) return;
  int rb, split;
  item_place(item, p.nrb, p.nsplit, p.block_rows, p.block_spans, rb, split);
  const int vt_begin = static_cast<int>((static_cast<int64_t>(p.nvt) * split) / p.nsplit);
  const int vt_end = static_cast<int>((static_cast<int64_t>(p.nvt) * (split + 1)) / p.nsplit);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wv = wave / kDzNWT;
  const int wt = wave % kDzNWT;
  const int l32 = lane & 31;
  const int half = lane >> 5;
  const int64_t t0 = static_cast<int64_t>(rb) * kDzTile;

  const uint16_t* fptr[Fast::NQ];
#pragma unroll
  for (int q = Fast::NQC; q < Fast::NQ; ++q) {
    int64_t i = t0 + Fast::row_of(q, wave, lane);
    i = (i < p.b) ? i : p.b - 1;  // rows past the end repeat the last one; their results are dropped
    const int64_t row = p.valids ? static_cast<int64_t>(p.valids[i]) : i;
    fptr[q] = p.e + row * p.stride_e + Fast::chunk_elems(wave, lane);
  }

  // The two rows of this lane (one per 32-row column block): fixed for the whole item.
  float r_lse2[kDzWT], r_g[kDzWT], r_h[kDzWT];
  int r_tgt[kDzWT];
#pragma unroll
  for (int ti = 0; ti < kDzWT; ++ti) {
    const int64_t i = t0 + wt * (32 * kDzWT) + ti * 32 + l32;
    float lse2 = INFINITY, g = 0.0f, h = 0.0f;
    int tgt = -1;
    if (i < p.b) {
      const int64_t row = p.valids ? static_cast<int64_t>(p.valids[i]) : i;
      lse2 = p.lse[i] * kLog2e;
      const int64_t tpos = row + p.shift;
      if (tpos < p.n_rows) {
        const int64_t t = p.targets[tpos] - p.target_offset;
        if (t >= 0 && t < p.v) tgt = static_cast<int>(t);
        g = p.grad_scale * (p.d_out_is_scalar ? p.d_out[0] : p.d_out[tpos]);
        if (p.d_lse != nullptr) h = p.d_lse[tpos];
      }
    }
    r_lse2[ti] = lse2;
    r_g[ti] = g;
    r_h[ti] = h;
    r_tgt[ti] = tgt;
  }

  // Staged blocks live in the token half of LDS stage 1, the one part of the ring that the early fetch of the
  // next tile (all of stage 0, the class half of stage 1) leaves alone.
  unsigned char* stage = smem + Fast::STAGE_BYTES + Fast::TILE_V * kDmaRowBytes + wave * kDzStageBytes;

  auto point_at_tile = [&](int vt) {
    const int64_t v0 = static_cast<int64_t>(vt) * kDzTile;
#pragma unroll
    for (int q = 0; q < Fast::NQC; ++q) {
      int64_t vr = v0 + Fast::row_of(q, wave, lane);
      vr = (vr < p.v) ? vr : p.v - 1;  // classes past the end repeat the last one; masked below
      fptr[q] = p.c + vr * p.stride_cv + Fast::chunk_elems(wave, lane);
    }
  };
  if (vt_begin < vt_end) {
    point_at_tile(vt_begin);
    Fast::prefetch(fptr, smem, static_cast<int>(p.d));
  }

  for (int vt = vt_begin; vt < vt_end; ++vt) {
    const int64_t v0 = static_cast<int64_t>(vt) * kDzTile;
    float* addend = s_addend + (vt & 1) * kDzTile;
    if (GENERAL) {
      if (tid < kDzTile) {  // published by the barriers of the main loop
        const int64_t vg = v0 + tid;
        float a = -INFINITY;
        if (vg < p.v) a = (p.bias != nullptr) ? Elem<T>::to_float(p.bias[vg]) : 0.0f;
        addend[tid] = a;
      }
    }
    f32x16 acc[kDzWV][kDzWT];
    Fast::run(acc, fptr, smem, static_cast<int>(p.d));  // (ends with a barrier: the ring is idle)
    // The next tile starts to arrive while this one's gradients are formed and stored.  Its loads sit ahead of the
    // stores below in the queue the main loop counts by: loads complete in order among themselves, so "at most QA
    // operations outstanding" at the top of run() still means that stage 0 has landed.
    if (vt + 1 < vt_end) {
      point_at_tile(vt + 1);
      Fast::prefetch(fptr, smem, static_cast<int>(p.d));
    }

    const int cls0 = static_cast<int>(v0) + wv * (32 * kDzWV);  // first class of this wave
    const float* wave_addend = addend + wv * (32 * kDzWV);
    const int sw = (l32 >> 1) & 7;  // 16-byte chunks of a staged row are XOR-swizzled with (row >> 1) & 7
#pragma unroll
    for (int ti = 0; ti < kDzWT; ++ti) {
      const float lse2 = r_lse2[ti], g = r_g[ti], gh = r_g[ti] + r_h[ti];
      const int tgt = r_tgt[ti];
      constexpr int kEs = OUT32 ? 4 : 2;                    // bytes per stored element
      constexpr int kViPer = kDzStageRow / (32 * kEs);      // 32-class blocks per staged block (2, or 1 for fp32)
      constexpr int kParts = kDzWV / kViPer;                // staged blocks per column block
      constexpr int kPieceElems = 16 / kEs;                 // elements per 16-byte piece
#pragma unroll
      for (int vh = 0; vh < kParts; ++vh) {
        // The gradients of one staged block.  One copy of the arithmetic per answer to "soft-capped?": asked per
        // logit, the (uniform) question costs two branches per element, a third of the epilogue's time.
        auto stage_block = [&](auto capped) {
#pragma unroll
          for (int vj = 0; vj < kViPer; ++vj) {
            const int vi = vh * kViPer + vj;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
              float dzv[4];
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int cl = vi * 32 + 8 * r4 + 4 * half + i;
                float x = acc[vi][ti][r4 * 4 + i];
                bool dead = false;
                if (GENERAL) {
                  const float add = wave_addend[cl];
                  dead = (add == -INFINITY);
                  x = dead ? 0.0f : x + add;
                }
                float s2, damp = 1.0f;
                if (decltype(capped)::value) {
                  const float t = __builtin_amdgcn_exp2f(x * p.sc.in_scale);
                  const float w = __builtin_amdgcn_rcpf(1.0f + t);
                  const float th = 1.0f - 2.0f * w;
                  s2 = p.sc.out_scale * th;
                  damp = 1.0f - th * th;
                } else {
                  s2 = x * kLog2e;
                }
                const float pr = __builtin_amdgcn_exp2f(s2 - lse2);
                float dz = pr * gh - ((cls0 + cl == tgt) ? g : 0.0f);
                if (decltype(capped)::value) dz *= damp;
                dzv[i] = dead ? 0.0f : dz;
              }
              const int col = (vj * 32 + 8 * r4 + 4 * half) * kEs;  // byte inside the staged row
              unsigned char* dst = stage + l32 * kDzStageRow + ((((col >> 4) ^ sw) << 4) | (col & 15));
              if (OUT32) {
                *reinterpret_cast<float4*>(dst) = make_float4(dzv[0], dzv[1], dzv[2], dzv[3]);
              } else {
                uint2 pk;
                pk.x = Elem<T>::pack2(dzv[0], dzv[1]);
                pk.y = Elem<T>::pack2(dzv[2], dzv[3]);
                *reinterpret_cast<uint2*>(dst) = pk;
              }
            }
          }
        };
        if (p.sc.on) {
          stage_block(std::true_type{});
        } else {
          stage_block(std::false_type{});
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the block is private to this wave: no barrier
        // 32 rows x 128 bytes leave as 16-byte pieces: one instruction covers 8 rows of 128 contiguous bytes
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int j = lane + 64 * k;
          const int row = j >> 3;
          const int pc = j & 7;
          const uint4 val = *reinterpret_cast<const uint4*>(stage + row * kDzStageRow + ((pc ^ ((row >> 1) & 7)) << 4));
          const int64_t gi = t0 + wt * (32 * kDzWT) + ti * 32 + row;
          const int64_t gcol = static_cast<int64_t>(cls0) + vh * (32 * kViPer) + pc * kPieceElems;
          if (gi < p.b) {
            unsigned char* dst = static_cast<unsigned char*>(p.dz) + (gi * p.ldz + gcol) * kEs;
            if (!GENERAL || gcol + kPieceElems <= p.v || (p.pad_store && gcol + kPieceElems <= p.ldz)) {
              *reinterpret_cast<uint4*>(dst) = val;
            } else if (OUT32) {
              const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (gcol + i < p.v) reinterpret_cast<uint32_t*>(dst)[i] = w[i];
            } else {
              const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (gcol + i < p.v) reinterpret_cast<uint16_t*>(dst)[i] = static_cast<uint16_t>(w[i >> 1] >> ((i & 1) * 16));
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next block is staged
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same kernel on the 16 x 16 x 32 main loop (DmaLogitTile16).  A lane holds, per 16-row block ti of its wave,
// ONE token row (lane % 16) and the classes 16 vi + 4 (lane / 16) + r of the wave's 128 (64); what a row needs (its
// log-sum-exp, upstream gradients, target) sits in LDS, one entry per row of the workgroup, instead of in
// registers.  The whole ring is busy during the epilogue (the main loop fetches both first stages of the next
// tile under its last two stages), so the staging blocks have LDS of their own: 16 rows x 128 bytes per wave,
// 64 classes of a row block at a time.
// ---------------------------------------------------------------------------------------------
constexpr int kDz16WV = 8, kDz16WT = 4;
constexpr int kDz16StageBytes = 16 * kDzStageRow;  // 16 rows of 128 bytes per wave

struct DzRow {
  float lse2, g, gh;
  int tgt;
};

// 2^(x2 - lse2) for gradients in fp32.  The difference as a whole number and a fraction of up to a half: rounded as one number, of 16 or so, it
// is off by 2^-21, and the result by as much.  x2, and lse2 = log-sum-exp times kLog2e, are rounded as they were in the forward, also by its
// soft-capping factor: of a row that one logit makes up it is that logit again, and the difference 0 (as a difference of natural
// logarithms it was 5e-7 there, and one with a factor of its own 9e-8 of a soft-capped logit).  Where they are far apart, lse2 falls short
// of the forward's by kLog2Slack of itself, which is of the difference.
// Distance from 64 bits, 2-norm, as a difference rounded as one number / of natural logarithms / so: dE of [64, 1000] x [50003, 1000] with soft-cap
// 30 2.57e-7 / 2.26e-7 / 2.09e-7, of [500, 2048] x [20000, 2048] 3.29e-7 / 3.1e-7 / 2.42e-7, of [400, 3072] x [3000, 3072] with targets of logits up
// to 15 8.09e-7 / 7.75e-7 / 8.00e-7, and with soft-cap 30 1.49e-6 / 1.73e-6 / 1.48e-6.  Six instructions per logit: nothing to be seen in
// the time of [2046, 3072] x [32064, 3072].
__device__ __forceinline__ float exp2_difference(float x2, float lse2) {
  const float n = __builtin_amdgcn_fmed3f(rintf(x2 - lse2), -256.0f, 256.0f);  // (rows past the end: lse2 = infinity, and 0)
  const float f = fmaf(n, kLog2Slack, x2 - (n + lse2));  // n + lse2: exact unless x2 is past lse2
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), static_cast<int>(n));
}

// Who holds what of a tile of ROWS x 256: 2 x 4 waves of 128 classes x 64 rows, or 4 x 2 of 64 x 96.
template <int ROWS>
struct Dz16Shape {
  static_assert(ROWS == kDzTile || ROWS == kMidRowBlock, "rows of a tile");
  static constexpr bool MID = ROWS == kMidRowBlock;
  static constexpr int WV = MID ? 4 : kDz16WV, WT = MID ? 6 : kDz16WT;
  static constexpr int NWV = MID ? 4 : kDzNWV, NWT = MID ? 2 : kDzNWT;
  template <typename T, bool PARTS, bool TAIL>
  using Tile = DmaLogitTile16<T, WV, WT, NWV, NWT, PARTS, TAIL>;
  static constexpr int LDS_BYTES =
      Tile<BF16, false, false>::LDS_BYTES + 2 * kDzTile * 4 + ROWS * static_cast<int>(sizeof(DzRow)) + NWV * NWT * kDz16StageBytes;
};

template <typename T, bool GENERAL, DzOut OUT, bool TAIL = false, int ROWS = kDzTile>
__device__ __forceinline__ void dense_dz16_item(const DzParams& p) {
  constexpr bool OUT32 = OUT == kDzFp32;
  constexpr bool PARTS = OUT == kDzParts;
  constexpr bool HALVES = PARTS && std::is_same<T, F16>::value;
  using Shape = Dz16Shape<ROWS>;
  constexpr int WV = Shape::WV, WT = Shape::WT;
  using Fast = typename Shape::template Tile<T, PARTS, TAIL>;
  extern __shared__ __align__(16) unsigned char smem[];
  float* s_addend = reinterpret_cast<float*>(smem + Fast::LDS_BYTES);                                   // [2][256]
  DzRow* s_rows = reinterpret_cast<DzRow*>(smem + Fast::LDS_BYTES + 2 * kDzTile * 4);                    // [ROWS]
  unsigned char* s_stage = smem + Fast::LDS_BYTES + 2 * kDzTile * 4 + ROWS * sizeof(DzRow);              // [8 waves]

  const int xcd = blockIdx.x & 7;
  const int slot = blockIdx.x >> 3;
  if (slot >= p.items_per_xcd) return;
  const int item = xcd * p.items_per_xcd + slot;
  if (item >= p.nitems) return;
  int rb, split;
  item_place(item, p.nrb, p.nsplit, p.block_rows, p.block_spans, rb, split);
  const int vt_begin = static_cast<int>((static_cast<int64_t>(p.nvt) * split) / p.nsplit);
  const int vt_end = static_cast<int>((static_cast<int64_t>(p.nvt) * (split + 1)) / p.nsplit);
  if (vt_begin >= vt_end) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wv = wave / Shape::NWT;
  const int wt = wave % Shape::NWT;
  const int r16 = lane & 15;
  const int kq = lane >> 4;
  const int64_t t0 = static_cast<int64_t>(rb) * ROWS;

  typename Fast::Source src;
  src.e_base = reinterpret_cast<const unsigned char*>(HALVES ? p.e_halves : p.e);
  src.chunk_bytes = 2u * static_cast<unsigned>(Fast::chunk_elems(wave, lane));
  src.row_in_block = static_cast<unsigned>(lane >> 3);
  const int64_t stride_e = HALVES ? kHalvesParts * p.d : p.stride_e, stride_cv = HALVES ? kHalvesParts * p.d : p.stride_cv;
  src.c_stride_bytes = static_cast<unsigned>(stride_cv * 2);
  src.terms = !PARTS ? 1 : HALVES ? kHalvesTerms : p.terms;
  // a sum in an accumulator times `unit` is a logit (a power of two); without an addend it rides in the first factor
  const float unit = HALVES ? p.halves_scale : 1.0f;
  const float in_scale = GENERAL ? p.sc.in_scale : p.sc.in_scale * unit;
  const float log2e = GENERAL ? kLog2e : kLog2e * unit;
  if constexpr (TAIL) Fast::set_tail(src, static_cast<int>(p.d));
#pragma unroll
  for (int q = Fast::NQC; q < Fast::NQ; ++q) {
    int64_t i = t0 + Fast::row_of(q, wave, lane);
    i = (i < p.b) ? i : p.b - 1;  // rows past the end repeat the last one; their results are dropped
    const int64_t row = (!PARTS && p.valids) ? static_cast<int64_t>(p.valids[i]) : i;
    src.e_off[q - Fast::NQC] = static_cast<unsigned>(row * stride_e * 2) + src.chunk_bytes;
  }
  auto set_class_tile = [&](int vt) {
    const int64_t v0 = static_cast<int64_t>(vt) * kDzTile;
    const int left = static_cast<int>(min(p.v - v0, static_cast<int64_t>(kDzTile)));
    Fast::set_class_tile(src, reinterpret_cast<const unsigned char*>(HALVES ? p.c_halves : p.c) + v0 * stride_cv * 2, left, wave);
  };

  unsigned char* stage = s_stage + wave * kDz16StageBytes;
  int buf = 0;
  set_class_tile(vt_begin);
  Fast::prefetch(src, smem, static_cast<int>(p.d));
  // What the rows of this workgroup need, fixed for the whole item (published by the first barrier of the main loop;
  // fetched behind the first stages of the ring, so that the two latencies overlap).
  if (tid < ROWS) {
    const int64_t i = t0 + tid;
    DzRow r = {INFINITY, 0.0f, 0.0f, -1};
    if (i < p.b) {
      const int64_t row = p.valids ? static_cast<int64_t>(p.valids[i]) : i;
      r.lse2 = p.lse[i] * kLog2e;
      const int64_t tpos = row + p.shift;
      if (tpos < p.n_rows) {
        const int64_t t = p.targets[tpos] - p.target_offset;
        if (t >= 0 && t < p.v) r.tgt = static_cast<int>(t);
        r.g = p.grad_scale * (p.d_out_is_scalar ? p.d_out[0] : p.d_out[tpos]);
        r.gh = r.g + ((p.d_lse != nullptr) ? p.d_lse[tpos] : 0.0f);
      }
    }
    s_rows[tid] = r;
  }

  for (int vt = vt_begin; vt < vt_end; ++vt) {
    const int64_t v0 = static_cast<int64_t>(vt) * kDzTile;
    float* addend = s_addend + (vt & 1) * kDzTile;
    if (GENERAL) {
      if (tid < kDzTile) {  // published by the barriers of the main loop
        const int64_t vg = v0 + tid;
        float a = -INFINITY;
        if (vg < p.v) {
          if (PARTS) a = (p.bias32 != nullptr) ? p.bias32[vg] : 0.0f;
          else a = (p.bias != nullptr) ? Elem<T>::to_float(p.bias[vg]) : 0.0f;
        }
        addend[tid] = a;
      }
    }
    f32x4 acc[WV][WT];
    Fast::run(acc, src, smem, static_cast<int>(p.d), buf, vt == vt_begin, [&] {
      if (vt + 1 < vt_end) set_class_tile(vt + 1);
    });

    const int cls0 = static_cast<int>(v0) + wv * (16 * WV);  // first class of this wave
    const float* wave_addend = addend + wv * (16 * WV);
    const int sw = (r16 >> 1) & 7;  // 16-byte chunks of a staged row are XOR-swizzled with (row >> 1) & 7
    // (left to itself the compiler forms the row part of every store address before the tile loop, holds the pairs
    // of registers through the main loop by spilling them, and the reload at the top of the epilogue waits for
    // the loads just issued for the next tile)
    int64_t wrow0 = t0 + wt * (16 * WT);  // first row of this wave
    asm volatile("" : "+s"(wrow0));
    constexpr int kEs = OUT32 ? 4 : 2;                  // bytes per stored element
    constexpr int kViPer = kDzStageRow / (16 * kEs);    // 16-class blocks per staged row (4, or 2 for fp32)
    constexpr int kParts = WV / kViPer;                 // staged blocks per row block
    constexpr int kPieceElems = 16 / kEs;               // elements per 16-byte piece
#pragma unroll
    for (int ti = 0; ti < WT; ++ti) {
      const DzRow rr = s_rows[wt * (16 * WT) + ti * 16 + r16];
#pragma unroll
      for (int vh = 0; vh < kParts; ++vh) {
        float rest[PARTS ? kViPer : 1][4];  // PARTS: what the parts stored so far leave of the gradients
        // The gradients of one staged block.  One copy of the arithmetic per answer to "soft-capped?".
        auto stage_block = [&](auto capped) {
#pragma unroll
          for (int vj = 0; vj < kViPer; ++vj) {
            const int vi = vh * kViPer + vj;
            float dzv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int cl = vi * 16 + 4 * kq + r;
              float x = acc[vi][ti][r];
              bool dead = false;
              if (GENERAL) {
                const float add = wave_addend[cl];
                dead = (add == -INFINITY);
                x = dead ? 0.0f : fmaf(x, unit, add);
              }
              float pr, damp = 1.0f;
              if (decltype(capped)::value) {
                const float t = __builtin_amdgcn_exp2f(x * in_scale);
                const float w = __builtin_amdgcn_rcpf(1.0f + t);
                const float th = 1.0f - 2.0f * w;
                pr = PARTS ? exp2_difference(p.sc.out_scale * th, rr.lse2) : __builtin_amdgcn_exp2f(p.sc.out_scale * th - rr.lse2);
                damp = 1.0f - th * th;
              } else {
                pr = PARTS ? exp2_difference(x * log2e, rr.lse2) : __builtin_amdgcn_exp2f(x * kLog2e - rr.lse2);
              }
              float dz = pr * rr.gh - ((cls0 + cl == rr.tgt) ? rr.g : 0.0f);
              if (decltype(capped)::value) dz *= damp;
              dzv[r] = dead ? 0.0f : dz;
            }
            const int col = (vj * 16 + 4 * kq) * kEs;  // byte inside the staged row
            unsigned char* dst = stage + r16 * kDzStageRow + ((((col >> 4) ^ sw) << 4) | (col & 15));
            if (PARTS) {
#pragma unroll
              for (int r = 0; r < 4; ++r) rest[vj][r] = dzv[r];
            } else if (OUT32) {
              *reinterpret_cast<float4*>(dst) = make_float4(dzv[0], dzv[1], dzv[2], dzv[3]);
            } else {
              uint2 pk;
              pk.x = Elem<T>::pack2(dzv[0], dzv[1]);
              pk.y = Elem<T>::pack2(dzv[2], dzv[3]);
              *reinterpret_cast<uint2*>(dst) = pk;
            }
          }
        };
        if (p.sc.on) {
          stage_block(std::true_type{});
        } else {
          stage_block(std::false_type{});
        }
        // 16 rows x 128 bytes leave as 16-byte pieces: one instruction covers 8 rows of 128 contiguous bytes
        auto store_block = [&](int part) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the block is private to this wave: no barrier
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const int j = lane + 64 * k;
            const int row = j >> 3;
            const int pc = j & 7;
            const uint4 val = *reinterpret_cast<const uint4*>(stage + row * kDzStageRow + ((pc ^ ((row >> 1) & 7)) << 4));
            const int64_t gi = wrow0 + ti * 16 + row;
            const int64_t gcol = static_cast<int64_t>(cls0) + vh * (16 * kViPer) + pc * kPieceElems;
            if constexpr (PARTS) {
              if (gi < p.b_store && gcol < p.ldz)
                *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.dz) + (gi * p.parts + part) * p.ldz + gcol) = val;
            } else if (gi < p.b) {
              unsigned char* dst = static_cast<unsigned char*>(p.dz) + (gi * p.ldz + gcol) * kEs;
              if (!GENERAL || gcol + kPieceElems <= p.v || (p.pad_store && gcol + kPieceElems <= p.ldz)) {
                *reinterpret_cast<uint4*>(dst) = val;
              } else if (OUT32) {
                const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                  if (gcol + i < p.v) reinterpret_cast<uint32_t*>(dst)[i] = w[i];
              } else {
                const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
                for (int i = 0; i < 8; ++i)
                  if (gcol + i < p.v) reinterpret_cast<uint16_t*>(dst)[i] = static_cast<uint16_t>(w[i >> 1] >> ((i & 1) * 16));
              }
            }
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next block is staged
        };
        if constexpr (PARTS) {
          // x = hi + mid + lo, each the bf16 nearest to what the ones before it leave; one staged block per part
#pragma unroll
          for (int part = 0; part < 3; ++part) {
            if (part >= p.parts) break;
#pragma unroll
            for (int vj = 0; vj < kViPer; ++vj) {
              uint2 pk;
              pk.x = Elem<BF16>::pack2(rest[vj][0], rest[vj][1]);
              pk.y = Elem<BF16>::pack2(rest[vj][2], rest[vj][3]);
              rest[vj][0] -= Elem<BF16>::to_float(static_cast<uint16_t>(pk.x));
              rest[vj][1] -= Elem<BF16>::to_float(static_cast<uint16_t>(pk.x >> 16));
              rest[vj][2] -= Elem<BF16>::to_float(static_cast<uint16_t>(pk.y));
              rest[vj][3] -= Elem<BF16>::to_float(static_cast<uint16_t>(pk.y >> 16));
              const int col = (vj * 16 + 4 * kq) * 2;
              *reinterpret_cast<uint2*>(stage + r16 * kDzStageRow + ((((col >> 4) ^ sw) << 4) | (col & 15))) = pk;
            }
            store_block(part);
          }
        } else {
          store_block(0);
        }
      }
    }
  }
  // the loads issued under the last tile (its own first stages once more) must land before the workgroup ends
  wait_vmcnt<0>();
}

template <typename T, bool GENERAL, DzOut OUT, bool TAIL = false, int ROWS = kDzTile>
__global__ __launch_bounds__(kDzThreads, 1) void dense_dz16_kernel(DzParams p) {
  dense_dz16_item<T, GENERAL, OUT, TAIL, ROWS>(p);
}

// Operands in parts: logits from halves of fp16 where the device found room for the values in them.
template <bool GENERAL>
__global__ __launch_bounds__(kDzThreads, 1) void dz_terms_kernel(DzParams p) {
  if (*p.wide == 0) dense_dz16_item<F16, GENERAL, kDzParts>(p);
  else dense_dz16_item<BF16, GENERAL, kDzParts>(p);
}

int dense_dz_launch(const void* e, const void* c, const void* bias,
                    const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                    const int32_t* valids, const int64_t* targets,
                    void* dz, int64_t ldz, int dz_is_fp32, int pad_store,
                    int64_t n_rows, int64_t b, int64_t v, int64_t d,
                    int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                    float grad_scale, int64_t shift, int64_t target_offset,
                    float softcap, int dtype, hipStream_t stream) {
  if (b < 0 || v <= 0 || d <= 0 || n_rows < 0 || shift < 0 || ldz < v) return CCE_ERR_INVALID_ARGUMENT;
  if (b == 0) return CCE_OK;
  if (e == nullptr || c == nullptr || lse == nullptr || d_out == nullptr || targets == nullptr || dz == nullptr)
    return CCE_ERR_INVALID_ARGUMENT;
  if (valids == nullptr && b > n_rows) return CCE_ERR_INVALID_ARGUMENT;
  if (d > (1 << 30) || v > (int64_t(1) << 31) - 512) return CCE_ERR_INVALID_ARGUMENT;
  if (dtype != CCE_DTYPE_BF16 && dtype != CCE_DTYPE_F16) return CCE_ERR_UNSUPPORTED_DTYPE;
  // direct-to-LDS main loop and 16-byte stores only
  const bool tail = d % kDmaBK != 0;
  if (!aligned16(e) || !aligned16(c) || !aligned16(dz) || !dense_width_ok(n_rows, d, stride_e, stride_cv) || (tail && dz_is_fp32) ||
      stride_e % 8 != 0 || stride_cv % 8 != 0 || stride_cd != 1 || ldz % (dz_is_fp32 ? 4 : 8) != 0)
    return CCE_ERR_MISALIGNED;

  DzParams p = {};
  p.e = static_cast<const uint16_t*>(e);
  p.c = static_cast<const uint16_t*>(c);
  p.bias = static_cast<const uint16_t*>(bias);
  p.valids = valids;
  p.lse = lse;
  p.d_out = d_out;
  p.d_lse = d_lse;
  p.targets = targets;
  p.dz = dz;
  p.ldz = ldz;
  p.n_rows = n_rows;
  p.b = b;
  p.v = v;
  p.d = d;
  p.stride_e = stride_e;
  p.stride_cv = stride_cv;
  p.shift = shift;
  p.target_offset = target_offset;
  p.grad_scale = grad_scale;
  p.d_out_is_scalar = d_out_is_scalar;
  p.pad_store = pad_store;
  // the 16 x 16 x 32 kernel addresses rows by 32-bit byte offsets and streams at least two stages per tile
  const bool k16 = dense_k16(n_rows, d, stride_e, stride_cv);
  const bool mid = k16 && !dz_is_fp32 && mid_row_blocks(b, v);
  const int block = mid ? kMidRowBlock : kDzTile;
  p.nrb = static_cast<int>((b + block - 1) / block);
  p.nvt = static_cast<int>((v + kDzTile - 1) / kDzTile);
  const SpanChoice spans = choose_spans(p.nrb, p.nvt);
  p.nsplit = spans.count;
  p.block_rows = spans.block_rows;
  p.block_spans = spans.block_spans;
  p.nitems = p.nrb * p.nsplit;
  p.items_per_xcd = (p.nitems + 7) / 8;
  p.sc = make_softcap(softcap);

  using FastB = DmaLogitTile<BF16, kDzWV, kDzWT, kDzNWV, kDzNWT>;
  const int lds = FastB::LDS_BYTES + 2 * kDzTile * 4;
  const int lds16 = mid ? Dz16Shape<kMidRowBlock>::LDS_BYTES : Dz16Shape<kDzTile>::LDS_BYTES;
  const bool general = (bias != nullptr) || (v % kDzTile != 0);
  const int grid = p.items_per_xcd * 8;
  hipError_t err;
#define CCE_LAUNCH_DZ2(TT, GE, O32)                                                               \
  do {                                                                                            \
    if (mid && tail) {                                                                            \
      auto kern = dense_dz16_kernel<TT, GE, kDz16Bit, true, kMidRowBlock>;                        \
      static LdsLimitOnce lds_limit;                                                              \
      err = lds_limit.set(kern, lds16);                                                           \
      if (err != hipSuccess) return status_from_hip(err);                                         \
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds16, stream, p);                   \
    } else if (mid) {                                                                             \
      auto kern = dense_dz16_kernel<TT, GE, kDz16Bit, false, kMidRowBlock>;                       \
      static LdsLimitOnce lds_limit;                                                              \
      err = lds_limit.set(kern, lds16);                                                           \
      if (err != hipSuccess) return status_from_hip(err);                                         \
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds16, stream, p);                   \
    } else if (k16 && tail) {                                                                     \
      auto kern = dense_dz16_kernel<TT, GE, kDz16Bit, true>;                                      \
      static LdsLimitOnce lds_limit;                                                              \
      err = lds_limit.set(kern, lds16);                                                           \
      if (err != hipSuccess) return status_from_hip(err);                                         \
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds16, stream, p);                   \
    } else if (k16) {                                                                             \
      auto kern = dense_dz16_kernel<TT, GE, (O32) ? kDzFp32 : kDz16Bit>;                          \
      static LdsLimitOnce lds_limit;                                                              \
      err = lds_limit.set(kern, lds16);                                                           \
      if (err != hipSuccess) return status_from_hip(err);                                         \
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds16, stream, p);                   \
    } else {                                                                                      \
      auto kern = dense_dz_kernel<TT, GE, O32>;                                                   \
      static LdsLimitOnce lds_limit;                                                              \
      err = lds_limit.set(kern, lds);                                                             \
      if (err != hipSuccess) return status_from_hip(err);                                         \
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds, stream, p);                     \
    }                                                                                             \
  } while (0)
#define CCE_LAUNCH_DZ(TT, GE)                                                                     \
  do {                                                                                            \
    if (dz_is_fp32) CCE_LAUNCH_DZ2(TT, GE, true); else CCE_LAUNCH_DZ2(TT, GE, false);             \
  } while (0)
  if (dtype == CCE_DTYPE_BF16) {
    if (general) CCE_LAUNCH_DZ(BF16, true); else CCE_LAUNCH_DZ(BF16, false);
  } else {
    if (general) CCE_LAUNCH_DZ(F16, true); else CCE_LAUNCH_DZ(F16, false);
  }
#undef CCE_LAUNCH_DZ
#undef CCE_LAUNCH_DZ2
  return status_from_hip(hipGetLastError());
}

// ---- dz of one chunk of classes with operands and result in bf16 parts (cce_fp32.hip) --------------------------
int dz_terms_launch(const uint16_t* e_parts, int64_t ld_e, const uint16_t* c_parts, int64_t ld_c, const uint16_t* e_halves,
                    const uint16_t* c_halves, const int* wide, float halves_scale, const float* bias,
                    const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                    const int32_t* valids, const int64_t* targets, uint16_t* dz_parts, int64_t ldz,
                    int64_t n_rows, int64_t b, int64_t b_store, int64_t v, int64_t part_d, int terms, int parts,
                    float grad_scale, int64_t shift, int64_t target_offset, float softcap, hipStream_t stream) {
  DzParams p = {};
  p.wide = wide;
  p.e_halves = e_halves;
  p.c_halves = c_halves;
  p.halves_scale = halves_scale;
  p.e = e_parts;
  p.c = c_parts;
  p.bias32 = bias;
  p.terms = terms;
  p.parts = parts;
  p.b_store = b_store;
  p.valids = valids;
  p.lse = lse;
  p.d_out = d_out;
  p.d_lse = d_lse;
  p.targets = targets;
  p.dz = dz_parts;
  p.ldz = ldz;
  p.n_rows = n_rows;
  p.b = b;
  p.v = v;
  p.d = part_d;
  p.stride_e = ld_e;
  p.stride_cv = ld_c;
  p.shift = shift;
  p.target_offset = target_offset;
  p.grad_scale = grad_scale;
  p.d_out_is_scalar = d_out_is_scalar;
  p.nrb = static_cast<int>((b + kDzTile - 1) / kDzTile);
  p.nvt = static_cast<int>((v + kDzTile - 1) / kDzTile);
  const SpanChoice spans = choose_spans(p.nrb, p.nvt);
  p.nsplit = spans.count;
  p.block_rows = spans.block_rows;
  p.block_spans = spans.block_spans;
  p.nitems = p.nrb * p.nsplit;
  p.items_per_xcd = (p.nitems + 7) / 8;
  p.sc = make_softcap(softcap);
  using Fast = DmaLogitTile16<BF16, kDz16WV, kDz16WT, kDzNWV, kDzNWT, true>;
  const int lds = Fast::LDS_BYTES + 2 * kDzTile * 4 + kDzTile * static_cast<int>(sizeof(DzRow)) + kDzNWV * kDzNWT * kDz16StageBytes;
  const int grid = p.items_per_xcd * 8;
  hipError_t err;
  auto launch = [&](auto kern, LdsLimitOnce& lds_limit) {
    err = lds_limit.set(kern, lds);
    if (err == hipSuccess) hipLaunchKernelGGL(kern, dim3(grid), dim3(kDzThreads), lds, stream, p);
    return err == hipSuccess;
  };
  static LdsLimitOnce limits[2];
  if (bias != nullptr || v % kDzTile != 0) {
    if (!launch(dz_terms_kernel<true>, limits[0])) return status_from_hip(err);
  } else {
    if (!launch(dz_terms_kernel<false>, limits[1])) return status_from_hip(err);
  }
  return status_from_hip(hipGetLastError());
}

}  // namespace cce

extern "C" int cce_backward_dz(const void* e, const void* c, const void* bias,
                               const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                               const int32_t* valids, const int64_t* targets,
                               void* dz, int64_t ldz, int dz_is_fp32,
                               int64_t n_rows, int64_t b, int64_t v, int64_t d,
                               int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                               float grad_scale, int64_t shift, int64_t target_offset,
                               float softcap, int dtype, void* stream) {
  if (b > 0 && d > 0 && d % cce::kDmaBK != 0) return CCE_ERR_MISALIGNED;
  return cce::dense_dz_launch(e, c, bias, lse, d_out, d_out_is_scalar, d_lse, valids, targets, dz, ldz, dz_is_fp32, 0,
                              n_rows, b, v, d, stride_e, stride_cv, stride_cd, grad_scale, shift, target_offset, softcap,
                              dtype, static_cast<hipStream_t>(stream));
}
