// One 256 x 256 tile of  Out[m][n] = sum_k A[m][k] * B[k][n]  on one compute unit with eight waves, two per SIMD, 2 (m) x 4 (n),
// each owning 128 x 64 of the tile: 8 x 4 accumulator blocks of 16 x 16.
//
// B is K-major (its reduction index is its row); A is K-major too (dC = dz^T . E) or has the reduction along its rows (dE =
// dz . C).  A stage is 64 reduction steps of either operand, 32 KB each, two stages in LDS (A0 A1 B0 B1), all by direct
// global -> LDS loads, eight per wave and stage:
//   Direct A  256 rows x 128 bytes, 16-byte chunks XOR-swizzled with (row >> 1) & 7; one load fills 8 rows, a fragment (16 rows x
//             32 steps) is one 16-byte read.
//   KMajor    64 rows x 512 bytes, the 32 chunks of a row XOR-swizzled with 4 (row & 3); one load fills 2 rows (lanes 0 - 31
//             one, 32 - 63 the next); a fragment is two LDS transpose reads (`ds_read_b64_tr_b16`) of four k rows per 16 lanes:
//             lane i of 16 supplies the address of row r0 + (i >> 2), columns c0 + 4 (i & 3) .. + 3, and receives the elements
//             [r0 .. r0 + 3][c0 + i].
// The rows of B may be gathered through an index vector (B_GATHER): a lane looks its row numbers up a step ahead of the loads.
//
// A stage is two steps of 32 MFMAs of 16 x 16 x 32: the step on its first half reads the fragments of the second half, the step on
// the second half those of the next stage's first half, and issues all loads of the stage after that into the ring stage it has
// just finished with.  A fragments are read again in place once their four MFMAs are issued, those of B are held twice; one barrier
// per stage, four MFMAs into its second step.
//
// What bounds it is power: the instruction reads and writes a quarter of the accumulator registers per MFMA and sums twice as many
// products before it touches them as the 32 x 32 x 16 one (the chip sustains 2.09 against 1.84 PFLOP/s of either from registers, with
// operands of full entropy), and two waves per SIMD cover each other's reads, loads and epilogues.  Counters of a launch of
// [8192, 2048] x [256000, 2048] (8000 classes): the pipe is busy 73 % of its cycles, 83 % of a compute unit's, at 1.8 of the 2.4 GHz;
// of the 6.2e5 cycles that a compute unit is busy, 1.3e5 are LDS bank conflicts (with K-major reads of four waves there were 2e3),
// and a wave waits for LDS 11 % of its time.  A loop of four waves with 128 x 128
// each on 32 x 32 x 16 has two thirds of the fragment reads and kept the pipe busier (75 % of the launch), at a lower clock.  Forward and backward
// with that loop / this one, ms: [15360, 4096] x [128256, 4096] 50.0 / 48.4, [8192, 2048] x [256000, 2048] 25.2 / 24.2, [65536, 3584] x
// [19008, 3584] 28.2 / 27.55, [3891, 1024] x [32000, 1024] 0.90 / 0.86, [8779, 2432] x [20995, 2432] in fp16 3.05 / 2.88, fp32 [2046, 3072] x
// [32064, 3072] 7.40 / 7.25.
//
// A column chunk past the matrix is fetched from the last chunk inside it instead (it only feeds outputs the caller drops).  A
// reduction that is not a multiple of 64 has one partial stage: it is the FIRST stage of the tile, fetched before the main
// loop by loads that ask per row whether the row exists and take a line of zeros when not, so that a non-finite value elsewhere
// never meets the product.
//
// TERMS: the operands are fp32 values in 16-bit parts, a_part / b_part bytes from part to part, and the reduction runs over the
// cross terms of the parts one after the other (kTermsFirst / kTermsSecond of cce_common.h: A is the first operand), whole
// stages only.
#pragma once

#include <utility>

#include "cce_common.h"

namespace cce {

typedef short tr_short4_t __attribute__((ext_vector_type(4)));

template <typename T, bool A_KM, bool B_GATHER = false, bool TERMS = false>
struct Tile8 {
  static_assert(!B_GATHER || !TERMS, "parts are compact");
  static constexpr int WM = 8, WN = 4;            // accumulator blocks per wave
  static constexpr int NW = 8;
  static constexpr int NT = 64 * NW;
  static constexpr int TILE = 256;
  static constexpr int BK = 64;
  static constexpr int OP_BYTES = 32 * 1024;      // one stage of one operand
  static constexpr int B_BASE = 2 * OP_BYTES;     // A stage 0, A stage 1, B stage 0, B stage 1
  static constexpr int LDS_BYTES = 4 * OP_BYTES;
  static constexpr int NQ = 4;                    // loads per wave, stage and operand
  using vec8 = typename Elem<T>::vec8;

  // ---- what a lane fetches ---------------------------------------------------------------------------
  static __device__ __forceinline__ int row_direct(int q, int wave, int lane) { return 8 * (q * NW + wave) + (lane >> 3); }
  static __device__ __forceinline__ int chunk_direct(int wave, int lane) {
    const int sw = (4 * (wave & 1) + (lane >> 4)) & 7;  // (row >> 1) & 7
    return ((lane & 7) ^ sw) * 8;
  }
  // KMajor: load q of a wave covers stage rows 2 (q NW + wave) and the next; this lane's is the (lane >> 5)-th
  static __device__ __forceinline__ int row_kmajor(int q, int wave) { return 2 * (q * NW + wave); }
  static __device__ __forceinline__ int chunk_kmajor(int wave, int lane) {
    const int r3 = (2 * (wave & 1) + (lane >> 5)) & 3;  // row & 3
    return ((lane & 31) ^ (r3 << 2)) * 8;
  }

  // A load takes a wave-uniform base, formed on the scalar unit, and a byte offset per lane.
  struct Source {
    const unsigned char* a_base;       // KMajor: row 0; Direct: row 0 of the tile, step 0 of the reduction
    unsigned a_off[A_KM ? 1 : NQ];     // KMajor: column chunk (and, for the upper lanes, a row); Direct: row and chunk of each load
    const unsigned char* b_base;       // row 0 (B_GATHER: of the matrix that the row numbers index)
    unsigned b_off;                    // as a_off of a KMajor A; B_GATHER: the column chunk alone
    uint32_t a_stride, b_stride;       // KMajor: bytes between consecutive k rows
    const int32_t* b_rows;             // B_GATHER: the k rows of B (k_total entries)
    int k_total;                       // length of the reduction (TERMS: of one term, a multiple of 64)
    int64_t a_part, b_part;            // TERMS: bytes from one part to the next
    int terms;                         // TERMS: 3 or 6
    int nk;                            // (plan) stages
    int partial;                       // (plan) 1: stage 0 is the partial last 64-step, stage t >= 1 is whole stage t - 1
  };
  static __device__ __forceinline__ void plan(Source& s) {
    const int whole = s.k_total / BK;
    s.partial = TERMS ? 0 : (s.k_total % BK) != 0;
    s.nk = TERMS ? s.terms * whole : whole + s.partial;
  }

  struct Geometry {
    int lane, wave, wm, wn;
    unsigned lds_base;
    // LDS byte addresses (inside a stage) of this lane's fragment reads; KMajor: one per pair of blocks (a step adds 16 KB, the
    // second block of a pair 32 bytes, the upper four k rows 2 KB); Direct: one per step (block i adds i * 2 KB)
    int a_addr[4];
    int b_addr[2];
  };
  static __device__ __forceinline__ Geometry geometry(unsigned char* lds) {
    Geometry g;
    g.lane = threadIdx.x & 63;
    g.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    g.wm = g.wave >> 2;
    g.wn = g.wave & 3;
    g.lds_base = static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds));
    const int r16 = g.lane & 15, kq = g.lane >> 4;
    const int tr_row = 8 * kq + ((g.lane >> 2) & 3);
    const int tr_col = 4 * (g.lane & 3);
    auto km = [&](int col) { return tr_row * 512 + ((((col >> 3) ^ ((tr_row & 3) << 2)) << 4) | ((col & 7) << 1)); };
#pragma unroll
    for (int x = 0; x < 4; ++x)
      g.a_addr[x] = A_KM ? km(g.wm * 128 + x * 32 + tr_col) : (g.wm * 128 + r16) * 128 + (((x * 4 + kq) ^ (r16 >> 1)) & 7) * 16;
#pragma unroll
    for (int x = 0; x < 2; ++x) g.b_addr[x] = B_BASE + km(g.wn * 64 + x * 32 + tr_col);
    return g;
  }

  // A stage of the reduction: its first step and, with TERMS, how far into the rows of A and B its parts lie.
  struct Pos {
    int k, term;
    int64_t a, b;
  };
  static __device__ __forceinline__ Pos first_pos(const Source& s) {
    Pos p = {s.partial ? s.k_total / BK * BK : 0, 0, 0, 0};
    if constexpr (TERMS) {
      p.term = kTermsAll - s.terms;
      p.a = term_part(kTermsFirst, p.term) * s.a_part;
      p.b = term_part(kTermsSecond, p.term) * s.b_part;
    }
    return p;
  }
  // Stage t from stage t - 1.
  static __device__ __forceinline__ void advance(Pos& p, const Source& s, int t) {
    if constexpr (TERMS) {
      p.k += BK;
      if (p.k == s.k_total) {
        p.k = 0;
        ++p.term;
        p.a = term_part(kTermsFirst, p.term) * s.a_part;
        p.b = term_part(kTermsSecond, p.term) * s.b_part;
      }
    } else {
      p.k = (t - s.partial) * BK;
    }
  }

  struct Ids {
    int v[B_GATHER ? NQ : 1];
  };

  // ---- loads of whole stages: nothing is checked ---------------------------------------------------------
  static __device__ __forceinline__ void look_up(Ids& ids, int q, const Source& s, int k0, const Geometry& g) {
    if (!B_GATHER) return;
    const int32_t* pair = s.b_rows + (k0 + row_kmajor(q, g.wave));  // uniform
    ids.v[B_GATHER ? q : 0] = pair[g.lane >> 5];
  }
  static __device__ __forceinline__ void issue_a(int q, const Source& s, const Pos& at, int stage_off, const Geometry& g) {
    const unsigned dst = g.lds_base + stage_off + (q * NW + g.wave) * 1024;
    if (A_KM)
      lds_dma16_sbase(s.a_base + static_cast<uint64_t>(static_cast<uint32_t>(at.k + row_kmajor(q, g.wave))) * s.a_stride + at.a,
                      s.a_off[0], dst);
    else
      lds_dma16_sbase(s.a_base + 2 * static_cast<int64_t>(at.k) + at.a, s.a_off[A_KM ? 0 : q], dst);
  }
  static __device__ __forceinline__ void issue_b(int q, const Source& s, const Ids& ids, const Pos& at, int stage_off,
                                                 const Geometry& g) {
    const unsigned dst = g.lds_base + B_BASE + stage_off + (q * NW + g.wave) * 1024;
    if (B_GATHER)
      lds_dma16(s.b_base + (static_cast<uint64_t>(static_cast<uint32_t>(ids.v[B_GATHER ? q : 0])) * s.b_stride + s.b_off), dst);
    else
      lds_dma16_sbase(s.b_base + static_cast<uint64_t>(static_cast<uint32_t>(at.k + row_kmajor(q, g.wave))) * s.b_stride + at.b,
                      s.b_off, dst);
  }

  // ---- loads of stage 0 (the partial stage when there is one): every row is asked for --------------------
  static __device__ __forceinline__ void issue_first(const Source& s, const Geometry& g) {
    const Pos at = first_pos(s);
    const unsigned char* zeros = reinterpret_cast<const unsigned char*>(g_zero_line) + (g.lane & 15) * 16;
    int id[NQ];  // (the row numbers of a gathered B are looked up first: the lookups and the loads share a queue)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int row = at.k + row_kmajor(q, g.wave) + (g.lane >> 5);
      id[q] = -1;
      if (row < s.k_total) id[q] = B_GATHER ? s.b_rows[row] : row;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (A_KM) {
        const int row = at.k + row_kmajor(q, g.wave);  // uniform; the lane's own row is one further for the upper lanes
        const unsigned char* src = s.a_base + static_cast<uint64_t>(static_cast<uint32_t>(row)) * s.a_stride + at.a + s.a_off[0];
        if (row + (g.lane >> 5) >= s.k_total) src = zeros;
        lds_dma16(src, g.lds_base + (q * NW + g.wave) * 1024);
      } else {
        issue_a(q, s, at, 0, g);
      }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const unsigned char* src;
      if (B_GATHER) {
        src = s.b_base + static_cast<uint64_t>(static_cast<uint32_t>(id[q])) * s.b_stride + s.b_off;
      } else {
        const int row = at.k + row_kmajor(q, g.wave);
        src = s.b_base + static_cast<uint64_t>(static_cast<uint32_t>(row)) * s.b_stride + at.b + s.b_off;
      }
      if (id[q] < 0) src = zeros;
      lds_dma16(src, g.lds_base + B_BASE + (q * NW + g.wave) * 1024);
    }
  }

  // ---- fragment reads --------------------------------------------------------------------------------
  struct Frag {
    tr_short4_t lo, hi;  // the lower and the upper four of eight consecutive k
  };
  static __device__ __forceinline__ vec8 value(const Frag& f) { return __builtin_bit_cast(vec8, f); }
  static __device__ __forceinline__ tr_short4_t read_tr(const unsigned char* at) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tr_short4_t*)(at));
  }
  static constexpr int kReadsA = A_KM ? 2 : 1;  // reads per fragment
  // `off`: the ring stage and, for KMajor operands, the step inside it; `half`: the step (Direct)
  static __device__ __forceinline__ void read_a(int i, int part, Frag (&a)[WM], const unsigned char* lds, int off, int half,
                                                const Geometry& g) {
    if (A_KM) {
      const tr_short4_t v = read_tr(lds + g.a_addr[i >> 1] + off + half * 16384 + (i & 1) * 32 + part * 2048);
      if (part) a[i].hi = v; else a[i].lo = v;
    } else {
      a[i] = __builtin_bit_cast(Frag, *reinterpret_cast<const uint4*>(lds + g.a_addr[half] + off + i * 2048));
    }
  }
  static __device__ __forceinline__ void read_b(int j, int part, Frag (&b)[WN], const unsigned char* lds, int off, int half,
                                                const Geometry& g) {
    const tr_short4_t v = read_tr(lds + g.b_addr[j >> 1] + off + half * 16384 + (j & 1) * 32 + part * 2048);
    if (part) b[j].hi = v; else b[j].lo = v;
  }

  // One step: 32 MFMAs on a[] and bc[]; under them, at most two memory instructions after each:
  //   READ  the fragments of the next step, in half `rhalf` of ring stage `roff`: a[i] once the last MFMA that uses the old
  //         one is issued, the others into bn[];
  //   LOAD  all loads of the stage `at` into ring stage `loff`;  IDS  the row numbers of B for the stage that starts at k0
  //   SYNC  (the second half of a stage) after four MFMAs this wave waits for its own loads of the next stage and for the
  //         reads it has in flight, then the barrier; reads and loads of such a step come after it.
  static constexpr int kSyncAt = 4;
  static constexpr int a_slot(bool sync, int i, int part) {
    const int at = (sync && i < 2 ? 5 + 2 * i : 4 * i + 3) + part;
    return at < 31 ? at : 31;
  }
  static constexpr int b_slot(bool sync, int j, int part) { return (sync ? 9 + 4 * j : 1 + 8 * j) + part; }
  static constexpr int load_slot(int q) { return q < 4 ? 8 + 4 * q : (q < 6 ? 25 + (q - 4) : 29 + (q - 6)); }

  template <bool READ, bool LOAD, bool SYNC, bool IDS>
  static __device__ __forceinline__ void step(f32x4 (&acc)[WM][WN], Frag (&a)[WM], const Frag (&bc)[WN], Frag (&bn)[WN],
                                              const unsigned char* lds, int roff, int rhalf, const Source& s, const Pos& at, int loff,
                                              Ids& ids, int k0, const Geometry& g) {
    static_for<WM * WN>([&](auto idx_c) {
      constexpr int idx = decltype(idx_c)::value;
      constexpr int i = idx / WN, j = idx % WN;
      if (SYNC && idx == kSyncAt) {
        wait_vmcnt<0>();
        if (B_GATHER) {
          // The looked-up rows are pinned as used here, where nothing is in flight: the compiler places its own wait for
          // them at their first use, and further down it would also wait for the direct-to-LDS loads.
#pragma unroll
          for (int q = 0; q < NQ; ++q) asm volatile("" : "+v"(ids.v[B_GATHER ? q : 0]));
        }
        __syncthreads();
      }
      acc[i][j] = Elem<T>::mfma16(value(a[i]), value(bc[j]), acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      if (READ) {
        static_for<WN>([&](auto n_c) {
          constexpr int n = decltype(n_c)::value;
          if (idx == b_slot(SYNC, n, 0)) read_b(n, 0, bn, lds, roff, rhalf, g);
          if (idx == b_slot(SYNC, n, 1)) read_b(n, 1, bn, lds, roff, rhalf, g);
        });
        static_for<WM>([&](auto m_c) {
          constexpr int m = decltype(m_c)::value;
          if (idx == a_slot(SYNC, m, 0)) read_a(m, 0, a, lds, roff, rhalf, g);
          if (kReadsA == 2 && idx == a_slot(SYNC, m, 1)) read_a(m, 1, a, lds, roff, rhalf, g);
        });
      }
      if (LOAD) {
        static_for<2 * NQ>([&](auto q_c) {
          constexpr int q = decltype(q_c)::value;
          if (idx == load_slot(q)) {
            if (q < NQ) issue_a(q, s, at, loff, g);
            else issue_b(q - NQ, s, ids, at, loff, g);
          }
        });
      }
      if (IDS && B_GATHER) {
        static_for<NQ>([&](auto q_c) {
          constexpr int q = decltype(q_c)::value;
          if (idx == 4 + 2 * q) look_up(ids, q, s, k0, g);
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  // acc = A . B over the whole reduction (k_total >= 1, plan() done); the LDS must be idle, and may be reused right after.
  static __device__ __forceinline__ void run(f32x4 (&acc)[WM][WN], const Source& s, unsigned char* lds, const Geometry& g) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int nk = s.nk;
    Ids ids = {};
    issue_first(s, g);
    Pos at = first_pos(s);
    if (nk > 1) {
      advance(at, s, 1);
#pragma unroll
      for (int q = 0; q < NQ; ++q) look_up(ids, q, s, at.k, g);
#pragma unroll
      for (int q = 0; q < NQ; ++q) issue_a(q, s, at, OP_BYTES, g);
#pragma unroll
      for (int q = 0; q < NQ; ++q) issue_b(q, s, ids, at, OP_BYTES, g);
      wait_vmcnt<2 * NQ>();  // the first stage has landed
    } else {
      wait_vmcnt<0>();
    }
    __syncthreads();
    Frag a[WM], b0[WN], b1[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      read_b(j, 0, b0, lds, 0, 0, g);
      read_b(j, 1, b0, lds, 0, 0, g);
    }
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      read_a(i, 0, a, lds, 0, 0, g);
      if (kReadsA == 2) read_a(i, 1, a, lds, 0, 0, g);
    }

    int cur = 0;
#pragma unroll 1
    for (int st = 0; st + 2 < nk; ++st) {
      advance(at, s, st + 2);
      step<true, false, false, true>(acc, a, b0, b1, lds, cur, 1, s, at, 0, ids, at.k, g);
      step<true, true, true, false>(acc, a, b1, b0, lds, OP_BYTES - cur, 0, s, at, cur, ids, 0, g);
      cur = OP_BYTES - cur;
    }
    if (nk > 1) {
      step<true, false, false, false>(acc, a, b0, b1, lds, cur, 1, s, at, 0, ids, 0, g);
      step<true, false, true, false>(acc, a, b1, b0, lds, OP_BYTES - cur, 0, s, at, 0, ids, 0, g);
      cur = OP_BYTES - cur;
    }
    step<true, false, false, false>(acc, a, b0, b1, lds, cur, 1, s, at, 0, ids, 0, g);
    step<false, false, false, false>(acc, a, b1, b0, lds, cur, 0, s, at, 0, ids, 0, g);
    __syncthreads();
  }

  // ---- the finished tile, as row pieces ----------------------------------------------------------------
  // A lane holds, of every block, column l % 16 and rows 4 (l / 16) + r.  Each wave passes its 128 x 64 part through LDS (idle
  // after run()), 16 rows at a time, and hands `f` pieces of 8 consecutive columns of one row:
  //     f(row, col, v)   row, col: position inside the 256 x 256 tile; v[8]: the values [row][col .. col + 7]
  // so that a piece is one 16-byte (16-bit data) or two 16-byte (fp32) accesses and 8 lanes cover 128 or 256
  // contiguous bytes of a row.  The staging area is private to the wave: no barrier.
  static constexpr int kPieceCols = 8;
  static constexpr int kStagePitch = (64 + 4) * 4;           // bytes per staged row
  static constexpr int kStageBytes = 16 * kStagePitch;       // per wave
  static_assert(NW * kStageBytes <= LDS_BYTES, "the staging areas reuse the ring");

  template <int I>
  static __device__ __forceinline__ void stage_rows(f32x4 (&acc)[WM][WN], unsigned char* stage, const Geometry& g) {
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<float*>(stage + (4 * (g.lane >> 4) + r) * kStagePitch + (j * 16 + (g.lane & 15)) * 4) = acc[I][j][r];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  template <typename F>
  static __device__ __forceinline__ void for_each_row_piece(f32x4 (&acc)[WM][WN], unsigned char* lds, const Geometry& g, F&& f) {
    unsigned char* stage = lds + g.wave * kStageBytes;
    static_for<WM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      stage_rows<i>(acc, stage, g);
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
        const int m = pass * 8 + (g.lane >> 3);
        const int c8 = (g.lane & 7) * kPieceCols;
        const float4 lo = *reinterpret_cast<const float4*>(stage + m * kStagePitch + c8 * 4);
        const float4 hi = *reinterpret_cast<const float4*>(stage + m * kStagePitch + c8 * 4 + 16);
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        f(g.wm * 128 + i * 16 + m, g.wn * 64 + c8, v);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are done before the next rows are staged
    });
  }

  // The same for an output that is combined with what memory holds (dE is summed over the chunks): `fetch(row,
  // col)` returns what `store(row, col, v, old)` needs of the old contents, fetched two slabs of 16 rows ahead.
  static constexpr int kAhead = 2;
  template <typename Old, typename Fetch, typename Store>
  static __device__ __forceinline__ void for_each_row_piece_rmw(f32x4 (&acc)[WM][WN], unsigned char* lds, const Geometry& g,
                                                                Fetch&& fetch, Store&& store) {
    unsigned char* stage = lds + g.wave * kStageBytes;
    const int c8 = (g.lane & 7) * kPieceCols;
    const int m_lane = g.lane >> 3;
    Old old[kAhead + 1][2];
    auto fetch_slab = [&](auto slab) {
      constexpr int i = decltype(slab)::value;
#pragma unroll
      for (int pass = 0; pass < 2; ++pass)
        old[i % (kAhead + 1)][pass] = fetch(g.wm * 128 + i * 16 + pass * 8 + m_lane, g.wn * 64 + c8);
    };
    static_for<kAhead>([&](auto slab) { fetch_slab(slab); });
    static_for<WM>([&](auto i_c) {
      constexpr int i = decltype(i_c)::value;
      stage_rows<i>(acc, stage, g);
      if constexpr (i + kAhead < WM) fetch_slab(std::integral_constant<int, i + kAhead>{});
#pragma unroll
      for (int pass = 0; pass < 2; ++pass) {
        const int m = pass * 8 + m_lane;
        const float4 lo = *reinterpret_cast<const float4*>(stage + m * kStagePitch + c8 * 4);
        const float4 hi = *reinterpret_cast<const float4*>(stage + m * kStagePitch + c8 * 4 + 16);
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        store(g.wm * 128 + i * 16 + m, g.wn * 64 + c8, v, old[i % (kAhead + 1)][pass]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are done before the next rows are staged
    });
  }
};

}  // namespace cce
