// cce_backward_dense: the unfiltered backward (gradient filter off) in one call.
//
// With every entry of dz = d loss / d logits in play the two gradient products are dense:
//     dE[rows] = dz . C          dC = dz^T . E[rows]          dBias = column sums of dz
// The reference forms them inside its one kernel with atomics on dE and dC
// (cut_cross_entropy/cce_backward.py:258-310).  On this chip a tile of dz can feed register-resident
// accumulators of only one of the two outputs at a time (a 256-row slab of dE or dC over D = 2304 .. 4096
// columns is 2.4 .. 4 MB of fp32, against 0.5 MB of registers per compute unit) and global float atomics are
// an order of magnitude too slow, so the vocabulary is walked in chunks and per chunk
//   1. dense_dz_kernel    recomputes the logits of the chunk and writes dz [B, vc] in the input type
//                         (the chunk is sized to stay in the last-level cache),
//   2. dense_dc_kernel    dC[chunk] = dz^T . E : complete for these classes, written once,
//      (2 and 3 are tiles of one launch, dense_products_kernel)
//   3. dense_de_kernel    dE += dz . C[chunk]  : accumulated across the chunks in d_e itself, in fp32 when the caller
//                         asked for an fp32 dE, else as d_e (16 bit) plus a 16-bit compensation term in the workspace,
//   4. dz_colsum_kernel   dBias[chunk], when wanted.
// Where the rows are many against the classes (a vocabulary shard: 65536 rows x 19008 classes) the walk goes over
// blocks of ROWS instead, each with the whole vocabulary: dE of a block is then complete after its one launch (written
// once, no compensation buffer of [b, d]) and it is dC that is carried from block to block, as a pair of 16-bit
// numbers with a [v, d] compensation buffer.  Same kernels, the roles of the two outputs exchanged.
// Where the tiles of a product are few and their reduction long (dE of a thousand rows against 50000 classes: 16 tiles
// of 800 stages on 256 compute units, and its mirror image, dC of a small vocabulary under many rows), the reduction
// itself is cut: a tile becomes several items, each with a range of the reduction and an fp32 slot [rows, d] of its
// own in the workspace, and split_sum_kernel adds the slots in a fixed order at the end (deterministic, no atomics).
// Both products run on the tile loop of cce_tile8.h (direct-to-LDS loads, LDS transpose reads for the
// operand whose reduction index is the row index).  Everything is enqueued on the caller's stream; nothing
// is allocated, no host synchronisation.
#include <algorithm>

#include "cce_dense.h"
#include "cce_tile8.h"

namespace cce {

struct ProductParams {
  const uint16_t* dz;   // [b][ldz]
  int64_t ldz;
  const uint16_t* c;    // first class of the chunk
  int64_t stride_cv;
  const uint16_t* e;
  int64_t stride_e;
  const int32_t* valids;
  float* de_f32;        // dE accumulated in fp32, in the caller's float d_e (rows of e, through valids); or nullptr:
  uint16_t* de_hi;      // dE accumulated as a pair of 16-bit values hi + lo: hi is the caller's d_e in the input type
  uint16_t* de_lo;      //   (rows of e), lo the compensation term in the workspace ([b][d], rows by valid-row number)
  int64_t ld_de;        // row stride of d_e (elements)
  int first_chunk;      // nothing accumulated yet: the pair is written, not read (de_lo == nullptr: the 16-bit d_e is
                        //   complete with this launch and written alone)
  void* d_c;            // first class of the chunk
  int64_t ld_dc;        // row stride of d_c (elements)
  int dc_fp32;
  int dc_accumulate;    // d_c (fp32) is added to, not written
  uint16_t* dc_lo;      // a 16-bit d_c carried over blocks of rows as a pair hi + lo: hi is d_c, lo this [n_cls][d]
  int dc_first;         //   compensation term in the workspace (nullptr: d_c is written once); the first block writes the pair
  int de_rows_by_number;  // the fp32 d_e is indexed by valid-row number (a [b, d] accumulator), not by row of e
  int64_t b;
  int d;
  int n_cls;            // classes in the chunk
  int tiles_n;          // column tiles of either output
  int dc_tiles, dc_per_xcd;  // items of dC (tiles x splits), places per XCD
  int de_tiles, de_per_xcd;
  int de_first;              // the dE items have the longer reduction and take the first block ids
  // A reduction cut into splits: split s of a tile runs over [s * len, min((s + 1) * len, total)) and leaves its
  // result in slot s, `slot` floats behind the one before (one split: the whole reduction, slot unused).
  int de_splits, dc_splits;
  int de_len, dc_len;        // classes / rows per split, multiples of 64
  int64_t de_slot, dc_slot;
  int de_init;               // an fp32 d_e is written, not added to (the first launch on a set of slots)
  // Operands and dz in 16-bit parts (TERMS): a row of c / e is [hi | mid | lo] of part_d columns each, a row of dz
  // [hi | mid | lo] of dz_part classes each; e is compact and b, n_cls are multiples of 64 (rows and classes that pad
  // them are zeros).  rows_out, cls_out: what of them exists; d may be anything (out_vec: 16-byte pieces may be stored).
  int terms, part_d, dz_part, out_vec;
  int64_t rows_out;
  int cls_out;
};

constexpr int kProdThreads = 512;  // eight waves, two per SIMD

// Item `block` of a group of `items` = tiles x splits items (tiles_n column tiles wide).  Block ids that land on one XCD get
// consecutive places in an order that keeps the 32 tiles an XCD works on at a time on few operand panels: a tile
// streams one A panel (its row of tiles) and one B panel (its column) through the XCD's L2, so 32 tiles of one or
// two rows of a wide output need 2 + 16 panels where a block of 4 x 8 tiles needs 12.  The columns are therefore
// cut into groups of at most 8 (as equal as possible), and the order walks a group row by row before it moves to
// the next group (E [15356, 4096] x C [128256, 4096], 16 column tiles: backward 39.3 -> 38.1 ms).
// The splits of a reduction are walked one after the other: neighbours then share the same range of the operands.
__device__ __forceinline__ bool product_tile_of(int block, int items, int splits, int per_xcd, int tiles_n, int& split,
                                                int& tm, int& tn) {
  const int xcd = block & 7;
  const int slot = block >> 3;
  int lin = xcd * per_xcd + slot;
  if (lin >= items) return false;
  const int tiles = items / splits;
  split = lin / tiles;
  lin -= split * tiles;
  const int tiles_m = tiles / tiles_n;
  const int groups = (tiles_n + 7) / 8;
  const int narrow = tiles_n / groups;          // width of the narrow groups; the first `wide` groups have one more
  const int wide = tiles_n - narrow * groups;
  const int in_wide = wide * tiles_m * (narrow + 1);
  int width, first_col;
  if (lin < in_wide) {
    width = narrow + 1;
    const int grp = lin / (tiles_m * width);
    lin -= grp * tiles_m * width;
    first_col = grp * width;
  } else {
    width = narrow;
    lin -= in_wide;
    const int grp = lin / (tiles_m * width);
    lin -= grp * tiles_m * width;
    first_col = wide * (narrow + 1) + grp * width;
  }
  tm = lin / width;
  tn = first_col + (lin - tm * width);
  return true;
}

// Eight consecutive floats of a row from column `col` on, of `d` columns in all; `vec`: rows are 16-byte aligned and d a
// multiple of 8.
__device__ __forceinline__ void load_piece(const float* row, int col, int d, bool vec, float (&v)[8]) {
  if (vec) {
    const float4 a = *reinterpret_cast<const float4*>(row + col), b = *reinterpret_cast<const float4*>(row + col + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (col + k < d) ? row[col + k] : 0.0f;
  }
}
__device__ __forceinline__ void store_piece(float* row, int col, int d, bool vec, const float (&v)[8]) {
  if (vec) {
    *reinterpret_cast<float4*>(row + col) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(row + col + 4) = make_float4(v[4], v[5], v[6], v[7]);
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (col + k < d) row[col + k] = v[k];
  }
}

// Where the operands of a tile lie: dE = dz . C (rows m0 on, columns n0 on, classes k0 on) and dC = dz^T . E (classes m0 on, rows
// k0 on).  Rows past the end repeat the last one, chunks past the `cols` columns of a matrix the last one inside it: their
// results are dropped.
template <typename Tile>
__device__ __forceinline__ void de_source(typename Tile::Source& s, const ProductParams& p, const typename Tile::Geometry& g,
                                          int64_t m0, int n0, int k0, int cols) {
  s.a_base = reinterpret_cast<const unsigned char*>(p.dz + m0 * p.ldz + k0);
  const int last = static_cast<int>(min(p.b - m0, static_cast<int64_t>(Tile::TILE))) - 1;
#pragma unroll
  for (int q = 0; q < Tile::NQ; ++q)
    s.a_off[q] = 2u * (static_cast<unsigned>(min(Tile::row_direct(q, g.wave, g.lane), last)) * static_cast<unsigned>(p.ldz) +
                       static_cast<unsigned>(Tile::chunk_direct(g.wave, g.lane)));
  s.a_stride = 0;
  s.b_base = reinterpret_cast<const unsigned char*>(p.c + k0 * p.stride_cv);
  s.b_stride = static_cast<uint32_t>(2 * p.stride_cv);
  s.b_off = (g.lane >> 5) * s.b_stride + 2u * static_cast<unsigned>(min(n0 + Tile::chunk_kmajor(g.wave, g.lane), cols - 8));
  s.b_rows = nullptr;
  s.k_total = min(p.de_len, p.n_cls - k0);
}
template <typename Tile, bool GATHER>
__device__ __forceinline__ void dc_source(typename Tile::Source& s, const ProductParams& p, const typename Tile::Geometry& g, int m0,
                                          int n0, int64_t k0, int64_t dz_cols, int cols) {
  const int chunk = Tile::chunk_kmajor(g.wave, g.lane);
  s.a_base = reinterpret_cast<const unsigned char*>(p.dz + k0 * p.ldz);
  s.a_stride = static_cast<uint32_t>(2 * p.ldz);
  s.a_off[0] = (g.lane >> 5) * s.a_stride + 2u * static_cast<unsigned>(min(static_cast<int64_t>(m0 + chunk), dz_cols - 8));
  s.b_base = reinterpret_cast<const unsigned char*>(p.e + (GATHER ? 0 : k0 * p.stride_e));
  s.b_stride = static_cast<uint32_t>(2 * p.stride_e);
  s.b_off = (GATHER ? 0u : (g.lane >> 5) * s.b_stride) + 2u * static_cast<unsigned>(min(n0 + chunk, cols - 8));
  s.b_rows = GATHER ? p.valids + k0 : nullptr;
  s.k_total = static_cast<int>(min(static_cast<int64_t>(p.dc_len), p.b - k0));
}

// The two products of operands in parts, fp32 results: the tiles below without what 16-bit gradients need.
__device__ __forceinline__ void terms_de_tile(const ProductParams& p, int split, int tm, int tn, unsigned char* smem) {
  using Tile = Tile8<BF16, false, false, true>;
  typename Tile::Geometry g = Tile::geometry(smem);
  const int64_t m0 = static_cast<int64_t>(tm) * Tile::TILE;
  const int n0 = tn * Tile::TILE;
  const int k0 = split * p.de_len;
  typename Tile::Source s;
  de_source<Tile>(s, p, g, m0, n0, k0, p.part_d);
  s.a_part = 2 * static_cast<int64_t>(p.dz_part);
  s.b_part = 2 * static_cast<int64_t>(p.part_d);
  s.terms = p.terms;
  Tile::plan(s);
  float* const de = p.de_f32 + split * p.de_slot;

  f32x4 acc[Tile::WM][Tile::WN];
  Tile::run(acc, s, smem, g);
  Tile::for_each_row_piece(acc, smem, g, [&](int row, int col, const float (&v)[8]) {
    const int64_t ri = m0 + row;
    const int cg = n0 + col;
    if (ri >= p.rows_out || cg >= p.d) return;
    const int64_t re = (p.valids != nullptr && !p.de_rows_by_number) ? static_cast<int64_t>(p.valids[ri]) : ri;
    float out[8];
    if (p.de_init) {
#pragma unroll
      for (int k = 0; k < 8; ++k) out[k] = v[k];
    } else {
      load_piece(de + re * p.ld_de, cg, p.d, p.out_vec != 0, out);
#pragma unroll
      for (int k = 0; k < 8; ++k) out[k] += v[k];
    }
    store_piece(de + re * p.ld_de, cg, p.d, p.out_vec != 0, out);
  });
}

__device__ __forceinline__ void terms_dc_tile(const ProductParams& p, int split, int tm, int tn, unsigned char* smem) {
  using Tile = Tile8<BF16, true, false, true>;
  typename Tile::Geometry g = Tile::geometry(smem);
  const int m0 = tm * Tile::TILE;
  const int n0 = tn * Tile::TILE;
  const int64_t k0 = static_cast<int64_t>(split) * p.dc_len;
  typename Tile::Source s;
  dc_source<Tile, false>(s, p, g, m0, n0, k0, p.dz_part, p.part_d);
  s.a_part = 2 * static_cast<int64_t>(p.dz_part);
  s.b_part = 2 * static_cast<int64_t>(p.part_d);
  s.terms = p.terms;
  Tile::plan(s);
  float* const dc = static_cast<float*>(p.d_c) + split * p.dc_slot;

  f32x4 acc[Tile::WM][Tile::WN];
  Tile::run(acc, s, smem, g);
  Tile::for_each_row_piece(acc, smem, g, [&](int row, int col, const float (&v)[8]) {
    const int cls = m0 + row;
    const int cg = n0 + col;
    if (cls >= p.cls_out || cg >= p.d) return;
    float* dst = dc + static_cast<int64_t>(cls) * p.ld_dc;
    float out[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = v[k];
    if (p.dc_accumulate) {
      float old[8];
      load_piece(dst, cg, p.d, p.out_vec != 0, old);
#pragma unroll
      for (int k = 0; k < 8; ++k) out[k] += old[k];
    }
    store_piece(dst, cg, p.d, p.out_vec != 0, out);
  });
}

// dE[row][col] += sum_class dz[row][class] * C[class][col]
template <typename T, bool SPLIT_DE>
__device__ __forceinline__ void dense_de_tile(const ProductParams& p, int split, int tm, int tn, unsigned char* smem) {
  using Tile = Tile8<T, false>;
  typename Tile::Geometry g = Tile::geometry(smem);
  const int64_t m0 = static_cast<int64_t>(tm) * Tile::TILE;
  const int n0 = tn * Tile::TILE;
  const int k0 = split * p.de_len;

  typename Tile::Source s;
  de_source<Tile>(s, p, g, m0, n0, k0, p.d);
  Tile::plan(s);
  float* const de_f32 = SPLIT_DE ? nullptr : p.de_f32 + split * p.de_slot;

  // What memory holds of a piece so far, fetched ahead of its use.
  struct Old {
    int64_t re;   // the piece's row of e (-1: the piece lies outside the matrix)
    uint4 a, b;   // fp32 dE: the eight sums; a 16-bit dE: the hi and the lo halves of the eight sums
  };
  auto fetch = [&](int row, int col) {
    Old o;
    o.re = -1;
    o.a = make_uint4(0u, 0u, 0u, 0u);
    o.b = make_uint4(0u, 0u, 0u, 0u);
    const int64_t ri = m0 + row;          // valid-row number
    const int cg = n0 + col;
    if (ri >= p.b || cg >= p.d) return o;
    o.re = (p.valids != nullptr && !p.de_rows_by_number) ? static_cast<int64_t>(p.valids[ri]) : ri;
    if (!SPLIT_DE) {
      if (p.de_init) return o;
      const uint4* src = reinterpret_cast<const uint4*>(de_f32 + o.re * p.ld_de + cg);
      o.a = src[0];
      o.b = src[1];
    } else if (!p.first_chunk) {  // (never with de_lo == nullptr: a d_e written alone is a first chunk)
      o.a = *reinterpret_cast<const uint4*>(p.de_hi + o.re * p.ld_de + cg);
      o.b = *reinterpret_cast<const uint4*>(p.de_lo + ri * p.d + cg);
    }
    return o;
  };
  f32x4 acc[Tile::WM][Tile::WN];
  Tile::run(acc, s, smem, g);

  Tile::template for_each_row_piece_rmw<Old>(acc, smem, g, fetch, [&](int row, int col, const float (&v)[8], const Old& o) {
    if (o.re < 0) return;
    const int64_t ri = m0 + row;
    const int cg = n0 + col;
    if (!SPLIT_DE) {
      float4* dst = reinterpret_cast<float4*>(de_f32 + o.re * p.ld_de + cg);
      float4 a = __builtin_bit_cast(float4, o.a), b = __builtin_bit_cast(float4, o.b);
      a.x += v[0]; a.y += v[1]; a.z += v[2]; a.w += v[3];
      b.x += v[4]; b.y += v[5]; b.z += v[6]; b.w += v[7];
      dst[0] = a;
      dst[1] = b;
    } else {
      // value so far = hi + lo (two 16-bit numbers: 16 bits of mantissa, where one would round the sum of a few
      // dozen chunks eight bits short); the new hi is the rounded total, so the last chunk leaves d_e final
      uint4* hi_ptr = reinterpret_cast<uint4*>(p.de_hi + o.re * p.ld_de + cg);
      uint4* lo_ptr = reinterpret_cast<uint4*>(p.de_lo + ri * p.d + cg);
      const uint32_t hw[4] = {o.a.x, o.a.y, o.a.z, o.a.w}, lw[4] = {o.b.x, o.b.y, o.b.z, o.b.w};
      uint32_t ho[4], lo_out[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float t[2], rest[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          t[h] = (Elem<T>::to_float(static_cast<uint16_t>(hw[k] >> (16 * h))) +
                  Elem<T>::to_float(static_cast<uint16_t>(lw[k] >> (16 * h)))) + v[2 * k + h];
        ho[k] = Elem<T>::pack2(t[0], t[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) rest[h] = t[h] - Elem<T>::to_float(static_cast<uint16_t>(ho[k] >> (16 * h)));
        lo_out[k] = Elem<T>::pack2(rest[0], rest[1]);
      }
      *hi_ptr = make_uint4(ho[0], ho[1], ho[2], ho[3]);
      if (p.de_lo != nullptr) *lo_ptr = make_uint4(lo_out[0], lo_out[1], lo_out[2], lo_out[3]);
    }
  });
}

// dC[class][col] = sum_row dz[row][class] * E[row][col]; GATHER: the rows of E come through valids
template <typename T, bool GATHER>
__device__ __forceinline__ void dense_dc_tile(const ProductParams& p, int split, int tm, int tn, unsigned char* smem) {
  using Tile = Tile8<T, true, GATHER>;
  typename Tile::Geometry g = Tile::geometry(smem);
  const int m0 = tm * Tile::TILE;
  const int n0 = tn * Tile::TILE;
  const int64_t k0 = static_cast<int64_t>(split) * p.dc_len;

  typename Tile::Source s;
  dc_source<Tile, GATHER>(s, p, g, m0, n0, k0, p.ldz, p.d);
  Tile::plan(s);

  f32x4 acc[Tile::WM][Tile::WN];
  Tile::run(acc, s, smem, g);

  if (p.dc_lo != nullptr) {
    // a 16-bit dC carried over blocks of rows: value so far = hi + lo, as dE is carried over chunks of classes
    struct Old {
      int ok;
      uint4 a, b;
    };
    auto fetch = [&](int row, int col) {
      Old o;
      o.ok = 0;
      o.a = make_uint4(0u, 0u, 0u, 0u);
      o.b = make_uint4(0u, 0u, 0u, 0u);
      const int cls = m0 + row;
      const int cg = n0 + col;
      if (cls >= p.n_cls || cg >= p.d) return o;
      o.ok = 1;
      if (!p.dc_first) {
        o.a = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.d_c) + static_cast<int64_t>(cls) * p.ld_dc + cg);
        o.b = *reinterpret_cast<const uint4*>(p.dc_lo + static_cast<int64_t>(cls) * p.d + cg);
      }
      return o;
    };
    Tile::template for_each_row_piece_rmw<Old>(acc, smem, g, fetch, [&](int row, int col, const float (&v)[8], const Old& o) {
      if (!o.ok) return;
      const int cls = m0 + row;
      const int cg = n0 + col;
      uint4* hi_ptr = reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.d_c) + static_cast<int64_t>(cls) * p.ld_dc + cg);
      uint4* lo_ptr = reinterpret_cast<uint4*>(p.dc_lo + static_cast<int64_t>(cls) * p.d + cg);
      const uint32_t hw[4] = {o.a.x, o.a.y, o.a.z, o.a.w}, lw[4] = {o.b.x, o.b.y, o.b.z, o.b.w};
      uint32_t ho[4], lo_out[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float t[2], rest[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          t[h] = (Elem<T>::to_float(static_cast<uint16_t>(hw[k] >> (16 * h))) +
                  Elem<T>::to_float(static_cast<uint16_t>(lw[k] >> (16 * h)))) + v[2 * k + h];
        ho[k] = Elem<T>::pack2(t[0], t[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) rest[h] = t[h] - Elem<T>::to_float(static_cast<uint16_t>(ho[k] >> (16 * h)));
        lo_out[k] = Elem<T>::pack2(rest[0], rest[1]);
      }
      *hi_ptr = make_uint4(ho[0], ho[1], ho[2], ho[3]);
      *lo_ptr = make_uint4(lo_out[0], lo_out[1], lo_out[2], lo_out[3]);
    });
    return;
  }
  Tile::for_each_row_piece(acc, smem, g, [&](int row, int col, const float (&v)[8]) {
    const int cls = m0 + row;
    const int cg = n0 + col;
    if (cls >= p.n_cls || cg >= p.d) return;
    const int64_t off = split * p.dc_slot + static_cast<int64_t>(cls) * p.ld_dc + cg;
    if (p.dc_fp32) {
      float4* dst = reinterpret_cast<float4*>(static_cast<float*>(p.d_c) + off);
      float4 a = make_float4(v[0], v[1], v[2], v[3]), b = make_float4(v[4], v[5], v[6], v[7]);
      if (p.dc_accumulate) {
        const float4 a0 = dst[0], b0 = dst[1];
        a.x += a0.x; a.y += a0.y; a.z += a0.z; a.w += a0.w;
        b.x += b0.x; b.y += b0.y; b.z += b0.z; b.w += b0.w;
      }
      dst[0] = a;
      dst[1] = b;
    } else {
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.d_c) + off) =
          make_uint4(Elem<T>::pack2(v[0], v[1]), Elem<T>::pack2(v[2], v[3]), Elem<T>::pack2(v[4], v[5]), Elem<T>::pack2(v[6], v[7]));
    }
  });
}

// Both products of one chunk in one launch.  Blocks are handed to compute units in id order as units fall free:
// the kind of tile with the longer reduction (dC: all B rows; dE: the classes of the chunk) takes the first block
// ids, so that the shorter tiles fill the last round of the longer ones.
template <typename T, bool SPLIT_DE>
__global__ __launch_bounds__(kProdThreads, 1) void dense_products_kernel(ProductParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int first_blocks = (p.de_first ? p.de_per_xcd : p.dc_per_xcd) * 8;
  const bool first = static_cast<int>(blockIdx.x) < first_blocks;
  const int block = first ? blockIdx.x : blockIdx.x - first_blocks;
  int split, tm, tn;
  if (first != (p.de_first != 0)) {
    if (!product_tile_of(block, p.dc_tiles, p.dc_splits, p.dc_per_xcd, p.tiles_n, split, tm, tn)) return;
    if (p.valids != nullptr) {
      dense_dc_tile<T, true>(p, split, tm, tn, smem);
    } else {
      dense_dc_tile<T, false>(p, split, tm, tn, smem);
    }
  } else {
    if (!product_tile_of(block, p.de_tiles, p.de_splits, p.de_per_xcd, p.tiles_n, split, tm, tn)) return;
    dense_de_tile<T, SPLIT_DE>(p, split, tm, tn, smem);
  }
}

// The same for operands in parts.
__global__ __launch_bounds__(kProdThreads, 1) void terms_products_kernel(ProductParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int first_blocks = (p.de_first ? p.de_per_xcd : p.dc_per_xcd) * 8;
  const bool first = static_cast<int>(blockIdx.x) < first_blocks;
  const int block = first ? blockIdx.x : blockIdx.x - first_blocks;
  int split, tm, tn;
  if (first != (p.de_first != 0)) {
    if (!product_tile_of(block, p.dc_tiles, p.dc_splits, p.dc_per_xcd, p.tiles_n, split, tm, tn)) return;
    terms_dc_tile(p, split, tm, tn, smem);
  } else {
    if (!product_tile_of(block, p.de_tiles, p.de_splits, p.de_per_xcd, p.tiles_n, split, tm, tn)) return;
    terms_de_tile(p, split, tm, tn, smem);
  }
}

// out[row(i)][:] (+)= sum over the slots of slot[s][i][:], in the order of the slots; eight columns per thread.  Bound
// by reading the slots: 4 bytes per element and slot.
template <typename T>
__global__ __launch_bounds__(256) void split_sum_kernel(const float* slots, int splits, int64_t rows, int d, int ld_slot,
                                                        const int32_t* ids, void* out, int64_t ld_out, int out_fp32, int add,
                                                        int out_vec) {
  const int per_row = (d + 7) / 8;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (item >= rows * per_row) return;
  const int64_t i = item / per_row;
  const int col = static_cast<int>(item - i * per_row) * 8;
  float v[8] = {};
  for (int s = 0; s < splits; ++s) {
    float x[8];
    load_piece(slots + (s * rows + i) * ld_slot, col, ld_slot, true, x);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] += x[k];
  }
  const int64_t row = (ids != nullptr ? static_cast<int64_t>(ids[i]) : i);
  if (out_fp32) {
    float* dst = static_cast<float*>(out) + row * ld_out;
    if (add) {
      float old[8];
      load_piece(dst, col, d, out_vec != 0, old);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] += old[k];
    }
    store_piece(dst, col, d, out_vec != 0, v);
  } else {
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + row * ld_out + col) =
        make_uint4(Elem<T>::pack2(v[0], v[1]), Elem<T>::pack2(v[2], v[3]), Elem<T>::pack2(v[4], v[5]), Elem<T>::pack2(v[6], v[7]));
  }
}

// d_bias[class] += sum over the rows of dz[row][class] (of the parts of it, where dz comes in parts).  A thread reads 16
// bytes of a row, 8 threads side by side whole lines of 64 classes, four rows in flight per thread; the 128 row lanes of a workgroup are
// added up in a fixed order, those of a wave by exchanges between its lanes, then the 16 waves in LDS.  Bound by reading dz.  Few
// classes make few workgroups: the rows are then cut into ranges, each with a workgroup, which leaves its sums, as floats, in
// the first two rows of its own range (no one reads dz any more, the workgroup itself has), and colsum_merge_kernel adds them up in
// their order.  (Narrower columns of whole reductions, down to a 16-byte one, with a tree of barriers in LDS, read as many times the lines.
// They took / it takes, us, dz in bf16: [54888] x 1088 80 / 20 + 6, [14264] x 4448 52 / 23 + 4, [4096] x 32000 50 / 47, [900] x 50257 26 / 19; in three
// parts: 253 / 34 + 10, 196 / 91 + 5, 123 / 96 + 5, 88 / 65, the first in two chunks of classes.)
constexpr int kColsumClasses = 64, kColsumLanes = 128;
// As a tree: a large entry among many small ones is rounded with every number that is added to it.  (The waves and the ranges one after the
// other: classes that are the label of one of 8192 rows had their dBias off by 4.0e-7, root mean square, now 2.9e-8.)
template <int N>
__device__ __forceinline__ float pairwise_sum(float (&v)[N]) {
#pragma unroll
  for (int half = N / 2; half >= 1; half /= 2)
#pragma unroll
    for (int k = 0; k < half; ++k) v[k] += v[k + half];
  return v[0];
}
template <typename T>
__global__ __launch_bounds__(1024) void dz_colsum_kernel(uint16_t* dz, int64_t ldz, int parts, int64_t b, int n_cls, int blocks, int ranges,
                                                         float* d_bias) {
  __shared__ float s_sum[1024 / 64][kColsumClasses];
  const int cl = threadIdx.x % 8, rl = threadIdx.x / 8;
  const int block = blockIdx.x % blocks, range = blockIdx.x / blocks;
  const int64_t begin = b * range / ranges, end = b * (range + 1) / ranges;
  const int cls = block * kColsumClasses + cl * 8;
  float sum[8] = {};
  if (cls < n_cls) {  // (a row of dz goes on in whole 16-byte pieces)
    auto value = [&](int64_t i, float (&x)[8]) {
      for (int part = parts - 1; part >= 0; --part) {
        const uint4 v = *reinterpret_cast<const uint4*>(dz + (i * parts + part) * ldz + cls);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] += Elem<T>::to_float(static_cast<uint16_t>(w[k >> 1] >> (16 * (k & 1))));
      }
    };
    // (the last time a row that does not exist is the last one again, and not added)
    auto four = [&](int64_t i, auto last) {
      float x[4][8] = {};
#pragma unroll
      for (int u = 0; u < 4; ++u) value(decltype(last)::value ? min(i + u * kColsumLanes, end - 1) : i + u * kColsumLanes, x[u]);
      if constexpr (decltype(last)::value) {
#pragma unroll
        for (int u = 1; u < 4; ++u)
#pragma unroll
          for (int k = 0; k < 8; ++k) x[u][k] = i + u * kColsumLanes < end ? x[u][k] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) sum[k] += (x[0][k] + x[1][k]) + (x[2][k] + x[3][k]);
    };
    int64_t i = begin + rl;
    for (; i + 3 * kColsumLanes < end; i += 4 * kColsumLanes) four(i, std::false_type{});
    if (i < end) four(i, std::true_type{});
  }
#pragma unroll
  for (int off = 32; off >= 8; off >>= 1)
#pragma unroll
    for (int k = 0; k < 8; ++k) sum[k] += __shfl_xor(sum[k], off, 64);
  if ((threadIdx.x & 63) < 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) s_sum[threadIdx.x >> 6][cl * 8 + k] = sum[k];
  }
  __syncthreads();
  if (threadIdx.x < kColsumClasses) {
    float wave_sum[1024 / 64];
#pragma unroll
    for (int w = 0; w < 1024 / 64; ++w) wave_sum[w] = s_sum[w][threadIdx.x];
    const float all = pairwise_sum(wave_sum);
    const int c = block * kColsumClasses + threadIdx.x;
    if (ranges == 1) {
      if (c < n_cls) d_bias[c] += all;
    } else if ((c & ~7) < n_cls) {
      reinterpret_cast<float*>(dz + (begin * parts + ((c >> 2) & 1)) * ldz + (c & ~7))[c & 3] = all;
    }
  }
}
__global__ __launch_bounds__(256) void colsum_merge_kernel(const uint16_t* dz, int64_t ldz, int parts, int64_t b, int n_cls, int ranges,
                                                           float* d_bias) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= n_cls) return;
  float sums[8] = {};
  for (int first = 0; first < ranges; first += 8) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t s = min(first + k, ranges - 1);
      const float x = reinterpret_cast<const float*>(dz + (b * s / ranges * parts + ((c >> 2) & 1)) * ldz + (c & ~7))[c & 3];
      sums[k] += first + k < ranges ? x : 0.0f;
    }
  }
  d_bias[c] += pairwise_sum(sums);
}

// The last reader of dz: its contents are gone afterwards.
int dz_colsum_launch(uint16_t* dz, int64_t ldz, int parts, int64_t b, int64_t n_cls, float* d_bias, int dtype,
                     hipStream_t stream) {
  const int blocks = static_cast<int>((n_cls + kColsumClasses - 1) / kColsumClasses);
  // two workgroups to a compute unit, and at least one row per row lane: never fewer than the two rows that the sums take
  int64_t ranges = 2 * compute_units() / blocks;
  if (ranges > b / kColsumLanes) ranges = b / kColsumLanes;
  if (ranges > 64) ranges = 64;
  if (ranges < 1) ranges = 1;
  const dim3 grid(static_cast<unsigned>(blocks * ranges));
  if (dtype == CCE_DTYPE_BF16)
    hipLaunchKernelGGL(dz_colsum_kernel<BF16>, grid, dim3(1024), 0, stream, dz, ldz, parts, b, static_cast<int>(n_cls), blocks,
                       static_cast<int>(ranges), d_bias);
  else
    hipLaunchKernelGGL(dz_colsum_kernel<F16>, grid, dim3(1024), 0, stream, dz, ldz, parts, b, static_cast<int>(n_cls), blocks,
                       static_cast<int>(ranges), d_bias);
  if (ranges > 1)
    hipLaunchKernelGGL(colsum_merge_kernel, dim3(static_cast<unsigned>((n_cls + 255) / 256)), dim3(256), 0, stream, dz, ldz, parts, b,
                       static_cast<int>(n_cls), static_cast<int>(ranges), d_bias);
  return status_from_hip(hipGetLastError());
}

static int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Finishing time of a launch of n1 items of length l1 and n2 of length l2 handed out, longer kind first, to the compute
// units as they fall free.  (With l1 >= l2 the units fall free at q l1 or (q + 1) l1, and the n2 short items end at the
// n2 smallest of {free + k l2}.)
static int64_t product_makespan(int64_t n1, int64_t l1, int64_t n2, int64_t l2) {
  const int64_t cus = compute_units();
  if (l1 < l2) {
    std::swap(n1, n2);
    std::swap(l1, l2);
  }
  const int64_t q = n1 / cus, r = n1 % cus;
  const int64_t early = q * l1, late = (q + 1) * l1;
  if (n2 == 0 || l2 == 0) return r > 0 ? late : early;
  auto done_by = [&](int64_t t) {
    return (cus - r) * ((t - early) / l2) + (t > late ? r * ((t - late) / l2) : 0);
  };
  auto first_end = [&](int64_t base) {  // the least base + k l2 by which all short items are done
    int64_t lo = 0, hi = n2;
    while (lo < hi) {
      const int64_t k = (lo + hi) / 2;
      if (done_by(base + k * l2) >= n2) hi = k; else lo = k + 1;
    }
    return base + lo * l2;
  };
  int64_t end = first_end(early);
  if (r > 0) {
    const int64_t other = first_end(late);
    end = other < end ? other : end;
    end = end < late ? late : end;
  }
  return end;
}

// How cce_backward_dense walks the [b, v] plane for a dz buffer of at most `max_dz_bytes`.
//   by classes  chunks of `unit` classes, all b rows each: dC of a chunk is complete, dE is carried over the chunks
//               (a 16-bit dE as a pair: fixed part of the workspace = its [b, d] compensation term);
//   by rows     blocks of `unit` rows, all v classes each: dE of a block is complete, dC is carried over the blocks
//               (fixed part = a [v, d] compensation term).
// Both walks take the same number of launches for the same buffer; what is carried is read and written once per
// launch, and its compensation term sits in the workspace for the whole call, so the walk goes by rows where the
// rows outnumber the classes two to one (measured, E [65536, 3584] x C [19008, 3584]: 36.1 ms and 581 MB by classes
// with 1024-class chunks, against the same 130 MB of dz by rows).  Only with 16-bit gradients: an fp32 dE is its own
// accumulator.  unit == 0: not even the smallest plan (256 classes / rows) fits.
//   splits      into how many ranges the reductions of dE and dC are cut.  The slots of the gradient that is carried are
//               then what is carried, in place of the pair and its compensation term; those of the other one are added up
//               after every launch.
struct DensePlan {
  bool by_rows;
  int64_t unit;
  int de_splits, dc_splits;
  int64_t fixed_bytes;  // what the size query promises to need beside the dz buffer
  int64_t comp_bytes;   // the compensation term this plan keeps (0 where the carried gradient sits in slots)
  int64_t dz_bytes;
  int64_t slot_bytes;   // of all slots
};
// (A block's rows of dz are whole vocabularies apart, and a tile of dE reaches 256 of them by 32-bit byte offsets: wider ones
// go by classes.)
static bool dense_walks_by_rows(int64_t b, int64_t v, bool gradients_16bit) {
  const int64_t v_pad = (v + 255) / 256 * 256;
  return gradients_16bit && b >= 2 * v_pad && v_pad <= (int64_t(1) << 23);
}

// A split of n steps of 64: multiples of whole stages, so that only the last one has a partial stage.
static int64_t split_stages(int64_t stages, int splits) { return (stages + splits - 1) / splits; }

// Estimated time of one launch pair (dz kernel, products) over `rows` rows and `cls` classes, in reduction stages of a
// product tile (64 steps of 256 x 256; 1.65 us where all units are busy): the dz tiles in rounds of all units, d / 64
// stages each, then the product items as they are handed out.  An item of a cut reduction leaves 256 KB of fp32 (and
// takes them in first, where slots are carried): up to 6 stages of time where every unit does so at once.
// whole_tiles: reductions counted in whole tiles of 256 steps, as the chunks of whole reductions are chosen.
static double launch_cost(int64_t rows, int64_t cls, int64_t d, int de_splits, int dc_splits, bool de_carried, bool dc_carried,
                          int terms = 1, bool whole_tiles = false) {
  const int64_t cus = compute_units();
  const int64_t tr = (rows + 255) / 256, tc = (cls + 255) / 256, tn = (d + 255) / 256;
  const int64_t dz = (tr * tc + cus - 1) / cus * tn * 4 * terms;
  auto item = [&](int64_t total, int splits, int64_t tiles, bool carried) {
    if (whole_tiles) return (total + 255) / 256 * 4;
    const int64_t len = split_stages((total + 63) / 64, splits) * terms;
    if (splits == 1) return len;
    const int64_t items = tiles * splits;
    return len + (4 + 6 * (items < cus ? items : cus) / cus) * (carried ? 2 : 1);
  };
  return static_cast<double>(dz + product_makespan(tc * tn * dc_splits, item(rows, dc_splits, tc * tn, dc_carried),
                                                   tr * tn * de_splits, item(cls, de_splits, tr * tn, de_carried)));
}

// Adding the slots up at the end: a launch, and reading them at 4 TB/s (6.6 MB in the time of a stage).
static double split_sum_cost(int64_t rows, int64_t d, int splits) {
  return splits == 1 ? 0.0 : 4.0 + static_cast<double>(splits) * static_cast<double>(rows * d) * 4.0 / 6.6e6;
}

// At least this many stages per split: below, an item is mostly its own start and end.
constexpr int64_t kMinSplitStages = 8;
constexpr int64_t kMaxChunkClasses = 16384;
constexpr double kCutMargin = 1.03, kMoreLaunchesMargin = 1.15;

static DensePlan dense_plan_uncached(int64_t b, int64_t v, int64_t d, bool g16, int64_t max_dz_bytes) {
  DensePlan pl = {};
  pl.by_rows = dense_walks_by_rows(b, v, g16);
  pl.de_splits = pl.dc_splits = 1;
  const int64_t v_pad = (v + 255) / 256 * 256, b_pad = (b + 255) / 256 * 256;
  pl.fixed_bytes = pl.by_rows ? align256(v * d * 2) : (g16 ? align256(b * d * 2) : 0);
  pl.comp_bytes = pl.fixed_bytes;
  const int64_t budget = max_dz_bytes + pl.fixed_bytes;  // what a plan may take in all
  double best = 1e300;

  // Takes a plan in if it fits and is estimated to be faster by `margin`.
  auto consider = [&](int64_t unit, int de_splits, int dc_splits, double margin) {
    const bool carried_cut = pl.by_rows ? dc_splits > 1 : de_splits > 1;
    const int64_t launches = pl.by_rows ? (b + unit - 1) / unit : (v + unit - 1) / unit;
    const int64_t comp = carried_cut ? 0 : pl.fixed_bytes;
    const int64_t dz = align256((pl.by_rows ? unit * v_pad : b * unit) * 2);
    const int64_t slot_rows = pl.by_rows ? std::min(unit, b) : b, slot_cls = pl.by_rows ? v : std::min(unit, v);
    const int64_t slots = align256(de_splits > 1 ? de_splits * slot_rows * d * 4 : 0) + align256(dc_splits > 1 ? dc_splits * slot_cls * d * 4 : 0);
    if (comp + dz + slots > budget || (margin > kCutMargin && slots > dz / 2)) return;
    auto launch = [&](int64_t n) {
      const int64_t rows = pl.by_rows ? n : b, cls = pl.by_rows ? v : n;
      double cost = 1.0 + launch_cost(rows, cls, d, de_splits, dc_splits, launches > 1 && !pl.by_rows, launches > 1 && pl.by_rows);
      return cost + (pl.by_rows ? split_sum_cost(rows, d, de_splits) : split_sum_cost(cls, d, dc_splits));
    };
    const int64_t whole = pl.by_rows ? b / unit : v / unit;
    const int64_t rest = pl.by_rows ? b - whole * unit : v - whole * unit;
    double cost = pl.by_rows ? split_sum_cost(v, d, dc_splits) : split_sum_cost(b, d, de_splits);
    if (whole > 0) cost += whole * launch(unit);
    if (rest > 0) cost += launch(rest);
    if (cost * margin >= best * (1.0 - 1e-9)) return;
    best = cost * margin;
    pl.unit = unit;
    pl.de_splits = de_splits;
    pl.dc_splits = dc_splits;
    pl.comp_bytes = comp;
    pl.dz_bytes = dz;
    pl.slot_bytes = slots;
  };

  // ---- whole reductions.  A carried 16-bit gradient is rounded once per launch, at places that go by the unit: the unit of
  // a plan without cuts is chosen by the estimate in whole tiles alone, apart from what the cut plans below are weighed
  // with, so that a shape which is not cut keeps the bits of its gradients whatever becomes of the other estimate, and by
  // rows it takes no launch more than the buffer asks for (E [65536, 3584] x C [19008, 3584]: ten blocks of 6656 rows;
  // twelve of 5632 take the same 28.9 ms, forward and backward, and round dC twice more).
  if (pl.by_rows) {
    int64_t rb = max_dz_bytes / (v_pad * 2) / 256 * 256;
    if (rb > b_pad) rb = b_pad;
    if (rb >= 256) {  // blocks of equal size: the last one is not a sliver
      const int64_t blocks = (b + rb - 1) / rb;
      rb = ((b + blocks - 1) / blocks + 255) / 256 * 256;
      consider(rb, 1, 1, 1.0);
    }
  } else {
    int64_t top = max_dz_bytes / (b * 2) / 256 * 256;
    if (top > kMaxChunkClasses) top = kMaxChunkClasses;
    int64_t unit = top >= v_pad ? v_pad : 0;
    double least = 1e300;
    for (int64_t vc = top; vc >= 256 && top < v_pad; vc -= 256) {
      const int64_t whole = v / vc, rest = v - whole * vc;
      double cost = static_cast<double>(whole) * (1.0 + launch_cost(b, vc, d, 1, 1, false, false, 1, true));
      if (rest > 0) cost += 1.0 + launch_cost(b, rest, d, 1, 1, false, false, 1, true);
      if (cost < least * (1.0 - 1e-9)) {
        least = cost;
        unit = vc;
      }
    }
    if (unit > 0) consider(unit, 1, 1, 1.0);
  }

  // ---- cut reductions, in as few launches as the budget allows (chunks past 16384 classes where the whole dz still
  // stays in the last-level cache), and a launch or two more: the slots compete with dz for the budget.  They have to win by
  // 3 %.  Where the slots leave room for none of those, in as few launches as they do leave room for (the budget is then
  // mostly what a filtered backward may take by itself: E [56512, 1024] x C [24608, 1024] ran 60 dE tiles of 385 stages beside
  // 388 dC tiles of 59; forward and backward 12.24 -> 11.03 ms in 17 smaller blocks with dE cut in three).  More launches of
  // shorter items are what the estimate knows least about (24911 x 68874 x 1280, by 6 % in the estimate: 17.8 ms became 19.6):
  // these have to win by 15 %, with slots of no more than half the dz buffer.
  static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
  const int64_t dz_cap = budget < (int64_t(256) << 20) ? budget : (int64_t(256) << 20);
  const int64_t along = pl.by_rows ? b_pad : v_pad;
  const int64_t dz_per_unit = (pl.by_rows ? v_pad : b) * 2;
  int64_t most = dz_cap / dz_per_unit / 256 * 256;
  if (most > along) most = along;
  if (most >= 256) {
    const int64_t least = (along + most - 1) / most;
    for (int se : kSplits) {
      for (int sc : kSplits) {
        if (se == 1 && sc == 1) continue;
        auto try_launches = [&](int64_t n, double margin) {
          const int64_t unit = ((along + n - 1) / n + 255) / 256 * 256;
          const int64_t rows = pl.by_rows ? unit : b, cls = pl.by_rows ? v : unit;
          if (se > 1 && (cls + 63) / 64 < se * kMinSplitStages) return;
          if (sc > 1 && (rows + 63) / 64 < sc * kMinSplitStages) return;
          consider(unit, se, sc, margin);
        };
        for (int64_t n = least; n <= least + 2; ++n) try_launches(n, kCutMargin);
        const int carried = pl.by_rows ? sc : se, other = pl.by_rows ? se : sc;
        const int64_t kept = carried > 1 ? carried * (pl.by_rows ? v : b) * d * 4 : pl.fixed_bytes;
        const int64_t room = (budget - kept) / (dz_per_unit + (other > 1 ? other * d * 4 : 0)) / 256 * 256;
        if (room < 256) continue;
        const int64_t fits = (along + room - 1) / room;
        if (fits > least + 2) {
          try_launches(fits, kMoreLaunchesMargin);
          try_launches(fits + 1, kMoreLaunchesMargin);
        }
      }
    }
  }
  return pl;
}

// The same questions come with every step of a training loop -- the size query with the caller's dz budget, then the
// call itself with the bytes that query answered -- so the last few answers of this thread are kept (a search weighs
// up to 64 chunk sizes and 400 ways to cut: 10 - 60 us of host time).
static DensePlan dense_plan(int64_t b, int64_t v, int64_t d, bool g16, int64_t max_dz_bytes) {
  struct Memo {
    int64_t b, v, d, bytes;
    bool g16;
    int cus;
    DensePlan answer;
  };
  constexpr int kMemos = 8;
  static thread_local Memo memo[kMemos] = {};
  static thread_local int next_slot = 0;
  const int cus = compute_units();
  for (int i = 0; i < kMemos; ++i) {
    const Memo& m = memo[i];
    if (m.b == b && m.v == v && m.d == d && m.bytes == max_dz_bytes && m.g16 == g16 && m.cus == cus && m.b != 0)
      return m.answer;
  }
  memo[next_slot] = {b, v, d, max_dz_bytes, g16, cus, dense_plan_uncached(b, v, d, g16, max_dz_bytes)};
  const DensePlan answer = memo[next_slot].answer;
  next_slot = (next_slot + 1) % kMemos;
  return answer;
}

// ---- the products of one chunk of classes with operands and dz in bf16 parts (cce_fp32.hip) ---------------------
// The walk over the classes for a dz of `dz_bytes_per_class` and a copy of C of `c_bytes_per_class`, either at most
// `most_bytes`, in chunks that are multiples of 256 classes; the reductions are cut as in cce_backward_dense.
static TermsPlan terms_plan_uncached(int64_t b, int64_t v, int64_t d, int terms, int64_t dz_bytes_per_class,
                                     int64_t c_bytes_per_class, int64_t most_bytes) {
  TermsPlan pl = {256, 1, 1};
  static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
  const int64_t v_pad = (v + 255) / 256 * 256;
  int64_t most = most_bytes / std::max(dz_bytes_per_class, c_bytes_per_class) / 256 * 256;
  most = std::min(std::max<int64_t>(most, 256), v_pad);
  const int64_t least = (v_pad + most - 1) / most;
  double best = 1e300;
  for (int64_t n = least; n <= least + 2; ++n) {
    const int64_t unit = ((v_pad + n - 1) / n + 255) / 256 * 256;
    const int64_t launches = (v + unit - 1) / unit;
    const int64_t rest = v - (launches - 1) * unit;
    for (int se : kSplits) {
      if (se > 1 && ((unit + 63) / 64 * terms < se * kMinSplitStages || se * b * d * 4 > most_bytes || unit / 64 < se)) break;
      for (int sc : kSplits) {
        if (sc > 1 && ((b + 63) / 64 * terms < sc * kMinSplitStages || sc * std::min(unit, v) * d * 4 > most_bytes ||
                       b / 64 < sc))
          break;
        auto launch = [&](int64_t cls) {
          return 1.0 + launch_cost(b, cls, d, se, sc, launches > 1, false, terms) + split_sum_cost(cls, d, sc);
        };
        double cost = static_cast<double>(launches - 1) * launch(unit) + launch(rest) + split_sum_cost(b, d, se);
        if (se > 1 || sc > 1) cost *= 1.03;
        if (cost < best * (1.0 - 1e-9)) {
          best = cost;
          pl.unit = unit;
          pl.de_splits = se;
          pl.dc_splits = sc;
        }
      }
    }
  }
  return pl;
}

// (asked by the size query and again by the call, with every step of a training loop, like dense_plan: 7 - 50 us each)
TermsPlan terms_plan(int64_t b, int64_t v, int64_t d, int terms, int64_t dz_bytes_per_class, int64_t c_bytes_per_class,
                     int64_t most_bytes) {
  struct Memo {
    int64_t b, v, d, dz, c, most;
    int terms, cus;
    TermsPlan answer;
  };
  constexpr int kMemos = 8;
  static thread_local Memo memo[kMemos] = {};
  static thread_local int next_slot = 0;
  const int cus = compute_units();
  for (int i = 0; i < kMemos; ++i) {
    const Memo& m = memo[i];
    if (m.b == b && m.v == v && m.d == d && m.dz == dz_bytes_per_class && m.c == c_bytes_per_class && m.most == most_bytes &&
        m.terms == terms && m.cus == cus)
      return m.answer;
  }
  const TermsPlan answer = terms_plan_uncached(b, v, d, terms, dz_bytes_per_class, c_bytes_per_class, most_bytes);
  memo[next_slot] = {b, v, d, dz_bytes_per_class, c_bytes_per_class, most_bytes, terms, cus, answer};
  next_slot = (next_slot + 1) % kMemos;
  return answer;
}

int terms_products_launch(const uint16_t* dz_parts, int64_t ldz, const uint16_t* c_parts, int64_t ld_c, const uint16_t* e_parts,
                          int64_t ld_e, const int32_t* valids, float* d_e, int64_t ld_de, bool de_by_number, bool de_init,
                          int64_t de_slot, int de_len, float* d_c, int64_t ld_dc, bool dc_add, int64_t dc_slot, int dc_len,
                          bool out_vec, int64_t b, int64_t b_pad, int64_t cls, int64_t cls_pad, int64_t d, int64_t part_d, int terms,
                          int parts, hipStream_t stream) {
  ProductParams p = {};
  p.dz = dz_parts;
  p.ldz = parts * ldz;
  p.dz_part = static_cast<int>(ldz);
  p.c = c_parts;
  p.stride_cv = ld_c;
  p.e = e_parts;
  p.stride_e = ld_e;
  p.valids = valids;
  p.de_f32 = d_e;
  p.ld_de = ld_de;
  p.de_rows_by_number = de_by_number ? 1 : 0;
  p.de_init = de_init ? 1 : 0;
  p.d_c = d_c;
  p.ld_dc = ld_dc;
  p.dc_accumulate = dc_add ? 1 : 0;
  p.b = b_pad;
  p.rows_out = b;
  p.n_cls = static_cast<int>(cls_pad);
  p.cls_out = static_cast<int>(cls);
  p.d = static_cast<int>(d);
  p.part_d = static_cast<int>(part_d);
  p.terms = terms;
  p.out_vec = out_vec ? 1 : 0;
  p.de_len = de_len;
  p.dc_len = dc_len;
  p.de_slot = de_slot;
  p.dc_slot = dc_slot;
  p.de_splits = static_cast<int>((cls_pad + de_len - 1) / de_len);
  p.dc_splits = static_cast<int>((b_pad + dc_len - 1) / dc_len);
  p.tiles_n = static_cast<int>((d + 255) / 256);
  p.dc_tiles = d_c != nullptr ? static_cast<int>((cls + 255) / 256) * p.tiles_n * p.dc_splits : 0;
  p.de_tiles = d_e != nullptr ? static_cast<int>((b + 255) / 256) * p.tiles_n * p.de_splits : 0;
  p.dc_per_xcd = (p.dc_tiles + 7) / 8;
  p.de_per_xcd = (p.de_tiles + 7) / 8;
  p.de_first = std::min<int64_t>(de_len, cls_pad) > std::min<int64_t>(dc_len, b_pad) ? 1 : 0;
  const int blocks = (p.dc_per_xcd + p.de_per_xcd) * 8;
  if (blocks == 0) return CCE_OK;
  const int lds = Tile8<BF16, true>::LDS_BYTES;
  auto kern = terms_products_kernel;
  static LdsLimitOnce lds_limit;
  const hipError_t err = lds_limit.set(kern, lds);
  if (err != hipSuccess) return status_from_hip(err);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kProdThreads), lds, stream, p);
  return status_from_hip(hipGetLastError());
}

int split_sum_launch(const float* slots, int count, int64_t rows, int64_t d, int64_t ld_slot, const int32_t* ids, float* out,
                     int64_t ld, bool add, bool out_vec, hipStream_t stream) {
  const unsigned blocks = static_cast<unsigned>((rows * ((d + 7) / 8) + 255) / 256);
  hipLaunchKernelGGL(split_sum_kernel<BF16>, dim3(blocks), dim3(256), 0, stream, slots, count, rows, static_cast<int>(d),
                     static_cast<int>(ld_slot), ids, out, ld, 1, add ? 1 : 0, out_vec ? 1 : 0);
  return status_from_hip(hipGetLastError());
}

}  // namespace cce

using namespace cce;

extern "C" int64_t cce_backward_dense_workspace_bytes(int64_t b, int64_t v, int64_t d, int d_e_in_workspace,
                                                      int64_t max_dz_bytes) {
  if (b <= 0 || v <= 0 || d <= 0) return 0;
  const DensePlan pl = dense_plan(b, v, d, d_e_in_workspace != 0, max_dz_bytes);
  if (pl.unit == 0) {  // the smallest plan
    const int64_t v_pad = (v + 255) / 256 * 256;
    return pl.fixed_bytes + align256(256 * (pl.by_rows ? v_pad : b) * 2);
  }
  return std::max(pl.comp_bytes + pl.dz_bytes + pl.slot_bytes, pl.fixed_bytes);
}

extern "C" int64_t cce_backward_dense_fixed_bytes(int64_t b, int64_t v, int64_t d, int d_e_in_workspace) {
  if (b <= 0 || v <= 0 || d <= 0) return 0;
  if (dense_walks_by_rows(b, v, d_e_in_workspace != 0)) return align256(v * d * 2);
  return d_e_in_workspace != 0 ? align256(b * d * 2) : 0;
}

extern "C" int64_t cce_backward_dense_dz_bytes(int64_t b, int64_t v, int64_t d, int d_e_in_workspace, int64_t units) {
  if (b <= 0 || v <= 0 || d <= 0 || units <= 0) return 0;
  const int64_t v_pad = (v + 255) / 256 * 256;
  const int64_t b_pad = (b + 255) / 256 * 256;
  const int64_t u = (units + 255) / 256 * 256;
  if (dense_walks_by_rows(b, v, d_e_in_workspace != 0)) return (u < b_pad ? u : b_pad) * v_pad * 2;
  return b * (u < v_pad ? u : v_pad) * 2;
}

extern "C" int cce_backward_dense(const void* e, const void* c, const void* bias,
                                  const float* lse, const float* d_out, int d_out_is_scalar, const float* d_lse,
                                  const int32_t* valids, const int64_t* targets,
                                  void* d_e, void* d_c, float* d_bias,
                                  void* workspace, int64_t workspace_bytes,
                                  int64_t n_rows, int64_t b, int64_t v, int64_t d,
                                  int64_t stride_e, int64_t stride_cv, int64_t stride_cd,
                                  float grad_scale, int d_e_is_fp32, int d_c_is_fp32,
                                  int64_t shift, int64_t target_offset,
                                  float softcap, int dtype, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (b < 0 || v <= 0 || d <= 0 || n_rows < 0 || shift < 0) return CCE_ERR_INVALID_ARGUMENT;
  if (b == 0) return CCE_OK;
  if (e == nullptr || c == nullptr || lse == nullptr || d_out == nullptr || targets == nullptr)
    return CCE_ERR_INVALID_ARGUMENT;
  if (valids == nullptr && b > n_rows) return CCE_ERR_INVALID_ARGUMENT;
  if (n_rows >= (int64_t(1) << 31) || b >= (int64_t(1) << 31) - 512 || v >= (int64_t(1) << 31) - 512 || d > (1 << 24))
    return CCE_ERR_INVALID_ARGUMENT;
  if (dtype != CCE_DTYPE_BF16 && dtype != CCE_DTYPE_F16) return CCE_ERR_UNSUPPORTED_DTYPE;
  if (d_e == nullptr && d_c == nullptr && d_bias == nullptr) return CCE_OK;
  if (!aligned16(e) || !aligned16(c) || !dense_width_ok(n_rows, d, stride_e, stride_cv) || stride_e % 8 != 0 || stride_cv % 8 != 0 || stride_cd != 1)
    return CCE_ERR_MISALIGNED;
  if (stride_e >= (int64_t(1) << 30) || stride_cv >= (int64_t(1) << 30)) return CCE_ERR_INVALID_ARGUMENT;
  if ((d_e != nullptr && !aligned16(d_e)) || (d_c != nullptr && !aligned16(d_c))) return CCE_ERR_MISALIGNED;
  if (workspace == nullptr || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
    return workspace == nullptr ? CCE_ERR_WORKSPACE_TOO_SMALL : CCE_ERR_MISALIGNED;

  // ---- plan: [16-bit compensation term of the gradient that is carried][dz buffer][slots of dE][slots of dC] ------
  const bool split_de = (d_e != nullptr) && !d_e_is_fp32;
  // (the walk by rows needs the caller to have sized the workspace for it: a 16-bit d_e is what the size query's
  // flag says, and a d_c in fp32 beside it is added to in place)
  const bool by_rows = dense_walks_by_rows(b, v, split_de);
  // the plan the size query made (both gradients wanted), so that its answer always suffices
  const DensePlan plan = dense_plan(b, v, d, split_de, workspace_bytes - cce_backward_dense_fixed_bytes(b, v, d, split_de));
  if (plan.unit == 0) return CCE_ERR_WORKSPACE_TOO_SMALL;
  unsigned char* const ws = static_cast<unsigned char*>(workspace);
  uint16_t* dz = reinterpret_cast<uint16_t*>(ws + plan.comp_bytes);
  float* const de_slots = reinterpret_cast<float*>(ws + plan.comp_bytes + plan.dz_bytes);
  float* const dc_slots =
      reinterpret_cast<float*>(ws + plan.comp_bytes + plan.dz_bytes +
                               (plan.de_splits > 1 ? align256(plan.de_splits * (by_rows ? std::min(plan.unit, b) : b) * d * 4) : 0));
  const int64_t vc = by_rows ? (v + 255) / 256 * 256 : plan.unit;
  const int64_t ldz = vc;
  const bool de_cut = d_e != nullptr && plan.de_splits > 1;
  const bool dc_cut = d_c != nullptr && plan.dc_splits > 1;
  const bool pair_de = split_de && !de_cut;  // dE leaves the products as 16-bit numbers

  ProductParams p = {};
  p.dz = dz;
  p.ldz = ldz;
  p.stride_cv = stride_cv;
  p.e = static_cast<const uint16_t*>(e);
  p.stride_e = stride_e;
  p.valids = valids;
  p.de_f32 = de_cut ? de_slots : (split_de ? nullptr : static_cast<float*>(d_e));
  p.de_hi = pair_de ? static_cast<uint16_t*>(d_e) : nullptr;
  p.de_lo = (pair_de && !by_rows) ? static_cast<uint16_t*>(workspace) : nullptr;
  p.ld_de = de_cut ? d : stride_e;
  p.dc_fp32 = dc_cut ? 1 : d_c_is_fp32;
  p.ld_dc = dc_cut ? d : stride_cv;
  p.dc_accumulate = 0;
  p.dc_lo = nullptr;
  p.dc_first = 1;
  p.de_rows_by_number = de_cut ? 1 : 0;
  p.de_init = 0;
  p.b = b;
  p.d = static_cast<int>(d);
  // Ranges of the reductions, fixed by the first launch, which is the largest: it fills every slot there is (seven stages
  // cut in five make four ranges of two, the last of them short), a later one has as many of them or fewer.
  const int64_t first_rows = by_rows ? std::min(plan.unit, b) : b, first_cls = by_rows ? v : std::min(vc, v);
  p.de_len = static_cast<int>(split_stages((first_cls + 63) / 64, de_cut ? plan.de_splits : 1) * 64);
  p.dc_len = static_cast<int>(split_stages((first_rows + 63) / 64, dc_cut ? plan.dc_splits : 1) * 64);
  const int de_nslots = static_cast<int>((first_cls + p.de_len - 1) / p.de_len);
  const int dc_nslots = static_cast<int>((first_rows + p.dc_len - 1) / p.dc_len);
  p.tiles_n = static_cast<int>((d + 255) / 256);
  auto set_items = [&](int64_t rows, int64_t cls) {  // the items of a launch over `rows` rows and `cls` classes
    p.b = rows;
    p.n_cls = static_cast<int>(cls);
    p.de_splits = static_cast<int>((cls + p.de_len - 1) / p.de_len);
    p.dc_splits = static_cast<int>((rows + p.dc_len - 1) / p.dc_len);
    p.de_slot = rows * d;  // slots are packed for what they hold: all rows or classes where they are carried
    p.dc_slot = cls * d;
    p.dc_tiles = (d_c != nullptr) ? static_cast<int>((cls + 255) / 256) * p.tiles_n * p.dc_splits : 0;
    p.de_tiles = (d_e != nullptr) ? static_cast<int>((rows + 255) / 256) * p.tiles_n * p.de_splits : 0;
    p.dc_per_xcd = (p.dc_tiles + 7) / 8;
    p.de_per_xcd = (p.de_tiles + 7) / 8;
    p.de_first = (std::min<int64_t>(p.de_len, cls) > std::min<int64_t>(p.dc_len, rows)) ? 1 : 0;
  };

  using TileB = Tile8<BF16, true>;
  const int lds = TileB::LDS_BYTES;
  hipError_t err;
#define CCE_LAUNCH_PRODUCT(KERN, BLOCKS)                                                            \
  do {                                                                                              \
    auto kern = KERN;                                                                               \
    static LdsLimitOnce lds_limit;                                                            \
    err = lds_limit.set(kern, lds);                                        \
    if (err != hipSuccess) return status_from_hip(err);                                             \
    hipLaunchKernelGGL(kern, dim3(BLOCKS), dim3(kProdThreads), lds, stream, p);                     \
  } while (0)
  // the products of the dz in the workspace (set_items() has been called), and dBias
  auto products = [&](int64_t rows, int64_t cls, float* bias_out) -> int {
    const int blocks = (p.dc_per_xcd + p.de_per_xcd) * 8;
    if (blocks > 0) {
      if (dtype == CCE_DTYPE_BF16) {
        if (pair_de) CCE_LAUNCH_PRODUCT((dense_products_kernel<BF16, true>), blocks);
        else CCE_LAUNCH_PRODUCT((dense_products_kernel<BF16, false>), blocks);
      } else {
        if (pair_de) CCE_LAUNCH_PRODUCT((dense_products_kernel<F16, true>), blocks);
        else CCE_LAUNCH_PRODUCT((dense_products_kernel<F16, false>), blocks);
      }
    }
    if (bias_out != nullptr) return dz_colsum_launch(dz, ldz, 1, rows, cls, bias_out, dtype, stream);
    return status_from_hip(hipGetLastError());
  };
#undef CCE_LAUNCH_PRODUCT

  auto sum_slots = [&](const float* slots, int count, int64_t rows, const int32_t* ids, void* out, int64_t ld, int fp32, int add) {
    const unsigned blocks = static_cast<unsigned>((rows * (d / 8) + 255) / 256);
    if (dtype == CCE_DTYPE_BF16)
      hipLaunchKernelGGL(split_sum_kernel<BF16>, dim3(blocks), dim3(256), 0, stream, slots, count, rows, static_cast<int>(d),
                         static_cast<int>(d), ids, out, ld, fp32, add, 1);
    else
      hipLaunchKernelGGL(split_sum_kernel<F16>, dim3(blocks), dim3(256), 0, stream, slots, count, rows, static_cast<int>(d),
                         static_cast<int>(d), ids, out, ld, fp32, add, 1);
  };

  const size_t es = 2;
  if (by_rows) {
    // ---- blocks of rows, the whole vocabulary each ------------------------------------------------------------
    const int64_t rb = plan.unit;
    p.c = static_cast<const uint16_t*>(c);
    p.first_chunk = 1;  // d_e of a block is complete with its launch
    p.de_init = 1;      // ... also where it is cut
    p.d_c = dc_cut ? static_cast<void*>(dc_slots) : d_c;
    p.dc_lo = (d_c != nullptr && !dc_cut && !d_c_is_fp32) ? static_cast<uint16_t*>(workspace) : nullptr;
    for (int64_t r0 = 0; r0 < b; r0 += rb) {
      const int64_t n = (b - r0 < rb) ? (b - r0) : rb;
      // Rows are numbered through valids when there is one (absolute rows of e: only the list moves on); without
      // one the block is the rows [r0, r0 + n) of e, and everything indexed by row moves with it.
      const int64_t shift_rows = (valids == nullptr) ? r0 : 0;
      const unsigned char* e_blk = static_cast<const unsigned char*>(e) + shift_rows * stride_e * es;
      const int32_t* valids_blk = valids ? valids + r0 : nullptr;
      const float* d_out_blk = d_out_is_scalar ? d_out : d_out + shift_rows;
      const float* d_lse_blk = d_lse ? d_lse + shift_rows : nullptr;
      int st = dense_dz_launch(e_blk, c, bias, lse + r0, d_out_blk, d_out_is_scalar, d_lse_blk, valids_blk,
                               targets + shift_rows, dz, ldz, 0, 1, n_rows - shift_rows, n, v, d, stride_e, stride_cv,
                               stride_cd, grad_scale, shift, target_offset, softcap, dtype, stream);
      if (st != CCE_OK) return st;
      p.e = reinterpret_cast<const uint16_t*>(e_blk);
      p.valids = valids_blk;
      if (pair_de) p.de_hi = static_cast<uint16_t*>(d_e) + shift_rows * stride_e;
      p.dc_first = (r0 == 0) ? 1 : 0;
      p.dc_accumulate = (r0 == 0) ? 0 : 1;  // an fp32 d_c (or its slots) is written by the first block and added to by the others
      set_items(n, v);
      st = products(n, v, d_bias);
      if (st != CCE_OK) return st;
      if (de_cut) sum_slots(de_slots, p.de_splits, n, valids_blk, static_cast<uint16_t*>(d_e) + shift_rows * stride_e, stride_e, 0, 0);
    }
  } else {
    for (int64_t v0 = 0; v0 < v; v0 += vc) {
      const int64_t n = (v - v0 < vc) ? (v - v0) : vc;
      const unsigned char* c_chunk = static_cast<const unsigned char*>(c) + v0 * stride_cv * es;
      const void* bias_chunk = bias ? static_cast<const unsigned char*>(bias) + v0 * es : nullptr;
      int st = dense_dz_launch(e, c_chunk, bias_chunk, lse, d_out, d_out_is_scalar, d_lse, valids, targets, dz, ldz, 0, 1,
                               n_rows, b, n, d, stride_e, stride_cv, stride_cd, grad_scale, shift, target_offset + v0,
                               softcap, dtype, stream);
      if (st != CCE_OK) return st;
      p.c = reinterpret_cast<const uint16_t*>(c_chunk);
      p.first_chunk = (v0 == 0) ? 1 : 0;
      p.de_init = (de_cut && v0 == 0) ? 1 : 0;  // (the caller's fp32 d_e is added to from the start)
      p.d_c = nullptr;
      if (d_c != nullptr)
        p.d_c = dc_cut ? static_cast<void*>(dc_slots) : static_cast<unsigned char*>(d_c) + v0 * stride_cv * (d_c_is_fp32 ? 4 : 2);
      set_items(b, n);
      st = products(b, n, d_bias != nullptr ? d_bias + v0 : nullptr);
      if (st != CCE_OK) return st;
      if (dc_cut)
        sum_slots(dc_slots, p.dc_splits, n, nullptr, static_cast<unsigned char*>(d_c) + v0 * stride_cv * (d_c_is_fp32 ? 4 : 2), stride_cv,
                  d_c_is_fp32, 0);
    }
  }

  if (de_cut && !by_rows) sum_slots(de_slots, de_nslots, b, valids, d_e, stride_e, d_e_is_fp32, 1);
  if (dc_cut && by_rows) sum_slots(dc_slots, dc_nslots, v, nullptr, d_c, stride_cv, d_c_is_fp32, 0);
  return status_from_hip(hipGetLastError());
}

// ---- the two products of one chunk on their own ----------------------------------------------------------------
extern "C" int cce_backward_products(const void* dz, int64_t ldz, const void* c, int64_t stride_cv,
                                     const void* e, int64_t stride_e, const int32_t* valids,
                                     float* d_e, int64_t ld_de, float* d_c, int64_t ld_dc, int d_c_accumulate,
                                     int64_t b, int64_t n_cls, int64_t d, int dtype, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (b < 0 || n_cls < 0 || d <= 0) return CCE_ERR_INVALID_ARGUMENT;
  if (b == 0 || n_cls == 0) return CCE_OK;
  if (dz == nullptr || (d_e != nullptr && c == nullptr) || (d_c != nullptr && e == nullptr)) return CCE_ERR_INVALID_ARGUMENT;
  if (dtype != CCE_DTYPE_BF16 && dtype != CCE_DTYPE_F16) return CCE_ERR_UNSUPPORTED_DTYPE;
  if (b >= (int64_t(1) << 31) - 512 || n_cls >= (int64_t(1) << 31) - 512 || d > (1 << 24)) return CCE_ERR_INVALID_ARGUMENT;
  if (ldz >= (int64_t(1) << 30) || stride_cv >= (int64_t(1) << 30) || stride_e >= (int64_t(1) << 30))
    return CCE_ERR_INVALID_ARGUMENT;
  if (d_e == nullptr && d_c == nullptr) return CCE_OK;
  // The tiles of dE reach their 256 rows of dz by 32-bit offsets.  Wider rows than that allows go block by block.
  if (d_e != nullptr && ldz > 0 && std::min<int64_t>(b, 256) * ldz * 2 >= (int64_t(1) << 32)) {
    const int64_t most = ((int64_t(1) << 32) - 1) / (2 * ldz);
    for (int64_t i = 0; i < b; i += most) {
      const int st = cce_backward_products(static_cast<const uint16_t*>(dz) + i * ldz, ldz, c, stride_cv,
                                           (e == nullptr || valids != nullptr) ? e : static_cast<const uint16_t*>(e) + i * stride_e,
                                           stride_e, valids == nullptr ? nullptr : valids + i, d_e + i * ld_de, ld_de, d_c, ld_dc,
                                           (d_c_accumulate || i > 0) ? 1 : 0, std::min(most, b - i), n_cls, d, dtype, stream_);
      if (st != CCE_OK) return st;
    }
    return CCE_OK;
  }
  if (!aligned16(dz) || ldz % 8 != 0 || ldz < (n_cls + 63) / 64 * 64 || d % 8 != 0) return CCE_ERR_MISALIGNED;
  if (d_e != nullptr && (!aligned16(c) || stride_cv % 8 != 0 || !aligned16(d_e) || ld_de % 4 != 0 || ld_de < d))
    return CCE_ERR_MISALIGNED;
  if (d_c != nullptr && (!aligned16(e) || stride_e % 8 != 0 || !aligned16(d_c) || ld_dc % 4 != 0 || ld_dc < d))
    return CCE_ERR_MISALIGNED;

  ProductParams p = {};
  p.dz = static_cast<const uint16_t*>(dz);
  p.ldz = ldz;
  p.c = static_cast<const uint16_t*>(c);
  p.stride_cv = stride_cv;
  p.e = static_cast<const uint16_t*>(e);
  p.stride_e = stride_e;
  p.valids = valids;
  p.de_f32 = d_e;
  p.de_hi = nullptr;
  p.de_lo = nullptr;
  p.ld_de = ld_de;
  p.de_rows_by_number = 1;
  p.de_init = 0;
  p.de_splits = p.dc_splits = 1;
  p.de_len = static_cast<int>((n_cls + 63) / 64 * 64);
  p.dc_len = static_cast<int>((b + 63) / 64 * 64);
  p.de_slot = p.dc_slot = 0;
  p.first_chunk = 0;
  p.d_c = d_c;
  p.ld_dc = ld_dc;
  p.dc_fp32 = 1;
  p.dc_accumulate = d_c_accumulate;
  p.dc_lo = nullptr;
  p.dc_first = 1;
  p.b = b;
  p.d = static_cast<int>(d);
  p.n_cls = static_cast<int>(n_cls);
  p.tiles_n = static_cast<int>((d + 255) / 256);
  p.dc_tiles = (d_c != nullptr) ? static_cast<int>((n_cls + 255) / 256) * p.tiles_n : 0;
  p.de_tiles = (d_e != nullptr) ? static_cast<int>((b + 255) / 256) * p.tiles_n : 0;
  p.dc_per_xcd = (p.dc_tiles + 7) / 8;
  p.de_per_xcd = (p.de_tiles + 7) / 8;
  p.de_first = (n_cls > b) ? 1 : 0;
  const int blocks = (p.dc_per_xcd + p.de_per_xcd) * 8;
  const int lds = Tile8<BF16, true>::LDS_BYTES;
  hipError_t err;
  if (dtype == CCE_DTYPE_BF16) {
    auto kern = dense_products_kernel<BF16, false>;
    static LdsLimitOnce lds_limit;
        err = lds_limit.set(kern, lds);
    if (err != hipSuccess) return status_from_hip(err);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kProdThreads), lds, stream, p);
  } else {
    auto kern = dense_products_kernel<F16, false>;
    static LdsLimitOnce lds_limit;
        err = lds_limit.set(kern, lds);
    if (err != hipSuccess) return status_from_hip(err);
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(kProdThreads), lds, stream, p);
  }
  return status_from_hip(hipGetLastError());
}
