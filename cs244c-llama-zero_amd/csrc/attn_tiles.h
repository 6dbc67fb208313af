// Shared pieces of the attention kernels: block orders, 16-bit MFMA operands,
// and the swizzled LDS tiles that are read as rows or transposed.
#pragma once
#include "lz_common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Workgroup -> (query block, batch, head), heaviest query blocks first.  The
// hardware deals workgroup i to XCD i % 8; when the (batch, kv head) pairs
// split evenly over the 8 XCDs, each XCD gets its own pairs, and all query
// heads of a pair's group and neighbouring query blocks run on that XCD at
// about the same time, so the K and V rows they stream are fetched into its
// L2 once instead of by workgroups spread over every XCD.
__device__ __forceinline__ void query_block_coords(int bid, int nqb, int B, int H, int KV, int& qb, int& b, int& h) {
  const int rep = H / KV, npairs = B * KV;
  if (npairs % 8 == 0) {
    const int xcd = bid % 8, j = bid / 8;
    const int per_q = (npairs / 8) * rep;  // workgroups of one query block on one XCD
    const int qr = j / per_q, rem = j - qr * per_q;
    const int pair = xcd + 8 * (rem / rep);
    b = pair / KV;
    h = (pair % KV) * rep + rem % rep;
    qb = nqb - 1 - qr;
  } else {
    const int bh = B * H;
    qb = nqb - 1 - bid / bh;
    b = (bid % bh) / H;
    h = bid % H;
  }
}

// Workgroup -> (key block, batch, kv head), first key blocks (the most
// queries at or after them) first; pairs split over XCDs as above, so the Q
// and dO rows a pair's key blocks read share an L2.
__device__ __forceinline__ void key_block_coords(int bid, int B, int KV, int& kvb, int& b, int& g) {
  const int npairs = B * KV;
  int pair;
  if (npairs % 8 == 0) {
    const int xcd = bid % 8, j = bid / 8, ppx = npairs / 8;
    kvb = j / ppx;
    pair = xcd + 8 * (j - kvb * ppx);
  } else {
    kvb = bid / npairs;
    pair = bid % npairs;
  }
  b = pair / KV;
  g = pair % KV;
}

// Elements e0..e0+7 of an accumulator -> an 8-element MFMA operand of the
// 16-bit format F (fragments travel as bf16x8_t: 16 raw bytes per lane).
template <typename F = FmtBF16>
__device__ __forceinline__ bf16x8_t pack8(const f32x16_t& v, int e0) {
  const uint4 w = make_uint4(F::pack2(v[e0], v[e0 + 1]), F::pack2(v[e0 + 2], v[e0 + 3]),
                             F::pack2(v[e0 + 4], v[e0 + 5]), F::pack2(v[e0 + 6], v[e0 + 7]));
  return __builtin_bit_cast(bf16x8_t, w);
}

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// One 32x32x16 MFMA on operands of the format F.
template <typename F>
__device__ __forceinline__ f32x16_t mfma16(const bf16x8_t& a, const bf16x8_t& b, const f32x16_t& c) {
  if constexpr (F::kDtype == LZ_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// x combined with the value of lane ^ 32 (both halves get the same result):
// v_permlane32_swap exchanges the halves of two registers without an LDS
// round trip.
__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <typename F = FmtBF16>
__device__ __forceinline__ void store_bf16x4(uint16_t* p, float a, float b, float c, float d) {
  uint2 w;
  w.x = (uint32_t)F::from_f(a) | ((uint32_t)F::from_f(b) << 16);
  w.y = (uint32_t)F::from_f(c) | ((uint32_t)F::from_f(d) << 16);
  *reinterpret_cast<uint2*>(p) = w;
}

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t* lds_v4i16_ptr;

// Chunk swizzle of a tile row r: keeps the 16-byte reads of 16 consecutive
// rows (row fragments) and the 8-byte transposed reads of 4 consecutive rows
// x 64 bytes (one half-wave of ds_read_b64_tr_b16) on distinct banks of the
// 64-bank LDS.
template <int HD>
__device__ __forceinline__ int tswz(int r) {
  if constexpr (HD == 128) return ((r & 3) << 2) | ((r >> 2) & 3);
  else if constexpr (HD == 64) return (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
  else return (r >> 2) & 3;  // 64-byte rows: four rows span the banks once
}

template <int HD>
__device__ __forceinline__ int toff(int r, int chunk) {
  return r * (HD * 2) + ((chunk ^ tswz<HD>(r)) << 4);
}

// Per-lane LDS offsets of the fragment reads of a tile.  tswz() depends only
// on the row modulo 16, so every offset splits into a per-lane part and a
// part that only depends on the 16-row block and the 32-column block.
template <int HD>
struct TileOffsets {
  static constexpr int RB = HD * 2;
  int row;              // row fragments: (lane % 32) * RB
  int chunk[HD / 16];   // row fragments: ((2*kk + lane/32) ^ tswz) * 16
  int tbase[2];         // transposed reads 1 and 2 (rows +0 and +8)
  int tcol[HD / 32];    // transposed reads: 32-column block i

  __device__ __forceinline__ void init(int lane) {
    const int l32 = lane & 31, half = lane >> 5;
    row = l32 * RB;
    const int sw = tswz<HD>(l32);
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) chunk[kk] = ((2 * kk + half) ^ sw) << 4;
    // lane 4j+q of each 16-lane group points at row r0 + j (+8), columns
    // c0 + 16*(group % 2) + 4q .. +3
    const int p = lane & 15;
    const int col = ((lane >> 4) & 1) * 16 + 4 * (p & 3);
    const int cl = col >> 3;
    int swh = 0;
#pragma unroll
    for (int rd = 0; rd < 2; ++rd) {
      const int r = 4 * half + (p >> 2) + 8 * rd;  // row within a 16-row block
      const int swr = tswz<HD>(r);
      tbase[rd] = r * RB + ((cl ^ (swr & 3)) << 4) + (col & 7) * 2;
      swh = swr >> 2;  // the same for both reads
    }
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) tcol[i] = (i ^ swh) << 6;
  }

  // Row fragment: row 32*t + lane%32, columns 16*kk + 8*(lane/32) .. +7.
  __device__ __forceinline__ bf16x8_t frag(const char* tile, int t, int kk) const {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(tile + t * 32 * RB + row + chunk[kk]));
  }

  // Transposed fragment for an MFMA operand whose k index runs over tile rows:
  // lane l gets column 32*i + l%32 at rows 16*ks + 8*(e/4) + 4*(l/32) + e%4
  // for k-slots e = 0..7 (the slot order of the accumulator layout).
  __device__ __forceinline__ bf16x8_t frag_t(const char* tile, int ks, int i) const {
    const char* blk = tile + ks * 16 * RB + tcol[i];
    const v4i16_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(blk + tbase[0]));
    const v4i16_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(blk + tbase[1]));
    const uint2 xw = __builtin_bit_cast(uint2, x), yw = __builtin_bit_cast(uint2, y);
    return __builtin_bit_cast(bf16x8_t, make_uint4(xw.x, xw.y, yw.x, yw.y));
  }
};

}  // namespace
