// Shared pieces of the bf16 / fp16 GEMM kernels: arguments, MFMA wrappers, the
// tile walk, LDS swizzles and the epilogue stores.
#pragma once
#include <algorithm>
#include <cmath>
#include "lz_common.h"

struct GemmArgs {
  const uint16_t* A;
  const uint16_t* B;
  void* C;
  const uint16_t* R;
  int64_t lda, ldb, ldc, ldr;
  int64_t M, N, K;
  float alpha, beta;
  int c_f32;      // output dtype fp32 (else the operands' 16-bit format)
  int vec_store;  // N, ldc, ldr multiples of 4 and pointers aligned
  int vec16;      // C rows (and R rows) start 16-byte aligned: row-contiguous 16-byte epilogue
  int r16;        // R rows 16-byte aligned too: the residual joins the 16-byte bf16 epilogue
  int64_t kper;   // K range of one split (multiple of 64); blockIdx.y is the split
  int64_t slab;   // elements between the fp32 partial slabs of consecutive splits
};

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// One 32x32x16 MFMA of the operand format F (FmtBF16 or FmtF16).  Fragments
// travel as bf16x8_t whatever the format: they are 16 raw bytes per lane.
template <typename F>
__device__ __forceinline__ f32x16_t mfma16(const bf16x8_t& a, const bf16x8_t& b, const f32x16_t& c) {
  if constexpr (F::kDtype == LZ_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// One 16x16x32 MFMA of the operand format F.  The direct-to-LDS kernels use
// this shape: on MI355X a stream of independent 16x16x32 MFMAs (128
// accumulator registers per wave, two waves per SIMD, as in these kernels)
// runs at about 2.39 GHz and 2.46 PFLOP/s, the same work as 32x32x16 MFMAs at
// about 2.14 GHz and 2.19 PFLOP/s: the same issue efficiency per clock, a
// higher clock under the power limit.  At the 256x256 tile, under sustained
// load, the forward product went from 1.23 to 1.31 PFLOP/s (O projection)
// and from 1.30 to 1.37 (gate|up); the gradient layouts, whose transposed
// LDS reads (ds_read_b64_tr_b16, about 150 bytes per clock per CU against
// about 220 for ds_read_b128) keep them near the LDS bound, by 1-2 %.
template <typename F>
__device__ __forceinline__ f32x4_t mfma_k32(const bf16x8_t& a, const bf16x8_t& b, const f32x4_t& c) {
  if constexpr (F::kDtype == LZ_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Accumulator fragments of an MI x MI MFMA tile (MI = 32: 32x32x16, 16 floats
// per lane; MI = 16: 16x16x32, 4 floats per lane).  The products are computed
// as D = B_tile . A_tile^T, so every lane holds groups of 4 consecutive output
// columns of one output row: group g (floats 4g..4g+3) of fragment (i, j) is
// row acc_row(i), columns acc_col(j, g) .. +3 of the wave's tile.
template <int MI>
struct Acc;
template <>
struct Acc<32> {
  typedef f32x16_t T;
  static constexpr int kGroups = 4;
};
template <>
struct Acc<16> {
  typedef f32x4_t T;
  static constexpr int kGroups = 1;
};
template <int MI>
__device__ __forceinline__ int acc_row(int i, int lane) {
  return i * MI + (lane & (MI - 1));
}
template <int MI>
__device__ __forceinline__ int acc_col(int j, int g, int lane) {
  return MI == 32 ? j * 32 + 8 * g + 4 * (lane >> 5) : j * 16 + 4 * (lane >> 4);
}

constexpr int kBK = 64;                 // K elements per stage
constexpr int kRowBytes = kBK * 2 + 16; // padded LDS row (144 B)

// Elementwise sum of two 8-value 16-bit pieces, rounded once.
template <typename F>
__device__ __forceinline__ uint4 add16x8(const uint4& a, const uint4& b) {
  const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
  uint32_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    o[k] = F::pack2(F::to_f(aw[k] & 0xffff) + F::to_f(bw[k] & 0xffff), F::to_f(aw[k] >> 16) + F::to_f(bw[k] >> 16));
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// A 16-bit output with a residual is rounded twice, as the reference's
// separate ops are (the nn.Linear output in bf16, then x + y in bf16,
// model/llama.py:158-159): the product is rounded to the format before R is
// added and the sum is rounded on the store.  fp32 outputs add R unrounded.
template <typename F>
__device__ __forceinline__ float with_residual(float v, uint32_t r16) { return F::round(v) + F::to_f(r16 & 0xffff); }

template <typename F>
__device__ __forceinline__ void store_out4(const GemmArgs& g, int64_t m, int64_t n, const float (&v)[4]) {
  float o[4] = {v[0] * g.alpha, v[1] * g.alpha, v[2] * g.alpha, v[3] * g.alpha};
  if (g.vec_store && n + 3 < g.N) {
    if (g.c_f32) {
      float4* cp = reinterpret_cast<float4*>(static_cast<float*>(g.C) + m * g.ldc + n);
      if (g.beta != 0.f) {
        float4 c = *cp;
        o[0] = fmaf(g.beta, c.x, o[0]); o[1] = fmaf(g.beta, c.y, o[1]);
        o[2] = fmaf(g.beta, c.z, o[2]); o[3] = fmaf(g.beta, c.w, o[3]);
      }
      if (g.R) {
        uint2 r = *reinterpret_cast<const uint2*>(g.R + m * g.ldr + n);
        o[0] += F::to_f(r.x & 0xffff); o[1] += F::to_f(r.x >> 16); o[2] += F::to_f(r.y & 0xffff); o[3] += F::to_f(r.y >> 16);
      }
      *cp = make_float4(o[0], o[1], o[2], o[3]);
    } else {
      uint2* cp = reinterpret_cast<uint2*>(static_cast<uint16_t*>(g.C) + m * g.ldc + n);
      if (g.beta != 0.f) {
        uint2 c = *cp;
        o[0] = fmaf(g.beta, F::to_f(c.x & 0xffff), o[0]); o[1] = fmaf(g.beta, F::to_f(c.x >> 16), o[1]);
        o[2] = fmaf(g.beta, F::to_f(c.y & 0xffff), o[2]); o[3] = fmaf(g.beta, F::to_f(c.y >> 16), o[3]);
      }
      if (g.R) {
        uint2 r = *reinterpret_cast<const uint2*>(g.R + m * g.ldr + n);
        o[0] = with_residual<F>(o[0], r.x & 0xffff); o[1] = with_residual<F>(o[1], r.x >> 16);
        o[2] = with_residual<F>(o[2], r.y & 0xffff); o[3] = with_residual<F>(o[3], r.y >> 16);
      }
      uint2 w;
      w.x = (uint32_t)F::from_f(o[0]) | ((uint32_t)F::from_f(o[1]) << 16);
      w.y = (uint32_t)F::from_f(o[2]) | ((uint32_t)F::from_f(o[3]) << 16);
      *cp = w;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t nn = n + e;
    if (nn >= g.N) break;
    float val = o[e];
    if (g.c_f32) {
      float* cp = static_cast<float*>(g.C) + m * g.ldc + nn;
      if (g.beta != 0.f) val = fmaf(g.beta, *cp, val);
      if (g.R) val += F::to_f(g.R[m * g.ldr + nn]);
      *cp = val;
    } else {
      uint16_t* cp = static_cast<uint16_t*>(g.C) + m * g.ldc + nn;
      if (g.beta != 0.f) val = fmaf(g.beta, F::to_f(*cp), val);
      if (g.R) val = with_residual<F>(val, g.R[m * g.ldr + nn]);
      *cp = F::from_f(val);
    }
  }
}

// Maps the linear workgroup id to a (tile_m, tile_n) pair.  Hardware places
// workgroup i on XCD i % 8; the remap gives each XCD a contiguous range of
// logical tiles, and the logical order walks groups of kGroupM M-tiles across
// all N-tiles so an XCD's concurrently running tiles share A rows and B rows.
__device__ __forceinline__ void tile_coords(int64_t pid, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
  constexpr int kXcd = 8, kGroupM = 4;
  const int64_t nblk = tiles_m * tiles_n;
  if (nblk % kXcd == 0) pid = (pid % kXcd) * (nblk / kXcd) + pid / kXcd;
  const int64_t per_group = (int64_t)kGroupM * tiles_n;
  const int64_t group = pid / per_group;
  const int64_t first_m = group * kGroupM;
  const int64_t gsize = min((int64_t)kGroupM, tiles_m - first_m);
  const int64_t in_group = pid - group * per_group;
  tm = first_m + in_group % gsize;
  tn = in_group / gsize;
}

// Chunk swizzle of a staged epilogue row of kRow bytes: rows that share a
// 256-byte bank window are told apart by the XOR, so 16 lanes writing one
// chunk of 16 consecutive rows (or reading 16 chunks of a row) hit 16
// distinct 16-byte bank groups.
template <int kRow>
__device__ __forceinline__ int epi_swz(int row) {
  constexpr int kPer256 = kRow >= 256 ? 1 : 256 / kRow;
  constexpr int kMask = (kRow / 16 - 1) < 15 ? (kRow / 16 - 1) : 15;
  return (row / kPer256) & kMask;
}

// Staged epilogue rows of kRow bytes: a power-of-two number of 16-byte chunks
// is XOR-swizzled in place (epi_swz); other widths (the 48-wide wave tiles of
// 192-wide tiles: 6 bf16 or 12 fp32 chunks) are padded by one chunk instead,
// an odd pitch in chunks that staggers consecutive rows over the bank groups.
template <int kRow>
constexpr bool epi_pow2() {
  return ((kRow / 16) & (kRow / 16 - 1)) == 0;
}
template <int kRow>
constexpr int epi_pitch() {
  return epi_pow2<kRow>() ? kRow : kRow + 16;
}
template <int kRow>
__device__ __forceinline__ int epi_off(int row, int chunk) {
  if constexpr (epi_pow2<kRow>()) return row * kRow + ((chunk ^ epi_swz<kRow>(row)) << 4);
  else return row * epi_pitch<kRow>() + (chunk << 4);
}
// LDS bytes one wave's region of store_tile16 takes: TM bf16 rows or TM/2 fp32
// rows of TN values.
template <int TM, int TN>
constexpr int epi_wave_bytes() {
  return TM * epi_pitch<TN * 2>() > (TM / 2) * epi_pitch<TN * 4>() ? TM * epi_pitch<TN * 2>()
                                                                    : (TM / 2) * epi_pitch<TN * 4>();
}

// Interior tiles, 16-byte path: each wave parks its TM x TN sub-tile in a
// private LDS region (rows of TN values, 16-byte chunks XOR-swizzled so that
// both the accumulator-layout writes and the row-wise reads are free of bank
// conflicts), then writes whole 16-byte pieces of consecutive row bytes, so a
// store instruction covers full cache lines.  fp32 output goes in two passes
// of TM/2 rows.  Needs WM*WN*epi_wave_bytes<TM, TN>() bytes of LDS (BM*BN*2
// for power-of-two wave tile widths).
// Parks a wave's TM x TN accumulator tile in its LDS region as 16-bit values
// (scaled by alpha, rounded once): rows of TN values (kRow = 2*TN bytes),
// 16-byte chunks XOR-swizzled by epi_swz, so that the accumulator-layout
// writes and the row-wise reads are free of bank conflicts.
template <typename F, int MI, int FM, int FN, int kRow>
__device__ __forceinline__ void park16(const typename Acc<MI>::T (&acc)[FM][FN], char* st, int lane, float alpha) {
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < Acc<MI>::kGroups; ++q) {
        const int row = acc_row<MI>(i, lane), byte = 2 * acc_col<MI>(j, q, lane);
        *reinterpret_cast<uint2*>(st + epi_off<kRow>(row, byte >> 4) + (byte & 15)) =
            make_uint2(F::pack2(acc[i][j][4 * q] * alpha, acc[i][j][4 * q + 1] * alpha),
                       F::pack2(acc[i][j][4 * q + 2] * alpha, acc[i][j][4 * q + 3] * alpha));
      }
}

template <typename F, int MI, int BM, int BN, int WM, int WN>
__device__ __forceinline__ void store_tile16(const GemmArgs& go, typename Acc<MI>::T (&acc)[BM / WM / MI][BN / WN / MI],
                                             int64_t m0, int64_t n0, char* smem, int lane, int wave) {
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / MI, FN = TN / MI;
  static_assert(FM % 2 == 0, "fp32 output is staged in two halves");
  const int wm = wave / WN, wn = wave % WN;
  const int64_t mrow0 = m0 + wm * TM, ncol0 = n0 + wn * TN;
  char* st = smem + wave * epi_wave_bytes<TM, TN>();
  if (!go.c_f32) {
    constexpr int kRow = TN * 2, kChunks = kRow / 16;  // bytes and 16-byte chunks per row
    static_assert(kChunks >= 4 && kChunks <= 64, "bf16 rows of 32 to 512 values");
    // beta == 0: stage bf16 values (the product rounded once) and store whole
    // 16-byte row pieces; a residual is added to each piece on the way out
    const bool plain = go.beta == 0.f && (go.R == nullptr || go.r16);
    if (plain) {
      park16<F, MI, FM, FN, kRow>(acc, st, lane, go.alpha);
      asm volatile("" ::: "memory");
      constexpr int kIters = TM * kChunks / 64;
      if (go.R == nullptr) {
        // 64 lanes x 16 bytes per store: whole rows (or 64-chunk row pieces)
#pragma unroll
        for (int t = 0; t < kIters; ++t) {
          const int idx = t * 64 + lane, row = idx / kChunks, chunk = idx % kChunks;
          const uint4 v = *reinterpret_cast<const uint4*>(st + epi_off<kRow>(row, chunk));
          st_nt16(static_cast<uint16_t*>(go.C) + (mrow0 + row) * go.ldc + ncol0 + chunk * 8, v);
        }
        return;
      }
      // with the residual: the R pieces of 8 stores are loaded together (R may
      // alias the output, so the compiler would not hoist them past the stores)
      constexpr int kBlk = kIters < 8 ? kIters : kIters % 8 == 0 ? 8 : kIters % 6 == 0 ? 6 : 4;
      static_assert(kIters % kBlk == 0, "store blocks must tile the wave's rows");
#pragma unroll
      for (int t0 = 0; t0 < kIters; t0 += kBlk) {
        uint4 rv[kBlk];
#pragma unroll
        for (int u = 0; u < kBlk; ++u) {
          const int idx = (t0 + u) * 64 + lane, row = idx / kChunks, chunk = idx % kChunks;
          rv[u] = *reinterpret_cast<const uint4*>(go.R + (mrow0 + row) * go.ldr + ncol0 + chunk * 8);
        }
#pragma unroll
        for (int u = 0; u < kBlk; ++u) {
          const int idx = (t0 + u) * 64 + lane, row = idx / kChunks, chunk = idx % kChunks;
          const uint4 v = *reinterpret_cast<const uint4*>(st + epi_off<kRow>(row, chunk));
          st_nt16(static_cast<uint16_t*>(go.C) + (mrow0 + row) * go.ldc + ncol0 + chunk * 8, add16x8<F>(v, rv[u]));
        }
      }
      return;
    }
  }
  // fp32 values staged (fp32 output, or bf16 output with beta / residual,
  // which are applied before the single rounding): two passes of TM/2 rows.
  // The stores go in blocks of kBlk: each block first issues all of its loads
  // of C (beta) and R, so that they are in flight together instead of one
  // load-use round trip per store (C and R may alias the output, so the
  // compiler cannot hoist them past the stores itself).
  constexpr int kRow = TN * 4, kChunks = kRow / 16;
  constexpr int kIters = (TM / 2) * kChunks / 64, kBlk = kIters < 4 ? kIters : 4;
  static_assert(kChunks >= 4 && kChunks <= 64, "fp32 rows of 16 to 256 values");
  static_assert(kIters % kBlk == 0, "store blocks must tile a pass");
  const bool has_c = go.beta != 0.f, has_r = go.R != nullptr;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int ii = 0; ii < FM / 2; ++ii) {
      const int i = p * (FM / 2) + ii;
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int q = 0; q < Acc<MI>::kGroups; ++q) {
          const int row = acc_row<MI>(ii, lane), chunk = acc_col<MI>(j, q, lane) >> 2;
          *reinterpret_cast<float4*>(st + epi_off<kRow>(row, chunk)) =
              make_float4(acc[i][j][4 * q] * go.alpha, acc[i][j][4 * q + 1] * go.alpha,
                          acc[i][j][4 * q + 2] * go.alpha, acc[i][j][4 * q + 3] * go.alpha);
        }
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t0 = 0; t0 < kIters; t0 += kBlk) {
      uint4 cpre[kBlk];  // beta's C: fp32 x4, or bf16 x4 in .x/.y
      uint2 rpre[kBlk];  // residual, bf16 x4
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        const int idx = (t0 + u) * 64 + lane, row = idx / kChunks, chunk = idx % kChunks;
        const int64_t m = mrow0 + p * (TM / 2) + row, n = ncol0 + chunk * 4;
        cpre[u] = make_uint4(0u, 0u, 0u, 0u);
        rpre[u] = make_uint2(0u, 0u);
        if (has_c) {
          if (go.c_f32) {
            cpre[u] = *reinterpret_cast<const uint4*>(static_cast<const float*>(go.C) + m * go.ldc + n);
          } else {
            const uint2 c = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(go.C) + m * go.ldc + n);
            cpre[u].x = c.x;
            cpre[u].y = c.y;
          }
        }
        if (has_r) rpre[u] = *reinterpret_cast<const uint2*>(go.R + m * go.ldr + n);
      }
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        const int idx = (t0 + u) * 64 + lane, row = idx / kChunks, chunk = idx % kChunks;
        const uint4 v = *reinterpret_cast<const uint4*>(st + epi_off<kRow>(row, chunk));
        const int64_t m = mrow0 + p * (TM / 2) + row, n = ncol0 + chunk * 4;
        float o[4] = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
        if (has_c) {
          const uint4 c = cpre[u];
          if (go.c_f32) {
            o[0] = fmaf(go.beta, __uint_as_float(c.x), o[0]); o[1] = fmaf(go.beta, __uint_as_float(c.y), o[1]);
            o[2] = fmaf(go.beta, __uint_as_float(c.z), o[2]); o[3] = fmaf(go.beta, __uint_as_float(c.w), o[3]);
          } else {
            o[0] = fmaf(go.beta, F::to_f(c.x & 0xffff), o[0]); o[1] = fmaf(go.beta, F::to_f(c.x >> 16), o[1]);
            o[2] = fmaf(go.beta, F::to_f(c.y & 0xffff), o[2]); o[3] = fmaf(go.beta, F::to_f(c.y >> 16), o[3]);
          }
        }
        if (has_r) {
          const uint2 r = rpre[u];
          if (go.c_f32) {
            o[0] += F::to_f(r.x & 0xffff); o[1] += F::to_f(r.x >> 16); o[2] += F::to_f(r.y & 0xffff); o[3] += F::to_f(r.y >> 16);
          } else {
            o[0] = with_residual<F>(o[0], r.x & 0xffff); o[1] = with_residual<F>(o[1], r.x >> 16);
            o[2] = with_residual<F>(o[2], r.y & 0xffff); o[3] = with_residual<F>(o[3], r.y >> 16);
          }
        }
        if (go.c_f32) {
          st_nt16(static_cast<float*>(go.C) + m * go.ldc + n, make_uint4(
              __float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])));
        } else {
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(go.C) + m * go.ldc + n) =
              make_uint2(F::pack2(o[0], o[1]), F::pack2(o[2], o[3]));
        }
      }
    }
    asm volatile("" ::: "memory");
  }
}

// Writes a workgroup's BM x BN accumulator tile (layout: Acc<MI>).
// Interior tiles with 16-byte aligned rows and wave tiles up to 64 wide take
// store_tile16; other interior tiles store each lane's 4-column groups
// straight from the accumulators (8 or 16 bytes) with the row address formed
// once per fragment row band; edge tiles go through LDS one MI-row band at a
// time and are written as whole rows with bounds checks, so the accumulators
// are never indexed dynamically.  `smem` must be free and at least
// max(WM*WN*MI*(BN/WN+4)*4, BM*BN*2) bytes.
template <typename F, int MI, int BM, int BN, int WM, int WN>
__device__ __forceinline__ void store_tile(const GemmArgs& go, typename Acc<MI>::T (&acc)[BM / WM / MI][BN / WN / MI],
                                           int64_t m0, int64_t n0, char* smem, int lane, int wave) {
  constexpr int TM = BM / WM, TN = BN / WN, FM = TM / MI, FN = TN / MI, G = Acc<MI>::kGroups;
  const int wm = wave / WN, wn = wave % WN;
  if constexpr (TN <= 64) {  // (wider wave tiles run out of registers in the staged path)
    if (m0 + BM <= go.M && n0 + BN <= go.N && go.vec16) {
      store_tile16<F, MI, BM, BN, WM, WN>(go, acc, m0, n0, smem, lane, wave);
      return;
    }
  }
  if (m0 + BM <= go.M && n0 + BN <= go.N && go.vec_store) {
    const int64_t ncol0 = n0 + wn * TN;
    if (go.c_f32) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int64_t m = m0 + wm * TM + acc_row<MI>(i, lane);
        float* crow = static_cast<float*>(go.C) + m * go.ldc + ncol0;
        const uint16_t* rrow = go.R ? go.R + m * go.ldr + ncol0 : nullptr;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q) {
            const int c = acc_col<MI>(j, q, lane);
            float4 o = make_float4(acc[i][j][4 * q] * go.alpha, acc[i][j][4 * q + 1] * go.alpha,
                                   acc[i][j][4 * q + 2] * go.alpha, acc[i][j][4 * q + 3] * go.alpha);
            float4* cp = reinterpret_cast<float4*>(crow + c);
            if (go.beta != 0.f) {
              const float4 cv = *cp;
              o.x = fmaf(go.beta, cv.x, o.x); o.y = fmaf(go.beta, cv.y, o.y);
              o.z = fmaf(go.beta, cv.z, o.z); o.w = fmaf(go.beta, cv.w, o.w);
            }
            if (rrow) {
              const uint2 r = *reinterpret_cast<const uint2*>(rrow + c);
              o.x += F::to_f(r.x & 0xffff); o.y += F::to_f(r.x >> 16); o.z += F::to_f(r.y & 0xffff); o.w += F::to_f(r.y >> 16);
            }
            *cp = o;
          }
      }
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int64_t m = m0 + wm * TM + acc_row<MI>(i, lane);
        uint16_t* crow = static_cast<uint16_t*>(go.C) + m * go.ldc + ncol0;
        const uint16_t* rrow = go.R ? go.R + m * go.ldr + ncol0 : nullptr;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int q = 0; q < G; ++q) {
            const int c = acc_col<MI>(j, q, lane);
            float o[4] = {acc[i][j][4 * q] * go.alpha, acc[i][j][4 * q + 1] * go.alpha,
                          acc[i][j][4 * q + 2] * go.alpha, acc[i][j][4 * q + 3] * go.alpha};
            uint2* cp = reinterpret_cast<uint2*>(crow + c);
            if (go.beta != 0.f) {
              const uint2 cv = *cp;
              o[0] = fmaf(go.beta, F::to_f(cv.x & 0xffff), o[0]); o[1] = fmaf(go.beta, F::to_f(cv.x >> 16), o[1]);
              o[2] = fmaf(go.beta, F::to_f(cv.y & 0xffff), o[2]); o[3] = fmaf(go.beta, F::to_f(cv.y >> 16), o[3]);
            }
            if (rrow) {
              const uint2 r = *reinterpret_cast<const uint2*>(rrow + c);
              o[0] = with_residual<F>(o[0], r.x & 0xffff); o[1] = with_residual<F>(o[1], r.x >> 16);
              o[2] = with_residual<F>(o[2], r.y & 0xffff); o[3] = with_residual<F>(o[3], r.y >> 16);
            }
            *cp = make_uint2(F::pack2(o[0], o[1]), F::pack2(o[2], o[3]));
          }
      }
    }
    return;
  }
  constexpr int kPitch = TN + 4;  // floats; 16-byte aligned, staggers the banks of consecutive rows
  float* stage = reinterpret_cast<float*>(smem) + wave * MI * kPitch;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < G; ++q)
        *reinterpret_cast<float4*>(stage + acc_row<MI>(0, lane) * kPitch + acc_col<MI>(j, q, lane)) =
            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    __syncthreads();
    const int64_t mband = m0 + wm * TM + i * MI, nband = n0 + wn * TN;
    for (int it = lane; it < MI * (TN / 4); it += 64) {
      const int r = it / (TN / 4), c4 = it % (TN / 4);
      const int64_t m = mband + r, n = nband + c4 * 4;
      if (m < go.M && n < go.N) {
        const float4 v4 = *reinterpret_cast<const float4*>(stage + r * kPitch + c4 * 4);
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
        store_out4<F>(go, m, n, v);
      }
    }
    __syncthreads();
  }
}

// LDS row swizzle: chunk c (8 K values) of row r sits in slot c ^ swz(r).
// For 4-chunk (64-byte) and 8-chunk (128-byte) rows this keeps the 16-byte
// reads of 8 or 16 consecutive rows on distinct banks.
template <int kChunks>
__device__ __forceinline__ int swz(int r) {
  if constexpr (kChunks == 4) return ((r >> 1) ^ (r >> 3)) & 3;
  else return ((r >> 1) ^ ((r & 1) << 2)) & 7;
}

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t* lds_v4i16_ptr;

}  // namespace
