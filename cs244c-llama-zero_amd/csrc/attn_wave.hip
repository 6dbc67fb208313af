// Attention on wave-private tiles: any sequence length, an explicit mask,
// attention dropout, head dims 32, 64 and 128, 16-bit or fp32 operands
// (reference: model/llama.py:72-133, as attn.hip).
//
// One workgroup owns 32 queries of a head (forward, dQ) or 32 keys of a kv
// head (dK/dV).  Its NW waves take every NW-th 32-row tile of the other side,
// each through LDS regions of its own (the next tile's rows wait in registers
// meanwhile), so the main loop has no workgroup barrier; the waves' partial
// results meet in LDS once, in a fixed order.  The calls that come here are
// bounded by latency, not by a unit: the 64- and 128-query tile kernels of
// attn.hip leave most of the chip idle on them and a one-wave-per-row kernel
// spends a wave reduction on each score.  Splitting the reduction over the
// waves gives NW times the workgroups' parallelism and 1/NW of the serial
// chain.
//
// Both operand policies share one data flow.  The accumulator of a 32x32 MFMA
// tile has lane = owned column (query, or key in dK/dV) and register r = row
// 8*(r/4) + 4*(lane/32) + r%4 of the other side's tile, and that layout is
// the B operand of the second product as it stands: rows() forms tile . own^T
// and cols() adds tile^T . P.
// Measured against the kernels these calls had before (us, forward + dQ + dK/dV
// device time, before -> after): heads 10/2 of 32, B 2, S 512: bf16 604 -> 38,
// fp32 627 -> 82; heads 12/4 of 64, B 4, S 500, bool mask, bf16 6246 -> 110;
// forward of heads 16/8 of 128, B 1, S 777, bf16 59 (and a transposed copy of
// V, 11) -> 19.  The exact weights and the second pass that non-finite sums ask
// for are 5 and 11 us of the two bf16 forward + backward figures.
//
//   PolF32: fp32 MFMAs (v_mfma_f32_32x32x2_f32) on fp32 tiles; fp32 and fp16
//     operands.  Every value after the load is fp32.
//   PolBF16: bf16 MFMAs on bf16 tiles.  The fp32 weights (probabilities, dS)
//     enter cols() as three bf16 terms that add up to them exactly (kSplit: 24
//     bits in pieces of eight, three MFMAs) or rounded to bf16 once, as the tile
//     kernels of attn.hip do.
// kExact policies keep fp32 values fp32 from the score to the last product:
// natural units and exp_accurate, no rounded weights.  In their products a row
// that an owned one does not see has weight 0, and 0 * inf is NaN (as is a
// zero term of a split weight times a visible inf), so a wave whose sums are
// not finite goes over its tiles again with cols_seen(), which leaves unseen
// rows out; finite inputs never do.
#include "attn_wave.h"

#include <type_traits>

#include "attn_tiles.h"

namespace {

// LDS written by this wave's lanes is read by its other lanes (and rewritten
// after such reads): LDS instructions of one wave execute in order, so only
// the compiler has to keep theirs.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// exp(d) for d <= 0 to about 1 ulp: 2^hi * (1 + lo ln 2) with hi + lo =
// d * log2(e) formed in two terms.  Below -150 (where the result is zero) d is
// replaced, so that -inf does not meet inf - inf in lo; a NaN stays one.
__device__ __forceinline__ float exp_accurate(float d) {
  d = d < -150.f ? -150.f : d;
  const float hi = d * kLog2e;
  const float lo = fmaf(d, kLog2e, -hi) + d * 1.9259629911266175e-8f;  // log2(e) - float(log2(e))
  const float p = __builtin_amdgcn_exp2f(hi);
  return fmaf(p * kLn2, lo, p);
}

// fp32 tiles: rows of HD + 4 floats (16 consecutive rows' 16-byte reads fall
// on distinct banks).
template <typename T, int HD_>
struct PolF32 {
  static constexpr int HD = HD_;
  static constexpr bool kExact = true, k16 = false;  // k16: 16-bit tiles
  static constexpr int RS = HD + 4, kTile = 32 * RS * 4;
  static constexpr int kPieces = HD / 8;  // 4-element pieces of a tile per lane
  typedef T Ptr;
  static constexpr bool kWide = sizeof(T) == 4;

  struct Own {
    float x[HD / 2];  // columns 8c + 4*half + e at [4c + e]
  };
  struct Stage {
    uint4 p[kWide ? kPieces : kPieces / 2];  // fp16: two pieces per uint4
  };

  static __device__ __forceinline__ float4 widen(uint2 w) {
    return make_float4(h2f(w.x & 0xffff), h2f(w.x >> 16), h2f(w.y & 0xffff), h2f(w.y >> 16));
  }
  static __device__ __forceinline__ void load_own(Own& f, const void* row, int half) {
#pragma unroll
    for (int c = 0; c < HD / 8; ++c) {
      float4 v;
      if constexpr (kWide) v = *reinterpret_cast<const float4*>(static_cast<const float*>(row) + 8 * c + 4 * half);
      else v = widen(*reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(row) + 8 * c + 4 * half));
      f.x[4 * c] = v.x;
      f.x[4 * c + 1] = v.y;
      f.x[4 * c + 2] = v.z;
      f.x[4 * c + 3] = v.w;
    }
  }
  static __device__ __forceinline__ float dot(const Own& a, const Own& b) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < HD / 2; ++i) s = fmaf(a.x[i], b.x[i], s);
    return s;
  }
  // rows row0 .. row0+31 of `base` (its row 0 = position 0), rows past S
  // re-reading row S-1
  static __device__ __forceinline__ void load(Stage& st, const void* base, int64_t ld, int row0, int S, int lane) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int p = lane + 64 * i;
      const int r = min(row0 + p / (HD / 4), S - 1), col = 4 * (p % (HD / 4));
      if constexpr (kWide) {
        st.p[i] = *reinterpret_cast<const uint4*>(static_cast<const float*>(base) + r * ld + col);
      } else {
        const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + r * ld + col);
        if (i % 2 == 0) {
          st.p[i / 2].x = w.x;
          st.p[i / 2].y = w.y;
        } else {
          st.p[i / 2].z = w.x;
          st.p[i / 2].w = w.y;
        }
      }
    }
  }
  // the staged rows into LDS; rows past S as zeros
  static __device__ __forceinline__ void store(const Stage& st, char* tile, int row0, int S, int lane) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int p = lane + 64 * i;
      const int r = p / (HD / 4), col = 4 * (p % (HD / 4));
      float4 v;
      if constexpr (kWide) v = __builtin_bit_cast(float4, st.p[i]);
      else v = widen(i % 2 == 0 ? make_uint2(st.p[i / 2].x, st.p[i / 2].y) : make_uint2(st.p[i / 2].z, st.p[i / 2].w));
      if (row0 + r >= S) v = make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<float4*>(tile + (r * RS + col) * 4) = v;
    }
  }
  static __device__ __forceinline__ float elem(const char* tile, int r, int c) {
    return *reinterpret_cast<const float*>(tile + (r * RS + c) * 4);
  }
  struct Ctx {
    int row, col;  // byte offsets of this lane's rows() and cols() reads
    __device__ __forceinline__ void init(int lane) {
      const int half = lane >> 5, l32 = lane & 31;
      row = (l32 * RS + 4 * half) * 4;
      col = (4 * half * RS + l32) * 4;
    }
  };
  static __device__ __forceinline__ void rows(const Ctx& cx, f32x16_t& s, const char* tile, const Own& own) {
#pragma unroll
    for (int c = 0; c < HD / 8; ++c) {
      const float4 a = *reinterpret_cast<const float4*>(tile + cx.row + c * 32);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, own.x[4 * c], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, own.x[4 * c + 1], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, own.x[4 * c + 2], s, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, own.x[4 * c + 3], s, 0, 0, 0);
    }
  }
  static __device__ __forceinline__ void cols(const Ctx& cx, f32x16_t (&acc)[HD / 32], const char* tile,
                                              const f32x16_t& p) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int i = 0; i < HD / 32; ++i) {
        const float a = *reinterpret_cast<const float*>(tile + cx.col + ((8 * (r >> 2) + (r & 3)) * RS + 32 * i) * 4);
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, p[r], acc[i], 0, 0, 0);
      }
  }
  static __device__ __forceinline__ void store4(void* row, int c, float a, float b, float d, float e) {
    if constexpr (kWide) *reinterpret_cast<float4*>(static_cast<float*>(row) + c) = make_float4(a, b, d, e);
    else store_bf16x4<FmtF16>(static_cast<uint16_t*>(row) + c, a, b, d, e);
  }
};

// 16 bytes from an 8-byte aligned address (the global loads of dout rows; one
// instruction either way).
typedef uint32_t u32x4a8_t __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ uint4 load16(const uint16_t* p) {
  const u32x4a8_t v = *reinterpret_cast<const u32x4a8_t*>(p);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

template <int HD_, bool kSplit>
struct PolBF16 {
  static constexpr int HD = HD_;
  static constexpr bool kExact = kSplit, k16 = true;
  static constexpr int kTile = 32 * HD * 2;
  static constexpr int kPieces = HD / 16;  // 8-element pieces of a tile per lane
  static constexpr int kTerms = kSplit ? 3 : 1;
  typedef uint16_t Ptr;

  struct Own {
    bf16x8_t x[HD / 16];  // columns 16kk + 8*half ..
  };
  struct Stage {
    uint4 p[kPieces];
  };
  static __device__ __forceinline__ void load_own(Own& f, const void* row, int half) {
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk)
      f.x[kk] = __builtin_bit_cast(bf16x8_t, load16(static_cast<const uint16_t*>(row) + 16 * kk + 8 * half));
  }
  static __device__ __forceinline__ float dot(const Own& a, const Own& b) {
    float s = 0.f;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      const uint4 x = __builtin_bit_cast(uint4, a.x[kk]), y = __builtin_bit_cast(uint4, b.x[kk]);
      const uint32_t xw[4] = {x.x, x.y, x.z, x.w}, yw[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = fmaf(bf2f(xw[e] & 0xffff), bf2f(yw[e] & 0xffff), s);
        s = fmaf(bf2f(xw[e] >> 16), bf2f(yw[e] >> 16), s);
      }
    }
    return s;
  }
  static __device__ __forceinline__ void load(Stage& st, const void* base, int64_t ld, int row0, int S, int lane) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int p = lane + 64 * i;
      const int r = min(row0 + p / (HD / 8), S - 1);
      st.p[i] = load16(static_cast<const uint16_t*>(base) + r * ld + 8 * (p % (HD / 8)));
    }
  }
  static __device__ __forceinline__ void store(const Stage& st, char* tile, int row0, int S, int lane) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int p = lane + 64 * i;
      const int r = p / (HD / 8);
      *reinterpret_cast<uint4*>(tile + toff<HD>(r, p % (HD / 8))) = row0 + r < S ? st.p[i] : make_uint4(0, 0, 0, 0);
    }
  }
  static __device__ __forceinline__ float elem(const char* tile, int r, int c) {
    return bf2f(*reinterpret_cast<const uint16_t*>(tile + toff<HD>(r, c >> 3) + (c & 7) * 2));
  }
  struct Ctx {
    TileOffsets<HD> to;
    __device__ __forceinline__ void init(int lane) { to.init(lane); }
  };
  static __device__ __forceinline__ void rows(const Ctx& cx, f32x16_t& s, const char* tile, const Own& own) {
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) s = mfma16<FmtBF16>(cx.to.frag(tile, 0, kk), own.x[kk], s);
  }
  static __device__ __forceinline__ void cols(const Ctx& cx, f32x16_t (&acc)[HD / 32], const char* tile,
                                              const f32x16_t& p) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      uint32_t w[kTerms][4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float p0 = p[8 * ks + 2 * e], p1 = p[8 * ks + 2 * e + 1];
        if constexpr (kSplit) {
          // the top eight significant bits of what is left, cut and not
          // rounded: each remainder is exact and the third has at most eight
#pragma unroll
          for (int t = 0; t < kTerms; ++t) {
            const uint32_t b0 = __float_as_uint(p0), b1 = __float_as_uint(p1);
            w[t][e] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
            p0 -= __uint_as_float(b0 & 0xffff0000u);
            p1 -= __uint_as_float(b1 & 0xffff0000u);
          }
        } else {
          w[0][e] = pack_bf16x2(p0, p1);
        }
      }
#pragma unroll
      for (int i = 0; i < HD / 32; ++i) {
        const bf16x8_t f = cx.to.frag_t(tile, ks, i);
#pragma unroll
        for (int t = kTerms - 1; t >= 0; --t)  // the smallest first
          acc[i] = mfma16<FmtBF16>(f, __builtin_bit_cast(bf16x8_t, make_uint4(w[t][0], w[t][1], w[t][2], w[t][3])), acc[i]);
      }
    }
  }
  static __device__ __forceinline__ void store4(void* row, int c, float a, float b, float d, float e) {
    store_bf16x4<FmtBF16>(static_cast<uint16_t*>(row) + c, a, b, d, e);
  }
};

// Units of the running maximum and of exp: natural for the exact policies (a
// mask of the type's lowest value would overflow in log2 units too), log2 for
// rounded causal bf16.
template <class P>
__device__ __forceinline__ float score_unit(float scale) {
  return P::kExact ? scale : scale * kLog2e;
}
template <class P>
__device__ __forceinline__ float exp_unit(float d) {
  if constexpr (P::kExact) return exp_accurate(d);
  else return __builtin_amdgcn_exp2f(d);
}

__device__ __forceinline__ float mask_elem(const LzWaveArgs& a, int64_t i) {
  if (a.mask_kind == 1) return static_cast<const uint8_t*>(a.mask)[i] ? 0.f : -INFINITY;
  if (a.mask_kind == 2) return static_cast<const float*>(a.mask)[i];
  if (a.mask_kind == 3) return bf2f(static_cast<const uint16_t*>(a.mask)[i]);
  return h2f(static_cast<const uint16_t*>(a.mask)[i]);
}

// Mask terms (0 / -inf for a bool mask) of one query against this lane's 16
// keys kv0 + 8*(r/4) + 4*half + r%4; keys past S are -inf.  Four adjacent
// keys come in one load when the mask's last dimension is dense.
__device__ __forceinline__ void mask_of_query(const LzWaveArgs& a, float (&mb)[16], int64_t off, int kv0, int half) {
  if (a.msk == 1 && kv0 + 32 <= a.S) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const int64_t i = off + kv0 + 8 * r4 + 4 * half;
      if (a.mask_kind == 1) {
        uint32_t w;
        __builtin_memcpy(&w, static_cast<const uint8_t*>(a.mask) + i, 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) mb[4 * r4 + e] = ((w >> (8 * e)) & 0xff) ? 0.f : -INFINITY;
      } else if (a.mask_kind == 2) {
        float w[4];
        __builtin_memcpy(w, static_cast<const float*>(a.mask) + i, 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) mb[4 * r4 + e] = w[e];
      } else {
        uint16_t w[4];
        __builtin_memcpy(w, static_cast<const uint16_t*>(a.mask) + i, 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) mb[4 * r4 + e] = a.mask_kind == 3 ? bf2f(w[e]) : h2f(w[e]);
      }
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int kv = kv0 + 8 * (r >> 2) + 4 * half + (r & 3);
    const float m = mask_elem(a, off + min(kv, a.S - 1) * a.msk);
    mb[r] = kv < a.S ? m : -INFINITY;
  }
}

// The mask terms of one key against this lane's 16 queries; rows past S are
// not read (the caller drops them).
__device__ __forceinline__ void mask_of_key(const LzWaveArgs& a, float (&mb)[16], int64_t off, int q0, int half) {
#pragma unroll
  for (int r = 0; r < 16; ++r)
    mb[r] = mask_elem(a, off + min(q0 + 8 * (r >> 2) + 4 * half + (r & 3), a.S - 1) * a.msq);
}

__device__ __forceinline__ float drop_of(const LzWaveArgs& a, int b, int h, int s, int kv) {
  const uint64_t i = (((uint64_t)b * a.H + h) * a.S + s) * a.S + kv;
  return lz_keep(a.drop_seed, i, a.drop_thresh) ? a.drop_scale : 0.0f;
}

__device__ __forceinline__ bool all_lanes_masked(const float (&mb)[16]) {
  float mx = mb[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) mx = fmaxf(mx, mb[r]);
  return __ballot(mx > -INFINITY) == 0;
}

template <class P>
__device__ __forceinline__ const void* row_ptr(const void* p, int64_t row, int64_t ld, int64_t col) {
  return static_cast<const typename P::Ptr*>(p) + row * ld + col;
}
template <class P>
__device__ __forceinline__ void* row_ptr_w(void* p, int64_t row, int64_t ld, int64_t col) {
  return static_cast<typename P::Ptr*>(p) + row * ld + col;
}

template <int N>
__device__ __forceinline__ void zero_acc(f32x16_t (&acc)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
}

// A tile straight into LDS (the second pass stages nothing ahead, so that it
// does not raise the kernel's registers).
template <class P>
__device__ __forceinline__ void copy_tile(const void* base, int64_t ld, char* tile, int row0, int S, int lane) {
  typename P::Stage st;
  P::load(st, base, ld, row0, S, lane);
  P::store(st, tile, row0, S, lane);
}

template <int N>
__device__ __forceinline__ bool all_finite(const f32x16_t (&acc)[N]) {
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(acc[i][r], 0.f, z);
  return __ballot(!(z == 0.f)) == 0;
}

// P::cols() one row of the tile at a time with fp32 multiply-adds, without the
// rows r of `hidden` (bit r: this lane's owned row does not see register r's).
template <class P>
__device__ __forceinline__ void cols_seen(f32x16_t (&acc)[P::HD / 32], const char* tile, const f32x16_t& w,
                                          uint32_t hidden, int lane) {
  const int l32 = lane & 31, half = lane >> 5;
#pragma unroll 1
  for (int row = 0; row < 32; ++row) {
    const int r = 4 * (row >> 3) + (row & 3), from = l32 + 8 * (row & 4);  // the lane whose register r is this row
    float x = w[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) x = e == r ? w[e] : x;
    x = __shfl(x, from, 64);
    const bool skip = (__shfl((int)hidden, from, 64) >> r) & 1;
#pragma unroll
    for (int i = 0; i < P::HD / 32; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float y = fmaf(x, P::elem(tile, row, 32 * i + 8 * (e >> 2) + 4 * half + (e & 3)), acc[i][e]);
        acc[i][e] = skip ? acc[i][e] : y;
        if (e % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // few reads in flight: few registers
      }
  }
}

// This wave's accumulators into its LDS region as [register][lane].
template <int N>
__device__ __forceinline__ void park_acc(char* region, const f32x16_t (&acc)[N], int lane) {
  float* f = reinterpret_cast<float*>(region) + lane;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) f[(16 * i + r) * 64] = acc[i][r];
}

// Sums the waves' parked accumulators (fixed order) and stores the row this
// lane owns: each wave takes every NW-th group of four adjacent columns.
template <class P, int NW>
__device__ __forceinline__ void sum_and_store(const char* smem, int stride, void* row, bool valid, float scale,
                                              int wave, int lane) {
  for (int g = wave; g < P::HD / 8; g += NW) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* f = reinterpret_cast<const float*>(smem + w * stride) + (4 * g) * 64 + lane;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += f[e * 64];
    }
    const int c = 32 * (g >> 2) + 8 * (g & 3) + 4 * (lane >> 5);
    if (valid) P::store4(row, c, v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
  }
}

template <class P, int NW, bool kGen>
__global__ void __launch_bounds__(64 * NW) attn_fwd_wave_kernel(LzWaveArgs a) {
  constexpr int HD = P::HD;
  constexpr int kRegion = 2 * P::kTile > HD * 128 ? 2 * P::kTile : HD * 128;
  __shared__ __attribute__((aligned(1024))) char smem[NW * kRegion];
  __shared__ float ml[NW][64];  // a query's running maximum (0..31) and sum (32..63) per wave

  const int S = a.S, H = a.H, nqt = (S + 31) / 32;
  int qb, b, h;
  query_block_coords(blockIdx.x, nqt, a.B, H, a.KV, qb, b, h);
  const int g = h / (H / a.KV);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int qrow = qb * 32 + l32, qc = min(qrow, S - 1);
  char* const Kt = smem + wave * kRegion;
  char* const Vt = Kt + P::kTile;
  typename P::Ctx cx;
  cx.init(lane);
  typename P::Own qf;
  P::load_own(qf, row_ptr<P>(a.q, (int64_t)b * S + qc, a.ldq, (int64_t)h * HD), half);
  const void* kbase = row_ptr<P>(a.k, (int64_t)b * S, a.ldk, (int64_t)g * HD);
  const void* vbase = row_ptr<P>(a.v, (int64_t)b * S, a.ldv, (int64_t)g * HD);
  const bool masked = kGen && a.mask_kind != 0;
  const int nt = masked ? nqt : qb + 1;
  const float u = score_unit<P>(a.scale);
  const int64_t moff = (int64_t)b * a.msb + (int64_t)h * a.msh + (int64_t)qc * a.msq;

  f32x16_t o[HD / 32];
  float m, l;
  auto pass = [&](auto seen_only) {
    zero_acc(o);
    m = -INFINITY;
    l = 0.f;
    typename P::Stage ks, vs;
    if (!seen_only && wave < nt) {
      P::load(ks, kbase, a.ldk, wave * 32, S, lane);
      P::load(vs, vbase, a.ldv, wave * 32, S, lane);
    }
    for (int t = wave; t < nt; t += NW) {
      const int kv0 = t * 32;
      if constexpr (seen_only) {
        copy_tile<P>(kbase, a.ldk, Kt, kv0, S, lane);
        copy_tile<P>(vbase, a.ldv, Vt, kv0, S, lane);
      } else {
        P::store(ks, Kt, kv0, S, lane);
        P::store(vs, Vt, kv0, S, lane);
      }
      wave_order();
      if (!seen_only && t + NW < nt) {
        P::load(ks, kbase, a.ldk, kv0 + 32 * NW, S, lane);
        P::load(vs, vbase, a.ldv, kv0 + 32 * NW, S, lane);
      }
      float mb[16];
      if constexpr (kGen) {
        if (masked) {
          mask_of_query(a, mb, moff, kv0, half);
          if (a.mask_kind == 1 && all_lanes_masked(mb)) continue;  // no query of this wave sees these keys
        }
      }
      f32x16_t s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
      P::rows(cx, s, Kt, qf);
      if (masked) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = mb[r] == -INFINITY ? -INFINITY : fmaf(s[r], u, mb[r]);
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] *= u;
        if (t == qb) {  // the diagonal tile (and the last one: keys past S lie past every query)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kv0 + 8 * (r >> 2) + 4 * half + (r & 3) > qrow) s[r] = -INFINITY;
        }
      }
      uint32_t hidden = 0;
      if constexpr (seen_only) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          hidden |= (masked ? s[r] == -INFINITY : kv0 + 8 * (r >> 2) + 4 * half + (r & 3) > qrow) ? 1u << r : 0u;
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx = max_halves(mx);
      const float m_new = fmaxf(m, mx);
      const float ms = m_new == -INFINITY ? 0.f : m_new;  // nothing seen yet: every term below is exp(-inf)
      const float alpha = exp_unit<P>(m - ms);
      m = m_new;
      float rs = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = exp_unit<P>(s[r] - ms);
        rs += s[r];
      }
      l = l * alpha + sum_halves(rs);
      if constexpr (kGen) {
        if (a.drop_thresh) {  // the normaliser sums the probabilities before dropout
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] *= drop_of(a, b, h, qc, kv0 + 8 * (r >> 2) + 4 * half + (r & 3));
        }
      }
#pragma unroll
      for (int i = 0; i < HD / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
      if constexpr (seen_only) cols_seen<P>(o, Vt, s, hidden, lane);
      else P::cols(cx, o, Vt, s);
      wave_order();  // the next tile's stores stay behind these reads
    }
  };
  pass(std::false_type{});
  if constexpr (P::kExact) {
    if (!all_finite(o)) pass(std::true_type{});
  }
  wave_order();
  park_acc(Kt, o, lane);
  if (half == 0) {
    ml[wave][l32] = m;
    ml[wave][l32 + 32] = l;
  }
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[w][l32]);
  const float Ms = M == -INFINITY ? 0.f : M;
  float f[NW], L = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    f[w] = exp_unit<P>(ml[w][l32] - Ms);
    L = fmaf(f[w], ml[w][l32 + 32], L);
  }
  const float inv = 1.f / L;  // a row with every key masked: 0 * inf = NaN
  for (int gq = wave; gq < HD / 8; gq += NW) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* p = reinterpret_cast<const float*>(smem + w * kRegion) + (4 * gq) * 64 + lane;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(f[w], p[e * 64], v[e]);
    }
    if (qrow < S)
      P::store4(row_ptr_w<P>(a.o, (int64_t)b * S + qrow, a.ldo, (int64_t)h * HD), 32 * (gq >> 2) + 8 * (gq & 3) + 4 * half,
                v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
  }
  if (wave == 0 && half == 0 && qrow < S) {
    float lse;
    if constexpr (P::kExact) lse = M + logf(L);
    else lse = (M + log2f(L)) * kLn2;
    a.lse[((int64_t)b * H + h) * S + qrow] = lse;
  }
}

template <class P, int NW, bool kGen>
__global__ void __launch_bounds__(64 * NW) attn_dq_wave_kernel(LzWaveArgs a) {
  constexpr int HD = P::HD;
  constexpr int kRegion = 2 * P::kTile > HD * 128 ? 2 * P::kTile : HD * 128;
  __shared__ __attribute__((aligned(1024))) char smem[NW * kRegion];

  const int S = a.S, H = a.H, nqt = (S + 31) / 32;
  int qb, b, h;
  query_block_coords(blockIdx.x, nqt, a.B, H, a.KV, qb, b, h);
  const int g = h / (H / a.KV);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int qrow = qb * 32 + l32, qc = min(qrow, S - 1);
  char* const Kt = smem + wave * kRegion;
  char* const Vt = Kt + P::kTile;
  typename P::Ctx cx;
  cx.init(lane);
  const int64_t grow = (int64_t)b * S + qc, li = ((int64_t)b * H + h) * S + qc;
  typename P::Own qf, df;
  P::load_own(qf, row_ptr<P>(a.q, grow, a.ldq, (int64_t)h * HD), half);
  P::load_own(df, row_ptr<P>(a.dout, grow, a.lddo, (int64_t)h * HD), half);
  float D;
  if (a.delta_w) {
    typename P::Own of;
    P::load_own(of, row_ptr<P>(a.o, grow, a.ldo, (int64_t)h * HD), half);
    D = sum_halves(P::dot(of, df));
    if (wave == 0 && half == 0 && qrow < S) a.delta_w[li] = D;
  } else {
    D = a.delta[li];
  }
  const float lse = a.lse[li];
  const float lu = P::kExact ? lse : lse * kLog2e;
  const void* kbase = row_ptr<P>(a.k, (int64_t)b * S, a.ldk, (int64_t)g * HD);
  const void* vbase = row_ptr<P>(a.v, (int64_t)b * S, a.ldv, (int64_t)g * HD);
  const bool masked = kGen && a.mask_kind != 0;
  const int nt = masked ? nqt : qb + 1;
  const float u = score_unit<P>(a.scale);
  const int64_t moff = (int64_t)b * a.msb + (int64_t)h * a.msh + (int64_t)qc * a.msq;
  // a query whose keys are all masked (lse -inf) has NaN gradients: its tiles are never skipped
  const bool may_skip = __ballot(lse == -INFINITY) == 0;

  f32x16_t dq[HD / 32];
  auto pass = [&](auto seen_only) {
    zero_acc(dq);
    typename P::Stage ks, vs;
    if (!seen_only && wave < nt) {
      P::load(ks, kbase, a.ldk, wave * 32, S, lane);
      P::load(vs, vbase, a.ldv, wave * 32, S, lane);
    }
    for (int t = wave; t < nt; t += NW) {
      const int kv0 = t * 32;
      if constexpr (seen_only) {
        copy_tile<P>(kbase, a.ldk, Kt, kv0, S, lane);
        copy_tile<P>(vbase, a.ldv, Vt, kv0, S, lane);
      } else {
        P::store(ks, Kt, kv0, S, lane);
        P::store(vs, Vt, kv0, S, lane);
      }
      wave_order();
      if (!seen_only && t + NW < nt) {
        P::load(ks, kbase, a.ldk, kv0 + 32 * NW, S, lane);
        P::load(vs, vbase, a.ldv, kv0 + 32 * NW, S, lane);
      }
      float mb[16];
      if constexpr (kGen) {
        if (masked) {
          mask_of_query(a, mb, moff, kv0, half);
          if (a.mask_kind == 1 && may_skip && all_lanes_masked(mb)) continue;
        }
      }
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = 0.f;
        dp[r] = 0.f;
      }
      P::rows(cx, s, Kt, qf);
      P::rows(cx, dp, Vt, df);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kv = kv0 + 8 * (r >> 2) + 4 * half + (r & 3);
        float x = s[r] * u;
        if (masked) x = mb[r] == -INFINITY ? -INFINITY : x + mb[r];
        const float p = exp_unit<P>(x - lu);
        float z = 1.f;
        if constexpr (kGen) {
          if (a.drop_thresh) z = drop_of(a, b, h, qc, kv);
        }
        dp[r] = p * (fmaf(z, dp[r], -D));
      }
      if (masked ? kv0 + 32 > S : t == qb) {
        const int last = masked ? S - 1 : qrow;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kv0 + 8 * (r >> 2) + 4 * half + (r & 3) > last) dp[r] = 0.f;
      }
      if constexpr (seen_only) {
        uint32_t hidden = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kv = kv0 + 8 * (r >> 2) + 4 * half + (r & 3);
          hidden |= (masked ? kv >= S || (mb[r] == -INFINITY && lse != -INFINITY) : kv > qrow) ? 1u << r : 0u;
        }
        cols_seen<P>(dq, Kt, dp, hidden, lane);
      } else {
        P::cols(cx, dq, Kt, dp);
      }
      wave_order();
    }
  };
  pass(std::false_type{});
  if constexpr (P::kExact) {
    if (!all_finite(dq)) pass(std::true_type{});
  }
  wave_order();
  park_acc(Kt, dq, lane);
  __syncthreads();
  sum_and_store<P, NW>(smem, kRegion, row_ptr_w<P>(a.dq, grow, a.lddq, (int64_t)h * HD), qrow < S, a.scale, wave, lane);
}

template <class P, int NW, bool kGen>
__global__ void __launch_bounds__(64 * NW) attn_dkdv_wave_kernel(LzWaveArgs a) {
  constexpr int HD = P::HD;
  constexpr int kRegion = 2 * P::kTile > HD * 128 ? 2 * P::kTile : HD * 128;
  __shared__ __attribute__((aligned(1024))) char smem[NW * kRegion];
  __shared__ __attribute__((aligned(16))) float rows_s[NW][64];  // a tile's lse (0..31) and delta (32..63)

  const int S = a.S, H = a.H, nqt = (S + 31) / 32, rep = H / a.KV;
  int kb, b, g;
  key_block_coords(blockIdx.x, a.B, a.KV, kb, b, g);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int kvrow = kb * 32 + l32, kvc = min(kvrow, S - 1);
  char* const Qt = smem + wave * kRegion;
  char* const Dt = Qt + P::kTile;
  typename P::Ctx cx;
  cx.init(lane);
  const int64_t grow = (int64_t)b * S + kvc;
  typename P::Own kf, vf;
  P::load_own(kf, row_ptr<P>(a.k, grow, a.ldk, (int64_t)g * HD), half);
  P::load_own(vf, row_ptr<P>(a.v, grow, a.ldv, (int64_t)g * HD), half);
  const bool masked = kGen && a.mask_kind != 0;
  const int first = masked ? 0 : kb, per = nqt - first, items = rep * per;
  const float u = score_unit<P>(a.scale);

  f32x16_t dk[HD / 32], dv[HD / 32];
  auto pass = [&](auto seen_only) {
    zero_acc(dk);
    zero_acc(dv);
    typename P::Stage qs, ds;
    float row_val = 0.f;
    auto row_value = [&](int h, int q0) {
      const int64_t li = ((int64_t)b * H + h) * S + min(q0 + l32, S - 1);
      return half == 0 ? a.lse[li] : a.delta[li];
    };
    auto fetch = [&](int it) {
      const int hq = it / per, q0 = (first + it - hq * per) * 32, h = g * rep + hq;
      P::load(qs, row_ptr<P>(a.q, (int64_t)b * S, a.ldq, (int64_t)h * HD), a.ldq, q0, S, lane);
      P::load(ds, row_ptr<P>(a.dout, (int64_t)b * S, a.lddo, (int64_t)h * HD), a.lddo, q0, S, lane);
      row_val = row_value(h, q0);
    };
    if (!seen_only && wave < items) fetch(wave);
    for (int it = wave; it < items; it += NW) {
      const int hq = it / per, qt = first + it - hq * per, q0 = qt * 32, h = g * rep + hq;
      if constexpr (seen_only) {
        copy_tile<P>(row_ptr<P>(a.q, (int64_t)b * S, a.ldq, (int64_t)h * HD), a.ldq, Qt, q0, S, lane);
        copy_tile<P>(row_ptr<P>(a.dout, (int64_t)b * S, a.lddo, (int64_t)h * HD), a.lddo, Dt, q0, S, lane);
        row_val = row_value(h, q0);
      } else {
        P::store(qs, Qt, q0, S, lane);
        P::store(ds, Dt, q0, S, lane);
      }
      rows_s[wave][lane] = row_val;
      const bool finite_rows = __ballot(half == 0 && row_val == -INFINITY) == 0;
      wave_order();
      if (!seen_only && it + NW < items) fetch(it + NW);
      float mb[16];
      if constexpr (kGen) {
        if (masked) {
          mask_of_key(a, mb, (int64_t)b * a.msb + (int64_t)h * a.msh + (int64_t)kvc * a.msk, q0, half);
          if (a.mask_kind == 1 && finite_rows && all_lanes_masked(mb)) continue;
        }
      }
      f32x16_t s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = 0.f;
        dp[r] = 0.f;
      }
      P::rows(cx, s, Qt, kf);
      P::rows(cx, dp, Dt, vf);
      f32x16_t pz;
      uint32_t hidden = 0;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const float4 l4 = *reinterpret_cast<const float4*>(&rows_s[wave][8 * r4 + 4 * half]);
        const float4 d4 = *reinterpret_cast<const float4*>(&rows_s[wave][32 + 8 * r4 + 4 * half]);
        const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dl[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * r4 + e;
          float x = s[r] * u;
          if (masked) x = mb[r] == -INFINITY ? -INFINITY : x + mb[r];
          const float p = exp_unit<P>(x - (P::kExact ? lv[e] : lv[e] * kLog2e));
          float z = 1.f;
          if constexpr (kGen) {
            if (a.drop_thresh) z = drop_of(a, b, h, q0 + 8 * r4 + 4 * half + e, kvc);
          }
          pz[r] = p * z;
          dp[r] = p * fmaf(z, dp[r], -dl[e]);
          if constexpr (seen_only) {
            const int qr = q0 + 8 * r4 + 4 * half + e;
            hidden |= (qr >= S || (masked ? mb[r] == -INFINITY && lv[e] != -INFINITY : qr < kvrow)) ? 1u << r : 0u;
          }
        }
      }
      if (q0 + 32 > S || (!masked && qt == kb)) {
        // queries past S, and (causal) the diagonal tile's queries before the key
        const int from = masked ? 0 : kvrow;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int qr = q0 + 8 * (r >> 2) + 4 * half + (r & 3);
          if (qr >= S || qr < from) {
            pz[r] = 0.f;
            dp[r] = 0.f;
          }
        }
      }
      if constexpr (seen_only) {
        cols_seen<P>(dv, Dt, pz, hidden, lane);
        cols_seen<P>(dk, Qt, dp, hidden, lane);
      } else {
        P::cols(cx, dv, Dt, pz);
        P::cols(cx, dk, Qt, dp);
      }
      wave_order();
    }
  };
  pass(std::false_type{});
  if constexpr (P::kExact) {
    if (!all_finite(dk) || !all_finite(dv)) pass(std::true_type{});
  }
  wave_order();
  const bool valid = kvrow < S;
  park_acc(Qt, dv, lane);
  __syncthreads();
  sum_and_store<P, NW>(smem, kRegion, row_ptr_w<P>(a.dv, grow, a.lddv, (int64_t)g * HD), valid, 1.0f, wave, lane);
  __syncthreads();
  park_acc(Qt, dk, lane);
  __syncthreads();
  sum_and_store<P, NW>(smem, kRegion, row_ptr_w<P>(a.dk, grow, a.lddk, (int64_t)g * HD), valid, a.scale, wave, lane);
}

// Waves per workgroup: eight (two per SIMD) for heads of 32 and 16-bit heads of
// 64, four where the LDS regions or the accumulators take more.  The general
// bf16 dK/dV kernel for heads of 64 spills 34 of its registers at eight waves
// and none at four, and is faster with eight: 12/4 heads, B 4, S 500, bool mask
// 49.6 against 69.1 us.  The general dK/dV kernels for heads of 128 spill at four
// (bf16 31, fp16 86, fp32 156 registers).
template <class P>
constexpr int waves_of() {
  return P::HD == 32 || (P::HD == 64 && P::k16) ? 8 : 4;
}

template <class P, bool kGen>
int launch_fwd(const LzWaveArgs& a, hipStream_t s) {
  constexpr int NW = waves_of<P>();
  const unsigned grid = (unsigned)((int64_t)a.B * a.H * ((a.S + 31) / 32));
  attn_fwd_wave_kernel<P, NW, kGen><<<grid, 64 * NW, 0, s>>>(a);
  return lz_check_launch("attention forward");
}

template <class P, bool kGen>
int launch_dq(const LzWaveArgs& a, hipStream_t s) {
  constexpr int NW = waves_of<P>();
  const unsigned grid = (unsigned)((int64_t)a.B * a.H * ((a.S + 31) / 32));
  attn_dq_wave_kernel<P, NW, kGen><<<grid, 64 * NW, 0, s>>>(a);
  return lz_check_launch("attention backward");
}

template <class P, bool kGen>
int launch_dkdv(const LzWaveArgs& a, hipStream_t s) {
  constexpr int NW = waves_of<P>();
  const unsigned grid = (unsigned)((int64_t)a.B * a.KV * ((a.S + 31) / 32));
  attn_dkdv_wave_kernel<P, NW, kGen><<<grid, 64 * NW, 0, s>>>(a);
  return lz_check_launch("attention backward");
}

template <class P, bool kGen>
int launch(const LzWaveArgs& a, LzWavePass pass, hipStream_t s) {
  if (pass == kWaveFwd) return launch_fwd<P, kGen>(a, s);
  return pass == kWaveDq ? launch_dq<P, kGen>(a, s) : launch_dkdv<P, kGen>(a, s);
}

}  // namespace

bool lz_attn_wave_ok(const LzWaveArgs& a, int dtype, int64_t hd, bool backward, bool dout8) {
  if (hd != 32 && hd != 64 && hd != 128) return false;
  if (dtype != LZ_BF16 && dtype != LZ_F16 && dtype != LZ_F32) return false;
  if ((int64_t)a.B * a.H * ((a.S + 31) / 32) >= (1ll << 31)) return false;
  // the rows are read in pieces of 8 (16-bit) or 4 (fp32) elements and
  // written four elements at a time
  const int64_t rd = dtype == LZ_F32 ? 4 : 8;
  const uintptr_t wr = dtype == LZ_F32 ? 15 : 7;
  auto reads = [&](const void* p, int64_t ld) { return lz_aligned16(p) && ld % rd == 0; };
  auto writes = [&](const void* p, int64_t ld) { return (reinterpret_cast<uintptr_t>(p) & wr) == 0 && ld % 4 == 0; };
  if (!reads(a.q, a.ldq) || !reads(a.k, a.ldk) || !reads(a.v, a.ldv)) return false;
  if (!backward) return writes(a.o, a.ldo);
  const bool dout_ok = reads(a.dout, a.lddo) ||
                       (dout8 && dtype != LZ_F32 && (reinterpret_cast<uintptr_t>(a.dout) & 7) == 0 && a.lddo % 4 == 0);
  return dout_ok && (a.delta_w == nullptr || reads(a.o, a.ldo)) && writes(a.dq, a.lddq) &&
         writes(a.dk, a.lddk) && writes(a.dv, a.lddv);
}

int lz_attn_wave_pass(const LzWaveArgs& a, int dtype, int64_t hd, LzWaveMode mode, LzWavePass pass, hipStream_t s) {
  const bool gen = mode == kWaveGeneral, split = mode == kWaveSplit;
  // (heads of 32 are never rounded: no tile kernel takes them)
#define LZ_WAVE(HD)                                                                              \
  (dtype == LZ_BF16 ? (gen                  ? launch<PolBF16<HD, true>, true>(a, pass, s)    \
                       : split || HD == 32 ? launch<PolBF16<HD, true>, false>(a, pass, s)   \
                                            : launch<PolBF16<HD, HD == 32>, false>(a, pass, s)) \
   : dtype == LZ_F16 ? (gen ? launch<PolF32<_Float16, HD>, true>(a, pass, s)                 \
                            : launch<PolF32<_Float16, HD>, false>(a, pass, s))               \
                     : (gen ? launch<PolF32<float, HD>, true>(a, pass, s)                    \
                            : launch<PolF32<float, HD>, false>(a, pass, s)))
  if (hd == 32) return LZ_WAVE(32);
  if (hd == 64) return LZ_WAVE(64);
  return LZ_WAVE(128);
#undef LZ_WAVE
}

int lz_attn_wave_bwd(const LzWaveArgs& a, int dtype, int64_t hd, LzWaveMode mode, hipStream_t s) {
  const int rc = lz_attn_wave_pass(a, dtype, hd, mode, kWaveDq, s);
  if (rc) return rc;
  LzWaveArgs k = a;  // dQ has written the delta it was asked to form
  if (k.delta_w) k.delta = k.delta_w;
  return lz_attn_wave_pass(k, dtype, hd, mode, kWaveDkdv, s);
}
