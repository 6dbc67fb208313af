// Causal grouped-query attention, flash style, on CDNA4 matrix cores
// (reference: model/llama.py:72-133 GroupedQueryAttention.forward with
// F.scaled_dot_product_attention(is_causal=True), K/V heads shared by
// H/KV query heads through repeat_interleave).
//
// Layouts (elements):
//   q/k/v : rows b*S + s of ld elements; head h occupies [h*hd, (h+1)*hd).  The
//           three may be column ranges of one fused QKV projection.
//   o     : same row layout with H heads.
//   lse   : [B, H, S] fp32, natural-log log-sum-exp of the scaled scores.
// The kv head of query head h is h / (H/KV); K/V are never expanded.
//
// MFMA tiling (v_mfma_f32_32x32x16_bf16).  The score tile is computed as
// S^T = K . Q^T so that each lane owns one query column: row statistics need
// one cross-half shuffle, and the probabilities already sit in the B-operand
// layout for O^T += V^T . P^T (the k-slots of the two operands are the same
// permutation of the 16 keys).  The backward splits into a dK/dV pass (one
// workgroup per 128 keys of a kv head, looping over the query heads of its
// group and the query blocks at or after the diagonal) and a dQ pass (one
// workgroup per 128 queries, looping over key blocks up to the diagonal); no
// atomics, deterministic.
#include <algorithm>
#include <cmath>

#include "attn_tiles.h"
#include "attn_wave.h"

namespace {

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  int64_t ldq, ldk, ldv;
  uint16_t* o;
  int64_t ldo;
  float* lse;
  // backward
  const uint16_t* dout; // rows like o
  int64_t lddo;
  const float* delta;   // [B,H,S] rowsum(dO*O)
  float* delta_w;       // the same rows, written by the dQ kernel that computes them (with o as O)
  uint16_t* dq;
  uint16_t* dk;
  uint16_t* dv;
  int64_t lddq, lddk, lddv;
  // backward with RoPE folded in: bf16 tables [>= S, hd] (row = position);
  // dq and dk are then the gradients of the un-rotated q and k
  const uint16_t* rcos;
  const uint16_t* rsin;
  int B, S, H, KV;
  float scale;
};

// One lane's row of a dQ or dK accumulator set (columns 32*i + 8*q4 +
// 4*half + e, the MFMA output layout), times `scale`, stored as bf16 at dst.
// With RoPE tables (cs/sn: the row's position, HD values each) the stored row
// is the gradient of the un-rotated input: the gradient pair (d1, d2) of
// columns (c, c + HD/2) in the format F becomes g1 = r(r(d1*c1) + r(d2*s2)) and
// g2 = r(r(d2*c2) - r(d1*s1)), rounding each product and sum to F as the
// separate RoPE backward pass (and the reference's bf16 autograd of
// x*cos + rotate_half(x)*sin, model/llama.py:35-39) does.  Columns c and
// c + HD/2 sit in accumulator blocks i and i + HD/64 of the same lane.
template <int HD, typename F = FmtBF16>
__device__ __forceinline__ void store_grad_row(uint16_t* dst, const f32x16_t (&acc)[HD / 32], float scale, int half,
                                               const uint16_t* cs, const uint16_t* sn) {
  if (cs == nullptr) {
#pragma unroll
    for (int i = 0; i < HD / 32; ++i)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int c = i * 32 + 8 * q4 + 4 * half;
        store_bf16x4<F>(dst + c, acc[i][4 * q4] * scale, acc[i][4 * q4 + 1] * scale, acc[i][4 * q4 + 2] * scale,
                     acc[i][4 * q4 + 3] * scale);
      }
    return;
  }
  // every table value this lane needs is loaded before the first store (the
  // stores may alias the tables as far as the compiler knows, so it would
  // otherwise wait for each group's loads in turn)
  constexpr int kHalf = HD / 2, kBlk = HD / 64;
  uint2 cw[kBlk][4][2], sw[kBlk][4][2];
#pragma unroll
  for (int i = 0; i < kBlk; ++i)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int c = i * 32 + 8 * q4 + 4 * half;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        cw[i][q4][hh] = *reinterpret_cast<const uint2*>(cs + c + hh * kHalf);
        sw[i][q4][hh] = *reinterpret_cast<const uint2*>(sn + c + hh * kHalf);
      }
    }
#pragma unroll
  for (int i = 0; i < kBlk; ++i)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int c = i * 32 + 8 * q4 + 4 * half;
      const uint32_t c1a[2] = {cw[i][q4][0].x, cw[i][q4][0].y}, c2a[2] = {cw[i][q4][1].x, cw[i][q4][1].y};
      const uint32_t s1a[2] = {sw[i][q4][0].x, sw[i][q4][0].y}, s2a[2] = {sw[i][q4][1].x, sw[i][q4][1].y};
      float g1[4], g2[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sh = (e & 1) * 16;
        const float c1 = F::to_f((uint16_t)(c1a[e >> 1] >> sh)), c2 = F::to_f((uint16_t)(c2a[e >> 1] >> sh));
        const float s1 = F::to_f((uint16_t)(s1a[e >> 1] >> sh)), s2 = F::to_f((uint16_t)(s2a[e >> 1] >> sh));
        const float d1 = F::round(acc[i][4 * q4 + e] * scale), d2 = F::round(acc[i + kBlk][4 * q4 + e] * scale);
        g1[e] = __fadd_rn(F::round(__fmul_rn(d1, c1)), F::round(__fmul_rn(d2, s2)));
        g2[e] = __fadd_rn(F::round(__fmul_rn(d2, c2)), -F::round(__fmul_rn(d1, s1)));
      }
      store_bf16x4<F>(dst + c, g1[0], g1[1], g1[2], g1[3]);
      store_bf16x4<F>(dst + c + kHalf, g2[0], g2[1], g2[2], g2[3]);
    }
}

// ---------------------------------------------------------------------------
// Tile path.  Every operand tile is a [64][HD] bf16 block
// of a row-major source (Q, dO, K or V rows), copied into LDS by
// buffer_load_dwordx4 ... lds with no staging registers, in unpadded rows whose
// 16-byte chunks are XOR-swizzled by tswz().  Operands that the MFMAs need
// with the other dimension innermost (V^T, K^T, Q^T, dO^T) are read from the
// same tiles with ds_read_b64_tr_b16: within each 16-lane group, lane 4j+q
// points at row k0+j, columns n0+4q..n0+4q+3, and lane i receives column
// n0+i, rows k0..k0+3.  So no transposed copy of any operand exists in HBM.
// kRagged instances take sequences that are not a multiple of 64: rows past
// the end are clamped in the loads and masked with the diagonal.
// Two LDS stages: the tiles of step i+1 are issued right after the barrier
// that opens step i (the barrier's fence waits for the loads of step i).
// ---------------------------------------------------------------------------
// Raw buffer starting at a tile's first row (src is the same for every
// lane): the DMA loads below take a 32-bit per-lane offset within the tile's
// 64 rows, which measured faster than 64-bit per-lane addresses.
__device__ __forceinline__ lz_v4i tile_rsrc(const uint16_t* src) { return lz_buffer_rsrc(src); }

__device__ __forceinline__ void lds_dma16(lz_v4i rsrc, uint32_t voff, char* dst) { lz_dma16(rsrc, voff, 0, dst); }

// A [64][HD] tile of rows `src` (stride ld elements) into LDS at `dst` by DMA:
// 64*HD*2/1024 wave loads split over the 4 waves.
template <int HD>
__device__ __forceinline__ void dma_tile(const uint16_t* src, int64_t ld, char* dst, int wave, int lane) {
  constexpr int kRowsPerLoad = 1024 / (HD * 2), kChunks = HD / 8;
  constexpr int kPer = 64 / kRowsPerLoad / 4;
  const lz_v4i rsrc = tile_rsrc(src);
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int r = (wave * kPer + q) * kRowsPerLoad + lane / kChunks;
    const int c = (lane % kChunks) ^ tswz<HD>(r);
    const uint32_t voff = (uint32_t)((r * ld + c * 8) * 2);
    if (q == 0) lz_dma16_first(rsrc, voff, 0, dst + (wave * kPer + q) * 1024);
    else lds_dma16(rsrc, voff, dst + (wave * kPer + q) * 1024);
  }
}

// dma_tile with rows past `nvalid` (1..63) clamped to the last valid one;
// their results are masked.
template <int HD>
__device__ __forceinline__ void dma_tile_tail(const uint16_t* src, int64_t ld, int nvalid, char* dst, int wave,
                                              int lane) {
  constexpr int kRowsPerLoad = 1024 / (HD * 2), kChunks = HD / 8;
  constexpr int kPer = 64 / kRowsPerLoad / 4;
  const lz_v4i rsrc = tile_rsrc(src);
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int r = (wave * kPer + q) * kRowsPerLoad + lane / kChunks;
    const int c = (lane % kChunks) ^ tswz<HD>(r);
    const uint32_t voff = (uint32_t)((min(r, nvalid - 1) * ld + c * 8) * 2);
    if (q == 0) lz_dma16_first(rsrc, voff, 0, dst + (wave * kPer + q) * 1024);
    else lds_dma16(rsrc, voff, dst + (wave * kPer + q) * 1024);
  }
}

// The tile of rows r0 .. r0+63 of a sequence of S rows (kRagged: its last
// rows may not exist).
template <int HD, bool kRagged>
__device__ __forceinline__ void dma_seq_tile(const uint16_t* base, int64_t ld, int r0, int S, char* dst, int wave,
                                             int lane) {
  const uint16_t* src = base + (int64_t)r0 * ld;
  if constexpr (kRagged) {
    if (S - r0 < 64) {
      dma_tile_tail<HD>(src, ld, S - r0, dst, wave, lane);
      return;
    }
  }
  dma_tile<HD>(src, ld, dst, wave, lane);
}

// 64 floats at src into LDS at dst by lanes 0-15 of the calling wave, and 64
// floats at src2 into dst + 256 by lanes 16-31 (src, src2 and dst uniform).
__device__ __forceinline__ void dma_rows64(const float* src, const float* src2, char* dst, int lane) {
  if (lane < 16) lz_dma16(lz_buffer_rsrc(src), 16 * lane, 0, dst);
  else if (lane < 32) lz_dma16(lz_buffer_rsrc(src2), 16 * (lane - 16), 0, dst);
}

// Forward on tiles: 128 queries per workgroup (32 per wave), 64-key steps,
// K and V tiles double-buffered in LDS (the next step's tiles are issued
// right after the barrier that opens a step).
template <int HD, typename F>
__device__ __forceinline__ void fwd_scores(f32x16_t (&s)[2], const TileOffsets<HD>& to, const char* Kt,
                                           const bf16x8_t (&qf)[HD / 16]) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
#pragma unroll
  for (int kk = 0; kk < HD / 16; ++kk)
#pragma unroll
    for (int t = 0; t < 2; ++t)
      s[t] = mfma16<F>(to.frag(Kt, t, kk), qf[kk], s[t]);
}

// Online softmax of one 64-key step and its P.V product.  s: the step's
// scores (lane = query column, registers = keys t*32 + 8*(r/4) + 4*half +
// r%4); MASK: keys with index > lim are masked (the diagonal step only, so
// that the other steps carry no masking instructions).  The running max m is
// kept in log2 units; l and O are rescaled only when some lane's max moves.
template <int HD, bool MASK, typename F>
__device__ __forceinline__ void fwd_softmax_pv(f32x16_t (&s)[2], f32x16_t (&o)[HD / 32], float& m, float& l,
                                               const TileOffsets<HD>& to, const char* Vt, float c, int lim, int half) {
  constexpr int BKV = 64;
  // the V^T fragments of the first 16 keys, read now so that the first P.V
  // MFMAs do not wait for LDS after the softmax
  bf16x8_t vf[2][HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) vf[0][i] = to.frag_t(Vt, 0, i);
  float mx = -INFINITY;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (MASK) {
        const int kv = t * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
        if (kv > lim) s[t][r] = -INFINITY;
      }
      mx = fmaxf(mx, s[t][r]);
    }
  mx = max_halves(mx);
  const float m_step = mx * c;
  if (__builtin_amdgcn_read_exec() & __ballot(m_step > m)) {  // some lane's max moved
    const float m_new = fmaxf(m, m_step);
    const float alpha = __builtin_amdgcn_exp2f(m - m_new);
    l *= alpha;
#pragma unroll
    for (int i = 0; i < HD / 32; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
    m = m_new;
  }
  const float nm = -m;
  float rs = 0.f;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s[t][r], c, nm));
      s[t][r] = p;
      rs += p;
    }
  l += sum_halves(rs);
#pragma unroll
  for (int ks = 0; ks < BKV / 16; ++ks) {
    if (ks + 1 < BKV / 16)  // the next 16 keys' fragments while these MFMAs run
#pragma unroll
      for (int i = 0; i < HD / 32; ++i) vf[(ks + 1) & 1][i] = to.frag_t(Vt, ks + 1, i);
    const bf16x8_t pb = pack8<F>(s[ks >> 1], 8 * (ks & 1));
#pragma unroll
    for (int i = 0; i < HD / 32; ++i)
      o[i] = mfma16<F>(vf[ks & 1][i], pb, o[i]);
  }
}

template <int HD, typename F, bool kRagged = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HD == 64 ? 4 : 2, HD == 64 ? 4 : 2))) attn_fwd_tile_kernel(AttnArgs a) {
  constexpr int BQ = 128, BKV = 64;
  constexpr int kTile = BKV * HD * 2;
  __shared__ __attribute__((aligned(1024))) char smem[4 * kTile];  // K slots 0, 1; V slots 0, 1
  char* const Ks = smem;
  char* const Vs = smem + 2 * kTile;

  const int S = a.S, H = a.H, KV = a.KV;
  const int nqb = (S + BQ - 1) / BQ;
  int qb, b, h;
  query_block_coords(blockIdx.x, nqb, a.B, H, KV, qb, b, h);
  const int g = h / (H / KV);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  TileOffsets<HD> to;
  to.init(lane);
  const int q0 = qb * BQ, qw0 = q0 + 32 * wave;
  const int qrow = qw0 + l32;

  bf16x8_t qf[HD / 16];
  {
    const uint16_t* qp = a.q + ((int64_t)b * S + min(qrow, S - 1)) * a.ldq + (int64_t)h * HD + 8 * half;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) qf[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qp + kk * 16));
  }
  f32x16_t o[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  float m = -INFINITY, l = 0.f;
  const float c = a.scale * kLog2e;

  const int kv_end = min(S, q0 + BQ);  // a multiple of 64 unless kRagged
  const int kv_end_w = qw0 < S ? min(S, qw0 + 32) : 0;  // a wave past the sequence computes nothing
  const uint16_t* kbase = a.k + (int64_t)b * S * a.ldk + (int64_t)g * HD;
  const uint16_t* vbase = a.v + (int64_t)b * S * a.ldv + (int64_t)g * HD;
  const int nsteps = kRagged ? (kv_end + BKV - 1) / BKV : kv_end / BKV;

  // Step it: wait for its K/V (and every wave's reads of step it-1), then
  // issue step it+1's tiles into the other slot.
  auto open_step = [&](int it) {
    dma_barrier();
    if (it + 1 < nsteps) {
      dma_seq_tile<HD, kRagged>(kbase, a.ldk, (it + 1) * BKV, S, Ks + ((it + 1) & 1) * kTile, wave, lane);
      dma_seq_tile<HD, kRagged>(vbase, a.ldv, (it + 1) * BKV, S, Vs + ((it + 1) & 1) * kTile, wave, lane);
    }
  };
  // This wave's last step holds its diagonal (the only step with masked
  // keys: 32 queries starting at a multiple of 32 against 64-key steps);
  // the loop before it has no branch, so the accumulators stay in place.
  const int last_w = kv_end_w > 0 ? (kv_end_w - 1) / BKV : -1;
  dma_seq_tile<HD, kRagged>(kbase, a.ldk, 0, S, Ks, wave, lane);
  dma_seq_tile<HD, kRagged>(vbase, a.ldv, 0, S, Vs, wave, lane);
  int it = 0;
  for (; it < last_w; ++it) {
    open_step(it);
    f32x16_t s[2];
    fwd_scores<HD, F>(s, to, Ks + (it & 1) * kTile, qf);
    fwd_softmax_pv<HD, false, F>(s, o, m, l, to, Vs + (it & 1) * kTile, c, 0, half);
  }
  if (last_w >= 0) {
    open_step(it);
    f32x16_t s[2];
    fwd_scores<HD, F>(s, to, Ks + (it & 1) * kTile, qf);
    fwd_softmax_pv<HD, true, F>(s, o, m, l, to, Vs + (it & 1) * kTile, c, qrow - it * BKV, half);
    ++it;
  }
  for (; it < nsteps; ++it) open_step(it);  // past this wave's diagonal: it only joins the barriers
  if (qrow < S) {
    const float inv_l = 1.0f / l;
    uint16_t* op = a.o + ((int64_t)b * S + qrow) * a.ldo + (int64_t)h * HD;
#pragma unroll
    for (int i = 0; i < HD / 32; ++i)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int hd = i * 32 + 8 * q4 + 4 * half;
        store_bf16x4<F>(op + hd, o[i][4 * q4] * inv_l, o[i][4 * q4 + 1] * inv_l, o[i][4 * q4 + 2] * inv_l,
                     o[i][4 * q4 + 3] * inv_l);
      }
    if (half == 0) a.lse[((int64_t)b * H + h) * S + qrow] = (m + log2f(l)) * kLn2;
  }
}

// The same for rows of any alignment, of which nvalid exist (the rest repeat
// the last one): 4 bytes per lane, one load per array.
__device__ __forceinline__ void dma_rows64_any(const float* src, const float* src2, int nvalid, char* dst, int lane) {
  const uint32_t voff = 4 * min(lane, nvalid - 1);
  lz_dma4_first(lz_buffer_rsrc(src), voff, dst);
  lz_dma4_first(lz_buffer_rsrc(src2), voff, dst + 256);
}

// A [64][HD] tile like dma_tile, loaded by the four waves of group `wg4`
// (wave index 0..3 within the group), rows past `nvalid` clamped to the last
// valid row (their results are masked).
template <int HD>
__device__ __forceinline__ void dma_tile_rows(const uint16_t* src, int64_t ld, int nvalid, char* dst, int wg4,
                                              int lane) {
  constexpr int kRowsPerLoad = 1024 / (HD * 2), kChunks = HD / 8;
  constexpr int kPer = 64 / kRowsPerLoad / 4;
  const lz_v4i rsrc = tile_rsrc(src);
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int r = (wg4 * kPer + q) * kRowsPerLoad + lane / kChunks;
    const int c = (lane % kChunks) ^ tswz<HD>(r);
    lds_dma16(rsrc, (uint32_t)((min(r, nvalid - 1) * ld + c * 8) * 2), dst + (wg4 * kPer + q) * 1024);
  }
}

// Issues the tiles of dK/dV step `step` for the 8-wave kernel: Q by waves
// 0-3, dO by waves 4-7, lse and delta by wave 0.
template <int HD, bool kRagged>
__device__ __forceinline__ void dkdv8_issue(const AttnArgs& a, int step, int nqs, int qstart, int b, int g, int rep,
                                            char* st, int wave, int lane) {
  constexpr int kTile = 64 * HD * 2;
  const int S = a.S;
  const int hq = step / nqs, q0 = qstart + (step - hq * nqs) * 64;
  const int h = g * rep + hq;
  if (wave < 4)
    dma_seq_tile<HD, kRagged>(a.q + (int64_t)b * S * a.ldq + (int64_t)h * HD, a.ldq, q0, S, st, wave, lane);
  else
    dma_seq_tile<HD, kRagged>(a.dout + (int64_t)b * S * a.lddo + (int64_t)h * HD, a.lddo, q0, S, st + kTile, wave - 4,
                              lane);
  if (wave == 0) {
    const int64_t off = ((int64_t)b * a.H + h) * S + q0;
    if constexpr (kRagged) dma_rows64_any(a.lse + off, a.delta + off, min(64, S - q0), st + 2 * kTile, lane);
    else dma_rows64(a.lse + off, a.delta + off, st + 2 * kTile, lane);
  }
}

// dK/dV with two waves per SIMD: 256 keys per workgroup of 8 waves (32 keys
// per wave), K fragments in registers, the workgroup's V tile in LDS (read
// back as fragments), 64-query steps over every query head of the kv head's
// group from the diagonal on: S^T = K Q^T and dP^T = V dO^T per 32-query
// half, P = exp(S*scale - lse), dS = P (dP - delta), then dV += P^T dO and
// dK += dS^T Q from transposed LDS reads.
// One 64-query step of the 8-wave dK/dV kernel for this wave's 32 keys:
// S^T and dP^T, P and dS, then dV += P^T dO and dK += dS^T Q.  MASK: the
// step crosses this wave's diagonal (or the sequence's end), so pairs with
// key > query (or query >= S) are dropped; the other steps carry no masking
// instructions.
template <int HD, bool MASK, typename F, bool kRagged>
__device__ __forceinline__ void dkdv_step(f32x16_t (&dk)[HD / 32], f32x16_t (&dv)[HD / 32], const TileOffsets<HD>& to,
                                          const char* Qt, const char* Vt, const bf16x8_t (&kf)[HD / 16], float c,
                                          int q0, int kvrow, int S, int wave, int half) {
  constexpr int kTile = 64 * HD * 2;
  const char* dOt = Qt + kTile;
  const float* lse_s = reinterpret_cast<const float*>(Qt + 2 * kTile);
  const float* D_s = lse_s + 64;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x16_t sc, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = 0.f;
      dp[r] = 0.f;
    }
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      sc = mfma16<F>(to.frag(Qt, t, kk), kf[kk], sc);
      dp = mfma16<F>(to.frag(dOt, t, kk), to.frag(Vt, wave, kk), dp);
      // keeps the fragment reads next to their MFMAs: two waves per SIMD
      // hide the latency, and the register budget is 256
      if constexpr (HD == 128) __builtin_amdgcn_sched_barrier(0);
    }
    // lane holds key column kvrow; query rows t*32 + 8*(r/4) + 4*half + r%4
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const int qlb = t * 32 + 8 * r4 + 4 * half;
      const float4 l4 = *reinterpret_cast<const float4*>(lse_s + qlb);
      const float4 d4 = *reinterpret_cast<const float4*>(D_s + qlb);
      const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
      const float dvv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * r4 + e;
        float p = __builtin_amdgcn_exp2f(fmaf(sc[r], c, -lv[e] * kLog2e));
        if constexpr (MASK) {
          p = kvrow <= q0 + qlb + e ? p : 0.f;
          if constexpr (kRagged) p = q0 + qlb + e < S ? p : 0.f;
        }
        dp[r] = p * (dp[r] - dvv[e]);
        sc[r] = p;
      }
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      const int ks = 2 * t + kh;
      const bf16x8_t pb = pack8<F>(sc, 8 * kh);
      const bf16x8_t dsb = pack8<F>(dp, 8 * kh);
#pragma unroll
      for (int i = 0; i < HD / 32; ++i) {
        dv[i] = mfma16<F>(to.frag_t(dOt, ks, i), pb, dv[i]);
        dk[i] = mfma16<F>(to.frag_t(Qt, ks, i), dsb, dk[i]);
        if constexpr (HD == 128) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <int HD, typename F, bool kRagged = false>
__global__ void __launch_bounds__(512) attn_bwd_dkdv_wide_kernel(AttnArgs a) {
  constexpr int BKV = 256, BQ = 64;
  constexpr int kTile = BQ * HD * 2;
  constexpr int kVTile = BKV * HD * 2;
  constexpr int kStage = 2 * kTile + 512;  // Q, dO, lse[64], delta[64]
  __shared__ __attribute__((aligned(1024))) char smem[kVTile + 2 * kStage];

  const int S = a.S, H = a.H, KV = a.KV, rep = H / KV;
  int kvb, b, g;
  key_block_coords(blockIdx.x, a.B, KV, kvb, b, g);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  TileOffsets<HD> to;
  to.init(lane);
  const int k0 = kvb * BKV, kw0 = k0 + 32 * wave;
  const int kvrow = kw0 + l32;
  const float c = a.scale * kLog2e;
  const char* Vt = smem;
  char* stages = smem + kVTile;

  {  // the V tile: 64-row quarters 2*(wave/4) and 2*(wave/4)+1
    const int quarter0 = 2 * (wave >> 2);
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
      const int r0 = k0 + 64 * (quarter0 + qq);
      dma_tile_rows<HD>(a.v + ((int64_t)b * S + min(r0, S - 1)) * a.ldv + (int64_t)g * HD, a.ldv, S - min(r0, S - 1),
                        smem + (quarter0 + qq) * kTile, wave & 3, lane);
    }
  }
  bf16x8_t kf[HD / 16];
  {
    const int64_t r = (int64_t)b * S + min(kvrow, S - 1);
    const uint16_t* kp = a.k + r * a.ldk + (int64_t)g * HD + 8 * half;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk)
      kf[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(kp + kk * 16));
  }
  f32x16_t dk[HD / 32], dv[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dk[i][r] = 0.f;
      dv[i][r] = 0.f;
    }

  const int qstart = (k0 / BQ) * BQ;
  const int nqs = kRagged ? (S - qstart + BQ - 1) / BQ : (S - qstart) / BQ;
  const int nsteps = rep * nqs;
  auto open_step = [&](int step) {
    dma_barrier();  // this step's tiles (and the V tile) landed, last step's reads retired
    if (step + 1 < nsteps)
      dkdv8_issue<HD, kRagged>(a, step + 1, nqs, qstart, b, g, rep, stages + ((step + 1) & 1) * kStage, wave, lane);
  };
  // Per query head, the 64-query blocks j = 0 .. nqs-1 (queries qstart + 64j
  // on) fall into three runs for this wave's keys kw0 .. kw0+31 (kw0 a
  // multiple of 32): blocks wholly before the keys (no work), blocks across
  // the diagonal (masked), blocks wholly after it (unmasked).  Every wave
  // opens every step, so the barriers match.
  const int rel = kw0 - qstart;  // 0 .. 224
  const int j_first = kw0 < S ? min(nqs, rel / BQ) : nqs;
  const int j_unmasked = kw0 < S ? min(nqs, (rel + 32 + BQ - 1) / BQ) : nqs;
  const int j_tail = kRagged && S % BQ && kw0 < S ? max(j_unmasked, nqs - 1) : nqs;  // a last block of fewer queries
  dkdv8_issue<HD, kRagged>(a, 0, nqs, qstart, b, g, rep, stages, wave, lane);
  int step = 0;
  for (int hq = 0; hq < rep; ++hq) {
    int j = 0;
    for (; j < j_first; ++j, ++step) open_step(step);
    for (; j < j_unmasked; ++j, ++step) {
      open_step(step);
      dkdv_step<HD, true, F, kRagged>(dk, dv, to, stages + (step & 1) * kStage, Vt, kf, c, qstart + j * BQ, kvrow, S,
                                      wave, half);
    }
    for (; j < j_tail; ++j, ++step) {
      open_step(step);
      dkdv_step<HD, false, F, kRagged>(dk, dv, to, stages + (step & 1) * kStage, Vt, kf, c, qstart + j * BQ, kvrow, S,
                                       wave, half);
    }
    if constexpr (kRagged) {
      for (; j < nqs; ++j, ++step) {
        open_step(step);
        dkdv_step<HD, true, F, true>(dk, dv, to, stages + (step & 1) * kStage, Vt, kf, c, qstart + j * BQ, kvrow, S,
                                     wave, half);
      }
    }
  }
  if (kvrow < S) {
    uint16_t* dkp = a.dk + ((int64_t)b * S + kvrow) * a.lddk + (int64_t)g * HD;
    uint16_t* dvp = a.dv + ((int64_t)b * S + kvrow) * a.lddv + (int64_t)g * HD;
    const bool rope = a.rcos != nullptr;
    store_grad_row<HD, F>(dkp, dk, a.scale, half, rope ? a.rcos + (int64_t)kvrow * HD : nullptr,
                       rope ? a.rsin + (int64_t)kvrow * HD : nullptr);
    store_grad_row<HD, F>(dvp, dv, 1.0f, half, nullptr, nullptr);
  }
}

// One 64-key step of the dQ kernel for this wave's 32 queries: S and dP, dS,
// then dQ += dS K.  MASK: the step holds this wave's diagonal, so keys past
// the query are dropped (the other steps carry no masking instructions).
template <int HD, bool MASK, typename F>
__device__ __forceinline__ void dq_step(f32x16_t (&dq)[HD / 32], const TileOffsets<HD>& to, const char* Kt,
                                        const bf16x8_t (&qf)[HD / 16], const bf16x8_t (&df)[HD / 16], float c, float nl2,
                                        float Dq, int k0, int qrow, int half) {
  constexpr int kTile = 64 * HD * 2;
  const char* Vt = Kt + kTile;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x16_t st, dpt;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      st[r] = 0.f;
      dpt[r] = 0.f;
    }
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      st = mfma16<F>(to.frag(Kt, t, kk), qf[kk], st);
      dpt = mfma16<F>(to.frag(Vt, t, kk), df[kk], dpt);
    }
    // the K^T fragments of the first 16 keys, read before dS is formed so
    // that the dQ MFMAs do not wait for LDS; the next 16 keys' during them
    bf16x8_t kt[2][HD / 32];
#pragma unroll
    for (int i = 0; i < HD / 32; ++i) kt[0][i] = to.frag_t(Kt, 2 * t, i);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float p = __builtin_amdgcn_exp2f(fmaf(st[r], c, nl2));
      if constexpr (MASK) {
        const int kv = k0 + t * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
        p = kv <= qrow ? p : 0.f;
      }
      dpt[r] = p * (dpt[r] - Dq);
    }
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      if (kh == 0)
#pragma unroll
        for (int i = 0; i < HD / 32; ++i) kt[1][i] = to.frag_t(Kt, 2 * t + 1, i);
      const bf16x8_t dsb = pack8<F>(dpt, 8 * kh);
#pragma unroll
      for (int i = 0; i < HD / 32; ++i)
        dq[i] = mfma16<F>(kt[kh][i], dsb, dq[i]);
    }
  }
}

// dQ on tiles: 128 queries per workgroup, 64-key steps up to the diagonal.
// kDelta: delta = rowsum(dO * O) of the workgroup's queries is computed here
// (from the dO fragments held in registers and the same columns of O, a.o)
// and written to a.delta_w for the dK/dV kernel that runs next, instead of
// read from a.delta.
template <int HD, typename F, bool kDelta = false, bool kRagged = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) attn_bwd_dq_tile_kernel(AttnArgs a) {
  constexpr int BQ = 128, BKV = 64;
  constexpr int kTile = BKV * HD * 2;
  constexpr int kStage = 2 * kTile;  // K, V
  __shared__ __attribute__((aligned(1024))) char smem[2 * kStage];

  const int S = a.S, H = a.H, KV = a.KV;
  const int nqb = (S + BQ - 1) / BQ;
  int qb, b, h;
  query_block_coords(blockIdx.x, nqb, a.B, H, KV, qb, b, h);
  const int g = h / (H / KV);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  TileOffsets<HD> to;
  to.init(lane);
  const int q0 = qb * BQ, qw0 = q0 + 32 * wave;
  const int qrow = qw0 + l32;
  const int qc = min(qrow, S - 1);
  const float c = a.scale * kLog2e;

  bf16x8_t qf[HD / 16], df[HD / 16];
  {
    const uint16_t* qp = a.q + ((int64_t)b * S + qc) * a.ldq + (int64_t)h * HD + 8 * half;
    const uint16_t* dp_ = a.dout + ((int64_t)b * S + qc) * a.lddo + (int64_t)h * HD + 8 * half;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      qf[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(qp + kk * 16));
      df[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(dp_ + kk * 16));
    }
  }
  const float nl2 = -a.lse[((int64_t)b * H + h) * S + qc] * kLog2e;
  float Dq;
  if constexpr (kDelta) {
    // each half of the wave holds half of the row's columns (8 of every 16)
    const uint16_t* op = a.o + ((int64_t)b * S + qc) * a.ldo + (int64_t)h * HD + 8 * half;
    float acc = 0.f;
#pragma unroll
    for (int kk = 0; kk < HD / 16; ++kk) {
      const uint4 ov = *reinterpret_cast<const uint4*>(op + kk * 16);
      const uint4 dv = __builtin_bit_cast(uint4, df[kk]);
      const uint32_t ow[4] = {ov.x, ov.y, ov.z, ov.w}, dw[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) {
        acc = fmaf(F::to_f(ow[k2] & 0xffff), F::to_f(dw[k2] & 0xffff), acc);
        acc = fmaf(F::to_f(ow[k2] >> 16), F::to_f(dw[k2] >> 16), acc);
      }
    }
    Dq = sum_halves(acc);
    if (qrow < S && half == 0) a.delta_w[((int64_t)b * H + h) * S + qrow] = Dq;
  } else {
    Dq = a.delta[((int64_t)b * H + h) * S + qc];
  }
  f32x16_t dq[HD / 32];
#pragma unroll
  for (int i = 0; i < HD / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[i][r] = 0.f;

  const int kv_end = min(S, q0 + BQ);
  const int kv_end_w = qw0 < S ? min(S, qw0 + 32) : 0;  // a wave past the sequence computes nothing
  const uint16_t* kbase = a.k + (int64_t)b * S * a.ldk + (int64_t)g * HD;
  const uint16_t* vbase = a.v + (int64_t)b * S * a.ldv + (int64_t)g * HD;
  const int nsteps = kRagged ? (kv_end + BKV - 1) / BKV : kv_end / BKV;

  auto open_step = [&](int it) {
    dma_barrier();  // this step's tiles landed (every wave's loads), last step's reads retired
    if (it + 1 < nsteps) {
      char* nxt = smem + ((it + 1) & 1) * kStage;
      dma_seq_tile<HD, kRagged>(kbase, a.ldk, (it + 1) * BKV, S, nxt, wave, lane);
      dma_seq_tile<HD, kRagged>(vbase, a.ldv, (it + 1) * BKV, S, nxt + kTile, wave, lane);
    }
  };
  // This wave's last step holds its diagonal (the only masked step); the
  // steps after it only join the barriers.
  const int last_w = kv_end_w > 0 ? (kv_end_w - 1) / BKV : -1;
  dma_seq_tile<HD, kRagged>(kbase, a.ldk, 0, S, smem, wave, lane);
  dma_seq_tile<HD, kRagged>(vbase, a.ldv, 0, S, smem + kTile, wave, lane);
  int it = 0;
  for (; it < last_w; ++it) {
    open_step(it);
    dq_step<HD, false, F>(dq, to, smem + (it & 1) * kStage, qf, df, c, nl2, Dq, it * BKV, qrow, half);
  }
  if (last_w >= 0) {
    open_step(it);
    dq_step<HD, true, F>(dq, to, smem + (it & 1) * kStage, qf, df, c, nl2, Dq, it * BKV, qrow, half);
    ++it;
  }
  for (; it < nsteps; ++it) open_step(it);
  if (qrow < S) {
    uint16_t* dqp = a.dq + ((int64_t)b * S + qrow) * a.lddq + (int64_t)h * HD;
    const bool rope = a.rcos != nullptr;
    store_grad_row<HD, F>(dqp, dq, a.scale, half, rope ? a.rcos + (int64_t)qrow * HD : nullptr,
                       rope ? a.rsin + (int64_t)qrow * HD : nullptr);
  }
}

// delta[b,h,s] = sum_d dO[b,s,h,d] * O[b,s,h,d]; one wave per (b, s, h) row.
template <typename T>
__global__ void __launch_bounds__(256) attn_delta_kernel(const T* __restrict__ o, int64_t ldo, const T* __restrict__ dout,
                                                          int64_t lddo, float* __restrict__ delta, int B, int S, int H,
                                                          int hd) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t total = (int64_t)B * S * H;
  if (row >= total) return;
  const int64_t bs = row / H;
  const int h = (int)(row - bs * H);
  const T* op = o + bs * ldo + (int64_t)h * hd;
  const T* dp = dout + bs * lddo + (int64_t)h * hd;
  float acc = 0.f;
  for (int d = lane; d < hd; d += 64) acc = fmaf(Elem<T>::load(op, d), Elem<T>::load(dp, d), acc);
  acc = wave_sum(acc);
  if (lane == 0) {
    const int64_t b = bs / S, s = bs - b * S;
    delta[(b * H + h) * S + s] = acc;
  }
}

// bf16 vector path: CPR = hd / 8 consecutive lanes share one (b, s, h) row,
// each loading 16 bytes of O and of dO (nontemporal: both are streamed
// once), so a workgroup reads 256 x 16 contiguous bytes of each; the row's
// partial sums meet through lane shuffles.  rows = B*S*H < 2^31.
template <int CPR>
__global__ void __launch_bounds__(256) attn_delta_vec_kernel(const uint16_t* __restrict__ o, int64_t ldo,
                                                              const uint16_t* __restrict__ dout, int64_t lddo,
                                                              float* __restrict__ delta, int S, int H, int rows) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int row = i / CPR, c = i % CPR;
  float acc = 0.f;
  if (row < rows) {
    const int bs = row / H, h = row - bs * H;
    const int64_t off = (int64_t)h * (CPR * 8) + c * 8;
    const v4u ov = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(o + bs * ldo + off));
    const v4u dv = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(dout + bs * lddo + off));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      acc = fmaf(bf2f(ov[k] & 0xffff), bf2f(dv[k] & 0xffff), acc);
      acc = fmaf(bf2f(ov[k] >> 16), bf2f(dv[k] >> 16), acc);
    }
  }
#pragma unroll
  for (int m = CPR / 2; m > 0; m >>= 1) acc += __shfl_xor(acc, m, 64);
  if (row < rows && c == 0) {
    const int bs = row / H, h = row - bs * H;
    const int b = bs / S, s = bs - b * S;
    delta[((int64_t)b * H + h) * S + s] = acc;
  }
}

// ---------------------------------------------------------------------------
// Generic path (any even head dim up to 256, any dtype and alignment): one
// wave per query row (forward, dQ) or key row (dK/dV), lanes split the head
// dim, fp32 online softmax.  Used where neither MFMA family applies.
// ---------------------------------------------------------------------------
template <typename T>
struct GenArgs {
  const T* q;
  const T* k;
  const T* v;
  int64_t ldq, ldk, ldv;
  T* o;
  int64_t ldo;
  float* lse;
  const T* dout;
  int64_t lddo;
  const float* delta;
  T* dq;
  T* dk;
  T* dv;
  int64_t lddq, lddk, lddv;
  int B, S, H, KV, hd;
  float scale;
  // explicit mask (SDPA's attn_mask; then no causal mask): kind 1 = bool
  // (bytes, nonzero keeps the score), 2 = fp32, 3 = bf16, 4 = fp16 (added to the
  // scaled score); element strides over [B, H, S(query), S(key)], 0 where
  // the mask broadcasts
  const void* mask;
  int mask_kind;
  int64_t msb, msh, msq, msk;
  // attention dropout (SDPA dropout_p): the probability of (b, h, query s,
  // key kv) is kept with scale 1/(1-p) when element ((b*H + h)*S + s)*S + kv
  // of the seed's stream is kept (lz_keep); drop_thresh 0 = no dropout
  uint32_t drop_thresh;
  float drop_scale;
  uint64_t drop_seed;
};

// Dropout factor of one attention probability (1 without dropout).
template <typename T>
__device__ __forceinline__ float drop_factor(const GenArgs<T>& a, int b, int h, int s, int kv) {
  if (a.drop_thresh == 0) return 1.0f;
  const uint64_t i = (((uint64_t)b * a.H + h) * a.S + s) * a.S + kv;
  return lz_keep(a.drop_seed, i, a.drop_thresh) ? a.drop_scale : 0.0f;
}

constexpr int kGenMax = 4;  // head dim up to 64 * kGenMax

// The scaled score of (b, h, query s, key kv) with the explicit mask applied:
// -inf where a bool mask is false, score + mask for a float mask.
template <typename T>
__device__ __forceinline__ float masked_score(const GenArgs<T>& a, float sc, int b, int h, int s, int kv) {
  const int64_t i = (int64_t)b * a.msb + (int64_t)h * a.msh + (int64_t)s * a.msq + (int64_t)kv * a.msk;
  if (a.mask_kind == 1) return static_cast<const uint8_t*>(a.mask)[i] ? sc : -INFINITY;
  if (a.mask_kind == 2) return sc + static_cast<const float*>(a.mask)[i];
  if (a.mask_kind == 3) return sc + bf2f(static_cast<const uint16_t*>(a.mask)[i]);
  return sc + h2f(static_cast<const uint16_t*>(a.mask)[i]);
}

template <typename T>
__global__ void __launch_bounds__(256) attn_fwd_generic_kernel(GenArgs<T> a) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t total = (int64_t)a.B * a.H * a.S;
  if (row >= total) return;
  const int s = (int)(row % a.S);
  const int64_t bh = row / a.S;
  const int h = (int)(bh % a.H), b = (int)(bh / a.H);
  const int g = h / (a.H / a.KV);
  const T* qp = a.q + ((int64_t)b * a.S + s) * a.ldq + (int64_t)h * a.hd;
  float qv[kGenMax], ov[kGenMax];
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    qv[j] = d < a.hd ? Elem<T>::load(qp, d) : 0.f;
    ov[j] = 0.f;
  }
  float m = -INFINITY, l = 0.f;
  const int kv_last = a.mask_kind ? a.S - 1 : s;  // an explicit mask replaces the causal one
  for (int kv = 0; kv <= kv_last; ++kv) {
    const T* kp = a.k + ((int64_t)b * a.S + kv) * a.ldk + (int64_t)g * a.hd;
    const T* vp = a.v + ((int64_t)b * a.S + kv) * a.ldv + (int64_t)g * a.hd;
    float dot = 0.f;
#pragma unroll
    for (int j = 0; j < kGenMax; ++j) {
      const int d = lane + 64 * j;
      if (d < a.hd) dot = fmaf(qv[j], Elem<T>::load(kp, d), dot);
    }
    float sc = wave_sum(dot) * a.scale;
    if (a.mask_kind) {
      sc = masked_score(a, sc, b, h, s, kv);
      if (sc == -INFINITY) continue;  // contributes nothing (and keeps m finite once it is)
    }
    const float m_new = fmaxf(m, sc);
    const float corr = expf(m - m_new), p = expf(sc - m_new);
    l = l * corr + p;  // the normaliser sums the probabilities before dropout
    const float pz = p * drop_factor(a, b, h, s, kv);
#pragma unroll
    for (int j = 0; j < kGenMax; ++j) {
      const int d = lane + 64 * j;
      if (d < a.hd) ov[j] = ov[j] * corr + pz * Elem<T>::load(vp, d);
    }
    m = m_new;
  }
  T* op = a.o + ((int64_t)b * a.S + s) * a.ldo + (int64_t)h * a.hd;
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    if (d < a.hd) Elem<T>::store(op, d, ov[j] / l);
  }
  if (lane == 0) a.lse[((int64_t)b * a.H + h) * a.S + s] = m + logf(l);
}

template <typename T>
__global__ void __launch_bounds__(256) attn_bwd_dq_generic_kernel(GenArgs<T> a) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t total = (int64_t)a.B * a.H * a.S;
  if (row >= total) return;
  const int s = (int)(row % a.S);
  const int64_t bh = row / a.S;
  const int h = (int)(bh % a.H), b = (int)(bh / a.H);
  const int g = h / (a.H / a.KV);
  const T* qp = a.q + ((int64_t)b * a.S + s) * a.ldq + (int64_t)h * a.hd;
  const T* dop = a.dout + ((int64_t)b * a.S + s) * a.lddo + (int64_t)h * a.hd;
  float qv[kGenMax], dov[kGenMax], acc[kGenMax];
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    qv[j] = d < a.hd ? Elem<T>::load(qp, d) : 0.f;
    dov[j] = d < a.hd ? Elem<T>::load(dop, d) : 0.f;
    acc[j] = 0.f;
  }
  const float lse = a.lse[((int64_t)b * a.H + h) * a.S + s];
  const float D = a.delta[((int64_t)b * a.H + h) * a.S + s];
  const int kv_last = a.mask_kind ? a.S - 1 : s;
  for (int kv = 0; kv <= kv_last; ++kv) {
    const T* kp = a.k + ((int64_t)b * a.S + kv) * a.ldk + (int64_t)g * a.hd;
    const T* vp = a.v + ((int64_t)b * a.S + kv) * a.ldv + (int64_t)g * a.hd;
    float dot = 0.f, dpd = 0.f;
#pragma unroll
    for (int j = 0; j < kGenMax; ++j) {
      const int d = lane + 64 * j;
      if (d < a.hd) {
        dot = fmaf(qv[j], Elem<T>::load(kp, d), dot);
        dpd = fmaf(dov[j], Elem<T>::load(vp, d), dpd);
      }
    }
    float sc = wave_sum(dot) * a.scale;
    if (a.mask_kind) sc = masked_score(a, sc, b, h, s, kv);
    const float p = expf(sc - lse);
    // dL/dP = Z * dO.V for the dropped-out P; D = rowsum(dO * O) is unchanged
    const float ds = p * (drop_factor(a, b, h, s, kv) * wave_sum(dpd) - D);
#pragma unroll
    for (int j = 0; j < kGenMax; ++j) {
      const int d = lane + 64 * j;
      if (d < a.hd) acc[j] = fmaf(ds, Elem<T>::load(kp, d), acc[j]);
    }
  }
  T* dqp = a.dq + ((int64_t)b * a.S + s) * a.lddq + (int64_t)h * a.hd;
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    if (d < a.hd) Elem<T>::store(dqp, d, acc[j] * a.scale);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) attn_bwd_dkdv_generic_kernel(GenArgs<T> a) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t total = (int64_t)a.B * a.KV * a.S;
  if (row >= total) return;
  const int kv = (int)(row % a.S);
  const int64_t bg = row / a.S;
  const int g = (int)(bg % a.KV), b = (int)(bg / a.KV);
  const int rep = a.H / a.KV;
  const T* kp = a.k + ((int64_t)b * a.S + kv) * a.ldk + (int64_t)g * a.hd;
  const T* vp = a.v + ((int64_t)b * a.S + kv) * a.ldv + (int64_t)g * a.hd;
  float kvv[kGenMax], vvv[kGenMax], dka[kGenMax], dva[kGenMax];
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    kvv[j] = d < a.hd ? Elem<T>::load(kp, d) : 0.f;
    vvv[j] = d < a.hd ? Elem<T>::load(vp, d) : 0.f;
    dka[j] = 0.f;
    dva[j] = 0.f;
  }
  for (int hq = 0; hq < rep; ++hq) {
    const int h = g * rep + hq;
    for (int s = a.mask_kind ? 0 : kv; s < a.S; ++s) {
      const T* qp = a.q + ((int64_t)b * a.S + s) * a.ldq + (int64_t)h * a.hd;
      const T* dop = a.dout + ((int64_t)b * a.S + s) * a.lddo + (int64_t)h * a.hd;
      float dot = 0.f, dpd = 0.f;
#pragma unroll
      for (int j = 0; j < kGenMax; ++j) {
        const int d = lane + 64 * j;
        if (d < a.hd) {
          dot = fmaf(Elem<T>::load(qp, d), kvv[j], dot);
          dpd = fmaf(Elem<T>::load(dop, d), vvv[j], dpd);
        }
      }
      const int64_t li = ((int64_t)b * a.H + h) * a.S + s;
      float sc = wave_sum(dot) * a.scale;
      if (a.mask_kind) sc = masked_score(a, sc, b, h, s, kv);
      const float p = expf(sc - a.lse[li]);
      const float z = drop_factor(a, b, h, s, kv);
      const float ds = p * (z * wave_sum(dpd) - a.delta[li]);
      const float pz = p * z;
#pragma unroll
      for (int j = 0; j < kGenMax; ++j) {
        const int d = lane + 64 * j;
        if (d < a.hd) {
          dva[j] = fmaf(pz, Elem<T>::load(dop, d), dva[j]);
          dka[j] = fmaf(ds, Elem<T>::load(qp, d), dka[j]);
        }
      }
    }
  }
  T* dkp = a.dk + ((int64_t)b * a.S + kv) * a.lddk + (int64_t)g * a.hd;
  T* dvp = a.dv + ((int64_t)b * a.S + kv) * a.lddv + (int64_t)g * a.hd;
#pragma unroll
  for (int j = 0; j < kGenMax; ++j) {
    const int d = lane + 64 * j;
    if (d < a.hd) {
      Elem<T>::store(dkp, d, dka[j] * a.scale);
      Elem<T>::store(dvp, d, dva[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// Small head dims (16, and 32 where the rows are not aligned for the
// wave-private kernels of attn_wave.hip): four lanes (a quad) per query row (forward, dQ)
// or key row (dK/dV), each holding a quarter of that row, its accumulators
// and the row's running softmax in registers; a workgroup of four waves owns
// 64 rows.  The other side's rows pass through LDS 64 at a time as fp32
// (written by consecutive threads, read by the 16 quads of a wave at four
// distinct addresses).  Dot products are summed over the quad with two DPP
// steps, which give all four lanes the same bits.
// ---------------------------------------------------------------------------

// rows [row0, row0 + n) of base[., ld] (columns 0 .. HD) into dst[64][HD] by
// 256 threads; rows from n on are zero.  Every load is unconditional (rows
// past n re-read row n-1), so they all issue before the first wait.
template <typename T, int HD>
__device__ __forceinline__ void stage_rows(float* dst, const T* base, int64_t ld, int64_t row0, int n, int tid) {
  constexpr int kPass = 64 * HD / 256;
  float x[kPass];
#pragma unroll
  for (int i = 0; i < kPass; ++i) {
    const int e = tid + 256 * i;
    const int r = min(e / HD, n - 1), d = e % HD;
    x[i] = Elem<T>::load(base + (row0 + r) * ld, d);
  }
#pragma unroll
  for (int i = 0; i < kPass; ++i) {
    const int e = tid + 256 * i;
    dst[e] = e / HD < n ? x[i] : 0.f;
  }
}

// DL values of a row from column c0 as fp32; rows the caller does not own
// read as zero
template <typename T, int DL>
__device__ __forceinline__ void load_part(float (&x)[DL], const T* p, bool own) {
#pragma unroll
  for (int d = 0; d < DL; ++d) x[d] = Elem<T>::load(p, d);
#pragma unroll
  for (int d = 0; d < DL; ++d) x[d] = own ? x[d] : 0.f;
}

// sum over the four lanes of a quad (quad_perm [1,0,3,2] then [2,3,0,1])
__device__ __forceinline__ float quad_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true));
  return x;
}

template <int DL>
__device__ __forceinline__ float dot_part(const float (&x)[DL], const float* row) {
  const float4* r4 = reinterpret_cast<const float4*>(row);
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < DL / 4; ++i) {
    const float4 t = r4[i];
    acc = fmaf(x[4 * i], t.x, acc);
    acc = fmaf(x[4 * i + 1], t.y, acc);
    acc = fmaf(x[4 * i + 2], t.z, acc);
    acc = fmaf(x[4 * i + 3], t.w, acc);
  }
  return acc;
}

// acc = acc * c + p * row
template <int DL>
__device__ __forceinline__ void axpby_part(float (&acc)[DL], float c, float p, const float* row) {
  const float4* r4 = reinterpret_cast<const float4*>(row);
#pragma unroll
  for (int i = 0; i < DL / 4; ++i) {
    const float4 t = r4[i];
    acc[4 * i] = fmaf(p, t.x, acc[4 * i] * c);
    acc[4 * i + 1] = fmaf(p, t.y, acc[4 * i + 1] * c);
    acc[4 * i + 2] = fmaf(p, t.z, acc[4 * i + 2] * c);
    acc[4 * i + 3] = fmaf(p, t.w, acc[4 * i + 3] * c);
  }
}

// grid: B * H * ceil(S / 64) workgroups of 256, query block fastest
template <typename T, int HD>
__global__ void __launch_bounds__(256) attn_fwd_quad_kernel(GenArgs<T> a) {
  constexpr int DL = HD / 4;
  __shared__ __attribute__((aligned(16))) float ks[64 * HD];
  __shared__ __attribute__((aligned(16))) float vs[64 * HD];
  const int tid = threadIdx.x, qd = tid & 3, rl = tid >> 2;
  const int nqb = (a.S + 63) / 64;
  const int qb = (int)(blockIdx.x % nqb);
  const int64_t bh = blockIdx.x / nqb;
  const int h = (int)(bh % a.H), b = (int)(bh / a.H);
  const int g = h / (a.H / a.KV);
  const int s = qb * 64 + rl;
  const bool valid = s < a.S;
  float q[DL], o[DL];
  load_part<T, DL>(q, a.q + ((int64_t)b * a.S + (valid ? s : 0)) * a.ldq + (int64_t)h * HD + qd * DL, valid);
#pragma unroll
  for (int d = 0; d < DL; ++d) o[d] = 0.f;
  const T* kb = a.k + (int64_t)b * a.S * a.ldk + (int64_t)g * HD;
  const T* vb = a.v + (int64_t)b * a.S * a.ldv + (int64_t)g * HD;
  const int kv_end = min(a.S, qb * 64 + 64);
  const int last = valid ? s : -1;  // causal: keys 0 .. s
  float m = -INFINITY, l = 0.f;
  for (int c0 = 0; c0 < kv_end; c0 += 64) {
    const int n = min(64, kv_end - c0);
    __syncthreads();  // the previous chunk's reads are done
    stage_rows<T, HD>(ks, kb, a.ldk, c0, n, tid);
    stage_rows<T, HD>(vs, vb, a.ldv, c0, n, tid);
    __syncthreads();
    const int jn = min(n, last - c0 + 1);  // the same for the four lanes of a row
    for (int j = 0; j < jn; ++j) {
      const float sc = quad_sum(dot_part<DL>(q, ks + j * HD + qd * DL)) * a.scale;
      const float m_new = fmaxf(m, sc);
      const float corr = expf(m - m_new), p = expf(sc - m_new);
      l = l * corr + p;
      axpby_part<DL>(o, corr, p, vs + j * HD + qd * DL);
      m = m_new;
    }
  }
  if (valid) {
    T* op = a.o + ((int64_t)b * a.S + s) * a.ldo + (int64_t)h * HD + qd * DL;
    const float inv = 1.f / l;
#pragma unroll
    for (int d = 0; d < DL; ++d) Elem<T>::store(op, d, o[d] * inv);
    if (qd == 0) a.lse[((int64_t)b * a.H + h) * a.S + s] = m + logf(l);
  }
}

template <typename T, int HD>
__global__ void __launch_bounds__(256) attn_bwd_dq_quad_kernel(GenArgs<T> a) {
  constexpr int DL = HD / 4;
  __shared__ __attribute__((aligned(16))) float ks[64 * HD];
  __shared__ __attribute__((aligned(16))) float vs[64 * HD];
  const int tid = threadIdx.x, qd = tid & 3, rl = tid >> 2;
  const int nqb = (a.S + 63) / 64;
  const int qb = (int)(blockIdx.x % nqb);
  const int64_t bh = blockIdx.x / nqb;
  const int h = (int)(bh % a.H), b = (int)(bh / a.H);
  const int g = h / (a.H / a.KV);
  const int s = qb * 64 + rl;
  const bool valid = s < a.S;
  const int64_t row = (int64_t)b * a.S + (valid ? s : 0);
  float q[DL], dov[DL], acc[DL];
  load_part<T, DL>(q, a.q + row * a.ldq + (int64_t)h * HD + qd * DL, valid);
  load_part<T, DL>(dov, a.dout + row * a.lddo + (int64_t)h * HD + qd * DL, valid);
#pragma unroll
  for (int d = 0; d < DL; ++d) acc[d] = 0.f;
  const int64_t li = ((int64_t)b * a.H + h) * a.S + (valid ? s : 0);
  const float lse = a.lse[li], D = a.delta[li];
  const T* kb = a.k + (int64_t)b * a.S * a.ldk + (int64_t)g * HD;
  const T* vb = a.v + (int64_t)b * a.S * a.ldv + (int64_t)g * HD;
  const int kv_end = min(a.S, qb * 64 + 64);
  const int last = valid ? s : -1;
  for (int c0 = 0; c0 < kv_end; c0 += 64) {
    const int n = min(64, kv_end - c0);
    __syncthreads();
    stage_rows<T, HD>(ks, kb, a.ldk, c0, n, tid);
    stage_rows<T, HD>(vs, vb, a.ldv, c0, n, tid);
    __syncthreads();
    const int jn = min(n, last - c0 + 1);
    for (int j = 0; j < jn; ++j) {
      const float* kr = ks + j * HD + qd * DL;
      const float p = expf(quad_sum(dot_part<DL>(q, kr)) * a.scale - lse);
      const float ds = p * (quad_sum(dot_part<DL>(dov, vs + j * HD + qd * DL)) - D);
      axpby_part<DL>(acc, 1.f, ds, kr);
    }
  }
  if (valid) {
    T* dqp = a.dq + ((int64_t)b * a.S + s) * a.lddq + (int64_t)h * HD + qd * DL;
#pragma unroll
    for (int d = 0; d < DL; ++d) Elem<T>::store(dqp, d, acc[d] * a.scale);
  }
}

// grid: B * KV * ceil(S / 64) workgroups of 256; a quad owns one key row and
// sums over the queries of every head in its group
template <typename T, int HD>
__global__ void __launch_bounds__(256) attn_bwd_dkdv_quad_kernel(GenArgs<T> a) {
  constexpr int DL = HD / 4;
  __shared__ __attribute__((aligned(16))) float qs[64 * HD];
  __shared__ __attribute__((aligned(16))) float dos[64 * HD];
  __shared__ float ls[64], dl[64];
  const int tid = threadIdx.x, qd = tid & 3, rl = tid >> 2;
  const int nkb = (a.S + 63) / 64;
  const int kbk = (int)(blockIdx.x % nkb);
  const int64_t bg = blockIdx.x / nkb;
  const int g = (int)(bg % a.KV), b = (int)(bg / a.KV);
  const int rep = a.H / a.KV;
  const int kv = kbk * 64 + rl;
  const bool valid = kv < a.S;
  const int64_t row = (int64_t)b * a.S + (valid ? kv : 0);
  float kr[DL], vr[DL], dk[DL], dv[DL];
  load_part<T, DL>(kr, a.k + row * a.ldk + (int64_t)g * HD + qd * DL, valid);
  load_part<T, DL>(vr, a.v + row * a.ldv + (int64_t)g * HD + qd * DL, valid);
#pragma unroll
  for (int d = 0; d < DL; ++d) {
    dk[d] = 0.f;
    dv[d] = 0.f;
  }
  const int first = valid ? kv : a.S;  // causal: queries kv .. S-1
  for (int hq = 0; hq < rep; ++hq) {
    const int h = g * rep + hq;
    const T* qb = a.q + (int64_t)b * a.S * a.ldq + (int64_t)h * HD;
    const T* dob = a.dout + (int64_t)b * a.S * a.lddo + (int64_t)h * HD;
    const int64_t li0 = ((int64_t)b * a.H + h) * a.S;
    for (int c0 = kbk * 64; c0 < a.S; c0 += 64) {
      const int n = min(64, a.S - c0);
      __syncthreads();
      stage_rows<T, HD>(qs, qb, a.ldq, c0, n, tid);
      stage_rows<T, HD>(dos, dob, a.lddo, c0, n, tid);
      if (tid < 64) {
        const int lr = min(tid, n - 1);
        const float lv = a.lse[li0 + c0 + lr], dvv = a.delta[li0 + c0 + lr];
        ls[tid] = lv;
        dl[tid] = dvv;
      }
      __syncthreads();
      for (int j = max(0, first - c0); j < n; ++j) {
        const float* qr = qs + j * HD + qd * DL;
        const float* dr = dos + j * HD + qd * DL;
        const float p = expf(quad_sum(dot_part<DL>(kr, qr)) * a.scale - ls[j]);
        const float ds = p * (quad_sum(dot_part<DL>(vr, dr)) - dl[j]);
        axpby_part<DL>(dv, 1.f, p, dr);
        axpby_part<DL>(dk, 1.f, ds, qr);
      }
    }
  }
  if (valid) {
    T* dkp = a.dk + row * a.lddk + (int64_t)g * HD + qd * DL;
    T* dvp = a.dv + row * a.lddv + (int64_t)g * HD + qd * DL;
#pragma unroll
    for (int d = 0; d < DL; ++d) {
      Elem<T>::store(dkp, d, dk[d] * a.scale);
      Elem<T>::store(dvp, d, dv[d]);
    }
  }
}

template <typename T>
void launch_fwd_small(const GenArgs<T>& a, hipStream_t s) {
  const unsigned grid = (unsigned)((int64_t)a.B * a.H * ((a.S + 63) / 64));
  if (a.hd == 16) attn_fwd_quad_kernel<T, 16><<<grid, 256, 0, s>>>(a);
  else attn_fwd_quad_kernel<T, 32><<<grid, 256, 0, s>>>(a);
}

template <typename T>
void launch_bwd_small(const GenArgs<T>& a, hipStream_t s) {
  const unsigned grid_q = (unsigned)((int64_t)a.B * a.H * ((a.S + 63) / 64));
  const unsigned grid_kv = (unsigned)((int64_t)a.B * a.KV * ((a.S + 63) / 64));
  if (a.hd == 16) {
    attn_bwd_dq_quad_kernel<T, 16><<<grid_q, 256, 0, s>>>(a);
    attn_bwd_dkdv_quad_kernel<T, 16><<<grid_kv, 256, 0, s>>>(a);
  } else {
    attn_bwd_dq_quad_kernel<T, 32><<<grid_q, 256, 0, s>>>(a);
    attn_bwd_dkdv_quad_kernel<T, 32><<<grid_kv, 256, 0, s>>>(a);
  }
}

// The tile loads address a tile's rows by 32-bit byte offsets from its first
// row: row strides below 2^22 elements keep a 64-row tile below 2^31 bytes.
constexpr int64_t kMaxTileLd = 1ll << 22;

bool strides_ok(int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo) {
  return ldq % 8 == 0 && ldk % 8 == 0 && ldv % 8 == 0 && ldo % 4 == 0 && ldq < kMaxTileLd && ldk < kMaxTileLd &&
         ldv < kMaxTileLd && ldo < kMaxTileLd;
}

bool mfma_ok(int dtype, int64_t hd, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, const void* q, const void* k,
             const void* v, const void* o) {
  return (dtype == LZ_BF16 || dtype == LZ_F16) && (hd == 64 || hd == 128) && strides_ok(ldq, ldk, ldv, ldo) &&
         lz_aligned16(q) && lz_aligned16(k) && lz_aligned16(v) && (reinterpret_cast<uintptr_t>(o) & 7) == 0;
}

int check_shape(int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd) {
  LZ_REQUIRE(B > 0 && S > 0 && H > 0 && KV > 0 && hd > 0, "attention: bad shape");
  LZ_REQUIRE(H % KV == 0, "attention: H (%lld) must be a multiple of KV (%lld)", (long long)H, (long long)KV);
  LZ_REQUIRE(hd <= 64 * kGenMax, "attention: head dim %lld > %d", (long long)hd, 64 * kGenMax);
  LZ_REQUIRE(B * H * lz_cdiv(S, 64) < (1ll << 31) && S < (1 << 30), "attention: problem too large");
  return LZ_OK;
}

LzWaveArgs wave_fwd_args(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, void* o,
                         int64_t ldo, float* lse, int64_t B, int64_t S, int64_t H, int64_t KV, float scale) {
  LzWaveArgs a{};
  a.q = q; a.k = k; a.v = v;
  a.ldq = ldq; a.ldk = ldk; a.ldv = ldv;
  a.o = o; a.ldo = ldo; a.lse = lse;
  a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.scale = scale;
  return a;
}

void wave_bwd_args(LzWaveArgs& a, const void* dout, int64_t lddo, const float* delta, void* dq, int64_t lddq, void* dk,
                   int64_t lddk, void* dv, int64_t lddv) {
  a.dout = dout; a.lddo = lddo; a.delta = delta;
  a.dq = dq; a.dk = dk; a.dv = dv;
  a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
}

// Where the tile kernels' workgroups are too few to fill the chip the
// wave-private kernels (a quarter or an eighth of the rows per workgroup, the
// other side split over its waves) are faster.  A tile kernel's time is one
// workgroup's chain of steps until its workgroups (`wgs`) fill the CUs; the
// wave kernels cut that chain and grow with the work.  So the line is a share
// of the CUs that rises with the steps of the chain: 64-key steps for the
// forward and dQ, for dK/dV the 64-query steps over every query head of the
// group, against its 32-key blocks in units of a tile workgroup's eight.
// Lines from both sides over B 1..32, S 32..2048 (whole and ragged), heads 12/4,
// 32/8, 8/8 of 64 and 16/8, 32/8, 32/32 of 128: over those 244 calls the rules
// are within 0.1 % (forward), 0.4 % (dQ) and 0.5 % (dK/dV) of the faster kernel
// in the geometric mean.  us, tile / wave:
//   forward, hd 64: 96 workgroups S 256 6.5 / 8.0, S 512 9.7 / 8.6, 192 S 1024
//     16.1 / 18.2, S 2048 27.9 / 26.7; hd 128: 64 S 192 7.0 / 8.5, S 512 13.2 / 11.4,
//     112 S 777 19.1 / 18.6, 128 S 1024 22.7 / 24.2
//   dQ, hd 64: 48 S 64 5.5 / 6.9, 96 S 512 11.3 / 13.9, S 1024 17.4 / 14.7, 192 S 2048
//     29.9 / 31.3; hd 128: 96 S 333 15.1 / 16.6, 112 S 777 25.1 / 22.5
//   dK/dV, hd 64, heads 8/8: 128 workgroups S 512 21.2 / 24.6, S 1024 35.5 / 31.9; heads
//     32/8: 128 S 2048 243 / 122, 256 S 2048 236 / 238; hd 128, heads 32/32: 64 S 256
//     23.6 / 18.3, 128 S 512 36.4 / 44.6, S 500 45.9 / 45.0; heads 16/8: 128 S 512 57.8 /
//     62.9, S 2048 193 / 169; heads of 128 at ragged lengths spill in the tile
//     kernel (16/8, S 777: 110 / 69)
bool wave_fwd_better(int64_t hd, int64_t S, int64_t wgs) {
  const double steps = (double)lz_cdiv(S, 64), share = (double)wgs / lz_num_cus();
  if (hd == 64) return steps >= 2 && share <= std::max(0.28, 0.9 - 2.5 / steps);
  return steps >= 4 && share <= 0.525 - 1.05 / steps;
}
bool wave_dq_better(int64_t S, int64_t wgs) {
  const double steps = (double)lz_cdiv(S, 64), share = (double)wgs / lz_num_cus();
  return steps >= 2 && share <= std::min(0.21 + 0.02 * steps, 0.55);
}
bool wave_dkdv_better(int64_t hd, int64_t S, int64_t pairs, int64_t rep) {  // pairs: B * KV
  const double cus = lz_num_cus(), steps = std::log2((double)(rep * lz_cdiv(S, 64)));
  if (pairs * lz_cdiv(S, 256) >= cus) return false;
  const double line = hd == 64 ? 0.04 + 0.12 * steps : (0.14 + 0.072 * steps) * (S % 64 ? 1.5 : 1.0);
  return pairs * lz_cdiv(S, 32) / 8.0 <= cus * std::max(0.125, line);
}

// The forward of 16-bit causal attention with head dim 64 or 128 (aligned as
// mfma_ok asks; fp16: S a multiple of 64).
int tiles_fwd(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, void* o, int64_t ldo,
              float* lse, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale, int dtype,
              hipStream_t s) {
  const int64_t grid = lz_cdiv(S, 128) * B * H;
  if (dtype == LZ_BF16 && wave_fwd_better(hd, S, grid)) {
    const LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, scale);
    if (lz_attn_wave_ok(w, dtype, hd, false)) return lz_attn_wave_pass(w, dtype, hd, kWaveRounded, kWaveFwd, s);
  }
  AttnArgs a{};
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
  a.ldq = ldq; a.ldk = ldk; a.ldv = ldv;
  a.o = (uint16_t*)o; a.ldo = ldo; a.lse = lse;
  a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.scale = scale;
  const unsigned g = (unsigned)grid;
  if (dtype == LZ_F16) {
    if (hd == 128) attn_fwd_tile_kernel<128, FmtF16><<<g, 256, 0, s>>>(a);
    else attn_fwd_tile_kernel<64, FmtF16><<<g, 256, 0, s>>>(a);
  } else if (S % 64) {
    if (hd == 128) attn_fwd_tile_kernel<128, FmtBF16, true><<<g, 256, 0, s>>>(a);
    else attn_fwd_tile_kernel<64, FmtBF16, true><<<g, 256, 0, s>>>(a);
  } else {
    if (hd == 128) attn_fwd_tile_kernel<128, FmtBF16><<<g, 256, 0, s>>>(a);
    else attn_fwd_tile_kernel<64, FmtBF16><<<g, 256, 0, s>>>(a);
  }
  return lz_check_launch("lz_attn_fwd");
}

template <int HD, typename F, bool kRagged>
void launch_dq_tiles(const AttnArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)(lz_cdiv(a.S, 128) * a.B * a.H);
  if (a.delta_w) attn_bwd_dq_tile_kernel<HD, F, true, kRagged><<<grid, 256, 0, s>>>(a);
  else attn_bwd_dq_tile_kernel<HD, F, false, kRagged><<<grid, 256, 0, s>>>(a);
}

template <int HD, typename F, bool kRagged>
void launch_dkdv_tiles(const AttnArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)(lz_cdiv(a.S, 256) * a.B * a.KV);
  attn_bwd_dkdv_wide_kernel<HD, F, kRagged><<<grid, 512, 0, s>>>(a);
}

// Its backward, with delta given or (delta_w) formed from o.
int tiles_bwd(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, const void* dout,
              int64_t lddo, const float* lse, const float* delta, void* dq, int64_t lddq, void* dk, int64_t lddk,
              void* dv, int64_t lddv, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale,
              const void* rope_cos, const void* rope_sin, int dtype, hipStream_t s, bool& rope_done, const void* o,
              int64_t ldo, float* delta_w) {
  AttnArgs a{};
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
  a.ldq = ldq; a.ldk = ldk; a.ldv = ldv;
  a.lse = const_cast<float*>(lse);
  a.dout = (const uint16_t*)dout; a.lddo = lddo;
  a.o = (uint16_t*)const_cast<void*>(o); a.ldo = ldo;
  a.delta_w = delta_w; a.delta = delta_w ? delta_w : delta;
  a.dq = (uint16_t*)dq; a.dk = (uint16_t*)dk; a.dv = (uint16_t*)dv;
  a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
  a.rcos = (const uint16_t*)rope_cos; a.rsin = (const uint16_t*)rope_sin;
  a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.scale = scale;
  LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, const_cast<void*>(o), ldo, const_cast<float*>(lse), B, S, H, KV,
                               scale);
  wave_bwd_args(w, dout, lddo, delta, dq, lddq, dk, lddk, dv, lddv);
  w.delta_w = delta_w;
  // dout rows at 8 bytes (a slice of a flat gradient): at lengths the tiles do
  // not divide they keep to kernels that load them through registers, as the
  // direct-to-LDS copies are made for 16-byte rows
  const bool dout8 = dtype == LZ_BF16 && S % 64 && !(lz_aligned16(dout) && lddo % 8 == 0);
  const bool can_wave = dtype == LZ_BF16 && lz_attn_wave_ok(w, dtype, hd, true, dout8);
  const bool wave_dq = can_wave && (dout8 || wave_dq_better(S, lz_cdiv(S, 128) * B * H));
  const bool wave_dkdv = can_wave && (dout8 || wave_dkdv_better(hd, S, B * KV, H / KV));
  rope_done = !wave_dq && !wave_dkdv;  // only the tile kernels rotate; the caller rotates after the others
  if (!rope_done) a.rcos = a.rsin = nullptr;
  // dQ first: it forms the delta that dK/dV reads when delta_w is set
  if (wave_dq) {
    const int rc = lz_attn_wave_pass(w, dtype, hd, kWaveRounded, kWaveDq, s);
    if (rc) return rc;
  } else if (dtype == LZ_F16) {
    if (hd == 128) launch_dq_tiles<128, FmtF16, false>(a, s);
    else launch_dq_tiles<64, FmtF16, false>(a, s);
  } else if (S % 64) {
    if (hd == 128) launch_dq_tiles<128, FmtBF16, true>(a, s);
    else launch_dq_tiles<64, FmtBF16, true>(a, s);
  } else {
    if (hd == 128) launch_dq_tiles<128, FmtBF16, false>(a, s);
    else launch_dq_tiles<64, FmtBF16, false>(a, s);
  }
  int rc = lz_check_launch("lz_attn_bwd");
  if (rc) return rc;
  if (wave_dkdv) {
    if (delta_w) w.delta = delta_w;
    return lz_attn_wave_pass(w, dtype, hd, kWaveRounded, kWaveDkdv, s);
  }
  if (dtype == LZ_F16) {
    if (hd == 128) launch_dkdv_tiles<128, FmtF16, false>(a, s);
    else launch_dkdv_tiles<64, FmtF16, false>(a, s);
  } else if (S % 64) {
    if (hd == 128) launch_dkdv_tiles<128, FmtBF16, true>(a, s);
    else launch_dkdv_tiles<64, FmtBF16, true>(a, s);
  } else {
    if (hd == 128) launch_dkdv_tiles<128, FmtBF16, false>(a, s);
    else launch_dkdv_tiles<64, FmtBF16, false>(a, s);
  }
  return lz_check_launch("lz_attn_bwd");
}

}  // namespace

// What lz_attn_fwd/bwd take for these arguments: 2 = MFMA on LDS tiles (S a
// multiple of 64), 1 = bf16 and the same head dims at other lengths, 0 = the
// rest.
LZ_EXPORT int lz_attn_path(int dtype, int64_t S, int64_t hd, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo) {
  const bool mfma = (dtype == LZ_BF16 || (dtype == LZ_F16 && S % 64 == 0)) && (hd == 64 || hd == 128) &&
                    strides_ok(ldq, ldk, ldv, ldo);
  return mfma ? (S % 64 == 0 ? 2 : 1) : 0;
}

// Which passes of causal attention on 16-byte aligned rows the tile kernels
// run: 1 forward, 2 dQ, 4 dK/dV (the others are wave-private or generic).
// Host only: attributes timings, and tests assert what they reach.
LZ_EXPORT int lz_attn_tiles(int dtype, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd) {
  if (B <= 0 || S <= 0 || KV <= 0 || H <= 0 || H % KV || (hd != 64 && hd != 128)) return 0;
  if (dtype == LZ_F16) return S % 64 ? 0 : 7;
  if (dtype != LZ_BF16) return 0;
  const int64_t wgs = lz_cdiv(S, 128) * B * H;
  return (wave_fwd_better(hd, S, wgs) ? 0 : 1) | (wave_dq_better(S, wgs) ? 0 : 2) |
         (wave_dkdv_better(hd, S, B * KV, H / KV) ? 0 : 4);
}

// Forward.  vt is ignored (no kernel reads a transposed operand).
LZ_EXPORT int lz_attn_fwd(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                          const void* /*vt*/, void* o, int64_t ldo, float* lse, int64_t B, int64_t S, int64_t H,
                          int64_t KV, int64_t hd, float scale, int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && o && lse, "lz_attn_fwd: null pointer");
  hipStream_t s = lz_stream(stream);
  const bool mfma = mfma_ok(dtype, hd, ldq, ldk, ldv, ldo, q, k, v, o);
  if (mfma && (dtype == LZ_BF16 || S % 64 == 0))
    return tiles_fwd(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, hd, scale, dtype, s);
  const LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, scale);
  if (lz_attn_wave_ok(w, dtype, hd, false)) return lz_attn_wave_pass(w, dtype, hd, kWaveSplit, kWaveFwd, s);
  const unsigned grid = (unsigned)lz_cdiv(B * H * S, 4);
  if (dtype == LZ_BF16) {
    GenArgs<uint16_t> a{};
    a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.o = (uint16_t*)o; a.ldo = ldo; a.lse = lse;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) launch_fwd_small(a, s);
    else attn_fwd_generic_kernel<uint16_t><<<grid, 256, 0, s>>>(a);
  } else if (dtype == LZ_F16) {
    GenArgs<_Float16> a{};
    a.q = (const _Float16*)q; a.k = (const _Float16*)k; a.v = (const _Float16*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.o = (_Float16*)o; a.ldo = ldo; a.lse = lse;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) launch_fwd_small(a, s);
    else attn_fwd_generic_kernel<_Float16><<<grid, 256, 0, s>>>(a);
  } else if (dtype == LZ_F32) {
    GenArgs<float> a{};
    a.q = (const float*)q; a.k = (const float*)k; a.v = (const float*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.o = (float*)o; a.ldo = ldo; a.lse = lse;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) launch_fwd_small(a, s);
    else attn_fwd_generic_kernel<float><<<grid, 256, 0, s>>>(a);
  } else {
    return lz_set_error(LZ_EINVAL, "lz_attn_fwd: bad dtype %d", dtype);
  }
  return lz_check_launch("lz_attn_fwd(generic)");
}

LZ_EXPORT int lz_attn_delta(const void* o, int64_t ldo, const void* dout, int64_t lddo, float* delta, int64_t B, int64_t S,
                            int64_t H, int64_t hd, int dtype, void* stream) {
  LZ_REQUIRE(B > 0 && S > 0 && H > 0 && hd > 0 && delta, "lz_attn_delta: bad arguments");
  const unsigned grid = (unsigned)lz_cdiv(B * S * H, 4);
  hipStream_t s = lz_stream(stream);
  const int64_t rows = B * S * H;
  const bool vec = dtype == LZ_BF16 && (hd == 32 || hd == 64 || hd == 128 || hd == 256) && lz_aligned16(o) &&
                   lz_aligned16(dout) && ldo % 8 == 0 && lddo % 8 == 0 && rows * (hd / 8) < (1ll << 31);
  if (vec) {
    const unsigned vgrid = (unsigned)lz_cdiv(rows * (hd / 8), 256);
    const uint16_t *o16 = (const uint16_t*)o, *d16 = (const uint16_t*)dout;
    if (hd == 32) attn_delta_vec_kernel<4><<<vgrid, 256, 0, s>>>(o16, ldo, d16, lddo, delta, (int)S, (int)H, (int)rows);
    else if (hd == 64) attn_delta_vec_kernel<8><<<vgrid, 256, 0, s>>>(o16, ldo, d16, lddo, delta, (int)S, (int)H, (int)rows);
    else if (hd == 128) attn_delta_vec_kernel<16><<<vgrid, 256, 0, s>>>(o16, ldo, d16, lddo, delta, (int)S, (int)H, (int)rows);
    else attn_delta_vec_kernel<32><<<vgrid, 256, 0, s>>>(o16, ldo, d16, lddo, delta, (int)S, (int)H, (int)rows);
  } else if (dtype == LZ_BF16)
    attn_delta_kernel<uint16_t><<<grid, 256, 0, s>>>((const uint16_t*)o, ldo, (const uint16_t*)dout, lddo, delta, (int)B, (int)S, (int)H, (int)hd);
  else if (dtype == LZ_F32)
    attn_delta_kernel<float><<<grid, 256, 0, s>>>((const float*)o, ldo, (const float*)dout, lddo, delta, (int)B, (int)S, (int)H, (int)hd);
  else if (dtype == LZ_F16)
    attn_delta_kernel<_Float16><<<grid, 256, 0, s>>>((const _Float16*)o, ldo, (const _Float16*)dout, lddo, delta, (int)B, (int)S, (int)H, (int)hd);
  else
    return lz_set_error(LZ_EINVAL, "lz_attn_delta: bad dtype %d", dtype);
  return lz_check_launch("lz_attn_delta");
}

LZ_EXPORT int lz_rope(void* x, int dtype, int64_t ld, int64_t rows, int64_t seq, int64_t nheads, int64_t hd,
                      const void* cos_t, const void* sin_t, int64_t pos_offset, int backward, void* stream);

namespace {

int attn_bwd_impl(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, const void* dout,
                  int64_t lddo, const float* lse, const float* delta, void* dq, int64_t lddq, void* dk, int64_t lddk,
                  void* dv, int64_t lddv, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale, const void* rope_cos, const void* rope_sin,
                  int dtype, hipStream_t s, bool& rope_done, const void* o = nullptr, int64_t ldo = 0,
                  float* delta_w = nullptr);

}  // namespace

// Backward.  qt, kt and dot are ignored (no kernel reads a transposed
// operand); delta comes from lz_attn_delta.  dq/dk/dv are written (not
// accumulated).  rope_cos/rope_sin (both or neither; tables [>= S, hd] in the
// activation dtype, row = position, as lz_rope takes): dq and dk come back
// as the gradients of q and k before RoPE, i.e. with lz_rope's backward
// already applied (in the bf16 MFMA kernels' epilogue, otherwise by lz_rope
// after them).
LZ_EXPORT int lz_attn_bwd(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                          const void* dout, int64_t lddo, const float* lse, const float* delta, const void* /*qt*/,
                          const void* /*kt*/, const void* /*dot*/, void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv,
                          int64_t lddv, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale,
                          const void* rope_cos, const void* rope_sin, int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && dout && lse && delta && dq && dk && dv, "lz_attn_bwd: null pointer");
  LZ_REQUIRE((rope_cos == nullptr) == (rope_sin == nullptr), "lz_attn_bwd: give both RoPE tables or neither");
  LZ_REQUIRE(rope_cos == nullptr || (hd % 2 == 0 && ((reinterpret_cast<uintptr_t>(rope_cos) |
                                                        reinterpret_cast<uintptr_t>(rope_sin)) & 7) == 0),
             "lz_attn_bwd: RoPE needs an even head dim and 8-byte aligned tables");
  hipStream_t s = lz_stream(stream);
  bool rope_done = false;
  rc = attn_bwd_impl(q, ldq, k, ldk, v, ldv, dout, lddo, lse, delta, dq, lddq, dk, lddk, dv, lddv, B, S, H, KV, hd,
                     scale, rope_cos, rope_sin, dtype, s, rope_done);
  if (rc || rope_cos == nullptr || rope_done) return rc;
  rc = lz_rope(dq, dtype, lddq, B * S, S, H, hd, rope_cos, rope_sin, 0, 1, stream);
  if (rc) return rc;
  return lz_rope(dk, dtype, lddk, B * S, S, KV, hd, rope_cos, rope_sin, 0, 1, stream);
}

// lz_attn_delta + lz_attn_bwd in one call for the LDS-tile kernels
// (lz_attn_path 2): the dQ kernel computes delta = rowsum(dO * O) from the
// dO rows it loads anyway and writes it to `delta` ([B, H, S] fp32, output),
// then the dK/dV kernel reads it.  Other shapes are refused.
LZ_EXPORT int lz_attn_bwd_with_o(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                                 const void* o, int64_t ldo, const void* dout, int64_t lddo, const float* lse,
                                 float* delta, void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv, int64_t lddv,
                                 int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale,
                                 const void* rope_cos, const void* rope_sin, int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && o && dout && lse && delta && dq && dk && dv, "lz_attn_bwd_with_o: null pointer");
  LZ_REQUIRE(lz_aligned16(o) && ldo % 8 == 0 && ldo >= H * hd, "lz_attn_bwd_with_o: O rows must be 16-byte aligned");
  LZ_REQUIRE((rope_cos == nullptr) == (rope_sin == nullptr), "lz_attn_bwd_with_o: give both RoPE tables or neither");
  LZ_REQUIRE(rope_cos == nullptr || (hd % 2 == 0 && ((reinterpret_cast<uintptr_t>(rope_cos) |
                                                        reinterpret_cast<uintptr_t>(rope_sin)) & 7) == 0),
             "lz_attn_bwd_with_o: RoPE needs an even head dim and 8-byte aligned tables");
  bool rope_done = false;
  rc = attn_bwd_impl(q, ldq, k, ldk, v, ldv, dout, lddo, lse, delta, dq, lddq, dk, lddk, dv, lddv, B, S, H, KV, hd,
                     scale, rope_cos, rope_sin, dtype, lz_stream(stream), rope_done, o, ldo, delta);
  if (rc || rope_cos == nullptr || rope_done) return rc;
  rc = lz_rope(dq, dtype, lddq, B * S, S, H, hd, rope_cos, rope_sin, 0, 1, stream);
  if (rc) return rc;
  return lz_rope(dk, dtype, lddk, B * S, S, KV, hd, rope_cos, rope_sin, 0, 1, stream);
}

namespace {

int attn_bwd_impl(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv, const void* dout,
                  int64_t lddo, const float* lse, const float* delta, void* dq, int64_t lddq, void* dk, int64_t lddk,
                  void* dv, int64_t lddv, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale, const void* rope_cos, const void* rope_sin,
                  int dtype, hipStream_t s, bool& rope_done, const void* o, int64_t ldo, float* delta_w) {
  const bool mfma = mfma_ok(dtype, hd, ldq, ldk, ldv, lddo, q, k, v, dout) && lddq % 4 == 0 && lddk % 4 == 0 &&
                    lddv % 4 == 0;
  LZ_REQUIRE(delta_w == nullptr || (mfma && S % 64 == 0),
             "lz_attn_bwd_with_o: this shape takes the other kernels (use lz_attn_delta + lz_attn_bwd)");
  if (mfma && (dtype == LZ_BF16 || S % 64 == 0))
    return tiles_bwd(q, ldq, k, ldk, v, ldv, dout, lddo, lse, delta, dq, lddq, dk, lddk, dv, lddv, B, S, H, KV, hd,
                     scale, rope_cos, rope_sin, dtype, s, rope_done, o, ldo, delta_w);
  LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, nullptr, 0, const_cast<float*>(lse), B, S, H, KV, scale);
  wave_bwd_args(w, dout, lddo, delta, dq, lddq, dk, lddk, dv, lddv);
  if (lz_attn_wave_ok(w, dtype, hd, true)) return lz_attn_wave_bwd(w, dtype, hd, kWaveSplit, s);
  const unsigned grid_q = (unsigned)lz_cdiv(B * H * S, 4);
  const unsigned grid_kv = (unsigned)lz_cdiv(B * KV * S, 4);
  if (dtype == LZ_BF16) {
    GenArgs<uint16_t> a{};
    a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.lse = const_cast<float*>(lse);
    a.dout = (const uint16_t*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (uint16_t*)dq; a.dk = (uint16_t*)dk; a.dv = (uint16_t*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) {
      launch_bwd_small(a, s);
    } else {
      attn_bwd_dq_generic_kernel<uint16_t><<<grid_q, 256, 0, s>>>(a);
      attn_bwd_dkdv_generic_kernel<uint16_t><<<grid_kv, 256, 0, s>>>(a);
    }
  } else if (dtype == LZ_F16) {
    GenArgs<_Float16> a{};
    a.q = (const _Float16*)q; a.k = (const _Float16*)k; a.v = (const _Float16*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.lse = const_cast<float*>(lse);
    a.dout = (const _Float16*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (_Float16*)dq; a.dk = (_Float16*)dk; a.dv = (_Float16*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) {
      launch_bwd_small(a, s);
    } else {
      attn_bwd_dq_generic_kernel<_Float16><<<grid_q, 256, 0, s>>>(a);
      attn_bwd_dkdv_generic_kernel<_Float16><<<grid_kv, 256, 0, s>>>(a);
    }
  } else if (dtype == LZ_F32) {
    GenArgs<float> a{};
    a.q = (const float*)q; a.k = (const float*)k; a.v = (const float*)v;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.lse = const_cast<float*>(lse);
    a.dout = (const float*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (float*)dq; a.dk = (float*)dk; a.dv = (float*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
    if (hd == 16 || hd == 32) {
      launch_bwd_small(a, s);
    } else {
      attn_bwd_dq_generic_kernel<float><<<grid_q, 256, 0, s>>>(a);
      attn_bwd_dkdv_generic_kernel<float><<<grid_kv, 256, 0, s>>>(a);
    }
  } else {
    return lz_set_error(LZ_EINVAL, "lz_attn_bwd: bad dtype %d", dtype);
  }
  return lz_check_launch("lz_attn_bwd(generic)");
}

}  // namespace

namespace {

template <class A>
void general_args(A& a, const void* mask, int mask_kind, const int64_t* mstride, float dropout_p, uint64_t seed) {
  a.mask = mask; a.mask_kind = mask_kind;
  if (mask_kind) {
    a.msb = mstride[0]; a.msh = mstride[1]; a.msq = mstride[2]; a.msk = mstride[3];
  }
  a.drop_thresh = (uint32_t)std::min(std::ceil((double)dropout_p * 16777216.0), 16777216.0);
  a.drop_scale = dropout_p < 1.f ? 1.0f / (1.0f - dropout_p) : 0.f;
  a.drop_seed = seed;
}

template <typename T>
void general_args(GenArgs<T>& a, const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                 const void* mask, int mask_kind, const int64_t* mstride, float dropout_p, uint64_t seed, int64_t B,
                 int64_t S, int64_t H, int64_t KV, int64_t hd, float scale) {
  a.q = (const T*)q; a.k = (const T*)k; a.v = (const T*)v;
  a.ldq = ldq; a.ldk = ldk; a.ldv = ldv;
  a.B = (int)B; a.S = (int)S; a.H = (int)H; a.KV = (int)KV; a.hd = (int)hd; a.scale = scale;
  general_args(a, mask, mask_kind, mstride, dropout_p, seed);
}

int check_general(const void* mask, int mask_kind, const int64_t* mstride, float dropout_p) {
  LZ_REQUIRE(mask_kind >= 0 && mask_kind <= 4, "attention mask: kind %d (0 causal, 1 bool, 2 fp32, 3 bf16, 4 fp16)",
             mask_kind);
  if (mask_kind) {
    LZ_REQUIRE(mask && mstride, "attention mask: null pointer");
    for (int i = 0; i < 4; ++i) LZ_REQUIRE(mstride[i] >= 0, "attention mask: negative stride");
  }
  LZ_REQUIRE(dropout_p >= 0.f && dropout_p <= 1.f, "attention dropout p %g not in [0, 1]", (double)dropout_p);
  return LZ_OK;
}

}  // namespace

// Attention with the options the tile paths do not take, on the wave-private
// kernels (attn_wave.hip; other head dims and unaligned rows: one wave per
// row) (model/llama.py:109-117, F.scaled_dot_product_attention):
//   - an explicit mask in place of the causal one (attn_mask with
//     is_causal=False): mask_kind 1 = bool bytes (nonzero: the key takes
//     part), 2 = fp32, 3 = bf16, 4 = fp16 (added to the scaled scores); mstride = its
//     element strides over [B, H, S(query), S(key)], 0 where it broadcasts;
//     mask_kind 0 = causal (mask and mstride ignored).  A row whose keys are
//     all masked gives NaN, as the reference's softmax of an all -inf row does;
//   - attention dropout (dropout_p): each probability kept with scale
//     1/(1-p) by element ((b*H + h)*S + s)*S + kv of seed's stream (the
//     stream lz_dropout uses), the normaliser summing them before dropout.
// Any head dim up to 256, any dtype.
LZ_EXPORT int lz_attn_fwd_general(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                                  const void* mask, int mask_kind, const int64_t* mstride, float dropout_p,
                                  uint64_t seed, void* o, int64_t ldo, float* lse, int64_t B, int64_t S, int64_t H,
                                  int64_t KV, int64_t hd, float scale, int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  rc = check_general(mask, mask_kind, mstride, dropout_p);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && o && lse, "lz_attn_fwd_general: null pointer");
  hipStream_t s = lz_stream(stream);
  LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, scale);
  if (lz_attn_wave_ok(w, dtype, hd, false)) {
    general_args(w, mask, mask_kind, mstride, dropout_p, seed);
    return lz_attn_wave_pass(w, dtype, hd, kWaveGeneral, kWaveFwd, s);
  }
  const unsigned grid = (unsigned)lz_cdiv(B * H * S, 4);
  if (dtype == LZ_BF16) {
    GenArgs<uint16_t> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.o = (uint16_t*)o; a.ldo = ldo; a.lse = lse;
    attn_fwd_generic_kernel<uint16_t><<<grid, 256, 0, s>>>(a);
  } else if (dtype == LZ_F16) {
    GenArgs<_Float16> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.o = (_Float16*)o; a.ldo = ldo; a.lse = lse;
    attn_fwd_generic_kernel<_Float16><<<grid, 256, 0, s>>>(a);
  } else if (dtype == LZ_F32) {
    GenArgs<float> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.o = (float*)o; a.ldo = ldo; a.lse = lse;
    attn_fwd_generic_kernel<float><<<grid, 256, 0, s>>>(a);
  } else {
    return lz_set_error(LZ_EINVAL, "lz_attn_fwd_general: bad dtype %d", dtype);
  }
  return lz_check_launch("lz_attn_fwd_general");
}

// Backward of lz_attn_fwd_general (same mask, dropout p and seed); delta
// from lz_attn_delta.
LZ_EXPORT int lz_attn_bwd_general(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                                  const void* dout, int64_t lddo, const float* lse, const float* delta,
                                  const void* mask, int mask_kind, const int64_t* mstride, float dropout_p,
                                  uint64_t seed, void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv,
                                  int64_t lddv, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale,
                                  int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  rc = check_general(mask, mask_kind, mstride, dropout_p);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && dout && lse && delta && dq && dk && dv, "lz_attn_bwd_general: null pointer");
  hipStream_t s = lz_stream(stream);
  LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, nullptr, 0, const_cast<float*>(lse), B, S, H, KV, scale);
  wave_bwd_args(w, dout, lddo, delta, dq, lddq, dk, lddk, dv, lddv);
  if (lz_attn_wave_ok(w, dtype, hd, true)) {
    general_args(w, mask, mask_kind, mstride, dropout_p, seed);
    return lz_attn_wave_bwd(w, dtype, hd, kWaveGeneral, s);
  }
  const unsigned grid_q = (unsigned)lz_cdiv(B * H * S, 4);
  const unsigned grid_kv = (unsigned)lz_cdiv(B * KV * S, 4);
  if (dtype == LZ_BF16) {
    GenArgs<uint16_t> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.lse = const_cast<float*>(lse); a.dout = (const uint16_t*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (uint16_t*)dq; a.dk = (uint16_t*)dk; a.dv = (uint16_t*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    attn_bwd_dq_generic_kernel<uint16_t><<<grid_q, 256, 0, s>>>(a);
    attn_bwd_dkdv_generic_kernel<uint16_t><<<grid_kv, 256, 0, s>>>(a);
  } else if (dtype == LZ_F16) {
    GenArgs<_Float16> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.lse = const_cast<float*>(lse); a.dout = (const _Float16*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (_Float16*)dq; a.dk = (_Float16*)dk; a.dv = (_Float16*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    attn_bwd_dq_generic_kernel<_Float16><<<grid_q, 256, 0, s>>>(a);
    attn_bwd_dkdv_generic_kernel<_Float16><<<grid_kv, 256, 0, s>>>(a);
  } else if (dtype == LZ_F32) {
    GenArgs<float> a{};
    general_args(a, q, ldq, k, ldk, v, ldv, mask, mask_kind, mstride, dropout_p, seed, B, S, H, KV, hd, scale);
    a.lse = const_cast<float*>(lse); a.dout = (const float*)dout; a.lddo = lddo; a.delta = delta;
    a.dq = (float*)dq; a.dk = (float*)dk; a.dv = (float*)dv; a.lddq = lddq; a.lddk = lddk; a.lddv = lddv;
    attn_bwd_dq_generic_kernel<float><<<grid_q, 256, 0, s>>>(a);
    attn_bwd_dkdv_generic_kernel<float><<<grid_kv, 256, 0, s>>>(a);
  } else {
    return lz_set_error(LZ_EINVAL, "lz_attn_bwd_general: bad dtype %d", dtype);
  }
  return lz_check_launch("lz_attn_bwd_general");
}

// Whether lz_attn_fwd_direct / lz_attn_bwd_direct take these shapes: head dim
// 32, 64 or 128, row strides of whole 16-byte pieces.
LZ_EXPORT int lz_attn_direct(int dtype, int64_t hd, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo) {
  const int64_t rd = dtype == LZ_F32 ? 4 : 8;
  return (dtype == LZ_BF16 || dtype == LZ_F16 || dtype == LZ_F32) && (hd == 32 || hd == 64 || hd == 128) &&
         ldq % rd == 0 && ldk % rd == 0 && ldv % rd == 0 && ldo % rd == 0;
}

// Causal attention of any sequence length that reads q, k and v (and o and
// dout in the backward) as they are stored: no transposed copies and no
// separate delta pass (the backward writes delta [B, H, S], which it forms
// from o and dout).  Shapes outside lz_attn_direct and unaligned pointers
// are refused.
LZ_EXPORT int lz_attn_fwd_direct(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                                 void* o, int64_t ldo, float* lse, int64_t B, int64_t S, int64_t H, int64_t KV,
                                 int64_t hd, float scale, int dtype, void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && o && lse, "lz_attn_fwd_direct: null pointer");
  const LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, scale);
  LZ_REQUIRE(lz_attn_direct(dtype, hd, ldq, ldk, ldv, ldo) && lz_attn_wave_ok(w, dtype, hd, false),
             "lz_attn_fwd_direct: unsupported head dim, dtype or alignment");
  if ((dtype == LZ_BF16 || S % 64 == 0) && mfma_ok(dtype, hd, ldq, ldk, ldv, ldo, q, k, v, o))
    return tiles_fwd(q, ldq, k, ldk, v, ldv, o, ldo, lse, B, S, H, KV, hd, scale, dtype, lz_stream(stream));
  return lz_attn_wave_pass(w, dtype, hd, kWaveSplit, kWaveFwd, lz_stream(stream));
}

LZ_EXPORT int lz_attn_bwd_direct(const void* q, int64_t ldq, const void* k, int64_t ldk, const void* v, int64_t ldv,
                                 const void* o, int64_t ldo, const void* dout, int64_t lddo, const float* lse,
                                 float* delta, void* dq, int64_t lddq, void* dk, int64_t lddk, void* dv, int64_t lddv,
                                 int64_t B, int64_t S, int64_t H, int64_t KV, int64_t hd, float scale, int dtype,
                                 void* stream) {
  int rc = check_shape(B, S, H, KV, hd);
  if (rc) return rc;
  LZ_REQUIRE(q && k && v && o && dout && lse && delta && dq && dk && dv, "lz_attn_bwd_direct: null pointer");
  LzWaveArgs w = wave_fwd_args(q, ldq, k, ldk, v, ldv, const_cast<void*>(o), ldo, const_cast<float*>(lse), B, S, H, KV,
                               scale);
  wave_bwd_args(w, dout, lddo, nullptr, dq, lddq, dk, lddk, dv, lddv);
  w.delta_w = delta;
  LZ_REQUIRE(lz_attn_direct(dtype, hd, ldq, ldk, ldv, ldo) && lz_attn_wave_ok(w, dtype, hd, true),
             "lz_attn_bwd_direct: unsupported head dim, dtype or alignment");
  bool rope_done = false;
  if ((dtype == LZ_BF16 || S % 64 == 0) && mfma_ok(dtype, hd, ldq, ldk, ldv, lddo, q, k, v, dout))
    return tiles_bwd(q, ldq, k, ldk, v, ldv, dout, lddo, lse, nullptr, dq, lddq, dk, lddk, dv, lddv, B, S, H, KV, hd,
                     scale, nullptr, nullptr, dtype, lz_stream(stream), rope_done, o, ldo, delta);
  return lz_attn_wave_bwd(w, dtype, hd, kWaveSplit, lz_stream(stream));
}
