// bf16 / fp16 GEMM for products whose 256-wide tiles would leave most of the
// chip idle (few rows: a generate() prompt, a small batch, a short sequence's
// gradients) or whose K is not a multiple of 64.
//
// BM x BN tiles of 64 or 128, four or eight waves, 64-deep K stages copied
// straight into LDS (buffer_load ... lds), kStages - 1 of them in flight.  Such
// a launch has at most a few tiles per CU, so its time is the serial chain of
// one tile's K steps plus the launch: what counts is that a step waits for
// LDS and not for HBM or L2.  Each step waits only for its own stage
// (vmcnt), crosses one barrier and issues the stage kStages - 1 ahead.  The
// last stage may be shorter than 64: its loads are clamped into the operand
// and the missing K values are zeroed in LDS (both operands, so that no stray
// inf or NaN meets a zero).
#include "gemm_pipe.h"

#include "gemm_tiles.h"

namespace {

// Chunk-pair swizzle of an M/N-major stage row of COLS values: tells apart, by
// an XOR of 32-byte pairs, the eight rows {0..3, 8..11} (+4) that a half-wave
// of ds_read_b64_tr_b16 reads 32 bytes of, within the 256-byte bank window
// (rows of 128 values span it once, rows of 64 values half of it).
template <int COLS>
__device__ __forceinline__ int swz_pair(int r) {
  if constexpr (COLS == 128) return (r & 3) | (((r >> 3) & 1) << 2);
  else return ((r >> 1) & 1) | (((r >> 3) & 1) << 1);
}

// One operand of a stage: ROWS (M or N) x 64 K, 128 * ROWS bytes, filled by
// wave loads of 1 KB spread over the waves.
template <bool KMAJOR, int ROWS, int kWaves>
struct PipeOperand {
  static constexpr int kLoads = ROWS / 8 / kWaves;  // wave loads per wave
  static constexpr int kRowBytes = KMAJOR ? 128 : ROWS * 2;
  static constexpr int kChunks = kRowBytes / 16, kRowsPerLoad = 64 / kChunks;
  lz_v4i rsrc;
  uint32_t voff[kLoads];
  uint32_t kadv;

  static __device__ __forceinline__ int row_of(int q, int wave, int lane) {
    return (wave * kLoads + q) * kRowsPerLoad + lane / kChunks;
  }
  static __device__ __forceinline__ int chunk_of(int r, int lane) {
    return (lane % kChunks) ^ (KMAJOR ? swz<8>(r) : 2 * swz_pair<ROWS>(r));
  }
  // rows (K-major) or columns (M/N-major) past the operand repeat its last ones
  __device__ __forceinline__ void init(const uint16_t* p, int64_t ld, int64_t row0, int64_t nrows, int64_t kbeg,
                                       int wave, int lane) {
    rsrc = lz_buffer_rsrc(KMAJOR ? p + row0 * ld + kbeg : p + kbeg * ld + row0);
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      const int r = row_of(q, wave, lane), c = chunk_of(r, lane);
      if constexpr (KMAJOR) voff[q] = (uint32_t)(((min(row0 + r, nrows - 1) - row0) * ld + c * 8) * 2);
      else voff[q] = (uint32_t)((r * ld + (min(row0 + c * 8, nrows - 8) - row0)) * 2);
    }
    kadv = (uint32_t)((KMAJOR ? 64 : 64 * ld) * 2);
  }
  __device__ __forceinline__ void issue(char* dst, int wave, int kt) const {
    if (kt == 0) lz_dma16_first(rsrc, voff[0], 0, dst + wave * kLoads * 1024);
    else lz_dma16(rsrc, voff[0], (uint32_t)kt * kadv, dst + wave * kLoads * 1024);
#pragma unroll
    for (int q = 1; q < kLoads; ++q)
      lz_dma16(rsrc, voff[q], (uint32_t)kt * kadv, dst + (wave * kLoads + q) * 1024);
  }
  // the last stage, of which only krem K values exist: the others' loads are
  // clamped to the last existing ones
  __device__ __forceinline__ void issue_tail(char* dst, int wave, int lane, int kt, int krem) const {
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      const int r = row_of(q, wave, lane), c = chunk_of(r, lane);
      const uint32_t back = KMAJOR ? 2 * max(0, c * 8 - (krem - 8)) : max(0, r - (krem - 1)) * (kadv / 64);
      lz_dma16_first(rsrc, voff[q] - back, (uint32_t)kt * kadv, dst + (wave * kLoads + q) * 1024);
    }
  }
  // zeros in the stage's K values from krem on
  static __device__ __forceinline__ void zero_tail(char* stage, int krem, int tid) {
    for (int i = tid; i < ROWS * 8; i += 64 * kWaves) {  // 16-byte chunks
      const int r = i / kChunks, slot = i % kChunks;
      const int k = KMAJOR ? chunk_of(r, slot) * 8 : r;
      if (k >= krem) *reinterpret_cast<uint4*>(stage + i * 16) = make_uint4(0, 0, 0, 0);
    }
  }
};

// Fragment offsets of a wave's NF 16-row blocks (the 16x16x32 operand layout:
// lane l holds row l % 16, K 8*(l/16) .. +7 of a 32-deep slice).
template <bool KMAJOR, int ROWS, int NF>
struct PipeFrags {
  static constexpr int kRowBytes = ROWS * 2;  // M/N-major stage row
  int kb[2], base[2], ioff[NF];

  __device__ __forceinline__ void init(int blk0, int lane) {
    if constexpr (KMAJOR) {
      const int r = blk0 * 16 + (lane & 15);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) kb[kk] = r * 128 + (((4 * kk + (lane >> 4)) ^ swz<8>(r)) << 4);
    } else {
      const int p = lane & 15, grp = lane >> 4, j = p >> 2, q = p & 3;
#pragma unroll
      for (int rd = 0; rd < 2; ++rd) base[rd] = (8 * grp + 4 * rd + j) * kRowBytes + ((q >> 1) << 4) + (q & 1) * 8;
      const int f = swz_pair<ROWS>(8 * grp + j);
#pragma unroll
      for (int i = 0; i < NF; ++i) ioff[i] = ((blk0 + i) ^ f) << 5;
    }
  }
  __device__ __forceinline__ bf16x8_t frag(const char* op, int f, int kk) const {
    if constexpr (KMAJOR) {
      return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(op + f * 16 * 128 + kb[kk]));
    } else {
      const char* blk = op + kk * 32 * kRowBytes + ioff[f];
      const v4i16_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(blk + base[0]));
      const v4i16_t y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(blk + base[1]));
      const uint2 xw = __builtin_bit_cast(uint2, x), yw = __builtin_bit_cast(uint2, y);
      return __builtin_bit_cast(bf16x8_t, make_uint4(xw.x, xw.y, yw.x, yw.y));
    }
  }
};

template <typename F, int BM, int BN, int WM, int WN, bool AK, bool BK, int kStages>
__global__ void __launch_bounds__(64 * WM * WN) gemm_pipe_kernel(GemmArgs g) {
  constexpr int kWaves = WM * WN, TM = BM / WM, TN = BN / WN, FM = TM / 16, FN = TN / 16;
  constexpr int kABytes = BM * 128, kStage = (BM + BN) * 128;
  constexpr int kLoads = PipeOperand<AK, BM, kWaves>::kLoads + PipeOperand<BK, BN, kWaves>::kLoads;  // per wave and stage
  static_assert(kWaves * epi_wave_bytes<TM, TN>() <= kStages * kStage, "epilogue staging does not fit");
  static_assert(kWaves * 16 * (TN + 4) * 4 <= kStages * kStage, "epilogue staging does not fit");
  __shared__ __attribute__((aligned(1024))) char smem[kStages * kStage];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t tm, tn;
  tile_coords(blockIdx.x, lz_cdiv(g.M, BM), lz_cdiv(g.N, BN), tm, tn);
  const int64_t m0 = tm * BM, n0 = tn * BN;
  const int64_t kbeg = (int64_t)blockIdx.y * g.kper, kend = min(g.K, kbeg + g.kper);
  const int ktiles = kend > kbeg ? (int)lz_cdiv(kend - kbeg, 64) : 0;
  const int krem = (int)(kend - kbeg) - (ktiles - 1) * 64;  // K values of the last stage, 1 .. 64

  PipeOperand<AK, BM, kWaves> la;
  PipeOperand<BK, BN, kWaves> lb;
  la.init(g.A, g.lda, m0, g.M, kbeg, wave, lane);
  lb.init(g.B, g.ldb, n0, g.N, kbeg, wave, lane);
  PipeFrags<AK, BM, FM> fra;
  PipeFrags<BK, BN, FN> frb;
  fra.init((wave / WN) * FM, lane);
  frb.init((wave % WN) * FN, lane);

  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  auto issue = [&](int kt) {
    char* st = smem + (kt % kStages) * kStage;
    if (kt == ktiles - 1 && krem < 64) {
      la.issue_tail(st, wave, lane, kt, krem);
      lb.issue_tail(st + kABytes, wave, lane, kt, krem);
    } else {
      la.issue(st, wave, kt);
      lb.issue(st + kABytes, wave, kt);
    }
  };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s)
    if (s < ktiles) issue(s);
  for (int kt = 0; kt < ktiles; ++kt) {
    // stage kt has landed (the stages issued after it may be in flight), and
    // every wave is done with stage kt - 1, whose slot the next issue refills
    if (kt + kStages - 2 < ktiles) wait_vmcnt<kLoads * (kStages - 2)>();
    else wait_vmcnt<0>();
    __syncthreads();
    if (kt + kStages - 1 < ktiles) issue(kt + kStages - 1);
    char* sa = smem + (kt % kStages) * kStage;
    char* sb = sa + kABytes;
    if (kt == ktiles - 1 && krem < 64) {
      PipeOperand<AK, BM, kWaves>::zero_tail(sa, krem, tid);
      PipeOperand<BK, BN, kWaves>::zero_tail(sb, krem, tid);
      __syncthreads();
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8_t fa[FN], fb[FM];
#pragma unroll
      for (int j = 0; j < FN; ++j) fa[j] = frb.frag(sb, j, kk);
#pragma unroll
      for (int i = 0; i < FM; ++i) fb[i] = fra.frag(sa, i, kk);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma_k32<F>(fa[j], fb[i], acc[i][j]);
    }
  }
  __syncthreads();  // every wave is done with the stages before the epilogue reuses LDS
  GemmArgs go = g;  // split-K: this split's fp32 slab
  if (g.slab) go.C = static_cast<float*>(g.C) + (int64_t)blockIdx.y * g.slab;
  store_tile<F, 16, BM, BN, WM, WN>(go, acc, m0, n0, smem, lane, wave);
}

// 64x64: four waves of 32x32, three stages (48 KB: three workgroups per CU);
// 64x128: eight waves of 32x32, three stages (72 KB: two); 128x128: eight waves
// of 64x32, two stages (64 KB: two).  Measured (us): eight waves instead of
// four 333x768x4096 at 128x128 46.4 -> 42.9, at 64x128 32.4 -> 27.9 (two waves
// per SIMD overlap one's LDS reads with the other's MFMAs); two workgroups
// per CU instead of one 4096x2048x2000 50.2 -> 33.1 (128x128, four stages ->
// two); two stages at 64 wide tiles lose 35 % once K reaches 4096; deeper
// pipelines (up to eight stages) and fragments read a slice ahead across the
// barrier gained nothing.
template <typename F, int BM, int BN, bool AK, bool BK>
int launch(const GemmArgs& g, int splits, hipStream_t s) {
  const int64_t tiles = lz_cdiv(g.M, BM) * lz_cdiv(g.N, BN);
  LZ_REQUIRE(tiles < (1ll << 31), "lz_gemm: too many tiles");
  constexpr int kWn = BN == 128 ? 4 : 2, kStages = BM == 128 ? 2 : 3;
  gemm_pipe_kernel<F, BM, BN, 2, kWn, AK, BK, kStages>
      <<<dim3((unsigned)tiles, (unsigned)splits), 128 * kWn, 0, s>>>(g);
  return lz_check_launch("lz_gemm");
}

template <typename F, int BM, int BN>
int launch_layout(const GemmArgs& g, bool ak, bool bk, int splits, hipStream_t s) {
  if (ak && bk) return launch<F, BM, BN, true, true>(g, splits, s);
  return ak ? launch<F, BM, BN, true, false>(g, splits, s) : launch<F, BM, BN, false, false>(g, splits, s);
}

template <typename F>
int launch_tile(const GemmArgs& g, bool ak, bool bk, int bm, int bn, int splits, hipStream_t s) {
  if (bm == 128 && bn == 128) return launch_layout<F, 128, 128>(g, ak, bk, splits, s);
  if (bm == 64 && bn == 128) return launch_layout<F, 64, 128>(g, ak, bk, splits, s);
  return launch_layout<F, 64, 64>(g, ak, bk, splits, s);
}

}  // namespace

int lz_gemm_pipe(const GemmArgs& g, bool f16, bool ak, bool bk, int bm, int bn, int splits, hipStream_t s) {
  return f16 ? launch_tile<FmtF16>(g, ak, bk, bm, bn, splits, s) : launch_tile<FmtBF16>(g, ak, bk, bm, bn, splits, s);
}
