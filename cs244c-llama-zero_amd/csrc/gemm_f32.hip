// fp32 GEMM on CDNA4 matrix cores (v_mfma_f32_32x32x2_f32):
//
//   C[M,N] = alpha * sum_k A(m,k) B(n,k)  (+ beta * C)  (+ R)
//
// The float32 twin of the bf16 product in gemm.hip, for models kept in fp32
// (the reference's `--dtype float32`, train.py:148-160 and
// train_zero.py:74,150-164, where nn.Linear runs in fp32).  Same operand
// layouts: an operand is K-major (A(m,k) = A[m*lda + k]) or M/N-major
// (A(m,k) = A[k*lda + m]), so forward, input-gradient and weight-gradient
// products read the stored tensors directly.  Products and sums stay fp32
// (gfx950 has no reduced-precision fp32 mode), so results are within a few
// fp32 ulps of the exact product; any M, N, K and leading dimension work:
// rows past M/N and K past the end are zero-filled in LDS, stores are masked.
//
// Tiling: a 256-thread workgroup (4 waves) owns one of three tiles, chosen by
// make_plan: 128 x 128 (2 x 2 waves of 64 x 64) or 64 x 64 (2 x 2 waves of
// 32 x 32) with K in 32-deep stages, or 32 x 32 with 128-deep stages whose
// four 32-deep slices go to one wave each (their sums meet in LDS, in a fixed
// order).  An fp32 MFMA keeps a matrix core busy for 64 cycles on two LDS
// reads, so even 32 x 32 wave tiles are MFMA-bound; what bounded the products
// of the small models was one 128 x 128 tile per CU on a few CUs, and the
// latency of one stage of loads per barrier.  Stages are double-buffered in
// LDS and the global loads run two stages ahead of them in registers.
//
// An operand stays in its own orientation in LDS: K-major rows padded to 36
// floats and read 16 bytes (four K) at a time, M/N-major K rows padded by 8
// floats and read one float at a time (transposing them on the way in cost
// four 8-way conflicting stores per load).  Half h of a wave takes the K
// values 8c + 4h + e of a slice in either orientation.
//
// The accumulators are flushed into a second set every 64 K, so a sum's
// rounding error grows with 64 + K/64 terms and not with K.
//
// Split-K: where the tiles alone leave CUs idle and K is long (a language-model
// head's input gradient reduces over the vocabulary), K is cut into slices of
// whole stages, one grid layer each; the slices write fp32 partial tiles into
// a workspace and a second kernel sums them in slice order, then applies
// alpha, beta*C and R as the unsplit epilogue does.  The result does not
// depend on timing.
#include "gemm_tiles.h"

namespace {

constexpr int kSliceK = 32;             // K per slice of a stage
constexpr int kRow = kSliceK + 4;       // padded K-major LDS row, floats
constexpr int kThreads = 256;

struct F32Args {
  const float* A;
  const float* B;
  void* C;
  const float* R;
  int64_t lda, ldb, ldc, ldr;
  int64_t M, N, K;
  float alpha, beta;
  int c_f32;   // fp32 output (else bf16)
  int64_t kper;  // K per grid layer (a multiple of kSliceK when split)
  int64_t slab;  // > 0: layer z writes raw fp32 partials at C + z * slab
};

struct Plan {
  int tile;  // 128, 64 or 32
  int splits;
  int64_t kper;
};

// Tile and split with the least estimated time (us): a launch, then per stage
// either the latency of one workgroup's chain or, with `rounds`
// workgroups per CU, the matrix cores' time for all of them, the output's
// bytes, and for a split the second kernel (2.2) and its partial tiles.
// Fitted to 1700 measured (product, tile, split) triples, five M x N x K
// families over 24 .. 8192 tokens; measured us, 128 x 128 register-transposed
// kernel with up to 64 splits -> this plan:
//   24 x 448 x 320    12.6 -> 6.2 (32)       1024 x 448 x 320     17.5 -> 9.0 (32)
//   1024 x 1792 x 320 33.2 -> 17.8 (64)      1024 x 320 x 8192   125.9 -> 60.3 (64, 16 splits)
//   4096 x 8192 x 320 228 -> 203 (64)        8192 x 1024 x 4096 weight gradient
//   1073 -> 582 (128, 2 splits)
// The 128 tile is up to 6 % faster than 64 x 64 where both fill the chip, and
// twice as slow where 64 x 64 tiles are fewer than the CUs.
Plan make_plan(int64_t M, int64_t N, int64_t K) {
  struct Tile {
    int size, deep;
    double start, chain, busy;  // us: launch and first stage; per stage, one workgroup alone and each of several on a CU
  };
  static constexpr Tile kTiles[] = {{32, 128, 3.5, 0.85, 0.90}, {64, 32, 4.6, 0.70, 0.56}, {128, 32, 6.0, 2.30, 2.10}};
  static constexpr int kSplits[] = {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32, 48, 64};
  constexpr double kBytesPerUs = 5e6;
  const int64_t cus = lz_num_cus();
  const double out = (double)M * N * sizeof(float) / kBytesPerUs;
  Plan best{64, 1, K};
  double least = INFINITY;
  for (const Tile& t : kTiles) {
    const int64_t tiles = lz_cdiv(M, t.size) * lz_cdiv(N, t.size), deep = t.deep;
    for (const int want : kSplits) {
      // a split keeps a stage of its own, and 8 workgroups per CU need no more
      if (want > 1 && (K < want * deep || tiles * want > 8 * cus)) break;
      const int64_t kper = want > 1 ? lz_cdiv(lz_cdiv(K, want), deep) * deep : K;
      const int64_t splits = want > 1 ? lz_cdiv(K, kper) : 1;
      const double stages = (double)lz_cdiv(kper, deep), rounds = (double)lz_cdiv(tiles * splits, cus);
      double us = t.start + std::max(stages * t.chain, rounds * stages * t.busy) + out;
      if (splits > 1) us += 2.2 + 2.0 * splits * out;
      if (us < least) {
        least = us;
        best = Plan{t.size, (int)splits, kper};
      }
    }
  }
  return best;
}

int64_t plan_workspace(const Plan& p, int64_t M, int64_t N) {
  return p.splits > 1 ? (int64_t)p.splits * M * N * (int64_t)sizeof(float) : 0;
}

typedef float f32x4a4_t __attribute__((ext_vector_type(4), aligned(4)));  // one 16-byte load of any row

// One operand's stage: ROWS of M (or N) x KS slices of kSliceK K.
template <bool KMAJOR, int ROWS, int KS>
struct Operand {
  static constexpr int kLd = KMAJOR ? kRow : ROWS + 8;              // LDS row, floats
  static constexpr int kSlice = (KMAJOR ? ROWS : kSliceK) * kLd;        // LDS floats of a slice
  static constexpr int kPieces = ROWS * KS * kSliceK / 4 / kThreads;    // four-float pieces per thread
  static constexpr int kPerRow = (KMAJOR ? KS * kSliceK : ROWS) / 4;    // pieces per stored row

  struct Regs {
    float4 v[kPieces];
  };

  // Stage at K offset k0 into registers.  kVec: 16-byte aligned rows of a
  // multiple of four floats; other rows take the same loads from addresses of
  // any float and single ones at their short end (one float at a time
  // 2048 x 2048 x 2048 with one such operand took 243 us, now 160).  Addresses past the operand are clamped into it:
  // rows past M/N only reach outputs that are never stored, K past kend is
  // zeroed by store().
  template <bool kVec>
  static __device__ __forceinline__ void load(Regs& r, const float* X, int64_t ld, int64_t rows, int64_t kend,
                                              int64_t r0, int64_t k0) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      const int i = threadIdx.x + kThreads * p;
      const int64_t outer = (KMAJOR ? r0 : k0) + i / kPerRow, inner = (KMAJOR ? k0 : r0) + i % kPerRow * 4;
      const int64_t nouter = KMAJOR ? rows : kend, ninner = KMAJOR ? kend : rows;
      const float* src = X + min(outer, nouter - 1) * ld;
      if constexpr (kVec) {
        r.v[p] = *reinterpret_cast<const float4*>(src + min(inner, ninner - 4));
      } else if (inner + 4 <= ninner) {
        const f32x4a4_t v = *reinterpret_cast<const f32x4a4_t*>(src + inner);
        r.v[p] = make_float4(v[0], v[1], v[2], v[3]);
      } else {
        r.v[p].x = src[min(inner, ninner - 1)];
        r.v[p].y = src[min(inner + 1, ninner - 1)];
        r.v[p].z = src[min(inner + 2, ninner - 1)];
        r.v[p].w = src[min(inner + 3, ninner - 1)];
      }
    }
  }

  // Registers -> LDS; krem: K values of this stage that exist.
  static __device__ __forceinline__ void store(const Regs& r, float* dst, int64_t krem) {
#pragma unroll
    for (int p = 0; p < kPieces; ++p) {
      const int i = threadIdx.x + kThreads * p;
      const int o = i / kPerRow, c = i % kPerRow * 4;
      float4 v = r.v[p];
      if constexpr (KMAJOR) {
        if (krem < KS * kSliceK) {
          v.x = c < krem ? v.x : 0.f;
          v.y = c + 1 < krem ? v.y : 0.f;
          v.z = c + 2 < krem ? v.z : 0.f;
          v.w = c + 3 < krem ? v.w : 0.f;
        }
        *reinterpret_cast<float4*>(dst + c / kSliceK * kSlice + o * kLd + c % kSliceK) = v;
      } else {
        if (o >= krem) v = make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(dst + o / kSliceK * kSlice + o % kSliceK * kLd + c) = v;
      }
    }
  }

  // This lane's values K = 8c + 4h + (0..3) of row `row` of a slice.
  static __device__ __forceinline__ float4 frag(const float* slice, int row, int c, int h) {
    if constexpr (KMAJOR) {
      return *reinterpret_cast<const float4*>(slice + row * kLd + 8 * c + 4 * h);
    } else {
      const float* s = slice + (8 * c + 4 * h) * kLd + row;
      return make_float4(s[0], s[kLd], s[2 * kLd], s[3 * kLd]);
    }
  }
};

// Barrier for LDS traffic only: the register prefetches stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void store_out(const F32Args& g, int64_t m, int64_t n, float acc) {
  if (m >= g.M || n >= g.N) return;
  if (g.slab > 0) {
    (static_cast<float*>(g.C) + (int64_t)blockIdx.y * g.slab)[m * g.N + n] = acc;
    return;
  }
  float val = acc * g.alpha;
  if (g.c_f32) {
    float* cp = static_cast<float*>(g.C) + m * g.ldc + n;
    if (g.beta != 0.f) val = fmaf(g.beta, *cp, val);
    if (g.R) val += g.R[m * g.ldr + n];
    *cp = val;
  } else {
    uint16_t* cp = static_cast<uint16_t*>(g.C) + m * g.ldc + n;
    if (g.beta != 0.f) val = fmaf(g.beta, bf2f(*cp), val);
    if (g.R) val += g.R[m * g.ldr + n];
    *cp = f2bf(val);
  }
}

// TILE x TILE per workgroup; KS = 4: each wave one slice of a stage, KS = 1:
// 2 x 2 waves.
template <int TILE, int KS, bool AK, bool BK, bool kVec>
__global__ void __launch_bounds__(kThreads, 2) gemm_f32_kernel(F32Args g) {
  using OpA = Operand<AK, TILE, KS>;
  using OpB = Operand<BK, TILE, KS>;
  constexpr int kWaveTile = KS == 1 ? TILE / 2 : TILE, kF = kWaveTile / 32;
  constexpr int kA = KS * OpA::kSlice, kStage = kA + KS * OpB::kSlice, kDeep = KS * kSliceK;
  __shared__ __attribute__((aligned(16))) float lds[2 * kStage];
  static_assert(KS == 1 || 2 * kStage >= 4 * 1024, "the waves' sums do not fit");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = KS == 1 ? (wave >> 1) * kWaveTile : 0, wn = KS == 1 ? (wave & 1) * kWaveTile : 0;
  const int slice = KS == 1 ? 0 : wave;
  const int li = lane & 31, h = lane >> 5;
  int64_t tm, tn;
  tile_coords(blockIdx.x, lz_cdiv(g.M, TILE), lz_cdiv(g.N, TILE), tm, tn);
  const int64_t m0 = tm * TILE, n0 = tn * TILE;
  const int64_t kbeg = (int64_t)blockIdx.y * g.kper, kend = min(g.K, kbeg + g.kper);
  const int nk = kend > kbeg ? (int)lz_cdiv(kend - kbeg, kDeep) : 0;

  f32x16_t acc[kF][kF], sum[kF][kF];
#pragma unroll
  for (int i = 0; i < kF; ++i)
#pragma unroll
    for (int j = 0; j < kF; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.f;
        sum[i][j][r] = 0.f;
      }

  typename OpA::Regs ra[2];
  typename OpB::Regs rb[2];
  auto fetch = [&](auto& a, auto& b, int kt) {
    OpA::template load<kVec>(a, g.A, g.lda, g.M, kend, m0, kbeg + (int64_t)kt * kDeep);
    OpB::template load<kVec>(b, g.B, g.ldb, g.N, kend, n0, kbeg + (int64_t)kt * kDeep);
  };
  auto put = [&](const auto& a, const auto& b, int kt) {
    float* st = lds + (kt & 1) * kStage;
    const int64_t krem = kend - (kbeg + (int64_t)kt * kDeep);
    OpA::store(a, st, krem);
    OpB::store(b, st + kA, krem);
  };
  // stage kt: its products, then stage kt + 1 (in registers a, b) into the
  // other buffer, last read before the previous barrier, and the loads of
  // stage kt + 3 in its place
  auto step = [&](auto& a, auto& b, int kt) {
    const float* As = lds + (kt & 1) * kStage + slice * OpA::kSlice;
    const float* Bs = lds + (kt & 1) * kStage + kA + slice * OpB::kSlice;
#pragma unroll
    for (int c = 0; c < kSliceK / 8; ++c) {
      float4 fa[kF], fb[kF];
#pragma unroll
      for (int i = 0; i < kF; ++i) fa[i] = OpA::frag(As, wm + 32 * i + li, c, h);
#pragma unroll
      for (int j = 0; j < kF; ++j) fb[j] = OpB::frag(Bs, wn + 32 * j + li, c, h);
#pragma unroll
      for (int i = 0; i < kF; ++i)
#pragma unroll
        for (int j = 0; j < kF; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].x, fb[j].x, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].y, fb[j].y, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].z, fb[j].z, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i].w, fb[j].w, acc[i][j], 0, 0, 0);
        }
    }
    if (kt + 1 < nk) put(a, b, kt + 1);
    if (kt + 3 < nk) fetch(a, b, kt + 3);
    lds_barrier();
  };
  if (nk > 0) {
    fetch(ra[0], rb[0], 0);
    if (nk > 1) fetch(ra[1], rb[1], 1);
    put(ra[0], rb[0], 0);
    if (nk > 2) fetch(ra[0], rb[0], 2);
    lds_barrier();
  }
  for (int kt = 0; kt < nk; kt += 2) {
    step(ra[1], rb[1], kt);
    if (kt + 1 < nk) step(ra[0], rb[0], kt + 1);
#pragma unroll
    for (int i = 0; i < kF; ++i)
#pragma unroll
      for (int j = 0; j < kF; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          sum[i][j][r] += acc[i][j][r];
          acc[i][j][r] = 0.f;
        }
  }

  // Accumulator register r of lane (li, h) in block (i, j) holds
  // C[m][n] with m = 8*(r/4) + 4*h + r%4 and n = li inside the 32 x 32 block:
  // each store instruction writes two 128-byte row segments.
  if constexpr (KS == 1) {
#pragma unroll
    for (int i = 0; i < kF; ++i)
#pragma unroll
      for (int j = 0; j < kF; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          store_out(g, m0 + wm + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3), n0 + wn + j * 32 + li, sum[i][j][r]);
  } else {
    // the four slices' sums as [slice][register][lane] (the last barrier is
    // behind every stage read); wave w adds and stores registers 4w .. 4w + 3
#pragma unroll
    for (int r = 0; r < 16; ++r) lds[(wave * 16 + r) * 64 + lane] = sum[0][0][r];
    lds_barrier();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float* p = lds + (4 * wave + e) * 64 + lane;
      store_out(g, m0 + 8 * wave + 4 * h + e, n0 + li, ((p[0] + p[1024]) + p[2048]) + p[3072]);
    }
  }
}

// C = alpha * sum_z part[z] (+ beta*C) (+ R), the slices summed in order.
__global__ void __launch_bounds__(256) splitk_reduce_f32_kernel(F32Args g, const float* __restrict__ part,
                                                                 int64_t slab, int splits) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= g.M * g.N) return;
  const int64_t m = i / g.N, n = i - m * g.N;
  float acc = 0.f;
  for (int z = 0; z < splits; ++z) acc += part[z * slab + i];
  store_out(g, m, n, acc);
}

template <int TILE, int KS, bool kVec>
int launch_tile(const F32Args& g, bool ak, bool bk, int splits, hipStream_t s) {
  const int64_t tiles = lz_cdiv(g.M, TILE) * lz_cdiv(g.N, TILE);
  LZ_REQUIRE(tiles < (1ll << 31), "lz_gemm_f32: too many tiles (M %lld, N %lld)", (long long)g.M, (long long)g.N);
  const dim3 grid((unsigned)tiles, (unsigned)splits);
  if (ak && bk) gemm_f32_kernel<TILE, KS, true, true, kVec><<<grid, kThreads, 0, s>>>(g);
  else if (ak) gemm_f32_kernel<TILE, KS, true, false, kVec><<<grid, kThreads, 0, s>>>(g);
  else if (bk) gemm_f32_kernel<TILE, KS, false, true, kVec><<<grid, kThreads, 0, s>>>(g);
  else gemm_f32_kernel<TILE, KS, false, false, kVec><<<grid, kThreads, 0, s>>>(g);
  return lz_check_launch("lz_gemm_f32");
}

int launch_f32(const F32Args& g, int tile, bool ak, bool bk, int splits, hipStream_t s) {
  // 16-byte loads: aligned rows of whole pieces (an operand's short end is
  // then a whole piece, never part of one)
  const bool vec = lz_aligned16(g.A) && lz_aligned16(g.B) && g.lda % 4 == 0 && g.ldb % 4 == 0 &&
                   ((!ak && !bk) || g.K % 4 == 0) && (ak || g.M % 4 == 0) && (bk || g.N % 4 == 0);
  if (tile == 128) return vec ? launch_tile<128, 1, true>(g, ak, bk, splits, s) : launch_tile<128, 1, false>(g, ak, bk, splits, s);
  if (tile == 64) return vec ? launch_tile<64, 1, true>(g, ak, bk, splits, s) : launch_tile<64, 1, false>(g, ak, bk, splits, s);
  return vec ? launch_tile<32, 4, true>(g, ak, bk, splits, s) : launch_tile<32, 4, false>(g, ak, bk, splits, s);
}

}  // namespace

// Workspace bytes lz_gemm_f32 uses for this shape (0 when K is not split).
LZ_EXPORT int64_t lz_gemm_f32_workspace(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return plan_workspace(make_plan(M, N, K), M, N);
}

// Number of K slices lz_gemm_f32 runs this shape in (1 = unsplit).
LZ_EXPORT int lz_gemm_f32_plan(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return make_plan(M, N, K).splits;
}

// fp32 operands, fp32 accumulation: C = alpha * sum_k A(m,k) B(n,k)
// (+ beta*C) (+ R), with the operand layouts of lz_gemm.  C: [M,N] fp32 or
// bf16 (ldc); R: optional fp32 [M,N] (ldr).  No alignment or size
// multiples are required; aligned rows of whole 16 bytes take the shorter loop.  `ws`
// (ws_bytes long, may be null) holds the partial products when K is split;
// with less than lz_gemm_f32_workspace() bytes the product runs unsplit.
LZ_EXPORT int lz_gemm_f32(const float* A, int64_t lda, int a_kmajor, const float* B, int64_t ldb, int b_kmajor, void* C,
                          int64_t ldc, int c_dtype, const float* R, int64_t ldr, int64_t M, int64_t N, int64_t K,
                          float alpha, float beta, void* ws, int64_t ws_bytes, void* stream) {
  LZ_REQUIRE(M >= 0 && N >= 0 && K >= 0, "lz_gemm_f32: negative shape");
  if (M == 0 || N == 0) return LZ_OK;
  LZ_REQUIRE(C, "lz_gemm_f32: null output");
  LZ_REQUIRE(K == 0 || (A && B), "lz_gemm_f32: null operand");
  LZ_REQUIRE(c_dtype == LZ_F32 || c_dtype == LZ_BF16, "lz_gemm_f32: bad output dtype %d", c_dtype);
  LZ_REQUIRE(K == 0 || (lda >= (a_kmajor ? K : M) && ldb >= (b_kmajor ? K : N)), "lz_gemm_f32: bad operand stride");
  LZ_REQUIRE(ldc >= N && (R == nullptr || ldr >= N), "lz_gemm_f32: bad output stride");
  LZ_REQUIRE(ws_bytes >= 0 && (ws == nullptr || lz_aligned16(ws)), "lz_gemm_f32: workspace must be 16-byte aligned");
  F32Args g;
  g.A = A;
  g.B = B;
  g.C = C;
  g.R = R;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.ldr = ldr;
  g.M = M;
  g.N = N;
  g.K = K;
  g.alpha = alpha;
  g.beta = beta;
  g.c_f32 = c_dtype == LZ_F32;
  g.kper = K;
  g.slab = 0;
  hipStream_t s = lz_stream(stream);
  const bool ak = a_kmajor != 0, bk = b_kmajor != 0;
  const Plan p = make_plan(M, N, K);
  if (p.splits == 1 || ws == nullptr || ws_bytes < plan_workspace(p, M, N)) return launch_f32(g, p.tile, ak, bk, 1, s);
  F32Args gs = g;  // partial products into fp32 slabs [splits][M][N]
  gs.C = ws;
  gs.kper = p.kper;
  gs.slab = M * N;
  int rc = launch_f32(gs, p.tile, ak, bk, p.splits, s);
  if (rc) return rc;
  splitk_reduce_f32_kernel<<<(unsigned)lz_cdiv(M * N, 256), 256, 0, s>>>(g, static_cast<const float*>(ws), gs.slab,
                                                                         p.splits);
  return lz_check_launch("lz_gemm_f32(split-K reduce)");
}
