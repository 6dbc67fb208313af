// Launches of the wave-private attention kernels (attn_wave.hip) for the entry
// points of attn.hip.
#pragma once
#include "lz_common.h"

struct LzWaveArgs {
  const void* q;
  const void* k;
  const void* v;
  int64_t ldq, ldk, ldv;
  void* o;  // written by the forward; read by the dQ kernel when it forms delta
  int64_t ldo;
  float* lse;
  const void* dout;
  int64_t lddo;
  const float* delta;
  float* delta_w;  // not null: the dQ kernel computes delta = rowsum(dO * O) and writes it here
  void* dq;
  void* dk;
  void* dv;
  int64_t lddq, lddk, lddv;
  int B, S, H, KV;
  float scale;
  // explicit mask in place of the causal one: kind 1 = bool bytes (nonzero
  // keeps the score), 2 = fp32, 3 = bf16, 4 = fp16 (added to the scaled
  // score), 0 = causal; element strides over [B, H, S(query), S(key)]
  const void* mask;
  int mask_kind;
  int64_t msb, msh, msq, msk;
  // attention dropout: probability (b, h, s, kv) is kept with drop_scale when
  // element ((b*H + h)*S + s)*S + kv of the seed's stream is (0 = none)
  uint32_t drop_thresh;
  float drop_scale;
  uint64_t drop_seed;
};

// Whether these kernels take the call: head dim 32, 64 or 128, rows aligned
// for their reads and writes (dout8: dout rows may start at any 8 bytes).
bool lz_attn_wave_ok(const LzWaveArgs& a, int dtype, int64_t hd, bool backward, bool dout8 = false);

// How a call is computed.  General: mask_kind and dropout are read (also when
// both are off, so that a call with dropout has the lse of one without);
// otherwise causal.  bf16 probabilities and dS enter their products with all
// their fp32 bits (three bf16 terms), except with kWaveRounded (one rounding,
// as in the tile kernels).
enum LzWaveMode { kWaveGeneral, kWaveSplit, kWaveRounded };

enum LzWavePass { kWaveFwd, kWaveDq, kWaveDkdv };

// One kernel; and the backward's two, dQ (which forms delta when delta_w is
// set) before dK/dV.
int lz_attn_wave_pass(const LzWaveArgs& a, int dtype, int64_t hd, LzWaveMode mode, LzWavePass pass, hipStream_t s);
int lz_attn_wave_bwd(const LzWaveArgs& a, int dtype, int64_t hd, LzWaveMode mode, hipStream_t s);
