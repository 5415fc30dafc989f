// The vectorised 1x128 activation quant as a device function, shared by the
// quant kernel (quant.hip) and the launch that runs it beside align
// (align.hip).
//
// Sixteen lanes own one 128-element group (a chunk of 16 B = 8 bf16 each), so
// every wave reads 1 KiB and writes 512 B contiguously with 128-bit loads; the
// group amax is a 16-lane xor-shuffle reduction.
//
// A row has W valid columns (W % 8 == 0, so a chunk is valid or not as a
// whole) and cpr = ceil(W/128)*16 chunks; the chunks past W are the zero
// padding of the reference's quant, which changes neither the amax nor the
// other codes.  Their zero codes are written where the output row has room
// for them (col < ldq).
#pragma once

#include "common.hpp"

namespace moe {

struct QuantArgs {
  const uint16_t* x;   // bf16 rows, stride W (2W for the SiLU*up form: gate | up)
  uint8_t* q;          // codes, row stride ldq (a multiple of 8)
  float* s;            // scales, cpr / 16 a row
  int64_t n_chunks;    // rows * cpr
  int64_t cpr;         // chunks of a row, padding included
  int64_t W;           // valid columns
  int64_t ldq;
};

// Block `blk` of THREADS threads takes UNROLL * THREADS chunks.  WHOLE: rows
// are whole groups and dense (W == ldq == 8 * cpr), so chunk ch sits at column
// 8 * ch of the flat tensor.
template <int THREADS, int UNROLL, bool SWIGLU, bool WHOLE>
MOE_DEVICE void quant_chunks(const QuantArgs& a, int64_t blk) {
  const int tid = threadIdx.x;
  const int64_t base = blk * THREADS * UNROLL;
  constexpr int NLOAD = SWIGLU ? 2 : 1;
  static_assert(WHOLE || !SWIGLU, "the SiLU*up form takes whole groups");
  v4i raw[UNROLL][NLOAD];
  int64_t row[UNROLL], col[UNROLL];
#pragma unroll
  for (int i = 0; i < UNROLL; ++i) {
    const int64_t ch = base + tid + i * THREADS;
    if constexpr (!WHOLE || SWIGLU) {
      // 32-bit division where it suffices (a 64-bit one is a long software routine)
      const bool small = a.n_chunks <= 0xFFFFFFFFll;
      row[i] = small ? (int64_t)((uint32_t)ch / (uint32_t)a.cpr) : ch / a.cpr;
      col[i] = (ch - row[i] * a.cpr) * 8;
    } else {
      row[i] = 0;
      col[i] = ch * 8;
    }
#pragma unroll
    for (int l = 0; l < NLOAD; ++l) raw[i][l] = (v4i){0, 0, 0, 0};
    if (ch < a.n_chunks) {
      if constexpr (SWIGLU) {
        const uint16_t* r = a.x + row[i] * 2 * a.W;
        raw[i][0] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(r + col[i]));
        raw[i][NLOAD - 1] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(r + a.W + col[i]));
      } else if (WHOLE || col[i] < a.W) {
        raw[i][0] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(a.x + row[i] * a.W + col[i]));
      }
    }
  }
#pragma unroll
  for (int i = 0; i < UNROLL; ++i) {
    const int64_t ch = base + tid + i * THREADS;
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = (uint32_t)raw[i][0][j];
      if constexpr (SWIGLU) {
        const uint32_t u = (uint32_t)raw[i][NLOAD - 1][j];
        v[2 * j] = silu_mul_bf16(lo_bf16(w), lo_bf16(u));
        v[2 * j + 1] = silu_mul_bf16(hi_bf16(w), hi_bf16(u));
      } else {
        v[2 * j] = lo_bf16(w);
        v[2 * j + 1] = hi_bf16(w);
      }
    }
    float amax = 0.0f;
    if constexpr (WHOLE) {
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    } else {
      // The general kernel's scale for every bit pattern: its maximum of two
      // passes a NaN over, while the three-operand maximum that this chain
      // becomes drops a number beside a signalling NaN, so NaNs are quieted.
      amax = fabsf(__builtin_canonicalizef(v[0]));
#pragma unroll
      for (int j = 1; j < 8; ++j) amax = fmaxf(amax, fabsf(__builtin_canonicalizef(v[j])));
    }
    // 16 lanes of one group are 16 consecutive lanes of the wave.
    amax = fmaxf(amax, __shfl_xor(amax, 1));
    amax = fmaxf(amax, __shfl_xor(amax, 2));
    amax = fmaxf(amax, __shfl_xor(amax, 4));
    amax = fmaxf(amax, __shfl_xor(amax, 8));
    const float sc = group_scale(amax);
    const float inv = 1.0f / sc;
    uint32_t lo, hi;
    if constexpr (WHOLE) {
      lo = quant4_e4m3(v[0], v[1], v[2], v[3], sc, inv);
      hi = quant4_e4m3(v[4], v[5], v[6], v[7], sc, inv);
    } else {  // the general kernel's codes, which differ for a NaN or an infinity
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = clamp_fp8(div_by(v[j], sc, inv));
      const bool pad = col[i] >= a.W;  // 0 / scale is no zero where the scale is infinite
      lo = pad ? 0u : pack4_e4m3(v[0], v[1], v[2], v[3]);
      hi = pad ? 0u : pack4_e4m3(v[4], v[5], v[6], v[7]);
    }
    if (ch < a.n_chunks) {
      // dense rows: chunk ch of the codes too, and no row and column kept through the codes' registers
      if (WHOLE || col[i] < a.ldq)
        __builtin_nontemporal_store((v2u){lo, hi},
                                    reinterpret_cast<v2u*>(a.q + (WHOLE ? ch * 8 : row[i] * a.ldq + col[i])));
      if ((tid & 15) == 0) a.s[ch >> 4] = sc;
    }
  }
}

// Whether the vectorised form takes rows of H columns at these pointers and
// strides: chunks and output words aligned, and a whole number of chunks.
inline bool quant_vectorised(const void* x, int64_t H, const void* q, int64_t ldq) {
  return H % 8 == 0 && ldq % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)q & 7) == 0;
}

inline QuantArgs quant_args(const void* x, int64_t T, int64_t H, void* q, int64_t ldq, float* s) {
  const int64_t cpr = (H + 127) / 128 * 16;
  return QuantArgs{(const uint16_t*)x, (uint8_t*)q, s, T * cpr, cpr, H, ldq};
}
inline bool quant_whole(const QuantArgs& a) { return a.W == 8 * a.cpr && a.ldq == a.W; }

}  // namespace moe
