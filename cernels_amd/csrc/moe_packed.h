// Packed expert weights (MFMA-fragment order): the layout's index map and the conventions that the packed GEMMs
// share for glu, the activation output between the two projections (see moe_gemm_packed.hip for its precision).
#pragma once

#include "moe_common.h"

namespace cmoe {

constexpr int kPkFrag = 512;  // bf16 elements of one fragment (1 KB)
// glu segments: scaled up below this largest |glu| (2^-8), down at or above 2^15; an all-zero segment
// records kGluAnyScale in gexp
constexpr float kGluSmall = 0.00390625f;
constexpr int kGluAnyScale = -128;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kModePkGateUp = 0;
constexpr int kModePkDown = 1;
constexpr int kModePkUp = 2;  // non-gated first projection (megablocks): glu[r, :] = act(X[tok(r), :] · W1_e)

// Packed layout of one projection, viewed as B[k][n] (reduction length Kd, KS = Kd/16 k-steps) cut
// into NF fragments of 32 columns:
//   gate_up: fragment c = gate columns [16c, 16c+16) then up columns [16c, 16c+16). Kd = H, NF = F/16.
//   down:    fragment c = output columns [32c, 32c+32).                           Kd = F, NF = H/32.
//   up:      (non-gated) fragment c = columns [32c, 32c+32), packed as a down projection with H and F
//            exchanged.                                                           Kd = H, NF = F/32.
// Fragments are bundled by eight (an N-tile: one fragment per wave) and stored k-step-major inside a
// tile, so the eight waves of a workgroup read one contiguous 8 KB run per k-step. Lane l of
// fragment (c, ks) holds B[16ks + 8(l/32) + j][column l%32 of the fragment], j = 0..7.
// Returns the fragment's index in 1 KB units.
__host__ __device__ inline long long packed_frag(int e, int c, int ks, int NF, int KS) {
    const int t = c >> 3, w = c & 7, nw = min(8, NF - 8 * t);
    return (long long)e * NF * KS + 8LL * KS * t + (long long)ks * nw + w;
}

// The forms of the packed path (mirrors cernels_moe_packed_form in include/cernels_moe.h).
constexpr int kFormGrouped = 0;       // persistent grouped GEMMs, equal item ranges per XCD
constexpr int kFormGroupedSplit = 1;  // the same, with the cost-balanced ranges that the route writes
constexpr int kFormFewSum = 2;        // few tokens, the sum over slots in the down kernel
constexpr int kFormFewRows = 3;       // few tokens, a Y row per pair and the combine
constexpr int kFormTiles = 4;         // streaming kernels over 32-row M-tiles
constexpr int kFormItems = 5;         // a workgroup per item of 128 rows

// Whether a glu segment whose largest |value| is m is stored scaled, and the power of two s it is then scaled by:
// m * 2^-s in [2^14, 2^15); s >= 1 for m >= 2^15 (inf or nan: s = 1), s <= -23 for 0 < m < 2^-8 (clamped at -126, so
// 2^s stays a normal fp32 and s an int8 other than kGluAnyScale).
__device__ __forceinline__ bool glu_needs_scale(float m) { return !(m < 32768.f) || (m < kGluSmall && m > 0.f); }
__device__ __forceinline__ int glu_scale_exp(float m) {
    const int s = __builtin_amdgcn_frexp_expf(m) - 15;
    return m < 32768.f ? max(-126, s) : max(1, s);
}

}  // namespace cmoe
