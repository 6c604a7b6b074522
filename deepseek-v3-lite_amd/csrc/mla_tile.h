// Types, swizzled LDS tiles and lane-pair reductions shared by the MLA attention
// kernels (mla.hip, mla_few.hip).
#pragma once

#include "common.h"
#include "mfma.h"

namespace dsmoe {

typedef short mla_v4s __attribute__((ext_vector_type(4)));
typedef float mla_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int mla_u32x4 __attribute__((ext_vector_type(4)));

constexpr float MLA_LOG2E = 1.4426950408889634f;

// Staged tiles are read both as MFMA fragments (ds_read_b128: eight columns
// of a row per lane) and transposed (ds_read_b64_tr_b16: four consecutive
// rows of a column per lane), so 16-byte chunk c of row r sits at
// c ^ mlb_g(r) inside each group of 16 chunks; sixteen consecutive rows at one
// chunk, and four consecutive rows (r = 0 mod 4) at four consecutive chunks
// (c = 0 mod 4), then fall on distinct banks.
__device__ __forceinline__ int mlb_off(int r, int c, int rb) {
  const int g = ((r & 3) << 2) | ((r >> 2) & 3);
  return r * rb + (((c & ~15) | ((c & 15) ^ g)) << 4);
}

// Reads of a staged tile with row bytes RB, the lane-dependent part of their
// offsets computed once per kernel (the swizzle sees only a row's low four
// bits and a chunk's low four, so rows R + .. with R = 0 mod 16 and chunk
// group k add R RB + 256 k as immediates):
//  * frag(t, R, st): the MFMA fragment of row R + (l & 31), 16-byte chunk
//    2 st + hi (columns 16 st + 8 hi .. + 7);
//  * tfrag(t, r0, ct): columns 32 ct .. + 31 over rows r0 .. r0 + 15
//    (r0 = 0 mod 16) by two ds_read_b64_tr_b16, the rows in the order the
//    score MFMA leaves in a lane's registers (lanes 0-31: r0 + {0-3, 8-11},
//    lanes 32-63: r0 + {4-7, 12-15}); lane l gets column 32 ct + (l & 31).
//    In a 16-lane group lane s addresses row s >> 2, columns 4 (s & 3) ..
//    + 3 (8-byte unit u), and receives one column of the four rows.
template <int RB>
struct MlbLane {
  int f[8], t0[4], t1[4];
  __device__ __forceinline__ explicit MlbLane(int lane) {
    const int hi = lane >> 5, l32 = lane & 31;
#pragma unroll
    for (int st = 0; st < 8; ++st) f[st] = mlb_off(l32, 2 * st + hi, RB);
    const int gq = lane >> 4, sl = lane & 15;
    const int r = 4 * (gq >> 1) + (sl >> 2);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      const int u = 8 * ct + 4 * (gq & 1) + (sl & 3);
      t0[ct] = mlb_off(r, u >> 1, RB) + ((u & 1) << 3);
      t1[ct] = mlb_off(r + 8, u >> 1, RB) + ((u & 1) << 3);
    }
  }
  __device__ __forceinline__ bf16x8_t frag(const char* t, int R, int st) const {
    return *reinterpret_cast<const bf16x8_t*>(t + f[st & 7] + R * RB + 256 * (st >> 3));
  }
  __device__ __forceinline__ bf16x8_t tfrag(const char* t, int r0, int ct) const {
    const int k = r0 * RB + 256 * (ct >> 2);
    const mla_v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) mla_v4s*)(t + t0[ct & 3] + k));
    const mla_v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) mla_v4s*)(t + t1[ct & 3] + k));
    typedef short v8s __attribute__((ext_vector_type(8)));
    const v8s v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8_t, v);
  }
};

// Maximum and sum over the two lanes that hold a query's keys (l, l + 32).
__device__ __forceinline__ float mla_pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float mla_pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}

}  // namespace dsmoe
