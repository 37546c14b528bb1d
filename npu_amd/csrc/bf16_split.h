// fp32 activations as three bf16 planes for v_mfma_f32_16x16x32_bf16.
#pragma once
#include "common.h"

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));

// A sign, 1 or -1, in the two forms that split3 takes it.
struct Sign {
  uint32_t bit;
  float f;
};

// The bf16 MFMA rounds its sums towards -infinity, so a product formed of x alone
// is low by about 2.5e-8 of its magnitude on average, in every output alike, which
// whatever averages the outputs (attention over the prompt's own V rows) does not
// average out.  Sums of steps are therefore formed of x and -x in turn and added
// with that sign: the two roundings cancel (bias at K = 2048 2.4e-8 -> 3e-11).
constexpr __device__ __forceinline__ Sign step_sign(int step) {
  return Sign{(uint32_t)step << 31, step & 1 ? -1.f : 1.f};
}

// sign x = h + m + l over 8 fp32 values -> three bf16x8 planes, exactly: h is
// truncated to bf16, m is the rest truncated, l = sign x - h - m has at most 8
// significant bits left.
__device__ __forceinline__ void split3(const gm_f32x4& xa, const gm_f32x4& xb, gm_u32x4 (&pl)[3],
                                       Sign sign = {0u, 1.f}) {
  const float v[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
  uint32_t hb[8], mb[8], lb[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hb[i] = (__float_as_uint(v[i]) ^ sign.bit) & 0xffff0000u;
    const float r = sign.f * v[i] - __uint_as_float(hb[i]);
    mb[i] = __float_as_uint(r) & 0xffff0000u;
    lb[i] = __float_as_uint(r - __uint_as_float(mb[i]));     // low 16 bits are zero
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    pl[0][d] = __builtin_amdgcn_perm(hb[2 * d + 1], hb[2 * d], 0x07060302u);
    pl[1][d] = __builtin_amdgcn_perm(mb[2 * d + 1], mb[2 * d], 0x07060302u);
    pl[2][d] = __builtin_amdgcn_perm(lb[2 * d + 1], lb[2 * d], 0x07060302u);
  }
}
