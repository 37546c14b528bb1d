// fp32 activations as three bf16 planes for v_mfma_f32_16x16x32_bf16.
#pragma once
#include "common.h"

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));

// x = h + m + l over 8 fp32 values -> three bf16x8 planes, exactly: h is x
// truncated to bf16, m is x - h truncated, l = x - h - m has at most 8
// significant bits left.
__device__ __forceinline__ void split3(const gm_f32x4& xa, const gm_f32x4& xb, gm_u32x4 (&pl)[3]) {
  const float v[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
  uint32_t hb[8], mb[8], lb[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hb[i] = __float_as_uint(v[i]) & 0xffff0000u;
    const float r = v[i] - __uint_as_float(hb[i]);
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
