// Grouped GEMMs over routed experts held as I8 rows (Q8_0 / Q4_K / Q5_K / Q6_K
// tensors, transcoded), for the MoE prefill (prefill.hip): the same segments of
// at most 32 tokens per expert, with fp32-exact activations as the decode
// kernels of these layers have them.
//
// Activations: each row times a power of two (its largest magnitude in [2^14,
// 2^15)), split into two f16 planes hi + lo (hi rounded, lo the rest rounded:
// 2^-24 of each value, where the decode kernels' limbs keep 2^-23 of each
// sub-block's largest), with the sum of every 32 values for the offsets.
// Weights: int8 quants are exact in f16; the two scales and the offset of a
// sub-block of 32 are applied in fp32 to its two half sums:
//   y += s0 (q[0..15] . x) + s1 (q[16..31] . x) + off sum(x)
// v_mfma_f32_16x16x32_f16 with the tokens as A and the weight rows as B, so the
// lane that decodes a row's quants also holds its scales for all its outputs;
// the half sums come from B operands whose other half is zero.
#include "kernels.h"
#include "moe_common.h"

using namespace gm_moe;

typedef _Float16 gm_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gm_f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t gm_u32x3 __attribute__((ext_vector_type(3)));

namespace {

constexpr int kSeg = 32;             // tokens per segment, two MFMA tiles
constexpr int kStep = 128;           // k per pipeline step: four sub-blocks
constexpr int kRowB = 2 * kStep;     // bytes of one row of one plane in LDS
constexpr int kPlane = kSeg * kRowB;

// fp32 rows -> planes hi, lo, the row's scale 2^-s and the sums of 32 (of the
// scaled values).  One wave per row; K % 256 == 0.
__global__ void __launch_bounds__(256) k_pf8_split(const float* __restrict__ src, int rows, int K,
                                                   uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                   float* __restrict__ scale, float* __restrict__ sums) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const gm_f32x4* x = reinterpret_cast<const gm_f32x4*>(src + (int64_t)r * K);
  float m = 0.f;
#pragma unroll 8
  for (int i = lane; i < K / 4; i += 64) {
    const gm_f32x4 v = x[i];
    m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  const int sh = 15 - (m > 0.f && m <= 3.4e38f ? max(__builtin_amdgcn_frexp_expf(m), -100) : 0);
  uint2* ph = reinterpret_cast<uint2*>(hi + (int64_t)r * K);
  uint2* pl = reinterpret_cast<uint2*>(lo + (int64_t)r * K);
#pragma unroll 4
  for (int i = lane; i < K / 4; i += 64) {
    const gm_f32x4 v = x[i];
    _Float16 h[4], l[4];
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float f = __builtin_ldexpf(v[c], sh);
      h[c] = (_Float16)f;
      l[c] = (_Float16)(f - (float)h[c]);
      s += f;
    }
    const gm_f16x2 h01 = {h[0], h[1]}, h23 = {h[2], h[3]}, l01 = {l[0], l[1]}, l23 = {l[2], l[3]};
    ph[i] = make_uint2(__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23));
    pl[i] = make_uint2(__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23));
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) s += __shfl_xor(s, o, 64);
    if ((lane & 7) == 0) sums[(int64_t)r * (K / 32) + i / 8] = s;
  }
  if (lane == 0) scale[r] = __builtin_ldexpf(1.0f, -sh);
}

// One pipeline step of a lane's weight row: octet q of four sub-blocks, and
// their {s0, s1, off}.
struct W8 {
  uint2 q[4];
  gm_u32x3 m[4];
};

__device__ __forceinline__ W8 w8_load(const uint8_t* __restrict__ row, int step, int q) {
  W8 w;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const uint8_t* sb = row + (step * 4 + s) * 48;
    w.q[s] = *reinterpret_cast<const uint2*>(sb + 8 * q);
    w.m[s] = *reinterpret_cast<const gm_u32x3*>(sb + 32);
  }
  return w;
}

// Four int8 -> f16: 0x6400 | (b ^ 0x80) is 1024 + 128 + b, exactly.
__device__ __forceinline__ void i8x4_f16(uint32_t b, uint32_t& o0, uint32_t& o1) {
  const uint32_t u = b ^ 0x80808080u;
  const gm_f16x2 c = {(_Float16)-1152.f, (_Float16)-1152.f};
  o0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + c);
  o1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + c);
}

struct Gemm8 {
  const uint8_t* w[2];     // routed experts [E][M][K / 32 * 48] (gate, up; or down)
  const uint8_t* wsh[2];   // the shared expert's rows, or NULL
  const uint16_t* hi;      // activation rows [.][K]
  const uint16_t* lo;
  const float* scale;
  const float* sums;       // [.][K / 32]
  float* out;              // [P + T][M]
  const int32_t* segs;
  const int32_t* offsets;
  const int32_t* sorted;   // gate/up: pair -> token row; NULL: activation rows are the pairs'
  int T, k, E, M, K, nrt;
};

template <int NMAT, int NT>
__device__ __forceinline__ void w8_step(const W8 (&w)[2], const uint8_t* __restrict__ act,
                                        const float* __restrict__ sums, int q, int l16,
                                        gm_f32x4 (&acc)[2][2]) {
  const bool low = q < 2;                                       // the lane's octet is in the first half
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    gm_f16x8 ah[NT], al[NT];
    gm_f32x4 xs[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int o = (16 * t + l16) * kRowB + 16 * ((4 * s + q) ^ l16);
      ah[t] = *reinterpret_cast<const gm_f16x8*>(act + o);
      al[t] = *reinterpret_cast<const gm_f16x8*>(act + kPlane + o);
      xs[t] = *reinterpret_cast<const gm_f32x4*>(sums + s * kSeg + 16 * t + 4 * q);
    }
#pragma unroll
    for (int n = 0; n < NMAT; ++n) {
      uint32_t b[4];
      i8x4_f16(w[n].q[s].x, b[0], b[1]);
      i8x4_f16(w[n].q[s].y, b[2], b[3]);
      const gm_u32x4 b0 = {low ? b[0] : 0u, low ? b[1] : 0u, low ? b[2] : 0u, low ? b[3] : 0u};
      const gm_u32x4 b1 = {low ? 0u : b[0], low ? 0u : b[1], low ? 0u : b[2], low ? 0u : b[3]};
      const gm_f16x8 B0 = __builtin_bit_cast(gm_f16x8, b0), B1 = __builtin_bit_cast(gm_f16x8, b1);
      const float s0 = __uint_as_float(w[n].m[s].x), s1 = __uint_as_float(w[n].m[s].y),
                  off = __uint_as_float(w[n].m[s].z);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const gm_f32x4 z = {0.f, 0.f, 0.f, 0.f};
        gm_f32x4 d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[t], B0, z, 0, 0, 0);
        gm_f32x4 d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[t], B1, z, 0, 0, 0);
        d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t], B0, d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[t], B1, d1, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[n][t][i] += fmaf(s0, d0[i], fmaf(s1, d1[i], off * xs[t][i]));
      }
    }
  }
}

// Block = (segment, 64 weight rows): wave w rows 16 w .. 16 w + 15 of NMAT
// matrices, all of the segment's tokens.  NMAT = 2: out = silu(gate) up; 1: out =
// down row times the activation row's scale.  The next step's weights (registers)
// and activation planes (straight into the other LDS buffer) load while a step is
// multiplied.
template <int NMAT>
__global__ void __launch_bounds__(256, 2) k_pf8_gemm(Gemm8 P) {
  __shared__ __attribute__((aligned(16))) uint8_t act[2][2 * kPlane];
  __shared__ __attribute__((aligned(16))) float sums[2][4 * kSeg];
  __shared__ int32_t in_row[kSeg], out_row[kSeg];
  const int slot = blockIdx.x >> 3;                             // as xcd_tile of prefill.hip
  const int seg = (slot / P.nrt) * 8 + (blockIdx.x & 7), rt = slot % P.nrt;
  if (seg >= P.segs[0]) return;
  const int e = P.segs[1 + 4 * seg], start = P.segs[2 + 4 * seg], n = P.segs[3 + 4 * seg];
  const bool shared = e == P.E;
  if (threadIdx.x < kSeg) {
    const int c = threadIdx.x < n ? threadIdx.x : 0;            // rows past n repeat the first
    const int pos = shared ? P.T * P.k + start + c : P.offsets[e] + start + c;
    in_row[threadIdx.x] = !P.sorted ? pos : shared ? start + c : P.sorted[pos] / P.k;
    out_row[threadIdx.x] = pos;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  const int K = P.K, row = rt * 64 + wave * 16 + l16, nt = (n + 15) >> 4;
  const int64_t rb = (int64_t)(K / 32) * 48;
  const uint8_t* wr[NMAT];
#pragma unroll
  for (int i = 0; i < NMAT; ++i)
    wr[i] = (shared ? P.wsh[i] : P.w[i] + (int64_t)e * P.M * rb) + row * rb;
  const int tt = threadIdx.x & 31, ts = (threadIdx.x >> 5) & 3;  // this thread's activation sum (first 128)
  const float* sp = P.sums + (int64_t)in_row[tt] * (K / 32) + ts;
  auto load_act = [&](int step, int buf) {                      // 1 KB: 4 rows of one plane
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int id = 4 * m + wave, pl = id >> 3, r4 = id & 7;
      if (r4 * 4 >= 16 * nt) continue;                          // wave-uniform
      const int r = 4 * r4 + (lane >> 4), g = l16 ^ (r & 15);
      __builtin_amdgcn_global_load_lds((pl ? P.lo : P.hi) + (int64_t)in_row[r] * K + step * kStep + 8 * g,
                                       act[buf] + pl * kPlane + r4 * 1024, 16, 0, 0);
    }
  };
  gm_f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[i][t] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
  W8 w[2], wn[2];
  load_act(0, 0);
#pragma unroll
  for (int i = 0; i < NMAT; ++i) w[i] = w8_load(wr[i], 0, q);
  if (threadIdx.x < 128) sums[0][ts * kSeg + tt] = sp[0];
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  const int ns = K / kStep;
  for (int s = 0; s < ns; ++s) {
    const int sn = s + 1 < ns ? s + 1 : s, b = s & 1;           // the last step re-reads itself, unused
#pragma unroll
    for (int i = 0; i < NMAT; ++i) wn[i] = w8_load(wr[i], sn, q);
    const float su = sp[sn * 4];
    if (s + 1 < ns) load_act(sn, b ^ 1);
    if (nt == 1) w8_step<NMAT, 1>(w, act[b], sums[b], q, l16, acc);
    else w8_step<NMAT, 2>(w, act[b], sums[b], q, l16, acc);
    if (threadIdx.x < 128) sums[b ^ 1][ts * kSeg + tt] = su;
#pragma unroll
    for (int i = 0; i < NMAT; ++i) w[i] = wn[i];
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  // lane l holds tokens 4 (l / 16) + i of a tile, weight row l % 16
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 16 * t + 4 * q + i;
      if (c >= n) continue;
      const float ds = P.scale[in_row[c]];
      float v = acc[0][t][i] * ds;
      if constexpr (NMAT == 2) v = gm_silu(v) * (acc[1][t][i] * ds);
      P.out[(int64_t)out_row[c] * P.M + row] = v;
    }
}

}  // namespace

int gm_pf8_split(const float* src, int rows, int K, const GmPf8Rows& a, hipStream_t s) {
  hipLaunchKernelGGL(k_pf8_split, dim3((rows + 3) / 4), dim3(256), 0, s, src, rows, K, a.hi, a.lo, a.scale, a.sums);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

int gm_pf8_gemm(const gm_moe_layer* L, bool down, const GmPf8Rows& a, const int32_t* segs, int nseg,
                const int32_t* offsets, const int32_t* sorted, int T, float* out, hipStream_t s) {
  const int M = down ? L->D : L->FF, K = down ? L->FF : L->D;
  auto u8 = [](const void* p) { return static_cast<const uint8_t*>(p); };
  Gemm8 P{};
  P.w[0] = u8(down ? L->down_exps : L->gate_exps);
  P.w[1] = u8(down ? nullptr : L->up_exps);
  P.wsh[0] = u8(down ? L->down_sh : L->gate_sh);
  P.wsh[1] = u8(down ? nullptr : L->up_sh);
  P.hi = a.hi; P.lo = a.lo; P.scale = a.scale; P.sums = a.sums;
  P.out = out; P.segs = segs; P.offsets = offsets; P.sorted = down ? nullptr : sorted;
  P.T = T; P.k = L->k; P.E = L->E; P.M = M; P.K = K; P.nrt = M / 64;
  const dim3 g((unsigned)((nseg + 7) / 8 * 8 * P.nrt));
  if (down) hipLaunchKernelGGL(k_pf8_gemm<1>, g, dim3(256), 0, s, P);
  else hipLaunchKernelGGL(k_pf8_gemm<2>, g, dim3(256), 0, s, P);
  GM_TRY(hipGetLastError());
  return GM_OK;
}
