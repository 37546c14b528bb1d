// Grouped GEMMs over routed experts held as I8 rows (Q8_0 / Q4_K / Q5_K / Q6_K
// tensors, transcoded), for the MoE prefill (prefill.hip): segments of at most 16
// tokens per expert, with activations no less exact than the decode kernels of
// these layers have them.
//
// Activations: each sub-block of 32 times a power of two (its largest magnitude in
// [2^14, 2^15)), split into two f16 planes hi + lo (hi rounded, lo the rest
// rounded): within 2^-23 of each value down to 2^-16 of the sub-block's largest,
// within 2^-39 of that below; the decode kernels' limbs keep 2^-23 of the
// sub-block's largest.  With them the sub-block's sum, for the offsets, and its
// scale 2^-s.
// Every other sub-block is held negated, with a negative scale: the f16 MFMA rounds
// its sums towards -infinity as the bf16 one does (bf16_split.h), which quants and
// offsets of one sign do not average out (Q8_0 / Q5_K experts at D = 2048: error
// against 64 bits 1.05e-6, now 1.8e-7; the decode kernels 5.4e-7).
// Weights: int8 quants are exact in f16; the two scales and the offset of a
// sub-block of 32 are applied in fp32 to its two half sums, then the activations':
//   y += 2^-s (s0 (q[0..15] . x) + s1 (q[16..31] . x) + off sum(x))
// v_mfma_f32_16x16x32_f16 with the tokens as A and the weight rows as B, so the
// lane that decodes a row's quants also holds its scales for all its outputs;
// the half sums come from B operands whose other half is zero.
#include "kernels.h"
#include "moe_common.h"

using namespace gm_moe;

typedef _Float16 gm_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gm_f16x2 __attribute__((ext_vector_type(2)));
typedef float gm_f32x2 __attribute__((ext_vector_type(2)));

namespace {

// fp32 rows -> planes hi, lo and meta [row][K / 32][2]: the sum of a sub-block's
// scaled values and its scale.  One wave per row, 8 lanes per sub-block; K % 256
// == 0.  (One scale per row left a sub-block 2^-24 of the row's largest 15 bits.)
__global__ void __launch_bounds__(256) k_pf8_split(const float* __restrict__ src, int rows, int K,
                                                   uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                                   float* __restrict__ meta) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const gm_f32x4* x = reinterpret_cast<const gm_f32x4*>(src + (int64_t)r * K);
  uint2* ph = reinterpret_cast<uint2*>(hi + (int64_t)r * K);
  uint2* pl = reinterpret_cast<uint2*>(lo + (int64_t)r * K);
  gm_f32x2* pm = reinterpret_cast<gm_f32x2*>(meta) + (int64_t)r * (K / 32);
  const int n = K / 256;
  constexpr int NL = 4;                                         // steps whose loads go out together
  for (int s0 = 0; s0 < n; s0 += NL) {
    gm_f32x4 v[NL];
#pragma unroll
    for (int u = 0; u < NL; ++u) v[u] = x[64 * min(s0 + u, n - 1) + lane];
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      if (s0 + u >= n) break;                                   // uniform
      const int i = 64 * (s0 + u) + lane;
      const float m = gm_max8(fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
      const int sh = 15 - (m > 0.f && m <= 3.4e38f ? max(__builtin_amdgcn_frexp_expf(m), -100) : 0);
      _Float16 h[4], l[4];
      float f[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        f[c] = __builtin_ldexpf(lane & 8 ? -v[u][c] : v[u][c], sh);
        h[c] = (_Float16)f[c];
        l[c] = (_Float16)(f[c] - (float)h[c]);
      }
      const gm_f16x2 h01 = {h[0], h[1]}, h23 = {h[2], h[3]}, l01 = {l[0], l[1]}, l23 = {l[2], l[3]};
      ph[i] = make_uint2(__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23));
      pl[i] = make_uint2(__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23));
      const float s = gm_sum8((f[0] + f[1]) + (f[2] + f[3]));
      if ((lane & 7) == 0) pm[i / 8] = gm_f32x2{s, __builtin_ldexpf(lane & 8 ? -1.0f : 1.0f, -sh)};
    }
  }
}

// Four int8 -> f16: 0x6400 | (b ^ 0x80) is 1024 + 128 + b, exactly.
__device__ __forceinline__ void i8x4_f16(uint32_t b, uint32_t& o0, uint32_t& o1) {
  const uint32_t u = b ^ 0x80808080u;
  const gm_f16x2 c = {(_Float16)-1152.f, (_Float16)-1152.f};
  o0 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + c);
  o1 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + c);
}

// N bytes per lane from global memory to dst + N lane (dst: wave-uniform, in LDS).
template <int N>
__device__ __forceinline__ void to_lds(const void* src, uint8_t* dst) {
  if constexpr (N == 16) __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
  else __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
}

// A block barrier behind the wave's LDS accesses only (__syncthreads() and the
// fences would also wait for the loads into LDS that are to stay in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct Gemm8 {
  const uint8_t* w[2];     // routed experts [E][M][K / 32 * 48] (gate, up; or down)
  const uint8_t* wsh[2];   // the shared expert's rows, or NULL
  const uint16_t* hi;      // activation rows [.][K]
  const uint16_t* lo;
  const float* meta;       // [.][K / 32][2]: sum, scale
  float* out;              // [P + T][M]
  const int32_t* segs;
  const int32_t* offsets;
  const int32_t* sorted;   // gate/up: pair -> token row; NULL: activation rows are the pairs'
  int T, k, E, M, K, nrt;
};

// Block = (segment of at most 16 tokens, RTB tiles of 64 weight rows): wave w rows
// 16 w .. 16 w + 15 of a tile of NMAT matrices, all of the segment's tokens.
// NMAT = 2: out = silu(gate) up; 1: out = the down row.
//
// Bound by the weights' way from HBM.  A step is 128 k (four sub-blocks); its
// weights (into the wave's own LDS), activation planes, sums and scales (into the
// block's) come straight from global memory, one step ahead.  A load instruction
// covers 5 1/3 weight rows of 192 contiguous bytes; loaded to registers as the MFMA
// wants them, 16 rows by an instruction, they came at 2.3 TB/s whatever was in
// flight (a probe of the two patterns alone: 3.1 and 6.9 TB/s).  Two buffers and
// two (gate/up) or three (down) blocks to a CU: one block with four or seven buffers
// had as much in flight but one wave per SIMD.  Segments of 32 tokens leave one
// gate/up block to a CU, and are slower however many tokens an expert has (block at
// D = 2048, FF = 512, 256 experts, k = 8: T = 500 559 against 422 us, 1000 794 / 678,
// 2500 1568 / 1431; at D = 512, FF = 256, 16 experts, k = 4: 100 49 / 43, 1000 85 / 81).
// D = 2048, FF = 512, 256 experts, 150 tokens (Q5_K / Q6_K, 1.2 GB of I8 rows), us:
//   gate/up 348 (16 rows an instruction) -> 270 (through LDS) -> 217 (a step's LDS
//   reads together, the next loads not waited for before them); down 177 -> 123
//   -> 111; 256 k a step: 316; one block of four buffers: 275 (down, seven: 184)
// Kernel durations with one scale per activation row 198 and 103, per sub-block 192
// and 101 (the activations' addresses are formed once, not per step).
// Granule g (16 bytes) of row r's step sits at position (g + 2 (r >> 2)) % 12 of
// its 12: the 16 rows' reads of 32 bytes fall evenly on the banks.
template <int NMAT, int RTB>
__global__ void __launch_bounds__(256) k_pf8_gemm(Gemm8 P) {
  constexpr int kStep = 128, kRowB = 2 * kStep, kWRow = 192, NW = 4;
  constexpr int SEG = kPf8Seg, PLANE = SEG * kRowB, NA = 2 * PLANE / 1024 / NW;   // act loads per wave and step
  constexpr int WB = NMAT * 16 * kWRow;                         // a wave's weight bytes per step
  constexpr int STAGE = 2 * PLANE + NW * WB + 8 * SEG * 4;      // planes, weights, meta [4][sum, scale][SEG]
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];   // [2][STAGE], then
  int32_t* in_row = reinterpret_cast<int32_t*>(smem + 2 * STAGE);  // [SEG]
  int32_t* out_row = in_row + SEG;
  const int slot = blockIdx.x >> 3;                             // as xcd_tile of prefill.hip
  const int seg = (slot / P.nrt) * 8 + (blockIdx.x & 7), rt = slot % P.nrt;
  if (seg >= P.segs[0]) return;
  const int e = P.segs[1 + 4 * seg], start = P.segs[2 + 4 * seg], n = P.segs[3 + 4 * seg];
  const bool shared = e == P.E;
  if (threadIdx.x < SEG) {
    const int c = (int)threadIdx.x < n ? threadIdx.x : 0;       // rows past n repeat the first
    const int pos = shared ? P.T * P.k + start + c : P.offsets[e] + start + c;
    in_row[threadIdx.x] = !P.sorted ? pos : shared ? start + c : P.sorted[pos] / P.k;
    out_row[threadIdx.x] = pos;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  const int K = P.K, ns = K / kStep, total = RTB * ns, row0 = (rt * RTB * NW + wave) * 16;
  const int64_t rb = (int64_t)(K / 32) * 48;
  const uint8_t* wp[NMAT];                                      // the wave's first row
#pragma unroll
  for (int i = 0; i < NMAT; ++i) wp[i] = (shared ? P.wsh[i] : P.w[i] + (int64_t)e * P.M * rb) + row0 * rb;
  auto turn = [](int r) { return 2 * (r >> 2); };
  int wo[3];                                                    // the lane's granules of a 16-row step
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int id = 64 * j + lane, r = id / 12;
    wo[j] = r * (int)rb + 16 * ((id % 12 + 12 - turn(r)) % 12);
  }
  int qo[4], mo[4];                                             // where row l16's octet q and scales are
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    qo[s] = l16 * kWRow + 16 * ((3 * s + (q >> 1) + turn(l16)) % 12) + 8 * (q & 1);
    mo[s] = l16 * kWRow + 16 * ((3 * s + 2 + turn(l16)) % 12);
  }
  // a step's 8 SEG sums and scales, one per lane of the first SEG / 8 waves (all their
  // lanes: see lds_load16 of prefill.hip)
  const int mi = 64 * wave + lane;
  const float* mp = P.meta + ((int64_t)in_row[mi % SEG] * (K / 32) + mi / (2 * SEG)) * 2 + mi / SEG % 2;
  const bool brings = __builtin_amdgcn_readfirstlane(wave) < SEG / 8;
  const uint16_t* ap[NA];                                       // the lane's activations: 4 rows an instruction
#pragma unroll
  for (int m = 0; m < NA; ++m) {
    const int id = NA * wave + m, r = 4 * (id % (SEG / 4)) + (lane >> 4);
    ap[m] = (id / (SEG / 4) ? P.lo : P.hi) + (int64_t)in_row[r] * K + 8 * (l16 ^ (r & 15));
  }
  auto load = [&](int it, int b) {
    const int tile = it / ns, s = it - tile * ns;
    uint8_t* st = smem + b * STAGE;
#pragma unroll
    for (int i = 0; i < NMAT; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j)
        to_lds<16>(wp[i] + (int64_t)tile * 16 * NW * rb + s * kWRow + wo[j],
                   st + 2 * PLANE + wave * WB + i * 16 * kWRow + j * 1024);
#pragma unroll
    for (int m = 0; m < NA; ++m) to_lds<16>(ap[m] + s * kStep, st + (NA * wave + m) * 1024);
    if (brings) to_lds<4>(mp + s * 8, st + 2 * PLANE + NW * WB + wave * 256);
  };
  gm_f32x4 acc[NMAT];
#pragma unroll
  for (int i = 0; i < NMAT; ++i) acc[i] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
  load(0, 0);
  const bool low = q < 2;                                       // the lane's octet is in the first half
  for (int it = 0; it < total; ++it) {
    __builtin_amdgcn_s_waitcnt(0xf70);                          // vmcnt(0)
    lds_barrier();                                              // everyone's part of step it; step it - 1 is done with
    if (it + 1 < total) load(it + 1, (it + 1) & 1);
    const uint8_t* st = smem + (it & 1) * STAGE;
    const uint8_t* wb = st + 2 * PLANE + wave * WB;
    const float* meta = reinterpret_cast<const float*>(st + 2 * PLANE + NW * WB);
    gm_f32x4 part[NMAT];                                        // the step's sums: a fourth of the running sum's additions
    gm_f16x8 ah[4], al[4];                                      // the LDS reads of all four sub-blocks go out together
    gm_f32x4 xs[4], xe[4], sc[4][NMAT];                         // sums, scales; sc: s0, s1, off
    gm_u32x2 w[4][NMAT];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int i = 0; i < NMAT; ++i) {
        w[s][i] = *reinterpret_cast<const gm_u32x2*>(wb + i * 16 * kWRow + qo[s]);
        sc[s][i] = *reinterpret_cast<const gm_f32x4*>(wb + i * 16 * kWRow + mo[s]);
      }
      const int o = l16 * kRowB + 16 * ((4 * s + q) ^ l16);
      ah[s] = *reinterpret_cast<const gm_f16x8*>(st + o);
      al[s] = *reinterpret_cast<const gm_f16x8*>(st + PLANE + o);
      xs[s] = *reinterpret_cast<const gm_f32x4*>(meta + 2 * s * SEG + 4 * q);
      xe[s] = *reinterpret_cast<const gm_f32x4*>(meta + (2 * s + 1) * SEG + 4 * q);
    }
    issue_fence();
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < NMAT; ++i) {
        uint32_t o[4];
        i8x4_f16(w[s][i].x, o[0], o[1]);
        i8x4_f16(w[s][i].y, o[2], o[3]);
        const gm_u32x4 b0 = {low ? o[0] : 0u, low ? o[1] : 0u, low ? o[2] : 0u, low ? o[3] : 0u};
        const gm_u32x4 b1 = {low ? 0u : o[0], low ? 0u : o[1], low ? 0u : o[2], low ? 0u : o[3]};
        const gm_f16x8 B0 = __builtin_bit_cast(gm_f16x8, b0), B1 = __builtin_bit_cast(gm_f16x8, b1);
        const gm_f32x4 z = {0.f, 0.f, 0.f, 0.f};
        gm_f32x4 d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[s], B0, z, 0, 0, 0);
        gm_f32x4 d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[s], B1, z, 0, 0, 0);
        d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s], B0, d0, 0, 0, 0);
        d1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[s], B1, d1, 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float v = fmaf(sc[s][i].x, d0[c], fmaf(sc[s][i].y, d1[c], sc[s][i].z * xs[s][c]));
          part[i][c] = s == 0 ? xe[s][c] * v : fmaf(xe[s][c], v, part[i][c]);
        }
      }
#pragma unroll
    for (int i = 0; i < NMAT; ++i) acc[i] += part[i];
    if ((it + 1) % ns == 0) {
      // a row tile is done: lane l holds tokens 4 (l / 16) + i, weight row l % 16
      const int row = row0 + (it / ns) * 16 * NW + l16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 4 * q + i;
        if (c < n) {
          float v = acc[0][i];
          if constexpr (NMAT == 2) v = gm_silu(v) * acc[NMAT - 1][i];
          P.out[(int64_t)out_row[c] * P.M + row] = v;
        }
#pragma unroll
        for (int m = 0; m < NMAT; ++m) acc[m][i] = 0.f;
      }
    }
  }
}

template <int NMAT, int RTB>
int launch8(Gemm8 P, int nseg, hipStream_t s) {
  constexpr size_t smem = 2 * (2 * kPf8Seg * 256 + 4 * NMAT * 16 * 192 + 8 * kPf8Seg * 4) + 2 * kPf8Seg * 4;
  static_assert((NMAT == 2 ? 2 : 3) * smem <= 160 * 1024, "LDS of a CU");
  P.nrt = P.M / (64 * RTB);
  if (int rc = gm_set_smem(k_pf8_gemm<NMAT, RTB>, smem)) return rc;
  hipLaunchKernelGGL((k_pf8_gemm<NMAT, RTB>), dim3((unsigned)((nseg + 7) / 8 * 8 * P.nrt)), dim3(256), smem, s, P);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

}  // namespace

int gm_pf8_split(const float* src, int rows, int K, const GmPf8Rows& a, hipStream_t s) {
  hipLaunchKernelGGL(k_pf8_split, dim3((rows + 3) / 4), dim3(256), 0, s, src, rows, K, a.hi, a.lo, a.meta);
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
  P.hi = a.hi; P.lo = a.lo; P.meta = a.meta;
  P.out = out; P.segs = segs; P.offsets = offsets; P.sorted = down ? nullptr : sorted;
  P.T = T; P.k = L->k; P.E = L->E; P.M = M; P.K = K;
  return down ? launch8<1, 4>(P, nseg, s) : launch8<2, 1>(P, nseg, s);   // M % 256 == 0: whole tiles
}
