// MoE block, prefill path (T > 8 tokens): grouped dequant-GEMMs on MFMA.
//
//   1. k_pf_prep_router, two roles in one launch:
//      prep blocks:   xn = rmsnorm(x) (or x) -> an f16 copy (gate/up operand),
//                     and each token's RMSNorm factor
//      router blocks: partial router dot products of x w_norm over K ranges and
//                     the shared scalar gate's on v_mfma_f32_16x16x32_bf16, x w_norm
//                     split in registers into three bf16 planes whose sum is it
//                     to ~2^-27, one MFMA per plane: every product of a bf16
//                     weight and a bf16 plane is exact in fp32; the RMSNorm
//                     factor multiplies the summed partials in step 3
//   3. k_pf_topk sums the router partials (times the RMSNorm factor, + bias),
//      then dispatch (dispatch.hip):
//      histogram -> exclusive scan -> stable scatter of (token, slot) pairs by
//      expert, the inverse permutation, and every expert's token list (and the
//      shared expert's, which takes all T tokens) cut into segments of <= 32
//      or 64 (pf_seg)
//   4. k_pf_gateup:   per (segment, 64 weight rows): h = silu(G x) * (U x).  The raw
//                     superblocks come through LDS, one superblock ahead, and are
//                     decoded to f16 integers (kvalue or grid magnitude times
//                     the integer part of the sub-block scale) straight into
//                     v_mfma_f32_16x16x32_f16 operands; the superblock's fp16 d
//                     multiplies the fp32 partial sum of each superblock.  The
//                     segment's activation tile is double-buffered in LDS.  h is
//                     stored as bf16 in expert-sorted row order.
//   5. k_pf_h16:      every h row scaled by a power of two into f16's range and
//                     converted exactly (the scale is kept per row)
//   6. k_pf_down:     per (segment, 2 x 128 or 2 x 256 weight rows): y_pair = Down_e h on
//                     v_mfma_f32_16x16x32_f16 with f16 integer weight operands as in
//                     4, fp32 out times the row's h scale; the segment's h tile is
//                     staged in LDS once per block
//   7. k_pf_combine:  y[t] = sum over t's experts in ascending id of w * y_pair
//                     + sigmoid gate * y_shared (+ x); fixed order, no atomics
//
// Reference semantics: the CPU loop of qwen/forward.py:563-665 (prefill takes
// that path in the reference; its NPU kernels are T = 1 only).
#include <type_traits>

#include "moe_common.h"

using namespace gm_moe;

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gm_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 gm_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gm_f16x2 __attribute__((ext_vector_type(2)));
typedef float gm_f32x2 __attribute__((ext_vector_type(2)));
typedef float gm_f32x8 __attribute__((ext_vector_type(8)));

namespace {

constexpr int kChunk = 256;         // K elements of a superblock

// f(integral_constant<int, n>) for the segment's tile count n = ntiles in
// [1, NT], as a chain of uniform branches (one instantiation per count).
template <int NT, class F>
__device__ __forceinline__ void nt_dispatch(int ntiles, F&& f) {
  if constexpr (NT > 1) {
    if (ntiles < NT) { nt_dispatch<NT - 1>(ntiles, f); return; }
  }
  f(std::integral_constant<int, NT>{});
}

struct PfWs {
  int32_t* counts;    // [E]
  int32_t* offsets;   // [E + 1]
  int32_t* sorted;    // [P]
  int32_t* inv;       // [P]   position of pair p in sorted order
  int32_t* segs;      // [1 + 4 * max_seg]  n_seg, then (expert, start, n, unused)
  float* rmsv;        // [T]        RMSNorm factor per token (1 without a norm), for k_pf_topk
  uint16_t* xh;       // [T][D]     f16 xn 2^s (gate/up operand)
  float* xsc;         // [T]        2^-s per token
  float* part;        // [kRouterSplit][T][ldp]  partial router dot products
  uint16_t* hb;       // [P + T][FF]  bf16 SwiGLU rows (sorted pairs, then shared per token)
  uint16_t* hh;       // [P + T][FF]  the same rows as scaled f16
  float* hsc;         // [P + T]      their scales
  float* yp;          // [P + T][D]   fp32 per-pair / shared outputs
  float* xn;          // [T][D]  fp32 xn, for a shared expert in other formats than the routed ones
  float* hsh;         // [T][FF] its fp32 SwiGLU rows
};

// A shared expert stored in other formats than the routed experts (the real
// model's K-quant shared experts, held as I8 rows, beside IQ routed experts; or
// a dense bf16 one) does not run as the GEMMs' ninth unit.  In I8 rows it runs
// as two dense f16 MFMA GEMMs of its own (k_pfs_gateup_i8 into the shared
// SwiGLU rows hb[P + t], k_pf_h16, k_pfs_down_i8 into yp[P + t]); in bf16 its T
// tokens run as one fp32 pass of the multi-token gate/up and down matvec
// kernels over xn.  Either way it writes the rows yp[P + t] the combine reads,
// and the routed experts keep the grouped GEMMs.
inline bool pf_shared_apart(const gm_moe_layer* L) {
  return L->gate_sh && (L->q_gate_sh != L->q_gate || L->q_down_sh != L->q_down);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

constexpr int kRouterSplit = 16;  // most K ranges of the router GEMM (partials summed in k_pf_topk)

// K ranges actually used: 256 wide (2 k-steps per wave; twice the blocks of
// 512-wide ranges, measured 11.0 against 12.4 us at D = 2048) up to D = 2048,
// then 512 wide when D allows.  At most kRouterSplit ranges (checked at entry).
int router_krange(int D) { return D <= 2048 || D % 512 ? 256 : 512; }
int router_split(int D) { return D / router_krange(D); }

// Row stride of the router partials: E rows + the shared gate row, padded to 4.
int router_ld(const gm_moe_layer* L) { return (L->E + 1 + 3) & ~3; }

int max_segments(int T, int k, int E, int seg) { return (T * k) / seg + E + (T + seg - 1) / seg + 1; }

// Tokens per segment of the IQ GEMMs.  Their kernels are bound by the decoding of
// weights to f16, once per segment, so an expert's tokens should fit one; but a
// segment of 64 halves the waves that a CU holds.  Block times at D = 2048, FF =
// 512, E = 256, k = 8 (32 / 64): T = 512 192 / 213 us, 768 231 / 235, 1024 268 /
// 257, 2048 437 / 381, 3072 612 / 523; at D = 512, FF = 256, E = 16, k = 4, where
// 64 leaves CUs without a block: T = 768 45 / 50, 1280 56 / 55, 2048 72 / 67.
constexpr int kSegMin = 32;
int pf_seg(const gm_moe_layer* L, int T) {
  const int64_t pairs = (int64_t)T * L->k;
  return L->FF <= 2 * kChunk && pairs >= 28 * (int64_t)L->E && pairs / 64 * (L->FF / 64) >= 512 ? 64 : kSegMin;
}

PfWs pf_layout(const gm_moe_layer* L, int T, uint8_t* base, size_t* total) {
  const size_t P = (size_t)T * L->k, E = L->E;
  size_t o = 0;
  PfWs w{};
  auto take = [&](size_t bytes) { uint8_t* p = base ? base + o : nullptr; o = align256(o + bytes); return p; };
  w.counts = reinterpret_cast<int32_t*>(take(E * 4));
  w.offsets = reinterpret_cast<int32_t*>(take((E + 1) * 4));
  w.sorted = reinterpret_cast<int32_t*>(take(P * 4));
  w.inv = reinterpret_cast<int32_t*>(take(P * 4));
  w.segs = reinterpret_cast<int32_t*>(take((1 + 4 * (size_t)max_segments(T, L->k, L->E, kSegMin)) * 4));
  w.rmsv = reinterpret_cast<float*>(take((size_t)T * 4));
  w.xh = reinterpret_cast<uint16_t*>(take((size_t)T * L->D * 2));
  w.xsc = reinterpret_cast<float*>(take((size_t)T * 4));
  w.part = reinterpret_cast<float*>(take((size_t)kRouterSplit * T * router_ld(L) * 4));
  w.hb = reinterpret_cast<uint16_t*>(take((P + T) * (size_t)L->FF * 2));
  w.hh = reinterpret_cast<uint16_t*>(take((P + T) * (size_t)L->FF * 2));
  w.hsc = reinterpret_cast<float*>(take((P + T) * 4));
  w.yp = reinterpret_cast<float*>(take((P + T) * (size_t)L->D * 4));
  if (pf_shared_apart(L)) {
    w.xn = reinterpret_cast<float*>(take((size_t)T * L->D * 4));
    w.hsh = reinterpret_cast<float*>(take((size_t)T * L->FF * 4));
  }
  if (total) *total = o;
  return w;
}

// Blocks run on the 8 XCDs round-robin (block b on XCD b % 8).  Segment
// seg goes to XCD seg % 8 and its nrt row tiles to consecutive slots there,
// so they share the segment's activation tile in one L2, and the grid's
// unused tail (it is sized for the most segments the routing can produce)
// is spread over all XCDs.  Grid size: a multiple of 8 * nrt.
__device__ __forceinline__ void xcd_tile(int b, int nrt, int& seg, int& rt) {
  const int slot = b >> 3;
  seg = (slot / nrt) * 8 + (b & 7);
  rt = slot - (slot / nrt) * nrt;
}

// ---------------------------------------------------------------- prep x
// xn = (x * rms) * w (qwen/forward.py:58-61) or x; xh = f16(xn 2^s) with the
// per-token power of two that puts max |xn| in [2^14, 2^15) (no f16 overflow
// whatever the input scale, and f16's 11 bits for every value down to 2^-10 of
// the token's maximum; rows below 2^-100 are scaled as if their maximum were
// 2^-100), xsc[t] = 2^-s, which the gate/up kernel multiplies into its sums,
// and rmsv[t] = rms (1 without a norm).  One block per token.
__device__ __forceinline__ float pf_block_max(float m, float* red4) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = m;
  __syncthreads();
  return fmaxf(fmaxf(red4[0], red4[1]), fmaxf(red4[2], red4[3]));
}

// 2^s for a row whose largest magnitude is m (m >= 0): m 2^s in [2^14, 2^15).
__device__ __forceinline__ int pf_f16_shift(float m) {
  const int E = m > 0.f && m <= 3.4e38f ? max(__builtin_amdgcn_frexp_expf(m), -100) : 0;
  return 15 - E;
}

__device__ __forceinline__ uint32_t pf_f16x2(gm_f32x2 v, int sh) {
  const gm_f32x2 vs = {__builtin_ldexpf(v.x, sh), __builtin_ldexpf(v.y, sh)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(vs, gm_f16x2));
}

__device__ __forceinline__ void pf_prep_token(int t, const float* __restrict__ x, int D,
                                              const float* __restrict__ norm_w, float eps,
                                              uint16_t* __restrict__ xh, float* __restrict__ xsc,
                                              float* __restrict__ xn32, float* __restrict__ rmsv, float* red,
                                              float* redm) {
  const gm_f32x2* x2 = reinterpret_cast<const gm_f32x2*>(x + (int64_t)t * D);
  const int n2 = D >> 1;
  int sh;
  if (D <= 4096) {                                             // uniform: the row held in registers
    constexpr int NQ = 4;                                      // 16-byte granules per thread
    const int n4 = D >> 2;
    const gm_f32x4* x4 = reinterpret_cast<const gm_f32x4*>(x + (int64_t)t * D);
    gm_f32x4 v[NQ], wv[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {                             // every load before the first use
      const int c = min((int)threadIdx.x + 256 * i, n4 - 1);   // past the row: a duplicate, not used
      v[i] = x4[c];
      wv[i] = norm_w ? reinterpret_cast<const gm_f32x4*>(norm_w)[c] : gm_f32x4{1.f, 1.f, 1.f, 1.f};
    }
    float rms = 1.f;
    if (norm_w) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        if ((int)threadIdx.x + 256 * i < n4)
          ss = fmaf(v[i].x, v[i].x, fmaf(v[i].y, v[i].y, fmaf(v[i].z, v[i].z, fmaf(v[i].w, v[i].w, ss))));
      ss = gm_wave_sum64(ss);
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
      __syncthreads();
      rms = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)D + eps);
    }
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      if (norm_w) {
        v[i].x = (v[i].x * rms) * wv[i].x; v[i].y = (v[i].y * rms) * wv[i].y;
        v[i].z = (v[i].z * rms) * wv[i].z; v[i].w = (v[i].w * rms) * wv[i].w;
      }
      if ((int)threadIdx.x + 256 * i < n4)
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    }
    sh = pf_f16_shift(pf_block_max(m, redm));
    if (threadIdx.x == 0) rmsv[t] = rms;
    uint2* qh = reinterpret_cast<uint2*>(xh) + (int64_t)t * n4;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int c = (int)threadIdx.x + 256 * i;
      if (c >= n4) break;
      qh[c] = make_uint2(pf_f16x2(gm_f32x2{v[i].x, v[i].y}, sh), pf_f16x2(gm_f32x2{v[i].z, v[i].w}, sh));
      if (xn32) reinterpret_cast<gm_f32x4*>(xn32 + (int64_t)t * D)[c] = v[i];
    }
  } else {
    // two passes over the row: x^2 and max |x w| (rms > 0 scales the maximum
    // exactly up to rounding, and the target range leaves a factor 2 of f16 room)
    const gm_f32x2* w2 = reinterpret_cast<const gm_f32x2*>(norm_w);
    float ss = 0.f, m = 0.f;
    for (int i = threadIdx.x; i < n2; i += 256) {
      const gm_f32x2 v = x2[i];
      const gm_f32x2 w = norm_w ? w2[i] : gm_f32x2{1.f, 1.f};
      ss = fmaf(v.x, v.x, fmaf(v.y, v.y, ss));
      m = fmaxf(m, fmaxf(fabsf(v.x * w.x), fabsf(v.y * w.y)));
    }
    float rms = 1.f;
    if (norm_w) {
      ss = gm_wave_sum64(ss);
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
      __syncthreads();
      rms = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)D + eps);
    }
    sh = pf_f16_shift(pf_block_max(m, redm) * rms);
    if (threadIdx.x == 0) rmsv[t] = rms;
    uint32_t* ph = reinterpret_cast<uint32_t*>(xh) + (int64_t)t * n2;
    for (int i = threadIdx.x; i < n2; i += 256) {
      gm_f32x2 v = x2[i];
      if (norm_w) { const gm_f32x2 w = w2[i]; v.x = (v.x * rms) * w.x; v.y = (v.y * rms) * w.y; }
      ph[i] = pf_f16x2(v, sh);
      if (xn32) reinterpret_cast<gm_f32x2*>(xn32 + (int64_t)t * D)[i] = v;
    }
  }
  if (threadIdx.x == 0) xsc[t] = __builtin_ldexpf(1.0f, -sh);
}

// ---------------------------------------------------------------- router
// Partial router dot products part[z][t][r] = (x[t] w_norm) . W[r] over the z-th
// K range of kr = 128 NK values (rows r < E of W and row E = the shared gate
// vector, qwen/forward.py:599-600, 608; the token's RMSNorm factor is applied to
// the summed partials by k_pf_topk, so no block needs a whole row of x).  Block:
// 64 rows x 16 tokens x one K range; wave w takes the w-th quarter of the range
// for all four 16-row tiles, and issues every operand load of its NK k-steps (x,
// the norm weights and the router rows) before its first MFMA (one memory round
// trip); x w_norm is formed in fp32 and split into three bf16 planes in
// registers.  The four waves' tiles are added in LDS in wave order.
// MFMA operand layout (16x16x32): lane l holds row / column l % 16 at
// k = 8 (l / 16) .. +7.

// An fp32 router (RF32) is split in registers into three bf16 pieces,
// w = w0 + w1 + w2 exactly (each piece holds the next 8 significant bits of
// the 24; exact unless |w| < 2^-100, where bf16 subnormals cut the last
// piece), and all nine piece products are accumulated.
// FOLD (layers with I8 experts, whose logits came from the decode kernels' fp32 FMAs
// before they had these GEMMs): a k-step is summed by itself, the lower pieces
// first, every other one of -x (neg), which cancels the MFMA's rounding towards
// -infinity; error of the logits against 64 bits at D = 2048 1.7e-7 -> 1.0e-7 (one
// token at a time 1.1e-7).
__device__ __forceinline__ void split3_bf16(const gm_u32x4 (&r)[2], gm_bf16x8 (&o)[3]) {
  gm_f32x8 v;
  v[0] = __uint_as_float(r[0].x); v[1] = __uint_as_float(r[0].y);
  v[2] = __uint_as_float(r[0].z); v[3] = __uint_as_float(r[0].w);
  v[4] = __uint_as_float(r[1].x); v[5] = __uint_as_float(r[1].y);
  v[6] = __uint_as_float(r[1].z); v[7] = __uint_as_float(r[1].w);
  o[0] = __builtin_convertvector(v, gm_bf16x8);
  const gm_f32x8 r0 = v - __builtin_convertvector(o[0], gm_f32x8);
  o[1] = __builtin_convertvector(r0, gm_bf16x8);
  const gm_f32x8 r1 = r0 - __builtin_convertvector(o[1], gm_f32x8);
  o[2] = __builtin_convertvector(r1, gm_bf16x8);
}

template <bool RF32, bool FOLD>
__device__ __forceinline__ void router_step(const gm_u32x4 (&a)[4][RF32 ? 2 : 1], const gm_u32x4 (&b)[3], bool neg,
                                            gm_f32x4 (&acc)[4]) {
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    gm_f32x4 d = FOLD ? gm_f32x4{0.f, 0.f, 0.f, 0.f} : acc[rt];
    if constexpr (RF32) {
      gm_bf16x8 ap[3];
      split3_bf16(a[rt], ap);
#pragma unroll
      for (int pa = 0; pa < 3; ++pa)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ap[FOLD ? 2 - pa : pa],
                                                      __builtin_bit_cast(gm_bf16x8, b[FOLD ? 2 - p : p]), d, 0, 0, 0);
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p)
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gm_bf16x8, a[rt][0]),
                                                    __builtin_bit_cast(gm_bf16x8, b[FOLD ? 2 - p : p]), d, 0, 0, 0);
    }
    acc[rt] = !FOLD ? d : neg ? acc[rt] - d : acc[rt] + d;
  }
}

template <int NK, bool RF32, bool FOLD>
__device__ __forceinline__ void pf_router_block(int rb, int tb, int z, const void* __restrict__ w,
                                                const void* __restrict__ wsh, const float* __restrict__ x,
                                                const float* __restrict__ norm_w, int T, int D, int E, int ldp,
                                                float* __restrict__ part, gm_f32x4 (*red)[4][64]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int nrows = E + (wsh ? 1 : 0);
  const int r0 = rb * 64;
  const int tok = tb * 16 + l16;
  const int tokc = tok < T ? tok : T - 1;
  const int k0 = (z * 4 + wave) * (32 * NK);
  const gm_f32x4* xrow = reinterpret_cast<const gm_f32x4*>(x + (int64_t)tokc * D + k0 + 8 * q);
  const gm_f32x4* nrow = reinterpret_cast<const gm_f32x4*>((norm_w ? norm_w : x) + k0 + 8 * q);
  constexpr int RW = RF32 ? 2 : 1;                              // 16-byte loads per 8 weights
  gm_u32x4 a[NK][4][RW];
  gm_f32x4 xv[NK][2], nv[NK][2];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int row = r0 + rt * 16 + l16;
    const void* pr = row < E ? router_row<RF32>(w, row, D) : (row == E && wsh ? wsh : w);
    const gm_u32x4* ar = reinterpret_cast<const gm_u32x4*>(static_cast<const char*>(pr) + (k0 + 8 * q) * 2 * RW);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
#pragma unroll
      for (int h = 0; h < RW; ++h) a[ks][rt][h] = ar[4 * RW * ks + h];
  }
#pragma unroll
  for (int ks = 0; ks < NK; ++ks)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xv[ks][h] = xrow[8 * ks + h];
      nv[ks][h] = nrow[8 * ks + h];                             // x again without a norm: not used
    }
  gm_f32x4 acc[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) acc[rt] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < NK; ++ks) {
    gm_u32x4 xw[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      gm_f32x4 v = norm_w ? xv[ks][h] * nv[ks][h] : xv[ks][h];
      if (FOLD && (ks & 1)) v = -v;
      xw[h] = __builtin_bit_cast(gm_u32x4, v);
    }
    gm_bf16x8 pl[3];
    split3_bf16(xw, pl);
    const gm_u32x4 b[3] = {__builtin_bit_cast(gm_u32x4, pl[0]), __builtin_bit_cast(gm_u32x4, pl[1]),
                           __builtin_bit_cast(gm_u32x4, pl[2])};
    router_step<RF32, FOLD>(a[ks], b, ks & 1, acc);
  }
  if (wave > 0) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) red[wave - 1][rt][lane] = acc[rt];
  }
  __syncthreads();
  if (wave > 0 || tok >= T) return;
#pragma unroll
  for (int v = 0; v < 3; ++v)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) acc[rt] += red[v][rt][lane];
  float* out = part + ((int64_t)z * T + tok) * ldp;
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int row = r0 + rt * 16 + 4 * q;
    if (row + 3 < nrows) *reinterpret_cast<gm_f32x4*>(out + row) = acc[rt];
    else
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (row + i < nrows) out[row + i] = acc[rt][i];
  }
}

// Blocks [0, n_rt): the router blocks (row block, token tile, K range) = (b %
// nrb, b / nrb % ntb, b / (nrb ntb)); blocks [n_rt, n_rt + T): the prep of
// token b - n_rt.  The two roles share nothing: the launch replaces a prep
// launch followed by a router launch.
template <int NK, bool RF32, bool FOLD>
__global__ void __launch_bounds__(256) k_pf_prep_router(const void* __restrict__ w, const void* __restrict__ wsh,
                                                        const float* __restrict__ x, const float* __restrict__ norm_w,
                                                        float eps, int T, int D, int E, int ldp,
                                                        float* __restrict__ part, int nrb, int ntb, int n_rt,
                                                        uint16_t* __restrict__ xh, float* __restrict__ xsc,
                                                        float* __restrict__ xn32, float* __restrict__ rmsv) {
  __shared__ gm_f32x4 red[3][4][64];
  __shared__ float pred[4], predm[4];
  const int b = blockIdx.x;
  if (b >= n_rt) {                                              // uniform per block
    pf_prep_token(b - n_rt, x, D, norm_w, eps, xh, xsc, xn32, rmsv, pred, predm);
    return;
  }
  pf_router_block<NK, RF32, FOLD>(b % nrb, (b / nrb) % ntb, b / (nrb * ntb), w, wsh, x, norm_w, T, D, E, ldp, part, red);
}

// One wave per token: logits = the token's RMSNorm factor x the sum of the
// nsplit <= NZ partials (fixed order) + bias, the shared gate sigmoid, and the top-k (ties -> lower id) with
// renormalised softmax weights (qwen/forward.py:609-611).  Every partial is
// loaded (clamped index) before any is summed.
template <int MAXV, int NZ>
__global__ void __launch_bounds__(256) k_pf_topk(const float* __restrict__ part, int ldp, int nsplit, int T, int E, int k,
                                                 int has_gate, const float* __restrict__ bias,
                                                 const float* __restrict__ rmsv,
                                                 float* __restrict__ logits, float* __restrict__ shg,
                                                 int32_t* __restrict__ ids, float* __restrict__ wts) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  const int64_t zs = (int64_t)T * ldp;
  const float* pt = part + (int64_t)t * ldp;
  const float rms = rmsv[t];
  float v[MAXV], pv[MAXV][NZ], pg[NZ];
  int ix[MAXV];
#pragma unroll
  for (int z = 0; z < NZ; ++z) {
    const int64_t zo = (int64_t)(z < nsplit ? z : nsplit - 1) * zs;
#pragma unroll
    for (int i = 0; i < MAXV; ++i) {
      const int r = lane + 64 * i;
      pv[i][z] = pt[zo + (r < E ? r : E - 1)];
    }
    pg[z] = pt[zo + E];
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    ix[i] = lane + 64 * i;
    const int r = ix[i] < E ? ix[i] : E - 1;
    float acc = 0.f;
#pragma unroll
    for (int z = 0; z < NZ; ++z) acc += z < nsplit ? pv[i][z] : 0.f;
    v[i] = rms * acc + (bias ? bias[r] : 0.f);
    if (ix[i] < E) logits[(int64_t)t * E + ix[i]] = v[i];
  }
  if (lane == 0) {                                          // no gate row: the shared expert is ungated
    float g = 0.f;
#pragma unroll
    for (int z = 0; z < NZ; ++z) g += z < nsplit ? pg[z] : 0.f;
    shg[t] = has_gate ? gm_sigmoid(rms * g) : 1.f;
  }
  int id;
  float wt;
  topk_finish<MAXV>(v, ix, E, k, id, wt);
  if (lane < k) {
    ids[(int64_t)t * k + lane] = id;
    wts[(int64_t)t * k + lane] = wt;
  }
}

// ------------------------------------------------------- raw superblocks
// The bytes of one superblock of one weight row that lane quarter q needs.
// Lane quarter q covers sub-blocks 2q and 2q+1 of every superblock; k-step j
// (0..7) of the superblock uses sub-block 2q + (j >> 2).
template <int QT> struct PfRaw;
template <> struct PfRaw<GM_QTYPE_IQ4_XS> {
  uint32_t h0, h1;      // d | scales_h, scales_l[0..3]
  uint32_t q[8];        // qs bytes 32q .. 32q+31 (sub-blocks 2q, 2q+1)
};
template <> struct PfRaw<GM_QTYPE_IQ3_XXS> {
  uint32_t d;           // fp16 bits
  uint32_t q[4];        // qs bytes 16q .. 16q+15 (sub-blocks 2q, 2q+1)
  uint32_t w0, w1;      // scale/sign words 2q, 2q+1
};

// IQ4_XS superblocks are 8-byte aligned (136 = 8 * 17, rows of whole superblocks).
__device__ __forceinline__ PfRaw<GM_QTYPE_IQ4_XS> pf_load_iq4(const uint8_t* __restrict__ sb, int q) {
  PfRaw<GM_QTYPE_IQ4_XS> r;
  const uint2 h = *reinterpret_cast<const uint2*>(sb);
  const uint2* p = reinterpret_cast<const uint2*>(sb + 8 + 32 * q);
  r.h0 = h.x; r.h1 = h.y;
#pragma unroll
  for (int i = 0; i < 4; ++i) { const uint2 v = p[i]; r.q[2 * i] = v.x; r.q[2 * i + 1] = v.y; }
  return r;
}

// IQ3_XXS superblocks are 2-byte aligned (98 B): dword loads re-aligned with
// v_alignbyte_b32.  Every dword read holds at least one byte of this
// superblock, so no read leaves the superblock's 4 KB page.
__device__ __forceinline__ PfRaw<GM_QTYPE_IQ3_XXS> pf_load_iq3(const uint8_t* __restrict__ sb, int q) {
  PfRaw<GM_QTYPE_IQ3_XXS> r;
  const int odd = (int)((reinterpret_cast<uintptr_t>(sb) >> 1) & 1);     // sb % 4 == 2 * odd
  const int rq = odd ? 0 : 2;                                           // (sb + 2) % 4
  const uint32_t* dp = reinterpret_cast<const uint32_t*>(sb - 2 * odd);
  const uint32_t dw = dp[0];
  r.d = odd ? (dw >> 16) : (dw & 0xffffu);
  const uint32_t* qp = reinterpret_cast<const uint32_t*>(sb + 2 + 16 * q - rq);
  uint32_t v[5];
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = qp[i];
  v[4] = qp[rq ? 4 : 3];
#pragma unroll
  for (int i = 0; i < 4; ++i) r.q[i] = __builtin_amdgcn_alignbyte(v[i + 1], v[i], rq);
  const uint32_t* wp = reinterpret_cast<const uint32_t*>(sb + 66 + 8 * q - rq);
  const uint32_t w0 = wp[0], w1 = wp[1], w2 = wp[rq ? 2 : 1];
  r.w0 = __builtin_amdgcn_alignbyte(w1, w0, rq);
  r.w1 = __builtin_amdgcn_alignbyte(w2, w1, rq);
  return r;
}

template <int QT>
__device__ __forceinline__ PfRaw<QT> pf_load(const uint8_t* __restrict__ sb, int q) {
  if constexpr (QT == GM_QTYPE_IQ4_XS) return pf_load_iq4(sb, q);
  else return pf_load_iq3(sb, q);
}

// Sub-block scales of the lane's two sub-blocks (2q, 2q+1): f16 weights hold only
// the integer factor, and the superblock factor pf_dscale is applied to the fp32
// partial sums:
//   IQ4_XS: d * (ls - 32)            -> integer ls - 32 in [-32, 31], factor d
//   IQ3_XXS: d * (0.5 + s4) * 0.5    -> integer 2 s4 + 1 in [1, 31], factor d / 4
// so every f16 weight is an integer product, exact up to 2048 in magnitude:
// |(2 s4 + 1) g| <= 1922 is always exact, |kv (ls - 32)| <= 4064 is rounded
// once to f16's 11 significant bits when odd and above 2048; f16's small
// exponent range never meets a tiny d.
// The lane's integer scales as an f16 pair {sub-block 2q, 2q + 1} (exact: 0x6400 |
// n is the f16 1024 + n) and the addends that go with them (u8x4_to_f16).
template <int QT>
struct PfF16Scale {
  gm_f16x2 s, c;
  __device__ __forceinline__ gm_f16x2 sh(int h) const { return gm_f16x2{s[h], s[h]}; }
  __device__ __forceinline__ gm_f16x2 ch(int h) const { return gm_f16x2{c[h], c[h]}; }
};

template <int QT>
__device__ __forceinline__ PfF16Scale<QT> pf_f16_scales(const PfRaw<QT>& r, int q) {
  PfF16Scale<QT> o;
  if constexpr (QT == GM_QTYPE_IQ4_XS) {
    const uint32_t sl = (r.h1 >> (8 * q)) & 0xffu, hi = r.h0 >> (16 + 4 * q);
    const uint32_t n = (sl & 0x0fu) | (sl & 0xf0u) << 12 | (hi & 3u) << 4 | (hi & 12u) << 18;
    o.s = __builtin_bit_cast(gm_f16x2, n | 0x64006400u) - gm_f16x2{(_Float16)1056.f, (_Float16)1056.f};
    o.c = o.s * gm_f16x2{(_Float16)-1152.f, (_Float16)-1152.f};
  } else {
    const uint32_t n = (r.w0 >> 28) << 1 | (r.w1 >> 28) << 17 | 0x00010001u;
    o.s = __builtin_bit_cast(gm_f16x2, n | 0x64006400u) - gm_f16x2{(_Float16)1024.f, (_Float16)1024.f};
    o.c = o.s * gm_f16x2{(_Float16)-1024.f, (_Float16)-1024.f};
  }
  return o;
}

template <int QT>
__device__ __forceinline__ float pf_dscale(const PfRaw<QT>& r) {
  if constexpr (QT == GM_QTYPE_IQ4_XS) return gm_h2f(r.h0 & 0xffffu);
  else return gm_h2f(r.d) * 0.25f;
}

// kvalues_iq4nl + 128 as unsigned bytes (entry n in byte n % 4 of word n / 4).
constexpr uint32_t kKvU[4] = {kGmKv[0] ^ 0x80808080u, kGmKv[1] ^ 0x80808080u, kGmKv[2] ^ 0x80808080u,
                              kGmKv[3] ^ 0x80808080u};

// Two-lookup XOR form of the table (see gm_lut16_xor), checked at compile time.
constexpr gm_iq4_xor::Tabs kKvUx = gm_iq4_xor::solve(kKvU);
static_assert(gm_iq4_xor::check(kKvU, kKvUx), "XOR lookup of kvalues + 128");

__device__ __forceinline__ uint32_t lut_kvu(uint32_t nib) { return gm_lut16_xor(kKvUx, nib); }

// Four unsigned bytes u -> two f16x2 holding (u - b) * s, rounded once (b = 128
// for IQ4_XS, 0 for IQ3_XXS's magnitudes): 0x6400 | u is the f16 1024 + u, and
// fma(1024 + u, s, c) with c = -(1024 + b) s (exact in f16 for |s| <= 32) is
// (u - b) s in one rounding.
__device__ __forceinline__ void u8x4_to_f16(uint32_t u, gm_f16x2 s, gm_f16x2 c, uint32_t& o0, uint32_t& o1) {
  const gm_f16x2 a = __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u));
  const gm_f16x2 b = __builtin_bit_cast(gm_f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u));
  o0 = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(a, s, c));
  o1 = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(b, s, c));
}

// IQ3_XXS sign table for k-step decode: entry i (7-bit ksigns index) holds the
// signs of ksigns(i) such that entry << p has those of weights 2p and 2p + 1 at
// bits 15 and 31, where the f16 pair p has its own (one dword: a fourth of the
// LDS traffic of byte masks for both halves).
__device__ __forceinline__ void pf_stage_signs(uint32_t* tab) {
  for (int i = threadIdx.x; i < 128; i += blockDim.x) {
    const uint32_t s = gm_ksigns((uint32_t)i);
    uint32_t m = 0;
#pragma unroll
    for (int p = 0; p < 4; ++p) m |= ((s >> (2 * p)) & 1u) << (15 - p) | ((s >> (2 * p + 1)) & 1u) << (31 - p);
    tab[i] = m;
  }
}

// f16 A operand of k-step j: 8 weights (scale folded in) at the lane's k-slots
// k = 32s + 8c + i (i < 8), s = 2q + (j >> 2), c = j & 3, so that the matching
// activations are 8 consecutive values:
//   IQ4_XS: the low (c < 2) or high (c >= 2) nibbles of qs bytes 8 (c & 1) .. + 7
//   IQ3_XXS: grid points 2c, 2c + 1 of the sub-block
template <int QT>
__device__ __forceinline__ gm_f16x8 a_f16(const PfRaw<QT>& r, int j, gm_f16x2 sc, gm_f16x2 cc,
                                          const uint32_t* __restrict__ grid,
                                          const uint32_t* __restrict__ sgn) {
  uint32_t o[4];
  if constexpr (QT == GM_QTYPE_IQ4_XS) {
    const int sl = j >> 2, c = j & 3, sh = 4 * (c >> 1);
    const uint32_t w0 = r.q[4 * sl + 2 * (c & 1)], w1 = r.q[4 * sl + 2 * (c & 1) + 1];
    u8x4_to_f16(lut_kvu((w0 >> sh) & 0x0f0f0f0fu), sc, cc, o[0], o[1]);
    u8x4_to_f16(lut_kvu((w1 >> sh) & 0x0f0f0f0fu), sc, cc, o[2], o[3]);
  } else {
    const int sl = j >> 2, g = j & 3;
    const uint32_t qw = r.q[2 * sl + (g >> 1)] >> (16 * (g & 1));
    const uint32_t ga = grid[qw & 0xffu], gb = grid[(qw >> 8) & 0xffu];
    const uint32_t w = sl ? r.w1 : r.w0;
    const uint32_t m = sgn[(w >> (7 * g)) & 127u];
    u8x4_to_f16(ga, sc, cc, o[0], o[1]);               // the magnitudes times the scale, then their signs
    u8x4_to_f16(gb, sc, cc, o[2], o[3]);
#pragma unroll
    for (int p = 0; p < 4; ++p) o[p] ^= (m << p) & 0x80008000u;
  }
  return __builtin_bit_cast(gm_f16x8, gm_u32x4{o[0], o[1], o[2], o[3]});
}

// Activation rows in LDS: every 16-byte granule (8 values) g of row r at slot
// g ^ (r & 15) of its row, so that the 16 rows a wave reads at once hit 16
// different bank groups without padding.  The B operand of k-step j, the 8
// activations of the lane's k-slots, is granule 4 (2q + (j >> 2)) + (j & 3) of a
// superblock; a gate/up row holds halves of superblocks (the k-steps of one
// half, granules 4q + (j & 3)).
template <int ROWB>
__device__ __forceinline__ gm_f16x8 b_lds(const uint8_t* tile, int r, int g) {
  return __builtin_bit_cast(gm_f16x8, *reinterpret_cast<const gm_u32x4*>(tile + r * ROWB + 16 * (g ^ (r & 15))));
}

// Half H (k-steps 4H .. 4H+3) of one superblock column of the gate and up
// rows against NT token tiles: f16 integer operands into the superblock's
// partial sums pg / pu.
template <int QT, int NT, int H>
__device__ __forceinline__ void gu_half(const PfRaw<QT>& wg, const PfRaw<QT>& wu, const PfF16Scale<QT>& sg,
                                        const PfF16Scale<QT>& su, int q, int l16, const uint8_t* __restrict__ xb,
                                        const uint32_t* __restrict__ grid, const uint32_t* __restrict__ sgn,
                                        gm_f32x4 (&pg)[NT], gm_f32x4 (&pu)[NT]) {
#pragma unroll
  for (int j = 4 * H; j < 4 * H + 4; ++j) {
    const gm_f16x8 A = a_f16<QT>(wg, j, sg.sh(H), sg.ch(H), grid, sgn);
    const gm_f16x8 U = a_f16<QT>(wu, j, su.sh(H), su.ch(H), grid, sgn);
    const int g = 4 * q + (j & 3);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const gm_f16x8 B = b_lds<256>(xb, t * 16 + l16, g);
      pg[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, B, pg[t], 0, 0, 0);
      pu[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(U, B, pu[t], 0, 0, 0);
    }
    if (j & 1) issue_fence();                          // two k-steps' operands live at a time
  }
}

// A superblock's partial sums times the superblock factor of each accumulator
// row (rows 4q + i, whose factors lanes 4q + i hold) into acc.
template <int NT>
__device__ __forceinline__ void pf_fold(float d, int q, const gm_f32x4 (&p)[NT], gm_f32x4 (&acc)[NT]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float di = __shfl(d, 4 * q + i, 64);
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t][i] = fmaf(di, p[t][i], acc[t][i]);
  }
}

// One superblock column of two down row tiles against NT token tiles: f16
// integer operands into the superblock's partial sums, then the partial sums
// times the superblock factor of each accumulator row into acc.
template <int QT, int NT, int ROWB>
__device__ __forceinline__ void dn_superblock(const PfRaw<QT>& w0, const PfRaw<QT>& w1, int q, int l16,
                                              const uint8_t* hbuf, const uint32_t* __restrict__ grid,
                                              const uint32_t* __restrict__ sgn, gm_f32x4 (&a0)[NT],
                                              gm_f32x4 (&a1)[NT]) {
  const PfF16Scale<QT> s0 = pf_f16_scales<QT>(w0, q), s1 = pf_f16_scales<QT>(w1, q);
  gm_f32x4 p0[NT], p1[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) { p0[t] = gm_f32x4{0.f, 0.f, 0.f, 0.f}; p1[t] = p0[t]; }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const gm_f16x8 A0 = a_f16<QT>(w0, j, s0.sh(j >> 2), s0.ch(j >> 2), grid, sgn);
    const gm_f16x8 A1 = a_f16<QT>(w1, j, s1.sh(j >> 2), s1.ch(j >> 2), grid, sgn);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const gm_f16x8 B = b_lds<ROWB>(hbuf, t * 16 + l16, 4 * (2 * q + (j >> 2)) + (j & 3));
      p0[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0, B, p0[t], 0, 0, 0);
      p1[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1, B, p1[t], 0, 0, 0);
    }
    if (j & 1) issue_fence();
  }
  pf_fold<NT>(pf_dscale<QT>(w0), q, p0, a0);
  pf_fold<NT>(pf_dscale<QT>(w1), q, p1, a1);
}

// ------------------------------------------------------------- h to f16
// One wave per SwiGLU row (FF <= 2048: 4 granules of 8 values per lane): the
// bf16 row scaled by 2^-e, e chosen so that its largest |value| lands in
// [2^14, 2^15), is exact in f16 (11 significand bits >= bf16's 8) for every
// value above 2^-29 of the largest; hsc[row] = 2^e, which the down kernel
// multiplies into its outputs.
__global__ void __launch_bounds__(256) k_pf_h16(const uint16_t* __restrict__ hb, int rows, int FF,
                                                uint16_t* __restrict__ hh, float* __restrict__ hsc) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const gm_u32x4* src = reinterpret_cast<const gm_u32x4*>(hb + (int64_t)r * FF);
  gm_u32x4* dst = reinterpret_cast<gm_u32x4*>(hh + (int64_t)r * FF);
  const int ng = FF >> 3;                                      // 16-byte granules per row
  constexpr int G = 4;                                         // FF <= 2048
  gm_u32x4 v[G];
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int g = lane + 64 * i;
    v[i] = src[g < ng ? g : ng - 1];
  }
  float m = 0.f;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
    for (int c = 0; c < 4; ++c)
      m = fmaxf(m, fmaxf(fabsf(gm_bf2f(w[c] & 0xffffu)), fabsf(gm_bf2f(w[c] >> 16))));
  }
  m = fmaxf(m, GM_DPP_F(m, GM_ROW_ROR8));
  m = fmaxf(m, GM_DPP_F(m, GM_ROW_ROR4));
  m = fmaxf(m, GM_DPP_F(m, GM_QPERM_2301));
  m = fmaxf(m, GM_DPP_F(m, GM_QPERM_1032));
  m = fmaxf(fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 0)),
                  __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 16))),
            fmaxf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 32)),
                  __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), 48))));
  // m in [2^(E-1), 2^E): scale so that the largest value lands in [2^14, 2^15)
  const int e = m > 0.f && m <= 3.4e38f ? __builtin_amdgcn_frexp_expf(m) - 15 : 0;
  const float down = __builtin_ldexpf(1.0f, -e);
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int g = lane + 64 * i;
    const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    uint32_t o[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const gm_f32x2 f = {gm_bf2f(w[c] & 0xffffu) * down, gm_bf2f(w[c] >> 16) * down};
      o[c] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, gm_f16x2));
    }
    if (g < ng) dst[g] = gm_u32x4{o[0], o[1], o[2], o[3]};
  }
  if (lane == 0) hsc[r] = m <= 3.4e38f ? __builtin_ldexpf(1.0f, e) : __builtin_nanf("");
}

// ------------------------------------------------ weight rows through LDS
// A wave load that takes 16 weight rows, as the A operands want them, asks for
// about five times the cache lines whose bytes it uses (a probe of the pattern:
// 3.1 TB/s, of contiguous runs 6.9).  So the lanes of a wave take consecutive
// 16-byte granules of its rows straight into LDS of its own, one step ahead, and
// read the operands from there.

// 16 bytes per lane into LDS at dst (the wave's, uniform) + 16 lane.
__device__ __forceinline__ void lds_load16(const void* src, uint8_t* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// Every lane takes part in every load: under a lane condition the compiler may
// merge two loads whose LDS destinations then differ between lanes.  Buffers are
// of whole loads, and lanes past the data read its last granule again.

// N consecutive granules (lane l of load j: granule 64 j + l) into LDS.
template <int N>
__device__ __forceinline__ void run_lds_load(const uint8_t* __restrict__ src, uint8_t* __restrict__ buf) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < (N + 63) / 64; ++j) {
    const int g = 64 * j + lane;
    lds_load16(src + 16 * (64 * j + 64 <= N ? g : min(g, N - 1)), buf + 1024 * j);
  }
}

// One superblock of 16 gate and 16 up IQ4_XS rows: 9 granules per row of 136
// bytes, the last one 8 bytes early so that it ends with the superblock.
constexpr int kIq4G = 9, kIq4Pitch = 16 * kIq4G, kIq4Tile = 16 * kIq4Pitch;
constexpr int kIq4Loads = (2 * 16 * kIq4G + 63) / 64;

// The lane's byte offsets of those granules from the gate tile (up = the up
// tile's distance from it).
__device__ __forceinline__ void iq4_offsets(int64_t up, int rb, int64_t (&off)[kIq4Loads]) {
#pragma unroll
  for (int j = 0; j < kIq4Loads; ++j) {
    const int id = min(64 * j + (int)(threadIdx.x & 63), 2 * 16 * kIq4G - 1), r = id / kIq4G, g = id - r * kIq4G;
    off[j] = (r < 16 ? 0 : up) + (r & 15) * rb + 16 * g - (g == 8 ? 8 : 0);
  }
}

__device__ __forceinline__ void iq4_lds_load(const uint8_t* __restrict__ gate, const int64_t (&off)[kIq4Loads],
                                             uint8_t* __restrict__ buf) {
#pragma unroll
  for (int j = 0; j < kIq4Loads; ++j) lds_load16(gate + off[j], buf + 1024 * j);
}

__device__ __forceinline__ PfRaw<GM_QTYPE_IQ4_XS> iq4_lds_read(const uint8_t* __restrict__ buf, int l16, int q) {
  PfRaw<GM_QTYPE_IQ4_XS> r;
  const uint8_t* p = buf + l16 * kIq4Pitch;
  const gm_u32x2 h = *reinterpret_cast<const gm_u32x2*>(p);
  r.h0 = h.x; r.h1 = h.y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const gm_u32x2 v = *reinterpret_cast<const gm_u32x2*>(p + 8 + 32 * q + 8 * i + (i == 3 && q == 3 ? 8 : 0));
    r.q[2 * i] = v.x; r.q[2 * i + 1] = v.y;
  }
  return r;
}

// Every LDS read issued so far has its data: what the reads took may be overwritten.
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// -------------------------------------------------------------- gate/up
// Block = (segment of at most ST tokens, 64 rows of FF); wave w -> rows 16w ..
// 16w+15 of both the gate and the up matrix, all of the segment's token tiles.
// A step is half a superblock: its activations are in one of two LDS buffers, the
// next step's on their way to the other (four blocks of 32 tokens to a CU, or three
// of 64).  IQ3_XXS rows come to registers, 16 rows a load: as decoded there they
// have not been tried through LDS.  At D = 2048, FF = 512, E = 256, k = 8 what bounds
// it is near even at T = 512: loads and barriers alone take 87 us (the rows' 285 MB
// at 3.3 TB/s and as many activation bytes from L2), decoding and MFMA alone 76,
// together 97 (113 with 16 rows to a load and the rows held in registers); at
// T = 4096, in segments of 64, 315 (416 in segments of 32, decoded twice as often).
template <int QT, int ST>
struct GuShape {
  static constexpr int ROWB = 256, TILE = ST * ROWB;              // bytes of an activation row and buffer
  static constexpr int G = ROWB / 16, NI = 16 * ROWB / 4096;           // granules per row, DMAs per wave and token tile
  static constexpr int WBYTES = QT == GM_QTYPE_IQ4_XS ? 4 * kIq4Loads * 1024 : 256 * 4 + 128 * 4;   // rows' way / tables
  static constexpr size_t SMEM = 2 * TILE + WBYTES + 2 * ST * 4;
};

// The next step's activations into the tile (no registers, no wait here): DMA
// instruction m of wave w writes 1 KB, granules 64 (NI w + m) .. + 63 of it.
template <int NI>
__device__ __forceinline__ void act_lds_load(const uint16_t* const (&ptr)[NI], int off, uint8_t* __restrict__ tile) {
#pragma unroll
  for (int m = 0; m < NI; ++m)
    lds_load16(ptr[m] + off, tile + ((threadIdx.x >> 6) * NI + m) * 1024);
}

// The K loop over NT token tiles.
template <int QT, int ST, int NT>
__device__ __forceinline__ void gu_loop(const uint8_t* __restrict__ gt, const uint8_t* __restrict__ ut, int64_t rb,
                                        int nsb, const uint16_t* const (&xp)[NT * GuShape<QT, ST>::NI],
                                        uint8_t* __restrict__ xl, uint8_t* __restrict__ wbuf,
                                        const uint32_t* __restrict__ grid, const uint32_t* __restrict__ sgn,
                                        gm_f32x4 (&ag)[NT], gm_f32x4 (&au)[NT]) {
  using S = GuShape<QT, ST>;
  constexpr bool IQ4 = QT == GM_QTYPE_IQ4_XS;
  constexpr int SBB = IQ4 ? GM_IQ4XS_BYTES : GM_IQ3XXS_BYTES;
  const int lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
#pragma unroll
  for (int t = 0; t < NT; ++t) { ag[t] = gm_f32x4{0.f, 0.f, 0.f, 0.f}; au[t] = ag[t]; }
  act_lds_load<NT * S::NI>(xp, 0, xl);
  int64_t woff[kIq4Loads];
  PfRaw<QT> wg, wu;
  if constexpr (IQ4) {
    iq4_offsets(ut - gt, (int)rb, woff);
    iq4_lds_load(gt, woff, wbuf);
  } else {
    wg = pf_load<QT>(gt + l16 * rb, q);
    wu = pf_load<QT>(ut + l16 * rb, q);
  }
  __builtin_amdgcn_s_waitcnt(0);                                        // the first step is in LDS
  __syncthreads();
  for (int sb = 0; sb < nsb; ++sb) {
    // next superblock's rows and, straight into the other LDS buffer, the next
    // activations (that buffer's last reader finished before the barrier)
    const bool more = sb + 1 < nsb;
    PfRaw<QT> wgn, wun;
    if constexpr (IQ4) {
      wg = iq4_lds_read(wbuf, l16, q);
      wu = iq4_lds_read(wbuf + kIq4Tile, l16, q);
      lds_reads_done();
    }
    act_lds_load<NT * S::NI>(xp, sb * kChunk + 32, xl + S::TILE);
    if constexpr (IQ4) {
      if (more) iq4_lds_load(gt + (sb + 1) * SBB, woff, wbuf);
    } else {
      const int sn = more ? sb + 1 : sb;                         // the last step re-reads itself
      wgn = pf_load<QT>(gt + l16 * rb + sn * SBB, q);
      wun = pf_load<QT>(ut + l16 * rb + sn * SBB, q);
    }
    const PfF16Scale<QT> sg = pf_f16_scales<QT>(wg, q), su = pf_f16_scales<QT>(wu, q);
    gm_f32x4 pg[NT], pu[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) { pg[t] = gm_f32x4{0.f, 0.f, 0.f, 0.f}; pu[t] = pg[t]; }
    gu_half<QT, NT, 0>(wg, wu, sg, su, q, l16, xl, grid, sgn, pg, pu);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (more) act_lds_load<NT * S::NI>(xp, (sb + 1) * kChunk, xl);
    gu_half<QT, NT, 1>(wg, wu, sg, su, q, l16, xl + S::TILE, grid, sgn, pg, pu);
    pf_fold<NT>(pf_dscale<QT>(wg), q, pg, ag);
    pf_fold<NT>(pf_dscale<QT>(wu), q, pu, au);
    if constexpr (!IQ4) {
      wg = wgn;
      wu = wun;
    }
    __builtin_amdgcn_s_waitcnt(0);                                      // the next step is in LDS
    __syncthreads();
  }
}

template <int QT, int ST>
__global__ void __launch_bounds__(256, ST == 32 ? 4 : 3) k_pf_gateup(
    gm_moe_layer P, const int32_t* __restrict__ segs, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ sorted, const uint16_t* __restrict__ xh, const float* __restrict__ xsc,
    uint16_t* __restrict__ hb, int T, int n_row_tiles) {
  using S = GuShape<QT, ST>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* xl = smem;                                                   // [2][ST][ROWB]
  uint8_t* wl = smem + 2 * S::TILE;                                     // [4 waves][gate, up tile, padding] (IQ4)
  uint32_t* grid = reinterpret_cast<uint32_t*>(wl);                     // [256] (IQ3)
  uint32_t* sgn = grid + 256;                                           // [128] (IQ3)
  int32_t* tok_row = reinterpret_cast<int32_t*>(wl + S::WBYTES);        // [ST]
  int32_t* out_row = tok_row + ST;                                      // [ST]
  int seg, rt;
  xcd_tile(blockIdx.x, n_row_tiles, seg, rt);
  if (seg >= segs[0]) return;
  const int e = segs[1 + 4 * seg], start = segs[2 + 4 * seg], n = segs[3 + 4 * seg];
  const int D = P.D, FF = P.FF, k = P.k, E = P.E;
  const bool shared = e == E;
  if constexpr (QT == GM_QTYPE_IQ3_XXS) {
    gm_stage_grid(grid);
    pf_stage_signs(sgn);
  }
  if (threadIdx.x < ST) {
    const int c = threadIdx.x;
    int tr = 0, orow = 0;
    if (c < n) {
      if (shared) { tr = start + c; orow = T * k + start + c; }
      else { const int pos = offsets[e] + start + c; tr = sorted[pos] / k; orow = pos; }
    } else {
      tr = shared ? start : sorted[offsets[e] + start] / k;     // a valid row of the segment
    }
    tok_row[c] = tr;
    out_row[c] = orow;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  const int64_t rb = gm_row_bytes(QT, D), tile = (int64_t)(rt * 64 + wave * 16) * rb;   // FF % 64 == 0: whole tiles
  const uint8_t* gbase = shared ? static_cast<const uint8_t*>(P.gate_sh)
                                : static_cast<const uint8_t*>(P.gate_exps) + (int64_t)e * FF * rb;
  const uint8_t* ubase = shared ? static_cast<const uint8_t*>(P.up_sh)
                                : static_cast<const uint8_t*>(P.up_exps) + (int64_t)e * FF * rb;
  const int ntiles = (n + 15) >> 4, r0 = rt * 64 + wave * 16 + 4 * q;
  nt_dispatch<ST / 16>(ntiles, [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    // lane i of DMA instruction m: slot s of row r, which holds granule s ^ (r & 15)
    const uint16_t* xp[NT * S::NI];
#pragma unroll
    for (int m = 0; m < NT * S::NI; ++m) {
      const int id = 64 * (wave * (NT * S::NI) + m) + lane, r = id / S::G, g = (id % S::G) ^ (r & 15);
      xp[m] = xh + (int64_t)tok_row[r] * D + 8 * (8 * (g >> 2) + (g & 3));
    }
    gm_f32x4 ag[NT], au[NT];
    gu_loop<QT, ST, NT>(gbase + tile, ubase + tile, rb, D / kChunk, xp, xl, wl + wave * kIq4Loads * 1024, grid, sgn, ag,
                            au);
    // C layout: lane l holds rows 4 (l / 16) + i of the 16-row tile, column l % 16
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int col = t * 16 + l16;
      if (col < n) {
        const float ds = xsc[tok_row[col]];                      // the token's f16 scale, undone exactly
        const gm_f32x4 g = ag[t] * ds, u = au[t] * ds;
        gm_f32x2 h01 = {gm_silu(g[0]) * u[0], gm_silu(g[1]) * u[1]};
        gm_f32x2 h23 = {gm_silu(g[2]) * u[2], gm_silu(g[3]) * u[3]};
        *reinterpret_cast<uint2*>(hb + (int64_t)out_row[col] * FF + r0) =
            make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(h01, gm_bf16x2)),
                       __builtin_bit_cast(uint32_t, __builtin_convertvector(h23, gm_bf16x2)));
      }
    }
  });
}

// ------------------------------------------------------------------ down
// Block of NW waves = (segment of at most ST tokens, rg_per_blk groups of 32 NW
// rows of D).  The segment's whole h tile (ST rows x FF, FF = 256 NSB) is staged
// in LDS once; the block then walks its row groups with the next group's rows on
// their way into LDS.  Wave w -> row tiles 2w, 2w+1 (16 rows each) of a group.
// Bound by the LDS gathers of the decode tables and VALU work about evenly (54% and
// 50% busy): 64 us at the sizes above and T = 512 (72 before), 230 at T = 4096 (295).
// Segments of 64: eight waves, one block to a CU (its LDS holds no second one).
// NSB is exact, three superblocks too (FF = 768 would else read past its rows).
template <int QT, int NSB, int ST, int NW>
struct DnShape {
  static constexpr int SBB = QT == GM_QTYPE_IQ4_XS ? GM_IQ4XS_BYTES : GM_IQ3XXS_BYTES;
  static constexpr int ROWB = NSB * 512, RUN = 2 * NSB * SBB;           // bytes of an h row, granules of a wave's rows
  static constexpr int WBUF = (RUN + 63) / 64 * 1024;                   // their LDS buffer
  static constexpr size_t SMEM = ST * (size_t)ROWB + 256 * 4 + 128 * 4 + ST * 4 + NW * WBUF;
};

template <int QT, int NSB, int ST, int NW, int NT>
__device__ __forceinline__ void dn_loop(const uint8_t* __restrict__ wrows, int64_t rb, uint8_t* __restrict__ wbuf,
                                        const uint8_t* hl, const uint32_t* __restrict__ grid,
                                        const uint32_t* __restrict__ sgn, int g0, int g1, int n,
                                        const float (&cs)[NT], float* __restrict__ yrow, int D) {
  using S = DnShape<QT, NSB, ST, NW>;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, l16 = lane & 15;
  PfRaw<QT> wc[2][NSB];
  auto take = [&]() {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) wc[m][sb] = pf_load<QT>(wbuf + ((m * 16 + l16) * NSB + sb) * S::SBB, q);
    lds_reads_done();
  };
  take();
  for (int g = g0; g < g1; ++g) {
    if (g + 1 < g1) run_lds_load<S::RUN>(wrows + (int64_t)(g + 1) * (32 * NW) * rb, wbuf);
    gm_f32x4 acc[2][NT];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[m][t] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
      dn_superblock<QT, NT, S::ROWB>(wc[0][sb], wc[1][sb], q, l16, hl + sb * 512, grid, sgn, acc[0], acc[1]);
    if (g + 1 < g1) {                                  // before this group's stores, which need not be waited for
      __builtin_amdgcn_s_waitcnt(0);
      take();
    }
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int r0 = g * (32 * NW) + wave * 32 + m * 16 + 4 * q;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int col = t * 16 + l16;
        if (col < n) *reinterpret_cast<gm_f32x4*>(yrow + (int64_t)col * D + r0) = acc[m][t] * cs[t];
      }
    }
  }
}

template <int QT, int NSB, int ST, int NW>
__global__ void __launch_bounds__(64 * NW, NSB > 2 ? 1 : 2) k_pf_down(gm_moe_layer P, const int32_t* __restrict__ segs,
                                                     const int32_t* __restrict__ offsets,
                                                     const uint16_t* __restrict__ hh, const float* __restrict__ hsc,
                                                     float* __restrict__ yp, int T, int n_blk, int rg_per_blk) {
  using S = DnShape<QT, NSB, ST, NW>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  uint8_t* hl = smem;                                                   // [ST][ROWB]
  uint32_t* grid = reinterpret_cast<uint32_t*>(smem + ST * S::ROWB);    // [256]
  uint32_t* sgn = grid + 256;                                           // [128]
  int32_t* in_row = reinterpret_cast<int32_t*>(sgn + 128);              // [ST]
  uint8_t* wl = reinterpret_cast<uint8_t*>(in_row + ST);                // [NW waves][32 rows]
  int seg, bi;
  xcd_tile(blockIdx.x, n_blk, seg, bi);
  if (seg >= segs[0]) return;
  const int e = segs[1 + 4 * seg], start = segs[2 + 4 * seg], n = segs[3 + 4 * seg];
  const int D = P.D, FF = P.FF, k = P.k, E = P.E;
  const bool shared = e == E;
  const int row0 = shared ? T * k + start : offsets[e] + start;        // rows of hb / yp
  if constexpr (QT == GM_QTYPE_IQ3_XXS) {
    gm_stage_grid(grid);
    pf_stage_signs(sgn);
  }
  if (threadIdx.x < ST) in_row[threadIdx.x] = row0 + (threadIdx.x < n ? threadIdx.x : 0);
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15;
  const int64_t rb = gm_row_bytes(QT, FF);
  const uint8_t* wrows = (shared ? static_cast<const uint8_t*>(P.down_sh)
                                 : static_cast<const uint8_t*>(P.down_exps) + (int64_t)e * D * rb) +
                         (int64_t)(wave * 32) * rb;
  const int n_groups = (D + 32 * NW - 1) / (32 * NW), g0 = bi * rg_per_blk;    // D % 256 == 0: whole groups
  const int g1 = g0 + rg_per_blk < n_groups ? g0 + rg_per_blk : n_groups;
  uint8_t* wbuf = wl + wave * S::WBUF;
  run_lds_load<S::RUN>(wrows + (int64_t)g0 * (32 * NW) * rb, wbuf);
  constexpr int G = S::ROWB / 16, NI = ST * G / (64 * NW);
  const int used = ((n + 15) & ~15) * G - 64 * __builtin_amdgcn_readfirstlane(wave);   // granules of the tiles in use
#pragma unroll
  for (int m = 0; m < NI; ++m) {                       // h rows, swizzled as b_lds reads them
    if (64 * NW * m >= used) break;
    const int id = 64 * (NW * m + wave) + lane, r = id / G, g = (id % G) ^ (r & 15);
    lds_load16(hh + (int64_t)in_row[r] * FF + 8 * g, hl + (NW * m + wave) * 1024);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  nt_dispatch<ST / 16>((n + 15) >> 4, [&](auto nt) {
    constexpr int NT = decltype(nt)::value;
    float cs[NT];                                                       // h scale of each output column
#pragma unroll
    for (int t = 0; t < NT; ++t) cs[t] = hsc[in_row[t * 16 + l16]];
    dn_loop<QT, NSB, ST, NW, NT>(wrows, rb, wbuf, hl, grid, sgn, g0, g1, n, cs, yp + (int64_t)row0 * D, D);
  });
}

template <int QT, int ST>
int launch_gateup(const gm_moe_layer* L, const PfWs& w, int nseg, int T, hipStream_t s) {
  const int nrt = L->FF / 64;
  constexpr size_t smem = GuShape<QT, ST>::SMEM;
  if (int rc = gm_set_smem(k_pf_gateup<QT, ST>, smem)) return rc;
  hipLaunchKernelGGL((k_pf_gateup<QT, ST>), dim3((nseg + 7) / 8 * 8 * nrt), dim3(256), smem, s, *L, w.segs,
                     w.offsets, w.sorted, w.xh, w.xsc, w.hb, T, nrt);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

template <int QT, int NSB, int ST, int NW>
int launch_down(const gm_moe_layer* L, const PfWs& w, int nseg, int T, hipStream_t s) {
  constexpr int kGroupsPerBlock = 2;
  const int n_blk = ((L->D + 32 * NW - 1) / (32 * NW) + kGroupsPerBlock - 1) / kGroupsPerBlock;
  constexpr size_t smem = DnShape<QT, NSB, ST, NW>::SMEM;
  if (int rc = gm_set_smem(k_pf_down<QT, NSB, ST, NW>, smem)) return rc;
  hipLaunchKernelGGL((k_pf_down<QT, NSB, ST, NW>), dim3((nseg + 7) / 8 * 8 * n_blk), dim3(64 * NW), smem, s, *L,
                     w.segs, w.offsets, w.hh, w.hsc, w.yp, T, n_blk, kGroupsPerBlock);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

// --------------------------------------------------------------- combine
// One block per token: y = sum_j w_j * yp[pos_j] over the token's experts in
// ascending id (= ascending sorted position), + shared gate * yp[P + t] (+ x).
__global__ void __launch_bounds__(256) k_pf_combine(const float* __restrict__ x, const float* __restrict__ yp,
                                                    const int32_t* __restrict__ inv, const float* __restrict__ wts,
                                                    const float* __restrict__ shg, int T, int k, int D, int has_sh,
                                                    int flags, float* __restrict__ y) {
  const int t = blockIdx.x;
  int pos[8];
  float w[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    pos[j] = j < k ? inv[t * k + j] : 0x7fffffff;
    w[j] = j < k ? wts[t * k + j] : 0.f;
  }
  // insertion sort by position (k <= 8)
#pragma unroll
  for (int i = 1; i < 8; ++i) {
#pragma unroll
    for (int j = i; j > 0; --j) {
      if (pos[j] < pos[j - 1]) {
        const int tp = pos[j]; pos[j] = pos[j - 1]; pos[j - 1] = tp;
        const float tw = w[j]; w[j] = w[j - 1]; w[j - 1] = tw;
      }
    }
  }
  const float sg = has_sh ? shg[t] : 0.f;
  const int Ptot = T * k, nq = D >> 2;
  const gm_f32x4* yp4 = reinterpret_cast<const gm_f32x4*>(yp);
  const gm_f32x4* x4 = reinterpret_cast<const gm_f32x4*>(x + (int64_t)t * D);
  constexpr int CS = 2;                      // column steps whose loads are issued together
  for (int c0 = threadIdx.x; c0 < nq; c0 += 256 * CS) {
    gm_f32x4 v[CS][9], xv[CS];
#pragma unroll
    for (int u = 0; u < CS; ++u) {
      const int c = min(c0 + 256 * u, nq - 1);                   // past the row: a duplicate, not stored
#pragma unroll
      for (int j = 0; j < 8; ++j) v[u][j] = yp4[(int64_t)(j < k ? pos[j] : pos[0]) * nq + c];
      v[u][8] = yp4[(int64_t)(has_sh ? Ptot + t : pos[0]) * nq + c];
      xv[u] = (flags & GM_MOE_RESIDUAL) ? x4[c] : gm_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < CS; ++u) {
      const int c = c0 + 256 * u;
      if (c >= nq) break;
      gm_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < k) {
          acc.x = fmaf(w[j], v[u][j].x, acc.x); acc.y = fmaf(w[j], v[u][j].y, acc.y);
          acc.z = fmaf(w[j], v[u][j].z, acc.z); acc.w = fmaf(w[j], v[u][j].w, acc.w);
        }
      if (has_sh) {
        acc.x += sg * v[u][8].x; acc.y += sg * v[u][8].y; acc.z += sg * v[u][8].z; acc.w += sg * v[u][8].w;
      }
      if (flags & GM_MOE_RESIDUAL) {
        acc.x = xv[u].x + acc.x; acc.y = xv[u].y + acc.y; acc.z = xv[u].z + acc.z; acc.w = xv[u].w + acc.w;
      }
      reinterpret_cast<gm_f32x4*>(y + (int64_t)t * D)[c] = acc;
    }
  }
}

// ------------------------------------------------- shared expert in I8 rows
// A shared expert held as I8 rows (the reference model's K-quant shared
// experts, transcoded) beside IQ routed experts runs as two dense GEMMs of its
// own over all T tokens, on the routed experts' f16 MFMA: A = the I8 weights
// decoded to f16 (s q + off, rounded once), B = the tokens' f16 rows (xh for
// gate/up, the scaled SwiGLU rows hh for down).  Wave tile: 16 weight rows x
// 16 kShTiles tokens over a K part, one I8 sub-block (32 k) per step, one
// decoded A operand for kShTiles MFMAs: lane l holds row l % 16 and k-octet
// o = l / 16 of A (8 quants, 8 bytes, and the sub-block's {s0, s1, off}),
// token l % 16 of each token tile and the same octet of B (16 bytes).
// Sub-blocks are loaded kShStep at a time into two register sets used in turn
// (no register copy at the loop latch), so one set's loads are in flight
// while the other is multiplied.
constexpr int kShStep = 2;
constexpr int kShTiles = 4;           // 16-token tiles per wave: one decoded A operand, 4 MFMAs

typedef uint32_t gm_u32x3 __attribute__((ext_vector_type(3)));

struct I8Oct {
  uint2 q;       // quants 8o .. 8o + 7 of the sub-block
  gm_u32x3 m;    // s0 (quants 0-15), s1 (16-31), off
};

__device__ __forceinline__ I8Oct i8_oct_load(const uint8_t* __restrict__ row, int sub, int o) {
  const uint8_t* sb = row + sub * 48;
  return I8Oct{*reinterpret_cast<const uint2*>(sb + 8 * o), *reinterpret_cast<const gm_u32x3*>(sb + 32)};
}

// The octet's 8 weights s q + off as f16 (each rounded once from fp32, where
// s q + off is the transcoded row's exact weight).
__device__ __forceinline__ gm_f16x8 i8_oct_f16(const I8Oct& r, int o) {
  const float sc = __uint_as_float(o < 2 ? r.m.x : r.m.y), off = __uint_as_float(r.m.z);
  gm_f16x8 a;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    a[b] = (_Float16)fmaf(sc, gm_sbyte(r.q.x, b), off);
    a[4 + b] = (_Float16)fmaf(sc, gm_sbyte(r.q.y, b), off);
  }
  return a;
}

// One pipeline stage: kShStep sub-blocks of NW weight rows and of the
// kShTiles token rows.
template <int NW>
struct ShStage {
  I8Oct w[NW][kShStep];
  gm_u32x4 b[kShStep][kShTiles];
};

template <int NW>
__device__ __forceinline__ void sh_stage_load(ShStage<NW>& st, const uint8_t* const (&wrow)[NW],
                                              const uint16_t* const (&brow)[kShTiles], int s0, int o) {
#pragma unroll
  for (int i = 0; i < kShStep; ++i) {
#pragma unroll
    for (int n = 0; n < NW; ++n) st.w[n][i] = i8_oct_load(wrow[n], s0 + i, o);
#pragma unroll
    for (int j = 0; j < kShTiles; ++j) st.b[i][j] = *reinterpret_cast<const gm_u32x4*>(brow[j] + 32 * (s0 + i));
  }
  issue_fence();
}

template <int NW>
__device__ __forceinline__ void sh_stage_mfma(const ShStage<NW>& st, int o, gm_f32x4 (&acc)[NW][kShTiles]) {
#pragma unroll
  for (int i = 0; i < kShStep; ++i) {
#pragma unroll
    for (int n = 0; n < NW; ++n) {
      const gm_f16x8 A = i8_oct_f16(st.w[n][i], o);
#pragma unroll
      for (int j = 0; j < kShTiles; ++j)
        acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, __builtin_bit_cast(gm_f16x8, st.b[i][j]), acc[n][j],
                                                           0, 0, 0);
    }
  }
  issue_fence();
}

// acc[n][j] = W_n[rows r0 .. r0 + 15] . brow[j] over sub-blocks [sb, sb + ns) (ns
// a multiple of 2 kShStep) for the lane's token of tile j.
template <int NW>
__device__ __forceinline__ void sh_gemm_tile(const uint8_t* const (&wrow)[NW], const uint16_t* const (&brow)[kShTiles],
                                             int sb, int ns, int o, gm_f32x4 (&acc)[NW][kShTiles]) {
#pragma unroll
  for (int n = 0; n < NW; ++n)
#pragma unroll
    for (int j = 0; j < kShTiles; ++j) acc[n][j] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
  ShStage<NW> sa, sb2;
  const int se = sb + ns;
  sh_stage_load<NW>(sa, wrow, brow, sb, o);
  for (int s0 = sb; s0 < se; s0 += 2 * kShStep) {
    sh_stage_load<NW>(sb2, wrow, brow, s0 + kShStep, o);
    sh_stage_mfma<NW>(sa, o, acc);
    const int s2 = s0 + 2 * kShStep < se ? s0 + 2 * kShStep : s0;      // the last round reloads, unused
    sh_stage_load<NW>(sa, wrow, brow, s2, o);
    sh_stage_mfma<NW>(sb2, o, acc);
  }
}

// K parts: the block's 4 waves split K into nkw parts (4, 2 or 1) of whole
// pipeline rounds and cover 4 / nkw token groups; the parts are added in LDS
// in part order by the group's part-0 wave.
inline int sh_kparts(int nsub) {
  return nsub % (8 * kShStep) == 0 ? 4 : nsub % (4 * kShStep) == 0 ? 2 : 1;
}

// Sums the block's K parts of acc (LDS red: 4 waves x NW x kShTiles x 256
// floats) into the part-0 wave of each token group; true on those waves.
template <int NW>
__device__ __forceinline__ bool sh_reduce(gm_f32x4 (&acc)[NW][kShTiles], int nkw, float* __restrict__ red) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, part = wave % nkw;
  gm_f32x4* r4 = reinterpret_cast<gm_f32x4*>(red);
  if (nkw > 1 && part != 0) {
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int j = 0; j < kShTiles; ++j) r4[((wave * NW + n) * kShTiles + j) * 64 + lane] = acc[n][j];
  }
  __syncthreads();
  if (part != 0) return false;
  for (int p = 1; p < nkw; ++p)
#pragma unroll
    for (int n = 0; n < NW; ++n)
#pragma unroll
      for (int j = 0; j < kShTiles; ++j) acc[n][j] += r4[(((wave + p) * NW + n) * kShTiles + j) * 64 + lane];
  return true;
}

// h[P + t] = silu(g) u for the shared expert, t < T: block (row tile of 16 FF
// rows, 4 / nkw token groups of 16 kShTiles tokens, nkw K parts each); bf16
// rows as k_pf_gateup writes them.
__global__ void __launch_bounds__(256) k_pfs_gateup_i8(const uint8_t* __restrict__ wg, const uint8_t* __restrict__ wu,
                                                       int FF, int D, const uint16_t* __restrict__ xh,
                                                       const float* __restrict__ xsc, int T, int nkw,
                                                       uint16_t* __restrict__ hsh) {
  __shared__ float red[4 * 2 * kShTiles * 256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, o = lane >> 4;
  const int gpb = 4 / nkw, part = wave % nkw, ns = D / 32 / nkw;
  const int r0 = blockIdx.x * 16, t0 = (blockIdx.y * gpb + wave / nkw) * 16 * kShTiles;
  const int64_t rb = (int64_t)(D / 32) * 48;
  const uint8_t* const wrow[2] = {wg + (r0 + l16) * rb, wu + (r0 + l16) * rb};
  const uint16_t* brow[kShTiles];
#pragma unroll
  for (int j = 0; j < kShTiles; ++j) {                         // tokens past T read a valid row, unstored
    const int t = t0 + 16 * j + l16;
    brow[j] = xh + (int64_t)(t < T ? t : T - 1) * D + 8 * o;
  }
  gm_f32x4 acc[2][kShTiles];
  sh_gemm_tile<2>(wrow, brow, part * ns, ns, o, acc);
  if (!sh_reduce<2>(acc, nkw, red)) return;
#pragma unroll
  for (int j = 0; j < kShTiles; ++j) {                         // C: rows r0 + 4 o + i, token column l16
    const int t = t0 + 16 * j + l16;
    if (t < T) {
      const float ds = xsc[t];
      const gm_f32x4 g = acc[0][j] * ds, u = acc[1][j] * ds;
      const gm_f32x2 h01 = {gm_silu(g[0]) * u[0], gm_silu(g[1]) * u[1]};
      const gm_f32x2 h23 = {gm_silu(g[2]) * u[2], gm_silu(g[3]) * u[3]};
      *reinterpret_cast<uint2*>(hsh + (int64_t)t * FF + r0 + 4 * o) =
          make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(h01, gm_bf16x2)),
                     __builtin_bit_cast(uint32_t, __builtin_convertvector(h23, gm_bf16x2)));
    }
  }
}

// y[t] = W_down h[t] for the shared expert from its scaled f16 rows (hh, scales
// hsc, as k_pf_h16 writes them): block (row tile of 16 D rows, 4 / nkw token
// groups, nkw K parts), fp32 rows y[t] that k_pf_combine adds last.
__global__ void __launch_bounds__(256) k_pfs_down_i8(const uint8_t* __restrict__ wd, int D, int FF,
                                                     const uint16_t* __restrict__ hh, const float* __restrict__ hsc,
                                                     int T, int nkw, float* __restrict__ y) {
  __shared__ float red[4 * kShTiles * 256];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, o = lane >> 4;
  const int gpb = 4 / nkw, part = wave % nkw, ns = FF / 32 / nkw;
  const int r0 = blockIdx.x * 16, t0 = (blockIdx.y * gpb + wave / nkw) * 16 * kShTiles;
  const int64_t rb = (int64_t)(FF / 32) * 48;
  const uint8_t* const wrow[1] = {wd + (r0 + l16) * rb};
  const uint16_t* brow[kShTiles];
#pragma unroll
  for (int j = 0; j < kShTiles; ++j) {
    const int t = t0 + 16 * j + l16;
    brow[j] = hh + (int64_t)(t < T ? t : T - 1) * FF + 8 * o;
  }
  gm_f32x4 acc[1][kShTiles];
  sh_gemm_tile<1>(wrow, brow, part * ns, ns, o, acc);
  if (!sh_reduce<1>(acc, nkw, red)) return;
#pragma unroll
  for (int j = 0; j < kShTiles; ++j) {
    const int t = t0 + 16 * j + l16;
    if (t < T) *reinterpret_cast<gm_f32x4*>(y + (int64_t)t * D + r0 + 4 * o) = acc[0][j] * hsc[t];
  }
}

// Steps 1-3: prep and router (xn32: also the fp32 rows xn, or NULL), top-k and
// dispatch into segs (shared_T: tokens of the shared expert's own segments, or 0).
// fold: see router_step.
int pf_route(const gm_moe_layer* L, const float* x, int T, uint8_t* ws, const GmMoeWs& lay, const PfWs& w,
             float* xn32, int shared_T, int32_t* segs, int seg_tok, bool fold, hipStream_t s) {
  const int D = L->D, E = L->E, k = L->k;
  float* logits = reinterpret_cast<float*>(ws + lay.logits);
  float* shg = reinterpret_cast<float*>(ws + lay.shg);
  int32_t* ids = reinterpret_cast<int32_t*>(ws + lay.ids);
  float* wts = reinterpret_cast<float*>(ws + lay.wts);
  const int nrows = E + (L->sh_gate_inp ? 1 : 0);
  const int ldp = router_ld(L);
  const int nsplit = router_split(D);
  {
    const int nrb = (nrows + 63) / 64, ntb = (T + 15) / 16, n_rt = nrb * ntb * nsplit;
    const dim3 g((unsigned)(n_rt + T));
    const bool f32 = L->q_router == GM_QTYPE_F32;
#define GM_PR(NK, F32, FOLD)                                                                                     \
  hipLaunchKernelGGL((k_pf_prep_router<NK, F32, FOLD>), g, dim3(256), 0, s, L->router, L->sh_gate_inp, x, L->norm_w, \
                     L->norm_eps, T, D, E, ldp, w.part, nrb, ntb, n_rt, w.xh, w.xsc, xn32, w.rmsv)
#define GM_PR2(NK, F32)              \
  do {                               \
    if (fold) GM_PR(NK, F32, true);  \
    else GM_PR(NK, F32, false);      \
  } while (0)
    if (router_krange(D) == 512 && f32) GM_PR2(4, true);
    else if (router_krange(D) == 512) GM_PR2(4, false);
    else if (f32) GM_PR2(2, true);
    else GM_PR2(2, false);
#undef GM_PR2
#undef GM_PR
  }
  GM_TRY(hipGetLastError());
  {
    const int hg = L->sh_gate_inp ? 1 : 0;
    const dim3 g((T + 3) / 4);
    if (E <= 256 && nsplit <= 4)
      hipLaunchKernelGGL((k_pf_topk<4, 4>), g, dim3(256), 0, s, w.part, ldp, nsplit, T, E, k, hg, L->router_bias,
                         w.rmsv, logits, shg, ids, wts);
    else if (E <= 256 && nsplit <= 8)
      hipLaunchKernelGGL((k_pf_topk<4, 8>), g, dim3(256), 0, s, w.part, ldp, nsplit, T, E, k, hg, L->router_bias,
                         w.rmsv, logits, shg, ids, wts);
    else if (E <= 256)
      hipLaunchKernelGGL((k_pf_topk<4, 16>), g, dim3(256), 0, s, w.part, ldp, nsplit, T, E, k, hg, L->router_bias,
                         w.rmsv, logits, shg, ids, wts);
    else if (nsplit <= 8)
      hipLaunchKernelGGL((k_pf_topk<8, 8>), g, dim3(256), 0, s, w.part, ldp, nsplit, T, E, k, hg, L->router_bias,
                         w.rmsv, logits, shg, ids, wts);
    else
      hipLaunchKernelGGL((k_pf_topk<8, 16>), g, dim3(256), 0, s, w.part, ldp, nsplit, T, E, k, hg, L->router_bias,
                         w.rmsv, logits, shg, ids, wts);
  }
  GM_TRY(hipGetLastError());
  return gm_launch_dispatch_seg(ids, T, k, E, w.counts, w.offsets, w.sorted, w.inv, segs, seg_tok, shared_T, s);
}

template <int QTG, int QTD>
int prefill_t(const gm_moe_layer* L, const float* x, float* y, int T, int flags, uint8_t* ws, const GmMoeWs& lay,
              hipStream_t s) {
  const int D = L->D, FF = L->FF, E = L->E, k = L->k;
  float* shg = reinterpret_cast<float*>(ws + lay.shg);
  float* wts = reinterpret_cast<float*>(ws + lay.wts);
  PfWs w = pf_layout(L, T, ws + lay.pre, nullptr);
  const bool has_sh = L->gate_sh != nullptr;
  const bool sh_apart = pf_shared_apart(L);
  const bool sh_gemm = has_sh && !sh_apart;          // the shared expert as the GEMMs' ninth unit
  // a shared expert in I8 rows: its own f16 MFMA GEMMs; other formats (bf16): the fp32 pass
  const bool sh_i8 = sh_apart && L->q_gate_sh == GM_QTYPE_I8 && L->q_up_sh == GM_QTYPE_I8 &&
                     L->q_down_sh == GM_QTYPE_I8;
  const bool sh_f32 = sh_apart && !sh_i8;
  const size_t P = (size_t)T * k;
  const int seg = pf_seg(L, T), nseg = max_segments(T, k, E, seg);
  if (int rc = pf_route(L, x, T, ws, lay, w, sh_f32 ? w.xn : nullptr, sh_gemm ? T : 0, w.segs, seg, false, s)) return rc;
  if (sh_f32) {                                      // shared expert rows yp[P + t], fp32
    if (int rc = gm_launch_gateup(L->q_gate_sh, L->gate_sh, L->up_sh, FF, D, w.xn, T, w.hsh, s)) return rc;
    if (int rc = gm_launch_matvec(L->q_down_sh, L->down_sh, D, FF, w.hsh, T, w.yp + P * D, s)) return rc;
  }
  if (int rc = seg == 64 ? launch_gateup<QTG, 64>(L, w, nseg, T, s) : launch_gateup<QTG, 32>(L, w, nseg, T, s))
    return rc;
  if (sh_i8) {                                       // shared SwiGLU rows hb[P + t] (D % 256 == 0)
    const int nkw = sh_kparts(D / 32), tok = 16 * kShTiles * (4 / nkw);    // tokens per block
    hipLaunchKernelGGL(k_pfs_gateup_i8, dim3(FF / 16, (T + tok - 1) / tok), dim3(256), 0, s,
                       static_cast<const uint8_t*>(L->gate_sh), static_cast<const uint8_t*>(L->up_sh), FF, D, w.xh,
                       w.xsc, T, nkw, w.hb + P * FF);
    GM_TRY(hipGetLastError());
  }
  {
    const int rows = T * k + (sh_gemm || sh_i8 ? T : 0);
    hipLaunchKernelGGL(k_pf_h16, dim3((rows + 3) / 4), dim3(256), 0, s, w.hb, rows, FF, w.hh, w.hsc);
    GM_TRY(hipGetLastError());
  }
  int rc;
  switch (FF / kChunk) {
    case 1: rc = seg == 64 ? launch_down<QTD, 1, 64, 8>(L, w, nseg, T, s) : launch_down<QTD, 1, 32, 4>(L, w, nseg, T, s); break;
    case 2: rc = seg == 64 ? launch_down<QTD, 2, 64, 8>(L, w, nseg, T, s) : launch_down<QTD, 2, 32, 4>(L, w, nseg, T, s); break;
    case 3: rc = launch_down<QTD, 3, 32, 4>(L, w, nseg, T, s); break;
    default: rc = launch_down<QTD, 4, 32, 4>(L, w, nseg, T, s); break;
  }
  if (rc) return rc;
  if (sh_i8) {                                       // shared expert rows yp[P + t] (FF % 256 == 0)
    const int nkw = sh_kparts(FF / 32), tok = 16 * kShTiles * (4 / nkw);
    hipLaunchKernelGGL(k_pfs_down_i8, dim3(D / 16, (T + tok - 1) / tok), dim3(256), 0, s,
                       static_cast<const uint8_t*>(L->down_sh), D, FF, w.hh + P * FF, w.hsc + P, T, nkw,
                       w.yp + P * D);
    GM_TRY(hipGetLastError());
  }
  hipLaunchKernelGGL(k_pf_combine, dim3(T), dim3(256), 0, s, x, w.yp, w.inv, wts, shg, T, k, D, has_sh ? 1 : 0,
                     flags, y);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

}  // namespace

size_t gm_prefill_scratch_bytes(const gm_moe_layer* L, int T) {
  size_t total = 0;
  pf_layout(L, T, nullptr, &total);
  return total;
}

// Layers whose routed experts (and shared expert, if any) are I8 rows, on the
// GEMMs of prefill_i8.hip: activations to 2^-23 of each sub-block's largest, as
// their decode kernels have, and the widths that those take (the same layer in a smaller workspace runs on
// them, and wider ones are refused there).
bool gm_pf8_ok(const gm_moe_layer* L) {
  const bool sh = !L->gate_sh || (L->q_gate_sh == GM_QTYPE_I8 && L->q_down_sh == GM_QTYPE_I8);
  return L->q_gate == GM_QTYPE_I8 && L->q_down == GM_QTYPE_I8 && sh && L->D % kChunk == 0 && L->FF % kChunk == 0 &&
         L->D <= 4096 && L->FF <= 2048;                         // router_split <= kRouterSplit
}

struct Pf8Ws {
  int32_t* segs;       // the segment list (of kPf8Seg tokens: more of them than PfWs's)
  float* xn;           // [T][D] fp32 rows
  float* h;            // [P + T][FF] fp32 SwiGLU rows
  GmPf8Rows xr, hr;    // their planes (hi of both and lo of h in PfWs's f16 rows)
};

static Pf8Ws pf8_layout(const gm_moe_layer* L, int T, const PfWs& w, uint8_t* base, size_t* total) {
  const size_t P = (size_t)T * L->k, D = L->D, FF = L->FF;
  size_t o = 0;
  auto take = [&](size_t bytes) { uint8_t* p = base ? base + o : nullptr; o = align256(o + bytes); return p; };
  Pf8Ws v{};
  v.segs = reinterpret_cast<int32_t*>(take((1 + 4 * (size_t)max_segments(T, L->k, L->E, kPf8Seg)) * 4));
  v.xn = reinterpret_cast<float*>(take(T * D * 4));
  v.xr = GmPf8Rows{w.xh, reinterpret_cast<uint16_t*>(take(T * D * 2)), reinterpret_cast<float*>(take(T * (D / 32) * 8))};
  v.h = reinterpret_cast<float*>(take((P + T) * FF * 4));
  v.hr = GmPf8Rows{w.hh, w.hb, reinterpret_cast<float*>(take((P + T) * (FF / 32) * 8))};
  if (total) *total = o;
  return v;
}

size_t gm_pf8_scratch_bytes(const gm_moe_layer* L, int T) {
  size_t total = 0;
  pf8_layout(L, T, PfWs{}, nullptr, &total);
  return total;
}

int gm_pf8_run(const gm_moe_layer* L, const float* x, float* y, int T, int flags, uint8_t* ws, const GmMoeWs& lay,
               hipStream_t s) {
  const int D = L->D, FF = L->FF, k = L->k;
  const PfWs w = pf_layout(L, T, ws + lay.pre, nullptr);
  const Pf8Ws v = pf8_layout(L, T, w, ws + lay.pre8, nullptr);
  const bool has_sh = L->gate_sh != nullptr;
  const int nseg = max_segments(T, k, L->E, kPf8Seg);
  if (int rc = pf_route(L, x, T, ws, lay, w, v.xn, has_sh ? T : 0, v.segs, kPf8Seg, true, s)) return rc;
  if (int rc = gm_pf8_split(v.xn, T, D, v.xr, s)) return rc;
  if (int rc = gm_pf8_gemm(L, false, v.xr, v.segs, nseg, w.offsets, w.sorted, T, v.h, s)) return rc;
  if (int rc = gm_pf8_split(v.h, T * k + (has_sh ? T : 0), FF, v.hr, s)) return rc;
  if (int rc = gm_pf8_gemm(L, true, v.hr, v.segs, nseg, w.offsets, w.sorted, T, w.yp, s)) return rc;
  hipLaunchKernelGGL(k_pf_combine, dim3(T), dim3(256), 0, s, x, w.yp, w.inv, reinterpret_cast<float*>(ws + lay.wts),
                     reinterpret_cast<float*>(ws + lay.shg), T, k, D, has_sh ? 1 : 0, flags, y);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

int gm_pf_run(const gm_moe_layer* L, const float* x, float* y, int T, int flags, uint8_t* ws, const GmMoeWs& lay,
              hipStream_t s) {
  if (L->D % kChunk || L->FF % kChunk || L->FF > 4 * kChunk)
    return gm_fail_arg("gm_moe_forward: prefill needs D and FF multiples of %d and FF <= %d", kChunk, 4 * kChunk);
  if (router_split(L->D) > kRouterSplit)
    return gm_fail_arg("gm_moe_forward: prefill supports D <= 8192 (a multiple of 512 above 4096); D=%d", L->D);
  const int qg = L->q_gate, qd = L->q_down;
  if (qg == GM_QTYPE_IQ4_XS && qd == GM_QTYPE_IQ3_XXS) return prefill_t<GM_QTYPE_IQ4_XS, GM_QTYPE_IQ3_XXS>(L, x, y, T, flags, ws, lay, s);
  if (qg == GM_QTYPE_IQ3_XXS && qd == GM_QTYPE_IQ4_XS) return prefill_t<GM_QTYPE_IQ3_XXS, GM_QTYPE_IQ4_XS>(L, x, y, T, flags, ws, lay, s);
  if (qg == GM_QTYPE_IQ4_XS && qd == GM_QTYPE_IQ4_XS) return prefill_t<GM_QTYPE_IQ4_XS, GM_QTYPE_IQ4_XS>(L, x, y, T, flags, ws, lay, s);
  if (qg == GM_QTYPE_IQ3_XXS && qd == GM_QTYPE_IQ3_XXS) return prefill_t<GM_QTYPE_IQ3_XXS, GM_QTYPE_IQ3_XXS>(L, x, y, T, flags, ws, lay, s);
  return gm_fail_arg("gm_moe_forward: unsupported routed formats gate/up %d down %d", qg, qd);
}
