// A prompt (T >= 2 tokens) through the core layers, all tokens in each launch:
// gated attention (qwen/forward.py:133-239) and the Gated DeltaNet (:292-431).
// Same functions, weights and state as the one-token path (core_decode.hip);
// fp32 activations, state and sums.  Up to kMaxTok tokens run at a time (the
// caller's workspace holds their intermediates); the caches and states carry a
// longer prompt from one such part to the next.
//
// Attention (gm_attn_prefill):
//   k_rms_row        h = rmsnorm(x, attn_norm)
//   dense            qkv = h Wqkv^T (gemm_bf16.hip / mv_bf16.hip)
//   k_pf_qk          q heads RMSNormed and rotated in place, k heads RMSNormed,
//                    rotated and written with v to the caches
//   k_pf_attn        online-softmax attention on fp32 MFMA, keys cut into parts
//                    where the tokens alone do not fill the chip
//   k_pf_attn_merge  the parts merged, times sigmoid(gate) (several parts only)
//   dense            y = out Wo^T (+ x)
// Gated DeltaNet (gm_ssm_prefill):
//   k_rms_row, dense mixed = h W_in^T and z = h W_gate^T in one launch
//   k_pf_ab          exp(g) and beta of every token and V head
//   k_pf_conv        the causal conv, SiLU, q / k L2 norms, and k . q per K head
//   k_pf_delta       the delta rule over the tokens, state in registers; the
//                    new conv state
//   k_pf_gnorm       rmsnorm(o_head, ssm_norm) * silu(z)
//   dense            y = o W_out^T (+ x)
#include "common.h"
#include "kernels.h"

namespace {

constexpr int kMaxTok = 1024;

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// ------------------------------------------------------------ attention
// One wave per head row of one token (4 rows per block): the q heads, then the
// kv heads.  Any even rope_dim <= Dh: the normalised row goes through LDS for
// the rotation's partner (i, i + rd / 2).
template <int DV>
__global__ void __launch_bounds__(256) k_pf_qk(float* __restrict__ qkv, int T, int Hq, int Hkv, int rd, int pos0,
                                               const float* __restrict__ q_norm, const float* __restrict__ k_norm,
                                               float eps, const float* __restrict__ cosr,
                                               const float* __restrict__ sinr, float* __restrict__ kc,
                                               float* __restrict__ vc) {
  constexpr int Dh = 64 * DV;
  __shared__ float rows[4][Dh];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nh = Hq + Hkv;
  const int64_t idx = (int64_t)blockIdx.x * 4 + wave;
  const bool live = idx < (int64_t)T * nh;                     // a wave past the end repeats the last row
  const int64_t id = live ? idx : (int64_t)T * nh - 1;
  const int t = (int)(id / nh), h = (int)(id % nh);
  const bool isq = h < Hq;
  float* tok = qkv + (int64_t)t * (2 * Hq + 2 * Hkv) * Dh;
  float* src = isq ? tok + (int64_t)2 * Dh * h : tok + (int64_t)2 * Dh * Hq + (int64_t)Dh * (h - Hq);
  const float* nw = isq ? q_norm : k_norm;
  float v[DV], n[DV];
  float ss = 0.f;
#pragma unroll
  for (int d = 0; d < DV; ++d) { v[d] = src[lane + 64 * d]; ss = fmaf(v[d], v[d], ss); }
  const float r = 1.0f / sqrtf(gm_wave_sum64(ss) / (float)Dh + eps);
#pragma unroll
  for (int d = 0; d < DV; ++d) { n[d] = (v[d] * r) * nw[lane + 64 * d]; rows[wave][lane + 64 * d] = n[d]; }
  __syncthreads();
  if (!live) return;
  const int half = rd >> 1;
  const float* cp = cosr + (int64_t)(pos0 + t) * rd;
  const float* sp = sinr + (int64_t)(pos0 + t) * rd;
  const int64_t crow = ((int64_t)(pos0 + t) * Hkv + (h - Hq)) * Dh;
#pragma unroll
  for (int d = 0; d < DV; ++d) {
    const int i = lane + 64 * d;
    float o = n[d];
    if (i < rd) o = o * cp[i] + (i < half ? -rows[wave][i + half] : rows[wave][i - half]) * sp[i];
    if (isq) {
      src[i] = o;
    } else {
      kc[crow + i] = o;
      vc[crow + i] = src[(int64_t)Dh * Hkv + i];
    }
  }
}

struct AttnP {
  const float* qkv;      // [T][(2 Hq + 2 Hkv) Dh]: rotated q (and its gate) per head
  const float* kc;       // [max_pos][Hkv][Dh]
  const float* vc;
  float* out;            // [T][Hq Dh]
  float* part;           // [nsplit][T Hq][Dh + 4]: {m, l, -, -, o} (nsplit > 1)
  int T, Hq, Hkv, pos0, nsplit, nblk;
  float scale;
};

// Whether the wave's V tile (k_pf_attn) holds an infinity or NaN.
template <int DV>
__device__ __forceinline__ bool v_not_finite(const float* V, const int (&vo)[4]) {
  bool odd = false;
#pragma unroll
  for (int g = 0; g < DV; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const gm_f32x4 v = *reinterpret_cast<const gm_f32x4*>(V + vo[i] + 64 * g);
#pragma unroll
      for (int c = 0; c < 4; ++c) odd |= !(fabsf(v[c]) < __builtin_inff());
    }
  return __any(odd);
}

// A tile's part of 64 output dims of k_pf_attn without the MFMAs: each row adds
// the keys up to its last one and never multiplies a later one.
template <int Dh>
__device__ __forceinline__ void v_masked(const float* V, int g, int key0, int last, const float (&p)[4],
                                         gm_f32x4 (&w)[4]) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
#pragma unroll 1
  for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 4 * k4 + i;
      const float pk = __shfl(p[i], 16 * k4 + l16, 64);
      if (key0 + key > last) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const gm_f32x4 v = *reinterpret_cast<const gm_f32x4*>(V + key * Dh + 4 * ((16 * g + 4 * q + e) ^ key));
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c][e] = fmaf(pk, v[c], w[c][e]);
      }
    }
}

// Attention of 64 query rows (16 per wave) of one kv head over one part of
// their keys, on v_mfma_f32_16x16x4_f32.  A kv head's rows are its T tokens x G
// = Hq / Hkv heads, head fastest, so a block's rows span few positions and
// nearly all their keys are common.  Keys come 16 at a time: the K and V rows
// of the next 16 go from global memory straight to LDS while these are used.
//   S^T = K Q^T   lane (l16, q) = (lane % 16, lane / 16): A = key l16, B = query
//                 l16, dims 16 s + 4 q + j in MFMA j of step s (one 16-byte LDS
//                 read, four MFMAs); the lane gets keys 4 q + i of query l16
//   O^T += V^T P^T  its scores are B operands as they lie: MFMA i takes key 4 q
//                 + i; A = dims 64 g + 4 l16 + c (one 16-byte LDS read, four
//                 tiles c); the lane gets dims 64 g + 16 q + 4 i + c of query l16
// so neither the scores nor K or V are ever transposed.  16-byte granule g of
// an LDS row r sits at g ^ (r & 15): the 16 keys that a wave reads at once hit
// different banks.  Scores are added up SC MFMAs at a time, and a tile's part of
// the output is formed by itself (OC chains), then o a + part (chains of MFMAs
// through all dims and keys: error of the layer against 64 bits 6.1e-7 at 1021
// tokens on 300 with heads of 256, one token at a time 3.3e-7).  Short chains for
// heads of up to 128, whose projections round less: 64 tokens on 500 with heads of
// 128 2.5e-7 -> 2.2e-7, one token at a time 2.2e-7.  For 256 the long ones: 2.5e-7
// against 3.0e-7, and the short ones cost 175 -> 207 us at 1021 tokens on 300.
template <int DV>
__global__ void __launch_bounds__(256, DV <= 4 ? 2 : 1) k_pf_attn(AttnP P) {
  constexpr int Dh = 64 * DV, NG = Dh / 4, NS = Dh / 16, TILE = 16 * Dh;   // floats of 16 rows
  constexpr int SC = DV <= 2 ? 2 : 8, OC = DV <= 2 ? 2 : 1;                // MFMAs in a chain of scores; chains of outputs
  extern __shared__ __attribute__((aligned(16))) float sm[];               // [2][K, V][TILE]
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int G = P.Hq / P.Hkv, R = P.T * G;
  // longest blocks first; the second part of a block's keys from the other end,
  // so that the two blocks of a CU are a long and a short one
  int b = blockIdx.x;
  const int split = b / (P.nblk * P.Hkv);
  b -= split * P.nblk * P.Hkv;
  const int hk = b % P.Hkv, bi = b / P.Hkv;
  const int blk = split & 1 ? bi : P.nblk - 1 - bi;
  const int r = min(blk * 64 + wave * 16 + l16, R - 1);                    // rows past R: never stored
  const int t = r / G, h = hk * G + (r - t * G);
  const int64_t ldq = (int64_t)(2 * P.Hq + 2 * P.Hkv) * Dh;
  const float* qrow = P.qkv + t * ldq + (int64_t)2 * Dh * h;
  const int last = P.pos0 + t;                                             // the row's last key
  const int first = __builtin_amdgcn_readfirstlane(last);                  // the least of the wave's
  const int nkeys = P.pos0 + min((blk * 64 + 63) / G, P.T - 1) + 1;        // of the block
  const int ntile = (nkeys + 15) / 16, per = (ntile + P.nsplit - 1) / P.nsplit;
  const int i0 = split * per, i1 = min(i0 + per, ntile);

  gm_f32x4 qv[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) qv[s] = *reinterpret_cast<const gm_f32x4*>(qrow + 16 * s + 4 * q);
  gm_f32x4 o[DV][4];
#pragma unroll
  for (int g = 0; g < DV; ++g)
#pragma unroll
    for (int c = 0; c < 4; ++c) o[g][c] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;

  auto load = [&](int tile, int buf) {                                     // 2 DV KB per wave, 1 KB an instruction
#pragma unroll
    for (int j = 0; j < DV; ++j) {
      const int gi = (wave * DV + j) * 64 + lane, row = gi / NG, g = (gi % NG) ^ (row & 15);
      const int64_t off = ((int64_t)min(tile * 16 + row, nkeys - 1) * P.Hkv + hk) * Dh + 4 * g;
      __builtin_amdgcn_global_load_lds(P.kc + off, sm + 2 * buf * TILE + (wave * DV + j) * 256, 16, 0, 0);
      __builtin_amdgcn_global_load_lds(P.vc + off, sm + (2 * buf + 1) * TILE + (wave * DV + j) * 256, 16, 0, 0);
    }
  };
  // the XOR touches the low four bits of a granule's number only: 4 addresses each
  int ko[4], vo[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    ko[u] = l16 * Dh + 4 * ((4 * u + q) ^ l16);
    vo[u] = (4 * q + u) * Dh + 4 * (l16 ^ (4 * q + u));
  }
  if (i0 < i1) load(i0, 0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int it = i0; it < i1; ++it) {
    const int buf = (it - i0) & 1;
    if (it + 1 < i1) load(it + 1, buf ^ 1);
    const float* K = sm + 2 * buf * TILE;
    const float* V = K + TILE;
    gm_f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS; s += 4) {                                      // 64 dims, 16 MFMAs
      constexpr int NC = 16 / SC;
      gm_f32x4 d[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) d[c] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const gm_f32x4 k = *reinterpret_cast<const gm_f32x4*>(K + ko[u] + 16 * s);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          gm_f32x4& a = d[NC == 2 ? u & 1 : 2 * u + j / 2];
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j], qv[s + u][j], a, 0, 0, 0);
        }
      }
#pragma unroll
      for (int h = NC / 2; h > 0; h /= 2)
#pragma unroll
        for (int c = 0; c < h; ++c) d[c] += d[c + h];
      sc += d[0];
    }
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = it * 16 + 4 * q + i <= last ? sc[i] * P.scale : -__builtin_inff();
    float mn = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
    mn = fmaxf(mn, __shfl_xor(mn, 16, 64));
    mn = fmaxf(fmaxf(mn, __shfl_xor(mn, 32, 64)), m);
    const float mr = mn == -__builtin_inff() ? 0.f : mn;                   // every key so far masked
    const float a = expf(m - mr);
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = expf(p[i] - mr);
    l = fmaf(l, a, (p[0] + p[1]) + (p[2] + p[3]));
    m = mn;
    // a key that is masked for some of the wave's rows has probability 0 there, and
    // 0 times a V value that is not finite would be NaN
    const bool odd = it * 16 + 15 > first && v_not_finite<DV>(V, vo);
#pragma unroll
    for (int g = 0; g < DV; ++g) {
      gm_f32x4 w[OC][4];
#pragma unroll
      for (int h = 0; h < OC; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) w[h][c] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
      if (!odd) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const gm_f32x4 v = *reinterpret_cast<const gm_f32x4*>(V + vo[i] + 64 * g);
#pragma unroll
          for (int c = 0; c < 4; ++c)
            w[i * OC / 4][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c], p[i], w[i * OC / 4][c], 0, 0, 0);
        }
      } else {
        v_masked<Dh>(V, g, it * 16, last, p, w[0]);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (OC == 2) w[0][c] += w[1][c];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[g][c][e] = fmaf(o[g][c][e], a, w[0][c][e]);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (blk * 64 + wave * 16 + l16 >= R) return;
  if (P.nsplit > 1) {
    float* pr = P.part + ((int64_t)split * P.T * P.Hq + (int64_t)t * P.Hq + h) * (Dh + 4);
    if (q == 0) { pr[0] = m; pr[1] = l; }
#pragma unroll
    for (int g = 0; g < DV; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<gm_f32x4*>(pr + 4 + 64 * g + 16 * q + 4 * i) =
            gm_f32x4{o[g][0][i], o[g][1][i], o[g][2][i], o[g][3][i]};
    return;
  }
  float* orow = P.out + ((int64_t)t * P.Hq + h) * Dh;
#pragma unroll
  for (int g = 0; g < DV; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 64 * g + 16 * q + 4 * i;
      const gm_f32x4 gt = *reinterpret_cast<const gm_f32x4*>(qrow + Dh + d);
      gm_f32x4 v;
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = (o[g][c][i] / l) * (1.0f / (1.0f + expf(-gt[c])));
      *reinterpret_cast<gm_f32x4*>(orow + d) = v;
    }
}

// out = (sum_s o_s e^(m_s - M)) / (sum_s l_s e^(m_s - M)) * sigmoid(gate), one
// thread per 4 dims; parts without a key of the row have m = -inf.
__global__ void __launch_bounds__(256) k_pf_attn_merge(AttnP P, int Dh) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int nq = Dh / 4;
  const int64_t row = i / nq, rows = (int64_t)P.T * P.Hq;
  if (row >= rows) return;
  const int d = 4 * (int)(i - row * nq), t = (int)(row / P.Hq), h = (int)(row - (int64_t)t * P.Hq);
  const float* p = P.part + row * (Dh + 4);
  const int64_t ss = rows * (Dh + 4);
  float M = -__builtin_inff();
  for (int s = 0; s < P.nsplit; ++s) M = fmaxf(M, p[s * ss]);
  float L = 0.f;
  gm_f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < P.nsplit; ++s) {
    const float f = p[s * ss] == -__builtin_inff() ? 0.f : expf(p[s * ss] - M);
    L = fmaf(p[s * ss + 1], f, L);
    const gm_f32x4 v = *reinterpret_cast<const gm_f32x4*>(p + s * ss + 4 + d);
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = fmaf(v[c], f, o[c]);
  }
  const gm_f32x4 g = *reinterpret_cast<const gm_f32x4*>(P.qkv + (int64_t)t * (2 * P.Hq + 2 * P.Hkv) * Dh +
                                                        (int64_t)2 * Dh * h + Dh + d);
#pragma unroll
  for (int c = 0; c < 4; ++c) o[c] = (o[c] / L) * (1.0f / (1.0f + expf(-g[c])));
  *reinterpret_cast<gm_f32x4*>(P.out + row * Dh + d) = o;
}

// ------------------------------------------------------------ Gated DeltaNet
// exp(g) and beta for 16 tokens x 64 of the 2 Hv alpha / beta rows (fp32
// weights) on v_mfma_f32_16x16x4_f32: the block's 8 waves take every eighth
// 16-wide k-step (all four row tiles each) and are added pairwise in LDS order.
// Each k-step is summed by itself and four of them pairwise: beta at D = 2048
// within 7.5e-8 of 64 bits (one chain through all of a wave's steps: 1.8e-7,
// which the state of the delta rule feels most).
// ab[t][r]: r < Hv exp(softplus(alpha_r . h + dt_bias) a), else beta.
__global__ void __launch_bounds__(512) k_pf_ab(const float* __restrict__ alpha, const float* __restrict__ beta,
                                               const float* __restrict__ dt_bias, const float* __restrict__ a,
                                               const float* __restrict__ hx, int T, int D, int Hv,
                                               float* __restrict__ ab) {
  __shared__ gm_f32x4 red[7][4][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q = lane >> 4;
  const int tok = blockIdx.x * 16 + l16, r0 = blockIdx.y * 64, nr = 2 * Hv;
  const float* xr = hx + (int64_t)min(tok, T - 1) * D + 4 * q;
  const float* wr[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = min(r0 + 16 * j + l16, nr - 1);
    wr[j] = (r < Hv ? alpha + (int64_t)r * D : beta + (int64_t)(r - Hv) * D) + 4 * q;
  }
  gm_f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
  auto load = [&](int k, gm_f32x4& x, gm_f32x4 (&w)[4]) {
    x = *reinterpret_cast<const gm_f32x4*>(xr + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const gm_f32x4*>(wr[j] + k);
  };
  auto step = [&](const gm_f32x4& x, const gm_f32x4& w) {
    gm_f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_16x16x4f32(w[e], x[e], d, 0, 0, 0);
    return d;
  };
  int k = 16 * wave;
  if (k + 384 < D) {                                            // four steps at a time, the next four on their way
    gm_f32x4 xn[4], wn[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) load(k + 128 * u, xn[u], wn[u]);
    for (; k + 384 < D; k += 512) {
      gm_f32x4 x[4], w[4][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        x[u] = xn[u];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[u][j] = wn[u][j];
      }
      const int k1 = k + 512 + 384 < D ? k + 512 : k;           // the last round reloads, unused
#pragma unroll
      for (int u = 0; u < 4; ++u) load(k1 + 128 * u, xn[u], wn[u]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] += (step(x[0], w[0][j]) + step(x[1], w[1][j])) + (step(x[2], w[2][j]) + step(x[3], w[3][j]));
    }
  }
  for (; k < D; k += 128) {
    gm_f32x4 x, w[4];
    load(k, x, w);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] += step(x, w[j]);
  }
  if (wave > 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave - 1][j][lane] = acc[j];
  }
  __syncthreads();
  if (wave > 0 || tok >= T) return;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    acc[j] = ((acc[j] + red[0][j][lane]) + (red[1][j][lane] + red[2][j][lane])) +
             ((red[3][j][lane] + red[4][j][lane]) + (red[5][j][lane] + red[6][j][lane]));
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + 16 * j + 4 * q + i;
      if (r >= nr) continue;
      const float s = acc[j][i];
      float o;
      if (r < Hv) {
        const float u = s + dt_bias[r];
        o = expf((u > 20.f ? u : log1pf(expf(u))) * a[r]);
      } else {
        o = 1.0f / (1.0f + expf(-s));
      }
      ab[(int64_t)tok * nr + r] = o;
    }
}

constexpr int kConvTok = 16;       // consecutive tokens of one wave

// The conv, SiLU and norms of one head's channels (CL = Sk / 64 per lane) over
// kConvTok tokens, the last ck - 1 inputs kept in registers (in[0 .. 6], oldest
// first, the newest at 6).
template <int CL>
struct ConvHead {
  float w[CL][8], in[CL][7];
  const float* src;
  int ld;
  __device__ __forceinline__ void init(const float* conv_w, const float* state, const float* mixed, int c0, int ck,
                                       int C, int t0) {
    const int lane = threadIdx.x & 63;
    src = mixed + c0 + lane;
    ld = C;
#pragma unroll
    for (int u = 0; u < CL; ++u) {
      const int c = c0 + lane + 64 * u;
#pragma unroll
      for (int j = 0; j < 8; ++j) w[u][j] = j < 8 - ck ? 0.f : conv_w[(int64_t)c * ck + j - (8 - ck)];
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        const int t = t0 - 7 + j;                               // the input of token t
        in[u][j] = j < 8 - ck ? 0.f
                 : t >= 0 ? mixed[(int64_t)t * C + c] : state[(int64_t)c * (ck - 1) + (ck - 1 + t)];
      }
    }
  }
  __device__ __forceinline__ void step(int t, float (&o)[CL]) {
#pragma unroll
    for (int u = 0; u < CL; ++u) {
      const float x = src[(int64_t)t * ld + 64 * u];
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 7; ++j) acc = fmaf(w[u][j], in[u][j], acc);
      acc = fmaf(w[u][7], x, acc);
#pragma unroll
      for (int j = 0; j < 6; ++j) in[u][j] = in[u][j + 1];
      in[u][6] = x;
      o[u] = acc / (1.0f + expf(-acc));
    }
  }
};

// One wave per (head, 16 tokens): heads [0, Hk) a K head's q and k rows and the
// products that k_pf_delta needs of them, heads [Hk, Hk + Hv) a V head's row.
// conv[t][C] as mixed; kq[t][head][kKq]: k_t . q_t, k_(t-i) . k_t and k_(t-i) . q_t
// for i = 1 .. 3 (those that leave a group of 4 tokens are not read).
constexpr int kKq = 8;

template <int CL>
__global__ void __launch_bounds__(256) k_pf_conv(const float* __restrict__ mixed, const float* __restrict__ w,
                                                 const float* __restrict__ state, int T, int ck, int Hk, int Hv,
                                                 float eps, float* __restrict__ conv, float* __restrict__ kq) {
  constexpr int Sk = 64 * CL;
  const int lane = threadIdx.x & 63, nt = (T + kConvTok - 1) / kConvTok;
  const int id = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= nt * (Hk + Hv)) return;
  const int hd = id / nt, t0 = (id % nt) * kConvTok, t1 = min(t0 + kConvTok, T), C = (2 * Hk + Hv) * Sk;
  if (hd >= Hk) {
    const int c0 = (Hk + hd) * Sk;
    ConvHead<CL> v;
    v.init(w, state, mixed, c0, ck, C, t0);
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
      float o[CL];
      v.step(t, o);
#pragma unroll
      for (int u = 0; u < CL; ++u) conv[(int64_t)t * C + c0 + lane + 64 * u] = o[u];
    }
    return;
  }
  const int cq = hd * Sk, ckk = (Hk + hd) * Sk;
  ConvHead<CL> qh, kh;
  qh.init(w, state, mixed, cq, ck, C, t0);
  kh.init(w, state, mixed, ckk, ck, C, t0);
  const float qs = 1.0f / sqrtf((float)Sk);
  float kp[3][CL];                                              // k of the 3 tokens before, the newest first
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int u = 0; u < CL; ++u) kp[i][u] = 0.f;
#pragma unroll 2
  for (int t = t0; t < t1; ++t) {
    float a[CL], b[CL];
    qh.step(t, a);
    kh.step(t, b);
    float sa = 0.f, sb = 0.f, sp[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < CL; ++u) { sa = fmaf(a[u], a[u], sa); sb = fmaf(b[u], b[u], sb); }
    const float ra = sqrtf(fmaxf(gm_wave_sum64(sa), eps)), rb = sqrtf(fmaxf(gm_wave_sum64(sb), eps));
#pragma unroll
    for (int u = 0; u < CL; ++u) {
      a[u] = a[u] / ra * qs;
      b[u] = b[u] / rb;
      sp[0] = fmaf(a[u], b[u], sp[0]);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        sp[1 + i] = fmaf(kp[i][u], b[u], sp[1 + i]);
        sp[4 + i] = fmaf(kp[i][u], a[u], sp[4 + i]);
      }
      kp[2][u] = kp[1][u];
      kp[1][u] = kp[0][u];
      kp[0][u] = b[u];
      conv[(int64_t)t * C + cq + lane + 64 * u] = a[u];
      conv[(int64_t)t * C + ckk + lane + 64 * u] = b[u];
    }
    float sl = 0.f;                                             // lane i < 7: product i
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      const float v = gm_wave_sum64(sp[i]);
      sl = lane == i ? v : sl;
    }
    if (lane < 7) kq[((int64_t)t * Hk + hd) * kKq + lane] = sl;
  }
}

// Tokens staged in LDS at a time (two buffers of k and q rows: 32 KB at S = 128).
template <int S>
constexpr int kDeltaTok = S <= 128 ? 16 : 8;

// The delta rule of 16 state columns of one V head over all T tokens: 16 lanes
// hold a column (S / 16 rows each, four consecutive ones per 64), 4 columns per
// wave.  Per token, with the state s of the token before:
//   d = (v - e (s . k)) beta,  o = e (s . q) + (k . q) d,  s = e s + k d
// Four tokens at a time: the dot products of all four run on the state before
// them, and what the tokens between add to it, d_i k_i scaled by the e in
// between, enters through the products k_i . k_j and k_i . q_j of k_pf_conv, so
// one reduction over the 16 lanes stands between two groups.  1000 tokens of 32
// heads of 128 x 128: 189 us (216 with a reduction between two tokens).  256 blocks:
// a wave is alone on its SIMD, and its issue, an instruction every 5 to 6 cycles,
// is the kernel's time.  k, q, v and the scalars of 16 tokens are staged in LDS two
// buffers deep; o leaves through LDS in 64-byte pieces.  The first blocks also
// write the new conv state (its old value was read by the launch before).
template <int S>
__global__ void __launch_bounds__(256) k_pf_delta(float* __restrict__ state, const float* __restrict__ conv,
                                                  const float* __restrict__ ab, const float* __restrict__ kq, int T,
                                                  int Hk, int Hv, float* __restrict__ o,
                                                  const float* __restrict__ mixed, float* __restrict__ conv_state,
                                                  int ck) {
  constexpr int RP = S / 16, NI = S / 64;                       // state rows per lane, in NI groups of 4
  constexpr int TOK = kDeltaTok<S>;
  constexpr int NKQ = TOK * 2 * S / 4 / 256;                    // 16-byte loads of k and q per thread and stage
  __shared__ __attribute__((aligned(16))) float skq[2][TOK][2][S];
  __shared__ __attribute__((aligned(16))) float sc[2][TOK][12];      // e, beta, the products of k_pf_conv
  __shared__ float sv[2][TOK][16], so[2][TOK][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, p = lane & 15, q = lane >> 4;
  const int hv = blockIdx.x, c0 = blockIdx.y * 16, hk = hv % Hk, C = (2 * Hk + Hv) * S;
  const int cw = wave * 4 + q, col = c0 + cw;                   // the lane's column
  {
    const int nb = gridDim.x * gridDim.y * 256;                 // new conv state: its last ck - 1 inputs
    for (int c = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x; c < C && ck > 1; c += nb) {
      float* st = conv_state + (int64_t)c * (ck - 1);
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (j < ck - 1) {
          const int t = T - (ck - 1) + j;
          st[j] = t >= 0 ? mixed[(int64_t)t * C + c] : st[j + T];
        }
    }
  }
  float* Sc = state + ((int64_t)hv * S) * S + col;
  float s[RP];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) s[4 * i + j] = Sc[(int64_t)(64 * i + 4 * p + j) * S];

  gm_f32x4 rkq[NKQ];
  float rv, rs;
  const int tv = threadIdx.x >> 4, cv = threadIdx.x & 15;       // tokens x 16 columns, scalars in cv < 9
  auto load = [&](int t0) {                                     // tokens past T repeat the last one, unused
#pragma unroll
    for (int i = 0; i < NKQ; ++i) {
      const int g = threadIdx.x + 256 * i, t = g / (2 * S / 4), r = g % (2 * S / 4), which = r / (S / 4);
      rkq[i] = *reinterpret_cast<const gm_f32x4*>(conv + (int64_t)min(t0 + t, T - 1) * C + (which ? 0 : Hk * S) +
                                                  hk * S + 4 * (r % (S / 4)));
    }
    const int64_t t = min(t0 + tv, T - 1);
    rv = conv[t * C + 2 * Hk * S + hv * S + c0 + cv];
    rs = cv >= 2 ? kq[(t * Hk + hk) * kKq + (cv < 9 ? cv - 2 : 0)] : ab[t * 2 * Hv + (cv == 1 ? Hv : 0) + hv];
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < NKQ; ++i) reinterpret_cast<gm_f32x4*>(skq[b])[threadIdx.x + 256 * i] = rkq[i];
    if (tv < TOK) {
      sv[b][tv][cv] = rv;
      if (cv < 9) sc[b][tv][cv] = rs;
    }
  };
  load(0);
  stage(0);
  __syncthreads();
  for (int t0 = 0, b = 0; t0 < T; t0 += TOK, b ^= 1) {
    load(min(t0 + TOK, T - 1));
    const int n = min(TOK, T - t0);
    auto step = [&](int t) {
      gm_f32x4 kv[NI], qv[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        kv[i] = *reinterpret_cast<const gm_f32x4*>(&skq[b][t][0][64 * i + 4 * p]);
        qv[i] = *reinterpret_cast<const gm_f32x4*>(&skq[b][t][1][64 * i + 4 * p]);
      }
      const gm_f32x4 e = *reinterpret_cast<const gm_f32x4*>(sc[b][t]);
      const float v = sv[b][t][cw];
      float a[NI], c[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        a[i] = s[4 * i] * kv[i].x;
        c[i] = s[4 * i] * qv[i].x;
#pragma unroll
        for (int j = 1; j < 4; ++j) { a[i] = fmaf(s[4 * i + j], kv[i][j], a[i]); c[i] = fmaf(s[4 * i + j], qv[i][j], c[i]); }
      }
#pragma unroll
      for (int i = 1; i < NI; ++i) { a[0] += a[i]; c[0] += c[i]; }
      const float sk = gm_row_sum16(a[0]), sq = gm_row_sum16(c[0]);
      const float d = (v - e.x * sk) * e.y;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[4 * i + j] = fmaf(kv[i][j], d, e.x * s[4 * i + j]);
      if (p == 0) so[b][t][cw] = fmaf(e.z, d, e.x * sq);
    };
    auto step4 = [&](int t) {
      gm_f32x4 kv[4][NI], qv[4][NI];
      float e[4], beta[4], v[4], kq0[4], kk[4][3], kq[4][3];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          kv[j][i] = *reinterpret_cast<const gm_f32x4*>(&skq[b][t + j][0][64 * i + 4 * p]);
          qv[j][i] = *reinterpret_cast<const gm_f32x4*>(&skq[b][t + j][1][64 * i + 4 * p]);
        }
        const gm_f32x4* r = reinterpret_cast<const gm_f32x4*>(sc[b][t + j]);
        const gm_f32x4 r0 = r[0], r1 = r[1];
        e[j] = r0.x; beta[j] = r0.y; kq0[j] = r0.z;
        kk[j][0] = r0.w; kk[j][1] = r1.x; kk[j][2] = r1.y;
        kq[j][0] = r1.z; kq[j][1] = r1.w; kq[j][2] = sc[b][t + j][8];
        v[j] = sv[b][t + j][cw];
      }
      float a[4], c[4];                                         // s . k_j and s . q_j
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float as[NI], cs[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          as[i] = s[4 * i] * kv[j][i].x;
          cs[i] = s[4 * i] * qv[j][i].x;
#pragma unroll
          for (int u = 1; u < 4; ++u) {
            as[i] = fmaf(s[4 * i + u], kv[j][i][u], as[i]);
            cs[i] = fmaf(s[4 * i + u], qv[j][i][u], cs[i]);
          }
        }
#pragma unroll
        for (int i = 1; i < NI; ++i) { as[0] += as[i]; cs[0] += cs[i]; }
        a[j] = gm_row_sum16(as[0]);
        c[j] = gm_row_sum16(cs[0]);
      }
      float d[4], out = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d[j] = (v[j] - e[j] * a[j]) * beta[j];
        const float oj = fmaf(kq0[j], d[j], e[j] * c[j]);
        out = (p & 3) == j ? oj : out;
#pragma unroll
        for (int l = j + 1; l < 4; ++l) {                       // token j's state under the later tokens
          a[l] = fmaf(kk[l][l - j - 1], d[j], e[j] * a[l]);
          c[l] = fmaf(kq[l][l - j - 1], d[j], e[j] * c[l]);
        }
      }
      so[b][t + (p & 3)][cw] = out;                             // four lanes the same value: no branch in the chain
      const float e23 = e[2] * e[3], e13 = e[1] * e23, e03 = e[0] * e13;
      const float d0 = d[0] * e13, d1 = d[1] * e23, d2 = d[2] * e[3];
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          s[4 * i + u] = fmaf(kv[3][i][u], d[3],
                              fmaf(kv[2][i][u], d2, fmaf(kv[1][i][u], d1, fmaf(kv[0][i][u], d0, e03 * s[4 * i + u]))));
    };
    if (n == TOK) {                                             // unrolled: the next tokens' LDS reads run ahead
#pragma unroll
      for (int t = 0; t < TOK; t += 4) step4(t);
    } else {
      int t = 0;
      for (; t + 4 <= n; t += 4) step4(t);
      for (; t < n; ++t) step(t);
    }
    stage(b ^ 1);
    __syncthreads();
    if (tv < n) o[(int64_t)(t0 + tv) * Hv * S + hv * S + c0 + cv] = so[b][tv][cv];
  }
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) Sc[(int64_t)(64 * i + 4 * p + j) * S] = s[4 * i + j];
}

// o <- rmsnorm(o_head, ssm_norm) * silu(z), one wave per head row.
template <int CL>
__global__ void __launch_bounds__(256) k_pf_gnorm(float* __restrict__ o, const float* __restrict__ nw,
                                                  const float* __restrict__ z, int64_t rows, float eps) {
  constexpr int S = 64 * CL;
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  float v[CL], zv[CL];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < CL; ++u) {
    v[u] = o[r * S + lane + 64 * u];
    zv[u] = z[r * S + lane + 64 * u];
  }
#pragma unroll
  for (int u = 0; u < CL; ++u) ss = fmaf(v[u], v[u], ss);
  const float k = 1.0f / sqrtf(gm_wave_sum64(ss) / (float)S + eps);
#pragma unroll
  for (int u = 0; u < CL; ++u)
    o[r * S + lane + 64 * u] = ((v[u] * k) * nw[lane + 64 * u]) * (zv[u] / (1.0f + expf(-zv[u])));
}

struct AttnWs { size_t h, qkv, out, part, total; int nblk, nsplit; };

// Key parts: the blocks of a few tokens do not fill the chip, so their keys are
// cut until there are about two blocks per CU: one part per 128 keys begun (129
// keys: two of 80 and 49) and 16 parts at most.  keys: cached positions with the
// prompt's own.
AttnWs attn_layout(const gm_attn_layer* L, int T, int keys) {
  AttnWs w{};
  const size_t Dh = (size_t)L->head_dim, Hq = (size_t)L->n_head, Hkv = (size_t)L->n_head_kv, Tz = (size_t)T;
  const int G = L->n_head / L->n_head_kv;
  w.nblk = (T * G + 63) / 64;
  const int want = 512 / (w.nblk * L->n_head_kv), most = (keys + 127) / 128;
  w.nsplit = want < 1 ? 1 : want > 16 ? 16 : want;
  if (w.nsplit > most) w.nsplit = most;
  size_t o = 0;
  w.h = o; o = align256(o + Tz * L->D * 4);
  w.qkv = o; o = align256(o + Tz * (2 * Hq + 2 * Hkv) * Dh * 4);
  w.out = o; o = align256(o + Tz * Hq * Dh * 4);
  w.part = o; o = align256(o + (w.nsplit > 1 ? (size_t)w.nsplit * Tz * Hq * (Dh + 4) * 4 : 0));
  w.total = o;
  return w;
}

struct SsmWs { size_t h, mixed, z, ab, conv, kq, o, total; };

SsmWs ssm_layout(const gm_ssm_layer* L, int T) {
  SsmWs w{};
  const size_t Tz = (size_t)T, Ck = (size_t)L->n_k_heads * L->d_state, di = (size_t)L->n_v_heads * L->d_state;
  const size_t C = 2 * Ck + di;
  size_t o = 0;
  w.h = o; o = align256(o + Tz * L->D * 4);
  w.mixed = o; o = align256(o + Tz * C * 4);
  w.z = o; o = align256(o + Tz * di * 4);
  w.ab = o; o = align256(o + Tz * 2 * L->n_v_heads * 4);
  w.conv = o; o = align256(o + Tz * C * 4);
  w.kq = o; o = align256(o + Tz * L->n_k_heads * kKq * 4);
  w.o = o; o = align256(o + Tz * di * 4);
  w.total = o;
  return w;
}

template <int DV>
int attn_part(const gm_attn_layer* L, const float* x, float* y, float* kc, float* vc, int T, int pos0, const float* cosr,
              const float* sinr, int flags, uint8_t* ws, hipStream_t s) {
  const AttnWs lay = attn_layout(L, T, pos0 + T);
  const int D = L->D, Hq = L->n_head, Hkv = L->n_head_kv, Dh = 64 * DV;
  float* h = reinterpret_cast<float*>(ws + lay.h);
  float* qkv = reinterpret_cast<float*>(ws + lay.qkv);
  float* out = reinterpret_cast<float*>(ws + lay.out);
  if (int rc = gm_launch_rms_row(x, L->attn_norm, D, T, L->eps, h, s)) return rc;
  if (int rc = gm_launch_dense(static_cast<const uint16_t*>(L->wqkv), (2 * Hq + 2 * Hkv) * Dh, nullptr, 0, D, h, T,
                               nullptr, qkv, nullptr, s))
    return rc;
  hipLaunchKernelGGL(k_pf_qk<DV>, dim3((T * (Hq + Hkv) + 3) / 4), dim3(256), 0, s, qkv, T, Hq, Hkv, L->rope_dim, pos0,
                     L->q_norm, L->k_norm, L->eps, cosr, sinr, kc, vc);
  GM_TRY(hipGetLastError());
  const AttnP P{qkv, kc, vc, out, reinterpret_cast<float*>(ws + lay.part), T, Hq, Hkv, pos0, lay.nsplit, lay.nblk,
                1.0f / sqrtf((float)Dh)};
  constexpr size_t smem = 4 * 16 * (size_t)(64 * DV) * sizeof(float);
  if (int rc = gm_set_smem(k_pf_attn<DV>, smem)) return rc;
  hipLaunchKernelGGL(k_pf_attn<DV>, dim3(lay.nblk * Hkv * lay.nsplit), dim3(256), smem, s, P);
  GM_TRY(hipGetLastError());
  if (lay.nsplit > 1) {
    const int64_t n = (int64_t)T * Hq * Dh / 4;
    hipLaunchKernelGGL(k_pf_attn_merge, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P, Dh);
    GM_TRY(hipGetLastError());
  }
  return gm_launch_dense(static_cast<const uint16_t*>(L->wo), D, nullptr, 0, Hq * Dh, out, T,
                         (flags & GM_MOE_RESIDUAL) ? x : nullptr, y, nullptr, s);
}

template <int S>
int ssm_part(const gm_ssm_layer* L, const float* x, float* y, float* conv_state, float* rec_state, int T, int flags,
             uint8_t* ws, hipStream_t s) {
  const SsmWs lay = ssm_layout(L, T);
  const int D = L->D, Hk = L->n_k_heads, Hv = L->n_v_heads, di = Hv * S, C = 2 * Hk * S + di;
  float* h = reinterpret_cast<float*>(ws + lay.h);
  float* mixed = reinterpret_cast<float*>(ws + lay.mixed);
  float* z = reinterpret_cast<float*>(ws + lay.z);
  float* ab = reinterpret_cast<float*>(ws + lay.ab);
  float* conv = reinterpret_cast<float*>(ws + lay.conv);
  float* kq = reinterpret_cast<float*>(ws + lay.kq);
  float* o = reinterpret_cast<float*>(ws + lay.o);
  if (int rc = gm_launch_rms_row(x, L->attn_norm, D, T, L->eps, h, s)) return rc;
  if (int rc = gm_launch_dense(static_cast<const uint16_t*>(L->w_in), C, static_cast<const uint16_t*>(L->w_gate), di,
                               D, h, T, nullptr, mixed, z, s))
    return rc;
  hipLaunchKernelGGL(k_pf_ab, dim3((T + 15) / 16, (2 * Hv + 63) / 64), dim3(512), 0, s, L->alpha, L->beta, L->dt_bias,
                     L->a, h, T, D, Hv, ab);
  GM_TRY(hipGetLastError());
  const int nw = (T + kConvTok - 1) / kConvTok * (Hk + Hv);
  hipLaunchKernelGGL(k_pf_conv<S / 64>, dim3((nw + 3) / 4), dim3(256), 0, s, mixed, L->conv1d, conv_state, T,
                     L->conv_k, Hk, Hv, L->eps, conv, kq);
  GM_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_pf_delta<S>, dim3(Hv, S / 16), dim3(256), 0, s, rec_state, conv, ab, kq, T, Hk, Hv, o, mixed,
                     conv_state, L->conv_k);
  GM_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_pf_gnorm<S / 64>, dim3((T * Hv + 3) / 4), dim3(256), 0, s, o, L->ssm_norm, z, (int64_t)T * Hv,
                     L->eps);
  GM_TRY(hipGetLastError());
  return gm_launch_dense(static_cast<const uint16_t*>(L->w_out), D, nullptr, 0, di, o, T,
                         (flags & GM_MOE_RESIDUAL) ? x : nullptr, y, nullptr, s);
}

}  // namespace

// Workspace of a prompt of T tokens in caches of max_pos positions: its parts
// are kMaxTok tokens and a rest, whose fewer tokens may have more key parts.
size_t gm_attn_prefill_ws(const gm_attn_layer* L, int T, int max_pos) {
  size_t most = attn_layout(L, T < kMaxTok ? T : kMaxTok, max_pos).total;
  if (T > kMaxTok && T % kMaxTok) {
    const size_t last = attn_layout(L, T % kMaxTok, max_pos).total;
    if (last > most) most = last;
  }
  return most;
}

size_t gm_ssm_prefill_ws(const gm_ssm_layer* L, int T) { return ssm_layout(L, T < kMaxTok ? T : kMaxTok).total; }

int gm_attn_prefill_run(const gm_attn_layer* L, const float* x, float* y, float* kc, float* vc, int T, int pos0,
                        const float* cosr, const float* sinr, int flags, uint8_t* ws, hipStream_t s) {
  for (int t = 0; t < T; t += kMaxTok) {
    const int n = T - t < kMaxTok ? T - t : kMaxTok;
    const float* xt = x + (int64_t)t * L->D;
    float* yt = y + (int64_t)t * L->D;
    int rc;
    switch (L->head_dim / 64) {
      case 1: rc = attn_part<1>(L, xt, yt, kc, vc, n, pos0 + t, cosr, sinr, flags, ws, s); break;
      case 2: rc = attn_part<2>(L, xt, yt, kc, vc, n, pos0 + t, cosr, sinr, flags, ws, s); break;
      case 4: rc = attn_part<4>(L, xt, yt, kc, vc, n, pos0 + t, cosr, sinr, flags, ws, s); break;
      default: rc = attn_part<8>(L, xt, yt, kc, vc, n, pos0 + t, cosr, sinr, flags, ws, s); break;
    }
    if (rc) return rc;
  }
  return GM_OK;
}

int gm_ssm_prefill_run(const gm_ssm_layer* L, const float* x, float* y, float* conv_state, float* rec_state, int T,
                       int flags, uint8_t* ws, hipStream_t s) {
  for (int t = 0; t < T; t += kMaxTok) {
    const int n = T - t < kMaxTok ? T - t : kMaxTok;
    const float* xt = x + (int64_t)t * L->D;
    float* yt = y + (int64_t)t * L->D;
    int rc;
    switch (L->d_state) {
      case 64: rc = ssm_part<64>(L, xt, yt, conv_state, rec_state, n, flags, ws, s); break;
      case 128: rc = ssm_part<128>(L, xt, yt, conv_state, rec_state, n, flags, ws, s); break;
      default: rc = ssm_part<256>(L, xt, yt, conv_state, rec_state, n, flags, ws, s); break;
    }
    if (rc) return rc;
  }
  return GM_OK;
}
