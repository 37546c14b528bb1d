// Dense bf16-weight GEMM for many tokens: y[t][m] = sum_k W[m][k] x[t][k]
// (+ add[t][m]), W bf16 row-major, x / y / add fp32, fp32 accumulation.  It
// serves the prompts' projections (NpuLinear, the core layers, lm_head); a few
// tokens on few rows stay on k_mv_bf16_mfma (mv_bf16.hip).
//
// v_mfma_f32_16x16x32_bf16 with the weight rows as A and the tokens as B, x
// split into three exact bf16 planes (bf16_split.h), so an MFMA triple is 8192
// exact bf16 x fp32 products.  Three MFMAs of 16 cycles share one A operand,
// which makes the operands' way, not the matrix cores, the bound:
//  * the weights of a tile (16 RT rows x 64 k) go through LDS, since every wave
//    of a block needs all of them;
//  * a wave has 16 tokens of its own, whose x goes from global memory to
//    registers and is split there, once per block (planes formed beforehand and
//    loaded instead, 6 bytes a value against 4: 134.6 -> 168 us at M = 9216,
//    K = 2048, T = 1021);
//  * both are loaded one step ahead in registers; what one block waits for its
//    loads (1.2 us a step when alone on a CU) two or three others fill.
// One token tile per wave against two at the same row count: 136 against 163 us
// there, 57 against 73 at T = 300 (more blocks, three to a CU).
// A step's 64 k are summed by themselves, the lower planes first, two row tiles'
// chains of MFMAs in turn, and then added to the running sum: error against 64
// bits 1.2e-7 (one chain through all steps: 5e-7 at K = 2048, 7e-7 at 4096; the
// few-token kernel: 2.5e-7), at the same speed as adding every 256 k (1.8e-7).
// Measured before (k_mv_bf16_mfma, every weight read per 16 tokens) and now, us:
//   M = 9216 K = 2048:  T = 24 26 -> 19, 57 41 -> 23, 120 76 -> 37, 300 199 -> 58, 1021 651 -> 141
//   M = 2048 K = 4096:  T = 100 44 -> 40, 300 114 -> 45, 1000 364 -> 77
//   M = 248320 K = 2048: T = 20 508 -> 274, 57 1051 -> 296
// (T = 1021: 819 TFLOP/s on the matrix cores; a large library product: 1120.)
#include "bf16_split.h"
#include "kernels.h"

#include <type_traits>

namespace {

constexpr int kBK = 64;                       // k values per step (two 32-wide MFMA k-steps)
struct GemmArgs {
  const uint16_t* w;     // [M][K]
  const uint16_t* w2;    // [M2][K] rows that follow w's (M2 = 0: none)
  const float* x;        // [T][K]
  const float* add;      // [T][M] or NULL
  float* y;              // [T][M]
  float* y2;             // [T][M2]
  int M, M2, K, T;
  int nc;                // token tiles
  int tiles, per_xcd;    // tiles in all, and per XCD (rounded up)
  int vec;               // y, y2, add rows 16-byte aligned: four outputs per store
};

template <int RT, int KS>
__global__ void __launch_bounds__(256 * KS, KS == 1 ? 2 : 1) k_gemm_bf16(GemmArgs P) {
  constexpr int NA = RT / 2;                                    // 16-byte granules of A per thread and step
  constexpr int ABUF = RT * 16 * 2 * kBK;                       // bytes of one A tile
  __shared__ __attribute__((aligned(16))) uint8_t smem[KS * 2 * ABUF];
  const int tile = (blockIdx.x & 7) * P.per_xcd + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= P.per_xcd || tile >= P.tiles) return;
  const int grp = KS > 1 ? threadIdx.x >> 8 : 0, tid = threadIdx.x & 255;
  const int wave = tid >> 6, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
  const int row0 = (tile / P.nc) * (16 * RT), tok0 = (tile % P.nc) * 64 + wave * 16;
  const int Mt = P.M + P.M2, K = P.K;
  uint8_t* abuf = smem + grp * 2 * ABUF;

  const uint16_t* ap[NA];
  int aoff[NA], agran[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    const int gi = tid + 256 * j, r = gi >> 3;
    const int row = min(row0 + r, Mt - 1);                      // rows past Mt: loaded, never stored
    ap[j] = row < P.M ? P.w + (int64_t)row * K : P.w2 + (int64_t)(row - P.M) * K;
    // granule g of a step holds k = 8 g .. + 7: two pieces of 4, for lane quarters
    // 2 (g & 1) and 2 (g & 1) + 1 of k-step g >> 2 (slots 4 (g >> 2) + quarter, XORed
    // with the row pair), the first or the second half of their 8 k's
    const int g = gi & 7, sl = (4 * (g >> 2) + 2 * (g & 1)) ^ ((r >> 1) & 7);
    agran[j] = g;
    aoff[j] = r * (2 * kBK) + 16 * sl + 8 * ((g >> 1) & 1);
  }
  const int tok = tok0 + l16;
  const float* xp = P.x + (int64_t)min(tok, P.T - 1) * K + 4 * q;

  const int nstep = (K + kBK - 1) / kBK, chunk = (nstep + KS - 1) / KS;
  const int s0 = grp * chunk, s1 = min(s0 + chunk, nstep);
  gm_u32x4 ar[NA];
  gm_f32x4 xr[2][2];
  auto load = [&](int s) {                                      // past the row: its last granule again, unused
    const int k0 = s * kBK;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 2; ++p) xr[h][p] = *reinterpret_cast<const gm_f32x4*>(xp + min(k0 + 32 * h, K - 32) + 16 * p);
#pragma unroll
    for (int j = 0; j < NA; ++j)
      ar[j] = *reinterpret_cast<const gm_u32x4*>(ap[j] + min(k0 + 8 * agran[j], K - 8));
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int j = 0; j < NA; ++j) {
      *reinterpret_cast<gm_u32x2*>(abuf + b * ABUF + aoff[j]) = gm_u32x2{ar[j].x, ar[j].y};
      *reinterpret_cast<gm_u32x2*>(abuf + b * ABUF + (aoff[j] ^ 16)) = gm_u32x2{ar[j].z, ar[j].w};
    }
  };

  gm_f32x4 acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = gm_f32x4{0.f, 0.f, 0.f, 0.f};

  load(min(s0, nstep - 1));
  stage(0);
  __syncthreads();
  auto step = [&](int i, auto odd) {
    constexpr Sign sign = step_sign(decltype(odd)::value);
    const int s = s0 + i;
    gm_f32x4 xc[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 2; ++p) xc[h][p] = xr[h][p];
    const bool more = i + 1 < chunk;
    if (more) load(min(s + 1, nstep - 1));
    if (s < s1) {
      const uint8_t* A = abuf + (i & 1) * ABUF;
      gm_u32x4 pl[2][3];
#pragma unroll
      for (int h = 0; h < 2; ++h) split3(xc[h][0], xc[h][1], pl[h], sign);
      const bool half = s * kBK + 32 >= K;                      // K % 64 == 32: half a last step
      constexpr int RG = 2;                                     // row tiles at a time: two independent chains
#pragma unroll
      for (int r0 = 0; r0 < RT; r0 += RG) {
        gm_bf16x8 a[RG][2];
        gm_f32x4 d[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r) {
          const int ra = 16 * (r0 + r) + l16;
#pragma unroll
          for (int h = 0; h < 2; ++h)
            a[r][h] = *reinterpret_cast<const gm_bf16x8*>(A + ra * (2 * kBK) + 16 * ((4 * h + q) ^ ((ra >> 1) & 7)));
          d[r] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
        }
        auto mul = [&](int h, int p) {
#pragma unroll
          for (int r = 0; r < RG; ++r)
            d[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r][h], __builtin_bit_cast(gm_bf16x8, pl[h][p]), d[r], 0, 0, 0);
        };
        if (!half) {
          mul(1, 2);
          mul(0, 2);
          mul(1, 1);
          mul(0, 1);
          mul(1, 0);
        } else {
          mul(0, 2);
          mul(0, 1);
        }
        mul(0, 0);
#pragma unroll
        for (int r = 0; r < RG; ++r) acc[r0 + r] += sign.f * d[r];
      }
    }
    if (more) stage((i + 1) & 1);
    __syncthreads();
  };
  for (int i = 0; i < chunk; i += 2) {                          // the signs as constants
    step(i, std::integral_constant<int, 0>{});
    if (i + 1 < chunk) step(i + 1, std::integral_constant<int, 1>{});
  }
  if constexpr (KS > 1) {                                       // K parts added in part order
    gm_f32x4* red = reinterpret_cast<gm_f32x4*>(smem);
    if (grp > 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r) red[(((grp - 1) * 4 + wave) * RT + r) * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int g = 0; g < KS - 1; ++g)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[r] += red[((g * 4 + wave) * RT + r) * 64 + lane];
  }
  // C layout: lane l holds rows 4 (l / 16) + i of a row tile, token column l % 16
  if (tok >= P.T) return;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = row0 + 16 * r + 4 * q;
    if (row >= Mt) continue;
    if (P.vec) {                                                // M % 4 == 0: four rows of one matrix
      const bool one = row < P.M;
      const int64_t o = one ? (int64_t)tok * P.M + row : (int64_t)tok * P.M2 + (row - P.M);
      gm_f32x4 v = acc[r];
      if (P.add && one) v = *reinterpret_cast<const gm_f32x4*>(P.add + o) + v;
      *reinterpret_cast<gm_f32x4*>((one ? P.y : P.y2) + o) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = row + i;
        if (m >= Mt) break;
        const bool one = m < P.M;
        const int64_t o = one ? (int64_t)tok * P.M + m : (int64_t)tok * P.M2 + (m - P.M);
        (one ? P.y : P.y2)[o] = P.add && one ? P.add[o] + acc[r][i] : acc[r][i];
      }
    }
  }
}

template <int RT, int KS>
int launch(GemmArgs P, hipStream_t s) {
  P.nc = (P.T + 63) / 64;
  P.tiles = ((P.M + P.M2 + 16 * RT - 1) / (16 * RT)) * P.nc;
  P.per_xcd = (P.tiles + 7) / 8;
  hipLaunchKernelGGL((k_gemm_bf16<RT, KS>), dim3(8 * P.per_xcd), dim3(256 * KS), 0, s, P);
  GM_TRY(hipGetLastError());
  return GM_OK;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

// Tile shape by how many blocks the call gives (T = 17 and up):
//   128 x 64 tiles when they fill the chip at least once (>= 300);
//   the same with K split over two halves of a 512-thread block (>= 128):
//     M = 2048 K = 4096 T = 1000 (256 tiles) 73 against 84 us, M = 9216 T = 120 (144) 35 against 41;
//   below that 64 x 64 tiles with K split over four quarters of a 1024-thread
//     block: M = 9216 T = 57 (72) 23 against 33 us, M = 2048 K = 4096 T = 300 (80) 44 against 64.
// Such a tile takes as long whatever part of the chip the tiles fill, while the
// few-token kernel's time goes with its 16 x 16 tiles; these are counted (few-token
// kernel / this one, us):
//   K = 4096, M = 2048: T = 65 (640) 31 / 40, 96 (768) 36 / 40, 97 (896) 42 / 40
//   K = 2048, M = 3072: T = 64 (768) 20 / 22, 65 (960) 23 / 22; M = 4096: T = 33 (768) 17 / 19, 49 (1024) 23 / 22
//   up to 32 tokens, K = 2048: M = 4096 (512) 13 / 18, 6144 (768) 18 / 17
//   K = 512, M = 4096: T = 65 (1280) 8.4 / 8.7, 96 (1536) 11 / 9
bool gm_gemm_bf16_takes(int rows, int K, int T) {
  return T > 16 && (int64_t)((rows + 15) / 16) * ((T + 15) / 16) >= (T <= 32 ? 736 : K < 1024 ? 1300 : 800);
}

int gm_launch_gemm_bf16(const uint16_t* w, int M, const uint16_t* w2, int M2, int K, const float* x, int T,
                        const float* add, float* y, float* y2, hipStream_t s) {
  GemmArgs P{w, w2, x, add, y, y2, M, w2 ? M2 : 0, K, T, 0, 0, 0, 0};
  P.vec = M % 4 == 0 && P.M2 % 4 == 0 && aligned16(y) && aligned16(y2) && aligned16(add);
  const int64_t t128 = (int64_t)((M + P.M2 + 127) / 128) * ((T + 63) / 64);
  if (t128 >= INT32_MAX / 16) return gm_fail_arg("gemm_bf16: %d rows x %d tokens is too large", M + P.M2, T);
  if (t128 >= 300) return launch<8, 1>(P, s);
  if (t128 >= 128) return launch<8, 2>(P, s);
  return launch<4, 4>(P, s);
}
