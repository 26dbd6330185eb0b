// gemv.hip -- linear layers of up to 4 rows (decode steps, the last rows of a window).
//
// Linear.Forward (src/LLM.Core/Layers/Layers.cs:29-37) for M <= 4 rows: y = epi(x @ W + b)
// (+ res) with W transposed as Wt[N][K], so a wave owns a column: its 64 lanes read the
// column's K values as contiguous 16-byte pieces, all of them in flight at once, and add
// up across the wave.  No partial sums and no second launch; with `ln` the LayerNorm of
// x runs in every wave's registers
// while its weights load.  HBM-bound for large K N; for small models a launch's fixed
// 2 us, so what counts is how few there are: 5 a layer where split-K products, their
// reductions, LayerNorms and the KV store took 9 (us per step: 4 layers, d 128: 141 -> 73;
// 16 layers, d 1024: 800 -> 482, 4 rows 866 -> 655; 12 layers, d 768, 2 rows: 571 -> 380).
//
// K > 1024 (mlp.proj): the four waves of a block take a quarter of K each, for four
// columns, and add up through LDS in wave order.
#include "kernels.hpp"

#include <math.h>

namespace fh {

namespace {

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

template <typename WT>
struct GemvArgs {
  const float* x;  // [M][K]
  const WT* Wt;    // [N][K]
  const float *ln_w, *ln_b, *bias, *res;
  float* y;  // [M][N]
  int M, K, N, kchunk;
  float eps;
  QkvStore<WT> kv;
};

constexpr int kOut = 0x7ffffff0;  // a byte offset past any operand: the load returns 0

template <typename WT, int MR, bool KS, int EPI>
__global__ __launch_bounds__(256) void k_gemv(GemvArgs<WT> g) {
  constexpr int VEC = 16 / sizeof(WT);
  constexpr int NI = 1024 / (64 * VEC);  // 16-byte pieces of a column per lane
  constexpr int NC = KS ? 4 : 1;         // columns per wave
  __shared__ float red[4][NC][MR];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col0 = blockIdx.x * 4 + (KS ? 0 : w);
  const int k0 = KS ? w * g.kchunk : 0, k1 = KS ? min(g.K, k0 + g.kchunk) : g.K;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<WT*>(g.Wt), (short)0, g.N * g.K * (int)sizeof(WT), 0x00020000);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.x), (short)0, g.M * g.K * 4, 0x00020000);
  u32x4_t wv[NC][NI];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int k = k0 + (64 * i + lane) * VEC;
      const bool on = k < k1 && col0 + c < g.N;
      wv[c][i] = __builtin_amdgcn_raw_buffer_load_b128(rw, on ? ((col0 + c) * g.K + k) * (int)sizeof(WT) : kOut, 0, 0);
    }
  float xv[MR][NI][VEC];
#pragma unroll
  for (int m = 0; m < MR; m++)
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int q = 0; q < VEC / 4; q++) {
        const int k = k0 + (64 * i + lane) * VEC + 4 * q;
        const bool on = k < k1 && m < g.M;
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rx, on ? (m * g.K + k) * 4 : kOut, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) xv[m][i][4 * q + j] = __uint_as_float(v[j]);
      }
  if constexpr (!KS) {
    if (g.ln_w) {
      const __amdgpu_buffer_rsrc_t rlw =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.ln_w), (short)0, g.K * 4, 0x00020000);
      const __amdgpu_buffer_rsrc_t rlb =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.ln_b), (short)0, g.K * 4, 0x00020000);
      float lw[NI][VEC], lb[NI][VEC];
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int q = 0; q < VEC / 4; q++) {
          const int k = (64 * i + lane) * VEC + 4 * q;
          const u32x4_t a = __builtin_amdgcn_raw_buffer_load_b128(rlw, k < g.K ? k * 4 : kOut, 0, 0);
          const u32x4_t b = __builtin_amdgcn_raw_buffer_load_b128(rlb, k < g.K ? k * 4 : kOut, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; j++) {
            lw[i][4 * q + j] = __uint_as_float(a[j]);
            lb[i][4 * q + j] = __uint_as_float(b[j]);
          }
        }
#pragma unroll
      for (int m = 0; m < MR; m++) {
        float s = 0.f, q2 = 0.f;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
          for (int j = 0; j < VEC; j++) s += xv[m][i][j];
        const float mu = wave_sum_dpp(s) / (float)g.K;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
          for (int j = 0; j < VEC; j++) {
            xv[m][i][j] = (64 * i + lane) * VEC < g.K ? xv[m][i][j] - mu : 0.f;  // K is a multiple of VEC
            q2 += xv[m][i][j] * xv[m][i][j];
          }
        const float rs = 1.f / sqrtf(wave_sum_dpp(q2) / (float)g.K + g.eps);
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
          for (int j = 0; j < VEC; j++) xv[m][i][j] = xv[m][i][j] * rs * lw[i][j] + lb[i][j];
      }
    }
  }
  float acc[NC][MR];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int m = 0; m < MR; m++) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < VEC; j++) {
          float wj;
          if constexpr (VEC == 4)
            wj = __uint_as_float(wv[c][i][j]);
          else
            wj = __uint_as_float(j & 1 ? wv[c][i][j / 2] & 0xffff0000u : wv[c][i][j / 2] << 16);
          s = fmaf(xv[m][i][j], wj, s);
        }
      acc[c][m] = wave_sum_dpp(s);
    }

  // results: lane m of the wave row m, or, over the waves' parts, thread c * MR + m
  int m = lane, col = col0;
  float v = 0.f;
  if constexpr (KS) {
    if (lane == 0)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int mm = 0; mm < MR; mm++) red[w][c][mm] = acc[c][mm];
    __syncthreads();
    if ((int)threadIdx.x >= NC * MR) return;
    const int c = threadIdx.x / MR;
    m = threadIdx.x % MR;
    col = col0 + c;
    v = red[0][c][m] + red[1][c][m] + red[2][c][m] + red[3][c][m];
  } else {
#pragma unroll
    for (int mm = 0; mm < MR; mm++)
      if (lane == mm) v = acc[0][mm];
  }
  if (m >= g.M || col >= g.N) return;
  if (g.bias) v += g.bias[col];
  if constexpr (EPI == EPI_GELU) v = gelu_tanh(v);
  if (g.res) v += g.res[(size_t)m * g.N + col];
  g.y[(size_t)m * g.N + col] = v;
  if constexpr (EPI == EPI_QKV) {
    // the K and V columns into the caches at the row's position, as k_kv_store writes them
    const int d = g.N / 3;
    if (col < d) return;
    const int pos = g.kv.src.pos_off + g.kv.src.pos_mul * *g.kv.src.step + m % g.kv.T;
    if ((unsigned)pos >= (unsigned)g.kv.ctx) return;
    const int hd = d / g.kv.H, cc = col < 2 * d ? col - d : col - 2 * d, h = cc / hd, e = cc % hd;
    const size_t dst = (((size_t)(m / g.kv.T) * g.kv.H + h) * g.kv.ctx + pos) * hd + e;
    (col < 2 * d ? g.kv.kc : g.kv.vc)[dst] = from_f32<WT>(v);
  }
}

template <typename WT, int MR, bool KS>
void launch_epi(hipStream_t st, int epi, const GemvArgs<WT>& g) {
  const dim3 grid((g.N + 3) / 4);
  if (epi == EPI_GELU)
    hipLaunchKernelGGL((k_gemv<WT, MR, KS, EPI_GELU>), grid, dim3(256), 0, st, g);
  else if (epi == EPI_QKV)
    hipLaunchKernelGGL((k_gemv<WT, MR, KS, EPI_QKV>), grid, dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((k_gemv<WT, MR, KS, EPI_NONE>), grid, dim3(256), 0, st, g);
}

}  // namespace

template <typename WT>
hipError_t launch_gemv(hipStream_t st, const float* x, int M, int K, const WT* Wt, int N, const float* ln_w,
                       const float* ln_b, float eps, const float* bias, int epi, const float* res, float* y,
                       const QkvStore<WT>* kv) {
  constexpr int VEC = 16 / sizeof(WT);
  if (!x || !Wt || !y || M <= 0 || M > 4 || K <= 0 || N <= 0 || K > 4096 || K % 8 != 0 ||
      (!ln_w) != (!ln_b) || (ln_w && K > 1024) || (epi == EPI_QKV) != (kv != nullptr) ||
      (size_t)N * K * sizeof(WT) >= (size_t)kOut)
    return hipErrorInvalidValue;
  if (kv && (!kv->kc || !kv->vc || !kv->src.step || kv->H <= 0 || kv->T <= 0 || M % kv->T != 0 || kv->ctx <= 0 ||
             N % 3 != 0 || N / 3 % kv->H != 0))
    return hipErrorInvalidValue;
  GemvArgs<WT> g{x, Wt, ln_w, ln_b, bias, res, y, M, K, N, 0, eps, kv ? *kv : QkvStore<WT>{}};
  g.kchunk = ((K + 3) / 4 + VEC - 1) / VEC * VEC;
  const bool ks = K > 1024;
  if (M == 1)
    ks ? launch_epi<WT, 1, true>(st, epi, g) : launch_epi<WT, 1, false>(st, epi, g);
  else if (M == 2)
    ks ? launch_epi<WT, 2, true>(st, epi, g) : launch_epi<WT, 2, false>(st, epi, g);
  else
    ks ? launch_epi<WT, 4, true>(st, epi, g) : launch_epi<WT, 4, false>(st, epi, g);
  return hipGetLastError();
}

template hipError_t launch_gemv<float>(hipStream_t, const float*, int, int, const float*, int, const float*,
                                       const float*, float, const float*, int, const float*, float*,
                                       const QkvStore<float>*);
template hipError_t launch_gemv<bf16_t>(hipStream_t, const float*, int, int, const bf16_t*, int, const float*,
                                        const float*, float, const float*, int, const float*, float*,
                                        const QkvStore<bf16_t>*);

}  // namespace fh
