// ops.hip -- the op-level ITensorBackend contract on device buffers.
//
// ITensorBackend (src/LLM.Core/Tensor/ITensorBackend.cs:18-266) is the
// reference's per-op plug-in seam: row-major fp32 tensors, explicit shapes,
// `accumulate` meaning +=, host index arrays uploaded per call.  These entry
// points implement every method of it (forward, backward, optimizer and the
// reductions) on device pointers, ordered on the context's stream; only the
// calls that return host values (the cross-entropy loss, the loss
// accumulation's end, the sums of squares) wait for the device.  The residency
// contract (InvalidateDeviceCache / EnsureHostCurrent) lives in the host
// mirror, which owns the device copies of its tensors.
//
// Elementwise kernels move 16 bytes to a load where the pointers allow it; rows of up to 1024 columns
// (softmax, LayerNorm, cross-entropy) stay in a wave's registers, of up to 32768 (cross-entropy) in
// a block's, wider ones take a block and several passes; column sums go by chunks of rows in a fixed
// order; the (batched) matmuls run on the split GEMM (gemm_split.hip), those of few k or of sizes
// past it on the tiled kernel here.  Results follow CpuBackend
// within the reference's own GPU-contract tolerances (GpuBackendTests.cs:23-24:
// 1e-4 forward, 1e-2 backward); the gathers, copies, masks and the embedding
// scatter-add (which adds each index's rows in ascending position, as the CPU
// loop does) are exact.
#include <math.h>
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "../../include/forge_hip.h"
#include "kernels.hpp"

namespace fh {

int set_error(int code, const char* msg);
hipStream_t context_stream(fh_context* c);
int context_device(fh_context* c);
int context_cus(fh_context* c);
struct OpsState;
OpsState*& context_ops(fh_context* c);

namespace {

constexpr int kT = 256;

__device__ __forceinline__ float ops_block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

__device__ __forceinline__ float ops_block_max(float v, float* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[w] = v;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// sum over a block of 256 in double (red: 256)
__device__ __forceinline__ double block_sum_double(double s, double* red) {
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  return red[0];
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

unsigned grid_for(size_t n) { return (unsigned)std::min<size_t>((n + kT - 1) / kT, 65536); }
unsigned grid_vec(size_t n, bool v4) { return grid_for(v4 ? (n + 3) / 4 : n); }

// ---- matmuls: y[s] (+)= op(a[s]) @ op(b[s]), 64x64 tiles, k steps of 16 ------------
// for few k, and for sizes that the split GEMM does not take (gemm_split_fits), with 64-bit offsets
// MODE 0 NN (a [M,K], b [K,N]), 1 NT (b [N,K]), 2 TN (a [K,M]).  Sums in S: the few products of
// fp32 elements are exact in double and hide behind the stores, so such a result is rounded once.
template <int MODE, typename S>
__global__ __launch_bounds__(256) void k_matmul(const float* __restrict__ a, const float* __restrict__ b,
                                                float* __restrict__ y, int M, int K, int N, int acc) {
  __shared__ float As[16][65];
  __shared__ float Bs[16][65];
  const int s = blockIdx.z;
  a += (size_t)s * M * K;
  b += (size_t)s * K * N;
  y += (size_t)s * M * N;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  S c[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
    for (int i = threadIdx.x; i < 1024; i += 256) {
      // A tile [16 k][64 m], B tile [16 k][64 n]
      int kk, mm;
      if (MODE == 2) {
        kk = i / 64, mm = i % 64;  // a[k][m]: m contiguous
      } else {
        mm = i / 16, kk = i % 16;  // a[m][k]: k contiguous
      }
      const int gm = m0 + mm, gk = k0 + kk;
      As[kk][mm] = (gm < M && gk < K) ? (MODE == 2 ? a[(size_t)gk * M + gm] : a[(size_t)gm * K + gk]) : 0.f;
      int kb, nn;
      if (MODE == 1) {
        nn = i / 16, kb = i % 16;  // b[n][k]
      } else {
        kb = i / 64, nn = i % 64;  // b[k][n]
      }
      const int gn = n0 + nn, gk2 = k0 + kb;
      Bs[kb][nn] = (gn < N && gk2 < K) ? (MODE == 1 ? b[(size_t)gn * K + gk2] : b[(size_t)gk2 * N + gn]) : 0.f;
    }
    __syncthreads();
    auto steps = [&](int from) {
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        S av[4], bv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) av[i] = As[from + kk][ty + 16 * i];
#pragma unroll
        for (int j = 0; j < 4; j++) bv[j] = Bs[from + kk][tx + 16 * j];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 4; j++) c[i][j] = fma(av[i], bv[j], c[i][j]);
      }
    };
    steps(0);
    if (sizeof(S) == 4 || k0 + 4 < K) steps(4);
    if (sizeof(S) == 4 || k0 + 8 < K) {
      steps(8);
      steps(12);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = m0 + ty + 16 * i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int n = n0 + tx + 16 * j;
      if (n >= N) continue;
      float& o = y[(size_t)m * N + n];
      o = acc ? o + (float)c[i][j] : (float)c[i][j];
    }
  }
}

// ---- head packing (PackHeads / UnpackHeads, CpuBackend.cs:225-262) ----------------
// HBM-bound copies.  A thread works within one (sequence, head) slot, so it divides by the head's
// width alone, and V (4 where widths, offsets and pointers are multiples of 16 bytes) floats move per
// load (48 slots of 331 x 64: 5.9 -> 3.4 us; three divisions per float before).  `wide` threads of
// a block share a slot, 256 / wide slots lie side by side: short slots (T of 1) fill a
// block too (16384 x 4 slots of 1 x 8: 4.4 us, a block to each 30).  blockIdx.z is one of up to three
// packed tensors whose columns follow each other (q, k and v in one launch: 4.9 us for three of 4 MB,
// 3.4 for one).  I: 64 bits where a slot or the slots are 2^31 or more.
struct PackSlices {
  float* packed[3];
};
template <int V, typename I>
__global__ __launch_bounds__(256) void k_pack_heads(float* __restrict__ wide_rows, int wide_cols, PackSlices slices,
                                                    I slots, int T, int H, int hd, int col_base, unsigned wide,
                                                    int unpack) {
  const unsigned per = hd / V, side = 256 / wide, ts = threadIdx.x / wide;
  if (ts >= side) return;
  const I n = (I)T * per;
  float* __restrict__ const packed = slices.packed[blockIdx.z];
  const int col = col_base + blockIdx.z * H * hd;
  for (I s = (I)blockIdx.y * side + ts; s < slots; s += (I)gridDim.y * side) {
    const I q = s / H, h = s % H;
    const size_t wide0 = (size_t)q * T * wide_cols + col + h * hd, packed0 = (size_t)s * T * hd;
    for (I i = (I)blockIdx.x * wide + (threadIdx.x - ts * wide); i < n; i += (I)gridDim.x * wide) {
      const I t = i / per, e = i % per * V;
      float* const pw = wide_rows + wide0 + (size_t)t * wide_cols + e;
      float* const pp = packed + packed0 + (size_t)i * V;
      if constexpr (V == 4) {
        if (unpack)
          *reinterpret_cast<float4*>(pw) = *reinterpret_cast<const float4*>(pp);
        else
          *reinterpret_cast<float4*>(pp) = *reinterpret_cast<const float4*>(pw);
      } else {
        if (unpack)
          *pw = *pp;
        else
          *pp = *pw;
      }
    }
  }
}

// ---- elementwise and row kernels -----------------------------------------------------
// Elementwise kernels: V floats (4 where the pointers, and for a bias its rows, are multiples of 16
// bytes) to a load, the last n % V by the first block's threads.
template <int V, typename F>
__device__ __forceinline__ void each_vec(size_t n, F f) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n / V; i += (size_t)gridDim.x * 256)
    f(i * V, std::integral_constant<int, V>());
  if (V > 1 && blockIdx.x == 0 && threadIdx.x < n % V) f(n - n % V + threadIdx.x, std::integral_constant<int, 1>());
}

template <int V>
struct Floats {
  float v[V];
  __device__ __forceinline__ void load(const float* p) {
    if constexpr (V == 4) {
      const float4 t = *reinterpret_cast<const float4*>(p);
      v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
    } else {
      v[0] = *p;
    }
  }
  __device__ __forceinline__ void store(float* p) const {
    if constexpr (V == 4)
      *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    else
      *p = v[0];
  }
};

// HBM-bound: a thread keeps V columns of the bias and walks down the rows, so no element divides by
// the row's width (2048 x 3072: 14.6 -> 8.8 us).  A block takes `wide` threads of a row and 256 / wide
// rows side by side (1048576 x 8: 7.6 us, one row to a block 92; x 1: 3.9 and 81).
template <int V>
__global__ __launch_bounds__(256) void k_add_bias(float* __restrict__ y, const float* __restrict__ bias,
                                                  unsigned rows, unsigned cols, unsigned wide) {
  const unsigned side = 256 / wide, tr = threadIdx.x / wide;
  const unsigned c = (blockIdx.x * wide + threadIdx.x - tr * wide) * V;
  if (c >= cols || tr >= side) return;
  Floats<V> b, t;
  b.load(bias + c);
#pragma unroll 4
  for (unsigned r = blockIdx.y * side + tr; r < rows; r += gridDim.y * side) {
    float* const p = y + (size_t)r * cols + c;
    t.load(p);
#pragma unroll
    for (int j = 0; j < V; j++) t.v[j] = t.v[j] + b.v[j];
    t.store(p);
  }
}

template <int V>
__global__ __launch_bounds__(256) void k_add_in_place(float* dst, const float* src, size_t n) {
  each_vec<V>(n, [&](size_t i, auto w) {
    Floats<decltype(w)::value> a, b;
    a.load(dst + i);
    b.load(src + i);
#pragma unroll
    for (int j = 0; j < decltype(w)::value; j++) a.v[j] = a.v[j] + b.v[j];
    a.store(dst + i);
  });
}

__global__ void k_scale(float* __restrict__ x, size_t n, float f) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    x[i] = x[i] * f;
}

__global__ void k_copy_block(const float* __restrict__ src, int src_cols, float* __restrict__ dst, int dst_cols,
                             int src_row, int src_col, int dst_row, int dst_col, int rows, int cols) {
  const size_t n = (size_t)rows * cols;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int r = (int)(i / cols), c = (int)(i % cols);
    dst[(size_t)(dst_row + r) * dst_cols + dst_col + c] = src[(size_t)(src_row + r) * src_cols + src_col + c];
  }
}

__global__ __launch_bounds__(256) void k_transpose_f32(const float* __restrict__ x, float* __restrict__ out, int rows,
                                                       int cols) {
  __shared__ float tile[32][33];
  const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int i = ty; i < 32; i += 8)
    if (r0 + i < rows && c0 + tx < cols) tile[i][tx] = x[(size_t)(r0 + i) * cols + c0 + tx];
  __syncthreads();
  for (int i = ty; i < 32; i += 8)
    if (c0 + i < cols && r0 + tx < rows) out[(size_t)(c0 + i) * rows + r0 + tx] = tile[tx][i];
}

// Column sums, HBM-bound: a block of four waves takes 64 columns of a chunk of rows, a
// lane one column; wave w adds rows w, w + 4, ... in order with 8 loads in flight, and the
// waves' sums add up in wave order.  The chunks are small enough to give every CU several
// blocks (2048 x 3072: one 256-row chunk per block and one load at a time took 60 us, this
// and the chunks' sum 10).  With one chunk the sums go straight into dst (dst[c] + sum),
// otherwise into part[chunk][c] for k_sum_chunks.
constexpr int kSumWaves = 4;
__global__ __launch_bounds__(64 * kSumWaves) void k_col_sums(const float* __restrict__ y, int rows, int cols,
                                                             int chunk_rows, float* __restrict__ dst,
                                                             float* __restrict__ part) {
  __shared__ float red[kSumWaves][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const int r0 = blockIdx.y * chunk_rows, r1 = min(rows, r0 + chunk_rows);
  float s = 0.f;
  if (c < cols) {
    int r = r0 + w;
    for (; r + 7 * kSumWaves < r1; r += 8 * kSumWaves) {
      float t[8];
#pragma unroll
      for (int i = 0; i < 8; i++) t[i] = y[(size_t)(r + i * kSumWaves) * cols + c];
#pragma unroll
      for (int i = 0; i < 8; i++) s += t[i];
    }
    for (; r < r1; r += kSumWaves) s += y[(size_t)r * cols + c];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w != 0 || c >= cols) return;
  for (int i = 1; i < kSumWaves; i++) s += red[i][lane];
  if (part)
    part[(size_t)blockIdx.y * cols + c] = s;
  else
    dst[c] = dst[c] + s;
}

// dst[k][c] += the sum of the chunks' part[chunk][k][c] for k < gridDim.y (dst0, dst1): 16
// waves take every 16th chunk each, 8 loads in flight, and add up in wave order.
constexpr int kChunkWaves = 16;
__global__ __launch_bounds__(64 * kChunkWaves) void k_sum_chunks(const float* __restrict__ part, int chunks, int cols,
                                                                 float* __restrict__ dst0, float* __restrict__ dst1) {
  __shared__ float red[kChunkWaves][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + lane;
  const size_t ld = (size_t)gridDim.y * cols;
  float s = 0.f;
  if (c < cols) {
    const float* p = part + (size_t)blockIdx.y * cols + c;
    int k = w;
    for (; k + 7 * kChunkWaves < chunks; k += 8 * kChunkWaves) {
      float t[8];
#pragma unroll
      for (int i = 0; i < 8; i++) t[i] = p[(size_t)(k + i * kChunkWaves) * ld];
#pragma unroll
      for (int i = 0; i < 8; i++) s += t[i];
    }
    for (; k < chunks; k += kChunkWaves) s += p[(size_t)k * ld];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w != 0 || c >= cols) return;
  for (int i = 1; i < kChunkWaves; i++) s += red[i][lane];
  float* dst = blockIdx.y ? dst1 : dst0;
  dst[c] = dst[c] + s;
}

// ---- LayerNorm (CpuBackend.cs:377-430), one block per row ------------------------------
__global__ __launch_bounds__(256) void k_ln_forward(const float* __restrict__ x, const float* __restrict__ w,
                                                    const float* __restrict__ b, float* __restrict__ out,
                                                    float* __restrict__ mean, float* __restrict__ rstd, int cols,
                                                    float eps) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const float* xr = x + (size_t)r * cols;
  float s = 0.f;
  for (int c = threadIdx.x; c < cols; c += 256) s += xr[c];
  const float mu = ops_block_sum(s, red) / (float)cols;
  float v = 0.f;
  for (int c = threadIdx.x; c < cols; c += 256) {
    const float dd = xr[c] - mu;
    v += dd * dd;
  }
  const float rs = 1.f / sqrtf(ops_block_sum(v, red) / (float)cols + eps);
  if (threadIdx.x == 0) {
    mean[r] = mu;
    rstd[r] = rs;
  }
  for (int c = threadIdx.x; c < cols; c += 256) out[(size_t)r * cols + c] = (xr[c] - mu) * rs * w[c] + b[c];
}

// The same for rows of at most 64 VPL columns: a wave keeps a row in registers (2048 x 768:
// 6.6 -> 4.4 us).
template <int VPL>
__global__ __launch_bounds__(256) void k_ln_forward_wave(const float* __restrict__ x, const float* __restrict__ w,
                                                         const float* __restrict__ b, float* __restrict__ out,
                                                         float* __restrict__ mean, float* __restrict__ rstd, int rows,
                                                         int cols, float eps) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const size_t at = (size_t)r * cols;
  float v[VPL], wc[VPL], bc[VPL], s = 0.f, q = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) v[i] = lane + 64 * i < cols ? x[at + lane + 64 * i] : 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    wc[i] = lane + 64 * i < cols ? w[lane + 64 * i] : 0.f;
    bc[i] = lane + 64 * i < cols ? b[lane + 64 * i] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < VPL; i++) s += v[i];
  const float mu = wave_sum_dpp(s) / (float)cols;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const float dd = lane + 64 * i < cols ? v[i] - mu : 0.f;
    q += dd * dd;
  }
  const float rs = 1.f / sqrtf(wave_sum_dpp(q) / (float)cols + eps);
  if (lane == 0) {
    mean[r] = mu;
    rstd[r] = rs;
  }
#pragma unroll
  for (int i = 0; i < VPL; i++)
    if (lane + 64 * i < cols) out[at + lane + 64 * i] = (v[i] - mu) * rs * wc[i] + bc[i];
}

// dx of every row and the column sums of dOut * xhat and dOut, reading dOut and x once: a
// wave keeps its row in registers (lane l: columns l, l + 64, ...; cols <= 64 VPL) and adds
// its rows' terms up per column; the block's waves add up in wave order into
// part[block][2][cols] (HBM-bound; 2048 x 768: 6 + 72 + 8 us for dx, the two column sums and
// their chunks, 8 + 4 this way).
template <int VPL>
__global__ __launch_bounds__(256) void k_ln_backward_rows(const float* __restrict__ dout, const float* __restrict__ x,
                                                          const float* __restrict__ w, const float* __restrict__ mean,
                                                          const float* __restrict__ rstd, float* __restrict__ dx,
                                                          int rows, int cols, int rows_per_block,
                                                          float* __restrict__ part) {
  __shared__ float red[4][64 * VPL];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r0 = blockIdx.x * rows_per_block, r1 = min(rows, r0 + rows_per_block);
  const float inv_n = 1.f / (float)cols;
  float wc[VPL], sw[VPL], sb[VPL];
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int c = lane + 64 * i;
    wc[i] = c < cols ? w[c] : 0.f;
    sw[i] = sb[i] = 0.f;
  }
  for (int r = r0 + wv; r < r1; r += 4) {
    const float* dr = dout + (size_t)r * cols;
    const float* xr = x + (size_t)r * cols;
    const float mu = mean[r], rs = rstd[r];
    float d[VPL], xh[VPL];
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      const int c = lane + 64 * i;
      d[i] = c < cols ? dr[c] : 0.f;
      xh[i] = c < cols ? xr[c] : 0.f;
    }
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      if (lane + 64 * i >= cols) continue;
      xh[i] = (xh[i] - mu) * rs;
      const float dxh = d[i] * wc[i];
      s1 += dxh;
      s2 += dxh * xh[i];
      sw[i] += d[i] * xh[i];
      sb[i] += d[i];
    }
    const float m1 = wave_sum_dpp(s1) * inv_n, m2 = wave_sum_dpp(s2) * inv_n;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      const int c = lane + 64 * i;
      if (c < cols) dx[(size_t)r * cols + c] = rs * (d[i] * wc[i] - m1 - xh[i] * m2);
    }
  }
#pragma unroll
  for (int k = 0; k < 2; k++) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < VPL; i++) red[wv][lane + 64 * i] = k ? sb[i] : sw[i];
    __syncthreads();
    for (int c = threadIdx.x; c < cols; c += 256)
      part[((size_t)blockIdx.x * 2 + k) * cols + c] = red[0][c] + red[1][c] + red[2][c] + red[3][c];
  }
}

// rows wider than the registers of a wave: dx by a block per row, the columns by chunks
__global__ __launch_bounds__(256) void k_ln_backward_dx(const float* __restrict__ dout, const float* __restrict__ x,
                                                        const float* __restrict__ w, const float* __restrict__ mean,
                                                        const float* __restrict__ rstd, float* __restrict__ dx,
                                                        int cols) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const float* dr = dout + (size_t)r * cols;
  const float* xr = x + (size_t)r * cols;
  const float mu = mean[r], rs = rstd[r];
  float s1 = 0.f, s2 = 0.f;
  for (int c = threadIdx.x; c < cols; c += 256) {
    const float xhat = (xr[c] - mu) * rs, dxhat = dr[c] * w[c];
    s1 += dxhat;
    s2 += dxhat * xhat;
  }
  const float inv_n = 1.f / (float)cols;
  const float m1 = ops_block_sum(s1, red) * inv_n;
  const float m2 = ops_block_sum(s2, red) * inv_n;
  for (int c = threadIdx.x; c < cols; c += 256) {
    const float xhat = (xr[c] - mu) * rs, dxhat = dr[c] * w[c];
    dx[(size_t)r * cols + c] = rs * (dxhat - m1 - xhat * m2);
  }
}

__global__ void k_ln_backward_cols(const float* __restrict__ dout, const float* __restrict__ x,
                                   const float* __restrict__ mean, const float* __restrict__ rstd, int rows, int cols,
                                   int chunk_rows, float* __restrict__ dw, float* __restrict__ db,
                                   float* __restrict__ part) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= cols) return;
  const int r0 = blockIdx.y * chunk_rows, r1 = min(rows, r0 + chunk_rows);
  float s = 0.f, s2 = 0.f;
#pragma unroll 4
  for (int r = r0; r < r1; r++) {
    const float d = dout[(size_t)r * cols + c];
    s += d * ((x[(size_t)r * cols + c] - mean[r]) * rstd[r]);
    s2 += d;
  }
  if (!part) {  // all rows in one chunk
    dw[c] = dw[c] + s;
    db[c] = db[c] + s2;
    return;
  }
  part[((size_t)blockIdx.y * 2) * cols + c] = s;
  part[((size_t)blockIdx.y * 2 + 1) * cols + c] = s2;
}

// ---- softmax (CpuBackend.cs:446-473; ITensorBackend.cs:117-130) ----------------------
// In place; with causal != 0 row r is query r % T of a packed [T,T] block: its
// keys past the query become -inf after the scale (Scale, CausalMask, Softmax).
__global__ __launch_bounds__(256) void k_softmax_rows(float* __restrict__ x, int cols, float scale, int causal) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  float* row = x + (size_t)r * cols;
  const int lim = causal ? r % cols : cols - 1;  // last unmasked column
  float mx = -INFINITY;
  for (int c = threadIdx.x; c <= lim; c += 256) mx = fmaxf(mx, row[c] * scale);
  mx = ops_block_max(mx, red);
  float s = 0.f;
  for (int c = threadIdx.x; c < cols; c += 256) {
    const float e = c <= lim ? expf(row[c] * scale - mx) : 0.f;
    row[c] = e;
    s += e;
  }
  const float inv = 1.f / ops_block_sum(s, red);
  for (int c = threadIdx.x; c < cols; c += 256) row[c] = row[c] * inv;
}

__global__ __launch_bounds__(256) void k_softmax_backward(const float* __restrict__ dout, const float* __restrict__ sm,
                                                          float* __restrict__ dx, int cols, float scale) {
  __shared__ float red[4];
  const int r = blockIdx.x;
  const float* dr = dout + (size_t)r * cols;
  const float* sr = sm + (size_t)r * cols;
  float d = 0.f;
  for (int c = threadIdx.x; c < cols; c += 256) d += dr[c] * sr[c];
  const float dot = ops_block_sum(d, red);
  for (int c = threadIdx.x; c < cols; c += 256) dx[(size_t)r * cols + c] = sr[c] * (dr[c] - dot) * scale;
}

// The same for rows of at most 64 VPL columns, HBM-bound: a wave keeps a row in registers
// (read once, written once) with all its loads in flight and needs no barrier (15888 rows of
// 331: forward 23.4 -> 10.5 us, backward 16.8 -> 10.7).
template <int VPL>
__global__ __launch_bounds__(256) void k_softmax_wave(float* __restrict__ x, int rows, int cols, float scale,
                                                      int causal) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  float* row = x + (size_t)r * cols;
  const int lim = causal ? r % cols : cols - 1;  // last unmasked column
  float v[VPL], mx = -INFINITY, s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) v[i] = lane + 64 * i <= lim ? row[lane + 64 * i] * scale : -INFINITY;
#pragma unroll
  for (int i = 0; i < VPL; i++) mx = fmaxf(mx, v[i]);
  mx = wave_max_dpp(mx);
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    v[i] = lane + 64 * i <= lim ? expf(v[i] - mx) : 0.f;
    s += v[i];
  }
  const float inv = 1.f / wave_sum_dpp(s);
#pragma unroll
  for (int i = 0; i < VPL; i++)
    if (lane + 64 * i < cols) row[lane + 64 * i] = v[i] * inv;
}

template <int VPL>
__global__ __launch_bounds__(256) void k_softmax_backward_wave(const float* __restrict__ dout,
                                                               const float* __restrict__ sm, float* __restrict__ dx,
                                                               int rows, int cols, float scale) {
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= rows) return;
  const size_t at = (size_t)r * cols;
  float d[VPL], p[VPL], s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int c = lane + 64 * i;
    d[i] = c < cols ? dout[at + c] : 0.f;
    p[i] = c < cols ? sm[at + c] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < VPL; i++)
    if (lane + 64 * i < cols) s += d[i] * p[i];
  const float dot = wave_sum_dpp(s);
#pragma unroll
  for (int i = 0; i < VPL; i++)
    if (lane + 64 * i < cols) dx[at + lane + 64 * i] = p[i] * (d[i] - dot) * scale;
}

// fn<VPL>(args) for the smallest VPL whose 64 VPL columns hold the row
#define ROW_WAVES(FN, cols, ...)        \
  do {                                  \
    if ((cols) <= 64)                   \
      FN<1> __VA_ARGS__;                \
    else if ((cols) <= 128)             \
      FN<2> __VA_ARGS__;                \
    else if ((cols) <= 256)             \
      FN<4> __VA_ARGS__;                \
    else if ((cols) <= 384)             \
      FN<6> __VA_ARGS__;                \
    else if ((cols) <= 512)             \
      FN<8> __VA_ARGS__;                \
    else if ((cols) <= 768)             \
      FN<12> __VA_ARGS__;               \
    else                                \
      FN<16> __VA_ARGS__;               \
  } while (0)
constexpr int kRowWaveCols = 1024;

// ---- GELU (CpuBackend.cs:477-514) ------------------------------------------------------
__device__ __forceinline__ float gelu_c() { return 0.7978845238685608f; }  // MathF.Sqrt(2f / MathF.PI)

// (1 + tanh u) / 2 is 1 / (1 + e^-2u): one exponential and a division where tanhf took both of its
// branches, and no cancellation where tanh u is near -1.  tanhf bound both kernels on the VALU; with 16
// bytes to a load they are HBM-bound (2048 x 3072: forward 13.3 -> 9.3 us, backward 18.8 -> 12.4).
__device__ __forceinline__ float gelu_gate(float v) {
  return 1.f / (1.f + expf(-2.f * (gelu_c() * (v + 0.044715f * v * v * v))));
}

template <int V>
__global__ __launch_bounds__(256) void k_gelu_forward(const float* x, float* out, size_t n) {
  each_vec<V>(n, [&](size_t i, auto w) {
    Floats<decltype(w)::value> a;
    a.load(x + i);
#pragma unroll
    for (int j = 0; j < decltype(w)::value; j++) a.v[j] = a.v[j] * gelu_gate(a.v[j]);
    a.store(out + i);
  });
}

template <int V>
__global__ __launch_bounds__(256) void k_gelu_backward(const float* dout, const float* x, float* dx, size_t n) {
  each_vec<V>(n, [&](size_t i, auto w) {
    Floats<decltype(w)::value> a, d;
    a.load(x + i);
    d.load(dout + i);
#pragma unroll
    for (int j = 0; j < decltype(w)::value; j++) {
      const float v = a.v[j], g = gelu_gate(v);
      const float du = gelu_c() * (1.f + 3.f * 0.044715f * v * v);
      d.v[j] = d.v[j] * (g + v * (2.f * g * (1.f - g)) * du);
    }
    d.store(dx + i);
  });
}

// ---- embedding (CpuBackend.cs:518-543) ----------------------------------------------------
__global__ void k_embedding_forward(const float* __restrict__ table, const int* __restrict__ idx,
                                    float* __restrict__ out, int D) {
  const int t = blockIdx.x;
  const float* src = table + (size_t)idx[t] * D;
  for (int c = threadIdx.x; c < D; c += blockDim.x) out[(size_t)t * D + c] = src[c];
}

// dTable[id] += dOut[t] for the positions t of each distinct id, in ascending order (the CPU
// loop's sums).  Block t works if no earlier position has its id: each thread compares a
// run of positions, a scan over the threads lists the later ones that match in LDS in order, and
// each thread adds up four columns at a time with 8 loads of each in flight (a text's commonest token
// comes up often: 80 of 2048 positions, one load at a time, took 15 us).  The ids are compared n^2
// times in all, 8 to a thread at n = 2048; up to kScatterIds positions that is less than sorting
// them on the host took.
constexpr int kScatterIds = 8192;
__global__ __launch_bounds__(256) void k_embedding_scatter(const float* __restrict__ dout, const int* __restrict__ idx,
                                                           int n, float* __restrict__ dtable, int D) {
  __shared__ int list[kScatterIds];
  __shared__ int counts[4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int id = idx[t];
  constexpr int R = kScatterIds / 256;
  const int run = (n + 255) / 256, j0 = tid * run, j1 = min(n, j0 + run);
  unsigned hits = 0;  // bit i: position j0 + i matches
#pragma unroll 8
  for (int i = 0; i < run; i++) hits |= (idx[min(j0 + i, n - 1)] == id && j0 + i < j1 ? 1u : 0u) << i;
  static_assert(R <= 32, "a run's matches fit a word");
  const unsigned before = t <= j0 ? 0u : t - j0 >= 32 ? ~0u : (1u << (t - j0)) - 1u;  // positions below t
  if (__syncthreads_or((hits & before) != 0)) return;
  const int cnt = __popc(hits);
  int incl = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  if (lane == 63) counts[w] = incl;
  __syncthreads();
  int at = incl - cnt, m = 0;
  for (int i = 0; i < 4; i++) {
    if (i < w) at += counts[i];
    m += counts[i];
  }
  for (unsigned h = hits; h; h &= h - 1) list[at++] = j0 + __ffs(h) - 1;
  __syncthreads();
  for (int c0 = 0; c0 < D; c0 += 1024) {
    float s[4];
    int c[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      c[u] = min(c0 + tid + 256 * u, D - 1);  // columns past D repeat the last one and are not stored
      s[u] = dtable[(size_t)id * D + c[u]];
    }
    int k = 0;
    for (; k + 8 <= m; k += 8) {
      float v[8][4];
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) v[i][u] = dout[(size_t)list[k + i] * D + c[u]];
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] = s[u] + v[i][u];
    }
    for (; k < m; k++)
#pragma unroll
      for (int u = 0; u < 4; u++) s[u] = s[u] + dout[(size_t)list[k] * D + c[u]];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (c0 + tid + 256 * u < D) dtable[(size_t)id * D + c[u]] = s[u];
  }
}

// The same for more positions, grouped on the host: uniq[u] is the id, pos[start[u] ..
// start[u+1]) its positions in order.
__global__ void k_embedding_backward(const float* __restrict__ dout, const int* __restrict__ uniq,
                                     const int* __restrict__ start, const int* __restrict__ pos,
                                     float* __restrict__ dtable, int D) {
  const int u = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= D) return;
  float* row = dtable + (size_t)uniq[u] * D;
  float s = row[c];
  for (int k = start[u]; k < start[u + 1]; k++) s = s + dout[(size_t)pos[k] * D + c];
  row[c] = s;
}

// ---- causal mask (CpuBackend.cs:551-557) ----------------------------------------------------
__global__ void k_causal_mask(float* __restrict__ s, size_t n, int T) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int j = (int)(i % T), q = (int)((i / T) % T);
    if (j > q) s[i] = -INFINITY;
  }
}

// ---- cross-entropy (CpuBackend.cs:594-644) --------------------------------------------------
// One block per position: probs (may alias logits) and the position's negative
// log-likelihood (0 when ignored).
__global__ __launch_bounds__(256) void k_ce_forward(const float* logits, const int* __restrict__ targets, float* probs,
                                                    int V, int ignore, float* __restrict__ nll) {
  __shared__ float red[4];
  const int t = blockIdx.x;
  const float* lr = logits + (size_t)t * V;
  float* pr = probs + (size_t)t * V;
  const int tg = targets[t];
  const bool ignored = tg == ignore;
  const float tl = ignored ? 0.f : lr[tg];
  float mx = -INFINITY;
  for (int v = threadIdx.x; v < V; v += 256) mx = fmaxf(mx, lr[v]);
  mx = ops_block_max(mx, red);  // every read of the row is done before the first write
  float s = 0.f;
  for (int v = threadIdx.x; v < V; v += 256) {
    const float e = expf(lr[v] - mx);
    pr[v] = e;
    s += e;
  }
  const float sum = ops_block_sum(s, red);
  const float inv = 1.f / sum;
  for (int v = threadIdx.x; v < V; v += 256) pr[v] = pr[v] * inv;
  if (threadIdx.x == 0) nll[t] = ignored ? 0.f : logf(sum) + mx - tl;
}

// The same for V <= 1024 PT: the row in the registers of 1024 threads, read once and
// written once, its loads all in flight (HBM-bound; 500 x 16257: 64 -> 15 us, where the block
// above reads or writes it five times).
template <int PT>
__global__ __launch_bounds__(1024) void k_ce_forward_row(const float* logits, const int* __restrict__ targets,
                                                         float* probs, int V, int ignore, float* __restrict__ nll) {
  __shared__ float red[2][16];
  const int t = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const float* lr = logits + (size_t)t * V;
  float* pr = probs + (size_t)t * V;
  const int tg = targets[t];
  const bool ignored = tg == ignore;
  const float tl = ignored ? 0.f : lr[tg];
  float v[PT], mx = -INFINITY, s = 0.f;
#pragma unroll
  for (int i = 0; i < PT; i++) {
    const int c = threadIdx.x + 1024 * i;
    v[i] = c < V ? lr[c] : -INFINITY;
  }
#pragma unroll
  for (int i = 0; i < PT; i++) mx = fmaxf(mx, v[i]);
  mx = wave_max_dpp(mx);
  if (lane == 0) red[0][w] = mx;
  __syncthreads();  // every read of the row is done before the first write
#pragma unroll
  for (int i = 0; i < 16; i++) mx = fmaxf(mx, red[0][i]);
#pragma unroll
  for (int i = 0; i < PT; i++) {
    v[i] = (int)threadIdx.x + 1024 * i < V ? expf(v[i] - mx) : 0.f;
    s += v[i];
  }
  s = wave_sum_dpp(s);
  if (lane == 0) red[1][w] = s;
  __syncthreads();
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i++) sum += red[1][i];
  const float inv = 1.f / sum;
#pragma unroll
  for (int i = 0; i < PT; i++) {
    const int c = threadIdx.x + 1024 * i;
    if (c < V) pr[c] = v[i] * inv;
  }
  if (threadIdx.x == 0) nll[t] = ignored ? 0.f : logf(sum) + mx - tl;
}

// The same for rows of at most 64 VPL columns: a wave to a row, no barrier (with the upload and the
// loss summed on the device, 65536 x 100: 103 us, 1024 threads to a row 323; 16000 x 300: 46 and 98).
template <int VPL>
__global__ __launch_bounds__(256) void k_ce_forward_wave(const float* logits, const int* __restrict__ targets,
                                                         float* probs, int T, int V, int ignore,
                                                         float* __restrict__ nll) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  const float* lr = logits + (size_t)t * V;
  float* pr = probs + (size_t)t * V;
  const int tg = targets[t];
  const bool ignored = tg == ignore;
  const float tl = ignored ? 0.f : lr[tg];
  float v[VPL], mx = -INFINITY, s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) v[i] = lane + 64 * i < V ? lr[lane + 64 * i] : -INFINITY;
#pragma unroll
  for (int i = 0; i < VPL; i++) mx = fmaxf(mx, v[i]);
  mx = wave_max_dpp(mx);
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    v[i] = lane + 64 * i < V ? expf(v[i] - mx) : 0.f;
    s += v[i];
  }
  const float sum = wave_sum_dpp(s), inv = 1.f / sum;
#pragma unroll
  for (int i = 0; i < VPL; i++)
    if (lane + 64 * i < V) pr[lane + 64 * i] = v[i] * inv;
  if (lane == 0) nll[t] = ignored ? 0.f : logf(sum) + mx - tl;
}

// acc (double, device) += sum of the T per-position terms, by one block in double (fixed order)
__global__ __launch_bounds__(256) void k_ce_accumulate(const float* __restrict__ nll, int T, double* __restrict__ acc) {
  __shared__ double red[256];
  double s = 0;
  for (int t = threadIdx.x; t < T; t += 256) s += (double)nll[t];
  s = block_sum_double(s, red);
  if (threadIdx.x == 0) acc[0] += s;
}

// HBM-bound: a block takes kCeCols columns of a position (blockIdx.x; blockIdx.y its part of
// the vocabulary), so no element divides by V and 8 loads per thread are in flight (500 x
// 16257: 21 -> 13 us).
constexpr unsigned kCeCols = 2048;
__global__ __launch_bounds__(256) void k_ce_backward(const float* probs, const int* __restrict__ targets, float* dl,
                                                     unsigned T, unsigned V, int ignore, float scale) {
  for (unsigned t = blockIdx.x; t < T; t += gridDim.x) {
    const int tg = targets[t];
    const size_t at = (size_t)t * V;
    for (unsigned c0 = blockIdx.y * kCeCols; c0 < V; c0 += gridDim.y * kCeCols) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const unsigned c = c0 + threadIdx.x + 256 * i;
        p[i] = tg != ignore && c < V ? probs[at + c] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const unsigned c = c0 + threadIdx.x + 256 * i;
        float g = p[i] * scale;
        if (tg == ignore)
          g = 0.f;
        else if ((int)c == tg)
          g = g - scale;
        if (c < V) dl[at + c] = g;
      }
    }
  }
}

// The same for V <= kCeFlat: a block takes kCeFlatPer elements of the positions one after the other,
// with a 32-bit division per element (with the targets' upload, 262144 x 10: 117 us, a block to each
// position 165; 65536 x 100: 40 and 59; 8000 x 600: 26.7 and 28.1; 4096 x 1024: 11.9 and 11.3).
constexpr int kCeFlat = 768, kCeFlatPer = 2048;
__global__ __launch_bounds__(256) void k_ce_backward_flat(const float* probs, const int* __restrict__ targets, float* dl,
                                                          size_t n, int V, int ignore, float scale) {
  const size_t base = (size_t)blockIdx.x * kCeFlatPer, t0 = base / V;
  const unsigned c0 = (unsigned)(base - t0 * V), left = (unsigned)min((size_t)kCeFlatPer, n - base);
  float p[8];
  int tg[8];
  unsigned c[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const unsigned j = min(threadIdx.x + 256u * i, left - 1), t = (c0 + j) / V;
    c[i] = c0 + j - t * V;
    tg[i] = targets[t0 + t];
    p[i] = probs[base + j];
  }
#pragma unroll
  for (int i = 0; i < 8; i++) {
    float g = p[i] * scale;
    if (tg[i] == ignore)
      g = 0.f;
    else if ((int)c[i] == tg[i])
      g = g - scale;
    if (threadIdx.x + 256u * i < left) dl[base + threadIdx.x + 256u * i] = g;
  }
}

// ---- sums of squares and AdamW (ITensorBackend.cs:214-265) ---------------------------------
// Sum x^2 of up to kSumsqTensors tensors in one launch: block j of a tensor's blocks adds
// elements j, j + its blocks, ... (in strides of 256) in double, the block's threads add up
// in a fixed tree, and k_sum_doubles adds the blocks' sums.  HBM-bound; a launch per tensor
// and a sum by one thread took 141 + 94 us for 20.5M elements in 16 tensors.
constexpr int kSumsqTensors = 64;
constexpr int kSumsqPerBlock = 8192;  // elements that a tensor gets a block for, up to kSumsqBlocks
constexpr int kSumsqBlocks = 512;
struct SumsqList {
  const float* x[kSumsqTensors];
  long long n[kSumsqTensors];
  int first[kSumsqTensors + 1];  // first block of each tensor
  int count;
};
__global__ __launch_bounds__(256) void k_sumsq(SumsqList l, double* __restrict__ part) {
  __shared__ double red[256];
  int t = 0;
  while (t + 1 < l.count && (int)blockIdx.x >= l.first[t + 1]) t++;
  const float* x = l.x[t];
  const size_t n = (size_t)l.n[t], step = (size_t)(l.first[t + 1] - l.first[t]) * 256;
  double s = 0;
  size_t i = (size_t)(blockIdx.x - l.first[t]) * 256 + threadIdx.x;
  for (; i + 7 * step < n; i += 8 * step) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = x[i + k * step];
#pragma unroll
    for (int k = 0; k < 8; k++) s += (double)v[k] * v[k];
  }
  for (; i < n; i += step) s += (double)x[i] * x[i];
  s = block_sum_double(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// out[0] = sum of part[0 .. n) by one block (fixed order)
__global__ __launch_bounds__(256) void k_sum_doubles(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double red[256];
  double s = 0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  s = block_sum_double(s, red);
  if (threadIdx.x == 0) out[0] = s;
}

// HBM-bound: 16 bytes read and 12 written per element, V (4 where the pointers are multiples of
// 16 bytes, the last n % 4 by one) to a load.  The moments stream past the caches: nothing reads them
// before the next update.  The gradients come from the norm or the backward before and the weights
// go to the next forward, so they stay cached (us per training step of forward, backward, norm and
// update, all streaming / none / the moments: d 256, 6 layers 1282 / 1260 / 1237; d 512, 8 layers 2804 /
// 2797 / 2768; d 768, 2 layers 1496 / 1518 / 1486; d 768, 12 layers 6951 / 7058 / 6970).
template <int V>
__global__ __launch_bounds__(256) void k_adamw(float* __restrict__ w, const float* __restrict__ g,
                                               float* __restrict__ m, float* __restrict__ v, size_t n, float lr,
                                               float b1, float b2, float eps, float wd, float bc1, float bc2,
                                               int decay) {
  auto step = [&](float gi, float& mi, float& vi, float& wi) {
    mi = b1 * mi + (1.f - b1) * gi;
    vi = b2 * vi + (1.f - b2) * gi * gi;
    if (decay) wi = wi - lr * wd * wi;
    const float mh = mi / bc1, vh = vi / bc2;
    wi = wi - lr * mh / (sqrtf(vh) + eps);
  };
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n / V; i += (size_t)gridDim.x * 256) {
    if constexpr (V == 4) {
      typedef float f4 __attribute__((ext_vector_type(4)));
      const f4 gv = reinterpret_cast<const f4*>(g)[i];
      f4 mv = __builtin_nontemporal_load(reinterpret_cast<f4*>(m) + i);
      f4 vv = __builtin_nontemporal_load(reinterpret_cast<f4*>(v) + i);
      f4 wv = reinterpret_cast<f4*>(w)[i];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float a = mv[j], b = vv[j], c = wv[j];
        step(gv[j], a, b, c);
        mv[j] = a, vv[j] = b, wv[j] = c;
      }
      __builtin_nontemporal_store(mv, reinterpret_cast<f4*>(m) + i);
      __builtin_nontemporal_store(vv, reinterpret_cast<f4*>(v) + i);
      reinterpret_cast<f4*>(w)[i] = wv;
    } else {
      step(g[i], m[i], v[i], w[i]);
    }
  }
  if (V > 1 && blockIdx.x == 0 && threadIdx.x < n % V) {
    const size_t i = n - n % V + threadIdx.x;
    step(g[i], m[i], v[i], w[i]);
  }
}

}  // namespace

constexpr int kStages = 8;
constexpr size_t kStageBytes = (size_t)1 << 16;  // 16384 indices; larger arrays are copied with a wait

// Per-context state of the op entry points: device scratch for uploaded index
// arrays and reduction partials, and the loss accumulation.
struct OpsState {
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  // pinned host memory that uploads leave from, so that a call returns without waiting for
  // its copy: kStages areas in turn, each with an event that says its last copy is done
  char* stage = nullptr;
  hipEvent_t stage_done[kStages] = {};
  int stage_next = 0;
  double* acc = nullptr;  // device loss accumulator + a result slot
  bool accumulating = false;
  long long accumulated_targets = 0;
};

void ops_state_free(OpsState* o) {
  if (!o) return;
  if (o->scratch) (void)hipFree(o->scratch);
  if (o->acc) (void)hipFree(o->acc);
  for (hipEvent_t e : o->stage_done)
    if (e) (void)hipEventDestroy(e);
  if (o->stage) (void)hipHostFree(o->stage);
  delete o;
}

}  // namespace fh

using namespace fh;

namespace {

int set_err(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  return set_error(code, buf);
}

#define HIP_TRY(expr)                                                                                         \
  do {                                                                                                        \
    hipError_t e_ = (expr);                                                                                   \
    if (e_ != hipSuccess)                                                                                     \
      return set_err(e_ == hipErrorOutOfMemory ? FH_ERR_OOM : FH_ERR_HIP, "%s failed: %s", #expr,            \
                     hipGetErrorString(e_));                                                                  \
  } while (0)

#define FH_TRY(expr)            \
  do {                          \
    int r_ = (expr);            \
    if (r_ != FH_OK) return r_; \
  } while (0)

int ops_begin(fh_context* c, OpsState** out) {
  if (!c) return set_err(FH_ERR_INVALID, "null context");
  HIP_TRY(hipSetDevice(context_device(c)));
  OpsState*& o = context_ops(c);
  if (!o) {
    o = new OpsState();
    if (hipMalloc(&o->acc, 2 * sizeof(double)) != hipSuccess) {
      delete o;
      o = nullptr;
      return set_err(FH_ERR_OOM, "allocating the loss accumulator failed");
    }
  }
  *out = o;
  return FH_OK;
}

// device scratch of at least `bytes` (the previous contents are not kept)
int ops_scratch(fh_context* c, OpsState* o, size_t bytes, void** p) {
  if (bytes > o->scratch_bytes) {
    HIP_TRY(hipStreamSynchronize(context_stream(c)));  // earlier kernels may still read the old scratch
    if (o->scratch) (void)hipFree(o->scratch);
    o->scratch = nullptr;
    o->scratch_bytes = 0;
    const size_t nb = std::max<size_t>(bytes, 1 << 16);
    if (hipMalloc(&o->scratch, nb) != hipSuccess) {
      o->scratch = nullptr;
      (void)hipGetLastError();  // the next launch's check is its own
      return set_err(FH_ERR_OOM, "allocating %zu bytes of scratch", nb);
    }
    o->scratch_bytes = nb;
  }
  *p = o->scratch;
  return FH_OK;
}

int op_launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_err(FH_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  return FH_OK;
}

#define OPS_PROLOGUE(c)    \
  OpsState* ops_ = nullptr; \
  FH_TRY(ops_begin((c), &ops_));                \
  hipStream_t st_ = context_stream(c);          \
  (void)ops_;                                   \
  (void)st_

#define OPS_ARG(cond, ...) \
  if (!(cond)) return set_err(FH_ERR_INVALID, __VA_ARGS__)

// Host ints to dev on the context's stream; the host array may go away on return.  It is
// copied into the next staging area (16 KB of targets or ids in a microsecond), whose event
// bounds how far the host runs ahead: waiting for each copy cost a training step 20-30 us per
// upload with the device idle.
int copy_ints(fh_context* c, OpsState* o, const int32_t* host, size_t n, int* dev) {
  hipStream_t st = context_stream(c);
  const size_t bytes = n * sizeof(int32_t);
  if (bytes > kStageBytes) {
    HIP_TRY(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, st));
    HIP_TRY(hipStreamSynchronize(st));
    return FH_OK;
  }
  if (!o->stage) {
    void* p = nullptr;
    HIP_TRY(hipHostMalloc(&p, kStages * kStageBytes, hipHostMallocDefault));
    o->stage = static_cast<char*>(p);
  }
  const int k = o->stage_next;
  if (o->stage_done[k])
    HIP_TRY(hipEventSynchronize(o->stage_done[k]));
  else
    HIP_TRY(hipEventCreateWithFlags(&o->stage_done[k], hipEventDisableTiming));
  char* from = o->stage + k * kStageBytes;
  std::memcpy(from, host, bytes);
  HIP_TRY(hipMemcpyAsync(dev, from, bytes, hipMemcpyHostToDevice, st));
  HIP_TRY(hipEventRecord(o->stage_done[k], st));
  o->stage_next = (k + 1) % kStages;
  return FH_OK;
}

int upload_ints(fh_context* c, OpsState* o, const int32_t* host, size_t n, int** dev) {
  void* p = nullptr;
  FH_TRY(ops_scratch(c, o, n * sizeof(int32_t), &p));
  *dev = static_cast<int*>(p);
  return copy_ints(c, o, host, n, *dev);
}

// the partial sums of a split K take at most this much of the context's scratch (64 MB)
constexpr size_t kSplitPartFloats = (size_t)16 << 20;

int matmul_common(fh_context* c, int mode, const void* a, const void* b, void* y, int slots, int M, int K, int N,
                  int acc) {
  OPS_PROLOGUE(c);
  OPS_ARG(a && b && y, "null buffer");
  OPS_ARG(slots > 0 && slots <= 65535 && M > 0 && K > 0 && N > 0, "slots (at most 65535), M, K and N must be positive");
  // Few k: the split GEMM's stage of 32 is mostly padding, and its results at K 1 are not all rounded
  // right.  Where y is added to, its wider tiles make up for that unless y is small (us, this kernel and
  // the split GEMM: 4096 x 1 x 4096 15.1 and 19.4, K 8 18.6 and 19.3, K 12 24 and 19.5; 65535 slots of
  // 8 x 8 x 8 134 and 200; adding to 48 slots of 331 x 8 x 331 17 and 11).
  const bool few = M < 1 << 22 && (K == 1 || (K <= 8 && (!acc || (size_t)M * N <= 1024)));
  if (!few && gemm_split_fits(slots, M, K, N)) {
    const int cus = context_cus(c);
    size_t pf = gemm_split_part_floats(slots, M, K, N, kSplitPartFloats, cus);
    void* part = nullptr;
    // a full device: K in one piece, which needs no scratch
    if (pf && ops_scratch(c, ops_, pf * sizeof(float), &part) != FH_OK) {
      part = nullptr;
      pf = 0;
    }
    HIP_TRY(launch_gemm_split(st_, mode, static_cast<const float*>(a), static_cast<const float*>(b), slots, M, K, N,
                              nullptr, 0, acc ? static_cast<const float*>(y) : nullptr, static_cast<float*>(y),
                              static_cast<float*>(part), pf, cus));
    return FH_OK;
  }
  dim3 grid((N + 63) / 64, (M + 63) / 64, slots);
  const float* fa = static_cast<const float*>(a);
  const float* fb = static_cast<const float*>(b);
  float* fy = static_cast<float*>(y);
  if (mode == 0)
    hipLaunchKernelGGL((few ? k_matmul<0, double> : k_matmul<0, float>), grid, dim3(256), 0, st_, fa, fb, fy, M, K, N,
                       acc);
  else if (mode == 1)
    hipLaunchKernelGGL((few ? k_matmul<1, double> : k_matmul<1, float>), grid, dim3(256), 0, st_, fa, fb, fy, M, K, N,
                       acc);
  else
    hipLaunchKernelGGL((few ? k_matmul<2, double> : k_matmul<2, float>), grid, dim3(256), 0, st_, fa, fb, fy, M, K, N,
                       acc);
  return op_launched("matmul");
}

// `count` packed tensors of slots * T * hd floats each, from (unpack: into) columns that follow each
// other in the wide rows
int launch_pack(hipStream_t st, float* wide, int wide_cols, const PackSlices& p, int count, int batch, int T, int H,
                int hd, int col_base, int unpack) {
  bool v4 = hd % 4 == 0 && wide_cols % 4 == 0 && col_base % 4 == 0 && aligned16(wide);
  for (int i = 0; i < count; i++) v4 = v4 && aligned16(p.packed[i]);
  const size_t n = (size_t)T * (hd / (v4 ? 4 : 1)), slots = (size_t)batch * H;
  const unsigned slot_threads = (unsigned)std::min<size_t>(n, 256), side = 256 / slot_threads;
  const dim3 grid((unsigned)std::min<size_t>((n + 255) / 256, 65535),
                  (unsigned)std::min<size_t>((slots + side - 1) / side, 65535), count);
  auto launch = [&](auto kernel, auto typed_slots) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, wide, wide_cols, p, typed_slots, T, H, hd, col_base,
                       slot_threads, unpack);
  };
  if (std::max(n, slots) < (size_t)1 << 31)
    launch(v4 ? k_pack_heads<4, unsigned> : k_pack_heads<1, unsigned>, (unsigned)slots);
  else
    launch(v4 ? k_pack_heads<4, size_t> : k_pack_heads<1, size_t>, slots);
  return op_launched(unpack ? "unpack heads" : "pack heads");
}

int softmax_common(fh_context* c, void* x, int rows, int cols, float scale, int causal) {
  OPS_PROLOGUE(c);
  OPS_ARG(x, "null buffer");
  OPS_ARG(rows > 0 && cols > 0, "rows and cols must be positive");
  float* fx = static_cast<float*>(x);
  if (cols <= kRowWaveCols)
    ROW_WAVES(k_softmax_wave, cols, <<<dim3((rows + 3) / 4), dim3(256), 0, st_>>>(fx, rows, cols, scale, causal));
  else
    hipLaunchKernelGGL(k_softmax_rows, dim3(rows), dim3(256), 0, st_, fx, cols, scale, causal);
  return op_launched("softmax");
}

}  // namespace

extern "C" {

int fh_op_matmul_nn(fh_context* c, const void* a, const void* b, void* y, int slots, int M, int K, int N, int acc) {
  return matmul_common(c, 0, a, b, y, slots, M, K, N, acc);
}
int fh_op_matmul_nt(fh_context* c, const void* a, const void* b, void* y, int slots, int M, int K, int N, int acc) {
  return matmul_common(c, 1, a, b, y, slots, M, K, N, acc);
}
int fh_op_matmul_tn(fh_context* c, const void* a, const void* b, void* y, int slots, int M, int K, int N, int acc) {
  return matmul_common(c, 2, a, b, y, slots, M, K, N, acc);
}

int fh_op_pack_heads(fh_context* c, const void* src, int src_cols, void* dst, int batch, int T, int n_heads,
                     int head_dim, int col_base) {
  OPS_PROLOGUE(c);
  OPS_ARG(src && dst, "null buffer");
  OPS_ARG(batch > 0 && T > 0 && n_heads > 0 && head_dim > 0 && col_base >= 0 &&
              col_base + n_heads * head_dim <= src_cols,
          "head slices outside the source rows");
  return launch_pack(st_, static_cast<float*>(const_cast<void*>(src)), src_cols, PackSlices{{static_cast<float*>(dst)}},
                     1, batch, T, n_heads, head_dim, col_base, 0);
}

int fh_op_unpack_heads(fh_context* c, const void* src, void* dst, int dst_cols, int batch, int T, int n_heads,
                       int head_dim, int col_base) {
  OPS_PROLOGUE(c);
  OPS_ARG(src && dst, "null buffer");
  OPS_ARG(batch > 0 && T > 0 && n_heads > 0 && head_dim > 0 && col_base >= 0 &&
              col_base + n_heads * head_dim <= dst_cols,
          "head slices outside the destination rows");
  return launch_pack(st_, static_cast<float*>(dst), dst_cols,
                     PackSlices{{static_cast<float*>(const_cast<void*>(src))}}, 1, batch, T, n_heads, head_dim,
                     col_base, 1);
}

int fh_op_pack_qkv_heads(fh_context* c, const void* src, int src_cols, void* q, void* k, void* v, int batch, int T,
                         int n_heads, int head_dim) {
  OPS_PROLOGUE(c);
  OPS_ARG(src && q && k && v, "null buffer");
  OPS_ARG(batch > 0 && T > 0 && n_heads > 0 && head_dim > 0 && 3ll * n_heads * head_dim <= src_cols,
          "head slices outside the source rows");
  return launch_pack(st_, static_cast<float*>(const_cast<void*>(src)), src_cols,
                     PackSlices{{static_cast<float*>(q), static_cast<float*>(k), static_cast<float*>(v)}}, 3, batch, T,
                     n_heads, head_dim, 0, 0);
}

int fh_op_unpack_qkv_heads(fh_context* c, const void* q, const void* k, const void* v, void* dst, int dst_cols,
                           int batch, int T, int n_heads, int head_dim) {
  OPS_PROLOGUE(c);
  OPS_ARG(q && k && v && dst, "null buffer");
  OPS_ARG(batch > 0 && T > 0 && n_heads > 0 && head_dim > 0 && 3ll * n_heads * head_dim <= dst_cols,
          "head slices outside the destination rows");
  auto f = [](const void* p) { return static_cast<float*>(const_cast<void*>(p)); };
  return launch_pack(st_, static_cast<float*>(dst), dst_cols, PackSlices{{f(q), f(k), f(v)}}, 3, batch, T, n_heads,
                     head_dim, 0, 1);
}

int fh_op_add_bias(fh_context* c, void* y, const void* bias, int rows, int cols) {
  OPS_PROLOGUE(c);
  OPS_ARG(y && bias && rows > 0 && cols > 0, "bad arguments");
  const bool v4 = cols % 4 == 0 && aligned16(y) && aligned16(bias);
  const int per_row = cols / (v4 ? 4 : 1), wide = std::min(per_row, 256), side = 256 / wide;
  const int strips = (per_row + wide - 1) / wide;
  // about 4096 blocks, so that a long column has several rows to a thread
  const dim3 grid(strips, std::min({rows / side + (rows % side != 0), (4096 + strips - 1) / strips, 65535}));
  hipLaunchKernelGGL(v4 ? k_add_bias<4> : k_add_bias<1>, grid, dim3(256), 0, st_, static_cast<float*>(y),
                     static_cast<const float*>(bias), (unsigned)rows, (unsigned)cols, (unsigned)wide);
  return op_launched("add bias");
}

int fh_op_sum_rows(fh_context* c, const void* dy, void* dbias, int rows, int cols) {
  OPS_PROLOGUE(c);
  OPS_ARG(dy && dbias && rows > 0 && cols > 0, "bad arguments");
  // chunks of at least 32 rows (64 when that is all of them) until there are about 1024 blocks
  const int strips = (cols + 63) / 64;
  const int want = std::max(1, std::min((rows + 31) / 32, (1024 + strips - 1) / strips));
  const int chunk_rows = rows <= 64 ? rows : (rows + want - 1) / want;
  const int chunks = (rows + chunk_rows - 1) / chunk_rows;
  float* part = nullptr;
  if (chunks > 1) {
    void* p = nullptr;
    FH_TRY(ops_scratch(c, ops_, (size_t)chunks * cols * sizeof(float), &p));
    part = static_cast<float*>(p);
  }
  hipLaunchKernelGGL(k_col_sums, dim3(strips, chunks), dim3(64 * kSumWaves), 0, st_, static_cast<const float*>(dy),
                     rows, cols, chunk_rows, static_cast<float*>(dbias), part);
  if (chunks > 1)
    hipLaunchKernelGGL(k_sum_chunks, dim3(strips), dim3(64 * kChunkWaves), 0, st_, part, chunks, cols,
                       static_cast<float*>(dbias), nullptr);
  return op_launched("sum rows");
}

int fh_op_add_in_place(fh_context* c, void* dst, const void* src, int64_t n) {
  OPS_PROLOGUE(c);
  OPS_ARG(dst && src && n > 0, "bad arguments");
  const bool v4 = aligned16(dst) && aligned16(src);
  hipLaunchKernelGGL(v4 ? k_add_in_place<4> : k_add_in_place<1>, dim3(grid_vec((size_t)n, v4)), dim3(256), 0, st_,
                     static_cast<float*>(dst),
                     static_cast<const float*>(src), (size_t)n);
  return op_launched("add in place");
}

int fh_op_copy(fh_context* c, const void* src, void* dst, int64_t n) {
  OPS_PROLOGUE(c);
  OPS_ARG(dst && src && n >= 0, "bad arguments");
  if (n > 0) HIP_TRY(hipMemcpyAsync(dst, src, (size_t)n * sizeof(float), hipMemcpyDeviceToDevice, st_));
  return FH_OK;
}

int fh_op_copy_block(fh_context* c, const void* src, int src_cols, void* dst, int dst_cols, int src_row, int src_col,
                     int dst_row, int dst_col, int rows, int cols) {
  OPS_PROLOGUE(c);
  OPS_ARG(src && dst && rows >= 0 && cols >= 0 && src_row >= 0 && src_col >= 0 && dst_row >= 0 && dst_col >= 0 &&
              src_col + cols <= src_cols && dst_col + cols <= dst_cols,
          "block outside the source or destination rows");
  const size_t n = (size_t)rows * cols;
  if (n == 0) return FH_OK;
  hipLaunchKernelGGL(k_copy_block, dim3(grid_for(n)), dim3(kT), 0, st_, static_cast<const float*>(src), src_cols,
                     static_cast<float*>(dst), dst_cols, src_row, src_col, dst_row, dst_col, rows, cols);
  return op_launched("copy block");
}

int fh_op_scale(fh_context* c, void* x, int64_t n, float factor) {
  OPS_PROLOGUE(c);
  OPS_ARG(x && n > 0, "bad arguments");
  hipLaunchKernelGGL(k_scale, dim3(grid_for((size_t)n)), dim3(kT), 0, st_, static_cast<float*>(x), (size_t)n, factor);
  return op_launched("scale");
}

int fh_op_transpose(fh_context* c, const void* x, void* out, int rows, int cols) {
  OPS_PROLOGUE(c);
  OPS_ARG(x && out && rows > 0 && cols > 0, "bad arguments");
  hipLaunchKernelGGL(k_transpose_f32, dim3((cols + 31) / 32, (rows + 31) / 32), dim3(256), 0, st_,
                     static_cast<const float*>(x), static_cast<float*>(out), rows, cols);
  return op_launched("transpose");
}

int fh_op_layernorm_forward(fh_context* c, const void* x, const void* w, const void* b, void* out, void* mean,
                            void* rstd, int rows, int cols, float eps) {
  OPS_PROLOGUE(c);
  OPS_ARG(x && w && b && out && mean && rstd && rows > 0 && cols > 0, "bad arguments");
  const float *fx = static_cast<const float*>(x), *fw = static_cast<const float*>(w), *fb = static_cast<const float*>(b);
  float *fo = static_cast<float*>(out), *fm = static_cast<float*>(mean), *fr = static_cast<float*>(rstd);
  if (cols <= kRowWaveCols)
    ROW_WAVES(k_ln_forward_wave, cols,
              <<<dim3((rows + 3) / 4), dim3(256), 0, st_>>>(fx, fw, fb, fo, fm, fr, rows, cols, eps));
  else
    hipLaunchKernelGGL(k_ln_forward, dim3(rows), dim3(256), 0, st_, fx, fw, fb, fo, fm, fr, cols, eps);
  return op_launched("layernorm forward");
}

int fh_op_layernorm_backward(fh_context* c, const void* dout, const void* x, const void* w, const void* mean,
                             const void* rstd, void* dx, void* dw, void* db, int rows, int cols) {
  OPS_PROLOGUE(c);
  OPS_ARG(dout && x && w && mean && rstd && dx && dw && db && rows > 0 && cols > 0, "bad arguments");
  const float *fd = static_cast<const float*>(dout), *fx = static_cast<const float*>(x);
  const float *fm = static_cast<const float*>(mean), *fr = static_cast<const float*>(rstd);
  // part[chunk][2][cols] of dW and dB: four rows a block (one a wave), more past 512 blocks
  const bool wide = cols > kRowWaveCols;
  const int per = wide ? std::max(32, (rows + 127) / 128) : std::max(4, ((rows + 511) / 512 + 3) / 4 * 4);
  const int chunks = (rows + per - 1) / per;
  void* p = nullptr;
  if (!wide || chunks > 1) FH_TRY(ops_scratch(c, ops_, (size_t)2 * chunks * cols * sizeof(float), &p));
  float* part = static_cast<float*>(p);
  const float* fw = static_cast<const float*>(w);
  float *fdx = static_cast<float*>(dx), *fdw = static_cast<float*>(dw), *fdb = static_cast<float*>(db);
  if (wide) {
    hipLaunchKernelGGL(k_ln_backward_dx, dim3(rows), dim3(256), 0, st_, fd, fx, fw, fm, fr, fdx, cols);
    hipLaunchKernelGGL(k_ln_backward_cols, dim3((cols + 255) / 256, chunks), dim3(256), 0, st_, fd, fx, fm, fr, rows,
                       cols, per, fdw, fdb, part);
  } else {
    ROW_WAVES(k_ln_backward_rows, cols,
              <<<dim3(chunks), dim3(256), 0, st_>>>(fd, fx, fw, fm, fr, fdx, rows, cols, per, part));
  }
  if (part)
    hipLaunchKernelGGL(k_sum_chunks, dim3((cols + 63) / 64, 2), dim3(64 * kChunkWaves), 0, st_, part, chunks, cols, fdw,
                       fdb);
  return op_launched("layernorm backward");
}

int fh_op_softmax_forward(fh_context* c, void* x, int rows, int cols) { return softmax_common(c, x, rows, cols, 1.f, 0); }

int fh_op_scaled_causal_softmax_forward(fh_context* c, void* scores, int rows, int T, float scale) {
  return softmax_common(c, scores, rows, T, scale, 1);
}

int fh_op_softmax_backward(fh_context* c, const void* dout, const void* sm, void* dx, int rows, int cols, float scale) {
  OPS_PROLOGUE(c);
  OPS_ARG(dout && sm && dx && rows > 0 && cols > 0, "bad arguments");
  const float *fd = static_cast<const float*>(dout), *fs = static_cast<const float*>(sm);
  float* fx = static_cast<float*>(dx);
  if (cols <= kRowWaveCols)
    ROW_WAVES(k_softmax_backward_wave, cols,
              <<<dim3((rows + 3) / 4), dim3(256), 0, st_>>>(fd, fs, fx, rows, cols, scale));
  else
    hipLaunchKernelGGL(k_softmax_backward, dim3(rows), dim3(256), 0, st_, fd, fs, fx, cols, scale);
  return op_launched("softmax backward");
}

int fh_op_gelu_forward(fh_context* c, const void* x, void* out, int64_t n) {
  OPS_PROLOGUE(c);
  OPS_ARG(x && out && n > 0, "bad arguments");
  const bool v4 = aligned16(x) && aligned16(out);
  hipLaunchKernelGGL(v4 ? k_gelu_forward<4> : k_gelu_forward<1>, dim3(grid_vec((size_t)n, v4)), dim3(256), 0, st_,
                     static_cast<const float*>(x),
                     static_cast<float*>(out), (size_t)n);
  return op_launched("gelu forward");
}

int fh_op_gelu_backward(fh_context* c, const void* dout, const void* x, void* dx, int64_t n) {
  OPS_PROLOGUE(c);
  OPS_ARG(dout && x && dx && n > 0, "bad arguments");
  const bool v4 = aligned16(dout) && aligned16(x) && aligned16(dx);
  hipLaunchKernelGGL(v4 ? k_gelu_backward<4> : k_gelu_backward<1>, dim3(grid_vec((size_t)n, v4)), dim3(256), 0, st_,
                     static_cast<const float*>(dout),
                     static_cast<const float*>(x), static_cast<float*>(dx), (size_t)n);
  return op_launched("gelu backward");
}

int fh_op_embedding_forward(fh_context* c, const void* table, int table_rows, const int32_t* indices, int n, void* out,
                            int D) {
  OPS_PROLOGUE(c);
  OPS_ARG(table && out && (indices || n == 0) && n >= 0 && D > 0 && table_rows > 0, "bad arguments");
  for (int t = 0; t < n; t++)
    if (indices[t] < 0 || indices[t] >= table_rows)
      return set_err(FH_ERR_RANGE, "index %d at position %d outside the table's %d rows", indices[t], t, table_rows);
  if (n == 0) return FH_OK;
  int* di = nullptr;
  FH_TRY(upload_ints(c, ops_, indices, (size_t)n, &di));
  hipLaunchKernelGGL(k_embedding_forward, dim3(n), dim3(256), 0, st_, static_cast<const float*>(table), di,
                     static_cast<float*>(out), D);
  return op_launched("embedding forward");
}

int fh_op_embedding_backward(fh_context* c, const void* dout, const int32_t* indices, int n, void* dtable,
                             int table_rows, int D) {
  OPS_PROLOGUE(c);
  OPS_ARG(dout && dtable && (indices || n == 0) && n >= 0 && D > 0 && table_rows > 0, "bad arguments");
  for (int t = 0; t < n; t++)
    if (indices[t] < 0 || indices[t] >= table_rows)
      return set_err(FH_ERR_RANGE, "index %d at position %d outside the table's %d rows", indices[t], t, table_rows);
  if (n == 0) return FH_OK;
  if (n <= kScatterIds) {
    int* di = nullptr;
    FH_TRY(upload_ints(c, ops_, indices, (size_t)n, &di));
    hipLaunchKernelGGL(k_embedding_scatter, dim3(n), dim3(256), 0, st_, static_cast<const float*>(dout), di, n,
                       static_cast<float*>(dtable), D);
    return op_launched("embedding backward");
  }
  // group the positions by id, ascending within each id
  std::vector<int> order(n);
  for (int t = 0; t < n; t++) order[t] = t;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return indices[x] < indices[y]; });
  std::vector<int> host;  // uniq[U] | start[U+1] | pos[n]
  std::vector<int> uniq, start;
  for (int k = 0; k < n; k++)
    if (k == 0 || indices[order[k]] != indices[order[k - 1]]) {
      uniq.push_back(indices[order[k]]);
      start.push_back(k);
    }
  start.push_back(n);
  const int U = (int)uniq.size();
  host.insert(host.end(), uniq.begin(), uniq.end());
  host.insert(host.end(), start.begin(), start.end());
  host.insert(host.end(), order.begin(), order.end());
  int* dev = nullptr;
  FH_TRY(upload_ints(c, ops_, host.data(), host.size(), &dev));
  hipLaunchKernelGGL(k_embedding_backward, dim3((D + 255) / 256, U), dim3(256), 0, st_,
                     static_cast<const float*>(dout), dev, dev + U, dev + 2 * U + 1, static_cast<float*>(dtable), D);
  return op_launched("embedding backward");
}

int fh_op_causal_mask(fh_context* c, void* scores, int64_t len, int T) {
  OPS_PROLOGUE(c);
  OPS_ARG(scores && T > 0 && len > 0 && len % ((int64_t)T * T) == 0, "scores must hold whole [T,T] blocks");
  hipLaunchKernelGGL(k_causal_mask, dim3(grid_for((size_t)len)), dim3(kT), 0, st_, static_cast<float*>(scores),
                     (size_t)len, T);
  return op_launched("causal mask");
}

int fh_op_cross_entropy_forward(fh_context* c, const void* logits, const int32_t* targets, void* probs, int T, int V,
                                int ignore_index, float* loss) {
  OPS_PROLOGUE(c);
  OPS_ARG(logits && probs && targets && loss && T > 0 && V > 0, "bad arguments");
  int count = 0;
  for (int t = 0; t < T; t++) {
    if (targets[t] == ignore_index) continue;
    if (targets[t] < 0 || targets[t] >= V)
      return set_err(FH_ERR_RANGE, "target %d at position %d outside [0,%d)", targets[t], t, V);
    count++;
  }
  void* p = nullptr;
  FH_TRY(ops_scratch(c, ops_, (size_t)T * (sizeof(int32_t) + sizeof(float)), &p));
  int* dt = static_cast<int*>(p);
  float* nll = reinterpret_cast<float*>(dt + T);
  FH_TRY(copy_ints(c, ops_, targets, (size_t)T, dt));
  const float* lg = static_cast<const float*>(logits);
  float* pr = static_cast<float*>(probs);
  if (V <= kRowWaveCols)
    ROW_WAVES(k_ce_forward_wave, V,
              <<<dim3((unsigned)(((size_t)T + 3) / 4)), dim3(256), 0, st_>>>(lg, dt, pr, T, V, ignore_index, nll));
  else if (V > 1024 * 32 || T >= 1 << 22)  // (a grid of 1024-thread blocks ends at 2^32 threads)
    hipLaunchKernelGGL(k_ce_forward, dim3(T), dim3(256), 0, st_, lg, dt, pr, V, ignore_index, nll);
  else if (V <= 1024 * 4)
    hipLaunchKernelGGL(k_ce_forward_row<4>, dim3(T), dim3(1024), 0, st_, lg, dt, pr, V, ignore_index, nll);
  else if (V <= 1024 * 16)
    hipLaunchKernelGGL(k_ce_forward_row<16>, dim3(T), dim3(1024), 0, st_, lg, dt, pr, V, ignore_index, nll);
  else
    hipLaunchKernelGGL(k_ce_forward_row<32>, dim3(T), dim3(1024), 0, st_, lg, dt, pr, V, ignore_index, nll);
  FH_TRY(op_launched("cross-entropy forward"));
  if (ops_->accumulating) {
    // the loss stays on the device until the accumulation ends (ITensorBackend.cs:154-161)
    hipLaunchKernelGGL(k_ce_accumulate, dim3(1), dim3(256), 0, st_, nll, T, ops_->acc);
    ops_->accumulated_targets += count;
    *loss = 0.f;
    return op_launched("loss accumulation");
  }
  std::vector<float> per(T);
  HIP_TRY(hipMemcpyAsync(per.data(), nll, (size_t)T * sizeof(float), hipMemcpyDeviceToHost, st_));
  HIP_TRY(hipStreamSynchronize(st_));
  double total = 0;
  for (int t = 0; t < T; t++)
    if (targets[t] != ignore_index) total += per[t];
  *loss = count == 0 ? 0.f : (float)(total / count);
  return FH_OK;
}

int fh_op_begin_loss_accumulation(fh_context* c) {
  OPS_PROLOGUE(c);
  if (ops_->accumulating) return set_err(FH_ERR_STATE, "Loss accumulation is already active.");
  HIP_TRY(hipMemsetAsync(ops_->acc, 0, sizeof(double), st_));
  ops_->accumulating = true;
  ops_->accumulated_targets = 0;
  return FH_OK;
}

int fh_op_end_loss_accumulation(fh_context* c, float* mean_loss) {
  OPS_PROLOGUE(c);
  OPS_ARG(mean_loss, "null result pointer");
  if (!ops_->accumulating) return set_err(FH_ERR_STATE, "Loss accumulation is not active.");
  double s = 0;
  HIP_TRY(hipMemcpyAsync(&s, ops_->acc, sizeof(double), hipMemcpyDeviceToHost, st_));
  HIP_TRY(hipStreamSynchronize(st_));
  ops_->accumulating = false;
  *mean_loss = ops_->accumulated_targets == 0 ? 0.f : (float)(s / (double)ops_->accumulated_targets);
  return FH_OK;
}

int fh_op_cross_entropy_backward(fh_context* c, const void* probs, const int32_t* targets, void* dlogits, int T, int V,
                                 int ignore_index) {
  OPS_PROLOGUE(c);
  OPS_ARG(probs && dlogits && targets && T > 0 && V > 0, "bad arguments");
  int count = 0;
  for (int t = 0; t < T; t++) {
    if (targets[t] == ignore_index) continue;
    if (targets[t] < 0 || targets[t] >= V)
      return set_err(FH_ERR_RANGE, "target %d at position %d outside [0,%d)", targets[t], t, V);
    count++;
  }
  const size_t n = (size_t)T * V;
  if (count == 0) {
    HIP_TRY(hipMemsetAsync(dlogits, 0, n * sizeof(float), st_));
    return FH_OK;
  }
  int* dt = nullptr;
  FH_TRY(upload_ints(c, ops_, targets, (size_t)T, &dt));
  const float* pr = static_cast<const float*>(probs);
  float* dl = static_cast<float*>(dlogits);
  const size_t blocks = (n + kCeFlatPer - 1) / kCeFlatPer;
  if (V <= kCeFlat && blocks < (1u << 24))
    hipLaunchKernelGGL(k_ce_backward_flat, dim3((unsigned)blocks), dim3(256), 0, st_, pr, dt, dl, n, V, ignore_index,
                       1.f / (float)count);
  else
    hipLaunchKernelGGL(k_ce_backward, dim3(std::min(T, 1 << 23), std::min(((unsigned)V + kCeCols - 1) / kCeCols, 65535u)),
                       dim3(256), 0, st_, pr, dt, dl, (unsigned)T, (unsigned)V, ignore_index, 1.f / (float)count);
  return op_launched("cross-entropy backward");
}

int fh_op_zero(fh_context* c, void* x, int64_t n) {
  OPS_PROLOGUE(c);
  OPS_ARG(x && n >= 0, "bad arguments");
  if (n > 0) HIP_TRY(hipMemsetAsync(x, 0, (size_t)n * sizeof(float), st_));
  return FH_OK;
}

int fh_op_sum_squares(fh_context* c, const void* x, int64_t n, double* out) {
  const void* xs[1] = {x};
  const int64_t ns[1] = {n};
  return fh_op_global_sum_squares(c, xs, ns, 1, out);
}

int fh_op_global_sum_squares(fh_context* c, const void* const* xs, const int64_t* ns, int count, double* out) {
  OPS_PROLOGUE(c);
  OPS_ARG(out && count >= 0 && (count == 0 || (xs && ns)), "bad arguments");
  *out = 0;
  if (count == 0) return FH_OK;
  for (int i = 0; i < count; i++) OPS_ARG(xs[i] && ns[i] >= 0, "bad tensor %d", i);
  auto blocks_of = [](int64_t n) {
    return (int)std::min<int64_t>(kSumsqBlocks, (n + kSumsqPerBlock - 1) / kSumsqPerBlock);
  };
  size_t blocks = 0;
  for (int i = 0; i < count; i++) blocks += blocks_of(ns[i]);
  void* p = nullptr;
  FH_TRY(ops_scratch(c, ops_, (blocks + 1) * sizeof(double), &p));
  double* res = static_cast<double*>(p);
  double* part = res + 1;
  size_t off = 0;
  for (int i = 0; i < count;) {
    SumsqList l{};
    int nb = 0;
    for (; i < count && l.count < kSumsqTensors; i++) {
      if (ns[i] == 0) continue;
      l.x[l.count] = static_cast<const float*>(xs[i]);
      l.n[l.count] = ns[i];
      l.first[l.count++] = nb;
      nb += blocks_of(ns[i]);
    }
    l.first[l.count] = nb;
    if (nb) hipLaunchKernelGGL(k_sumsq, dim3(nb), dim3(256), 0, st_, l, part + off);
    off += nb;
  }
  hipLaunchKernelGGL(k_sum_doubles, dim3(1), dim3(256), 0, st_, part, (int)off, res);
  FH_TRY(op_launched("sum of squares"));
  HIP_TRY(hipMemcpyAsync(out, res, sizeof(double), hipMemcpyDeviceToHost, st_));
  HIP_TRY(hipStreamSynchronize(st_));
  return FH_OK;
}

int fh_op_adamw_step(fh_context* c, void* w, const void* g, void* m, void* v, int64_t n, float lr, float beta1,
                     float beta2, float eps, float weight_decay, int step, int is_matrix) {
  OPS_PROLOGUE(c);
  OPS_ARG(w && g && m && v && n > 0 && step >= 1, "bad arguments");
  const float bc1 = 1.f - powf(beta1, (float)step);
  const float bc2 = 1.f - powf(beta2, (float)step);
  const int decay = weight_decay != 0.f && is_matrix;
  float *fw = static_cast<float*>(w), *fm = static_cast<float*>(m), *fv = static_cast<float*>(v);
  const float* fg = static_cast<const float*>(g);
  if (aligned16(w) && aligned16(g) && aligned16(m) && aligned16(v))
    hipLaunchKernelGGL(k_adamw<4>, dim3(grid_for(((size_t)n + 3) / 4)), dim3(kT), 0, st_, fw, fg, fm, fv, (size_t)n, lr,
                       beta1, beta2, eps, weight_decay, bc1, bc2, decay);
  else
    hipLaunchKernelGGL(k_adamw<1>, dim3(grid_for((size_t)n)), dim3(kT), 0, st_, fw, fg, fm, fv, (size_t)n, lr, beta1,
                       beta2, eps, weight_decay, bc1, bc2, decay);
  return op_launched("adamw step");
}

}  // extern "C"
