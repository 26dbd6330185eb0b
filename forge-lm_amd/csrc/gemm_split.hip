// gemm_split.hip -- fp32 matrix products on the bf16 matrix cores (gfx950).
//
// y = op(a) @ op(b) in fp32 precision: each operand element is split exactly into
// three bf16 values (x = x1 + x2 + x3, each the rounding of what the ones before
// leave: 3 x 8 significant bits hold fp32's 24), and the six products whose weight is
// above fp32's own rounding, x1 y1, x1 y2, x2 y1, x1 y3, x2 y2 and x3 y1, are summed in
// fp32 by v_mfma_f32_32x32x16_bf16.  The three left out are below 2^-26 of x y, under
// the 2^-24 that each fp32 multiply-add rounds by.
//
// Why: the fp32 matrix instruction runs at 157 TFLOP/s and plain FMA code at half of
// that; six bf16 products at 2.5 PFLOP/s are worth 417.  What bounds the kernel is the
// work around the MFMAs: the split (11 VALU instructions per two elements) and the LDS
// traffic (three planes per operand), so a block keeps 128 x 128 results and a wave
// 64 x 64, which reads 12 KB of fragments for 24 MFMAs per 16 k.  Two to three blocks
// share a CU: one's split and barriers run under another's MFMAs.
//
// The operands are read in place, in either order, without a transposed copy.  KC: k
// contiguous (a of NN and NT, b of NT), two 16-byte loads per 8 k of a row.  RC: rows
// contiguous (b of NN and TN, a of TN), eight 4-byte loads per 8 k of a row, coalesced
// across lanes; 8 k of one row meet in one thread either way, so the layout costs
// nothing after the load.
//
// Rounding: the matrix core cuts what it adds off about 8 bits below the sum's last one,
// always downwards.  That is small beside the rounding itself but of one sign, and 6 K / 16
// of them showed where columns of results are added up (a bias gradient over 2048 rows came
// out 1.8e-6 off, 0.5e-6 with fp32 instructions).  So a and the sums change sign every two
// stages and the cuts cancel: 0.41e-6 there (K 768) and 0.83e-6 at K 3072 (fp32 1.0e-6); the
// results themselves 0.42e-6 and 0.85e-6 (fp32 0.50e-6 and 0.99e-6).  It costs 2-5% of the time.
//
// Infinities and NaN: a split of them makes products the fp32 sum would not have (inf *
// 0), so a block whose sums are not all finite computes its tile again on the fp32 matrix
// cores.  A finite result cannot have met one.  A product of NaN alone takes about twice
// its time (2048 x 768 x 3072: 69 -> 141 us, with one row of NaN 113; scalar multiply-adds
// in place of the matrix cores took 5700 in both).
//
// Small elements: bf16 ends at 2^-133 as fp32 does at 2^-149, so the three parts hold less than
// 24 bits of an element below 2^-111 (sums of elements near 2^-118 came out 9e-6 off, near 2^-126
// 2e-3).  What is lost is at most 2^-134 of the other element, so it shows where the sum itself is
// tiny: a block with a sum below 2^-80 that is not zero computes its tile again as well, which keeps
// fp32's precision for other elements up to 2^29 / K^0.5.
#include <algorithm>

#include "kernels.hpp"
#include "mfma_epi.hpp"

namespace fh {

namespace {

constexpr int SK = 32;  // k per stage: 64 bytes of bf16 per row and plane
constexpr int FLIP = 2;  // stages between sign changes
constexpr uint32_t kTiny = (127u - 80u) << 23;  // bits of 2^-80

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// 16-byte chunk c of row r is stored at chunk c ^ g(r), with g different over rows r, r + 4,
// r + 8, r + 12 (16 rows of one chunk fill the 64 banks that reads see) and over pairs of rows (8 rows
// fill the 32 that writes see): no bank conflicts either way.  bits 2-3 of r alone cost the
// row-contiguous operands 5% of the CU's cycles each in write conflicts.
__device__ __forceinline__ int split_swz(int r, int c) { return c ^ (((r >> 1) ^ (r >> 3 & 1)) & 3); }

// two elements -> their three bf16 parts, packed (round to nearest even at each step;
// the subtractions are exact)
__device__ __forceinline__ void split2(float x, float y, uint32_t& p1, uint32_t& p2, uint32_t& p3) {
  auto pack = [](float a, float b) {
    const bf16x2_t v = {(__bf16)a, (__bf16)b};
    uint32_t p = __builtin_bit_cast(uint32_t, v);
    asm("" : "+v"(p));  // one conversion: without it the compiler converts the low half again to subtract it
    return p;
  };
  p1 = pack(x, y);
  const float x1 = x - __uint_as_float(p1 << 16), y1 = y - __uint_as_float(p1 & 0xffff0000u);
  p2 = pack(x1, y1);
  p3 = pack(x1 - __uint_as_float(p2 << 16), y1 - __uint_as_float(p2 & 0xffff0000u));
}

struct SplitArgs {
  const float* a;
  const float* b;
  int M, K, N;
  int slots, splits, kchunk;
  int gm, gn;
  const float* bias;  // [N] or null
  const float* res;   // added to y (y itself to accumulate), or null
  int gelu;
  float* y;
  float* part;  // splits > 1: partial sums [splits][slots * M][N]
};

// Tile rows [row0, row0 + R) of one operand, k steps of SK from kb on.
// unit u of thread t holds 8 consecutive k of one row: KC: row t / 4 + 64 u, chunk
// t % 4; RC: row t % 64 + 64 u, chunk t / 64.
template <int R, bool KC>
struct Operand {
  static constexpr int U = R / 64;
  const char* base;   // first element of the current stage
  int64_t left;       // bytes from base to the end of what may be read
  int64_t step;       // bytes per stage
  int off[KC ? U : 8];  // byte offsets of the loads within a stage
  int row, chunk;

  __device__ __forceinline__ void init(const float* p, int ld, int rows, int row0, int K, int kb, int tid) {
    if constexpr (KC) {
      row = tid >> 2;
      chunk = tid & 3;
      base = reinterpret_cast<const char*>(p + (size_t)row0 * ld + kb);
      left = ((int64_t)min(R, rows - row0) * ld - kb) * 4;
      step = SK * 4;
#pragma unroll
      for (int u = 0; u < U; u++) off[u] = ((row + 64 * u) * ld + 8 * chunk) * 4;
    } else {
      row = tid & 63;
      chunk = tid >> 6;
      base = reinterpret_cast<const char*>(p + (size_t)kb * ld + row0);
      left = ((int64_t)(K - kb) * ld - row0) * 4;
      step = (int64_t)SK * ld * 4;
#pragma unroll
      for (int j = 0; j < 8; j++) off[j] = ((8 * chunk + j) * ld + row) * 4;
    }
  }

  // bounded loads: past the operand's end they return 0 (a KC row past the last one, an
  // RC k past the last one; the range is checked dword by dword, and a KC load of a whole
  // stage lies inside or outside as a whole)
  // `on` false (a stage past the last): every load out of bounds, no branch around them
  template <bool TAIL>
  __device__ __forceinline__ void load(float (&v)[U][8], bool on) {
    const int num = !on ? 0 : (int)(left > 0x7ffffffc ? 0x7ffffffc : left);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), (short)0, num, 0x00020000);
    if constexpr (KC && !TAIL) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
          const u32x4_t w = __builtin_amdgcn_raw_buffer_load_b128(rs, off[KC ? u : 0] + 16 * q, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; j++) v[u][4 * q + j] = __uint_as_float(w[j]);
        }
    } else {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < 8; j++)
          v[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rs, KC ? off[KC ? u : 0] + 4 * j : off[KC ? 0 : j] + 256 * u, 0, 0));
    }
    if (!TAIL && on) {
      base += step;
      left -= step;
    }
  }

  // the last stage of a K that is no multiple of SK: a KC row runs on into the next one
  __device__ __forceinline__ void mask(float (&v)[U][8], int krem) {
    if constexpr (KC) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < 8; j++) v[u][j] = 8 * chunk + j < krem ? v[u][j] : 0.f;
    }
  }

  // the elements as they are, 128 bytes a row: 16-byte chunk c of row r at c ^ (r & 7)
  __device__ __forceinline__ void store_f32(char* lds, const float (&v)[U][8]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int q = 0; q < 2; q++)
        *reinterpret_cast<float4*>(lds + (row + 64 * u) * 128 + 16 * ((2 * chunk + q) ^ (row & 7))) =
            make_float4(v[u][4 * q], v[u][4 * q + 1], v[u][4 * q + 2], v[u][4 * q + 3]);
  }

  // `sign`: 0 or the sign bit, flipped into every element
  __device__ __forceinline__ void store(char* lds, const float (&v)[U][8], uint32_t sign = 0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      uint32_t p[3][4];
#pragma unroll
      for (int j = 0; j < 4; j++)
        split2(__uint_as_float(__float_as_uint(v[u][2 * j]) ^ sign),
               __uint_as_float(__float_as_uint(v[u][2 * j + 1]) ^ sign), p[0][j], p[1][j], p[2][j]);
      const int at = (row + 64 * u) * 64 + 16 * split_swz(row, chunk);
#pragma unroll
      for (int s = 0; s < 3; s++)
        *reinterpret_cast<uint4*>(lds + s * R * 64 + at) = make_uint4(p[s][0], p[s][1], p[s][2], p[s][3]);
    }
  }
};

template <int BM, int BN, bool AKC, bool BKC>
__global__ __launch_bounds__(256, 3) void k_gemm_split(SplitArgs g) {
  constexpr int MT = BM / 64, NT = BN / 64;  // 32 x 32 accumulators per wave (2 x 2 waves)
  // The 64 x 64 tile has registers for a second accumulator: the five small products go there, so
  // the large sums are rounded K / 16 times and not 6 K / 16 (48 heads of 331 x 64: 3.4e-7 -> 1.4e-7
  // against 64 bits; windows of 33 to 128 rows at d 128: 2.6e-7 -> 1.8e-7, fp32 instructions 2.3e-7) at
  // the same time.  128 x 64 would take 156 registers where it has 128: three blocks a CU, not four.
  constexpr int NACC = MT * NT > 1 ? 1 : 2;
  __shared__ __align__(16) char smem[3 * (BM + BN) * 64];
  char* const As = smem;
  char* const Bs = smem + 3 * BM * 64;

  // each XCD (blocks reach them in turn) takes a contiguous run of tiles: neighbours in a
  // row of tiles share their A rows in one L2, and 8 K splits give each XCD one slice of K
  const int total = gridDim.x, bid = blockIdx.x;
  const int x = bid & 7, q = total >> 3, rem = total & 7;
  int t = x * q + min(x, rem) + (bid >> 3);
  const int tn = t % g.gn;
  t /= g.gn;
  const int tm = t % g.gm;
  t /= g.gm;
  const int split = t % g.splits, slot = t / g.splits;
  const int m0 = tm * BM, n0 = tn * BN;
  const int kb = split * g.kchunk, ke = min(g.K, kb + g.kchunk);
  const float* a = g.a + (size_t)slot * g.M * g.K;
  const float* b = g.b + (size_t)slot * g.K * g.N;

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w & 1, wn = w >> 1;
  const int fr = lane & 31, fh = lane >> 5;

  Operand<BM, AKC> oa;
  Operand<BN, BKC> ob;
  oa.init(a, AKC ? g.K : g.M, g.M, m0, g.K, kb, tid);
  ob.init(b, BKC ? g.K : g.N, g.N, n0, g.K, kb, tid);
  float va[MT][8], vb[NT][8];

  // acc[0]: the x1 y1 products, acc[1] (the same where registers are short) the five small ones
  f32x16_t acc[NACC][MT][NT];
#pragma unroll
  for (int c = 0; c < NACC; c++)
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[c][i][j][r] = 0.f;

  auto compute = [&]() {
#pragma unroll
    for (int kk = 0; kk < SK / 16; kk++) {
      bf16x8_t af[3][MT], bf[3][NT];
#pragma unroll
      for (int s = 0; s < 3; s++) {
#pragma unroll
        for (int i = 0; i < MT; i++)
          af[s][i] = *reinterpret_cast<const bf16x8_t*>(As + s * BM * 64 + (wm * (BM / 2) + i * 32 + fr) * 64 +
                                                        16 * split_swz(fr, 2 * kk + fh));
#pragma unroll
        for (int j = 0; j < NT; j++)
          bf[s][j] = *reinterpret_cast<const bf16x8_t*>(Bs + s * BN * 64 + (wn * (BN / 2) + j * 32 + fr) * 64 +
                                                        16 * split_swz(fr, 2 * kk + fh));
      }
      // the small products first, every accumulator once per step
      constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
      for (int p = 0; p < 6; p++)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
          for (int j = 0; j < NT; j++)
            acc[p < 5 ? NACC - 1 : 0][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                af[PA[p]][i], bf[PB[p]][j], acc[p < 5 ? NACC - 1 : 0][i][j], 0, 0, 0);
    }
  };

  const int nst = (ke - kb) / SK, krem = (ke - kb) % SK;
  uint32_t sign = 0;
  auto flip = [&]() {
    sign ^= 0x80000000u;
#pragma unroll
    for (int c = 0; c < NACC; c++)
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[c][i][j][r] = -acc[c][i][j][r];
  };
  auto put = [&]() {
    oa.store(As, va, sign);
    ob.store(Bs, vb);
    __syncthreads();
  };
  // stage st + 1 loads into registers while stage st is multiplied from LDS.  A second
  // register stage, or two LDS stages with the split between the MFMAs, measured slower
  // at every size (8192 x 4096 x 4096: 181-190 against 220 TFLOP/s): fewer blocks per CU
  oa.template load<false>(va, nst > 0);
  ob.template load<false>(vb, nst > 0);
  for (int st = 0; st < nst; st++) {
    put();
    oa.template load<false>(va, st + 1 < nst);
    ob.template load<false>(vb, st + 1 < nst);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before the MFMAs, not between them
    compute();
    if (st % FLIP == FLIP - 1) flip();
    __syncthreads();
  }
  if (krem) {
    // the rest of a K that is no multiple of SK, with nothing to hide its loads behind
    oa.template load<true>(va, true);
    ob.template load<true>(vb, true);
    oa.mask(va, krem);
    ob.mask(vb, krem);
    put();
    compute();
  }
  if (sign) flip();
  if constexpr (NACC == 2) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][i][j][r] += acc[1][i][j][r];
  }

  // ---- results ------------------------------------------------------------------------
  const size_t yrow = (size_t)slot * g.M + m0;
  const int rows = min(BM, g.M - m0);
  const bool parts = g.part != nullptr;
  float* const out = parts ? g.part + (size_t)split * g.slots * g.M * g.N : g.y;
  // the thread's place again, from a copy that the compiler takes for another value: kept in registers
  // through the loop, what the rest derives from it displaced what the loop needs
  int tid2 = threadIdx.x;
  asm("" : "+v"(tid2));
  const int lane2 = tid2 & 63, fr2 = lane2 & 31, fh2 = lane2 >> 5;
  // rows and columns past the end may be flagged too: that costs time only.  Two instructions an
  // element: a maximum that keeps NaN, and a minimum of the bits without sign, less one (0 wraps)
  float most = 0.f;
  uint32_t least = ~0u;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        most = __builtin_elementwise_maximum(most, fabsf(acc[0][i][j][r]));
        least = min(least, (__float_as_uint(acc[0][i][j][r]) << 1) - 1);
      }
  const bool bad = !(most < INFINITY) || least < 2 * kTiny - 1;
  if (__syncthreads_or(bad)) {
    // the tile again on the fp32 matrix cores, which give what fp32 arithmetic gives
    oa.init(a, AKC ? g.K : g.M, g.M, m0, g.K, kb, tid2);
    ob.init(b, BKC ? g.K : g.N, g.N, n0, g.K, kb, tid2);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][i][j][r] = 0.f;
    for (int st = 0; st < nst + (krem != 0); st++) {
      if (st < nst) {
        oa.template load<false>(va, true);
        ob.template load<false>(vb, true);
      } else {
        oa.template load<true>(va, true);
        ob.template load<true>(vb, true);
        oa.mask(va, krem);
        ob.mask(vb, krem);
      }
      oa.store_f32(As, va);
      ob.store_f32(As + BM * 128, vb);
      __syncthreads();
      // a step's two k are k and k + 16 of the stage: 16 bytes of a row feed four steps.  (Unrolled, these
      // steps cost the loop above registers: 768 x 2048 x 3072 TN 74.9 -> 76.9 us.)
#pragma unroll 1
      for (int kk = 0; kk < SK / 8; kk++) {
        float4 af[MT], bf[NT];
        const int at = fr2 * 128 + 16 * ((4 * fh2 + kk) ^ (fr2 & 7));
#pragma unroll
        for (int i = 0; i < MT; i++)
          af[i] = *reinterpret_cast<const float4*>(As + (wm * (BM / 2) + i * 32) * 128 + at);
#pragma unroll
        for (int j = 0; j < NT; j++)
          bf[j] = *reinterpret_cast<const float4*>(As + BM * 128 + (wn * (BN / 2) + j * 32) * 128 + at);
        auto step = [&](auto pick) {
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
              acc[0][i][j] =
                  __builtin_amdgcn_mfma_f32_32x32x2f32(pick(af[i]), pick(bf[j]), acc[0][i][j], 0, 0, 0);
        };
        step([](const float4& v) { return v.x; });
        step([](const float4& v) { return v.y; });
        step([](const float4& v) { return v.z; });
        step([](const float4& v) { return v.w; });
      }
      __syncthreads();
    }
  }
  const __amdgpu_buffer_rsrc_t ry = rows_rsrc(out, yrow, rows, g.N, 4);
  const __amdgpu_buffer_rsrc_t rres = !parts && g.res ? rows_rsrc(g.res, yrow, rows, g.N, 4) : ry;
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const int col = n0 + wn * (BN / 2) + j * 32 + fr2;
    if (col >= g.N) continue;
    const float bcol = !parts && g.bias ? g.bias[col] : 0.f;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int tr = wm * (BM / 2) + i * 32;
      if (parts)
        mfma_store_tile<EPI_NONE, false, false, 2>(acc[0][i][j], lane2, tr, col, g.N, 0.f, ry, ry);
      else if (g.gelu)
        mfma_store_tile<EPI_GELU, false, false>(acc[0][i][j], lane2, tr, col, g.N, bcol, ry, ry);
      else if (g.res)
        mfma_store_tile<EPI_NONE, true, false>(acc[0][i][j], lane2, tr, col, g.N, bcol, rres, ry);
      else
        mfma_store_tile<EPI_NONE, false, false>(acc[0][i][j], lane2, tr, col, g.N, bcol, ry, ry);
    }
  }
}

template <int BM, int BN>
hipError_t launch_tile(hipStream_t st, int mode, unsigned blocks, const SplitArgs& g) {
  if (mode == 0)
    hipLaunchKernelGGL((k_gemm_split<BM, BN, true, false>), dim3(blocks), dim3(256), 0, st, g);
  else if (mode == 1)
    hipLaunchKernelGGL((k_gemm_split<BM, BN, true, true>), dim3(blocks), dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((k_gemm_split<BM, BN, false, false>), dim3(blocks), dim3(256), 0, st, g);
  return hipGetLastError();
}

}  // namespace

namespace {

struct SplitPlan {
  int bm, bn, splits;
};

constexpr size_t kMaxBlocks = (size_t)1 << 24;  // of 256 threads

constexpr int kTiles[3][2] = {{128, 128}, {128, 64}, {64, 64}};

size_t split_blocks(int bm, int bn, int slots, int M, int N) {
  return (size_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * slots;
}

// Tile and K splits by a cost in microseconds, fitted to the times of every tile and split over
// 92 products (40 .. 16257 rows, K 64 .. 16257, plain and batched; weights cold): what it picks
// is 1.4% off the fastest in the geometric mean and 10% at worst.  A launch costs `fixed`, and
// `round` more per round of blocks over the CUs; a stage costs a CU `unit` per block of its own
// (a large tile does the most per operand byte: 217 / 190 / 168 TFLOP/s at 8192 x 4096 x 4096),
// a lone block no less than `alone` (its chain of load, split, LDS and MFMAs); splitting K costs a
// second launch and the partial sums' way through memory.  M 2048, K 3072, N 768: 128 x 128 tiles in
// 5 splits, 72 us with their sum, unsplit 109; 100 x 768 x 768: 64 x 64 in 12 splits, 11.3, unsplit 23.
SplitPlan split_plan(int slots, int M, int K, int N, size_t part_floats, int cus) {
  constexpr double fixed[3] = {4.6, 3.9, 4.1}, round[3] = {1.5, 0.7, 0.24};
  constexpr double alone[3] = {1.78, 1.2, 0.77}, unit[3] = {1.17, 0.74, 0.45};
  constexpr int counts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};
  const double mn = (double)slots * M * N;
  SplitPlan best{64, 64, 1};
  double best_us = 1e300;
  for (int i = 0; i < 3; i++) {
    const double tiles = (double)split_blocks(kTiles[i][0], kTiles[i][1], slots, M, N);
    for (int S : counts) {
      if (S > 1 && (K < S * 2 * SK || mn * S > (double)part_floats || tiles * S >= (double)kMaxBlocks)) break;
      const double rounds = (double)(((size_t)tiles * S + cus - 1) / cus);
      const int stages = ((K + S - 1) / S + SK - 1) / SK;
      double us = fixed[i] + rounds * round[i] + stages * std::max(alone[i], rounds * unit[i]);
      if (S > 1) us += 2.8 + mn * (S + 1) * 4 / 5.2e6;
      if (us < best_us) {
        best_us = us;
        best = SplitPlan{kTiles[i][0], kTiles[i][1], S};
      }
    }
  }
  return best;
}

// y == null: only the partial sums part[splits][slots * M][N]
hipError_t run_split(hipStream_t st, int mode, const float* a, const float* b, int slots, int M, int K, int N,
                     const float* bias, int gelu, const float* res, float* y, float* part, const SplitPlan& p,
                     int* splits) {
  SplitArgs g{};
  g.a = a;
  g.b = b;
  g.M = M;
  g.K = K;
  g.N = N;
  g.slots = slots;
  g.kchunk = ((K + p.splits - 1) / p.splits + SK - 1) / SK * SK;
  g.splits = (K + g.kchunk - 1) / g.kchunk;  // every split has work
  g.gm = (M + p.bm - 1) / p.bm;
  g.gn = (N + p.bn - 1) / p.bn;
  g.bias = bias;
  g.gelu = gelu;
  g.res = res;
  g.y = y;
  g.part = !y || g.splits > 1 ? part : nullptr;
  if (splits) *splits = g.splits;
  const unsigned blocks = (unsigned)(split_blocks(p.bm, p.bn, slots, M, N) * g.splits);
  hipError_t e;
  if (p.bm == 128 && p.bn == 128)
    e = launch_tile<128, 128>(st, mode, blocks, g);
  else if (p.bm == 128)
    e = launch_tile<128, 64>(st, mode, blocks, g);
  else
    e = launch_tile<64, 64>(st, mode, blocks, g);
  if (e != hipSuccess || !g.part || !y) return e;
  return launch_splitk_epilogue(st, part, g.splits, slots * M, N, bias, gelu ? EPI_GELU : EPI_NONE, res, y);
}

}  // namespace

bool gemm_split_fits(int slots, int M, int K, int N) {
  // 32-bit byte offsets: 128 rows of K floats (KC), 32 k of M or N floats (RC) and the 128 rows of N
  // floats that a tile writes; and a grid below 2^32 threads
  return slots > 0 && M > 0 && K > 0 && N > 0 && M < (1 << 24) && K < (1 << 22) && N < (1 << 22) &&
         (int64_t)slots * M < (1 << 30) && split_blocks(64, 64, slots, M, N) < kMaxBlocks;
}

hipError_t launch_gemm_split(hipStream_t st, int mode, const float* a, const float* b, int slots, int M, int K, int N,
                             const float* bias, int gelu, const float* res, float* y, float* part,
                             size_t part_floats, int cus) {
  if (!a || !b || !y || mode < 0 || mode > 2 || (gelu && res) || !gemm_split_fits(slots, M, K, N))
    return hipErrorInvalidValue;
  const SplitPlan p = split_plan(slots, M, K, N, part ? part_floats : 0, cus > 0 ? cus : 256);
  return run_split(st, mode, a, b, slots, M, K, N, bias, gelu, res, y, part, p, nullptr);
}

hipError_t launch_gemm_split_parts(hipStream_t st, const float* a, const float* b, int M, int K, int N, float* part,
                                   size_t part_floats, int cus, int* splits) {
  if (!a || !b || !part || !splits || !gemm_split_fits(1, M, K, N) || (size_t)M * N > part_floats)
    return hipErrorInvalidValue;
  const SplitPlan p = split_plan(1, M, K, N, part_floats, cus > 0 ? cus : 256);
  return run_split(st, 1, a, b, 1, M, K, N, nullptr, 0, nullptr, nullptr, part, p, splits);
}

size_t gemm_split_part_floats(int slots, int M, int K, int N, size_t most, int cus) {
  if (!gemm_split_fits(slots, M, K, N)) return 0;
  const SplitPlan p = split_plan(slots, M, K, N, most, cus > 0 ? cus : 256);
  return p.splits > 1 ? (size_t)p.splits * slots * M * N : 0;
}

}  // namespace fh
