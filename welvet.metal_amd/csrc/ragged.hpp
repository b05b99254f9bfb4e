// ragged.hpp (part of dense.hip) — Dense forward and dX for rows that do not start on a chunk
// boundary (an input width that is no multiple of the format's chunk: 4
// elements for 32-bit formats, 8 for 16-bit, 16 for 8-bit, 32 below), any
// format, any batch.
//
// A chunk of E codes may start at any bit of the packed body: a lane loads
// the dwords that cover it (one more than a chunk has) and shifts them into
// the aligned chunk the other kernels' decode takes.  Products and sums are
// f64 (each f32 operand widened): on the VALU for one row of x, for up to four
// where the weights are few (eight where rows are also long) and for dX of few
// rows or outputs, else on the f64 MFMA.
//
// What bounds them: short rows, the launch and one load-compute-reduce chain
// (4-6 us); large ones, the f64 matrix rate (half of fp32's) and the chunk
// loads.  Measured against the kernels they replaced (a block per output row
// that re-read the weights for every batch row; dX a thread per output), us:
// Float32 1001 -> 777 b100 99 -> 11.6, Int8 393 -> 362 b20 16.1 -> 5.1, NF4
// 4095^2 b1 15.5 -> 11.3, b20 238 -> 29.5.  x staged through LDS with
// whole-row loads and 16-byte-aligned chunk loads with a shift were measured
// and not kept: equal at 4095^2, 10-25% slower below (1001 -> 777 b20 Int8
// 7.3 against 6.5, Float32 8.7 / 6.7), the staging lengthens the chain.
#pragma once

#include <algorithm>

#include "codec.hpp"
#include "kernel_formats.hpp"
#include "kernels.hpp"

namespace wh {
namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

struct RaggedArgs {
  const uint8_t *body;
  const float *lut;
  float scale, minv;
  const float *A;  // x [M][K], or dpre [M][K] for dX
  int M, K, N;     // product dims; a stored row has `cols` elements
  int cols;
  int nst;  // k stages
  int gx;   // tiles along N (one-dimensional grid: tile = blockIdx.x)
};

// NE codes (a chunk, or its first NE) from element `elem` of the body on.
// Reads at most 4 bytes past them: inside the store's padding for every
// elem < n.
template <int F, int NE = FI<F>::kE>
__device__ inline void load_chunk_at(const uint8_t *__restrict__ body, int64_t elem, uint32_t (&w)[FI<F>::kW]) {
  constexpr int BITS = FI<F>::kBits, W = (NE * BITS + 31) / 32;
  struct __attribute__((packed, aligned(4))) Words { uint32_t v[W]; };
  if constexpr (BITS >= 32) {
    const Words p = *(const Words *)(body + elem * (BITS / 8));
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = p.v[i];
  } else {
    const int64_t bit = elem * BITS;
    const uint8_t *p = body + (bit >> 5) * 4;
    const uint32_t sh = (uint32_t)bit & 31u;
    const Words v = *(const Words *)p;
    const uint32_t last = *(const uint32_t *)(p + 4 * W);
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = __builtin_amdgcn_alignbit(i + 1 < W ? v.v[i + 1] : last, v.v[i], sh);
  }
}

// NK (a multiple of 4, or 1 or 2) consecutive values of a row of K floats
// from k on; `whole`: all of them lie inside the row.  Otherwise each load is
// clamped to the row's last value (the caller zeroes what lies past it).
template <int NK>
__device__ inline void load_row(const float *__restrict__ row, int k, int K, bool whole, float (&v)[NK]) {
  if (whole) {
    if constexpr (NK % 4 == 0) {
      struct __attribute__((packed, aligned(4))) Quad { float f[4]; };
#pragma unroll
      for (int q = 0; q < NK; q += 4) {
        const Quad p = *(const Quad *)(row + k + q);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[q + t] = p.f[t];
      }
    } else {
#pragma unroll
      for (int q = 0; q < NK; ++q) v[q] = row[k + q];
    }
  } else {
#pragma unroll
    for (int q = 0; q < NK; ++q) v[q] = row[min(k + q, K - 1)];
  }
}

// Row products, B rows of x (grid row 1: the last B of M): a block holds 4 / S
// output rows, S waves share one, its pieces of P codes dealt to their lanes in
// turn.  One row: up to four codes per lane (a whole chunk leaves most lanes of
// a short row idle), but one of Complex64, whose imaginary halves are not
// loaded: two strided dwords per lane take longer than one (4095 -> 1000 b1 9.0
// us, with one 6.9).  More rows, of which most start off a 16-byte boundary: one code
// per lane, so each row's loads are whole cache lines (four dwords per lane of
// a 16-byte-strided row take 39 cycles each: 4095^2 b2 32 us).
template <int F, int B>
constexpr int ragged_piece() {
  return B > 1 || F == FC64 ? 1 : FI<F>::kE < 4 ? FI<F>::kE : 4;
}
template <int F, int B>
__global__ void __launch_bounds__(256) ragged_gemv_kernel(RaggedArgs a, int S, const double *bias, int bias_len,
                                                          int act, float *pre, float *post) {
  using I = FI<F>;
  constexpr int P = ragged_piece<F, B>(), W = I::kW;
  __shared__ __align__(16) float lut_s[I::kTable];
  __shared__ double red[4][B];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if constexpr (I::kLut) {
    TabCopy<F> tab;
    tab.load(a.lut, tid);
    tab.store(lut_s, tid);
    __syncthreads();
  }
  const int part = wave & (S - 1);
  const int row = min((int)blockIdx.x * (4 / S) + wave / S, a.N - 1);
  double acc[B];
#pragma unroll
  for (int b = 0; b < B; ++b) acc[b] = 0.0;
  const int npieces = (a.K + P - 1) / P, m0 = blockIdx.y == 0 ? 0 : a.M - B;
  const int64_t base = (int64_t)row * a.cols;
  const float *x = a.A + (int64_t)m0 * a.K;
  for (int c = part * 64 + lane; c < npieces; c += 64 * S) {
    const int k = c * P;
    uint32_t w[W];
    load_chunk_at<F, P>(a.body, base + k, w);
    const bool whole = k + P <= a.K;
    float xv[B][P];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int64_t off = (int64_t)b * a.K;
      if (B == 1 && whole) {
        load_x<P>(x + k, xv[b]);
      } else {
#pragma unroll
        for (int e = 0; e < P; ++e) xv[b][e] = x[off + min(k + e, a.K - 1)];
      }
    }
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const bool in = whole || k + e < a.K;
      const double wv = in ? (double)chunk_value<F>(w, e, lut_s, a.scale, a.minv) : 0.0;
#pragma unroll
      for (int b = 0; b < B; ++b) acc[b] = fma(wv, in ? (double)xv[b][e] : 0.0, acc[b]);
    }
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const double s = wave_sum(acc[b]);
    if (lane == 0) red[wave][b] = s;
  }
  __syncthreads();
  if (tid < (4 / S) * B) {  // thread t: output row t / B of the block, batch row t % B
    const int r = tid / B, b = tid % B, o = blockIdx.x * (4 / S) + r;
    double t = 0.0;
    for (int i = 0; i < S; ++i) t += red[r * S + i][b];
    // a row that both halves hold is the first one's: the epilogue may read
    // what it overwrites (kSwiGated)
    if (o < a.N && (blockIdx.y == 0 || m0 + b >= B))
      bias_act_store(t, o, bias, bias_len, act, pre, post, (int64_t)(m0 + b) * a.N + o);
  }
}

// k per lane and stage of the MFMA kernels: lane group h = lane / 16 supplies
// k = k0 + KR h + t at step t, a run of KR consecutive elements of its row.
template <int F>
struct RaggedShape {
  static constexpr int E = FI<F>::kE;
  static constexpr int KR = E >= 8 ? 32 : 4 * E;
  static constexpr int NCH = KR / E;
  static constexpr int ST = 4 * KR;
};

// Sum over the block's waves (each holds the same T tiles over its own k
// stages) in wave order, one output element per thread and turn; store(mt,
// nt, i, j, sum) with i, j the row and column in the 16 x 16 tile.
// v_mfma_f64_16x16x4: register r of lane (j, h) is row 4 r + h, column j.
template <int T, int NT, typename Store>
__device__ inline void ragged_sum(double *ex, const doublex4 (&acc)[T], int nwaves, Store store) {
  const int tid = threadIdx.x, lane = tid & 63, g = tid >> 6;
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) ex[((g * T + t) * 4 + r) * 64 + lane] = acc[t][r];
  __syncthreads();
  for (int q = tid; q < T * 256; q += nwaves * 64) {
    double s = 0.0;
    for (int w = 0; w < nwaves; ++w) s += ex[w * T * 256 + q];
    const int t = q >> 8, r = (q >> 6) & 3, l = q & 63;
    store(t / NT, t % NT, 4 * r + (l >> 4), l & 15, s);
  }
}

// Forward: C[m][n] = sum_k x[m][k] W[n][k] on
// v_mfma_f64_16x16x4_f64.  A wave owns MT x NT tiles of 16 x 16 and walks k
// stages g, g + KG, ...; the block's waves share the tiles and split the
// stages, so K is never split across blocks (no partial tiles in memory).
template <int F, int MT, int NT, int KG>
__global__ void __launch_bounds__(64 * KG) ragged_gemm_kernel(RaggedArgs a, const double *bias, int bias_len,
                                                              int act, float *pre, float *post) {
  using I = FI<F>;
  using S = RaggedShape<F>;
  constexpr int E = S::E, W = I::kW, KR = S::KR, NCH = S::NCH, ST = S::ST;
  __shared__ __align__(16) float lut_s[I::kTable];
  __shared__ double ex[KG * MT * NT * 256];
  const int tid = threadIdx.x, lane = tid & 63, g = tid >> 6, nw = blockDim.x >> 6;
  const int j = lane & 15, h = lane >> 4;
  const int n0 = blockIdx.x % a.gx * 16 * NT, m0 = blockIdx.x / a.gx * 16 * MT;
  if constexpr (I::kLut) {
    TabCopy<F> tab;
    tab.load(a.lut, tid);
    tab.store(lut_s, tid);
    __syncthreads();
  }
  const float *xr[MT];
  int64_t wr[NT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xr[t] = a.A + (int64_t)min(m0 + 16 * t + j, a.M - 1) * a.K;
#pragma unroll
  for (int t = 0; t < NT; ++t) wr[t] = (int64_t)min(n0 + 16 * t + j, a.N - 1) * a.cols;
  doublex4 acc[MT * NT];
#pragma unroll
  for (int t = 0; t < MT * NT; ++t) acc[t] = doublex4{0.0, 0.0, 0.0, 0.0};
  const int klast = (a.K - 1) / E * E;
  for (int s = g; s < a.nst; s += nw) {
    const int k0 = s * ST + KR * h;
    const bool whole = (s + 1) * ST <= a.K;  // uniform over the wave
    uint32_t w[NT][NCH][W];
    float x[MT][KR];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < NCH; ++c) load_chunk_at<F>(a.body, wr[t] + min(k0 + c * E, klast), w[t][c]);
#pragma unroll
    for (int t = 0; t < MT; ++t) load_row<KR>(xr[t], k0, a.K, whole, x[t]);
#pragma unroll
    for (int q = 0; q < KR; ++q) {
      const bool in = whole || k0 + q < a.K;
      double bv[NT], av[MT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        bv[t] = in ? (double)chunk_value<F>(w[t][q / E], q % E, lut_s, a.scale, a.minv) : 0.0;
#pragma unroll
      for (int t = 0; t < MT; ++t) av[t] = in ? (double)x[t][q] : 0.0;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt * NT + nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[mt], bv[nt], acc[mt * NT + nt], 0, 0, 0);
    }
  }
  ragged_sum<MT * NT, NT>(ex, acc, nw, [&](int mt, int nt, int i, int jj, double s) {
    const int m = m0 + 16 * mt + i, n = n0 + 16 * nt + jj;
    if (m < a.M && n < a.N) bias_act_store(s, n, bias, bias_len, act, pre, post, (int64_t)m * a.N + n);
  });
}

// dX: C[m][i] = sum_o dpre[m][o] W[o][i], K = rows, N = cols.  A wave decodes
// the 16-column pieces of a stage's rows into its own LDS tile (pitch 17) and
// reads them back as B operands; otherwise as ragged_gemm_kernel.  next_pre:
// the layer below's piecewise activation derivative is applied to the stored
// fl32, as gemm_regt_kernel does.
template <int F>
struct RaggedTShape {
  static constexpr int E = FI<F>::kE;
  static constexpr int KR = E >= 4 ? 16 : 8;
  static constexpr int ST = 4 * KR;
  static constexpr int DE = E >= 16 ? 16 : E;   // elements a chunk load decodes
  static constexpr int CPR = 16 / DE;           // chunk loads per row piece
  static constexpr int NCH = ST * CPR / 64;     // chunk loads per lane and stage
  static constexpr int P = 17;
  static_assert(ST * CPR % 64 == 0, "whole chunk loads per lane");
};
template <int F, int MT, int KG>
__global__ void __launch_bounds__(64 * KG) ragged_dx_kernel(RaggedArgs a, float *out, const float *next_pre,
                                                            int next_act) {
  using I = FI<F>;
  using S = RaggedTShape<F>;
  using V = typename I::Acc;
  constexpr int E = S::E, W = I::kW, KR = S::KR, ST = S::ST, DE = S::DE, CPR = S::CPR, NCH = S::NCH, P = S::P;
  __shared__ __align__(16) float lut_s[I::kTable];
  __shared__ V tile[KG][ST * P];
  __shared__ double ex[KG * MT * 256];
  const int tid = threadIdx.x, lane = tid & 63, g = tid >> 6, nw = blockDim.x >> 6;
  const int j = lane & 15, h = lane >> 4;
  const int n0 = blockIdx.x % a.gx * 16, m0 = blockIdx.x / a.gx * 16 * MT;
  if constexpr (I::kLut) {
    TabCopy<F> tab;
    tab.load(a.lut, tid);
    tab.store(lut_s, tid);
    __syncthreads();
  }
  const float *xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xr[t] = a.A + (int64_t)min(m0 + 16 * t + j, a.M - 1) * a.K;
  doublex4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = doublex4{0.0, 0.0, 0.0, 0.0};
  V *tw = tile[g];
  for (int s = g; s < a.nst; s += nw) {
    const int k0 = s * ST;
    const bool whole = k0 + ST <= a.K;
    uint32_t w[NCH][W];
    float x[MT][KR];
    // load c: row q / CPR, piece q % CPR of the row's 16 columns
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int q = lane + 64 * c;
      const int o = min(k0 + q / CPR, a.K - 1), col = min(n0 + (q % CPR) * DE, a.N - 1);
      load_chunk_at<F>(a.body, (int64_t)o * a.cols + col, w[c]);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) load_row<KR>(xr[t], k0 + KR * h, a.K, whole, x[t]);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int q = lane + 64 * c;
      const bool in = whole || k0 + q / CPR < a.K;
#pragma unroll
      for (int e = 0; e < DE; ++e) {
        const V v = chunk_value<F>(w[c], e, lut_s, a.scale, a.minv);
        tw[(q / CPR) * P + (q % CPR) * DE + e] = in ? v : V(0);
      }
    }
    // one wave's LDS operations complete in order: its tile is whole before
    // it is read, and read before the next stage overwrites it
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < KR; ++q) {
      const bool in = whole || k0 + KR * h + q < a.K;
      const double bv = (double)tw[(KR * h + q) * P + j];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? (double)x[t][q] : 0.0, bv, acc[t], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  ragged_sum<MT, 1>(ex, acc, nw, [&](int mt, int, int i, int jj, double s) {
    const int m = m0 + 16 * mt + i, n = n0 + jj;
    if (m >= a.M || n >= a.N) return;
    const int64_t idx = (int64_t)m * a.N + n;
    float v = (float)s;
    if (next_pre != nullptr) v = v * act_prime_piecewise(next_pre[idx], next_act);
    out[idx] = v;
  });
}

RaggedArgs ragged_args(const DevStore &w, const float *A, int M, int K, int N, int f) {
  return RaggedArgs{kernel_body(w, f), w.lut, w.scale, w.minv, A, M, K, N, w.cols, 0, 0};
}

template <int F>
hipError_t ragged_forward(RaggedArgs a, const double *bias, int bias_len, int act, float *pre, float *post,
                          hipStream_t s) {
  // up to 4 rows as row products; from 8 M weights on the MFMA reads them at
  // least as fast (4095^2 Int8 b2 / b4 17.3 / 17.5 us against 18.1 / 22.7).  5
  // to 8 rows as two halves where K is long: the MFMA's one chain per 16 x 16
  // outputs is then the time (Float32 4095 -> 100 b5 17.3 us against 5.1, 4095
  // -> 1000 b8 18.4 / 11.5; 2047^2 b8 stays on it, 11.2 us), from 512 on for
  // Complex64, whose loads there are strided (1001 -> 777 b5 9.7 / 6.1).
  const bool few = (int64_t)a.K * a.N <= ((int64_t)8 << 20);
  if (a.M == 1 || (a.M <= 4 && few) || (a.M <= 8 && few && a.K >= (F == FC64 ? 512 : 3072))) {
    const int P = a.M == 1 ? ragged_piece<F, 1>() : 1;
    const int npieces = (a.K + P - 1) / P;
    const int S = npieces > 128 ? 4 : npieces > 64 ? 2 : 1;
    const dim3 blocks((a.N + 4 / S - 1) / (4 / S), a.M <= 4 ? 1 : 2);
    const int B = a.M <= 4 ? a.M : (a.M + 1) / 2;
    if (B == 1) ragged_gemv_kernel<F, 1><<<blocks, 256, 0, s>>>(a, S, bias, bias_len, act, pre, post);
    else if (B == 2) ragged_gemv_kernel<F, 2><<<blocks, 256, 0, s>>>(a, S, bias, bias_len, act, pre, post);
    else if (B == 3) ragged_gemv_kernel<F, 3><<<blocks, 256, 0, s>>>(a, S, bias, bias_len, act, pre, post);
    else ragged_gemv_kernel<F, 4><<<blocks, 256, 0, s>>>(a, S, bias, bias_len, act, pre, post);
    return hipGetLastError();
  }
  a.nst = (a.K + RaggedShape<F>::ST - 1) / RaggedShape<F>::ST;
  // 32 x 32 outputs per block where that still fills the CUs (each load then
  // feeds two tiles), else 16 x 16 on twice the waves
  const int gx32 = (a.N + 31) / 32, gy32 = (a.M + 31) / 32;
  if ((int64_t)gx32 * gy32 >= num_cus()) {
    a.gx = gx32;
    ragged_gemm_kernel<F, 2, 2, 4><<<gx32 * gy32, 64 * std::min(4, a.nst), 0, s>>>(a, bias, bias_len, act, pre, post);
  } else {
    a.gx = (a.N + 15) / 16;
    ragged_gemm_kernel<F, 1, 1, 8><<<a.gx * ((a.M + 15) / 16), 64 * std::min(8, a.nst), 0, s>>>(a, bias, bias_len,
                                                                                               act, pre, post);
  }
  return hipGetLastError();
}

// dX of few terms or few outputs, bound by the launch and one load chain: L
// lanes (1 or 64) per output walk the rows of W, one code each.
template <int F, int L>
__global__ void __launch_bounds__(256) ragged_dx_few_kernel(RaggedArgs a, float *out, const float *next_pre,
                                                            int next_act) {
  using I = FI<F>;
  __shared__ __align__(16) float lut_s[I::kTable];
  const int tid = threadIdx.x;
  if constexpr (I::kLut) {
    TabCopy<F> tab;
    tab.load(a.lut, tid);
    tab.store(lut_s, tid);
    __syncthreads();
  }
  const int total = a.M * a.N, q = blockIdx.x * (256 / L) + tid / L, qc = min(q, total - 1);
  const int m = qc / a.N, i = qc % a.N;
  double s = 0.0;
#pragma unroll 4
  for (int o = tid % L; o < a.K; o += L) {
    uint32_t w[I::kW];
    load_chunk_at<F, 1>(a.body, (int64_t)o * a.cols + i, w);
    s = fma((double)chunk_value<F>(w, 0, lut_s, a.scale, a.minv), (double)a.A[(int64_t)m * a.K + o], s);
  }
  if constexpr (L > 1) s = wave_sum(s);
  if (q < total && tid % L == 0) {
    float v = (float)s;
    if (next_pre != nullptr) v = v * act_prime_piecewise(next_pre[q], next_act);
    out[q] = v;
  }
}

template <int F>
hipError_t ragged_dx(RaggedArgs a, float *dX, const float *next_pre, int next_act, hipStream_t s) {
  // up to 16 terms (a quarter of a stage) or 1024 outputs: the MFMA kernel's
  // staging and exchange are most of its time (Float32 10 rows of 777 b8 4.0
  // us, 3.2 here; 777 rows of 10 b8 5.4 / 4.5)
  const int64_t total = (int64_t)a.M * a.N;
  if (a.K <= 16 && total <= 65536) {
    ragged_dx_few_kernel<F, 1><<<(int)((total + 255) / 256), 256, 0, s>>>(a, dX, next_pre, next_act);
    return hipGetLastError();
  }
  if (total <= 1024) {
    ragged_dx_few_kernel<F, 64><<<(int)((total + 3) / 4), 256, 0, s>>>(a, dX, next_pre, next_act);
    return hipGetLastError();
  }
  a.nst = (a.K + RaggedTShape<F>::ST - 1) / RaggedTShape<F>::ST;
  a.gx = (a.N + 15) / 16;
  const int gy32 = (a.M + 31) / 32;
  if ((int64_t)a.gx * gy32 >= 2 * num_cus())
    ragged_dx_kernel<F, 2, 4><<<a.gx * gy32, 64 * std::min(4, a.nst), 0, s>>>(a, dX, next_pre, next_act);
  else
    ragged_dx_kernel<F, 1, 8><<<a.gx * ((a.M + 15) / 16), 64 * std::min(8, a.nst), 0, s>>>(a, dX, next_pre, next_act);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_ragged_forward(const DevStore &w, int batch, const float *x, const double *bias, int bias_len,
                                 int act, float *pre, float *post, hipStream_t s) {
  const int f = kernel_fmt(w.dtype);
  if (kernel_body(w, f) == nullptr) return hipErrorInvalidValue;
  const RaggedArgs a = ragged_args(w, x, batch, w.cols, w.rows, f);
#define WH_RF(F) return ragged_forward<F>(a, bias, bias_len, act, pre, post, s);
  WH_FMT_SWITCH(f, WH_RF)
#undef WH_RF
}

hipError_t launch_ragged_dx(const DevStore &w, int batch, const float *dpre, float *dX, const float *next_pre,
                            int next_act, hipStream_t s) {
  const int f = kernel_fmt(w.dtype);
  if (kernel_body(w, f) == nullptr) return hipErrorInvalidValue;
  const RaggedArgs a = ragged_args(w, dpre, batch, w.rows, w.cols, f);
#define WH_RD(F) return ragged_dx<F>(a, dX, next_pre, next_act, s);
  WH_FMT_SWITCH(f, WH_RD)
#undef WH_RD
}

}  // namespace wh
