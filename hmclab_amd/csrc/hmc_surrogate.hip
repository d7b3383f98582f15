// Learned surrogate potential for the trajectory: an MLP
//   f(x) = w3 . silu(W2 silu(W1 xn + b1) + b2) + b3,   xn = (x - x_mean) / x_scale
// modelling the likelihood misfit (chi_lik ~ f_mean + f_scale * f).  Its input
// gradient drives the leapfrog; the Metropolis test keeps the exact FP64
// Hamiltonian, so the chain targets the exact posterior.  FP32 master
// weights; GEMMs on bf16 MFMA (or FP32 SIMT for checks); training minimises
//   alpha (f - y)^2 + beta/D ||grad f - t||^2
// with hand-written double backpropagation and Adam (Kingma & Ba 2015).
#include <algorithm>
#include <numeric>
#include <random>
#include <type_traits>
#include <vector>

#include "hmc_internal.hpp"

struct hmc_surrogate;

namespace hmc {

// ---------------------------------------------------------------------------
// FP32 GEMM (mode f32): C[m][n] = alpha * sum_k A(m,k) B(n,k) + beta * C[m][n]
//   A(m,k) = TA ? A[k*lda + m] : A[m*lda + k];  B(n,k) = TB ? B[k*ldb + n] : B[n*ldb + k]
// 64x64x32 tiles, 256 threads; dimensions must be multiples of the tile (the
// surrogate pads every dimension to 64).
// ---------------------------------------------------------------------------
constexpr int SG_T = 64, SG_K = 32;

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_sgemm(const float* __restrict__ A, int64_t lda,
                                               const float* __restrict__ B, int64_t ldb,
                                               float* __restrict__ C, int64_t ldc, int K,
                                               float alpha, float beta) {
  __shared__ __attribute__((aligned(16))) float As[SG_T][SG_K + 1];
  __shared__ __attribute__((aligned(16))) float Bs[SG_T][SG_K + 1];
  const int tid = threadIdx.x;
  const int64_t m0 = (int64_t)blockIdx.y * SG_T, n0 = (int64_t)blockIdx.x * SG_T;
  // staging: 64 x 32 elements per operand, 8 per thread
  auto stage = [&](const float* __restrict__ P, int64_t ld, bool trans, int64_t r0, int k0,
                   float (*S)[SG_K + 1]) {
    if (!trans) {
      const int r = tid >> 2, kk = (tid & 3) * 8;
      const float* src = P + (r0 + r) * ld + k0 + kk;
#pragma unroll
      for (int e = 0; e < 8; ++e) S[r][kk + e] = src[e];
    } else {
      const int kk = tid >> 3, r = (tid & 7) * 8;
      const float* src = P + (int64_t)(k0 + kk) * ld + r0 + r;
#pragma unroll
      for (int e = 0; e < 8; ++e) S[r + e][kk] = src[e];
    }
  };
  // each thread a 4 x 4 micro tile
  const int tm = (tid >> 4) * 4, tn = (tid & 15) * 4;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += SG_K) {
    __syncthreads();
    stage(A, lda, TA, m0, k0, As);
    stage(B, ldb, TB, n0, k0, Bs);
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < SG_K; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += As[tm + i][k] * Bs[tn + j][k];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float* cp = C + (m0 + tm + i) * ldc + n0 + tn + j;
      *cp = alpha * acc[i][j] + (beta != 0.f ? beta * *cp : 0.f);
    }
}

// ---------------------------------------------------------------------------
// element-wise pieces
// ---------------------------------------------------------------------------
__device__ inline float sig(float z) { return 1.f / (1.f + __expf(-z)); }
__device__ inline float silu_f(float z) { return z * sig(z); }
__device__ inline float dsilu_f(float z) {
  const float s = sig(z);
  return s * (1.f + z * (1.f - s));
}
__device__ inline float d2silu_f(float z) {
  const float s = sig(z);
  return s * (1.f - s) * (2.f + z * (1.f - 2.f * s));
}

// Z += bias; A = silu(Z); S = silu'(Z)   over [rows][H]
__global__ void k_act(float* Z, float* Aout, float* S, const float* bias, int64_t rows, int H) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * H) return;
  const float z = Z[i] + bias[i % H];
  Z[i] = z;
  Aout[i] = silu_f(z);
  S[i] = dsilu_f(z);
}

// f[b] = A2[b].w3 + b3 ; U2 = S2 * w3      (one block of 256 per row)
__global__ void k_head(const float* A2, const float* S2, const float* w3, const float* b3, float* U2,
                       float* f, int H) {
  __shared__ float red[256];
  const int64_t b = blockIdx.x;
  float acc = 0.f;
  for (int i = threadIdx.x; i < H; i += 256) {
    acc += A2[b * H + i] * w3[i];
    U2[b * H + i] = S2[b * H + i] * w3[i];
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) f[b] = red[0] + b3[0];
}

__global__ void k_mul(float* out, const float* a, const float* b, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = a[i] * b[i];
}

// normalise chain rows (state dtype, stride ldx) into Xn [rows][Dp] (zero padded)
template <typename T>
__global__ void k_norm(const T* X, int64_t ldx, float* Xn, int64_t Dp, int64_t D, const float* xm,
                       const float* xs, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * Dp) return;
  const int64_t b = i / Dp, j = i % Dp;
  Xn[i] = (j < D) ? ((float)X[b * ldx + j] - xm[j]) / xs[j] : 0.f;
}

// surrogate kick + drift: g = G[b][j] * gscale_j + prior'(x); then as EpiLeap
template <typename T>
__global__ void k_sur_leap(T* x, T* p, int64_t ldx, const float* G, int64_t Dp, int64_t D,
                           const float* gscale, const double* eps, const double* beta, double kick,
                           double drift, double drift2, int64_t rows, DevModel md) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * D) return;
  const int64_t b = i / D, j = i % D;
  const double e = eps[b];
  const double ke = beta ? kick * e * beta[b] : kick * e;
  const int64_t o = b * ldx + j;
  T xv = x[o], pv = p[o];
  T g = (T)(G[b * Dp + j] * gscale[j]) + prior_grad<T>(md, j, xv);
  if (out_of_bounds(md, j, (double)xv)) g = (T)INFINITY;
  pv -= (T)ke * g;
  xv += (T)(drift * e) * kgrad<T>(md, j, pv);
  corrector<T>(md, j, xv, pv);
  if (drift2 != 0.0) {
    xv += (T)(drift2 * e) * kgrad<T>(md, j, pv);
    corrector<T>(md, j, xv, pv);
  }
  x[o] = xv;
  p[o] = pv;
}

// training-batch targets: r = f - y ; df = 2 alpha r / Bt ; E = G - T ; dG = 2 beta/D E / Bt;
// loss partial per row
__global__ void k_residuals(const float* f, const float* y, const float* G, const float* Tg,
                            float* df, float* dG, float* lrow, int64_t Dp, int64_t D, float alpha,
                            float beta, int Bt) {
  __shared__ float red[256];
  const int64_t b = blockIdx.x;
  float acc = 0.f;
  for (int64_t j = threadIdx.x; j < Dp; j += 256) {
    const float e = (j < D) ? G[b * Dp + j] - Tg[b * Dp + j] : 0.f;
    dG[b * Dp + j] = 2.f * beta / (float)D * e / (float)Bt;
    acc += e * e;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float r = f[b] - y[b];
    df[b] = 2.f * alpha * r / (float)Bt;
    lrow[b] = alpha * r * r + beta / (float)D * red[0];
  }
}

// dS = dU * V ; dV = dU * S   (in place: dU -> dV, out dS)
__global__ void k_split(const float* dU, const float* V, const float* S, float* dS, float* dV, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  dS[i] = dU[i] * V[i];
  dV[i] = dU[i] * S[i];
}

// dZ2 = dU2*w3 * silu''(Z2) + df (x) w3 * S2 ; also dw3 partial pieces handled by k_colsum
__global__ void k_dz2(const float* dU2, const float* w3, const float* Z2, const float* S2,
                      const float* df, float* dZ2, int64_t rows, int H) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * H) return;
  const int64_t b = i / H;
  const int h = (int)(i % H);
  dZ2[i] = dU2[i] * w3[h] * d2silu_f(Z2[i]) + df[b] * w3[h] * S2[i];
}

// dZ1 = dS1 * silu''(Z1) + dA1 * S1
__global__ void k_dz1(const float* dS1, const float* Z1, const float* dA1, const float* S1, float* dZ1,
                      int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dZ1[i] = dS1[i] * d2silu_f(Z1[i]) + dA1[i] * S1[i];
}

// out[h] = sum_b X[b][h] * (Y ? Y[b][h] : 1) (+ sum_b w[b] * W[b][h])   fixed order
__global__ void k_colsum(const float* X, const float* Y, const float* wv, const float* Wm, float* out,
                         int64_t rows, int H) {
  const int h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= H) return;
  float acc = 0.f;
  for (int64_t b = 0; b < rows; ++b) {
    acc += X[b * H + h] * (Y ? Y[b * H + h] : 1.f);
    if (wv) acc += wv[b] * Wm[b * H + h];
  }
  out[h] = acc;
}

__global__ void k_sum(const float* v, int64_t n, float* out) {
  __shared__ float red[256];
  float acc = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += 256) acc += v[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// Adam step of parameter i with gradient gi; returns the new value
struct AdamStep {
  float *w, *m, *v;
  float lr, b1, b2, c1, c2, eps;
  // moments and value wo, mo, vo as loaded by the caller
  __device__ __forceinline__ float apply(int64_t i, float gi, float wo, float mo, float vo) const {
    const float mi = b1 * mo + (1.f - b1) * gi;
    const float vi = b2 * vo + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = wo - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    return wi;
  }
  __device__ __forceinline__ float apply(int64_t i, float gi) const { return apply(i, gi, w[i], m[i], v[i]); }
};

__global__ void k_adam(AdamStep a, const float* g, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a.apply(i, g[i]);
}

// gather normalised training rows: Xn[b] = X[idx[b]], Tn[b] = T[idx[b]], yb[b] = y[idx[b]]
__global__ void k_gather(const float* Xall, const float* Tall, const float* yall, const int32_t* idx,
                         float* Xn, float* Tn, float* yb, int64_t Dp, int64_t rows) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * Dp) return;
  const int64_t b = i / Dp, j = i % Dp;
  const int64_t src = (int64_t)idx[b] * Dp + j;
  Xn[i] = Xall[src];
  Tn[i] = Tall[src];
  if (j == 0) yb[b] = yall[idx[b]];
}

// ---------------------------------------------------------------------------
// bf16 products of the evaluation and training passes
//   C[m][n] = sum_k A[m][k] B[n][k]   (+ a second product, added after it)
// on bf16 planes whose rows are k-contiguous, FP32 accumulation in ascending k
// (v_mfma_f32_32x32x16_bf16, one 16-deep step after the other, so a result does
// not depend on the tile).  A block of WM x WN waves computes 32 WM x 32 WN
// outputs; its operand tiles stream global -> LDS with direct-to-LDS loads
// through an S-stage ring of 64-wide k-tiles, rows swizzled in 16-byte chunks
// by (row & 7).
//
// What bounds it: these products are small (256 x 512 outputs are 128 tiles of
// 32 x 32), so each block's chain of k-tiles and its loads in flight, not the
// matrix cores.  One wave per 32 x 32 tile keeps 7 k-tiles (56 KB) in flight
// and needs no barrier; in a long product a second wave issues all the loads, so
// the first runs only LDS reads and MFMAs; 64 x 64 blocks take the products with
// many outputs.  The fragments of a k-tile are read while the MFMAs of the one
// before run, and the two products of a weight gradient are two loops (a test
// per k-tile made the accumulators travel through plain registers).
// 256 x 512 x 8192: 30 us (194 us with 64 x 64 tiles staged through registers as
// float32); 256 x 512 x 512: 7 us (15 us).
// ---------------------------------------------------------------------------
#define HMC_LDS __attribute__((address_space(3)))

template <int N>
__device__ inline void sur_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt out of range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}

struct SurOperands {
  const uint16_t *a = nullptr, *b = nullptr;
  int64_t lda = 0, ldb = 0;
  int K = 0;
};

template <int WM, int WN, int LW, int S, class Epi>
__global__ __launch_bounds__((WM * WN + LW) * 64) void k_sur_gemm(SurOperands p0, SurOperands p1, int gm, int gn,
                                                                  Epi epi) {
  constexpr int BK = 64, CW = WM * WN, NW = CW + LW, BM = 32 * WM, BN = 32 * WN;
  constexpr int NL = LW > 0 ? LW : CW;   // waves that load
  constexpr int A_GROUPS = BM / 8, GROUPS = (BM + BN) / 8, GPW = GROUPS / NL;   // 1 KB loads
  constexpr int STAGE = (BM + BN) * BK;
  static_assert(GROUPS % NL == 0 && GPW * (S - 2) < 64, "load groups");
  __shared__ __attribute__((aligned(1024))) uint16_t smem[S * STAGE];

  // tiles dealt to the XCDs in contiguous n-major ranges (an XCD reads its own
  // rows of B and all of the smaller A)
  const int T = gm * gn, chunk = (T + 7) / 8, t = ((int)blockIdx.x % 8) * chunk + (int)blockIdx.x / 8;
  if (t >= T) return;
  const int64_t m_blk = (int64_t)(t % gm) * BM, n_blk = (int64_t)(t / gm) * BN;
  const int tid = threadIdx.x, lane = tid & 63, w = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool loader = LW == 0 || w >= CW, computes = LW == 0 || w < CW;
  const int lw = LW > 0 ? w - CW : w;    // index among the loading waves
  const int wm = w / WN, wn = w % WN;
  const int q = lane >> 5, r = lane & 31, lrow = lane >> 3;

  // this lane's source of each of the wave's load groups, advanced per k-tile
  const int nk0 = p0.K / BK, nk = nk0 + p1.K / BK;
  const uint16_t* src[GPW];
  auto aim = [&](const SurOperands& p) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < GPW; ++i) {
      const int g = lw * GPW + i;
      const bool is_a = g < A_GROUPS;
      const int row = (is_a ? g : g - A_GROUPS) * 8 + lrow;
      const uint16_t* base = is_a ? p.a : p.b;
      const int64_t at = is_a ? (m_blk + row) * p.lda : (n_blk + row) * p.ldb;
      src[i] = base + at + ((lane & 7) ^ (row & 7)) * 8;
    }
  };
  auto issue = [&](int kt, int st) __attribute__((always_inline)) {
    if (kt == nk0) aim(p1);
    uint16_t* stage = smem + st * STAGE;
#pragma unroll
    for (int i = 0; i < GPW; ++i) {
      __builtin_amdgcn_global_load_lds((const void*)src[i], (HMC_LDS void*)(stage + (lw * GPW + i) * 8 * BK), 16, 0, 0);
      src[i] += BK;
    }
  };
  if (loader) {
    aim(p0);
#pragma unroll
    for (int s0 = 0; s0 < S - 1; ++s0)
      if (s0 < nk) issue(s0, s0);
  }
  floatx16 acc, first;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = first[v] = 0.f;
  bf16x8 af[2][4] = {}, bf[2][4] = {};
  const int ra = wm * 32 + r, rb = wn * 32 + r;
  auto mfmas = [&](auto set) __attribute__((always_inline)) {
    constexpr int p = decltype(set)::value;
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[p][s], bf[p][s], acc, 0, 0, 0);
  };
  // k-tile kt with its fragments in set p; the MFMAs of the k-tile before it
  // (set 1 - p, unless kt is the product's first) run while they are read
  auto tile = [&](int kt, auto set, auto is_first) __attribute__((always_inline)) {
    constexpr int p = decltype(set)::value;
    if (loader) {
      if (kt + S - 2 < nk) sur_wait_vmcnt<GPW * (S - 2)>();
      else sur_wait_vmcnt<0>();
    }
    // this wave's LDS reads of the stage about to be refilled have returned
    // (naming the fragments keeps the compiler from moving their reads past
    // this point); with several waves, all of them have passed the barrier
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(af[1 - p][0]), "+v"(af[1 - p][1]), "+v"(af[1 - p][2]), "+v"(af[1 - p][3]), "+v"(bf[1 - p][0]),
                   "+v"(bf[1 - p][1]), "+v"(bf[1 - p][2]), "+v"(bf[1 - p][3])
                 :
                 : "memory");
    if constexpr (NW > 1) {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (computes) {
      const uint16_t* As = smem + (kt % S) * STAGE;
      const uint16_t* Bs = As + BM * BK;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int c = 2 * s + q;   // k = 16 s + 8 q + e
        af[p][s] = *reinterpret_cast<const bf16x8*>(&As[ra * BK + ((c ^ (ra & 7)) << 3)]);
        bf[p][s] = *reinterpret_cast<const bf16x8*>(&Bs[rb * BK + ((c ^ (rb & 7)) << 3)]);
      }
      if constexpr (!decltype(is_first)::value) mfmas(std::integral_constant<int, 1 - p>{});
    }
    if (loader && kt + S - 1 < nk) issue(kt + S - 1, (kt + S - 1) % S);
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  auto product = [&](int kt, int end) __attribute__((always_inline)) {
    tile(kt, Set0{}, std::true_type{});
    for (++kt; kt + 2 <= end; kt += 2) {
      tile(kt, Set1{}, std::false_type{});
      tile(kt + 1, Set0{}, std::false_type{});
    }
    if (kt < end) {
      tile(kt, Set1{}, std::false_type{});
      if (computes) mfmas(Set1{});
    } else if (computes) {
      mfmas(Set0{});
    }
  };
  product(0, nk0);
  if (nk > nk0) {
    first = acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    product(nk0, nk);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = acc[v] + first[v];
  }
  if (!computes) return;
  // lane (q, r) holds rows 8 g + 4 q + v (g, v = 0..3) of column r
  epi.apply(m_blk + wm * 32, 4 * q, n_blk + wn * 32 + r, acc);
}

// the lane's 16 values of src at rows b0 + 8 g + q4 + v of column h, loaded
// before an epilogue's first store (a store between them would order them)
__device__ __forceinline__ floatx16 load16(const float* src, int64_t b0, int q4, int64_t h, int64_t ld) {
  floatx16 o;
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = src[(b0 + 8 * (i / 4) + q4 + i % 4) * ld + h];
  return o;
}

// 4 consecutive batch rows of one column as bf16: the transposed plane's 8-byte
// store
__device__ __forceinline__ void put_t4(uint16_t* pT, int64_t o, const float v[4]) {
  const uint32_t h0 = f32_to_bf16_bits(v[0]), h1 = f32_to_bf16_bits(v[1]), h2 = f32_to_bf16_bits(v[2]),
                 h3 = f32_to_bf16_bits(v[3]);
  *reinterpret_cast<uint2*>(&pT[o]) = uint2{h0 | (h1 << 16), h2 | (h3 << 16)};
}

// Epilogues: m = batch row b, n = column; rows b0 + 8 g + q4 + v.

// Z1 = acc + b1; A1 = silu(Z1), S1 = silu'(Z1)
struct SurZ1 {
  const float* bias;
  float *z, *s;
  uint16_t *a, *aT;   // aT may be null (evaluation)
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const float bh = bias[h];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float av[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        const float zz = acc[4 * g + v] + bh;
        z[o] = zz;
        s[o] = dsilu_f(zz);
        av[v] = silu_f(zz);
        a[o] = f32_to_bf16_bits(av[v]);
      }
      if (aT) put_t4(aT, h * R + b0 + 8 * g + q4, av);
    }
  }
};

// Z2 = acc + b2; A2 = silu(Z2), S2 = silu'(Z2), U2 = S2 w3
struct SurZ2 {
  const float *bias, *w3;
  float *z, *a, *s;
  uint16_t *u, *uT;
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const float bh = bias[h], wh = w3[h];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float uv[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        const float zz = acc[4 * g + v] + bh;
        z[o] = zz;
        a[o] = silu_f(zz);
        const float ss = dsilu_f(zz);
        s[o] = ss;
        uv[v] = ss * wh;
        u[o] = f32_to_bf16_bits(uv[v]);
      }
      if (uT) put_t4(uT, h * R + b0 + 8 * g + q4, uv);
    }
  }
};

// V1 = acc; U1 = S1 V1
struct SurV1 {
  const float* s1;
  float* v1;
  uint16_t *u, *uT;
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const floatx16 ss = load16(s1, b0, q4, h, H);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float uv[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        v1[o] = acc[4 * g + v];
        uv[v] = ss[4 * g + v] * acc[4 * g + v];
        u[o] = f32_to_bf16_bits(uv[v]);
      }
      if (uT) put_t4(uT, h * R + b0 + 8 * g + q4, uv);
    }
  }
};

// input gradient of the evaluation: out[b][j] = acc gscale_j (raw units, FP64)
struct SurEvalGrad {
  const float* gscale;
  double* out;
  int64_t D, B;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t j, const floatx16& acc) const {
    if (j >= D) return;
    const double gs = (double)gscale[j];
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t b = b0 + 8 * g + q4 + v;
        if (b < B) out[b * D + j] = (double)acc[4 * g + v] * gs;
      }
  }
};

// training: E = acc - t, dG = 2 beta / D E / R, tile sums of E^2 per batch row
struct SurResid {
  const float* t;        // [.][Dp], row idx[b]
  const int32_t* idx;    // or null: row b
  uint16_t *dg, *dgT;
  float* lpart;          // [Dp / 32][R]
  int64_t D, Dp, R;
  float beta;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t j, const floatx16& acc) const {
    const int r = threadIdx.x & 31;
    float tt[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int64_t b = b0 + 8 * (i / 4) + q4 + i % 4;
      tt[i] = t[(idx ? idx[b] : b) * Dp + j];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float dv[4], e2[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t b = b0 + 8 * g + q4 + v;
        const float e = (j < D) ? acc[4 * g + v] - tt[4 * g + v] : 0.f;
        dv[v] = 2.f * beta / (float)D * e / (float)R;
        e2[v] = e * e;
        dg[b * Dp + j] = f32_to_bf16_bits(dv[v]);
      }
      put_t4(dgT, j * R + b0 + 8 * g + q4, dv);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) e2[v] += __shfl_xor(e2[v], off, 32);
        if (r == 0) lpart[(j / 32) * R + b0 + 8 * g + q4 + v] = e2[v];
      }
    }
  }
};

// dU1 = acc; dS1 = dU1 V1, dV1 = dU1 S1
struct SurDU1 {
  const float *v1, *s1;
  float* ds1;
  uint16_t *dv, *dvT;
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const floatx16 vv = load16(v1, b0, q4, h, H), ss = load16(s1, b0, q4, h, H);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float dd[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        ds1[o] = acc[4 * g + v] * vv[4 * g + v];
        dd[v] = acc[4 * g + v] * ss[4 * g + v];
        dv[o] = f32_to_bf16_bits(dd[v]);
      }
      put_t4(dvT, h * R + b0 + 8 * g + q4, dd);
    }
  }
};

// dU2 = acc; dZ2 = dU2 w3 silu''(Z2) + df w3 S2
struct SurDU2 {
  const float *w3, *z2, *s2, *df;
  float *du, *dzf;
  uint16_t *dz, *dzT;
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const floatx16 zz = load16(z2, b0, q4, h, H), ss = load16(s2, b0, q4, h, H), dfb = load16(df, b0, q4, 0, 1);
    const float wh = w3[h];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float dd[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 4 * g + v;
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        du[o] = acc[i];
        dd[v] = acc[i] * wh * d2silu_f(zz[i]) + dfb[i] * wh * ss[i];
        dzf[o] = dd[v];
        dz[o] = f32_to_bf16_bits(dd[v]);
      }
      put_t4(dzT, h * R + b0 + 8 * g + q4, dd);
    }
  }
};

// dA1 = acc; dZ1 = dS1 silu''(Z1) + dA1 S1
struct SurDA1 {
  const float *ds1, *z1, *s1;
  float* dzf;
  uint16_t* dzT;
  int64_t H, R;
  __device__ __forceinline__ void apply(int64_t b0, int q4, int64_t h, const floatx16& acc) const {
    const floatx16 dd1 = load16(ds1, b0, q4, h, H), zz = load16(z1, b0, q4, h, H), ss = load16(s1, b0, q4, h, H);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float dd[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 4 * g + v;
        const int64_t o = (b0 + 8 * g + q4 + v) * H + h;
        dd[v] = fmaf(acc[i], ss[i], dd1[i] * d2silu_f(zz[i]));
        dzf[o] = dd[v];
      }
      put_t4(dzT, h * R + b0 + 8 * g + q4, dd);
    }
  }
};

// weight gradient W[m][n] (m = hidden unit, n = input): stored, or (training)
// the Adam step and the new weight's planes [m][n] and [n][m]
struct SurWeight {
  float* g;            // gradient, or null: Adam
  AdamStep adam;
  int64_t off;         // of the matrix in the packed parameters
  uint16_t *h, *t;     // planes
  int64_t ld, ldt;     // row strides of W (and plane h) and of plane t
  __device__ __forceinline__ void apply(int64_t m0, int q4, int64_t n, const floatx16& acc) const {
    if (g) {
#pragma unroll
      for (int i = 0; i < 16; ++i) g[off + (m0 + 8 * (i / 4) + q4 + i % 4) * ld + n] = acc[i];
      return;
    }
    const floatx16 wo = load16(adam.w + off, m0, q4, n, ld), mo = load16(adam.m + off, m0, q4, n, ld),
                   vo = load16(adam.v + off, m0, q4, n, ld);
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      float wv[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int i = 4 * gq + v;
        const int64_t o = (m0 + 8 * gq + q4 + v) * ld + n;
        wv[v] = adam.apply(off + o, acc[i], wo[i], mo[i], vo[i]);
        h[o] = f32_to_bf16_bits(wv[v]);
      }
      put_t4(t, n * ldt + m0 + 8 * gq + q4, wv);
    }
  }
};

// f[b] = A2[b] . w3 + b3 (fixed tree); df = 2 alpha (f - y) / R when training
__global__ void k_sur_head(const float* a2, const float* w3, const float* b3, const float* y, const int32_t* idx,
                           float alpha, float* f, float* df, int H, int R) {
  __shared__ float red[256];
  const int64_t b = blockIdx.x;
  float acc = 0.f;
  for (int i = threadIdx.x; i < H; i += 256) acc += a2[b * H + i] * w3[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const float fv = red[0] + b3[0];
    f[b] = fv;
    if (df) df[b] = 2.f * alpha * (fv - y[idx ? idx[b] : b]) / (float)R;
  }
}

// e2[b] = sum over the column tiles of lpart[tile][b]: 32 batch rows per block,
// 8 threads each
__global__ __launch_bounds__(256) void k_sur_e2(const float* __restrict__ lpart, int tiles, int R,
                                                float* __restrict__ e2) {
  __shared__ float red[8][32];
  const int b = threadIdx.x & 31, k = threadIdx.x >> 5;
  float s = 0.f;
#pragma unroll 8
  for (int t = k; t < tiles; t += 8) s += lpart[(int64_t)t * R + blockIdx.x * 32 + b];
  red[k][b] = s;
  __syncthreads();
  if (k == 0) {
    for (int i = 1; i < 8; ++i) s += red[i][b];
    e2[blockIdx.x * 32 + b] = s;
  }
}

// Column sums over the batch in row order, 32 rows of loads ahead of their
// sums: block (x, 0) dw3 = sum_b dU2 S2 + df A2, (x, 1) db2 = sum_b dZ2, (x, 2)
// db1 = sum_b dZ1; block (0, 3) db3 = sum_b df and the batch loss
// sum_b alpha r^2 + beta / D sum E^2 (e2: k_sur_e2's sums).  Gradients are stored (g) or take their
// Adam step (g null).  One column per thread and 64 columns per block: the sums
// are serial chains, so the loads in flight bound them (256 rows of 512
// columns: 31 us per sum with 256-column blocks and a load per step).
struct SurFinish {
  const float *du2, *s2, *a2, *dz2, *dz1, *e2, *f, *y, *df;
  const int32_t* idx;
  float* g;
  AdamStep adam;
  int64_t ow3, ob2, ob1, ob3;
  float* loss;
  int H, R, D;
  float alpha, beta;
};
__global__ __launch_bounds__(64) void k_sur_finish(SurFinish p) {
  constexpr int U = 32;
  auto put = [&](int64_t o, float v) {
    if (p.g) p.g[o] = v;
    else p.adam.apply(o, v);
  };
  const int h = blockIdx.x * 64 + threadIdx.x, which = blockIdx.y;
  if (which < 3) {   // H and R are multiples of 64
    float acc = 0.f;
    if (which == 0) {
      for (int b0 = 0; b0 < p.R; b0 += U) {
        float du[U], ss[U], aa[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t o = (int64_t)(b0 + u) * p.H + h;
          du[u] = p.du2[o];
          ss[u] = p.s2[o];
          aa[u] = p.a2[o];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          acc += du[u] * ss[u];
          acc += p.df[b0 + u] * aa[u];
        }
      }
      put(p.ow3 + h, acc);
    } else {
      const float* z = which == 1 ? p.dz2 : p.dz1;
      for (int b0 = 0; b0 < p.R; b0 += U) {
        float zz[U];
#pragma unroll
        for (int u = 0; u < U; ++u) zz[u] = z[(int64_t)(b0 + u) * p.H + h];
#pragma unroll
        for (int u = 0; u < U; ++u) acc += zz[u];
      }
      put((which == 1 ? p.ob2 : p.ob1) + h, acc);
    }
    return;
  }
  if (blockIdx.x != 0) return;
  // 256 strided sums, then a fixed tree
  __shared__ float red[2][256];
  for (int i = threadIdx.x; i < 256; i += 64) {
    float sd = 0.f, sl = 0.f;
    for (int b = i; b < p.R; b += 256) {
      const float r = p.f[b] - p.y[p.idx ? p.idx[b] : b];
      sd += p.df[b];
      sl += p.alpha * r * r + p.beta / (float)p.D * p.e2[b];
    }
    red[0][i] = sd;
    red[1][i] = sl;
  }
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    for (int i = threadIdx.x; i < s; i += 64) {
      red[0][i] += red[0][i + s];
      red[1][i] += red[1][i + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    put(p.ob3, red[0][0]);
    *p.loss = red[1][0];
  }
}

// bf16 planes of rows idx[b] (or b) of X [.][Dp]: x[b][j] and, transposed
// through LDS, xT[j][b].  One 64 x 64 tile per block.
__global__ __launch_bounds__(256) void k_sur_rows(const float* __restrict__ X, const int32_t* __restrict__ idx,
                                                  int64_t Dp, int64_t R, uint16_t* __restrict__ x,
                                                  uint16_t* __restrict__ xT) {
  __shared__ uint16_t tile[64][66];
  const int64_t j0 = (int64_t)blockIdx.x * 64, b0 = (int64_t)blockIdx.y * 64;
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
  float f[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int64_t b = b0 + r0 + 4 * k;
    f[k] = X[(idx ? idx[b] : b) * Dp + j0 + c];
  }
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int r = r0 + 4 * k;
    const uint16_t v = f32_to_bf16_bits(f[k]);
    x[(b0 + r) * Dp + j0 + c] = v;
    tile[c][r] = v;
  }
  if (!xT) return;
  __syncthreads();
  for (int r = r0; r < 64; r += 4) xT[(j0 + r) * R + b0 + c] = tile[r][c];
}

// parameters without W1's padding columns: W1 [H][D], then the rest
__global__ void k_sur_pack(const float* __restrict__ p, int64_t H, int64_t D, int64_t Dp, int64_t n,
                           float* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = i < H * D ? p[(i / D) * Dp + i % D] : p[i - H * D + H * Dp];
}

// host rows (f64 [n][D]) -> float32 [n][Dp], zero in the padding columns:
// mode 0 as given, 1 ((float)v - mean) / scale in float32, 2 (v - mean) / scale
// in FP64, 3 v scale / fs in FP64
__global__ void k_sur_load(const double* __restrict__ src, int64_t n, int64_t D, int64_t Dp,
                           const float* __restrict__ xm, const float* __restrict__ xs, double fs, int mode,
                           float* __restrict__ dst) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n * Dp; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / Dp, j = i % Dp;
    float o = 0.f;
    if (j < D) {
      const double v = src[b * D + j];
      if (mode == 0) o = (float)v;
      else if (mode == 1) o = ((float)v - xm[j]) / xs[j];
      else if (mode == 2) o = (float)((v - (double)xm[j]) / (double)xs[j]);
      else o = (float)(v * (double)xs[j] / fs);
    }
    dst[i] = o;
  }
}

// ---------------------------------------------------------------------------
// host object
// ---------------------------------------------------------------------------
// Buffers of the bf16 evaluation and training passes, for up to `rows` rows
struct TrainBufs {
  int64_t rows = 0;
  // operand planes: [b][k] and transposed [k][b] (suffix T)
  uint16_t *x = nullptr, *xT = nullptr, *dg = nullptr, *dgT = nullptr, *a1 = nullptr, *a1T = nullptr, *u2 = nullptr,
           *u2T = nullptr, *u1 = nullptr, *u1T = nullptr, *dv1 = nullptr, *dv1T = nullptr, *dz2 = nullptr,
           *dz2T = nullptr, *dz1T = nullptr;
  float *z1 = nullptr, *s1 = nullptr, *z2 = nullptr, *a2 = nullptr, *s2 = nullptr, *v1 = nullptr, *ds1 = nullptr,
        *du2 = nullptr, *dz2f = nullptr, *dz1f = nullptr;
  float *f = nullptr, *df = nullptr, *e2 = nullptr;
  float* lpart = nullptr;   // [Dp / 32][rows] sums of (grad f - t)^2
};

struct Surrogate {
  TrainBufs tb;
  int64_t D = 0, Dp = 0, H = 0;
  int mode = 0;                  // 0 bf16 MFMA, 1 fp32 SIMT
  hipStream_t stream = nullptr;
  std::vector<void*> owned;
  // parameters (packed: W1 | b1 | W2 | b2 | w3 | b3) and Adam moments
  float* P = nullptr;
  float* Pm = nullptr;
  float* Pv = nullptr;
  float* dP = nullptr;
  int64_t nP = 0, oW1 = 0, ob1 = 0, oW2 = 0, ob2 = 0, ow3 = 0, ob3 = 0;
  int64_t adam_t = 0;
  // normalisation
  float* xm = nullptr;
  float* xs = nullptr;
  float* gscale = nullptr;      // f_scale / x_scale
  float* xsinv = nullptr;       // 1 / x_scale
  double f_mean = 0.0, f_scale = 1.0;
  // work buffers for up to Bmax rows
  int64_t Bmax = 0;
  float *Xn = nullptr, *Z1 = nullptr, *A1 = nullptr, *S1 = nullptr, *Z2 = nullptr, *A2 = nullptr,
        *S2 = nullptr, *U2 = nullptr, *V1 = nullptr, *U1 = nullptr, *G = nullptr, *f = nullptr;
  float *Tn = nullptr, *yb = nullptr, *df = nullptr, *dG = nullptr, *dU1 = nullptr, *dS1 = nullptr,
        *dV1 = nullptr, *dU2 = nullptr, *dZ2 = nullptr, *dA1 = nullptr, *dZ1 = nullptr, *lrow = nullptr,
        *scal = nullptr;
  int32_t* idx = nullptr;
  // bf16 MFMA trajectory stage: weight planes (rebuilt when the parameters
  // change) and per-stage operands for up to Bh rows
  uint16_t *w1h = nullptr, *w1t = nullptr, *w2h = nullptr, *w2t = nullptr;
  bool planes_ok = false;
  int64_t Bh = 0;
  uint16_t *xh = nullptr, *a1h = nullptr, *u2h = nullptr, *u1h = nullptr;
  float* s1h = nullptr;
  const void* planes_for = nullptr;   // chain set whose positions xh holds
  float* ws = nullptr;
  size_t ws_elems = 0;

  float* W1() { return P + oW1; }
  float* b1() { return P + ob1; }
  float* W2() { return P + oW2; }
  float* b2() { return P + ob2; }
  float* w3() { return P + ow3; }
  float* b3() { return P + ob3; }
};

// float32 mode: full-precision copies of every intermediate
static void ensure_rows(Surrogate& s, int64_t rows) {
  rows = round_up(rows, 64);
  if (rows <= s.Bmax) return;
  auto F = [&](size_t n) { return (float*)dev_alloc(s.owned, n * sizeof(float)); };
  const int64_t RD = rows * s.Dp, RH = rows * s.H;
  s.Xn = F(RD); s.G = F(RD); s.Tn = F(RD); s.dG = F(RD);
  s.Z1 = F(RH); s.A1 = F(RH); s.S1 = F(RH); s.Z2 = F(RH); s.A2 = F(RH); s.S2 = F(RH);
  s.U2 = F(RH); s.V1 = F(RH); s.U1 = F(RH); s.dU1 = F(RH); s.dS1 = F(RH); s.dV1 = F(RH);
  s.dU2 = F(RH); s.dZ2 = F(RH); s.dA1 = F(RH); s.dZ1 = F(RH);
  s.f = F(rows); s.yb = F(rows); s.df = F(rows); s.lrow = F(rows); s.scal = F(64);
  s.idx = (int32_t*)dev_alloc(s.owned, rows * sizeof(int32_t));
  s.Bmax = rows;
}

// bf16 mode: operand planes ([row][k] and, where a product over the batch
// reads it, the transpose) and the float32 values the epilogues need again
static void ensure_train_rows(Surrogate& s, int64_t rows) {
  rows = round_up(rows, 64);
  TrainBufs& t = s.tb;
  if (rows <= t.rows) return;
  auto F = [&](size_t n) { return (float*)dev_alloc(s.owned, n * sizeof(float)); };
  auto U = [&](size_t n) { return (uint16_t*)dev_alloc(s.owned, n * 2); };
  const int64_t RD = rows * s.Dp, RH = rows * s.H;
  t.x = U(RD); t.xT = U(RD); t.dg = U(RD); t.dgT = U(RD);
  t.a1 = U(RH); t.a1T = U(RH); t.u2 = U(RH); t.u2T = U(RH); t.u1 = U(RH); t.u1T = U(RH);
  t.dv1 = U(RH); t.dv1T = U(RH); t.dz2 = U(RH); t.dz2T = U(RH); t.dz1T = U(RH);
  t.z1 = F(RH); t.s1 = F(RH); t.z2 = F(RH); t.a2 = F(RH); t.s2 = F(RH); t.v1 = F(RH); t.ds1 = F(RH);
  t.du2 = F(RH); t.dz2f = F(RH); t.dz1f = F(RH);
  t.f = F(rows); t.df = F(rows); t.e2 = F(rows);
  t.lpart = F((s.Dp / 32) * rows);
  t.rows = rows;
}

template <bool TA, bool TB>
static void gemm(Surrogate& s, const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                 int64_t ldc, int64_t M, int64_t N, int64_t K, float alpha, float beta) {
  HMC_REQUIRE(M % SG_T == 0 && N % SG_T == 0 && K % SG_K == 0, HMC_ERR_STATE, "surrogate GEMM padding");
  const dim3 grid((unsigned)(N / SG_T), (unsigned)(M / SG_T));
  hipLaunchKernelGGL((k_sgemm<TA, TB>), grid, dim3(256), 0, s.stream, A, lda, B, ldb, C, ldc, (int)K, alpha, beta);
  HMC_HIP(hipGetLastError());
}

static inline dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

// dst[r][c] = bf16(src[r][c]) (trans 0) or dst[c][r] = bf16(src[r][c]) (trans 1)
__global__ void k_weight_plane(const float* __restrict__ src, int64_t lds, int64_t rows, int64_t cols,
                               uint16_t* __restrict__ dst, int64_t ldd, int trans) {
  const int64_t n = rows * cols;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / cols, c = i % cols;
    const uint16_t v = f32_to_bf16_bits(src[r * lds + c]);
    if (trans) dst[c * ldd + r] = v;
    else dst[r * ldd + c] = v;
  }
}

// bf16 normalised rows Xh[b][j] = bf16((x - xm_j) / xs_j) for b < B, zero in the
// padding (rows up to `rows`, columns up to Dp)
// one workgroup row per chain row (blockIdx.y), 4 columns per thread
template <typename T>
__global__ void k_norm_bf16(const T* __restrict__ X, int64_t ldx, uint16_t* __restrict__ Xh, int Dp, int D,
                            const float* __restrict__ xm, const float* __restrict__ xsinv, int B) {
  const int b = blockIdx.y;
  for (int j0 = 4 * (blockIdx.x * blockDim.x + threadIdx.x); j0 < Dp; j0 += 4 * gridDim.x * blockDim.x) {
    uint32_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + e;
      h[e] = (b < B && j < D) ? f32_to_bf16_bits(((float)X[(int64_t)b * ldx + j] - xm[j]) * xsinv[j]) : 0u;
    }
    *reinterpret_cast<uint2*>(&Xh[(int64_t)b * Dp + j0]) = uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
  }
}

// (launched on `st`, the stream of the GEMMs that read the planes)
static void ensure_planes(Surrogate& s, hipStream_t st) {
  if (s.planes_ok) return;
  // parameters written on the surrogate's own stream (training) are complete
  HMC_HIP(hipStreamSynchronize(s.stream));
  const int64_t H = s.H, Dp = s.Dp, Hp = round_up(H, 256), Dpp = round_up(Dp, 256);
  if (!s.w1h) {
    s.w1h = (uint16_t*)dev_alloc(s.owned, (size_t)Hp * Dp * 2);
    s.w1t = (uint16_t*)dev_alloc(s.owned, (size_t)Dpp * H * 2);
    s.w2h = (uint16_t*)dev_alloc(s.owned, (size_t)Hp * H * 2);
    s.w2t = (uint16_t*)dev_alloc(s.owned, (size_t)Hp * H * 2);
  }
  const dim3 grid(4096);
  hipLaunchKernelGGL(k_weight_plane, grid, dim3(256), 0, st, s.W1(), Dp, H, Dp, s.w1h, Dp, 0);
  hipLaunchKernelGGL(k_weight_plane, grid, dim3(256), 0, st, s.W1(), Dp, H, Dp, s.w1t, H, 1);
  hipLaunchKernelGGL(k_weight_plane, grid, dim3(256), 0, st, s.W2(), H, H, H, s.w2h, H, 0);
  hipLaunchKernelGGL(k_weight_plane, grid, dim3(256), 0, st, s.W2(), H, H, H, s.w2t, H, 1);
  HMC_HIP(hipGetLastError());
  HMC_HIP(hipStreamSynchronize(st));   // later readers may be on another stream
  s.planes_ok = true;
}

static void ensure_bf16_rows(Surrogate& s, int64_t B, int n_cu) {
  const int64_t rows = round_up(B, 256);
  if (rows > s.Bh) {
    s.xh = (uint16_t*)dev_alloc(s.owned, (size_t)rows * s.Dp * 2);
    s.a1h = (uint16_t*)dev_alloc(s.owned, (size_t)rows * s.H * 2);
    s.u2h = (uint16_t*)dev_alloc(s.owned, (size_t)rows * s.H * 2);
    s.u1h = (uint16_t*)dev_alloc(s.owned, (size_t)rows * s.H * 2);
    s.s1h = (float*)dev_alloc(s.owned, (size_t)rows * s.H * 4);
    s.Bh = rows;
  }
  const size_t e = surrogate_split_workspace(s.D, s.H, B, n_cu);
  if (e > s.ws_elems) {
    s.ws = (float*)dev_alloc(s.owned, e * 4);
    s.ws_elems = e;
  }
}

// forward + input gradient for `rows` normalised rows in s.Xn (rows multiple of 64)
static void forward_grad(Surrogate& s, int64_t rows) {
  const int64_t H = s.H, Dp = s.Dp;
  gemm<false, false>(s, s.Xn, Dp, s.W1(), Dp, s.Z1, H, rows, H, Dp, 1.f, 0.f);      // Z1 = Xn W1^T
  hipLaunchKernelGGL(k_act, g1(rows * H), dim3(256), 0, s.stream, s.Z1, s.A1, s.S1, s.b1(), rows, (int)H);
  gemm<false, false>(s, s.A1, H, s.W2(), H, s.Z2, H, rows, H, H, 1.f, 0.f);         // Z2 = A1 W2^T
  hipLaunchKernelGGL(k_act, g1(rows * H), dim3(256), 0, s.stream, s.Z2, s.A2, s.S2, s.b2(), rows, (int)H);
  hipLaunchKernelGGL(k_head, dim3((unsigned)rows), dim3(256), 0, s.stream, s.A2, s.S2, s.w3(), s.b3(),
                     s.U2, s.f, (int)H);
  gemm<false, true>(s, s.U2, H, s.W2(), H, s.V1, H, rows, H, H, 1.f, 0.f);           // V1 = U2 W2
  hipLaunchKernelGGL(k_mul, g1(rows * H), dim3(256), 0, s.stream, s.U1, s.S1, s.V1, rows * H);
  gemm<false, true>(s, s.U1, H, s.W1(), Dp, s.G, Dp, rows, Dp, H, 1.f, 0.f);          // G = U1 W1
  HMC_HIP(hipGetLastError());
}

// loss and parameter gradients for one normalised batch (Xn, Tn, yb) of `rows`
static void backward(Surrogate& s, int64_t rows, float alpha, float beta) {
  const int64_t H = s.H, Dp = s.Dp;
  hipLaunchKernelGGL(k_residuals, dim3((unsigned)rows), dim3(256), 0, s.stream, s.f, s.yb, s.G, s.Tn, s.df,
                     s.dG, s.lrow, Dp, s.D, alpha, beta, (int)rows);
  float* gW1 = s.dP + s.oW1;
  float* gb1 = s.dP + s.ob1;
  float* gW2 = s.dP + s.oW2;
  float* gb2 = s.dP + s.ob2;
  float* gw3 = s.dP + s.ow3;
  float* gb3 = s.dP + s.ob3;
  gemm<true, true>(s, s.U1, H, s.dG, Dp, gW1, Dp, H, Dp, rows, 1.f, 0.f);            // dW1 = U1^T dG
  gemm<false, false>(s, s.dG, Dp, s.W1(), Dp, s.dU1, H, rows, H, Dp, 1.f, 0.f);       // dU1 = dG W1^T
  hipLaunchKernelGGL(k_split, g1(rows * H), dim3(256), 0, s.stream, s.dU1, s.V1, s.S1, s.dS1, s.dV1, rows * H);
  gemm<true, true>(s, s.U2, H, s.dV1, H, gW2, H, H, H, rows, 1.f, 0.f);              // dW2 = U2^T dV1
  gemm<false, false>(s, s.dV1, H, s.W2(), H, s.dU2, H, rows, H, H, 1.f, 0.f);         // dU2 = dV1 W2^T
  // dw3 = sum_b dU2*S2 + sum_b df*A2 ; db3 = sum df
  hipLaunchKernelGGL(k_colsum, g1(H), dim3(256), 0, s.stream, s.dU2, s.S2, s.df, s.A2, gw3, rows, (int)H);
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, s.stream, s.df, rows, gb3);
  hipLaunchKernelGGL(k_dz2, g1(rows * H), dim3(256), 0, s.stream, s.dU2, s.w3(), s.Z2, s.S2, s.df, s.dZ2,
                     rows, (int)H);
  gemm<true, true>(s, s.dZ2, H, s.A1, H, gW2, H, H, H, rows, 1.f, 1.f);              // dW2 += dZ2^T A1
  hipLaunchKernelGGL(k_colsum, g1(H), dim3(256), 0, s.stream, s.dZ2, nullptr, nullptr, nullptr, gb2, rows,
                     (int)H);
  gemm<false, true>(s, s.dZ2, H, s.W2(), H, s.dA1, H, rows, H, H, 1.f, 0.f);          // dA1 = dZ2 W2
  hipLaunchKernelGGL(k_dz1, g1(rows * H), dim3(256), 0, s.stream, s.dS1, s.Z1, s.dA1, s.S1, s.dZ1, rows * H);
  gemm<true, true>(s, s.dZ1, H, s.Xn, Dp, gW1, Dp, H, Dp, rows, 1.f, 1.f);           // dW1 += dZ1^T Xn
  hipLaunchKernelGGL(k_colsum, g1(H), dim3(256), 0, s.stream, s.dZ1, nullptr, nullptr, nullptr, gb1, rows,
                     (int)H);
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, s.stream, s.lrow, rows, s.scal);
  HMC_HIP(hipGetLastError());
}

// the next Adam step (advances the step count)
static AdamStep next_adam(Surrogate& s, float lr) {
  s.adam_t += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)s.adam_t), c2 = 1.f - std::pow(b2, (float)s.adam_t);
  return AdamStep{s.P, s.Pm, s.Pv, lr, b1, b2, c1, c2, 1e-8f};
}

static void adam(Surrogate& s, float lr) {
  s.planes_ok = false;
  hipLaunchKernelGGL(k_adam, g1(s.nP), dim3(256), 0, s.stream, next_adam(s, lr), s.dP, s.nP);
  HMC_HIP(hipGetLastError());
}

// ---- bf16 evaluation and training passes ------------------------------------
template <class Epi>
static void sur_gemm(Surrogate& s, int64_t M, int64_t N, const SurOperands& p0, const SurOperands& p1, const Epi& epi) {
  // 32 x 32 tiles while there are few, with a second wave that only loads in a
  // long product
  auto go = [&](auto wm, auto wn, auto lw, auto st) {
    constexpr int WM = decltype(wm)::value, WN = decltype(wn)::value, LW = decltype(lw)::value, S = decltype(st)::value;
    const int gm = (int)(M / (32 * WM)), gn = (int)(N / (32 * WN));
    hipLaunchKernelGGL((k_sur_gemm<WM, WN, LW, S, Epi>), dim3((unsigned)((gm * gn + 7) / 8 * 8)),
                       dim3((WM * WN + LW) * 64), 0, s.stream, p0, p1, gm, gn, epi);
  };
  using std::integral_constant;
  using I0 = integral_constant<int, 0>;
  using I1 = integral_constant<int, 1>;
  using I2 = integral_constant<int, 2>;
  if ((M / 32) * (N / 32) > 256) go(I2{}, I2{}, I0{}, integral_constant<int, 4>{});
  else if (p0.K + p1.K <= 1024) go(I1{}, I1{}, I0{}, integral_constant<int, 8>{});
  else go(I1{}, I1{}, I1{}, integral_constant<int, 9>{});
  HMC_HIP(hipGetLastError());
}

// planes of rows idx of X (float32 [.][Dp]), forward to U1; f and (training) df
static void bf16_forward(Surrogate& s, int64_t R, const float* X, const int32_t* idx, const float* y, float alpha,
                         bool train) {
  const int64_t H = s.H, Dp = s.Dp;
  TrainBufs& t = s.tb;
  hipLaunchKernelGGL(k_sur_rows, dim3((unsigned)(Dp / 64), (unsigned)(R / 64)), dim3(256), 0, s.stream, X, idx, Dp, R,
                     t.x, train ? t.xT : nullptr);
  HMC_HIP(hipGetLastError());
  const SurOperands none{};
  sur_gemm(s, R, H, SurOperands{t.x, s.w1h, Dp, Dp, (int)Dp}, none,
           SurZ1{s.b1(), t.z1, t.s1, t.a1, train ? t.a1T : nullptr, H, R});                      // Z1 = Xn W1^T
  sur_gemm(s, R, H, SurOperands{t.a1, s.w2h, H, H, (int)H}, none,
           SurZ2{s.b2(), s.w3(), t.z2, t.a2, t.s2, t.u2, train ? t.u2T : nullptr, H, R});        // Z2 = A1 W2^T
  hipLaunchKernelGGL(k_sur_head, dim3((unsigned)R), dim3(256), 0, s.stream, t.a2, s.w3(), s.b3(), y, idx, alpha, t.f,
                     train ? t.df : nullptr, (int)H, (int)R);
  sur_gemm(s, R, H, SurOperands{t.u2, s.w2t, H, H, (int)H}, none,
           SurV1{t.s1, t.v1, t.u1, train ? t.u1T : nullptr, H, R});                              // V1 = U2 W2
}

// loss and parameter gradients (into dP), or with `step` the Adam update of
// the parameters and of the weight planes
static void bf16_train_batch(Surrogate& s, int64_t R, const float* X, const float* T, const float* y,
                             const int32_t* idx, float alpha, float beta, const AdamStep* step, float* loss) {
  const int64_t H = s.H, Dp = s.Dp;
  TrainBufs& t = s.tb;
  const SurOperands none{};
  bf16_forward(s, R, X, idx, y, alpha, true);
  sur_gemm(s, R, Dp, SurOperands{t.u1, s.w1t, H, H, (int)H}, none,
           SurResid{T, idx, t.dg, t.dgT, t.lpart, s.D, Dp, R, beta});                            // G = U1 W1
  sur_gemm(s, R, H, SurOperands{t.dg, s.w1h, Dp, Dp, (int)Dp}, none,
           SurDU1{t.v1, t.s1, t.ds1, t.dv1, t.dv1T, H, R});                                      // dU1 = dG W1^T
  sur_gemm(s, R, H, SurOperands{t.dv1, s.w2h, H, H, (int)H}, none,
           SurDU2{s.w3(), t.z2, t.s2, t.df, t.du2, t.dz2f, t.dz2, t.dz2T, H, R});               // dU2 = dV1 W2^T
  sur_gemm(s, R, H, SurOperands{t.dz2, s.w2t, H, H, (int)H}, none,
           SurDA1{t.ds1, t.z1, t.s1, t.dz1f, t.dz1T, H, R});                                     // dA1 = dZ2 W2
  const AdamStep ad = step ? *step : AdamStep{};
  float* g = step ? nullptr : s.dP;
  hipLaunchKernelGGL(k_sur_e2, dim3((unsigned)(R / 32)), dim3(256), 0, s.stream, t.lpart, (int)(Dp / 32), (int)R, t.e2);
  hipLaunchKernelGGL(k_sur_finish, dim3((unsigned)(H / 64), 4), dim3(64), 0, s.stream,
                     SurFinish{t.du2, t.s2, t.a2, t.dz2f, t.dz1f, t.e2, t.f, y, t.df, idx, g, ad, s.ow3, s.ob2, s.ob1,
                               s.ob3, loss, (int)H, (int)R, (int)s.D, alpha, beta});
  HMC_HIP(hipGetLastError());
  // dW2 = U2^T dV1 + dZ2^T A1, dW1 = U1^T dG + dZ1^T Xn
  sur_gemm(s, H, H, SurOperands{t.u2T, t.dv1T, R, R, (int)R}, SurOperands{t.dz2T, t.a1T, R, R, (int)R},
           SurWeight{g, ad, s.oW2, s.w2h, s.w2t, H, H});
  sur_gemm(s, H, Dp, SurOperands{t.u1T, t.dgT, R, R, (int)R}, SurOperands{t.dz1T, t.xT, R, R, (int)R},
           SurWeight{g, ad, s.oW1, s.w1h, s.w1t, Dp, H});
}

// gradient of the surrogate at the chains' trajectory positions + kick/drift
void surrogate_kick_drift(Chains& c, double kick, double drift, double drift2, bool first) {
  Surrogate& s = *reinterpret_cast<Surrogate*>(c.surrogate);
  Problem& p = *c.p;
  if (s.mode == 0) {
    // bf16 MFMA: normalised rows, then four pipelined GEMMs whose last
    // epilogue applies the kick and drift
    ensure_planes(s, p.stream);
    ensure_bf16_rows(s, c.B, p.n_cu);
    hipEvent_t ev;
    time_begin(c, 5, ev);
    // the first stage of a trajectory normalises the rows (up to the GEMM's
    // 128-row chain tile: padding rows become zeros); later stages read the
    // plane the previous stage's kick/drift epilogue wrote
    if (first || s.planes_for != &c) {
      HMC_REQUIRE(s.Dp % 4 == 0 && s.Bh < 65536, HMC_ERR_STATE, "surrogate row layout");
      const dim3 grid((unsigned)std::max<int64_t>(1, std::min<int64_t>((s.Dp / 4 + 255) / 256, 8)),
                      (unsigned)round_up(c.B, 128));
      if (p.state_dtype == HMC_F64)
        hipLaunchKernelGGL(k_norm_bf16<double>, grid, dim3(256), 0, p.stream, (const double*)c.xt, c.ldx, s.xh,
                           (int)s.Dp, (int)s.D, s.xm, s.xsinv, (int)c.B);
      else
        hipLaunchKernelGGL(k_norm_bf16<float>, grid, dim3(256), 0, p.stream, (const float*)c.xt, c.ldx, s.xh,
                           (int)s.Dp, (int)s.D, s.xm, s.xsinv, (int)c.B);
      HMC_HIP(hipGetLastError());
      s.planes_for = &c;
    }
    SurGemm g;
    g.D = s.D;
    g.Dp = s.Dp;
    g.H = s.H;
    g.xh = s.xh;
    g.w1h = s.w1h;
    g.w1t = s.w1t;
    g.w2h = s.w2h;
    g.w2t = s.w2t;
    g.b1 = s.b1();
    g.b2 = s.b2();
    g.w3 = s.w3();
    g.gscale = s.gscale;
    g.xm = s.xm;
    g.xsinv = s.xsinv;
    g.a1h = s.a1h;
    g.u2h = s.u2h;
    g.u1h = s.u1h;
    g.s1 = s.s1h;
    g.ws = s.ws;
    g.ws_elems = s.ws_elems;
    surrogate_stage_bf16(c, g, kick, drift, drift2);
    time_end(c, 5, ev);
    return;
  }
  const int64_t rows = round_up(c.B, 64);
  ensure_rows(s, rows);
  // launches go to the problem's stream for the duration of the call
  struct StreamSwap {
    Surrogate& s;
    hipStream_t saved;
    ~StreamSwap() { s.stream = saved; }
  } swap{s, s.stream};
  s.stream = p.stream;
  hipEvent_t ev;
  time_begin(c, 5, ev);
  if (p.state_dtype == HMC_F64)
    hipLaunchKernelGGL(k_norm<double>, g1(rows * s.Dp), dim3(256), 0, s.stream, (const double*)c.xt, c.ldx,
                       s.Xn, s.Dp, s.D, s.xm, s.xs, rows);
  else
    hipLaunchKernelGGL(k_norm<float>, g1(rows * s.Dp), dim3(256), 0, s.stream, (const float*)c.xt, c.ldx,
                       s.Xn, s.Dp, s.D, s.xm, s.xs, rows);
  forward_grad(s, rows);
  time_end(c, 5, ev);
  hipEvent_t ev2;
  time_begin(c, 6, ev2);
  if (p.state_dtype == HMC_F64)
    hipLaunchKernelGGL(k_sur_leap<double>, g1(c.B * p.d), dim3(256), 0, s.stream, (double*)c.xt, (double*)c.pt,
                       c.ldx, s.G, s.Dp, p.d, s.gscale, c.eps, (const double*)c.beta, kick, drift, drift2, c.B,
                       p.model());
  else
    hipLaunchKernelGGL(k_sur_leap<float>, g1(c.B * p.d), dim3(256), 0, s.stream, (float*)c.xt, (float*)c.pt,
                       c.ldx, s.G, s.Dp, p.d, s.gscale, c.eps, (const double*)c.beta, kick, drift, drift2, c.B,
                       p.model());
  HMC_HIP(hipGetLastError());
  time_end(c, 6, ev2);
}

}  // namespace hmc

struct hmc_surrogate {
  hmc::Surrogate s;
};

using namespace hmc;

extern "C" {

int hmc_surrogate_create(int64_t dimensions, int64_t hidden, uint64_t seed, hmc_surrogate** out) {
  return guarded("hmc_surrogate_create", [&] {
    HMC_REQUIRE(out && dimensions > 0 && hidden > 0 && hidden % 64 == 0, HMC_ERR_ARG,
                "dimensions > 0 and hidden a positive multiple of 64 are required");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
      (void)hipGetLastError();
      throw Error{HMC_ERR_HIP, "no HIP device is visible"};
    }
    auto* h = new hmc_surrogate();
    Surrogate& s = h->s;
    try {
      HMC_HIP(hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking));
      s.D = dimensions;
      s.Dp = round_up(dimensions, 64);
      s.H = hidden;
      s.oW1 = 0;
      s.ob1 = s.oW1 + s.H * s.Dp;
      s.oW2 = s.ob1 + s.H;
      s.ob2 = s.oW2 + s.H * s.H;
      s.ow3 = s.ob2 + s.H;
      s.ob3 = s.ow3 + s.H;
      s.nP = s.ob3 + 1;
      s.P = (float*)dev_alloc(s.owned, s.nP * 4);
      s.Pm = (float*)dev_alloc(s.owned, s.nP * 4);
      s.Pv = (float*)dev_alloc(s.owned, s.nP * 4);
      s.dP = (float*)dev_alloc(s.owned, s.nP * 4);
      // Glorot-uniform initialisation, zero biases
      std::vector<float> P0(s.nP, 0.f);
      std::mt19937_64 g(seed);
      auto fill = [&](int64_t off, int64_t rows, int64_t cols, int64_t ld, int64_t fan_in, int64_t fan_out) {
        std::uniform_real_distribution<float> U(-1.f, 1.f);
        const float a = std::sqrt(6.f / (float)(fan_in + fan_out));
        for (int64_t r = 0; r < rows; ++r)
          for (int64_t c = 0; c < cols; ++c) P0[off + r * ld + c] = a * U(g);
      };
      fill(s.oW1, s.H, s.D, s.Dp, s.D, s.H);
      fill(s.oW2, s.H, s.H, s.H, s.H, s.H);
      fill(s.ow3, 1, s.H, s.H, s.H, 1);
      h2d(s.P, P0.data(), s.nP * 4);
      std::vector<float> ones(s.Dp, 1.f), zeros(s.Dp, 0.f);
      s.xm = (float*)dev_alloc(s.owned, s.Dp * 4);
      s.xs = (float*)dev_alloc(s.owned, s.Dp * 4);
      s.gscale = (float*)dev_alloc(s.owned, s.Dp * 4);
      s.xsinv = (float*)dev_alloc(s.owned, s.Dp * 4);
      h2d(s.xs, ones.data(), s.Dp * 4);
      h2d(s.gscale, ones.data(), s.Dp * 4);
      h2d(s.xsinv, ones.data(), s.Dp * 4);
    } catch (...) {
      for (void* p : s.owned) (void)hipFree(p);
      if (s.stream) (void)hipStreamDestroy(s.stream);
      delete h;
      throw;
    }
    *out = h;
  });
}

int hmc_surrogate_destroy(hmc_surrogate* h) {
  return guarded("hmc_surrogate_destroy", [&] {
    if (!h) return;
    (void)hipStreamSynchronize(h->s.stream);
    for (void* p : h->s.owned) (void)hipFree(p);
    (void)hipStreamDestroy(h->s.stream);
    delete h;
  });
}

int hmc_surrogate_set_mode(hmc_surrogate* h, int mode) {
  return guarded("hmc_surrogate_set_mode", [&] {
    HMC_REQUIRE(h && (mode == 0 || mode == 1), HMC_ERR_ARG, "mode must be 0 (bf16 MFMA) or 1 (fp32)");
    h->s.mode = mode;
  });
}

int hmc_surrogate_set_normalization(hmc_surrogate* h, const double* x_mean, const double* x_scale,
                                    double f_mean, double f_scale) {
  return guarded("hmc_surrogate_set_normalization", [&] {
    HMC_REQUIRE(h && x_mean && x_scale && f_scale > 0.0, HMC_ERR_ARG, "invalid normalisation");
    Surrogate& s = h->s;
    std::vector<float> m(s.Dp, 0.f), sc(s.Dp, 1.f), gs(s.Dp, 0.f), si(s.Dp, 0.f);
    for (int64_t j = 0; j < s.D; ++j) {
      HMC_REQUIRE(x_scale[j] > 0.0, HMC_ERR_ARG, "x_scale must be positive");
      m[j] = (float)x_mean[j];
      sc[j] = (float)x_scale[j];
      gs[j] = (float)(f_scale / x_scale[j]);
      si[j] = (float)(1.0 / x_scale[j]);
    }
    h2d(s.xm, m.data(), s.Dp * 4);
    h2d(s.xs, sc.data(), s.Dp * 4);
    h2d(s.gscale, gs.data(), s.Dp * 4);
    h2d(s.xsinv, si.data(), s.Dp * 4);
    s.planes_for = nullptr;
    s.f_mean = f_mean;
    s.f_scale = f_scale;
  });
}

// parameters as one packed float32 vector: W1 (H x D) | b1 | W2 (H x H) | b2 | w3 | b3
int hmc_surrogate_param_count(hmc_surrogate* h, int64_t* n) {
  return guarded("hmc_surrogate_param_count", [&] {
    HMC_REQUIRE(h && n, HMC_ERR_ARG, "NULL argument");
    const Surrogate& s = h->s;
    *n = s.H * s.D + s.H + s.H * s.H + s.H + s.H + 1;
  });
}

// device allocations of one call
struct FreeList {
  std::vector<void*> v;
  ~FreeList() {
    for (void* p : v) (void)hipFree(p);
  }
};

static void pack_unpack(Surrogate& s, float* host, bool to_device, float* dev) {
  // host layout is unpadded (W1 H x D); device rows are padded to Dp
  if (!to_device) {
    const int64_t np = s.H * s.D + s.nP - s.ob1;
    if (s.D == s.Dp) {
      d2h(host, dev, np * 4);
      return;
    }
    FreeList tmp;   // packed on the device, one contiguous copy (a pitched copy runs row by row)
    float* buf = (float*)dev_alloc(tmp.v, np * 4);
    hipLaunchKernelGGL(k_sur_pack, dim3((unsigned)std::min<int64_t>((np + 255) / 256, 8192)), dim3(256), 0, s.stream,
                       dev, s.H, s.D, s.Dp, np, buf);
    HMC_HIP(hipGetLastError());
    HMC_HIP(hipMemcpyAsync(host, buf, np * 4, hipMemcpyDeviceToHost, s.stream));
    HMC_HIP(hipStreamSynchronize(s.stream));
    return;
  }
  std::vector<float> buf(s.nP, 0.f);
  int64_t k = 0;
  for (int64_t r = 0; r < s.H; ++r)
    for (int64_t c = 0; c < s.D; ++c, ++k) buf[s.oW1 + r * s.Dp + c] = host[k];
  const int64_t tail = s.nP - s.ob1;
  for (int64_t i = 0; i < tail; ++i, ++k) buf[s.ob1 + i] = host[k];
  h2d(dev, buf.data(), s.nP * 4);
}

int hmc_surrogate_get_params(hmc_surrogate* h, float* params) {
  return guarded("hmc_surrogate_get_params", [&] {
    HMC_REQUIRE(h && params, HMC_ERR_ARG, "NULL argument");
    HMC_HIP(hipStreamSynchronize(h->s.stream));
    pack_unpack(h->s, params, false, h->s.P);
  });
}

int hmc_surrogate_set_params(hmc_surrogate* h, const float* params) {
  return guarded("hmc_surrogate_set_params", [&] {
    HMC_REQUIRE(h && params, HMC_ERR_ARG, "NULL argument");
    HMC_HIP(hipStreamSynchronize(h->s.stream));
    pack_unpack(h->s, const_cast<float*>(params), true, h->s.P);
    h->s.planes_ok = false;
    h->s.adam_t = 0;
    dzero(h->s.Pm, h->s.nP * 4);
    dzero(h->s.Pv, h->s.nP * 4);
  });
}

// rows (n x D, host f64) into float32 device rows dst [n][Dp] (k_sur_load's
// mode), through a staging buffer of at most 64 MB
static void load_rows(Surrogate& s, const double* rows, int64_t n, int mode, double fs, float* dst) {
  const int64_t chunk = std::max<int64_t>(1, std::min<int64_t>(n, ((int64_t)64 << 20) / (8 * s.D)));
  void* stage = nullptr;
  if (hipMalloc(&stage, (size_t)chunk * s.D * 8) != hipSuccess) {
    (void)hipGetLastError();
    throw Error{HMC_ERR_NOMEM, "surrogate staging buffer"};
  }
  try {
    for (int64_t a = 0; a < n; a += chunk) {
      const int64_t m = std::min(chunk, n - a);
      HMC_HIP(hipMemcpyAsync(stage, rows + a * s.D, (size_t)m * s.D * 8, hipMemcpyHostToDevice, s.stream));
      hipLaunchKernelGGL(k_sur_load, dim3((unsigned)std::min<int64_t>((m * s.Dp + 255) / 256, 8192)), dim3(256), 0,
                         s.stream, (const double*)stage, m, s.D, s.Dp, s.xm, s.xs, fs, mode, dst + a * s.Dp);
      HMC_HIP(hipGetLastError());
    }
    HMC_HIP(hipStreamSynchronize(s.stream));
  } catch (...) {
    (void)hipFree(stage);
    throw;
  }
  (void)hipFree(stage);
}

// float32 device rows for a call: [rows][Dp], zero in the padding rows
static float* call_rows(Surrogate& s, std::vector<void*>& tmp, int64_t rows) {
  return (float*)dev_alloc(tmp, (size_t)rows * s.Dp * 4);
}

int hmc_surrogate_eval(hmc_surrogate* h, const double* X, int64_t B, double* f, double* g) {
  return guarded("hmc_surrogate_eval", [&] {
    HMC_REQUIRE(h && X && B > 0, HMC_ERR_ARG, "invalid argument");
    Surrogate& s = h->s;
    const int64_t rows = round_up(B, 64);
    std::vector<float> hf(rows);
    FreeList tmp;
    if (s.mode == 0) {
      ensure_train_rows(s, rows);
      ensure_planes(s, s.stream);
      float* dx = call_rows(s, tmp.v, rows);
      double* dg = g ? (double*)dev_alloc(tmp.v, (size_t)B * s.D * 8) : nullptr;
      load_rows(s, X, B, 1, 1.0, dx);
      bf16_forward(s, rows, dx, nullptr, nullptr, 0.f, false);
      if (g) {
        sur_gemm(s, rows, s.Dp, SurOperands{s.tb.u1, s.w1t, s.H, s.H, (int)s.H}, SurOperands{},
                 SurEvalGrad{s.gscale, dg, s.D, B});
        HMC_HIP(hipMemcpyAsync(g, dg, (size_t)B * s.D * 8, hipMemcpyDeviceToHost, s.stream));
      }
      HMC_HIP(hipMemcpyAsync(hf.data(), s.tb.f, rows * 4, hipMemcpyDeviceToHost, s.stream));
      HMC_HIP(hipStreamSynchronize(s.stream));
    } else {
      ensure_rows(s, rows);
      HMC_HIP(hipMemsetAsync(s.Xn, 0, (size_t)rows * s.Dp * 4, s.stream));
      load_rows(s, X, B, 1, 1.0, s.Xn);
      forward_grad(s, rows);
      std::vector<float> hg(rows * s.Dp), gs(s.Dp);
      HMC_HIP(hipMemcpyAsync(hf.data(), s.f, rows * 4, hipMemcpyDeviceToHost, s.stream));
      HMC_HIP(hipMemcpyAsync(hg.data(), s.G, hg.size() * 4, hipMemcpyDeviceToHost, s.stream));
      HMC_HIP(hipMemcpyAsync(gs.data(), s.gscale, s.Dp * 4, hipMemcpyDeviceToHost, s.stream));
      HMC_HIP(hipStreamSynchronize(s.stream));
      if (g)
        for (int64_t b = 0; b < B; ++b)
          for (int64_t j = 0; j < s.D; ++j) g[b * s.D + j] = (double)hg[b * s.Dp + j] * (double)gs[j];
    }
    if (f)
      for (int64_t b = 0; b < B; ++b) f[b] = s.f_mean + s.f_scale * (double)hf[b];
  });
}

// Loss and packed parameter gradient of one batch, in normalised units:
// y (B) and t (B x D) are targets of f and of grad_xn f.
int hmc_surrogate_loss_grad(hmc_surrogate* h, const double* Xn, const double* y, const double* t, int64_t B,
                            double alpha, double beta, double* loss, float* grad) {
  return guarded("hmc_surrogate_loss_grad", [&] {
    HMC_REQUIRE(h && Xn && y && t && B > 0 && B % 64 == 0, HMC_ERR_ARG, "batch must be a positive multiple of 64");
    Surrogate& s = h->s;
    std::vector<float> hy(B);
    for (int64_t b = 0; b < B; ++b) hy[b] = (float)y[b];
    FreeList tmp;
    float l = 0.f;
    if (s.mode == 0) {
      ensure_train_rows(s, B);
      ensure_planes(s, s.stream);
      float *dx = call_rows(s, tmp.v, B), *dt = call_rows(s, tmp.v, B), *dy = (float*)dev_alloc(tmp.v, (B + 1) * 4);
      h2d(dy, hy.data(), B * 4);
      load_rows(s, Xn, B, 0, 1.0, dx);
      load_rows(s, t, B, 0, 1.0, dt);
      bf16_train_batch(s, B, dx, dt, dy, nullptr, (float)alpha, (float)beta, nullptr, dy + B);
      HMC_HIP(hipMemcpyAsync(&l, dy + B, 4, hipMemcpyDeviceToHost, s.stream));
    } else {
      ensure_rows(s, B);
      h2d(s.yb, hy.data(), B * 4);
      load_rows(s, Xn, B, 0, 1.0, s.Xn);
      load_rows(s, t, B, 0, 1.0, s.Tn);
      forward_grad(s, B);
      backward(s, B, (float)alpha, (float)beta);
      HMC_HIP(hipMemcpyAsync(&l, s.scal, 4, hipMemcpyDeviceToHost, s.stream));
    }
    HMC_HIP(hipStreamSynchronize(s.stream));
    if (loss) *loss = (double)l / (double)B;
    if (grad) pack_unpack(s, grad, false, s.dP);
  });
}

// Train on N rows (X: N x D f64 raw positions, chi: N raw misfits, grad: N x D raw gradients)
// for `epochs` passes of shuffled batches (batch a multiple of 64); normalisation must be set.
int hmc_surrogate_train(hmc_surrogate* h, const double* X, const double* chi, const double* grad, int64_t N,
                        int64_t batch, int64_t epochs, double lr, double alpha, double beta, uint64_t seed,
                        double* loss_history) {
  return guarded("hmc_surrogate_train", [&] {
    HMC_REQUIRE(h && X && chi && grad && N >= batch && batch > 0 && batch % 64 == 0 && epochs > 0, HMC_ERR_ARG,
                "invalid training arguments");
    Surrogate& s = h->s;
    const int64_t nb = N / batch;
    if (s.mode == 0) {
      ensure_train_rows(s, batch);
      ensure_planes(s, s.stream);
    } else {
      ensure_rows(s, batch);
    }
    // normalised training set on the device
    FreeList tmp;
    float *dX = call_rows(s, tmp.v, N), *dT = call_rows(s, tmp.v, N), *dy = (float*)dev_alloc(tmp.v, (size_t)N * 4);
    int32_t* idx = (int32_t*)dev_alloc(tmp.v, (size_t)N * 4);
    float* dl = (float*)dev_alloc(tmp.v, (size_t)nb * 4);
    std::vector<float> hy(N), hl(nb);
    for (int64_t i = 0; i < N; ++i) hy[i] = (float)((chi[i] - s.f_mean) / s.f_scale);
    h2d(dy, hy.data(), N * 4);
    load_rows(s, X, N, 2, 1.0, dX);
    load_rows(s, grad, N, 3, s.f_scale, dT);   // d f_n / d x_n
    std::vector<int32_t> perm(N);
    std::iota(perm.begin(), perm.end(), 0);
    std::mt19937_64 g(seed);
    for (int64_t e = 0; e < epochs; ++e) {
      std::shuffle(perm.begin(), perm.end(), g);
      HMC_HIP(hipMemcpyAsync(idx, perm.data(), N * 4, hipMemcpyHostToDevice, s.stream));
      HMC_HIP(hipStreamSynchronize(s.stream));   // perm is shuffled again while the epoch runs
      for (int64_t b = 0; b < nb; ++b) {
        if (s.mode == 0) {
          const AdamStep step = next_adam(s, (float)lr);   // updates the planes too
          bf16_train_batch(s, batch, dX, dT, dy, idx + b * batch, (float)alpha, (float)beta, &step, dl + b);
        } else {
          hipLaunchKernelGGL(k_gather, g1(batch * s.Dp), dim3(256), 0, s.stream, dX, dT, dy, idx + b * batch, s.Xn,
                             s.Tn, s.yb, s.Dp, batch);
          forward_grad(s, batch);
          backward(s, batch, (float)alpha, (float)beta);
          adam(s, (float)lr);
          HMC_HIP(hipMemcpyAsync(dl + b, s.scal, 4, hipMemcpyDeviceToDevice, s.stream));
        }
      }
      HMC_HIP(hipMemcpyAsync(hl.data(), dl, nb * 4, hipMemcpyDeviceToHost, s.stream));
      HMC_HIP(hipStreamSynchronize(s.stream));
      double acc = 0.0;
      for (int64_t b = 0; b < nb; ++b) acc += (double)hl[b] / (double)batch;
      if (loss_history) loss_history[e] = acc / (double)nb;
    }
  });
}

int hmc_chains_set_surrogate(hmc_chains* hc, hmc_surrogate* hs) {
  return guarded("hmc_chains_set_surrogate", [&] {
    HMC_REQUIRE(hc, HMC_ERR_ARG, "NULL chains");
    Chains& c = hc->c;
    if (hs) {
      HMC_REQUIRE(hs->s.D == c.p->d, HMC_ERR_ARG, "surrogate dimension does not match the problem");
      HMC_REQUIRE(c.p->resolved_engine() == HMC_ENGINE_GEMM, HMC_ERR_UNSUPPORTED,
                  "surrogate trajectories run on the GEMM engine");
    }
    c.surrogate = hs ? &hs->s : nullptr;
  });
}

}  // extern "C"
