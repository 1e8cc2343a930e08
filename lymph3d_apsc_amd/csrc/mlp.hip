// mlp.hip -- liblymph_mlp.so: fully connected network (GELU) trained and
// evaluated with hand-written BF16 MFMA kernels for gfx950 (MI355X).
//
// GEMM: C[M][N] = sum_k A(m,k) B(k,n), bf16 operands, FP32 accumulation on
// v_mfma_f32_16x16x32_bf16.  TM x TM output tile (TM = 128, or 64 for small
// or split-k GEMMs) per 256-thread workgroup, each of the 4 waves owning a
// (TM/2)^2 quarter as (TM/32)^2 MFMA tiles; k advances 64 at a time through
// LDS tiles stored k-contiguous for both operands, so every lane's MFMA
// fragment is one 16-byte LDS read.  Operands may be k-contiguous
// in memory (row-major A, "W[n][k]" B: 16-byte loads copied as they are) or
// m/n-contiguous (16-byte loads along m/n, transposed into LDS), which covers
// the forward pass (X W^T), the input gradient (dZ W) and the weight
// gradient (dZ^T X) without transposed copies.  Epilogues fuse bias + GELU
// (forward, keeping the FP32 pre-activation) and the GELU derivative
// (backward).  Networks whose inputs and hidden layers are at most 512 wide take
// the fragment-order kernels further down instead (k_slab, k_layer, k_wide,
// k_update).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <utility>
#include <vector>

#include "../../include/lymph_mlp.h"

namespace {

typedef uint16_t bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

thread_local std::string g_err;
int fail(int code, std::string m) {
  g_err = std::move(m);
  return code;
}
#define HIP_TRY(x)                                                                          \
  do {                                                                                      \
    hipError_t e_ = (x);                                                                    \
    if (e_ != hipSuccess) return fail(LYMPH_MLP_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// float -> bfloat16, round to nearest even (NaN kept quiet)
__host__ __device__ inline bf16_t f2bf(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ inline float bf2f(bf16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) +
         z * 0.39894228040143268f * expf(-0.5f * z * z);
}

constexpr int BK = 64, LDK = BK + 8;  // LDS row: 64 k + 8 pad (144 B)
enum { EPI_F32 = 0, EPI_GELU_FWD = 1, EPI_GELU_BWD = 2 };

struct GemmArgs {
  int M, N, K;
  const bf16_t* A;  // A(m,k) = A_KC ? A[m*lda + k] : A[k*lda + m]
  int lda;
  const bf16_t* B;  // B(k,n) = B_KC ? B[n*ldb + k] : B[k*ldb + n]
  int ldb;
  float* C32;  // EPI_F32: result (+ bias);   EPI_GELU_FWD: pre-activation z
  bf16_t* C16; // EPI_GELU_FWD: gelu(z);      EPI_GELU_BWD: acc * gelu'(aux)
  int ldc;
  const float* bias;  // [N] or null
  const float* aux;   // EPI_GELU_BWD: pre-activation, ldc layout
  int kchunk;         // k range per blockIdx.z (multiple of BK)
  float* part;        // split-k partial sums [z][M][N], or null for a direct epilogue
};

// One TM x 64 operand tile in TM/32 16-byte pieces per thread: global ->
// registers (issued before the previous tile's MFMAs), registers -> LDS with
// k contiguous.
//  KC (k contiguous in memory): piece c = tid + 256 j is row c/8, k 8(c%8)..+7,
//    stored as it is.
//  not KC (rows contiguous in memory): thread tid owns rows 8 mg..8 mg+7 and
//    k rows RK kg..RK kg+RK-1 (mg = tid % (TM/8), kg = tid / (TM/8), RK = TM/32):
//    RK loads of 8 rows each, coalesced along the rows; in registers each row's
//    RK k values are gathered and written as one RK*2-byte LDS store.  The k
//    chunks (8 values) of row r are XOR-swizzled by (r/16) % 8 so that the 16
//    rows a wave writes at once fall in distinct banks; a 16-row MFMA tile has
//    one swizzle, so the fragment reads stay conflict-free.
template <bool KC>
__device__ inline int lds_k(int row, int k) {
  if (KC) return k;
  return ((((k >> 3) ^ (row >> 4)) & 7) << 3) | (k & 7);
}

template <bool KC, int TM>
__device__ inline void fetch(uint4 (&v)[TM / 32], const bf16_t* __restrict__ g, int ld, int r0,
                             int R, int k0, int ke, int tid) {
  constexpr int RK = TM / 32;
#pragma unroll
  for (int j = 0; j < RK; ++j) {
    v[j] = make_uint4(0u, 0u, 0u, 0u);
    if (KC) {
      const int c = tid + 256 * j;
      const int r = c >> 3, kc = (c & 7) * 8;
      if (r0 + r < R && k0 + kc < ke)
        v[j] = *reinterpret_cast<const uint4*>(g + (size_t)(r0 + r) * ld + k0 + kc);
    } else {
      const int mg = tid % (TM / 8), kk = (tid / (TM / 8)) * RK + j, rc = mg * 8;
      if (k0 + kk < ke && r0 + rc < R)
        v[j] = *reinterpret_cast<const uint4*>(g + (size_t)(k0 + kk) * ld + r0 + rc);
    }
  }
}

__device__ inline uint32_t word(const uint4& v, int w) {
  return w == 0 ? v.x : (w == 1 ? v.y : (w == 2 ? v.z : v.w));
}

template <bool KC, int TM>
__device__ inline void put(bf16_t* __restrict__ s, const uint4 (&v)[TM / 32], int tid) {
  constexpr int RK = TM / 32;
  if (KC) {
#pragma unroll
    for (int j = 0; j < RK; ++j) {
      const int c = tid + 256 * j;
      *reinterpret_cast<uint4*>(s + (c >> 3) * LDK + (c & 7) * 8) = v[j];
    }
  } else {
    static_assert(RK == 2 || RK == 4, "tile rows");
    const int mg = tid % (TM / 8), kb = (tid / (TM / 8)) * RK;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int row = mg * 8 + q;
      // element q of k row j: half (q & 1) of word q / 2 of v[j]
      uint32_t h[RK];
#pragma unroll
      for (int j = 0; j < RK; ++j) h[j] = (q & 1) ? (word(v[j], q >> 1) >> 16) : (word(v[j], q >> 1) & 0xffffu);
      bf16_t* dst = s + row * LDK + lds_k<false>(row, kb);
      if constexpr (RK == 4)
        *reinterpret_cast<uint2*>(dst) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
      else
        *reinterpret_cast<uint32_t*>(dst) = h[0] | (h[1] << 16);
    }
  }
}

template <int EPI>
__device__ inline void epilogue(const GemmArgs& g, int m, int n, float v) {
  const size_t o = (size_t)m * g.ldc + n;
  if (EPI == EPI_F32) {
    g.C32[o] = g.bias ? v + g.bias[n] : v;
  } else if (EPI == EPI_GELU_FWD) {
    const float z = v + g.bias[n];
    g.C32[o] = z;
    g.C16[o] = f2bf(gelu(z));
  } else {
    g.C16[o] = f2bf(v * gelu_grad(g.aux[o]));
  }
}

// TM x TM output tile per 256-thread workgroup; 2 x 2 waves, each owning a
// (TM/2) x (TM/2) quarter as (TM/32) x (TM/32) MFMA tiles of 16 x 16.
template <bool A_KC, bool B_KC, int EPI, int TM>
__global__ __launch_bounds__(256, TM == 128 ? 3 : 1) void k_gemm(GemmArgs g) {
  constexpr int T = TM / 32;  // MFMA tiles per wave per dimension
  __shared__ __attribute__((aligned(16))) bf16_t sA[TM * LDK];
  __shared__ __attribute__((aligned(16))) bf16_t sB[TM * LDK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TM;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TM / 2);
  const int kb = blockIdx.z * g.kchunk;
  const int ke = min(g.K, kb + g.kchunk);
  f32x4 acc[T][T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  uint4 ra[T], rb[T];
  fetch<A_KC, TM>(ra, g.A, g.lda, m0, g.M, kb, ke, tid);
  fetch<B_KC, TM>(rb, g.B, g.ldb, n0, g.N, kb, ke, tid);
  for (int k0 = kb; k0 < ke; k0 += BK) {
    put<A_KC, TM>(sA, ra, tid);
    put<B_KC, TM>(sB, rb, tid);
    __syncthreads();
    if (k0 + BK < ke) {  // next tile in flight while this one is multiplied
      fetch<A_KC, TM>(ra, g.A, g.lda, m0, g.M, k0 + BK, ke, tid);
      fetch<B_KC, TM>(rb, g.B, g.ldb, n0, g.N, k0 + BK, ke, tid);
    }
#pragma unroll
    for (int ks = 0; ks < BK; ks += 32) {
      bf16x8 af[T], bfg[T];
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const int row = wm + i * 16 + fr;
        af[i] = *reinterpret_cast<const bf16x8*>(sA + row * LDK + lds_k<A_KC>(row, ks + fk));
      }
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const int row = wn + j * 16 + fr;
        bfg[j] = *reinterpret_cast<const bf16x8*>(sB + row * LDK + lds_k<B_KC>(row, ks + fk));
      }
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfg[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  // D fragment: lane holds rows 4*(lane/16) + r, column lane % 16 of each 16x16 tile
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + (lane >> 4) * 4 + r;
        const int n = n0 + wn + j * 16 + (lane & 15);
        if (m >= g.M || n >= g.N) continue;
        if (g.part)
          g.part[((size_t)blockIdx.z * g.M + m) * g.N + n] = acc[i][j][r];
        else
          epilogue<EPI>(g, m, n, acc[i][j][r]);
      }
}

// split-k: sum the S partial tiles in order, then the epilogue
template <int EPI>
__global__ void k_splitk(GemmArgs g, int S) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)g.M * g.N) return;
  const int m = (int)(i / g.N), n = (int)(i % g.N);
  float v = 0.f;
  for (int z = 0; z < S; ++z) v += g.part[((size_t)z * g.M + m) * g.N + n];
  epilogue<EPI>(g, m, n, v);
}

__global__ void k_gather(const float* __restrict__ X, int w, const int* __restrict__ idx, int B,
                         bf16_t* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)B * w) return;
  const int b = (int)(i / w), k = (int)(i % w);
  out[i] = f2bf(X[(size_t)idx[b] * w + k]);
}

// dY = scale * (y - t) in bf16; per-block partial sums of (y - t)^2.  Each
// thread takes 8 consecutive outputs of one row (N is a multiple of 8): two
// 16-byte loads of Y and of the target row, one 16-byte store of dY.
constexpr int kLossPer = 8 * 256;  // outputs per workgroup
__global__ __launch_bounds__(256) void k_loss(const float* __restrict__ Y, int N,
                                              const float* __restrict__ T,
                                              const int* __restrict__ idx, int B, float scale,
                                              bf16_t* __restrict__ dY, float* __restrict__ part) {
  __shared__ float red[256];
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  float d2 = 0.f;
  if (i < (size_t)B * N) {
    const int b = (int)(i / N), n = (int)(i % N);
    const float4* y = reinterpret_cast<const float4*>(Y + i);
    const float4* t = reinterpret_cast<const float4*>(T + (size_t)idx[b] * N + n);
    const float4 y0 = y[0], y1 = y[1], t0 = t[0], t1 = t[1];
    const float d[8] = {y0.x - t0.x, y0.y - t0.y, y0.z - t0.z, y0.w - t0.w,
                        y1.x - t1.x, y1.y - t1.y, y1.z - t1.z, y1.w - t1.w};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      o[k] = (uint32_t)f2bf(scale * d[2 * k]) | ((uint32_t)f2bf(scale * d[2 * k + 1]) << 16);
      d2 += d[2 * k] * d[2 * k] + d[2 * k + 1] * d[2 * k + 1];
    }
    *reinterpret_cast<uint4*>(dY + i) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  red[threadIdx.x] = d2;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// deterministic sum of n partials by one 256-thread workgroup: thread t adds
// partials t, t+256, ... in order, then a fixed tree over the threads
__global__ __launch_bounds__(256) void k_sum(const float* __restrict__ part, int n, float scale,
                                             float* __restrict__ out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = (float)(red[0] * scale);
}

// out[n] = sum_b D[b][n]: 64 columns per workgroup as 8 groups of 8 (one
// 16-byte load per row); 32 row groups per column group, row group g adding
// rows g, g + 32, ... in order, then the 32 partials of each column in order
// (deterministic).  N is a multiple of 8.
__global__ __launch_bounds__(256) void k_colsum(const bf16_t* __restrict__ D, int B, int N,
                                                float* __restrict__ out) {
  __shared__ float red[32][65];
  const int cg = threadIdx.x & 7, rg = threadIdx.x >> 3;
  const int n0 = blockIdx.x * 64 + cg * 8;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (n0 < N)
    for (int b = rg; b < B; b += 32) {
      const uint4 v = *reinterpret_cast<const uint4*>(D + (size_t)b * N + n0);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        s[2 * k] += bf2f((bf16_t)(w[k] & 0xffffu));
        s[2 * k + 1] += bf2f((bf16_t)(w[k] >> 16));
      }
    }
#pragma unroll
  for (int k = 0; k < 8; ++k) red[rg][cg * 8 + k] = s[k];
  __syncthreads();
  if (threadIdx.x < 64) {
    const int n = blockIdx.x * 64 + threadIdx.x;
    float t = 0.f;
    for (int g = 0; g < 32; ++g) t += red[g][threadIdx.x];
    if (n < N) out[n] = t;
  }
}

__global__ void k_to_bf16(const float* __restrict__ a, bf16_t* __restrict__ b, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = f2bf(a[i]);
}


// ---------------------------------------------------------------------------
// Networks whose inputs and hidden layers are at most kSlabW wide (the receiver
// network; the all-traces network, whose output layer is wide).
//
// Weights are kept in the order the matrix cores read them (pack_pos: W for
// the forward pass, its columns for the input gradients), and so are the
// activations and gradients between layers, so that one 16-byte load per lane
// is a whole MFMA fragment and a wave's load is 1 KB in one piece: no LDS
// staging, no transposes.  The products run over k in the same 32-wide steps,
// in the same order, as k_gemm's: the same bits.
constexpr int kSlabW = 512;       // widest layer: 8 waves x 4 tiles of 16 columns in one pass
constexpr int kSlabL = 16;        // most layers
constexpr int kSlabLd = kSlabW + 8;  // LDS row of activations: 16-byte reads of 8 rows in distinct banks

// fragment order of a [R][C] matrix contracted over C: tile r / 16, step
// c / 32, then lane (c % 32) / 8 * 16 + r % 16 holding c % 8; `steps` per tile
__host__ __device__ inline size_t pack_pos(int r, int c, int steps) {
  return ((size_t)(r >> 4) * steps + (c >> 5)) * 512 + ((((c >> 3) & 3) << 4) + (r & 15)) * 8 + (c & 7);
}
__host__ __device__ inline int steps_of(int c) { return (c + 31) >> 5; }
__host__ __device__ inline int tiles_of(int r) { return (r + 15) >> 4; }
// tiles per wave (8 waves), and the packed matrix' tiles: whole passes, so no
// load needs a bound (the padding is zero)
__host__ __device__ inline int tpw_of(int r) { return (tiles_of(r) + 7) >> 3; }
__host__ __device__ inline size_t pack_size(int r, int c) { return (size_t)tpw_of(r) * 8 * steps_of(c) * 512; }

struct SlabArgs {
  int L, B;                 // layers, valid rows
  int w[kSlabL + 1];        // widths
  const bf16_t* Wf[kSlabL]; // W_l packed
  const float* bias[kSlabL];
  const float* X;           // inputs [B][w[0]]
  float* Y;                 // outputs [B][w[L]]; null: the last layer's gelu goes to Hp
  bf16_t* Hp;               // packed [rows][w[L]] (a wide output layer follows)
};

// fragment f of the packed matrix: a uniform base and the lane's 16 bytes
__device__ __forceinline__ u32x4 frag(const bf16_t* W, size_t f, int lane) {
  return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(W + f * 512) + (uint32_t)lane * 16u);
}

// the first fragments of a wave's tiles (PF of them, step by step)
template <int PF, int TPW>
__device__ __forceinline__ void frag_first(u32x4 (&pf)[PF], const bf16_t* W, int steps, int wave, int lane) {
  constexpr int CH = PF / TPW;  // steps in flight
#pragma unroll
  for (int s = 0; s < CH; ++s)
#pragma unroll
    for (int i = 0; i < TPW; ++i)
      pf[s * TPW + i] = frag(W, (size_t)(wave + 8 * i) * steps + min(s, steps - 1), lane);
}
template <int PF>
__device__ __forceinline__ void frag_first_any(u32x4 (&pf)[PF], const bf16_t* W, int tpw, int steps, int wave,
                                               int lane) {
  if (tpw == 4) frag_first<PF, 4>(pf, W, steps, wave, lane);
  else if (tpw == 3) frag_first<PF, 3>(pf, W, steps, wave, lane);
  else if (tpw == 2) frag_first<PF, 2>(pf, W, steps, wave, lane);
  else frag_first<PF, 1>(pf, W, steps, wave, lane);
}

// acc[i][m] += W tile (wave + 8 i) times the slab's rows 16 m..16 m + 15; pf
// holds the first fragments (frag_first), each refilled as it is used
template <int MR, int PF, int TPW>
__device__ __forceinline__ void slab_product(f32x4 (&acc)[4][MR / 16], u32x4 (&pf)[PF], const bf16_t* W, int steps,
                                             const bf16_t* sH, int wave, int lane) {
  constexpr int CH = PF / TPW;  // steps in flight
  const bf16_t* a = sH + (lane & 15) * kSlabLd + (lane >> 4) * 8;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int m = 0; m < MR / 16; ++m) acc[i][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 h[MR / 16], hn[MR / 16];
  auto rows = [&](bf16x8 (&v)[MR / 16], int step) {
#pragma unroll
    for (int m = 0; m < MR / 16; ++m) v[m] = *reinterpret_cast<const bf16x8*>(a + m * 16 * kSlabLd + step * 32);
  };
  auto use = [&](int s) {
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const bf16x8 w = __builtin_bit_cast(bf16x8, pf[s * TPW + i]);
#pragma unroll
      for (int m = 0; m < MR / 16; ++m)
        acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, h[m], acc[i][m], 0, 0, 0);
    }
  };
  rows(h, 0);
  // whole chunks refill without a branch (the last step again past the end):
  // with one, every use would wait for all loads in flight; and in this order,
  // or the compiler gathers the refills at the chunk's end
  const int whole = steps / CH * CH;
#pragma unroll 1
  for (int s0 = 0; s0 < whole; s0 += CH)
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      rows(hn, min(s0 + s + 1, steps - 1));
      use(s);
#pragma unroll
      for (int i = 0; i < TPW; ++i)
        pf[s * TPW + i] = frag(W, (size_t)(wave + 8 * i) * steps + min(s0 + s + CH, steps - 1), lane);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < MR / 16; ++m) h[m] = hn[m];
    }
#pragma unroll
  for (int s = 0; s < CH; ++s)
    if (whole + s < steps) {
      rows(h, whole + s);
      use(s);
    }
}
template <int MR, int PF>
__device__ __forceinline__ void slab_product_any(f32x4 (&acc)[4][MR / 16], u32x4 (&pf)[PF], const bf16_t* W, int tpw,
                                                 int steps, const bf16_t* sH, int wave, int lane) {
  if (tpw == 4) slab_product<MR, PF, 4>(acc, pf, W, steps, sH, wave, lane);
  else if (tpw == 3) slab_product<MR, PF, 3>(acc, pf, W, steps, sH, wave, lane);
  else if (tpw == 2) slab_product<MR, PF, 2>(acc, pf, W, steps, sH, wave, lane);
  else slab_product<MR, PF, 1>(acc, pf, W, steps, sH, wave, lane);
}

// Four neighbouring columns n0..n0+3 of slab row m into LDS; columns past the
// layer's width are zeros (the next contraction runs in whole steps of 32)
__device__ __forceinline__ void slab_put(bf16_t* sH, int m, int n0, const uint32_t (&h)[4]) {
  *reinterpret_cast<uint2*>(sH + m * kSlabLd + n0) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
}

// Forward pass of one slab of MR rows through the whole network: rows are
// independent, so a workgroup needs no other's results and the activations
// never leave LDS.  8 waves x TPW column tiles; D fragments: lane holds
// columns 16 t + 4 (lane / 16) + r of row 16 m + lane % 16.  Bound by the
// weights' way into the CUs (each slab reads all of them from L2) and the
// error functions.  Receiver network (32-512x5-64), 16,384 rows: 64 batches
// of 7 launches took 5.6 ms, one launch takes 0.106 ms (340 TFLOP/s).
template <int MR, int PF>
__global__ __launch_bounds__(512, 2) void k_slab(SlabArgs g) {
  constexpr int MT = MR / 16;
  __shared__ __attribute__((aligned(16))) bf16_t sH[MR * kSlabLd];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b0 = blockIdx.x * MR;
  const int q4 = (lane >> 4) * 4, mr = lane & 15;
  u32x4 pf[PF];
  frag_first_any<PF>(pf, g.Wf[0], tpw_of(g.w[1]), steps_of(g.w[0]), wave, lane);
  {  // the slab's inputs in bf16, zeros past the rows and past the width
    const int K = g.w[0], Kp = steps_of(K) * 32;
    for (int e = tid; e < MR * (Kp / 4); e += 512) {
      const int m = e / (Kp / 4), k = (e % (Kp / 4)) * 4;
      uint32_t h[4] = {0u, 0u, 0u, 0u};
      if (b0 + m < g.B && k < K) {
        const float4 x = *reinterpret_cast<const float4*>(g.X + (size_t)(b0 + m) * K + k);
        h[0] = f2bf(x.x); h[1] = f2bf(x.y); h[2] = f2bf(x.z); h[3] = f2bf(x.w);
      }
      slab_put(sH, m, k, h);
    }
  }
  __syncthreads();
  f32x4 acc[4][MT];
  for (int l = 0; l < g.L; ++l) {
    const int N = g.w[l + 1], tpw = tpw_of(N), nt = tiles_of(N);
    const bool last = g.Y && l + 1 == g.L;
    slab_product_any<MR, PF>(acc, pf, g.Wf[l], tpw, steps_of(g.w[l]), sH, wave, lane);
    if (l + 1 < g.L) frag_first_any<PF>(pf, g.Wf[l + 1], tpw_of(g.w[l + 2]), steps_of(N), wave, lane);
    __syncthreads();  // every wave has read this layer's input
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = wave + 8 * i;
      if (i >= tpw || t >= nt) continue;
      const int n0 = t * 16 + q4;
      const bool in = n0 < N;  // widths are multiples of 8: all four columns or none
      const float4 bv = in ? *reinterpret_cast<const float4*>(g.bias[l] + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
      const float b[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int row = b0 + m * 16 + mr;
        if (last) {
          if (in && row < g.B)
            *reinterpret_cast<float4*>(g.Y + (size_t)row * N + n0) =
                make_float4(acc[i][m][0] + b[0], acc[i][m][1] + b[1], acc[i][m][2] + b[2], acc[i][m][3] + b[3]);
          continue;
        }
        uint32_t h[4] = {0u, 0u, 0u, 0u};
        if (in)
#pragma unroll
          for (int r = 0; r < 4; ++r) h[r] = f2bf(gelu(acc[i][m][r] + b[r]));
        if (l + 1 < g.L)
          slab_put(sH, m * 16 + mr, n0, h);
        else if (in)
          *reinterpret_cast<uint2*>(g.Hp + pack_pos(row, n0, steps_of(N))) =
              make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
      }
    }
    if (nt & 1) {  // the last step's second tile
      const uint32_t zero[4] = {0u, 0u, 0u, 0u};
      for (int e = tid; e < MR * 4; e += 512) slab_put(sH, e >> 2, nt * 16 + (e & 3) * 4, zero);
    }
    __syncthreads();
  }
}

// Training: one launch per layer and direction.  A slab kernel as above left
// the chip idle here -- 16 slabs at batch 256, each pulling all 2.3 MB of
// weights into one CU at about 60 GB/s, 84 us forward and back -- so every
// 16 x 16 tile of a layer is a wave of its own (512 of them at 256 x 512),
// all its fragments in flight at once: one trip to memory per launch, 3.7 to
// 4.7 us each.  Receiver network, batch 256: a step of 30 launches took 178
// us, these 12 take 57 us (k_update 11 us of them; 61 and 16 while the
// transposed copies were rows, of which a load takes 64 bytes at a time).
enum { LAYER_FWD = 0, LAYER_LOSS = 1, LAYER_BWD = 2, LAYER_OUT = 3 };
struct LayerArgs {
  int N, K, B, ts;     // output width, contraction, rows, steps of a transposed copy's row
  const bf16_t* W;     // packed [N][K]
  const bf16_t* in;    // packed [rows][K]; null: rows idx[b] of X
  const float* X;
  const int* idx;      // null: rows 0, 1, ...
  bf16_t* XT;          // X's rows in bf16, transposed and packed [K][rows]
  const float* bias;   // forward
  bf16_t* out;         // packed [rows][N]: gelu(z), dY or dZ
  bf16_t* outT;        // transposed, packed [N][rows]
  f32x4* dg;           // gelu'(z) as the lanes hold it, one per tile and lane
  const float* T;      // loss: targets, row idx[b]
  float scale;         // loss: 2 / (B N)
  float* part;         // loss: per wave, sum of (y - t)^2
  float* Y;            // LAYER_OUT: outputs [B][N]
  int rw;              // k_wide: waves of a workgroup along the rows
};

// workgroups of 2 waves: column tile wg % tiles, row tiles 2 (wg / tiles) + wave
__host__ __device__ inline int layer_wgs(int N, int B) { return tiles_of(N) * ((B + 31) >> 5); }

// End of one 16 x 16 tile from its sums; dg, bv, tv: gelu'(z), bias and target
// of the lane's four columns.  With sT the transposed copy goes there (its
// column 0, row 0 of the tile).  Returns the lane's part of the loss.
template <int EPI>
__device__ __forceinline__ float layer_end(const LayerArgs& g, int mt, int t, int lane, f32x4 acc, f32x4 dg,
                                           float4 bv, float4 tv, bf16_t* sT = nullptr, int ldT = 0) {
  const int nt = tiles_of(g.N), row = mt * 16 + (lane & 15), n0 = t * 16 + (lane >> 4) * 4;
  const bool ok = n0 < g.N && row < g.B;  // widths are multiples of 8: all four columns or none
  const float b[4] = {bv.x, bv.y, bv.z, bv.w}, tt[4] = {tv.x, tv.y, tv.z, tv.w};
  if (EPI == LAYER_OUT) {
    if (ok)
      *reinterpret_cast<float4*>(g.Y + (size_t)row * g.N + n0) =
          make_float4(acc[0] + b[0], acc[1] + b[1], acc[2] + b[2], acc[3] + b[3]);
    return 0.f;
  }
  uint32_t h[4] = {0u, 0u, 0u, 0u};
  float d2 = 0.f;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (EPI == LAYER_FWD) {
      const float z = acc[r] + b[r];
      const float e1 = 1.0f + erff(z * 0.70710678118654752f);
      h[r] = f2bf(0.5f * z * e1);
      dg[r] = 0.5f * e1 + z * 0.39894228040143268f * expf(-0.5f * z * z);
    } else if (EPI == LAYER_BWD) {
      h[r] = f2bf(acc[r] * dg[r]);
    } else {
      const float d = (acc[r] + b[r]) - tt[r];
      if (ok) d2 += d * d;
      h[r] = f2bf(g.scale * d);
    }
  }
  if (EPI == LAYER_FWD) g.dg[((size_t)mt * nt + t) * 64 + lane] = dg;
  if (ok) {
    if (g.out)
      *reinterpret_cast<uint2*>(g.out + pack_pos(row, n0, steps_of(g.N))) =
          make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    if (!sT)
#pragma unroll
      for (int r = 0; r < 4; ++r) g.outT[pack_pos(n0 + r, row, g.ts)] = (bf16_t)h[r];
  }
  if (sT)
#pragma unroll
    for (int r = 0; r < 4; ++r) sT[((lane >> 4) * 4 + r) * ldT + (lane & 15)] = (bf16_t)h[r];
  return d2;
}

template <int EPI, bool GATHER>
__device__ __forceinline__ void layer_tile(const LayerArgs& g, int wg) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = tiles_of(g.N), t = wg % nt, mt = wg / nt * 2 + wave;
  if (mt * 16 >= g.B) return;
  const int steps = steps_of(g.K);
  const int row = mt * 16 + (lane & 15), n0 = t * 16 + (lane >> 4) * 4;
  const bool in = n0 < g.N, ok = in && row < g.B;  // widths are multiples of 8: all four columns or none
  f32x4 dg = {0.f, 0.f, 0.f, 0.f};
  if (EPI == LAYER_BWD) dg = g.dg[((size_t)mt * nt + t) * 64 + lane];
  float4 bv = make_float4(0.f, 0.f, 0.f, 0.f), tv = bv;
  if (EPI != LAYER_BWD && in) bv = *reinterpret_cast<const float4*>(g.bias + n0);
  if (EPI == LAYER_LOSS && ok) tv = *reinterpret_cast<const float4*>(g.T + (size_t)g.idx[row] * g.N + n0);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  constexpr int CH = GATHER ? 4 : 16;  // steps in flight
#pragma unroll 1
  for (int s0 = 0; s0 < steps; s0 += CH) {
    u32x4 w[CH], h[CH];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int st = min(s0 + s, steps - 1);
      w[s] = frag(g.W, (size_t)t * steps + st, lane);
      if (!GATHER) {
        h[s] = frag(g.in, (size_t)mt * steps + st, lane);
      } else {
        const int k = st * 32 + (lane >> 4) * 8;
        uint32_t v[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        if (row < g.B && k < g.K) {
          const float* x = g.X + (size_t)(g.idx ? g.idx[row] : row) * g.K + k;
          const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
          v[0] = f2bf(a.x); v[1] = f2bf(a.y); v[2] = f2bf(a.z); v[3] = f2bf(a.w);
          v[4] = f2bf(b.x); v[5] = f2bf(b.y); v[6] = f2bf(b.z); v[7] = f2bf(b.w);
          if (t == 0 && s0 + s < steps)
#pragma unroll
            for (int r = 0; r < 8; ++r) g.XT[pack_pos(k + r, row, g.ts)] = (bf16_t)v[r];
        }
        h[s] = u32x4{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
      }
    }
#pragma unroll
    for (int s = 0; s < CH; ++s)
      if (s0 + s < steps)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[s]),
                                                      __builtin_bit_cast(bf16x8, h[s]), acc, 0, 0, 0);
  }
  float d2 = layer_end<EPI>(g, mt, t, lane, acc, dg, bv, tv);
  if (EPI == LAYER_LOSS) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) d2 += __shfl_down(d2, o, 64);
    if (lane == 0) g.part[(size_t)mt * nt + t] = d2;
  }
}

// acc[i][j] += W tile (t0 + i) times row tile (m0 + j) over steps s0..s1 - 1,
// both in fragment order, D steps' fragments in flight.  Tiles past the last are
// the last one again.
template <int T, int D>
__device__ __forceinline__ void block_product(f32x4 (&acc)[T][T], const bf16_t* W, const bf16_t* in, int t0, int nt,
                                              int m0, int nm, int steps, int s0, int s1, int lane) {
  size_t wt[T], ht[T];
#pragma unroll
  for (int i = 0; i < T; ++i) {
    wt[i] = (size_t)min(t0 + i, nt - 1) * steps;
    ht[i] = (size_t)min(m0 + i, nm - 1) * steps;
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  u32x4 w[D][T], h[D][T];
  auto get = [&](int d, int s) {
    s = min(s, s1 - 1);
#pragma unroll
    for (int i = 0; i < T; ++i) w[d][i] = frag(W, wt[i] + s, lane);
#pragma unroll
    for (int i = 0; i < T; ++i) h[d][i] = frag(in, ht[i] + s, lane);
  };
  auto use = [&](int d) {
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[d][i]),
                                                            __builtin_bit_cast(bf16x8, h[d][j]), acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) get(d, s0 + d);
  int s = s0;
#pragma unroll 1
  for (; s + D <= s1; s += D)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      use(d);
      get(d, s + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (s + d < s1) use(d);
}

// LDS ordering within one wave: fences at wavefront scope around a
// code-motion barrier
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wide output layer, forward: every wave T x T tiles of 16 x 16, so that W's
// fragments are read B / 16 T times and the rows' N / 16 T times where k_layer
// reads them once per tile.  4 waves a workgroup, rw of them along the rows; an
// XCD takes every eighth group of columns for all rows, so W comes into one L2
// only.  Bound by the way of W and the targets
// (39 MB each at 256 x 38,400) from HBM, of the gradients back (two copies of
// 20 MB) and of the rows from L2.  EPI LAYER_LOSS fuses the loss: outputs are
// not stored.
template <int T, int EPI>
__global__ __launch_bounds__(256, 2) void k_wide(LayerArgs g) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = tiles_of(g.N), nm = tiles_of(g.B), steps = steps_of(g.K);
  const int wr = (nm + T * g.rw - 1) / (T * g.rw), li = blockIdx.x >> 3;
  const int m0 = (li % wr * g.rw + wave % g.rw) * T;
  const int t0 = ((li / wr * 8 + (blockIdx.x & 7)) * (4 / g.rw) + wave / g.rw) * T;
  float d2 = 0.f;
  // a wave's gradients transposed: they leave as whole fragments
  constexpr int LDT = 16 * T + 8;
  __shared__ __attribute__((aligned(16))) bf16_t sT[EPI == LAYER_LOSS ? 4 * 16 * T * LDT : 8];
  bf16_t* st = sT + (EPI == LAYER_LOSS ? wave * 16 * T * LDT : 0);
  if (m0 < nm && t0 < nt) {
    float4 bv[T], tv[T][T];  // biases and targets on their way while the products run
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int row = (m0 + j) * 16 + (lane & 15);
      const int src = EPI == LAYER_LOSS && row < g.B ? g.idx[row] : -1;
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const int n0 = (t0 + i) * 16 + (lane >> 4) * 4;
        tv[i][j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (src >= 0 && n0 < g.N) tv[i][j] = *reinterpret_cast<const float4*>(g.T + (size_t)src * g.N + n0);
      }
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const int n0 = (t0 + i) * 16 + (lane >> 4) * 4;
      bv[i] = n0 < g.N ? *reinterpret_cast<const float4*>(g.bias + n0) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    f32x4 acc[T][T];
    block_product<T, T == 4 ? 2 : 4>(acc, g.W, g.in, t0, nt, m0, nm, steps, 0, steps, lane);
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
      for (int j = 0; j < T; ++j)
        if (t0 + i < nt && m0 + j < nm)
          d2 += layer_end<EPI>(g, m0 + j, t0 + i, lane, acc[i][j], f32x4{0.f, 0.f, 0.f, 0.f}, bv[i], tv[i][j],
                               EPI == LAYER_LOSS ? st + i * 16 * LDT + j * 16 : nullptr, LDT);
    if (EPI == LAYER_LOSS) {
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T / 2; ++j) {  // whole fragments: T is even, and so is m0
          const int n = (t0 + i) * 16 + (lane & 15), c = j * 32 + (lane >> 4) * 8;
          if (n < g.N && m0 * 16 + c < g.B)
            *reinterpret_cast<uint4*>(g.outT + ((size_t)(t0 + i) * g.ts + m0 / 2 + j) * 512 + lane * 8) =
                *reinterpret_cast<const uint4*>(st + (i * 16 + (lane & 15)) * LDT + c);
        }
    }
  }
  if (EPI == LAYER_LOSS) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) d2 += __shfl_down(d2, o, 64);
    if (lane == 0) g.part[(size_t)blockIdx.x * 4 + wave] = d2;
  }
}

// Its input gradient: a long contraction (N of the output layer) for few
// tiles, so the contraction is split as in gemm() and the parts, stored as the
// lanes hold them, are added in order by k_split_end.  An XCD takes every
// eighth part, whose operands then fit its L2.  256 x 512 from 38,400: 28 us,
// 19 where dZ and W are still in the Infinity Cache (2 x 2 tiles a wave 39; more
// steps in flight change nothing) and 5 for the sums, where the GEMM and its
// sums took 47.
template <int T>
__global__ __launch_bounds__(256, 2) void k_split(LayerArgs g, int S, int chunk, f32x4* ws) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt = tiles_of(g.N), nm = tiles_of(g.B), steps = steps_of(g.K);
  const int wr = (nm + 2 * T - 1) / (2 * T), wgs = wr * ((nt + 2 * T - 1) / (2 * T)), li = blockIdx.x >> 3;
  const int z = li / wgs * 8 + (blockIdx.x & 7), o = li % wgs;
  const int m0 = (o % wr * 2 + (wave & 1)) * T, t0 = (o / wr * 2 + (wave >> 1)) * T;
  if (z >= S || m0 >= nm || t0 >= nt) return;
  f32x4 acc[T][T];
  block_product<T, 4>(acc, g.W, g.in, t0, nt, m0, nm, steps, z * chunk, min(steps, (z + 1) * chunk), lane);
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
      if (t0 + i < nt && m0 + j < nm)
        ws[(((size_t)z * nm + m0 + j) * nt + t0 + i) * 64 + lane] = acc[i][j];
}

__global__ __launch_bounds__(64) void k_split_end(LayerArgs g, int S, const f32x4* ws) {
  const int lane = threadIdx.x, nt = tiles_of(g.N), nm = tiles_of(g.B);
  const int mt = blockIdx.x / nt, t = blockIdx.x % nt;
  const f32x4 dg = g.dg[((size_t)mt * nt + t) * 64 + lane];
  const size_t stride = (size_t)nm * nt * 64;
  const f32x4* p = ws + ((size_t)mt * nt + t) * 64 + lane;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int z = 0; z < S; ++z) v += p[z * stride];
  const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
  layer_end<LAYER_BWD>(g, mt, t, lane, v, dg, none, none);
}

struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ float adam_one(float& w, float& m, float& v, float g, const AdamArgs& a) {
  const float mi = a.b1 * m + (1.f - a.b1) * g;
  const float vi = a.b2 * v + (1.f - a.b2) * g * g;
  m = mi;
  v = vi;
  w = w - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + a.eps);
  return w;
}

__global__ void k_adam(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                       const float* __restrict__ gr, bf16_t* __restrict__ wb, size_t n, AdamArgs a) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float wi = w[i], mi = m[i], vi = v[i];
  adam_one(wi, mi, vi, gr[i], a);
  m[i] = mi;
  v[i] = vi;
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

struct UpdateLayer {
  int N, K, first;      // W is [N][K]; first workgroup of its weight tiles
  const bf16_t *DT, *HT;  // dZ^T [N][rows], H^T [K][rows], packed
  size_t woff, boff;
  bf16_t *Wf, *Wd;      // packed copies
};
struct UpdateArgs {
  int L, B, ts, first_bias, n_part;  // ts: steps of DT's and HT's rows
  UpdateLayer y[kSlabL];
  float *P, *M, *V;  // ADAM: updated in place
  float* G;          // !ADAM: gradients
  AdamArgs a;
  const float* part;
  float part_scale;
  float* loss;
};

// Weight gradients dW_l = dZ_l^T H_l of every layer in one launch, with the
// Adam update of the master weights, both moments and the bf16 copies in the
// epilogue (ADAM), or the gradients stored (!ADAM).  64 x 16 (k x n) of W per
// workgroup of 2 waves, 32 x 16 per wave, fragments straight from the
// transposed operands (packed along the batch); D
// fragments hold four neighbouring k of one n, so masters and moments move in
// 16-byte pieces.  Bound by their 24 bytes per weight and by the trip to
// memory (a gradient buffer in between would add 8 bytes and a launch).
// Joined to the launch of a lower layer's input gradient instead, each layer's
// update made those launches 8.3 us long where they take 4.2: 75 us a step
// against 63.  The workgroups from first_bias on sum the biases' columns (in
// k_colsum's order), the last one the loss.  PARTS > 1: that many pairs of
// waves share the batch and add their sums in order (see update_parts).
template <bool ADAM, int PARTS>
__global__ __launch_bounds__(128 * PARTS) void k_update(UpdateArgs u) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6 & 1), part = __builtin_amdgcn_readfirstlane(tid >> 7);
  const int wg = blockIdx.x;
  __shared__ f32x4 sP[PARTS > 1 ? PARTS - 1 : 1][PARTS > 1 ? 2 : 1][64][2];
  if (wg == (int)gridDim.x - 1) {  // the loss
    __shared__ double red[128];
    if (part == 0) {
      double s = 0.0;
#pragma unroll 8
      for (int i = tid; i < u.n_part; i += 128) s += u.part[i];
      red[tid] = s;
    }
    __syncthreads();
    for (int w = 64; w > 0; w >>= 1) {
      if (tid < w) red[tid] += red[tid + w];
      __syncthreads();
    }
    if (tid == 0) u.loss[0] = (float)(red[0] * u.part_scale);
    return;
  }
  if (wg >= u.first_bias) {  // 4 bias entries per workgroup, 32 lanes each
    int o = wg - u.first_bias, l = 0;
    while (o >= u.y[l].N / 4) o -= u.y[l++].N / 4;
    const UpdateLayer& y = u.y[l];
    const int gp = lane & 31, half = lane >> 5;
    const int n = o * 4 + wave * 2 + half;  // widths are multiples of 8
    float s = 0.f;
    if constexpr (PARTS == 1) {
      for (int b = gp; b < u.B; b += 32) s += bf2f(y.DT[pack_pos(n, b, u.ts)]);
    } else {
#pragma unroll 8
      for (int b = 32 * part + gp; b < u.B; b += 32 * PARTS) s += bf2f(y.DT[pack_pos(n, b, u.ts)]);
      if (part > 0) sP[part - 1][wave][lane][0][0] = s;
      __syncthreads();
      if (part > 0) return;
#pragma unroll
      for (int j = 0; j < PARTS - 1; ++j) s += sP[j][wave][lane][0][0];
    }
    float t = 0.f;
#pragma unroll
    for (int j = 0; j < 32; ++j) t += __shfl(s, half * 32 + j, 64);
    if (gp == 0) {
      const size_t i = y.boff + n;
      if (ADAM) {
        float w = u.P[i], m = u.M[i], v = u.V[i];
        adam_one(w, m, v, t, u.a);
        u.P[i] = w; u.M[i] = m; u.V[i] = v;
      } else {
        u.G[i] = t;
      }
    }
    return;
  }
  int l = u.L - 1;
  while (wg < u.y[l].first) --l;
  const UpdateLayer& y = u.y[l];
  const int tk = (y.K + 63) / 64, o = wg - y.first;
  const int k0 = (o % tk) * 64 + wave * 32, n0 = (o / tk) * 16;
  const bool on = k0 < y.K && n0 < y.N;
  if (PARTS == 1 && !on) return;
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  f32x4 acc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // masters and moments on their way while the products run
  float4 pw[2], pm[2], pv[2];
  if (ADAM && part == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + 16 * i + (lane >> 4) * 4, n = n0 + fr;
      if (k < y.K && n < y.N) {
        const size_t at = y.woff + (size_t)n * y.K + k;
        pw[i] = *reinterpret_cast<const float4*>(u.P + at);
        pm[i] = *reinterpret_cast<const float4*>(u.M + at);
        pv[i] = *reinterpret_cast<const float4*>(u.V + at);
      }
    }
  }
  constexpr int CH = 4;
#pragma unroll 1
  for (int s0 = 32 * CH * part; s0 < u.B && on; s0 += 32 * CH * PARTS) {
    uint4 a[CH][2], b[CH];
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int bb = s0 + 32 * s + fk, n = n0 + fr;
      b[s] = a[s][0] = a[s][1] = make_uint4(0u, 0u, 0u, 0u);
      const size_t st = (size_t)(s0 / 32 + s) * 512 + lane * 8;
      if (bb < u.B && n < y.N) b[s] = *reinterpret_cast<const uint4*>(y.DT + (size_t)(n0 >> 4) * u.ts * 512 + st);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int k = k0 + 16 * i + fr;
        if (bb < u.B && k < y.K)
          a[s][i] = *reinterpret_cast<const uint4*>(y.HT + (size_t)((k0 >> 4) + i) * u.ts * 512 + st);
      }
    }
#pragma unroll
    for (int s = 0; s < CH; ++s)
      if (s0 + 32 * s < u.B)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s][i]),
                                                           __builtin_bit_cast(bf16x8, b[s]), acc[i], 0, 0, 0);
  }
  if constexpr (PARTS > 1) {
    if (part > 0)
#pragma unroll
      for (int i = 0; i < 2; ++i) sP[part - 1][wave][lane][i] = acc[i];
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int j = 0; j < PARTS - 1; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] += sP[j][wave][lane][i];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = k0 + 16 * i + (lane >> 4) * 4, n = n0 + fr;
    if (k >= y.K || n >= y.N) continue;
    const size_t at = y.woff + (size_t)n * y.K + k;
    if (!ADAM) {
      *reinterpret_cast<float4*>(u.G + at) = make_float4(acc[i][0], acc[i][1], acc[i][2], acc[i][3]);
      continue;
    }
    float4 w = pw[i], m = pm[i], v = pv[i];
    const uint32_t h0 = f2bf(adam_one(w.x, m.x, v.x, acc[i][0], u.a));
    const uint32_t h1 = f2bf(adam_one(w.y, m.y, v.y, acc[i][1], u.a));
    const uint32_t h2 = f2bf(adam_one(w.z, m.z, v.z, acc[i][2], u.a));
    const uint32_t h3 = f2bf(adam_one(w.w, m.w, v.w, acc[i][3], u.a));
    *reinterpret_cast<float4*>(u.P + at) = w;
    *reinterpret_cast<float4*>(u.M + at) = m;
    *reinterpret_cast<float4*>(u.V + at) = v;
    const uint2 hw = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
    if (y.Wf) *reinterpret_cast<uint2*>(y.Wf + pack_pos(n, k, steps_of(y.K))) = hw;
    if (y.Wd) {
      const int sn = steps_of(y.N);
      y.Wd[pack_pos(k, n, sn)] = (bf16_t)h0;
      y.Wd[pack_pos(k + 1, n, sn)] = (bf16_t)h1;
      y.Wd[pack_pos(k + 2, n, sn)] = (bf16_t)h2;
      y.Wd[pack_pos(k + 3, n, sn)] = (bf16_t)h3;
    }
  }
}

// four floats, streaming (NT) or cached
template <bool NT>
__device__ __forceinline__ float4 load4(const float* p) {
  const auto* q = reinterpret_cast<const f32x4*>(p);
  const f32x4 t = NT ? __builtin_nontemporal_load(q) : *q;
  return make_float4(t[0], t[1], t[2], t[3]);
}
template <bool NT>
__device__ __forceinline__ void store4(float* p, float4 v) {
  const f32x4 t = {v.x, v.y, v.z, v.w};
  if (NT) __builtin_nontemporal_store(t, reinterpret_cast<f32x4*>(p));
  else *reinterpret_cast<f32x4*>(p) = t;
}

// k_update of a wide output layer: 32 x 128 (n x k) of W per workgroup of 4
// waves.  The products go to LDS, from where masters, moments and gradients
// move as whole rows and both packed copies as whole fragments.  Bound by its
// 28 bytes per weight: 38,400 x 512 in 110 us (5.2 TB/s; with 256 k 150, with
// 64 183, as k_update's tiles 231; NT: see wide_nt), where the gradient product, the column sums
// and the update took 130.
constexpr int kUpN = 32, kUpK = 128, kUpT = kUpK / 64, kUpLd = kUpK + 4, kUpLb = kUpK + 8;
template <bool ADAM, bool NT>
__global__ __launch_bounds__(256, 3) void k_update_wide(UpdateArgs u, int l) {
  __shared__ __attribute__((aligned(16))) float sG[kUpN * kUpLd];
  __shared__ __attribute__((aligned(16))) bf16_t sW[kUpN * kUpLb];
  __shared__ float sB[kUpN][33];
  const UpdateLayer& y = u.y[l];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tk = (y.K + kUpK - 1) / kUpK;
  const int k0 = (int)(blockIdx.x % tk) * kUpK, n0 = (int)(blockIdx.x / tk) * kUpN;
  const int kw = min(kUpK, y.K - k0), rowq = kw / 4;  // k of this workgroup, pieces of 4 per row
  const bool bias = k0 == 0 && wave == 0;  // its products' rows are the biases' terms
  constexpr int E = kUpN * kUpK / 4 / 256;
  float4 pw[E], pm[E], pv[E];
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  f32x4 acc[kUpT][2];
#pragma unroll
  for (int i = 0; i < kUpT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float sum[2][8] = {};
  constexpr int CH = 4;
  uint4 a[CH][kUpT], b[CH][2];
  auto get = [&](int s0) {
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int bb = s0 + 32 * s + fk;
      const size_t st = (size_t)(s0 / 32 + s) * 512 + lane * 8;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        b[s][j] = make_uint4(0u, 0u, 0u, 0u);
        if (bb < u.B && n0 + 16 * j + fr < y.N)
          b[s][j] = *reinterpret_cast<const uint4*>(y.DT + (size_t)(n0 / 16 + j) * u.ts * 512 + st);
      }
#pragma unroll
      for (int i = 0; i < kUpT; ++i) {
        const int k = (wave * kUpT + i) * 16 + fr;
        a[s][i] = make_uint4(0u, 0u, 0u, 0u);
        if (bb < u.B && k < kw)
          a[s][i] = *reinterpret_cast<const uint4*>(y.HT + (size_t)(k0 / 16 + wave * kUpT + i) * u.ts * 512 + st);
      }
    }
  };
  auto use = [&]() {
#pragma unroll
    for (int s = 0; s < CH; ++s) {
#pragma unroll
      for (int i = 0; i < kUpT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s][i]),
                                                              __builtin_bit_cast(bf16x8, b[s][j]), acc[i][j], 0, 0, 0);
      if (bias)  // column sums in k_colsum's order: the rows 32 apart first
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t h[4] = {b[s][j].x, b[s][j].y, b[s][j].z, b[s][j].w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            sum[j][2 * q] += bf2f((bf16_t)(h[q] & 0xffffu));
            sum[j][2 * q + 1] += bf2f((bf16_t)(h[q] >> 16));
          }
        }
    }
  };
  get(0);
#pragma unroll 1
  for (int s0 = 32 * CH; s0 < u.B; s0 += 32 * CH) {
    use();
    get(s0);
  }
  // masters and moments on their way while the last products run
  if (ADAM) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const int e = tid + 256 * j, n = n0 + e / rowq;
      if (e < kUpN * rowq && n < y.N) {
        const size_t at = y.woff + (size_t)n * y.K + k0 + e % rowq * 4;
        pw[j] = load4<NT>(u.P + at);
        pm[j] = load4<NT>(u.M + at);
        pv[j] = load4<NT>(u.V + at);
      }
    }
  }
  use();
#pragma unroll
  for (int i = 0; i < kUpT; ++i)  // lane: four neighbouring k of one n
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<f32x4*>(sG + (16 * j + fr) * kUpLd + wave * 16 * kUpT + 16 * i + (lane >> 4) * 4) = acc[i][j];
  if (ADAM && kw < kUpK)  // the copies' last steps and tiles are padded with zeros
    for (int e = tid; e < kUpN * kUpLb / 8; e += 256) reinterpret_cast<uint4*>(sW)[e] = make_uint4(0u, 0u, 0u, 0u);
  if (bias)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 8; ++q) sB[16 * j + fr][fk + q] = sum[j][q];
  __syncthreads();
  if (bias && tid < kUpN && n0 + tid < y.N) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < 32; ++q) t += sB[tid][q];
    const size_t i = y.boff + n0 + tid;
    if (ADAM) {
      float w = u.P[i], m = u.M[i], v = u.V[i];
      adam_one(w, m, v, t, u.a);
      u.P[i] = w; u.M[i] = m; u.V[i] = v;
    } else {
      u.G[i] = t;
    }
  }
#pragma unroll
  for (int j = 0; j < E; ++j) {
    const int e = tid + 256 * j;
    if (e >= kUpN * rowq) continue;
    const int r = e / rowq, k = e % rowq * 4, n = n0 + r;
    uint2 hw = make_uint2(0u, 0u);
    if (n < y.N) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(sG + r * kUpLd + k);
      const size_t at = y.woff + (size_t)n * y.K + k0 + k;
      if (!ADAM) {
        *reinterpret_cast<f32x4*>(u.G + at) = g;
        continue;
      }
      float4 w = pw[j], m = pm[j], v = pv[j];
      const uint32_t h0 = f2bf(adam_one(w.x, m.x, v.x, g[0], u.a));
      const uint32_t h1 = f2bf(adam_one(w.y, m.y, v.y, g[1], u.a));
      const uint32_t h2 = f2bf(adam_one(w.z, m.z, v.z, g[2], u.a));
      const uint32_t h3 = f2bf(adam_one(w.w, m.w, v.w, g[3], u.a));
      store4<NT>(u.P + at, w);
      store4<NT>(u.M + at, m);
      store4<NT>(u.V + at, v);
      hw = make_uint2(h0 | (h1 << 16), h2 | (h3 << 16));
    }
    if (ADAM) *reinterpret_cast<uint2*>(sW + r * kUpLb + k) = hw;
  }
  if (!ADAM) return;
  __syncthreads();
  // fragments of both copies: (n tile, k step) and k tile x this n step
  const int sk = steps_of(y.K), sn = steps_of(y.N);
  for (int f = wave; f < kUpK / 8; f += 4) {
    if (f < kUpK / 16) {
      const int t = n0 / 16 + (f & 1), st = k0 / 32 + (f >> 1);
      if (t < tiles_of(y.N) && st < sk)
        *reinterpret_cast<uint4*>(y.Wf + ((size_t)t * sk + st) * 512 + lane * 8) =
            *reinterpret_cast<const uint4*>(sW + ((f & 1) * 16 + fr) * kUpLb + (f >> 1) * 32 + fk);
    } else {
      const int t = k0 / 16 + f - kUpK / 16;
      if (t >= tiles_of(y.K)) continue;
      uint32_t h[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bf16_t* c = sW + (fk + 2 * q) * kUpLb + (f - kUpK / 16) * 16 + fr;
        h[q] = (uint32_t)c[0] | ((uint32_t)c[kUpLb] << 16);
      }
      *reinterpret_cast<uint4*>(y.Wd + ((size_t)t * sn + n0 / 32) * 512 + lane * 8) = make_uint4(h[0], h[1], h[2], h[3]);
    }
  }
}

template <int EPI, bool GATHER>
__global__ __launch_bounds__(128) void k_layer(LayerArgs g) {
  layer_tile<EPI, GATHER>(g, blockIdx.x);
}

// Rows idx of X in bf16 in both fragment orders (a wave per 16 rows x 32
// columns, transposed through LDS): see rows_apart().
__global__ __launch_bounds__(256) void k_rows(const float* __restrict__ X, const int* __restrict__ idx, int B, int K,
                                              int ts, bf16_t* __restrict__ HP, bf16_t* __restrict__ XT) {
  constexpr int LDR = 24;  // 16 rows, padded to keep 16-byte pieces aligned
  __shared__ __attribute__((aligned(16))) bf16_t sX[4][32 * LDR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, steps = steps_of(K);
  const int w = blockIdx.x * 4 + wave, mt = w / steps, k0 = w % steps * 32;
  if (mt * 16 >= B) return;
  const int row = mt * 16 + (lane & 15), q = (lane >> 4) * 8;
  uint32_t v[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  if (row < B && k0 + q < K) {
    const float* x = X + (size_t)idx[row] * K + k0 + q;
    const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
    v[0] = f2bf(a.x); v[1] = f2bf(a.y); v[2] = f2bf(a.z); v[3] = f2bf(a.w);
    v[4] = f2bf(b.x); v[5] = f2bf(b.y); v[6] = f2bf(b.z); v[7] = f2bf(b.w);
  }
  *reinterpret_cast<uint4*>(HP + ((size_t)mt * steps + k0 / 32) * 512 + lane * 8) =
      make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
  bf16_t* s = sX[wave];
#pragma unroll
  for (int r = 0; r < 8; ++r) s[(q + r) * LDR + (lane & 15)] = (bf16_t)v[r];
  wave_lds_sync();
  const int k = lane >> 1, r0 = (lane & 1) * 8;  // widths and batches are multiples of 8
  if (k0 + k < K && mt * 16 + r0 < B)
    *reinterpret_cast<uint4*>(XT + pack_pos(k0 + k, mt * 16 + r0, ts)) =
        *reinterpret_cast<const uint4*>(s + k * LDR + r0);
}

// bf16 copies of every layer's W [N][K] in both fragment orders, a lane's 16
// bytes of a fragment per thread, Wf's fragments first; all layers in one launch
// (with one each and 2-byte stores 32-512x5-64's parameters took 20 us longer)
struct PackLayer {
  const float* W;
  int N, K;
  bf16_t *Wf, *Wd;    // Wd: null for the first layer
  unsigned first;     // workgroup
};
struct PackArgs {
  int L;
  PackLayer y[kSlabL];
};
__global__ __launch_bounds__(256) void k_pack(PackArgs p) {
  int l = p.L - 1;
  while (blockIdx.x < p.y[l].first) --l;
  const PackLayer& y = p.y[l];
  const size_t nf = (size_t)tiles_of(y.N) * steps_of(y.K) * 64, nd = (size_t)tiles_of(y.K) * steps_of(y.N) * 64;
  size_t i = (size_t)(blockIdx.x - y.first) * 256 + threadIdx.x;
  if (i >= nf + (y.Wd ? nd : 0)) return;
  const bool f = i < nf;
  if (!f) i -= nf;
  // row r of the packed matrix, columns c..c + 7: W's row r, or its column r
  const int steps = steps_of(f ? y.K : y.N), lane = (int)(i & 63);
  const int r = (int)(i / 64 / steps) * 16 + (lane & 15), c = (int)(i / 64 % steps) * 32 + (lane >> 4) * 8;
  uint32_t v[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
  if (r < (f ? y.N : y.K) && c < (f ? y.K : y.N))  // widths are multiples of 8
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = f2bf(f ? y.W[(size_t)r * y.K + c + q] : y.W[(size_t)(c + q) * y.K + r]);
  *reinterpret_cast<uint4*>((f ? y.Wf : y.Wd) + i * 8) =
      make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
}

unsigned blocks(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

struct LymphMlp {
  int L = 0, max_batch = 0;
  std::vector<int> w;                  // widths
  std::vector<size_t> woff, boff;      // offsets of W_l, b_l in the parameter vector
  size_t n_params = 0;
  float *P = nullptr, *G = nullptr, *Mo = nullptr, *Vo = nullptr;  // master, grad, Adam
  bf16_t* Wb = nullptr;                // bf16 copy (W parts used; b parts unused)
  std::vector<bf16_t*> H;              // H[0] input .. H[L-1] (bf16 activations)
  std::vector<float*> Z;               // Z[0..L-2] pre-activations
  float* Y = nullptr;                  // [B][w_L]
  bf16_t *dY = nullptr, *dZa = nullptr, *dZb = nullptr;
  float *part = nullptr, *loss = nullptr;
  int* idx = nullptr;
  int n_data = 0;
  float *X = nullptr, *T = nullptr;
  int adam_t = 0;
  float* ws = nullptr;  // split-k partial sums, sized by the largest split GEMM seen
  size_t ws_floats = 0;
  // training's sample order and per-step losses, grown to the longest call
  int* dorder = nullptr;
  size_t dorder_cap = 0;
  float* dloss = nullptr;
  size_t dloss_cap = 0;
  // slab networks (inputs and hidden layers <= kSlabW; wide: the output layer
  // is wider): packed weights, activations and gradients, packed and
  // transposed, and gelu' per tile
  bool slab = false, wide = false;
  bf16_t* hp = nullptr;  // forward of a wide network: the last activations, packed
  size_t hp_cap = 0;
  std::vector<bf16_t*> Wf, Wd, HT, DT, HP, DP;
  std::vector<f32x4*> dg;
  // inputs and outputs of host-side calls: one batch with the network, grown
  // (own) up to upload_rows() and chunk_rows()
  struct Buf {
    float* p = nullptr;
    size_t cap = 0;
    bool own = false;
  } in, out;
  std::vector<void*> owned;
  // every kernel and copy of this network runs on its own stream, so that
  // networks trained from different host threads overlap on the GPU
  hipStream_t stream = nullptr;
};

namespace {

template <class T>
int dalloc(LymphMlp* m, T** p, size_t n) {
  *p = nullptr;
  if (n == 0) n = 1;
  if (hipMalloc((void**)p, n * sizeof(T)) != hipSuccess)
    return fail(LYMPH_MLP_ERR_HIP, "hipMalloc(" + std::to_string(n * sizeof(T)) + " B) failed");
  m->owned.push_back((void*)*p);
  return 0;
}

// Launch: 128 x 128 tiles when they still give >= 256 workgroups, else
// 64 x 64; a GEMM with few tiles and a long k range (the input gradient of the
// output layer: k = 38,400) is split along k over up to kMaxSplit workgroups
// per tile (32 x 32 = 1024 workgroups there) and reduced in order.
constexpr int kMaxSplit = 32;
// parts of a contraction over K for an [M][N] result, of kchunk each
int split_of(int M, int N, int K, int* kchunk) {
  const int TM = blocks(N, 128) * blocks(M, 128) >= 256 ? 128 : 64;
  int S = 1;
  if (blocks(N, TM) * blocks(M, TM) < 256 && K > 1024) S = std::min<int>(kMaxSplit, (K + 1023) / 1024);
  *kchunk = (int)(blocks(blocks(K, S), BK) * BK);
  return (int)blocks(K, *kchunk);
}
// The same for a wide layer's input gradient.  Where the GEMM would not split,
// k_split still does from 4,096 outputs on, into 8 parts (one per XCD): k_layer
// reads W again for every 16 rows.  us per step, k_layer / split: 8-512x3-38,400
// at batch 2,048 1047 / 762, 4,096 2050 / 1478 (the GEMM 1934), 8,192 4032 / 3011
// (3452); 8-512-8,192 at 8,192 901 / 760 (888); 512x2-4,096 at 4,096 239 / 221;
// 8-512-2,048 at 2,048 even, at 16,384 644 / 690.
int wide_parts(int M, int N, int K, int* kchunk) {
  const int S = split_of(M, N, K, kchunk);
  if (S > 1 || K < 4096) return S;
  *kchunk = (int)(blocks(blocks(K, 8), BK) * BK);
  return (int)blocks(K, *kchunk);
}
// split-k workspace: grown on the first call of a larger shape
int need_ws(LymphMlp* m, size_t floats) {
  if (floats <= m->ws_floats) return 0;
  (void)hipStreamSynchronize(m->stream);
  if (m->ws) (void)hipFree(m->ws);
  m->ws = nullptr;
  m->ws_floats = 0;
  if (hipMalloc(&m->ws, floats * sizeof(float)) != hipSuccess)
    return fail(LYMPH_MLP_ERR_HIP, "hipMalloc of the split-k workspace failed");
  m->ws_floats = floats;
  return 0;
}
template <bool A_KC, bool B_KC, int EPI>
int gemm(LymphMlp* m, GemmArgs a) {
  if (a.M <= 0 || a.N <= 0 || a.K <= 0) return 0;
  const bool big = blocks(a.N, 128) * blocks(a.M, 128) >= 256;
  const int TM = big ? 128 : 64;
  const int S = split_of(a.M, a.N, a.K, &a.kchunk);
  a.part = nullptr;
  if (S > 1) {
    if (int rc = need_ws(m, (size_t)S * a.M * a.N)) return rc;
    a.part = m->ws;
  }
  dim3 grid(blocks(a.N, TM), blocks(a.M, TM), S);
  if (big)
    k_gemm<A_KC, B_KC, EPI, 128><<<grid, 256, 0, m->stream>>>(a);
  else
    k_gemm<A_KC, B_KC, EPI, 64><<<grid, 256, 0, m->stream>>>(a);
  if (S > 1) k_splitk<EPI><<<blocks((size_t)a.M * a.N, 256), 256, 0, m->stream>>>(a, S);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : fail(LYMPH_MLP_ERR_HIP, std::string("k_gemm: ") + hipGetErrorString(e));
}

// forward of B rows of H[0]; last layer into Y
int forward(LymphMlp* m, int B) {
  for (int l = 0; l < m->L; ++l) {
    GemmArgs a{};
    a.M = B; a.N = m->w[l + 1]; a.K = m->w[l];
    a.A = m->H[l]; a.lda = m->w[l];
    a.B = m->Wb + m->woff[l]; a.ldb = m->w[l];
    a.ldc = m->w[l + 1];
    a.bias = m->P + m->boff[l];
    if (l + 1 < m->L) {
      a.C32 = m->Z[l];
      a.C16 = m->H[l + 1];
      if (int rc = gemm<true, true, EPI_GELU_FWD>(m, a)) return rc;
    } else {
      a.C32 = m->Y;
      if (int rc = gemm<true, true, EPI_F32>(m, a)) return rc;
    }
  }
  return 0;
}

// loss of Y against T rows idx (device), gradients into G
int backward(LymphMlp* m, int B, const float* T, const int* idx, float* loss_out) {
  const int NL = m->w[m->L];
  const size_t ny = (size_t)B * NL;
  const unsigned nb = blocks(ny, kLossPer);
  k_loss<<<nb, 256, 0, m->stream>>>(m->Y, NL, T, idx, B, 2.0f / (float)ny, m->dY, m->part);
  k_sum<<<1, 256, 0, m->stream>>>(m->part, (int)nb, 1.0f / (float)ny, loss_out);
  bf16_t* dZ = m->dY;
  for (int l = m->L - 1; l >= 0; --l) {
    const int N = m->w[l + 1], K = m->w[l];
    GemmArgs a{};  // dW_l = dZ_l^T H_l
    a.M = N; a.N = K; a.K = B;
    a.A = dZ; a.lda = N;
    a.B = m->H[l]; a.ldb = K;
    a.C32 = m->G + m->woff[l]; a.ldc = K;
    if (int rc = gemm<false, false, EPI_F32>(m, a)) return rc;
    k_colsum<<<blocks(N, 64), 256, 0, m->stream>>>(dZ, B, N, m->G + m->boff[l]);
    if (l > 0) {  // dZ_{l-1} = (dZ_l W_l) * gelu'(Z_{l-1})
      bf16_t* nxt = (dZ == m->dZa) ? m->dZb : m->dZa;
      GemmArgs d{};
      d.M = B; d.N = K; d.K = N;
      d.A = dZ; d.lda = N;
      d.B = m->Wb + m->woff[l]; d.ldb = K;
      d.C16 = nxt; d.ldc = K;
      d.aux = m->Z[l - 1];
      if (int rc = gemm<true, false, EPI_GELU_BWD>(m, d)) return rc;
      dZ = nxt;
    }
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : fail(LYMPH_MLP_ERR_HIP, std::string("backward: ") + hipGetErrorString(e));
}

int grow(LymphMlp* m, LymphMlp::Buf& b, size_t n) {
  if (n <= b.cap) return 0;
  HIP_TRY(hipStreamSynchronize(m->stream));
  float* q = nullptr;
  if (hipMalloc((void**)&q, n * sizeof(float)) != hipSuccess)
    return fail(LYMPH_MLP_ERR_HIP, "hipMalloc(" + std::to_string(n * sizeof(float)) + " B) failed");
  if (b.own) (void)hipFree(b.p);
  b = {q, n, true};
  return 0;
}

// Tiles of 16 per wave and direction of a wide layer's k_wide, 1: k_layer.
// The larger a wave's block, the less of the rows' activations every group of
// columns reads again (256 rows x 38,400: 47 us with 4 x 4 tiles, 57 with 2 x
// 2, 70 with 4 x 1; 40 since wide_nt), as long as about two waves a SIMD are left: 1024 blocks
// of 4 x 4, 512 of 2 x 2.
int wide_tile(int N, int B) {
  const size_t t = (size_t)tiles_of(N) * tiles_of(B);
  return t >= 16 * 1024 ? 4 : t >= 4 * 512 ? 2 : 1;
}
// its launch; returns the waves (entries of the loss sum)
template <int EPI>
int launch_wide(LymphMlp* m, LayerArgs& a) {
  const int T = wide_tile(a.N, a.B), nt = tiles_of(a.N), nm = tiles_of(a.B);
  if (T == 1) {
    k_layer<EPI, false><<<(unsigned)layer_wgs(a.N, a.B), 128, 0, m->stream>>>(a);
    return nt * nm;
  }
  a.rw = nm > 2 * T ? 4 : nm > T ? 2 : 1;
  const unsigned wr = blocks(nm, T * a.rw), cg = blocks(nt, T * (4 / a.rw));
  const unsigned wgs = 8 * blocks(cg, 8) * wr;
  if (T == 4) k_wide<4, EPI><<<wgs, 256, 0, m->stream>>>(a);
  else k_wide<2, EPI><<<wgs, 256, 0, m->stream>>>(a);
  return (int)wgs * 4;
}

// Rows of a forward pass at a time: as many as have 64 MB of inputs or outputs,
// or a batch of up to 150 MB in whole groups of k_wide's 256 rows: beyond, the
// outputs no longer stay in the Infinity Cache on their way out.  ms of a pass of
// 8-512x3-38,400, one launch / pieces (the GEMMs): 2,048 rows 0.246 / 0.183
// (0.207), 4,096 0.463 / 0.366 (0.402); 8-64-32,768, 4,096 rows 0.228 / 0.136
// (0.157).
int chunk_rows(const LymphMlp* m) {
  auto rows = [&](size_t mb) { return (int)((mb << 18) / (unsigned)std::max(m->w[0], m->w[m->L])); };
  const int most = rows(150), whole = most >= 256 ? most / 256 * 256 : std::max(most / 32 * 32, 32);
  return std::max(rows(64) / 32 * 32, std::min(m->max_batch, whole));
}
// Rows of host inputs at a time, whole passes of `pass` rows: at most 64 MB, a
// pass at least.  The buffer stays with the network, so it does not grow with
// the rows of a call.
int upload_rows(const LymphMlp* m, int pass) {
  return std::max(pass, (int)((16u << 20) / (unsigned)m->w[0]) / pass * pass);
}

// Whether a forward pass of up to 32 rows takes a launch per layer, through the
// training's buffers (which hold whole tiles of max_batch rows): in a slab a
// single CU pulls every layer's weights in turn, which past about 300 KB a layer
// takes longer than the launches.  us of a pass, slab / launches (the GEMMs), 1
// row: nine layers of 512 77 / 39 (57), sixteen 136 / 64 (100), six of 512 42 / 28
// (39), 32-512x5-64 36 / 22 (35); eight of 384 (288 KB each) 39 by the slab (42).
bool few_rows_by_layer(const LymphMlp* m, int n, int layers) {
  if (n > 32 || tiles_of(n) > tiles_of(m->max_batch) || layers < 2) return false;
  size_t bytes = 0;
  for (int l = 0; l < layers; ++l) bytes += pack_size(m->w[l + 1], m->w[l]) * sizeof(bf16_t);
  return bytes > (size_t)layers * 300 * 1024;
}

// Outputs of n <= chunk_rows() rows (device).  16 rows a slab until every CU
// has one (4096 rows), then 32: the weights are read once per slab, and two
// slabs of 32 fit a CU's registers.  A wide output layer takes the slabs'
// activations from memory in a launch of its own, which spreads it over the chip.
int slab_forward(LymphMlp* m, int n, const float* X, float* Y) {
  if (n <= 0) return 0;
  SlabArgs a{};
  a.L = m->wide ? m->L - 1 : m->L;
  a.B = n;
  for (int l = 0; l <= a.L; ++l) a.w[l] = m->w[l];
  for (int l = 0; l < a.L; ++l) {
    a.Wf[l] = m->Wf[l];
    a.bias[l] = m->P + m->boff[l];
  }
  a.X = X;
  if (few_rows_by_layer(m, n, a.L)) {
    for (int l = 0; l < m->L; ++l) {
      LayerArgs o{};
      o.N = m->w[l + 1]; o.K = m->w[l]; o.B = n; o.ts = steps_of(m->max_batch);
      o.W = m->Wf[l]; o.in = m->HP[l]; o.bias = m->P + m->boff[l];
      o.X = X; o.XT = m->HT[0]; o.Y = Y;
      const unsigned wgs = (unsigned)layer_wgs(o.N, n);
      if (l + 1 < m->L) {
        o.out = m->HP[l + 1]; o.outT = m->HT[l + 1]; o.dg = m->dg[l];
        if (l == 0) k_layer<LAYER_FWD, true><<<wgs, 128, 0, m->stream>>>(o);
        else k_layer<LAYER_FWD, false><<<wgs, 128, 0, m->stream>>>(o);
      } else if (m->wide) {
        launch_wide<LAYER_OUT>(m, o);
      } else {
        k_layer<LAYER_OUT, false><<<wgs, 128, 0, m->stream>>>(o);
      }
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(LYMPH_MLP_ERR_HIP, std::string("k_layer: ") + hipGetErrorString(e));
  }
  if (m->wide) {
    const size_t need = pack_size((n + 31) / 32 * 32, a.w[a.L]);
    if (need > m->hp_cap) {  // zeros: the padding of the last step is never written
      HIP_TRY(hipStreamSynchronize(m->stream));
      if (m->hp) (void)hipFree(m->hp);
      m->hp = nullptr;
      m->hp_cap = 0;
      HIP_TRY(hipMalloc(&m->hp, need * sizeof(bf16_t)));
      HIP_TRY(hipMemsetAsync(m->hp, 0, need * sizeof(bf16_t), m->stream));
      m->hp_cap = need;
    }
    a.Hp = m->hp;
  } else {
    a.Y = Y;
  }
  if (n <= 4096)
    k_slab<16, 16><<<blocks(n, 16), 512, 0, m->stream>>>(a);
  else
    k_slab<32, 16><<<blocks(n, 32), 512, 0, m->stream>>>(a);
  if (m->wide) {
    const int l = m->L - 1;
    LayerArgs o{};
    o.N = m->w[m->L]; o.K = m->w[l]; o.B = n;
    o.W = m->Wf[l]; o.in = m->hp; o.bias = m->P + m->boff[l]; o.Y = Y;
    launch_wide<LAYER_OUT>(m, o);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : fail(LYMPH_MLP_ERR_HIP, std::string("k_slab: ") + hipGetErrorString(e));
}

// Whether a wide layer's masters and moments are streamed past the caches: from
// half of the Infinity Cache on they push out the packed weights, the gradients
// and the targets that the step's other launches read.  us per step of an
// 8-512x3-N network at batch 256, cached / streamed: 49 MB of them 80.9 / 84.8,
// 98 MB 107 / 112, 123 MB 128 / 129, 147 MB 144 / 139, 184 MB 187 / 159, 236 MB
// (N = 38,400) 235 / 198.
bool wide_nt(const LymphMlp* m) {
  return (size_t)m->w[m->L] * m->w[m->L - 1] * 12 > ((size_t)128 << 20);
}

// Whether a step's input rows are packed by a launch of their own (k_rows).
// Every column tile of the first layer otherwise gathers and converts them
// again, which wide inputs do not hide: us per step, in the layer / apart (both
// with one sum per tile of k_update), one layer of 512 x 512 at batch 256 22 /
// 12, 4,096 100 / 55, 65,536 1610 / 700 (with the GEMMs 28, 75 and 1040); 256 x 256 at 256 15.2 / 12.2.  Inputs of at
// most 128 cost less than the launch: 128-256x2 at batch 512 21.6 / 23.3,
// 64-512 at 1,024 18.5 / 20.8, 32-512x5-64 at 256 56.4 / 57.4.
bool rows_apart(const LymphMlp* m) { return m->w[0] > 128; }

// Pairs of waves per tile of k_update.  With one, a wave walks the whole batch,
// and few tiles (wgs workgroups) leave the chip idle meanwhile; four in a
// workgroup keep four times the loads in flight.  us per step, 1 / 4, at batch
// 2,048 and 16,384: 64-512 32.1 / 21.8 and 191 / 126 (the GEMMs: 44 and 169),
// 8-512 27.2 / 18.4 and 169 / 72 (46 and 135), 512-512 (256 workgroups) 33.2 /
// 24.8 and 190 / 111.  Where the tiles fill the chip both are even: 32-512x5-64
// (1,088) 121 / 126 and 725 / 707.  Smaller batches keep one sum in the rows'
// order (64-512 at 1,024: 18.1 / 13.9; at 256 even).
constexpr int kUpParts = 4;
int update_parts(int wgs, int B) { return B >= 2048 && wgs <= 256 ? kUpParts : 1; }

// One step on rows idx of X, T: gradients into G (adam == null) or applied.
// L forward launches (wide inputs packed by one more), L - 1 backward (a wide
// layer's in two), one update.
int slab_step(LymphMlp* m, int B, const float* X, const float* T, const int* idx, float* loss,
              const AdamArgs* adam) {
  const size_t ny = (size_t)B * m->w[m->L];
  const int L = m->L;
  hipStream_t st = m->stream;
  int n_part = tiles_of(B) * tiles_of(m->w[L]);
  const bool packed = rows_apart(m);
  if (packed)
    k_rows<<<blocks((size_t)tiles_of(B) * steps_of(m->w[0]), 4), 256, 0, st>>>(
        X, idx, B, m->w[0], steps_of(m->max_batch), m->HP[0], m->HT[0]);
  for (int l = 0; l < L; ++l) {
    LayerArgs a{};
    a.N = m->w[l + 1]; a.K = m->w[l]; a.B = B; a.ts = steps_of(m->max_batch);
    a.W = m->Wf[l];
    a.in = m->HP[l];
    a.X = X; a.idx = idx; a.XT = m->HT[0];
    a.bias = m->P + m->boff[l];
    const unsigned wgs = (unsigned)layer_wgs(a.N, B);
    if (l + 1 < L) {
      a.out = m->HP[l + 1]; a.outT = m->HT[l + 1]; a.dg = m->dg[l];
      if (l == 0 && !packed) k_layer<LAYER_FWD, true><<<wgs, 128, 0, st>>>(a);
      else k_layer<LAYER_FWD, false><<<wgs, 128, 0, st>>>(a);
    } else {
      a.out = m->DP[l]; a.outT = m->DT[l];
      a.T = T; a.scale = 2.0f / (float)ny; a.part = m->part;
      if (m->wide) n_part = launch_wide<LAYER_LOSS>(m, a);
      else if (l == 0 && !packed) k_layer<LAYER_LOSS, true><<<wgs, 128, 0, st>>>(a);
      else k_layer<LAYER_LOSS, false><<<wgs, 128, 0, st>>>(a);
    }
  }
  for (int l = L - 1; l >= 1; --l) {  // dZ_{l-1} = (dZ_l W_l) gelu'(z_{l-1})
    LayerArgs a{};
    a.N = m->w[l]; a.K = m->w[l + 1]; a.B = B; a.ts = steps_of(m->max_batch);
    a.W = m->Wd[l];
    a.in = m->DP[l];
    a.out = l > 1 ? m->DP[l - 1] : nullptr; a.outT = m->DT[l - 1]; a.dg = m->dg[l - 1];
    int kchunk = 0;
    const int S = l == L - 1 && m->wide ? wide_parts(B, a.N, a.K, &kchunk) : 1;
    if (S == 1) {
      k_layer<LAYER_BWD, false><<<(unsigned)layer_wgs(a.N, B), 128, 0, st>>>(a);
      continue;
    }
    const int nt = tiles_of(a.N), nm = tiles_of(B);
    if (int rc = need_ws(m, (size_t)S * nt * nm * 256)) return rc;
    f32x4* ws = reinterpret_cast<f32x4*>(m->ws);
    if (nm >= 8)
      k_split<4><<<8 * blocks(S, 8) * blocks(nm, 8) * blocks(nt, 8), 256, 0, st>>>(a, S, kchunk / 32, ws);
    else
      k_split<2><<<8 * blocks(S, 8) * blocks(nm, 4) * blocks(nt, 4), 256, 0, st>>>(a, S, kchunk / 32, ws);
    k_split_end<<<(unsigned)(nt * nm), 64, 0, st>>>(a, S, ws);
  }
  UpdateArgs u{};
  u.L = L;
  u.B = B;
  u.ts = steps_of(m->max_batch);
  u.P = m->P; u.M = m->Mo; u.V = m->Vo; u.G = m->G;
  if (adam) u.a = *adam;
  // a wide layer's weights in a launch of their own where it fills the chip
  const int big = (int)(blocks(m->w[L], kUpN) * blocks(m->w[L - 1], kUpK));
  const int apart = m->wide && big >= 256 ? L - 1 : -1;
  int wgs = 0, bias = 0;
  for (int l = 0; l < L; ++l) {
    UpdateLayer& y = u.y[l];
    y.N = m->w[l + 1];
    y.K = m->w[l];
    y.first = wgs;
    if (l != apart) wgs += (int)(blocks(y.N, 16) * blocks(y.K, 64));
    if (l != apart) bias += y.N / 4;
    y.DT = m->DT[l];
    y.HT = m->HT[l];
    y.woff = m->woff[l];
    y.boff = m->boff[l];
    y.Wf = m->Wf[l];
    y.Wd = m->Wd[l];
  }
  u.first_bias = wgs;
  u.part = m->part;
  u.n_part = n_part;
  u.part_scale = 1.0f / (float)ny;
  u.loss = loss;
  if (apart >= 0) {
    if (!adam) k_update_wide<false, false><<<big, 256, 0, st>>>(u, apart);
    else if (wide_nt(m)) k_update_wide<true, true><<<big, 256, 0, st>>>(u, apart);
    else k_update_wide<true, false><<<big, 256, 0, st>>>(u, apart);
  }
  if (update_parts(wgs, B) > 1) {
    if (adam) k_update<true, kUpParts><<<wgs + bias + 1, 128 * kUpParts, 0, st>>>(u);
    else k_update<false, kUpParts><<<wgs + bias + 1, 128 * kUpParts, 0, st>>>(u);
  } else {
    if (adam) k_update<true, 1><<<wgs + bias + 1, 128, 0, st>>>(u);
    else k_update<false, 1><<<wgs + bias + 1, 128, 0, st>>>(u);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : fail(LYMPH_MLP_ERR_HIP, std::string("training step: ") + hipGetErrorString(e));
}

int need(const LymphMlp* m) { return m ? 0 : fail(LYMPH_MLP_ERR_ARG, "null network"); }

}  // namespace

extern "C" {

const char* lymph_mlp_last_error(void) { return g_err.c_str(); }

int lymph_mlp_destroy(LymphMlp* m) {
  if (!m) return 0;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  for (void* p : m->owned) (void)hipFree(p);
  if (m->ws) (void)hipFree(m->ws);
  if (m->hp) (void)hipFree(m->hp);
  if (m->dorder) (void)hipFree(m->dorder);
  if (m->dloss) (void)hipFree(m->dloss);
  if (m->in.own) (void)hipFree(m->in.p);
  if (m->out.own) (void)hipFree(m->out.p);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return 0;
}

int lymph_mlp_create(int n_layers, const int32_t* widths, int max_batch, LymphMlp** out) {
  if (!out) return fail(LYMPH_MLP_ERR_ARG, "out is null");
  *out = nullptr;
  if (n_layers < 1 || !widths) return fail(LYMPH_MLP_ERR_ARG, "need at least one layer");
  if (max_batch < 8 || max_batch % 8) return fail(LYMPH_MLP_ERR_ARG, "max_batch must be a positive multiple of 8");
  for (int l = 0; l <= n_layers; ++l)
    if (widths[l] < 8 || widths[l] % 8) return fail(LYMPH_MLP_ERR_ARG, "widths must be positive multiples of 8");
  int dev = 0;
  if (hipGetDeviceCount(&dev) != hipSuccess || dev == 0)
    return fail(LYMPH_MLP_ERR_HIP, "no HIP device: liblymph_mlp needs an MI355X (gfx950)");
  auto* m = new LymphMlp;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
    delete m;
    return fail(LYMPH_MLP_ERR_HIP, "hipStreamCreate failed");
  }
  m->L = n_layers;
  m->max_batch = max_batch;
  m->w.assign(widths, widths + n_layers + 1);
  size_t off = 0;
  int maxh = 8;
  for (int l = 0; l < n_layers; ++l) {
    m->woff.push_back(off);
    off += (size_t)m->w[l + 1] * m->w[l];
    m->boff.push_back(off);
    off += (size_t)m->w[l + 1];
    if (l + 1 < n_layers) maxh = std::max(maxh, m->w[l + 1]);
  }
  m->n_params = off;
  // one allocation: the buffers that start as zeros first, then the others
  struct Want { void** p; size_t bytes; };
  std::vector<Want> zeros, rest;
  auto zero = [&](auto** p, size_t n) { zeros.push_back({(void**)p, n * sizeof(**p)}); };
  auto al = [&](auto** p, size_t n) { rest.push_back({(void**)p, n * sizeof(**p)}); };
  zero(&m->P, off);
  zero(&m->Mo, off);
  zero(&m->Vo, off);
  al(&m->G, off);
  const int NL = m->w[n_layers];
  m->wide = n_layers > 1 && NL > kSlabW;
  m->slab = n_layers <= kSlabL && *std::max_element(m->w.begin(), m->w.end() - 1) <= kSlabW &&
            (NL <= kSlabW || m->wide);
  m->wide = m->wide && m->slab;
  if (m->slab) {
    for (auto* v : {&m->Wf, &m->Wd, &m->HT, &m->DT, &m->HP, &m->DP}) v->assign(n_layers, nullptr);
    m->dg.assign(n_layers, nullptr);
    for (int l = 0; l < n_layers; ++l) {
      const int N = m->w[l + 1], K = m->w[l];
      zero(&m->Wf[l], pack_size(N, K));
      al(&m->HT[l], pack_size(K, max_batch));
      al(&m->DT[l], pack_size(N, max_batch));
      if (l > 0) {  // operands of the next layer's launch, either way
        zero(&m->Wd[l], pack_size(K, N));
        zero(&m->HP[l], pack_size(max_batch, K));
        zero(&m->DP[l], pack_size(max_batch, N));
      }
      if (l == 0 && rows_apart(m)) al(&m->HP[0], pack_size(max_batch, K));
      if (l + 1 < n_layers) al(&m->dg[l], (size_t)tiles_of(max_batch) * tiles_of(N) * 64);
    }
  } else {
    zero(&m->Wb, off);
    m->H.assign(n_layers, nullptr);
    m->Z.assign(n_layers, nullptr);
    for (int l = 0; l < n_layers; ++l) al(&m->H[l], (size_t)max_batch * m->w[l]);
    for (int l = 0; l + 1 < n_layers; ++l) al(&m->Z[l], (size_t)max_batch * m->w[l + 1]);
    al(&m->Y, (size_t)max_batch * NL);
    al(&m->dY, (size_t)max_batch * NL);
    al(&m->dZa, (size_t)max_batch * maxh);
    al(&m->dZb, (size_t)max_batch * maxh);
  }
  // k_loss: a sum per workgroup; the layer kernels: one per wave, of whole
  // groups of 8 workgroups (launch_wide: 2 x 2 tiles a wave or more)
  const size_t mt = tiles_of(max_batch), nt = tiles_of(NL);
  al(&m->part, std::max((size_t)blocks((size_t)max_batch * NL, 256), mt * nt + 16 * mt + 2 * nt + 128));
  al(&m->loss, 1);
  al(&m->idx, (size_t)max_batch);
  m->in.cap = (size_t)max_batch * m->w[0];
  m->out.cap = (size_t)max_batch * NL;
  al(&m->in.p, m->in.cap);
  al(&m->out.p, m->out.cap);
  size_t total = 0, cleared = 0;
  for (auto* v : {&zeros, &rest}) {
    for (auto& q : *v) total += (q.bytes + 255) / 256 * 256;
    if (v == &zeros) cleared = total;
  }
  char* base = nullptr;
  if (int rc = dalloc(m, &base, total)) {
    lymph_mlp_destroy(m);
    return rc;
  }
  for (auto* v : {&zeros, &rest})
    for (auto& q : *v) {
      *q.p = base;
      base += (q.bytes + 255) / 256 * 256;
    }
  if (hipMemsetAsync(m->P, 0, cleared, m->stream) != hipSuccess ||
      hipStreamSynchronize(m->stream) != hipSuccess) {
    lymph_mlp_destroy(m);
    return fail(LYMPH_MLP_ERR_HIP, "hipMemset failed");
  }
  *out = m;
  return 0;
}

int lymph_mlp_n_params(const LymphMlp* m, int64_t* n) {
  if (int rc = need(m)) return rc;
  if (n) *n = (int64_t)m->n_params;
  return 0;
}

int lymph_mlp_set_params(LymphMlp* m, const float* p) {
  if (int rc = need(m)) return rc;
  if (!p) return fail(LYMPH_MLP_ERR_ARG, "null params");
  HIP_TRY(hipMemcpyAsync(m->P, p, m->n_params * 4, hipMemcpyHostToDevice, m->stream));
  if (m->slab) {
    PackArgs p{};
    p.L = m->L;
    unsigned wgs = 0;
    for (int l = 0; l < m->L; ++l) {
      const int N = m->w[l + 1], K = m->w[l];
      p.y[l] = {m->P + m->woff[l], N, K, m->Wf[l], m->Wd[l], wgs};
      const size_t nf = (size_t)tiles_of(N) * steps_of(K), nd = (size_t)tiles_of(K) * steps_of(N);
      wgs += blocks((nf + (m->Wd[l] ? nd : 0)) * 64, 256);
    }
    k_pack<<<wgs, 256, 0, m->stream>>>(p);
  } else {
    k_to_bf16<<<blocks(m->n_params, 256), 256, 0, m->stream>>>(m->P, m->Wb, m->n_params);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemsetAsync(m->Mo, 0, m->n_params * 4, m->stream));
  HIP_TRY(hipMemsetAsync(m->Vo, 0, m->n_params * 4, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  m->adam_t = 0;
  return 0;
}

int lymph_mlp_get_params(const LymphMlp* m, float* p) {
  if (int rc = need(m)) return rc;
  if (!p) return fail(LYMPH_MLP_ERR_ARG, "null params");
  HIP_TRY(hipMemcpyAsync(p, m->P, m->n_params * 4, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return 0;
}

int lymph_mlp_set_data(LymphMlp* m, int n, const float* x, const float* y) {
  if (int rc = need(m)) return rc;
  if (n < 1 || !x || !y) return fail(LYMPH_MLP_ERR_ARG, "empty data set");
  const size_t nx = (size_t)n * m->w[0], ny = (size_t)n * m->w[m->L];
  (void)hipStreamSynchronize(m->stream);
  for (float** q : {&m->X, &m->T})
    if (*q) {
      for (auto& o : m->owned)
        if (o == (void*)*q) o = nullptr;
      (void)hipFree(*q);
      *q = nullptr;
    }
  if (int rc = dalloc(m, &m->X, nx)) return rc;
  if (int rc = dalloc(m, &m->T, ny)) return rc;
  HIP_TRY(hipMemcpyAsync(m->X, x, nx * 4, hipMemcpyHostToDevice, m->stream));
  HIP_TRY(hipMemcpyAsync(m->T, y, ny * 4, hipMemcpyHostToDevice, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  m->n_data = n;
  return 0;
}

int lymph_mlp_train(LymphMlp* m, int n_steps, int batch, const int32_t* order, float lr,
                    float beta1, float beta2, float eps, float* losses) {
  if (int rc = need(m)) return rc;
  if (!m->X) return fail(LYMPH_MLP_ERR_STATE, "no training data: call lymph_mlp_set_data");
  if (batch < 8 || batch > m->max_batch || batch % 8)
    return fail(LYMPH_MLP_ERR_ARG, "batch must be a multiple of 8 and at most max_batch");
  if (n_steps < 0 || !order) return fail(LYMPH_MLP_ERR_ARG, "bad steps/order");
  for (size_t i = 0; i < (size_t)n_steps * batch; ++i)
    if (order[i] < 0 || order[i] >= m->n_data) return fail(LYMPH_MLP_ERR_ARG, "sample index out of range");
  const size_t n_order = std::max<size_t>(1, (size_t)n_steps * batch);
  const size_t n_loss = std::max<size_t>(1, (size_t)n_steps);
  if (n_order > m->dorder_cap || n_loss > m->dloss_cap) {  // grown, then reused by later calls
    HIP_TRY(hipStreamSynchronize(m->stream));
    if (m->dorder) (void)hipFree(m->dorder);
    if (m->dloss) (void)hipFree(m->dloss);
    m->dorder = nullptr;
    m->dloss = nullptr;
    m->dorder_cap = m->dloss_cap = 0;
    HIP_TRY(hipMalloc(&m->dorder, sizeof(int) * n_order));
    HIP_TRY(hipMalloc(&m->dloss, sizeof(float) * n_loss));
    m->dorder_cap = n_order;
    m->dloss_cap = n_loss;
  }
  int* dorder = m->dorder;
  float* dloss = m->dloss;
  HIP_TRY(hipMemcpyAsync(dorder, order, sizeof(int) * (size_t)n_steps * batch, hipMemcpyHostToDevice,
                         m->stream));
  int rc = 0;
  for (int s = 0; s < n_steps && !rc; ++s) {
    const int* idx = dorder + (size_t)s * batch;
    m->adam_t++;
    const AdamArgs ad{lr, beta1, beta2, eps, 1.0f / (1.0f - std::pow(beta1, (float)m->adam_t)),
                      1.0f / (1.0f - std::pow(beta2, (float)m->adam_t))};
    if (m->slab) {
      rc = slab_step(m, batch, m->X, m->T, idx, dloss + s, &ad);
      if (rc) m->adam_t--;
      continue;
    }
    k_gather<<<blocks((size_t)batch * m->w[0], 256), 256, 0, m->stream>>>(m->X, m->w[0], idx, batch, m->H[0]);
    rc = forward(m, batch);
    if (!rc) rc = backward(m, batch, m->T, idx, dloss + s);
    if (rc) {
      m->adam_t--;
    } else {
      k_adam<<<blocks(m->n_params, 256), 256, 0, m->stream>>>(m->P, m->Mo, m->Vo, m->G, m->Wb, m->n_params, ad);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) rc = fail(LYMPH_MLP_ERR_HIP, std::string("k_adam: ") + hipGetErrorString(e));
    }
  }
  if (!rc && losses && n_steps > 0 &&
      hipMemcpyAsync(losses, dloss, sizeof(float) * n_steps, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    rc = fail(LYMPH_MLP_ERR_HIP, "loss copy failed");
  if (hipStreamSynchronize(m->stream) != hipSuccess && !rc) rc = fail(LYMPH_MLP_ERR_HIP, "training failed");
  return rc;
}

int lymph_mlp_gradients(LymphMlp* m, int batch, const float* x, const float* y, float* grads,
                        float* loss) {
  if (int rc = need(m)) return rc;
  if (batch < 8 || batch > m->max_batch || batch % 8)
    return fail(LYMPH_MLP_ERR_ARG, "batch must be a multiple of 8 and at most max_batch");
  if (!x || !y) return fail(LYMPH_MLP_ERR_ARG, "null batch");
  const size_t nx = (size_t)batch * m->w[0], ny = (size_t)batch * m->w[m->L];
  if (int rc = grow(m, m->in, nx)) return rc;
  if (int rc = grow(m, m->out, ny)) return rc;
  float *dx = m->in.p, *dy = m->out.p;
  std::vector<int> id(batch);
  for (int i = 0; i < batch; ++i) id[i] = i;
  int rc = 0;
  if (hipMemcpyAsync(dx, x, nx * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
      hipMemcpyAsync(dy, y, ny * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
      hipMemcpyAsync(m->idx, id.data(), 4 * batch, hipMemcpyHostToDevice, m->stream) != hipSuccess)
    rc = fail(LYMPH_MLP_ERR_HIP, "upload failed");
  if (!rc && m->slab) {
    rc = slab_step(m, batch, dx, dy, m->idx, m->loss, nullptr);
  } else if (!rc) {
    k_gather<<<blocks(nx, 256), 256, 0, m->stream>>>(dx, m->w[0], m->idx, batch, m->H[0]);
    rc = forward(m, batch);
    if (!rc) rc = backward(m, batch, dy, m->idx, m->loss);
  }
  if (!rc && grads &&
      hipMemcpyAsync(grads, m->G, m->n_params * 4, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    rc = fail(LYMPH_MLP_ERR_HIP, "gradient copy failed");
  if (!rc && loss && hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    rc = fail(LYMPH_MLP_ERR_HIP, "loss copy failed");
  if (hipStreamSynchronize(m->stream) != hipSuccess && !rc) rc = fail(LYMPH_MLP_ERR_HIP, "gradients failed");
  return rc;
}

int lymph_mlp_predict(LymphMlp* m, int n, const float* x, float* y) {
  if (int rc = need(m)) return rc;
  if (n < 0 || (n > 0 && (!x || !y))) return fail(LYMPH_MLP_ERR_ARG, "bad inputs");
  const int w0 = m->w[0], NL = m->w[m->L];
  const int pass = m->slab ? chunk_rows(m) : m->max_batch, up = upload_rows(m, pass);
  if (int rc = grow(m, m->in, (size_t)std::min(n, up) * w0)) return rc;
  if (m->slab)
    if (int rc = grow(m, m->out, (size_t)std::min(n, pass) * NL)) return rc;
  const float* dx = m->in.p;
  int rc = 0;
  std::vector<int> id(m->slab ? 0 : m->max_batch);
  for (int i = 0; i < (int)id.size(); ++i) id[i] = i;
  if (!m->slab &&
      hipMemcpyAsync(m->idx, id.data(), 4 * id.size(), hipMemcpyHostToDevice, m->stream) != hipSuccess)
    rc = fail(LYMPH_MLP_ERR_HIP, "upload failed");
  for (int b0 = 0; b0 < n && !rc; b0 += pass) {
    const int B = std::min(pass, n - b0), at = b0 % up;  // up is a multiple of pass
    if (at == 0 && hipMemcpyAsync(m->in.p, x + (size_t)b0 * w0, (size_t)std::min(up, n - b0) * w0 * 4,
                                  hipMemcpyHostToDevice, m->stream) != hipSuccess) {
      rc = fail(LYMPH_MLP_ERR_HIP, "upload failed");
      break;
    }
    const float* xb = dx + (size_t)at * w0;
    if (m->slab) {
      rc = slab_forward(m, B, xb, m->out.p);
    } else {
      k_gather<<<blocks((size_t)B * w0, 256), 256, 0, m->stream>>>(xb, w0, m->idx, B, m->H[0]);
      rc = forward(m, B);
    }
    if (!rc && hipMemcpyAsync(y + (size_t)b0 * NL, m->slab ? m->out.p : m->Y, (size_t)B * NL * 4,
                              hipMemcpyDeviceToHost, m->stream) != hipSuccess)
      rc = fail(LYMPH_MLP_ERR_HIP, "download failed");
  }
  if (hipStreamSynchronize(m->stream) != hipSuccess && !rc) rc = fail(LYMPH_MLP_ERR_HIP, "prediction failed");
  return rc;
}

int lymph_mlp_time_predict(LymphMlp* m, int n, int reps, double* ms) {
  if (int rc = need(m)) return rc;
  if (!m->X || n < 1 || n > m->n_data || reps < 1) return fail(LYMPH_MLP_ERR_ARG, "bad n/reps or no data");
  std::vector<int> id(m->max_batch);
  for (int i = 0; i < m->max_batch; ++i) id[i] = i;
  HIP_TRY(hipMemcpyAsync(m->idx, id.data(), 4 * m->max_batch, hipMemcpyHostToDevice, m->stream));
  const int chunk = chunk_rows(m);
  if (m->slab)
    if (int rc = grow(m, m->out, (size_t)std::min(n, chunk) * m->w[m->L])) return rc;
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  int rc = 0;
  HIP_TRY(hipEventRecord(e0, m->stream));
  for (int r = 0; r < reps && !rc; ++r) {
    if (m->slab) {
      for (int b0 = 0; b0 < n && !rc; b0 += chunk)
        rc = slab_forward(m, std::min(chunk, n - b0), m->X + (size_t)b0 * m->w[0], m->out.p);
      continue;
    }
    for (int b0 = 0; b0 < n && !rc; b0 += m->max_batch) {
      const int B = std::min(m->max_batch, n - b0);
      k_gather<<<blocks((size_t)B * m->w[0], 256), 256, 0, m->stream>>>(m->X + (size_t)b0 * m->w[0], m->w[0],
                                                          m->idx, B, m->H[0]);
      rc = forward(m, B);
    }
  }
  HIP_TRY(hipEventRecord(e1, m->stream));
  HIP_TRY(hipEventSynchronize(e1));
  float f = 0.f;
  HIP_TRY(hipEventElapsedTime(&f, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (ms) *ms = f / reps;
  return rc;
}

}  // extern "C"
