// surrogate.hip -- the learned node-interval surrogate on MI355X (gfx950):
// a bf16 MLP on the MFMA units (forward, backward, Adam), the node encode
// and gate kernels, and the surrogate evolve that routes rejected nodes to
// the FP64 integrator.  C ABI of include/gal_surrogate.h.
//
// Matrix products are v_mfma_f32_16x16x32_bf16 tiles with fp32 accumulators.
// Inference runs the four layers in one kernel (mlp_forward_fused), a training
// step is three launches (train_rows_kernel, train_weights_kernel,
// adam_kernel).  Weight gradients are split over the batch, every split writes
// its own fp32 partial sum and the Adam kernel adds them in a fixed order, so
// training is deterministic.  gemm_kernel is the plain layer by layer product
// that the fused forward is compared with: each 256-thread workgroup owns a
// 64 x 64 tile, each of its four waves a 32 x 32 quarter, operand tiles of
// 64 x 32 staged in LDS as [row][k].
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cmath>
#include <vector>
#include <algorithm>

#include "../../include/gal_ode.h"
#include "../../include/gal_surrogate.h"
#include "constants.hpp"
#include "physics.hpp"
#include "batch.hpp"

using namespace gal;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // in a caller's buffer of floats

constexpr int kIn = GAL_MLP_INPUTS, kHid = GAL_MLP_HIDDEN, kOut = GAL_MLP_OUTPUTS, kOutLd = GAL_MLP_OUT_LD;
constexpr int kLayers = 4;
constexpr int kFanIn[kLayers] = {kIn, kHid, kHid, kHid};
constexpr int kFanOut[kLayers] = {kHid, kHid, kHid, kOut};
constexpr int kLdW[kLayers] = {kHid, kHid, kHid, kOutLd};  // bf16 weight row stride (fan_out padded to 8)

constexpr int64_t param_count() {
  int64_t p = 0;
  for (int l = 0; l < kLayers; ++l) p += (int64_t)kFanIn[l] * kFanOut[l] + kFanOut[l];
  return p;
}
constexpr int64_t kParams = param_count();

// ---- bf16 ------------------------------------------------------------------
// round to nearest even; NaN stays quiet NaN (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
// two or four values in one instruction each two
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ __forceinline__ uint2 f2bf4(f32x4 v) { return make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3])); }
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

// SiLU, z / (1 + exp(-z)).  The network's epilogues are bound by vector
// instructions, and an IEEE division is eleven of them with two changes of
// the denormal mode.  The quotient from the hardware reciprocal and one
// residual correction is four: q = z r, q + r (z - d q), where the residual
// is exact in one fma, so the result is the correctly rounded quotient but
// for ties within 2^-46.  That holds while d = 1 + exp(-z) and z are far
// from the ends of the range; beyond |z| = 80 (and for infinities, where the
// residual would be NaN) silu_far divides.  A NaN takes either to NaN.
constexpr float kSiluNear = 80.0f;
__device__ __forceinline__ float silu_near(float z) {
  const float d = 1.0f + __expf(-z);
  const float r = __builtin_amdgcn_rcpf(d);
  const float q = z * r;
  return fmaf(fmaf(-d, q, z), r, q);
}
__device__ __forceinline__ float silu_far(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu(float z) {   // both, and a select
  const float near = silu_near(z), far = silu_far(z);
  return fabsf(z) > kSiluNear ? far : near;
}
__device__ __forceinline__ float abs_max4(f32x4 z) {
  return fmaxf(fmaxf(fabsf(z[0]), fabsf(z[1])), fmaxf(fabsf(z[2]), fabsf(z[3])));
}
// Its derivative, with the same two forms of the logistic function.
template <bool FAR>
__device__ __forceinline__ float dsilu(float z) {
  const float d = 1.0f + __expf(-z);
  const float r = __builtin_amdgcn_rcpf(d);
  const float s = FAR && fabsf(z) > kSiluNear ? 1.0f / d : fmaf(fmaf(-d, r, 1.0f), r, r);
  return s * (1.0f + z * (1.0f - s));
}

// ---- MFMA GEMM ---------------------------------------------------------------
constexpr int TM = 64, TN = 64, TK = 32, LDT = TK + 8;
enum Epi { EPI_SILU = 0, EPI_LINEAR = 1 };

struct GemmArgs {
  const uint16_t* A;  // [m][k], row stride lda
  const uint16_t* B;  // [k][n], row stride ldb
  int M, N, K, lda, ldb, ldc;
  int n_valid;        // epilogue writes columns n < n_valid
  const float* bias;
  uint16_t* out_bf;   // SILU: activation
  float* out_f;       // LINEAR: output
};

template <int EPI>
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[TM * LDT];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[TN * LDT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  for (int k0 = 0; k0 < g.K; k0 += TK) {
    {  // rows of A are contiguous in k
      const int r = tid >> 2, c = (tid & 3) * 8;
      uint4 v = zero;
      if (m0 + r < g.M && k0 + c < g.K) v = *reinterpret_cast<const uint4*>(g.A + (size_t)(m0 + r) * g.lda + k0 + c);
      *reinterpret_cast<uint4*>(As + r * LDT + c) = v;
    }
    {  // B: contiguous in n, transposed into LDS
      const int kk = tid >> 3, c = (tid & 7) * 8;
      uint4 v = zero;
      if (k0 + kk < g.K && n0 + c < g.N) v = *reinterpret_cast<const uint4*>(g.B + (size_t)(k0 + kk) * g.ldb + n0 + c);
      const uint16_t* e = reinterpret_cast<const uint16_t*>(&v);
#pragma unroll
      for (int j = 0; j < 8; ++j) Bs[(c + j) * LDT + kk] = e[j];
    }
    __syncthreads();
    bf16x8 a[2], b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(As + (wm * 32 + i * 16 + (lane & 15)) * LDT + (lane >> 4) * 8);
      a[i] = __builtin_bit_cast(bf16x8, v);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint4 v = *reinterpret_cast<const uint4*>(Bs + (wn * 32 + j * 16 + (lane & 15)) * LDT + (lane >> 4) * 8);
      b[j] = __builtin_bit_cast(bf16x8, v);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    __syncthreads();
  }
  // C(m, n) of accumulator register r: m = 4*(lane/16) + r, n = lane % 16 within the 16 x 16 tile.
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * 32 + i * 16 + (lane >> 4) * 4 + r;
        const int n = n0 + wn * 32 + j * 16 + (lane & 15);
        if (m >= g.M || n >= g.n_valid) continue;
        const float c = acc[i][j][r];
        const size_t o = (size_t)m * g.ldc + n;
        const float z = c + g.bias[n];
        if (EPI == EPI_SILU) {
          // as in the fused kernel: the division only where some lane needs it
          // (100,000 rows 213 us; both forms for every value 225 us, a
          // division for every value 220 us)
          float h;
          if (__builtin_expect(__any(fabsf(z) > kSiluNear), 0)) h = silu(z);
          else h = silu_near(z);
          g.out_bf[o] = f2bf(h);
        } else {
          g.out_f[o] = z;
        }
      }
}

// ---- weights in fragment order ------------------------------------------------
// The fused kernels read a wave's MFMA operand of weights, 16 columns x 32 k
// with eight consecutive k per lane, as one contiguous KiB: fragment
// (c / 16, k / 32), lane 16 (k / 8 mod 4) + c mod 16, element k mod 8.  From
// rows of 512 bytes the same operand touches 16 cache lines and uses half of
// each.
__host__ __device__ constexpr size_t frag_offset(int c, int k, int n_k) {
  return ((size_t)(c / 16) * (n_k / 32) + k / 32) * 512 + ((k / 8) % 4 * 16 + c % 16) * 8 + k % 8;
}

// ---- fused inference forward ---------------------------------------------
// The whole network for FR rows per workgroup in one kernel: the rows'
// activations stay in LDS from layer to layer.  Wave w computes all rows x
// columns [64w, 64w+64) of a hidden layer, and one of the two column tiles of
// half the rows of the output layer.  A wave's columns are its own, so it
// reads its weight fragments straight from memory in fragment order into
// registers, KG k chunks at a time, with no LDS staging and no workgroup
// barrier inside a layer.  The weights are the MFMA's A operand, so a lane
// ends with four consecutive columns of one row: it adds one bias vector,
// rounds two values per instruction and writes 8 bytes to LDS (16 to the
// output).  The arithmetic is the per-layer GEMMs' (same products, same k
// order, same bias + SiLU epilogue and bf16 rounding), so the outputs are
// bit-identical to them.
//
// Bound by the epilogue's vector instructions, ten for each activation, beside
// 16 x 16 x 32 products that take a third as long; four waves on a SIMD hide
// some of the products and waits under them.  500,000 rows with their output
// buffer: 254 us with 64 rows per workgroup, 260 us with 128 rows and two waves
// on a SIMD (interleaving one half's products with the other half's epilogue
// within each wave: 264), and 420 us with an IEEE division, the bf16 rounding
// in integer instructions, two-byte LDS writes and weights read from
// transposed rows that each call copied anew.
//
// Few rows are bound by the chain of the four layers instead, and 32 rows per
// workgroup make it shorter and the workgroups more: 1000 rows 9 us against 14
// (128 rows: 22), 20,000 rows 18 against 22.  From 32,768 rows on they would no
// longer all be on the chip at once, and 60,000 rows take 42 us against 40.
constexpr int LDH = kHid + 8;           // activation row stride (bf16)
constexpr int LDX = kIn + 8;            // input row stride (bf16)
constexpr int kFewRows = 32768;
constexpr int kManyRows = 64;           // rows per workgroup of more than kFewRows
constexpr int kFusedThreads = 256;
// Rows of one launch: a launch of 2^32 threads or more is refused.
constexpr int64_t kLaunchRows = int64_t{1} << 29;
static_assert((kLaunchRows + kManyRows - 1) / kManyRows * kFusedThreads < (int64_t{1} << 32),
              "a launch must have fewer than 2^32 threads");

struct FusedArgs {
  const uint16_t* x;                 // [n][kIn] bf16
  const uint16_t* wf[kLayers];       // bf16, fragment order: frag_offset(n, k, kFanIn[l])
  const float* bias[kLayers];
  float* out;                        // [n][kOutLd]
  int n;
};

template <int FR, int KG_MAX, int K, bool LAST>
__device__ __forceinline__ void fused_layer(const FusedArgs& a, int l, const uint16_t* __restrict__ A, int lda,
                                            uint16_t* __restrict__ H, int r0) {
  constexpr int NK = K / TK;
  constexpr int KG = NK < KG_MAX ? NK : KG_MAX;                    // k chunks per register group
  constexpr int JT = LAST ? 1 : 4;                       // column tiles per wave
  // the wave's number as a scalar: so are its addresses, but for the lane
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nbase = LAST ? (wave & 1) * 16 : wave * 64;
  constexpr int IT = LAST ? FR / 32 : FR / 16;           // row tiles per wave
  const int ibase = LAST ? (wave >> 1) * IT : 0;
  const uint16_t* __restrict__ wf = a.wf[l] + (size_t)(nbase / 16) * NK * 512 + lane * 8;
  f32x4 acc[IT][JT];
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  {
    for (int g0 = 0; g0 < NK; g0 += KG) {
      uint4 bq[KG][JT];
#pragma unroll
      for (int kk = 0; kk < KG; ++kk)
#pragma unroll
        for (int j = 0; j < JT; ++j)
          bq[kk][j] = *reinterpret_cast<const uint4*>(wf + (size_t)(j * NK + g0 + kk) * 512);
#pragma unroll
      for (int kk = 0; kk < KG; ++kk) {
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          const uint4 v = *reinterpret_cast<const uint4*>(A + ((ibase + i) * 16 + (lane & 15)) * lda + (g0 + kk) * TK +
                                                          (lane >> 4) * 8);
          const bf16x8 av = __builtin_bit_cast(bf16x8, v);
#pragma unroll
          for (int j = 0; j < JT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bq[kk][j]), av, acc[i][j],
                                                                0, 0, 0);
        }
      }
    }
  }
  // every wave has read this layer's input before any epilogue overwrites H
  __syncthreads();
  // column nbase + 16 j + 4 (lane / 16) + r of row 16 i + lane mod 16
  const int c0 = nbase + (lane >> 4) * 4;
  const float* __restrict__ bias = a.bias[l];
  f32x4 b[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) b[j][r] = bias[LAST ? min(c0 + r, kOut - 1) : c0 + j * 16 + r];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int row = (ibase + i) * 16 + (lane & 15);
    if (LAST) {
      if (r0 + row >= a.n) continue;
      const f32x4 z = acc[i][0] + b[0];
      float* o = a.out + (size_t)(r0 + row) * kOutLd + c0;
      if (c0 + 3 < kOut) {
        *reinterpret_cast<f32x4_a4*>(o) = z;
      } else {
        o[0] = z[0]; o[1] = z[1]; o[2] = z[2];
      }
    } else {
      float far = 0.0f;
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        acc[i][j] += b[j];
        far = fmaxf(far, abs_max4(acc[i][j]));
      }
      uint16_t* h = H + row * LDH + c0;
      if (__builtin_expect(__any(far > kSiluNear), 0)) {   // uniform: the rare block lies apart
#pragma unroll
        for (int j = 0; j < JT; ++j) {
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = silu(acc[i][j][r]);
          *reinterpret_cast<uint2*>(h + j * 16) = f2bf4(v);
        }
      } else {
#pragma unroll
        for (int j = 0; j < JT; ++j) {
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = silu_near(acc[i][j][r]);
          *reinterpret_cast<uint2*>(h + j * 16) = f2bf4(v);
        }
      }
    }
  }
}

template <int FR, int KG>
__global__ __launch_bounds__(kFusedThreads, 4) void mlp_forward_fused(FusedArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t H[FR * LDH];
  __shared__ __attribute__((aligned(16))) uint16_t X[FR * LDX];
  const int tid = threadIdx.x;
  const int r0 = blockIdx.x * FR;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  for (int e = tid; e < FR * (kIn / 8); e += kFusedThreads) {
    const int r = e / (kIn / 8), c = (e % (kIn / 8)) * 8;
    uint4 v = zero;
    if (r0 + r < a.n) v = *reinterpret_cast<const uint4*>(a.x + (size_t)(r0 + r) * kIn + c);
    *reinterpret_cast<uint4*>(X + r * LDX + c) = v;
  }
  __syncthreads();
  fused_layer<FR, KG, kIn, false>(a, 0, X, LDX, H, r0);
  __syncthreads();
#pragma unroll 1
  for (int l = 1; l < 3; ++l) {   // one copy of the layer's code in the instruction cache
    fused_layer<FR, KG, kHid, false>(a, l, H, LDH, H, r0);
    __syncthreads();
  }
  fused_layer<FR, KG, kHid, true>(a, 3, H, LDH, H, r0);
}

// ---- training support kernels ----------------------------------------------
// Network outputs enter sinh(); beyond +-20 they are clipped (sinh(20) = 2.4e8).
constexpr float kOutClip = 20.0f;

// ---- the training step: rows, weight gradients, Adam ---------------------------
// Three launches make a step.  rows: forward, loss and the gradients with
// respect to every pre-activation, 32 rows of the batch per workgroup, with
// the activations in LDS and registers.  weights: all weight and bias
// gradients as split partial sums.  Adam: the sums over the splits and the
// update.  At 8192 rows they take 22 + 16 + 7.5 us.  A launch for each
// product, sum and copy (18 of them, none of which fills the chip) took
// 200 us.
//
// What rows leaves for weights is laid out in blocks of 32 rows,
// [block][unit][32 rows]: a workgroup's block is written in one piece, and a
// product over rows reads its MFMA operands (16 units x 32 rows) as contiguous
// KiB, with no transposition through LDS.  Rows past the end of the batch are
// zeros.
constexpr int RB = 32;                   // rows per block: one k chunk of the weight gradients
constexpr int kRowThreads = 512;         // wave w: hidden units [32w, 32w+32) of all 32 rows
constexpr int LDF = kOutLd + 1;          // fp32 row stride of the output tile

struct RowsArgs {
  const uint16_t* x;                     // the rows, or the data set's rows when perm is set
  const float* target;
  const int* perm;
  const long long* cursor;
  long long ds_n;
  int n;
  const uint16_t* wf[kLayers];           // frag_offset(n, k, fan_in)
  const uint16_t* wb[kLayers];           // frag_offset(k, n, padded fan_out)
  const float* bias[kLayers];
  uint16_t* xt;                          // [block][unit][32]: inputs,
  uint16_t* ht[3];                       //   activations,
  uint16_t* dzt[3];                      //   gradients wrt pre-activations,
  uint16_t* dot;                         //   gradients wrt outputs
  float* row_loss;
  float w[32], sigma[32];
  unsigned head_mask;
  float head_w, inv_wsum, inv_B;
};

// NK k chunks of a wave's 32 x 32 tile: rows of A (LDS) times its weights.
template <int NK>
__device__ __forceinline__ void rows_product(const uint16_t* __restrict__ A, int lda, const uint4 (&w)[NK][2],
                                             f32x4 (&acc)[2][2]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint4 v = *reinterpret_cast<const uint4*>(A + (i * 16 + (lane & 15)) * lda + kk * TK + (lane >> 4) * 8);
      const bf16x8 av = __builtin_bit_cast(bf16x8, v);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, w[kk][j]), acc[i][j],
                                                            0, 0, 0);
    }
}

// A wave's weight fragments of two adjacent 16-column tiles.
template <int NK>
__device__ __forceinline__ void rows_weights(const uint16_t* __restrict__ w, int tile, uint4 (&q)[NK][2]) {
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      q[kk][j] = *reinterpret_cast<const uint4*>(w + (size_t)((tile + j) * NK + kk) * 512 + (threadIdx.x & 63) * 8);
}

__device__ __forceinline__ uint2 zero_past(uint2 v, int valid) {  // keep the first `valid` of four bf16
  if (valid < 4) {
    v.y = valid < 3 ? 0u : v.y & 0xffffu;
    v.x = valid < 1 ? 0u : (valid < 2 ? v.x & 0xffffu : v.x);
  }
  return v;
}

// Four consecutive rows of one unit to the LDS tile (when a later layer reads
// it) and to the block for the weight gradients.
__device__ __forceinline__ void rows_store(uint2 v, uint16_t* __restrict__ tile, uint16_t* __restrict__ block, int row,
                                           int unit, int valid_rows) {
  if (tile) {
    tile[(row + 0) * LDH + unit] = (uint16_t)v.x;
    tile[(row + 1) * LDH + unit] = (uint16_t)(v.x >> 16);
    tile[(row + 2) * LDH + unit] = (uint16_t)v.y;
    tile[(row + 3) * LDH + unit] = (uint16_t)(v.y >> 16);
  }
  *reinterpret_cast<uint2*>(block + (size_t)unit * RB + row) = zero_past(v, valid_rows - row);
}

// Bias, SiLU and rounding of a hidden layer; z (bf16) stays for the backward.
template <bool FAR>
__device__ __forceinline__ void rows_activate(const f32x4 (&acc)[2][2], uint16_t* __restrict__ tile,
                                              uint16_t* __restrict__ block, int valid_rows) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f32x4 h;
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = FAR ? silu(acc[i][j][r]) : silu_near(acc[i][j][r]);
      rows_store(f2bf4(h), tile, block, i * 16 + (lane >> 4) * 4, wave * 32 + j * 16 + (lane & 15), valid_rows);
    }
}

__device__ __forceinline__ void rows_hidden(f32x4 (&acc)[2][2], const float (&bias)[2], uint2 (&z)[2][2],
                                            uint16_t* __restrict__ tile, uint16_t* __restrict__ block,
                                            int valid_rows) {
  float far = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      acc[i][j] += bias[j];
      z[i][j] = f2bf4(acc[i][j]);
      far = fmaxf(far, abs_max4(acc[i][j]));
    }
  if (__builtin_expect(__any(far > kSiluNear), 0))
    rows_activate<true>(acc, tile, block, valid_rows);
  else
    rows_activate<false>(acc, tile, block, valid_rows);
}

// Gradient wrt a hidden layer's pre-activation.
template <bool FAR>
__device__ __forceinline__ void rows_chain(const f32x4 (&acc)[2][2], const f32x4 (&z)[2][2],
                                           uint16_t* __restrict__ tile, uint16_t* __restrict__ block,
                                           int valid_rows) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f32x4 d;
#pragma unroll
      for (int r = 0; r < 4; ++r) d[r] = acc[i][j][r] * dsilu<FAR>(z[i][j][r]);
      rows_store(f2bf4(d), tile, block, i * 16 + (lane >> 4) * 4, wave * 32 + j * 16 + (lane & 15), valid_rows);
    }
}

__device__ __forceinline__ void rows_gradient(const f32x4 (&acc)[2][2], const uint2 (&zq)[2][2],
                                              uint16_t* __restrict__ tile, uint16_t* __restrict__ block,
                                              int valid_rows) {
  f32x4 z[2][2];
  float far = 0.0f;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint2 q = zq[i][j];
      z[i][j] = f32x4{bf2f((uint16_t)q.x), bf2f((uint16_t)(q.x >> 16)), bf2f((uint16_t)q.y),
                      bf2f((uint16_t)(q.y >> 16))};
      far = fmaxf(far, abs_max4(z[i][j]));
    }
  if (__builtin_expect(__any(far > kSiluNear), 0))
    rows_chain<true>(acc, z, tile, block, valid_rows);
  else
    rows_chain<false>(acc, z, tile, block, valid_rows);
}

// [unit][32 rows] of an LDS tile of 32 rows x 32 columns (threads 0..127).
__device__ __forceinline__ void rows_transpose(const uint16_t* __restrict__ tile, uint16_t* __restrict__ block,
                                               int valid_rows) {
  const int u = threadIdx.x >> 2, r = (threadIdx.x & 3) * 8;
  if (u >= 32) return;
  uint32_t q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = r + 2 * e < valid_rows ? tile[(r + 2 * e) * LDX + u] : 0u;
    const uint32_t hi = r + 2 * e + 1 < valid_rows ? tile[(r + 2 * e + 1) * LDX + u] : 0u;
    q[e] = lo | hi << 16;
  }
  *reinterpret_cast<uint4*>(block + u * RB + r) = make_uint4(q[0], q[1], q[2], q[3]);
}

// Bound by the serial chain of layers: eight waves share a layer's 256 units,
// and each asks for the next layer's weights before it starts on this one's
// products, so that memory is waited for once.  A workgroup's 570 KB of
// weights come from the L2; 32 rows make 256 workgroups of a batch of 8192.
__global__ __launch_bounds__(kRowThreads, 2) void train_rows_kernel(RowsArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t X[RB * LDX];
  __shared__ __attribute__((aligned(16))) uint16_t H[2][RB * LDH];
  __shared__ float O[RB * LDF], R[RB * LDF];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t blk = blockIdx.x;
  const int r0 = blockIdx.x * RB;
  const int valid = min(RB, a.n - r0);
  uint16_t* const hb[3] = {a.ht[0] + blk * kHid * RB, a.ht[1] + blk * kHid * RB, a.ht[2] + blk * kHid * RB};
  uint16_t* const db[3] = {a.dzt[0] + blk * kHid * RB, a.dzt[1] + blk * kHid * RB, a.dzt[2] + blk * kHid * RB};

  // this thread's row of the batch: sixteen threads to a row
  const int row = tid >> 4, c = tid & 15;
  float2 t = make_float2(0.0f, 0.0f);
  uint4 xv = make_uint4(0u, 0u, 0u, 0u);
  if (row < valid) {
    long long src = r0 + row;
    if (a.perm) {
      src += *a.cursor;
      if (src >= a.ds_n) src %= a.ds_n;
      src = a.perm[src];
    }
    if (c < 4) xv = *reinterpret_cast<const uint4*>(a.x + src * kIn + c * 8);
    t.x = a.target[src * kOutLd + 2 * c];
    t.y = a.target[src * kOutLd + 2 * c + 1];
  }
  // loads return in order: what is small and needed soon goes first
  float b[3][2];
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int j = 0; j < 2; ++j) b[l][j] = a.bias[l][wave * 32 + j * 16 + (lane & 15)];
  const int out_col = (wave & 1) * 16 + (lane & 15);           // of waves 0..3
  const float b_out = a.bias[3][min(out_col, kOut - 1)];
  const float2 vw = make_float2(a.w[2 * c], a.w[2 * c + 1]);
  const float2 vs = make_float2(a.sigma[2 * c], a.sigma[2 * c + 1]);
  uint4 w1[1][2], w2[8][2], w3[8][2], w4[8];
  rows_weights(a.wf[0], wave * 2, w1);
  rows_weights(a.wf[1], wave * 2, w2);
  if (c < 4) *reinterpret_cast<uint4*>(X + row * LDX + c * 8) = xv;
  __syncthreads();
  rows_transpose(X, a.xt + blk * kIn * RB, valid);
  f32x4 acc[2][2];
  uint2 z1[2][2], z2[2][2], z3[2][2];
  rows_product(X, LDX, w1, acc);
  rows_hidden(acc, b[0], z1, H[0], hb[0], valid);
  __syncthreads();
  rows_weights(a.wf[2], wave * 2, w3);
  rows_product(H[0], LDH, w2, acc);
  rows_hidden(acc, b[1], z2, H[1], hb[1], valid);
  __syncthreads();
  if (wave < 4) {  // the output layer: one 16 x 16 tile for each of four waves
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
      w4[kk] = *reinterpret_cast<const uint4*>(a.wf[3] + (size_t)((wave & 1) * 8 + kk) * 512 + lane * 8);
  }
  rows_weights(a.wb[3], wave * 2, w1);
  rows_product(H[1], LDH, w3, acc);
  rows_hidden(acc, b[2], z3, H[0], hb[2], valid);
  __syncthreads();
  rows_weights(a.wb[2], wave * 2, w2);
  if (wave < 4) {
    const int i = wave >> 1;
    f32x4 o = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const uint4 v = *reinterpret_cast<const uint4*>(H[0] + (i * 16 + (lane & 15)) * LDH + kk * TK + (lane >> 4) * 8);
      o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, v), __builtin_bit_cast(bf16x8, w4[kk]), o,
                                                  0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) O[(i * 16 + (lane >> 4) * 4 + r) * LDF + out_col] = o[r] + b_out;
  }
  __syncthreads();
  // The loss and its gradient, two variables per thread.  The error head's
  // target is the row's largest error; the squares are added in the order of
  // the variables by one thread per row.
  {
    const int v = 2 * c;
    const float2 o = make_float2(O[row * LDF + v], O[row * LDF + v + 1]);
    const float2 res = make_float2(o.x - t.x, o.y - t.y);
    R[row * LDF + v] = res.x;
    R[row * LDF + v + 1] = res.y;
    const float t31 = __shfl(t.y, (lane & 48) | 15);
    uint16_t* d = X + row * LDX;
    float emax = 0.0f;
    // targets are asinh((r - m)/sigma) of the residual r: the error of the
    // residual itself is sigma |sinh(o) - sinh(t)|
    if (c < 15) {
      if ((a.head_mask >> v) & 1u)
        emax = fmaxf(emax, vs.x * fabsf(sinhf(fminf(fmaxf(o.x, -kOutClip), kOutClip)) - sinhf(t.x)));
      if ((a.head_mask >> (v + 1)) & 1u)
        emax = fmaxf(emax, vs.y * fabsf(sinhf(fminf(fmaxf(o.y, -kOutClip), kOutClip)) - sinhf(t.y)));
      d[v] = f2bf(2.0f * vw.x * res.x * a.inv_wsum * a.inv_B);
      d[v + 1] = f2bf(2.0f * vw.y * res.y * a.inv_wsum * a.inv_B);
    }
#pragma unroll
    for (int m = 8; m > 0; m >>= 1) emax = fmaxf(emax, __shfl_xor(emax, m));
    // a sample whose target was clipped carries a flag in column 31: its true
    // error is at least 1 (asinh units), so the head learns to reject it
    if (t31 != 0.0f) emax = fmaxf(emax, 1.0f);
    if (c == 15) {
      const float rh = o.x - logf(emax + 1.0e-7f);
      R[row * LDF + GAL_MLP_HEAD] = rh;
      d[GAL_MLP_HEAD] = f2bf(2.0f * a.head_w * rh * a.inv_B);
      d[31] = 0;
    }
  }
  __syncthreads();
  rows_transpose(X, a.dot + blk * kOutLd * RB, valid);
  if (tid >= kRowThreads - RB) {  // the last wave's lanes: one per row
    const int rr = tid - (kRowThreads - RB);
    float mse = 0.0f;
#pragma unroll
    for (int v = 0; v < 30; ++v) {
      const float res = R[rr * LDF + v];
      mse += a.w[v] * res * res;
    }
    const float rh = R[rr * LDF + GAL_MLP_HEAD];
    if (rr < valid) a.row_loss[r0 + rr] = mse * a.inv_wsum + a.head_w * rh * rh;
  }
  rows_product(X, LDX, w1, acc);
  rows_gradient(acc, z3, H[1], db[2], valid);
  __syncthreads();
  rows_weights(a.wb[1], wave * 2, w3);
  rows_product(H[1], LDH, w2, acc);
  rows_gradient(acc, z2, H[0], db[1], valid);
  __syncthreads();
  rows_product(H[0], LDH, w3, acc);
  rows_gradient(acc, z1, nullptr, db[0], valid);
}

// Weight gradients act^T . grad and bias gradients (column sums of grad) of
// all layers, over one split of the rows each: partial[split][k][n].  A wave
// owns a 32 x 32 tile, and a workgroup's four tiles share operands through
// the L1.  A block of 32 rows is one k chunk, whose fragments are contiguous.
// Consecutive workgroups take the same part of consecutive splits: with a
// multiple of eight splits an XCD's L2 holds the splits it works on.
constexpr int kWeightParts = 36;                       // workgroups per split for the products: 2 + 16 + 16 + 2
constexpr int kBiasParts = 4;                         // and for the column sums, a layer each

struct WeightArgs {
  const uint16_t* act[kLayers];
  const uint16_t* grad[kLayers];
  float* pw[kLayers];
  float* pb[kLayers];
  int n, splits, rows_per_split;         // rows_per_split: a multiple of RB
  // the step's loss, counters and learning rate (one further workgroup)
  const float* row_loss;
  float* loss_partial;
  float inv_B;
  float* loss;                           // null: a training step's loss_hist
  float* loss_hist;
  int hist_cap;
  long long* step;
  long long* cursor;
  int* local;
  int advance;
  float lr0, lr_min, beta1, beta2;
  int64_t total_steps;
  float* rates;                          // lr and the two bias corrections of the step
};

// Sum of the rows' losses, 256 rows to a partial sum, and a training step's
// counters.
__device__ void finish_step(const WeightArgs& a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nb = (a.n + 255) / 256;
  constexpr int G = 4;   // partial sums under way in a wave
  for (int b0 = wave * G; b0 < nb; b0 += 4 * G) {
    float v[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = (b0 + g) * 256 + q * 64 + lane;
        v[g][q] = a.row_loss[min(r, a.n - 1)];
        if (r >= a.n) v[g][q] = 0.0f;
      }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float s = (v[g][0] + v[g][2]) + (v[g][1] + v[g][3]);
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
      if (lane == 0 && b0 + g < nb) a.loss_partial[b0 + g] = s;
    }
  }
  __threadfence_block();
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.0f;
#pragma unroll 8
    for (int b = 0; b < nb; ++b) s += a.loss_partial[b];
    if (a.loss) *a.loss = s * a.inv_B;
    if (a.advance) {
      const int ls = *a.local;
      if (ls < a.hist_cap) a.loss_hist[ls] = s * a.inv_B;
      *a.local = ls + 1;
      *a.cursor += a.n;
    }
  }
  if (a.advance && threadIdx.x == 64) {
    const long long step = *a.step + 1;
    *a.step = step;
    const double t = (double)step;
    const double frac = fmin(t, (double)a.total_steps) / (double)a.total_steps;
    a.rates[0] = (float)(a.lr_min + 0.5 * (a.lr0 - a.lr_min) * (1.0 + cos(kPi * frac)));
    a.rates[1] = (float)(1.0 - pow((double)a.beta1, t));
    a.rates[2] = (float)(1.0 - pow((double)a.beta2, t));
  }
}

__global__ __launch_bounds__(256) void train_weights_kernel(WeightArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x == 0) {  // first: its chain of loads and sums is the longest
    finish_step(a);
    return;
  }
  const int part = (blockIdx.x - 1) / a.splits, split = (blockIdx.x - 1) % a.splits;
  const int nblk = (a.n + RB - 1) / RB, per = a.rows_per_split / RB;
  const int b0 = split * per, b1 = min(nblk, b0 + per);
  if (part >= kWeightParts) {
    // a unit per lane; the sums of the rows q, q + 4, ... are kept apart
    int u = (part - kWeightParts) * 256 + threadIdx.x;
    const int l = min(u / kHid, 3);
    u -= l * kHid;
    const int units = l == 3 ? kOutLd : kHid;
    if (u >= units) return;
    const uint16_t* g = a.grad[0];
    float* pb = a.pb[0];
    if (l == 1) { g = a.grad[1]; pb = a.pb[1]; }
    if (l == 2) { g = a.grad[2]; pb = a.pb[2]; }
    if (l == 3) { g = a.grad[3]; pb = a.pb[3]; }
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int b = b0; b < b1; ++b) {
      const uint4* e = reinterpret_cast<const uint4*>(g + ((size_t)b * units + u) * RB);
#pragma unroll
      for (int i = 0; i < RB / 8; ++i) {
        const uint4 v = e[i];
        s[0] += bf2f((uint16_t)v.x);
        s[1] += __uint_as_float(v.x & 0xffff0000u);
        s[2] += bf2f((uint16_t)v.y);
        s[3] += __uint_as_float(v.y & 0xffff0000u);
        s[0] += bf2f((uint16_t)v.z);
        s[1] += __uint_as_float(v.z & 0xffff0000u);
        s[2] += bf2f((uint16_t)v.w);
        s[3] += __uint_as_float(v.w & 0xffff0000u);
      }
    }
    pb[(size_t)split * units + u] = (s[0] + s[1]) + (s[2] + s[3]);
    return;
  }
  // the wave's tile: rows [mt, mt+32) x columns [nt, nt+32) of layer l
  const uint16_t *A, *G;
  float* pw;
  int mt, nt, M, N;
  if (part < 32) {
    const int p = part & 15;
    A = part < 16 ? a.act[1] : a.act[2];
    G = part < 16 ? a.grad[1] : a.grad[2];
    pw = part < 16 ? a.pw[1] : a.pw[2];
    M = kHid; N = kHid;
    mt = (p >> 2) * 64 + (wave >> 1) * 32;
    nt = (p & 3) * 64 + (wave & 1) * 32;
  } else if (part < 34) {
    A = a.act[0]; G = a.grad[0]; pw = a.pw[0];
    M = kIn; N = kHid;
    mt = 0;
    nt = (part & 1) * 128 + wave * 32;
  } else {
    A = a.act[3]; G = a.grad[3]; pw = a.pw[3];
    M = kHid; N = kOutLd;
    mt = (part & 1) * 128 + wave * 32;
    nt = 0;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int at = (lane & 15) * RB + (lane >> 4) * 8;
  const uint16_t* pa = A + (size_t)mt * RB + at;
  const uint16_t* pg = G + (size_t)nt * RB + at;
  // four k chunks' operands in flight at a time
  constexpr int KU = 4;
  int b = b0;
  for (; b + KU <= b1; b += KU) {
    uint4 av[KU][2], gv[KU][2];
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        av[u][i] = *reinterpret_cast<const uint4*>(pa + ((size_t)(b + u) * M + i * 16) * RB);
        gv[u][i] = *reinterpret_cast<const uint4*>(pg + ((size_t)(b + u) * N + i * 16) * RB);
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[u][i]),
                                                              __builtin_bit_cast(bf16x8, gv[u][j]), acc[i][j], 0, 0, 0);
  }
  for (; b < b1; ++b) {
    uint4 av[2], gv[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      av[i] = *reinterpret_cast<const uint4*>(pa + ((size_t)b * M + i * 16) * RB);
      gv[i] = *reinterpret_cast<const uint4*>(pg + ((size_t)b * N + i * 16) * RB);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[i]),
                                                            __builtin_bit_cast(bf16x8, gv[j]), acc[i][j], 0, 0, 0);
  }
  float* out = pw + ((size_t)split * M + mt + (lane >> 4) * 4) * N + nt + (lane & 15);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) out[(size_t)(i * 16 + r) * N + j * 16] = acc[i][j][r];
}

struct AdamArgs {
  float* param;
  float* m;
  float* v;
  uint16_t* wbf[kLayers];
  uint16_t* wf[kLayers];
  uint16_t* wb[kLayers];
  float* grad_out;
  const float* pw;
  const float* pb;
  int64_t w_off[kLayers], b_off[kLayers], pw_off[kLayers], pb_off[kLayers];
  int splits;
  float beta1, beta2, eps;
  const float* rates;   // WeightArgs::rates
  int apply;
};

// Sum the split partials into the gradient (fixed order) and take one Adam
// step; keeps the bf16 copies of each weight in step with its fp32 master.
__global__ __launch_bounds__(256) void adam_kernel(AdamArgs a) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kParams) return;
  int l = 0, k = 0, n = 0;
  bool is_b = false;
#pragma unroll
  for (int j = 0; j < kLayers; ++j) {
    if (p >= a.w_off[j] && p < a.b_off[j]) {
      const int64_t q = p - a.w_off[j];
      l = j; k = (int)(q / kFanOut[j]); n = (int)(q % kFanOut[j]);
    } else if (p >= a.b_off[j] && p < a.b_off[j] + kFanOut[j]) {
      l = j; n = (int)(p - a.b_off[j]); is_b = true;
    }
  }
  float g = 0.0f;
  if (is_b) {
#pragma unroll 16
    for (int s = 0; s < a.splits; ++s) g += a.pb[a.pb_off[l] + (int64_t)s * kLdW[l] + n];
  } else {
#pragma unroll 16
    for (int s = 0; s < a.splits; ++s) g += a.pw[a.pw_off[l] + ((int64_t)s * kFanIn[l] + k) * kLdW[l] + n];
  }
  if (a.grad_out) a.grad_out[p] = g;
  if (!a.apply) return;
  const float lr = a.rates[0], bc1 = a.rates[1], bc2 = a.rates[2];
  // which product is rounded is written out: a last bit here grows over the steps
  const float m = fmaf(g, 1.0f - a.beta1, a.beta1 * a.m[p]);
  const float v = fmaf(g, g * (1.0f - a.beta2), a.beta2 * a.v[p]);
  a.m[p] = m;
  a.v[p] = v;
  const float w = a.param[p] - lr * (m / bc1) / (sqrtf(v / bc2) + a.eps);
  a.param[p] = w;
  if (!is_b) {
    const uint16_t b = f2bf(w);
    a.wbf[l][(size_t)k * kLdW[l] + n] = b;
    a.wf[l][frag_offset(n, k, kFanIn[l])] = b;
    a.wb[l][frag_offset(k, n, kLdW[l])] = b;
  }
}

__global__ void weights_to_bf16_kernel(const float* __restrict__ param, int64_t w_off, int fan_in, int fan_out,
                                       int ldw, uint16_t* __restrict__ wbf, uint16_t* __restrict__ wf,
                                       uint16_t* __restrict__ wb) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (int64_t)fan_in * fan_out) return;
  const int k = (int)(q / fan_out), n = (int)(q % fan_out);
  const uint16_t b = f2bf(param[w_off + q]);
  wbf[(size_t)k * ldw + n] = b;
  wf[frag_offset(n, k, fan_in)] = b;
  wb[frag_offset(k, n, ldw)] = b;
}

// A kernel and not a memset, which a caller's graph replays wrongly.
__global__ void reset_count_kernel(int* count) {
  if (threadIdx.x == 0) *count = 0;
}

__global__ void reset_train_kernel(long long* cursor, int* local) {
  if (threadIdx.x == 0) {
    *cursor = 0;
    *local = 0;
  }
}

// ---- node encoding ------------------------------------------------------------
enum Role : int { R_MASS, R_METAL, R_ANGMOM, R_ENERGY, R_BH, R_UNIT, R_CONST, R_SPIN, R_FIRST_ORDER };

__device__ __forceinline__ int var_role(int v) {
  switch (v) {
    case GAL_V_HOT_MASS: case GAL_V_HOT_OUTFLOWED_MASS: case GAL_V_HOT_UNACCRETED_MASS:
    case GAL_V_DISK_MASS_STELLAR: case GAL_V_DISK_MASS_STELLAR_FORMED: case GAL_V_DISK_MASS_GAS:
    case GAL_V_SPHEROID_MASS_STELLAR: case GAL_V_SPHEROID_MASS_STELLAR_FORMED: case GAL_V_SPHEROID_MASS_GAS:
      return R_MASS;
    case GAL_V_HOT_ABUNDANCES: case GAL_V_HOT_OUTFLOWED_ABUNDANCES: case GAL_V_HOT_UNACCRETED_ABUNDANCES:
    case GAL_V_DISK_ABUNDANCES_STELLAR: case GAL_V_DISK_ABUNDANCES_GAS: case GAL_V_SPHEROID_ABUNDANCES_STELLAR:
    case GAL_V_SPHEROID_ABUNDANCES_GAS:
      return R_METAL;
    case GAL_V_HOT_ANGULAR_MOMENTUM: case GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM: case GAL_V_DISK_ANGULAR_MOMENTUM:
    case GAL_V_SPHEROID_ANGULAR_MOMENTUM:
      return R_ANGMOM;
    case GAL_V_HOT_ENERGY_RADIATED: return R_ENERGY;
    case GAL_V_BH_MASS: return R_BH;
    case GAL_V_BH_SPIN: return R_UNIT;
    case GAL_V_SPIN_ANGULAR_MOMENTUM: return R_SPIN;
    // not fed to the network: advanced by the first-order step of the rate at
    // the interval's start (outer radius, bound mass and stripped gas)
    case GAL_V_HOT_OUTER_RADIUS: case GAL_V_SATELLITE_BOUND_MASS: case GAL_V_HOT_STRIPPED_MASS:
    case GAL_V_HOT_STRIPPED_ABUNDANCES:
      return R_FIRST_ORDER;
    default: return R_CONST;
  }
}

// Variables fed to the network, in state order.
__constant__ int kInputVars[GAL_SURR_N_INPUT_VARS] = {
    GAL_V_HOT_MASS, GAL_V_HOT_ABUNDANCES, GAL_V_HOT_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_MASS,
    GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_ABUNDANCES, GAL_V_HOT_UNACCRETED_MASS,
    GAL_V_HOT_UNACCRETED_ABUNDANCES, GAL_V_DISK_MASS_STELLAR, GAL_V_DISK_MASS_STELLAR_FORMED,
    GAL_V_DISK_ABUNDANCES_STELLAR, GAL_V_DISK_MASS_GAS, GAL_V_DISK_ABUNDANCES_GAS, GAL_V_DISK_ANGULAR_MOMENTUM,
    GAL_V_SPHEROID_MASS_STELLAR, GAL_V_SPHEROID_MASS_STELLAR_FORMED, GAL_V_SPHEROID_ABUNDANCES_STELLAR,
    GAL_V_SPHEROID_MASS_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS, GAL_V_SPHEROID_ANGULAR_MOMENTUM, GAL_V_BH_MASS,
    GAL_V_BH_SPIN};

struct NodeFrame {
  Halo H;
  double unit;      // f_b M_halo(t0)
  double s_mass, s_metal, s_ang, s_energy;
  double failed;
};

__device__ __forceinline__ NodeFrame node_frame(const double* __restrict__ P, const DerivedConstants& D,
                                                const NodePar& np, double t0, double spin_j) {
  NodeFrame f;
  f.H = halo(P, D, np, t0, spin_j);
  f.unit = D.f_baryon * f.H.mass;
  f.s_mass = 1.0e-4 * f.unit;
  f.s_metal = 1.0e-6 * f.unit;
  f.s_ang = 1.0e-4 * f.unit * f.H.r_vir * f.H.v_vir;
  f.s_energy = D.unit_energy * f.H.mass * f.H.v_vir * f.H.v_vir * 1.0e-3;
  f.failed = (f.H.a3 > D.a3_reion && f.H.v_vir < P[GAL_P_VELOCITY_SUPPRESSION_REIONIZATION]) ? 1.0 : 0.0;
  return f;
}

__device__ __forceinline__ double var_scale(const NodeFrame& f, int role) {
  switch (role) {
    case R_MASS: return f.s_mass;
    case R_METAL: return f.s_metal;
    case R_ANGMOM: return f.s_ang;
    case R_ENERGY: return f.s_energy;
    default: return 1.0;
  }
}

// The first-order increment of each trained variable in asinh space from one
// RHS evaluation at t0: for a growing quantity the Euler step taken in y,
// asinh((y + f dt)/s) - asinh(y/s) (exact for a constant rate); for a
// decaying one the Euler step taken in u, f dt / sqrt(s^2 + y^2) (exact for
// exponential decay, and never overshoots through zero).  The network
// learns only what this misses.
__device__ __forceinline__ void euler_baseline(const double* __restrict__ P, const DerivedConstants& D,
                                               const double* __restrict__ tab, const CoolingDesc& cd, int mode,
                                               const NodePar& np, const NodeFrame& f, double t0, double dt,
                                               const double (&y0)[kNV], double (&du)[kNV]) {
  double rate[kNV];
  rhs(P, D, tab, cd, mode, np, t0, y0, rate);
#pragma unroll
  for (int v = 0; v < kNV; ++v) {
    const int role = var_role(v);
    double d = 0.0;
    if (role == R_ENERGY) {
      d = asinh(rate[v] * dt / f.s_energy);
    } else if (role != R_CONST && role != R_SPIN && role != R_FIRST_ORDER) {
      const double s = var_scale(f, role);
      if (rate[v] >= 0.0)
        d = asinh((y0[v] + rate[v] * dt) / s) - asinh(y0[v] / s);          // linear growth
      else if (y0[v] > 0.0)
        d = asinh(y0[v] * exp(rate[v] * dt / y0[v]) / s) - asinh(y0[v] / s);  // decay on y/|f|
      else
        d = rate[v] * dt * rsqrt(s * s + y0[v] * y0[v]);
    }
    du[v] = d;
  }
}

__global__ __launch_bounds__(256) void encode_kernel(int n, int ld, const double* __restrict__ y0,
                                                     const double* __restrict__ y1, const double* __restrict__ npa,
                                                     const double* __restrict__ t0a, const double* __restrict__ t1a,
                                                     const double* __restrict__ P, DerivedConstants D,
                                                     const double* __restrict__ tab, CoolingDesc cd, int mode,
                                                     const float* __restrict__ norm, uint16_t* __restrict__ x,
                                                     float* __restrict__ x_raw, float* __restrict__ target) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const NodePar np = load_node_par(npa, ld, i);
  const double t0 = t0a[i];
  const double dt = t1a[i] - t0;
  const NodeFrame f = node_frame(P, D, np, t0, y0[GAL_V_SPIN_ANGULAR_MOMENTUM * (size_t)ld + i]);
  float in[kIn];
#pragma unroll
  for (int j = 0; j < GAL_SURR_N_INPUT_VARS; ++j) {
    const int v = kInputVars[j];
    in[j] = (float)asinh(y0[v * (size_t)ld + i] / var_scale(f, var_role(v)));
  }
  const double dtp = fmax(dt, 1.0e-12);
  in[22] = (float)log(dtp);
  in[23] = (float)(log10(f.H.mass) - 11.0);
  in[24] = (float)(0.1 * t0);
  in[25] = (float)((np.satellite ? 0.0 : np.m_rate) * dt / f.H.mass);
  in[26] = (float)log(fmax(f.H.lambda, 1.0e-4));
  in[27] = (float)(y0[GAL_V_HOT_OUTER_RADIUS * (size_t)ld + i] * f.H.inv_r_vir);
  in[28] = (float)(f.H.v_vir / 200.0);
  in[29] = (float)f.failed;
  in[30] = (float)log(dtp * f.H.inv_t_dyn);
  in[31] = 0.0f;
  if (x_raw) {
#pragma unroll
    for (int j = 0; j < kIn; ++j) x_raw[(size_t)i * kIn + j] = in[j];
  }
  if (x) {
#pragma unroll
    for (int j = 0; j < kIn; ++j) {
      const float z = norm ? (in[j] - norm[j]) / norm[kIn + j] : in[j];
      x[(size_t)i * kIn + j] = f2bf(z);
    }
  }
  if (target && y1) {
    double ys[kNV], du[kNV];
#pragma unroll
    for (int v = 0; v < kNV; ++v) ys[v] = y0[v * (size_t)ld + i];
    euler_baseline(P, D, tab, cd, mode, np, f, t0, dt, ys, du);
    float* tg = target + (size_t)i * kOutLd;
    for (int v = 0; v < GAL_NVAR; ++v) {
      const int role = var_role(v);
      const double a = ys[v], b = y1[v * (size_t)ld + i];
      double d = 0.0;
      if (role == R_ENERGY) {
        d = asinh((b - a) / f.s_energy) - du[v];
      } else if (role != R_CONST && role != R_SPIN && role != R_FIRST_ORDER) {
        const double s = var_scale(f, role);
        d = asinh(b / s) - asinh(a / s) - du[v];
      }
      float z = (float)d;
      if (norm) z = (float)asinh((d - (double)norm[2 * kIn + v]) / (double)norm[3 * kIn + v]);
      tg[v] = z;
    }
    tg[GAL_MLP_HEAD] = 0.0f;
    tg[31] = 0.0f;
  }
}

struct GateArgs {
  int n, ld;
  double* y;
  const double* np;
  const double* t0;
  const double* t1;
  const float* out;
  const float* norm;
  double* scale;
  int* status;
  int* accepted;
  int* reject_list;
  int* reject_count;
  int index_offset;   // global index of node 0 of this call (chunking)
  const double* P;
  const double* tab;
  DerivedConstants D;
  CoolingDesc cd;
  int mode;
  gal_surrogate_gate gate;
};

// Decode the network's increments for one node, check them and either
// commit the new state or queue the node for the integrator.
__global__ __launch_bounds__(256) void apply_kernel(GateArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool reject = false;
  if (i < a.n) {
    const size_t ld = (size_t)a.ld;
    const NodePar np = load_node_par(a.np, a.ld, i);
    const double t0 = a.t0[i];
    const double dt = a.t1[i] - t0;
    double y0[kNV], y1[kNV];
#pragma unroll
    for (int v = 0; v < kNV; ++v) y0[v] = a.y[v * ld + i];
    if (dt > 0.0) {
      const NodeFrame f = node_frame(a.P, a.D, np, t0, y0[GAL_V_SPIN_ANGULAR_MOMENTUM]);
      const float* o = a.out + (size_t)i * kOutLd;
      const float* nm = a.norm;
      bool ok = (double)o[GAL_MLP_HEAD] <= a.gate.log_error_max;
      double rate[kNV];
      rhs(a.P, a.D, a.tab, a.cd, a.mode, np, t0, y0, rate);
#pragma unroll
      for (int v = 0; v < kNV; ++v) {
        const int role = var_role(v);
        if (role == R_CONST) {
          y1[v] = y0[v];
        } else if (role == R_FIRST_ORDER) {
          y1[v] = y0[v] + rate[v] * dt;
        } else if (role == R_SPIN) {
          y1[v] = y0[v] + (np.satellite ? 0.0 : np.spin_rate) * dt;
        } else {
          // u1 = asinh(y0/s) + du + c with du the first-order increment of
          // euler_baseline and c = m + sigma sinh(o) the network's residual.
          // Written as u1 = asinh(Y/s) + C for the first-order end point Y,
          // y1 = s sinh(u1) = Y cosh C + sqrt(s^2 + Y^2) sinh C: no asinh,
          // and sinh C, cosh C from one expm1 (accurate for small C).
          const double ov = fmin(fmax((double)o[v], -(double)kOutClip), (double)kOutClip);
          double C = (double)nm[2 * kIn + v] + (double)nm[3 * kIn + v] * sinh(ov);
          const double s = var_scale(f, role);
          const double step = rate[v] * dt;
          double Y;
          if (role == R_ENERGY) {
            Y = step;                                  // energy: y1 = y0 + s sinh(asinh(f dt/s) + c)
          } else if (rate[v] >= 0.0) {
            Y = y0[v] + step;                          // linear growth
          } else if (y0[v] > 0.0) {
            Y = y0[v] * exp(step / y0[v]);             // decay on y/|f|
          } else {
            Y = y0[v];                                 // Euler step in u
            C += step * rsqrt(s * s + y0[v] * y0[v]);
          }
          const double em = expm1(C);
          const double e = 1.0 + em;
          const double sinh_c = 0.5 * em * (1.0 + 1.0 / e);
          const double cosh_c = 1.0 + 0.5 * em * em / e;
          const double w = Y * cosh_c + sqrt(s * s + Y * Y) * sinh_c;
          y1[v] = role == R_ENERGY ? y0[v] + w : w;
        }
        // a small negative value of a non-negative quantity is set to zero,
        // as the reference's post-step fixes do after an integrator step
        if (var_non_negative(v) && y1[v] < 0.0 && role != R_ENERGY &&
            y1[v] >= -a.gate.negative_tolerance * var_scale(f, role))
          y1[v] = 0.0;
        ok = ok && isfinite(y1[v]);
        ok = ok && !(var_non_negative(v) && y1[v] < 0.0);
      }
      // Baryon budget: accretion f_b Mdot dt is the only source; black-hole
      // growth is the only sink (radiated and jet energy).
      const double accreted = np.satellite ? 0.0 : a.D.f_baryon * np.m_rate * dt;
      auto baryons = [](const double* s) {
        return s[GAL_V_HOT_MASS] + s[GAL_V_HOT_OUTFLOWED_MASS] + s[GAL_V_HOT_UNACCRETED_MASS] +
               s[GAL_V_HOT_STRIPPED_MASS] + s[GAL_V_DISK_MASS_GAS] + s[GAL_V_DISK_MASS_STELLAR] +
               s[GAL_V_SPHEROID_MASS_GAS] + s[GAL_V_SPHEROID_MASS_STELLAR] + s[GAL_V_BH_MASS];
      };
      auto metals = [](const double* s) {
        return s[GAL_V_HOT_ABUNDANCES] + s[GAL_V_HOT_OUTFLOWED_ABUNDANCES] + s[GAL_V_HOT_UNACCRETED_ABUNDANCES] +
               s[GAL_V_HOT_STRIPPED_ABUNDANCES] + s[GAL_V_DISK_ABUNDANCES_GAS] + s[GAL_V_DISK_ABUNDANCES_STELLAR] +
               s[GAL_V_SPHEROID_ABUNDANCES_GAS] + s[GAL_V_SPHEROID_ABUNDANCES_STELLAR];
      };
      const double mb0 = baryons(y0), mb1 = baryons(y1);
      const double dbh = fmax(y1[GAL_V_BH_MASS] - y0[GAL_V_BH_MASS], 0.0);
      const double rm = mb1 - mb0 - accreted;
      const double tol_m = a.gate.mass_tolerance * (mb0 + accreted);
      ok = ok && rm <= tol_m && rm >= -(tol_m + a.gate.bh_slack * dbh);
      // Metal budget: the yield of newly formed stars is the only source.
      const double formed = (y1[GAL_V_DISK_MASS_STELLAR_FORMED] - y0[GAL_V_DISK_MASS_STELLAR_FORMED]) +
                            (y1[GAL_V_SPHEROID_MASS_STELLAR_FORMED] - y0[GAL_V_SPHEROID_MASS_STELLAR_FORMED]);
      const double src = a.P[GAL_P_METAL_YIELD] * formed;
      const double z0 = metals(y0), z1 = metals(y1);
      const double rz = z1 - z0 - src;
      const double tol_z = a.gate.metal_tolerance * (z0 + fabs(src)) + 1.0e-3 * f.s_metal;
      ok = ok && rz <= tol_z && rz >= -(tol_z + 0.1 * a.gate.bh_slack * dbh);
      if (ok) {
        double sc[kNV];
        scales(a.P, a.D, np, t0, y0, sc);
#pragma unroll
        for (int v = 0; v < kNV; ++v) {
          a.y[v * ld + i] = y1[v];
          if (a.scale) a.scale[v * ld + i] = sc[v];
        }
      }
      reject = !ok;
    }
    if (!reject) a.status[i] = GAL_STATUS_SUCCESS;
    a.accepted[i] = reject ? 0 : 1;
  }
  // Wave-aggregated append of the rejected nodes.
  const unsigned long long mask = __ballot(reject);
  if (mask) {
    const int lane = __lane_id();
    const int leader = __ffsll((long long)mask) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(a.reject_count, __popcll(mask));
    base = __shfl(base, leader);
    if (reject) {
      const unsigned long long below = lane ? (mask & ((1ull << lane) - 1ull)) : 0ull;
      a.reject_list[base + __popcll(below)] = a.index_offset + i;
    }
  }
}

}  // namespace

// ============================================================================
// The network handle
// ============================================================================
struct gal_mlp {
  int device = 0;
  int batch = 0, splits = 0;
  int64_t w_off[kLayers] = {}, b_off[kLayers] = {}, pw_off[kLayers] = {}, pb_off[kLayers] = {};
  float* d_param = nullptr;
  float* d_m = nullptr;
  float* d_v = nullptr;
  uint16_t* d_wbf[kLayers] = {};
  uint16_t* d_wf[kLayers] = {};   // the same in fragment order, columns as operand rows (forward)
  uint16_t* d_wb[kLayers] = {};   // and rows as operand rows (backward)
  // blocks of 32 rows, [block][unit][32], of the batch under way
  uint16_t* d_xt = nullptr;
  uint16_t* d_ht[3] = {};
  uint16_t* d_dzt[3] = {};
  uint16_t* d_dot = nullptr;
  float* d_row_loss = nullptr;
  float* d_rates = nullptr;
  float* d_pw = nullptr;
  float* d_pb = nullptr;
  float* d_loss_partial = nullptr;
  long long* d_step = nullptr;
  long long* d_cursor = nullptr;
  int* d_local = nullptr;
  float* d_loss_hist = nullptr;
  int loss_hist_cap = 0;
  float lr0 = 1.0e-3f, lr_min = 1.0e-5f, beta1 = 0.9f, beta2 = 0.999f, eps = 1.0e-8f;
  int64_t total_steps = 1;
  float var_w[32] = {}, sigma[32] = {};
  unsigned head_mask = 0;
  float head_w = 0.1f, inv_wsum = 0.0f;
  long long ds_n = 0;
  const uint16_t* ds_x = nullptr;
  const float* ds_t = nullptr;
  const int* ds_perm = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  // the captured step, and kGraphSteps of them: the GPU idles for 8 us between
  // two graphs and not at all within one
  hipGraph_t graph[2] = {};
  hipGraphExec_t exec[2] = {};
  int inf_rows = 0;
  uint16_t* d_ix = nullptr;
  uint16_t* d_ih[2] = {};
  float* d_iout = nullptr;
  int rej_cap = 0;
  int* d_rej = nullptr;
  int* d_rej_count = nullptr;
};

namespace {

constexpr int kInferChunk = 1 << 17;

template <int EPI>
int gemm(const GemmArgs& g, hipStream_t s) {
  // Operand loads are 16-byte vectors along the contiguous dimension.
  if (g.K % 8 || g.lda % 8 || g.N % 8 || g.ldb % 8) return GAL_E_INVALID;
  const dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM);
  if (grid.y > 65535u) return GAL_E_INVALID;
  hipLaunchKernelGGL(gemm_kernel<EPI>, grid, dim3(256), 0, s, g);
  return hipGetLastError() == hipSuccess ? GAL_OK : GAL_E_HIP;
}

GemmArgs gemm_args(const uint16_t* A, const uint16_t* B, int M, int N, int K, int lda, int ldb, int ldc) {
  GemmArgs g{};
  g.A = A; g.B = B; g.M = M; g.N = N; g.K = K; g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.n_valid = N;
  return g;
}

#define GAL_TRY(x)                 \
  do {                             \
    const int rc_ = (x);           \
    if (rc_ != GAL_OK) return rc_; \
  } while (0)

// Forward through the four layers for n rows of x, one launch each.
int forward(gal_mlp* m, int n, const uint16_t* x, uint16_t* const h[3], float* out, hipStream_t s) {
  const uint16_t* in = x;
  for (int l = 0; l < 3; ++l) {
    GemmArgs g = gemm_args(in, m->d_wbf[l], n, kFanOut[l], kFanIn[l], kFanIn[l], kLdW[l], kFanOut[l]);
    g.bias = m->d_param + m->b_off[l];
    g.out_bf = h[l];
    GAL_TRY((gemm<EPI_SILU>(g, s)));
    in = h[l];
  }
  GemmArgs g = gemm_args(in, m->d_wbf[3], n, kOutLd, kHid, kHid, kLdW[3], kOutLd);
  g.n_valid = kOut;
  g.bias = m->d_param + m->b_off[3];
  g.out_f = out;
  return gemm<EPI_LINEAR>(g, s);
}

// Rows of a split of n rows: a multiple of the weight gradients' k chunk.
int split_rows(const gal_mlp* m, int n) { return ((n + m->splits - 1) / m->splits + RB - 1) / RB * RB; }

// Forward, loss and gradients of n rows: the weights' partial sums.  With perm
// the rows are the batch at the cursor of the permuted data set, and the step's
// counters, loss and learning rate move on.
int grad_pass(gal_mlp* m, int n, const uint16_t* x, const float* target, const int* perm, float* loss,
              hipStream_t s) {
  RowsArgs a{};
  a.x = x;
  a.target = target;
  a.perm = perm;
  a.cursor = m->d_cursor;
  a.ds_n = m->ds_n;
  a.n = n;
  WeightArgs g{};
  for (int l = 0; l < kLayers; ++l) {
    a.wf[l] = m->d_wf[l];
    a.wb[l] = m->d_wb[l];
    a.bias[l] = m->d_param + m->b_off[l];
    g.act[l] = l ? m->d_ht[l - 1] : m->d_xt;
    g.grad[l] = l < 3 ? m->d_dzt[l] : m->d_dot;
    g.pw[l] = m->d_pw + m->pw_off[l];
    g.pb[l] = m->d_pb + m->pb_off[l];
  }
  a.xt = m->d_xt;
  for (int l = 0; l < 3; ++l) { a.ht[l] = m->d_ht[l]; a.dzt[l] = m->d_dzt[l]; }
  a.dot = m->d_dot;
  a.row_loss = m->d_row_loss;
  for (int v = 0; v < 32; ++v) { a.w[v] = m->var_w[v]; a.sigma[v] = m->sigma[v]; }
  a.head_mask = m->head_mask;
  a.head_w = m->head_w;
  a.inv_wsum = m->inv_wsum;
  a.inv_B = 1.0f / (float)n;
  hipLaunchKernelGGL(train_rows_kernel, dim3((n + RB - 1) / RB), dim3(kRowThreads), 0, s, a);
  g.n = n;
  g.rows_per_split = split_rows(m, n);
  g.splits = (n + g.rows_per_split - 1) / g.rows_per_split;
  g.row_loss = m->d_row_loss;
  g.loss_partial = m->d_loss_partial;
  g.inv_B = a.inv_B;
  g.loss = loss;
  g.loss_hist = m->d_loss_hist;
  g.hist_cap = m->loss_hist_cap;
  g.step = m->d_step;
  g.cursor = m->d_cursor;
  g.local = m->d_local;
  g.advance = perm != nullptr;
  g.lr0 = m->lr0; g.lr_min = m->lr_min; g.beta1 = m->beta1; g.beta2 = m->beta2;
  g.total_steps = m->total_steps;
  g.rates = m->d_rates;
  hipLaunchKernelGGL(train_weights_kernel, dim3(g.splits * (kWeightParts + kBiasParts) + 1), dim3(256), 0, s, g);
  return hipGetLastError() == hipSuccess ? GAL_OK : GAL_E_HIP;
}

AdamArgs adam_args(gal_mlp* m, int n, float* grad_out, int apply) {
  AdamArgs a{};
  a.param = m->d_param; a.m = m->d_m; a.v = m->d_v;
  for (int l = 0; l < kLayers; ++l) {
    a.wbf[l] = m->d_wbf[l];
    a.wf[l] = m->d_wf[l];
    a.wb[l] = m->d_wb[l];
    a.w_off[l] = m->w_off[l]; a.b_off[l] = m->b_off[l]; a.pw_off[l] = m->pw_off[l]; a.pb_off[l] = m->pb_off[l];
  }
  const int rps = split_rows(m, n);
  a.splits = (n + rps - 1) / rps;
  a.grad_out = grad_out;
  a.pw = m->d_pw; a.pb = m->d_pb;
  a.beta1 = m->beta1; a.beta2 = m->beta2; a.eps = m->eps;
  a.rates = m->d_rates;
  a.apply = apply;
  return a;
}

int record_train_step(gal_mlp* m, hipStream_t s) {
  const int B = m->batch;
  GAL_TRY(grad_pass(m, B, m->ds_x, m->ds_t, m->ds_perm, nullptr, s));
  hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((kParams + 255) / 256)), dim3(256), 0, s,
                     adam_args(m, B, nullptr, 1));
  return hipGetLastError() == hipSuccess ? GAL_OK : GAL_E_HIP;
}

constexpr int kGraphSteps = 8;

void release_graph(gal_mlp* m) {
  for (int k = 0; k < 2; ++k) {
    if (m->exec[k]) hipGraphExecDestroy(m->exec[k]);
    if (m->graph[k]) hipGraphDestroy(m->graph[k]);
    m->exec[k] = nullptr;
    m->graph[k] = nullptr;
  }
}

// Capture `steps` training steps as graph k unless that is there.
int ensure_graph(gal_mlp* m, int k, int steps) {
  if (m->exec[k]) return GAL_OK;
  HIP_TRY(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
  int rc = GAL_OK;
  for (int i = 0; i < steps && rc == GAL_OK; ++i) rc = record_train_step(m, m->stream);
  hipGraph_t g = nullptr;
  const hipError_t e = hipStreamEndCapture(m->stream, &g);
  if (rc != GAL_OK || e != hipSuccess) {
    if (g) hipGraphDestroy(g);
    hipGetLastError();
    return rc != GAL_OK ? rc : GAL_E_HIP;
  }
  const hipError_t ie = hipGraphInstantiate(&m->exec[k], g, nullptr, nullptr, 0);
  if (ie != hipSuccess) {
    m->exec[k] = nullptr;
    hipGraphDestroy(g);
    HIP_TRY(ie);
  }
  m->graph[k] = g;
  return GAL_OK;
}

int ensure_inference(gal_mlp* m, int rows) {
  if (rows <= m->inf_rows) return GAL_OK;
  hipFree(m->d_ix); hipFree(m->d_ih[0]); hipFree(m->d_ih[1]); hipFree(m->d_iout);
  m->d_ix = nullptr; m->d_ih[0] = m->d_ih[1] = nullptr; m->d_iout = nullptr; m->inf_rows = 0;
  if (hipMalloc(&m->d_ix, sizeof(uint16_t) * kIn * (size_t)rows) != hipSuccess ||
      hipMalloc(&m->d_ih[0], sizeof(uint16_t) * kHid * (size_t)rows) != hipSuccess ||
      hipMalloc(&m->d_ih[1], sizeof(uint16_t) * kHid * (size_t)rows) != hipSuccess ||
      hipMalloc(&m->d_iout, sizeof(float) * kOutLd * (size_t)rows) != hipSuccess)
    return GAL_E_NOMEM;
  m->inf_rows = rows;
  return GAL_OK;
}

// Per-layer GEMM path.
int infer_layers(gal_mlp* m, int n, const uint16_t* x, float* out, hipStream_t s) {
  uint16_t* h[3] = {m->d_ih[0], m->d_ih[1], m->d_ih[0]};
  return forward(m, n, x, h, out, s);
}

// The fused one-kernel forward.
int infer(gal_mlp* m, int n, const uint16_t* x, float* out, hipStream_t s) {
  if (n <= 0) return GAL_OK;
  FusedArgs a{};
  a.x = x;
  for (int l = 0; l < kLayers; ++l) { a.wf[l] = m->d_wf[l]; a.bias[l] = m->d_param + m->b_off[l]; }
  a.out = out;
  a.n = n;
  if (n <= kFewRows)
    hipLaunchKernelGGL((mlp_forward_fused<32, 4>), dim3((n + 31) / 32), dim3(kFusedThreads), 0, s, a);
  else
    hipLaunchKernelGGL((mlp_forward_fused<kManyRows, 2>), dim3((n + kManyRows - 1) / kManyRows), dim3(kFusedThreads), 0, s,
                       a);
  return hipGetLastError() == hipSuccess ? GAL_OK : GAL_E_HIP;
}

}  // namespace

extern "C" {

int64_t gal_mlp_param_count(void) { return kParams; }

int gal_mlp_create(int batch, gal_mlp** out) {
  if (!out || batch < 1 || batch > 65535 * TM) return GAL_E_INVALID;
  *out = nullptr;
  gal_mlp* m = new gal_mlp();
  hipGetDevice(&m->device);
  m->batch = batch;
  m->splits = std::max(1, std::min(32, batch / 256));
  int64_t off = 0, pw = 0, pb = 0;
  for (int l = 0; l < kLayers; ++l) {
    m->w_off[l] = off;
    off += (int64_t)kFanIn[l] * kFanOut[l];
    m->b_off[l] = off;
    off += kFanOut[l];
    m->pw_off[l] = pw;
    pw += (int64_t)m->splits * kFanIn[l] * kLdW[l];
    m->pb_off[l] = pb;
    pb += (int64_t)m->splits * kLdW[l];
  }
  const size_t B = (size_t)(batch + RB - 1) / RB * RB;
  bool ok = hipMalloc(&m->d_param, sizeof(float) * kParams) == hipSuccess &&
            hipMalloc(&m->d_m, sizeof(float) * kParams) == hipSuccess &&
            hipMalloc(&m->d_v, sizeof(float) * kParams) == hipSuccess &&
            hipMalloc(&m->d_xt, sizeof(uint16_t) * kIn * B) == hipSuccess &&
            hipMalloc(&m->d_dot, sizeof(uint16_t) * kOutLd * B) == hipSuccess &&
            hipMalloc(&m->d_row_loss, sizeof(float) * B) == hipSuccess &&
            hipMalloc(&m->d_rates, sizeof(float) * 3) == hipSuccess &&
            hipMalloc(&m->d_pw, sizeof(float) * pw) == hipSuccess &&
            hipMalloc(&m->d_pb, sizeof(float) * pb) == hipSuccess &&
            hipMalloc(&m->d_loss_partial, sizeof(float) * ((B + 255) / 256)) == hipSuccess &&
            hipMalloc(&m->d_step, sizeof(long long)) == hipSuccess &&
            hipMalloc(&m->d_cursor, sizeof(long long)) == hipSuccess &&
            hipMalloc(&m->d_local, sizeof(int)) == hipSuccess;
  for (int l = 0; l < kLayers && ok; ++l)
    ok = hipMalloc(&m->d_wbf[l], sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess &&
         hipMalloc(&m->d_wf[l], sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess &&
         hipMalloc(&m->d_wb[l], sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess;
  for (int l = 0; l < 3 && ok; ++l)
    ok = hipMalloc(&m->d_ht[l], sizeof(uint16_t) * kHid * B) == hipSuccess &&
         hipMalloc(&m->d_dzt[l], sizeof(uint16_t) * kHid * B) == hipSuccess;
  // the training stream is created on the first training call: every stream
  // holds a hardware queue for the rest of the process, and inference-only
  // handles never need one
  ok = ok && hipEventCreateWithFlags(&m->ev_in, hipEventDisableTiming) == hipSuccess &&
       hipEventCreateWithFlags(&m->ev_out, hipEventDisableTiming) == hipSuccess;
  if (ok) {
    ok = hipMemset(m->d_param, 0, sizeof(float) * kParams) == hipSuccess &&
         hipMemset(m->d_m, 0, sizeof(float) * kParams) == hipSuccess &&
         hipMemset(m->d_v, 0, sizeof(float) * kParams) == hipSuccess &&
         hipMemset(m->d_step, 0, sizeof(long long)) == hipSuccess;
    for (int l = 0; l < kLayers && ok; ++l)
      ok = hipMemset(m->d_wbf[l], 0, sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess &&
           hipMemset(m->d_wf[l], 0, sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess &&
           hipMemset(m->d_wb[l], 0, sizeof(uint16_t) * kFanIn[l] * kLdW[l]) == hipSuccess;
    ok = ok && hipDeviceSynchronize() == hipSuccess;
  }
  if (!ok) {
    gal_mlp_destroy(m);
    return GAL_E_NOMEM;
  }
  for (int v = 0; v < 30; ++v) { m->var_w[v] = 1.0f; m->sigma[v] = 1.0f; }
  m->inv_wsum = 1.0f / 30.0f;
  *out = m;
  return GAL_OK;
}

int gal_mlp_destroy(gal_mlp* m) {
  if (!m) return GAL_OK;
  release_graph(m);
  hipFree(m->d_param); hipFree(m->d_m); hipFree(m->d_v);
  for (int l = 0; l < kLayers; ++l) { hipFree(m->d_wbf[l]); hipFree(m->d_wf[l]); hipFree(m->d_wb[l]); }
  hipFree(m->d_xt); hipFree(m->d_dot); hipFree(m->d_row_loss); hipFree(m->d_rates);
  for (int l = 0; l < 3; ++l) { hipFree(m->d_ht[l]); hipFree(m->d_dzt[l]); }
  hipFree(m->d_pw); hipFree(m->d_pb); hipFree(m->d_loss_partial);
  hipFree(m->d_step); hipFree(m->d_cursor); hipFree(m->d_local); hipFree(m->d_loss_hist);
  hipFree(m->d_ix); hipFree(m->d_ih[0]); hipFree(m->d_ih[1]); hipFree(m->d_iout);
  hipFree(m->d_rej); hipFree(m->d_rej_count);
  if (m->ev_in) hipEventDestroy(m->ev_in);
  if (m->ev_out) hipEventDestroy(m->ev_out);
  if (m->stream) hipStreamDestroy(m->stream);
  delete m;
  return GAL_OK;
}

int gal_mlp_set_params(gal_mlp* m, const float* params, int64_t n) {
  if (!m || !params || n != kParams) return GAL_E_INVALID;
  HIP_TRY(hipMemcpy(m->d_param, params, sizeof(float) * kParams, hipMemcpyHostToDevice));
  HIP_TRY(hipMemset(m->d_m, 0, sizeof(float) * kParams));
  HIP_TRY(hipMemset(m->d_v, 0, sizeof(float) * kParams));
  HIP_TRY(hipMemset(m->d_step, 0, sizeof(long long)));
  for (int l = 0; l < kLayers; ++l) {
    const int64_t cnt = (int64_t)kFanIn[l] * kFanOut[l];
    hipLaunchKernelGGL(weights_to_bf16_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, 0,
                       (const float*)m->d_param, m->w_off[l], kFanIn[l], kFanOut[l], kLdW[l], m->d_wbf[l], m->d_wf[l], m->d_wb[l]);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipDeviceSynchronize());
  return GAL_OK;
}

int gal_mlp_get_params(gal_mlp* m, float* params, int64_t n) {
  if (!m || !params || n != kParams) return GAL_E_INVALID;
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(params, m->d_param, sizeof(float) * kParams, hipMemcpyDeviceToHost));
  return GAL_OK;
}

int gal_mlp_set_adam(gal_mlp* m, double lr, double lr_min, double beta1, double beta2, double eps,
                     int64_t total_steps) {
  if (!m || !(lr > 0.0) || lr_min < 0.0 || !(beta1 >= 0.0 && beta1 < 1.0) || !(beta2 >= 0.0 && beta2 < 1.0) ||
      !(eps > 0.0) || total_steps < 1)
    return GAL_E_INVALID;
  m->lr0 = (float)lr; m->lr_min = (float)lr_min; m->beta1 = (float)beta1; m->beta2 = (float)beta2;
  m->eps = (float)eps; m->total_steps = total_steps;
  release_graph(m);
  return GAL_OK;
}

int gal_mlp_set_loss(gal_mlp* m, const float* var_weight, const float* target_sigma, const int* head_vars,
                     double head_weight) {
  if (!m || !var_weight || !target_sigma || !head_vars || head_weight < 0.0) return GAL_E_INVALID;
  double ws = 0.0;
  unsigned mask = 0;
  for (int v = 0; v < 30; ++v) {
    if (var_weight[v] < 0.0f) return GAL_E_INVALID;
    m->var_w[v] = var_weight[v];
    m->sigma[v] = target_sigma[v];
    ws += var_weight[v];
    if (head_vars[v]) mask |= 1u << v;
  }
  if (!(ws > 0.0)) return GAL_E_INVALID;
  m->inv_wsum = (float)(1.0 / ws);
  m->head_mask = mask;
  m->head_w = (float)head_weight;
  release_graph(m);
  return GAL_OK;
}

int gal_mlp_forward_d(gal_mlp* m, int64_t n, const uint16_t* x, float* out, void* stream) {
  if (!m || n < 0 || (n > 0 && (!x || !out))) return GAL_E_INVALID;
  hipStream_t s = (hipStream_t)stream;
  if (n == 0) return GAL_OK;
  for (int64_t c0 = 0; c0 < n; c0 += kLaunchRows) {
    const int nc = (int)std::min<int64_t>(kLaunchRows, n - c0);
    GAL_TRY(infer(m, nc, x + c0 * kIn, out + c0 * kOutLd, s));
  }
  return GAL_OK;
}

int gal_mlp_forward_layers_d(gal_mlp* m, int64_t n, const uint16_t* x, float* out, void* stream) {
  if (!m || n < 0 || (n > 0 && (!x || !out))) return GAL_E_INVALID;
  hipStream_t s = (hipStream_t)stream;
  const int chunk = (int)std::min<int64_t>(n, kInferChunk);
  if (n == 0) return GAL_OK;
  GAL_TRY(ensure_inference(m, chunk));
  for (int64_t c0 = 0; c0 < n; c0 += chunk) {
    const int nc = (int)std::min<int64_t>(chunk, n - c0);
    GAL_TRY(infer_layers(m, nc, x + c0 * kIn, out + c0 * kOutLd, s));
  }
  return GAL_OK;
}

int gal_mlp_gradient_d(gal_mlp* m, int n, const uint16_t* x, const float* target, float* grad, float* loss,
                       void* stream) {
  if (!m || n < 1 || n > m->batch || !x || !target) return GAL_E_INVALID;
  hipStream_t s = (hipStream_t)stream;
  GAL_TRY(grad_pass(m, n, x, target, nullptr, loss, s));
  if (grad)
    hipLaunchKernelGGL(adam_kernel, dim3((unsigned)((kParams + 255) / 256)), dim3(256), 0, s,
                       adam_args(m, n, grad, 0));
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

int gal_mlp_set_dataset(gal_mlp* m, int64_t n, const uint16_t* x, const float* target, const int* perm) {
  if (!m || n < 1 || !x || !target || !perm) return GAL_E_INVALID;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(target)) & 15u) return GAL_E_INVALID;
  m->ds_n = n; m->ds_x = x; m->ds_t = target; m->ds_perm = perm;
  release_graph(m);
  return GAL_OK;
}

int gal_mlp_train_d(gal_mlp* m, int n_steps, int use_graph, float* loss_trace, void* stream) {
  if (!m || n_steps < 0 || !m->ds_x) return GAL_E_INVALID;
  if (n_steps == 0) return GAL_OK;
  if (!m->stream) HIP_TRY(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
  if (n_steps > m->loss_hist_cap) {
    release_graph(m);
    hipFree(m->d_loss_hist);
    m->d_loss_hist = nullptr;
    m->loss_hist_cap = 0;
    HIP_TRY(hipMalloc(&m->d_loss_hist, sizeof(float) * (size_t)n_steps));
    m->loss_hist_cap = n_steps;
  }
  hipStream_t cs = (hipStream_t)stream;
  HIP_TRY(hipEventRecord(m->ev_in, cs));
  HIP_TRY(hipStreamWaitEvent(m->stream, m->ev_in, 0));
  hipLaunchKernelGGL(reset_train_kernel, dim3(1), dim3(64), 0, m->stream, m->d_cursor, m->d_local);
  HIP_TRY(hipGetLastError());
  if (use_graph) {
    const int many = n_steps / kGraphSteps, rest = n_steps % kGraphSteps;
    if (many) GAL_TRY(ensure_graph(m, 1, kGraphSteps));
    if (rest) GAL_TRY(ensure_graph(m, 0, 1));
    for (int i = 0; i < many; ++i) HIP_TRY(hipGraphLaunch(m->exec[1], m->stream));
    for (int i = 0; i < rest; ++i) HIP_TRY(hipGraphLaunch(m->exec[0], m->stream));
  } else {
    for (int i = 0; i < n_steps; ++i) GAL_TRY(record_train_step(m, m->stream));
  }
  if (loss_trace)
    HIP_TRY(hipMemcpyAsync(loss_trace, m->d_loss_hist, sizeof(float) * n_steps, hipMemcpyDeviceToDevice, m->stream));
  HIP_TRY(hipEventRecord(m->ev_out, m->stream));
  HIP_TRY(hipStreamWaitEvent(cs, m->ev_out, 0));
  return GAL_OK;
}

int gal_surrogate_encode_d(gal_ode_batch* h, int n, int ld, const double* y0, const double* y1,
                           const double* node_par, const double* t0, const double* t1, const float* norm,
                           uint16_t* x, float* x_raw, float* target, void* stream) {
  if (!h || n < 0 || ld < n || !h->have_physics) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!y0 || !node_par || !t0 || !t1 || (target && !y1)) return GAL_E_INVALID;
  if (target && !h->have_table) return GAL_E_INVALID;
  hipLaunchKernelGGL(encode_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n, ld, y0, y1, node_par,
                     t0, t1, (const double*)h->d_params, h->D, (const double*)h->d_table, h->cd,
                     (int)h->params[GAL_P_PHYSICS_MODE], norm, x, x_raw, target);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

static int apply_chunk(gal_ode_batch* h, const gal_surrogate_gate* gate, int n, int ld, double* y,
                       const double* node_par, const double* t0, const double* t1, const float* mlp_out,
                       const float* norm, double* scale, int* status, int* accepted, int* reject_list,
                       int* reject_count, int index_offset, hipStream_t s) {
  GateArgs a{};
  a.n = n; a.ld = ld; a.y = y; a.np = node_par; a.t0 = t0; a.t1 = t1; a.out = mlp_out; a.norm = norm;
  a.scale = scale; a.status = status; a.accepted = accepted; a.reject_list = reject_list;
  a.reject_count = reject_count; a.index_offset = index_offset;
  a.P = h->d_params; a.tab = h->d_table; a.D = h->D; a.cd = h->cd; a.mode = (int)h->params[GAL_P_PHYSICS_MODE];
  a.gate = *gate;
  hipLaunchKernelGGL(apply_kernel, dim3((n + 255) / 256), dim3(256), 0, s, a);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

int gal_surrogate_apply_d(gal_ode_batch* h, const gal_surrogate_gate* gate, int n, int ld, double* y,
                          const double* node_par, const double* t0, const double* t1, const float* mlp_out,
                          const float* norm, double* scale, int* status, int* accepted, int* reject_list,
                          int* reject_count, void* stream) {
  if (!h || !gate || n < 0 || ld < n || !h->have_physics || !h->have_table) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!y || !node_par || !t0 || !t1 || !mlp_out || !norm || !status || !accepted || !reject_list || !reject_count)
    return GAL_E_INVALID;
  return apply_chunk(h, gate, n, ld, y, node_par, t0, t1, mlp_out, norm, scale, status, accepted, reject_list,
                     reject_count, 0, (hipStream_t)stream);
}

int gal_surrogate_evolve_d(gal_ode_batch* h, gal_mlp* m, const float* norm, const gal_surrogate_gate* gate,
                           int n, int ld, double* y, const double* node_par, const double* t_start,
                           const double* t_end, double* h_step, double* scale, int* status, int* accepted,
                           int* n_rejected, void* stream) {
  if (!h || !m || !norm || !gate || n < 0 || ld < n || n > h->n_max || !h->have_physics || !h->have_table)
    return GAL_E_INVALID;
  if (n_rejected) *n_rejected = 0;
  if (n == 0) return GAL_OK;
  if (!y || !node_par || !t_start || !t_end || !h_step || !status || !accepted) return GAL_E_INVALID;
  if ((h->flags & GAL_FLAG_SCALES_PROVIDED) && !scale) return GAL_E_INVALID;
  hipStream_t s = (hipStream_t)stream;
  if (n > m->rej_cap) {
    hipFree(m->d_rej);
    m->d_rej = nullptr;
    m->rej_cap = 0;
    HIP_TRY(hipMalloc(&m->d_rej, sizeof(int) * (size_t)n));
    m->rej_cap = n;
  }
  if (!m->d_rej_count) HIP_TRY(hipMalloc(&m->d_rej_count, sizeof(int)));
  const int chunk = std::min(n, kInferChunk);
  GAL_TRY(ensure_inference(m, chunk));
  hipLaunchKernelGGL(reset_count_kernel, dim3(1), dim3(64), 0, s, m->d_rej_count);
  HIP_TRY(hipGetLastError());
  for (int c0 = 0; c0 < n; c0 += chunk) {
    const int nc = std::min(chunk, n - c0);
    GAL_TRY(gal_surrogate_encode_d(h, nc, ld, y + c0, nullptr, node_par + c0, t_start + c0, t_end + c0, norm,
                                   m->d_ix, nullptr, nullptr, s));
    GAL_TRY(infer(m, nc, m->d_ix, m->d_iout, s));
    // With provided scales the integrator's scales stay the caller's.
    double* sc = (h->flags & GAL_FLAG_SCALES_PROVIDED) ? nullptr : (scale ? scale + c0 : nullptr);
    GAL_TRY(apply_chunk(h, gate, nc, ld, y + c0, node_par + c0, t_start + c0, t_end + c0, m->d_iout, norm, sc,
                        status + c0, accepted + c0, m->d_rej, m->d_rej_count, c0, s));
  }
  // The integrator takes the rejected list with its count in device memory,
  // so nothing here waits for the GPU: the call only enqueues work on s
  // unless the caller asks for the count on the host.
  GAL_TRY(gal_ode_evolve_subset(h, n, ld, y, node_par, t_start, t_end, h_step, scale, status, nullptr, m->d_rej, n,
                                s, m->d_rej_count));
  if (n_rejected) {
    int n_rej = 0;
    HIP_TRY(hipMemcpyAsync(&n_rej, m->d_rej_count, sizeof(int), hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    *n_rejected = n_rej;
  }
  return GAL_OK;
}

}  // extern "C"
