// Split-proposal network: 32 inputs (normalised node class histogram [16],
// node depth, candidate u, v and threshold, then 10 statistics of the
// candidate on a class-stratified subsample of the node: the estimated left
// fraction of classes 0..7, the estimated gain relative to the node's best
// estimate, the estimated overall left fraction; zero where not measured)
// -> 3 hidden layers of 256 units (GELU, tanh form) -> one output: the
// predicted gain (plain-trainer records) or the correction of the estimated
// relative gain (subsample records).
//
// Numerics: BF16 weights and activations, FP32 accumulation on the gfx950
// matrix cores (v_mfma_f32_16x16x32_bf16), FP32 bias / GELU / output layer,
// FP32 master weights and Adam state.  Gradients of the hidden layers are
// carried in BF16 between the matrix products, as the activations are.
//
// Kernels (256-thread blocks, 4 wave64s; 128-row tiles):
//   k_mlp_fwd     all layers fused, 128 (or 64 / 32) rows per block; the
//                 tile's activations stay in LDS.  A wave owns 64 output
//                 columns: 8 x 4 MFMA 16x16 tiles, one operand (activations)
//                 from LDS, the other (weights, stored in MFMA fragment order,
//                 tix()) from L2 through a register ring that runs ahead over
//                 the layers; two waves per SIMD (registers capped at 256), so
//                 one wave's epilogue overlaps another's MFMAs.  Bound by the
//                 epilogue's VALU work: 2^20 rows 560 us (520 TFLOP/s) at first,
//                 400 with the constants of the GELU folded, packed BF16
//                 conversion, 8-byte LDS stores and the output layer on the
//                 matrix cores, 340 (860 TFLOP/s) with the ring: VALU pipe 76%
//                 busy (7.5 operations an activation), matrix cores 40%.
//                 Batches of 4096 training rows: 17.4 -> 12.4 us, the backward
//                 15.5 -> 10.0 us (waits for L2 loads).
//                 Training mode also stores the BF16 GELU
//                 derivatives G = gelu'(z) of the pre-activations (the
//                 backward multiplies by them) and the BF16 activations H in
//                 MFMA fragment blocks
//                 (tix(); the weight gradient reads each operand as 1 KiB of
//                 contiguous memory).
//   k_mlp_bwd     dL/dy, then dZ3 -> dZ2 -> dZ1 with the transposed weights,
//                 dZ^T stored in BF16.
//   k_mlp_wgrad   dW = dZ^T H over one split of the batch, per 64x32 tile,
//                 into a per-split partial (no atomics: deterministic).
//   k_mlp_wgrad64 the same for inputs a multiple of 64 wide, per 64x64 tile
//                 (2x2 MFMA tiles per wave).
//   bgrad_group   output-layer weight and output-bias partials, in extra
//                 blocks of k_mlp_wgrad (the hidden biases' partials come
//                 from the weight-gradient blocks themselves).
//   k_mlp_adam    sums the split partials in fixed order, applies Adam,
//                 refreshes the BF16 weight copies and sums the step's loss.
//   k_mlp_pack    FP32 master -> BF16 copies and transposed copies in fragment
//                 order; clears the Adam state.
//   k_topk        per node, the `keep` best of K scores (radix select on the
//                 orderable score bits, ties to the lower candidate index),
//                 written in increasing candidate order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>

#pragma clang fp contract(off)

namespace pd {
namespace mlp {

constexpr int IN = 32;     // logical inputs
constexpr int INP = 32;    // padded input row (bf16 elements)
constexpr int HID = 256;
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + HID * IN;
constexpr int OFF_W2 = OFF_B1 + HID;
constexpr int OFF_B2 = OFF_W2 + HID * HID;
constexpr int OFF_W3 = OFF_B2 + HID;
constexpr int OFF_B3 = OFF_W3 + HID * HID;
constexpr int OFF_W4 = OFF_B3 + HID;
constexpr int OFF_B4 = OFF_W4 + HID;
constexpr int NPARAM = OFF_B4 + 1;
constexpr int ROWS = 64;        // rows per block of the backward pass from MID_BATCH rows
constexpr int ROWS_BIG = 128;   // ... and from BIG_BATCH rows on (weights re-read from L2 once per tile)
constexpr int ROWS_SMALL = 32;  // ... and below MID_BATCH rows (more blocks for the chip)
constexpr uint32_t BIG_BATCH = 32768;
constexpr uint32_t MID_BATCH = 8192;  // the training forward likewise: 128 / 64 / 32-row tiles
constexpr int FWD_ROWS = 128;   // rows per block of the forward pass (weights re-read from L2 once per tile)
constexpr int THREADS = 256;    // 4 wave64s
constexpr int LDA = HID + 8;    // LDS row stride in bf16 elements (16 B pad)
constexpr int SPLIT = 512;      // batch rows are padded to a multiple of this; a weight-gradient partial
                                // covers a power-of-two multiple of it (the step's `split`)
constexpr int HIST_IN = 16;     // class-histogram inputs

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even (finite inputs)
__host__ __device__ inline uint16_t f2bf(float f)
{
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

// Element (n, r) of a training-time activation or gradient matrix with rows n
// (a layer's 256 units, layers stacked) and columns r (the batch, ldb a
// multiple of 32), stored as 16 x 32 blocks of 1 KiB in MFMA-fragment order:
// block (n / 16, r / 32), inside it lane l = 16 ((r % 32) / 8) + n % 16 of a
// 16x16x32 operand holds elements 8 l .. 8 l + 7 (r % 8).  A wave reads one
// operand fragment as 1 KiB of contiguous memory; the rows of a block's
// columns r .. r + 7 are 8 contiguous elements.
__host__ __device__ __forceinline__ size_t tix(uint32_t n, uint32_t r, uint32_t ldb)
{
  return ((size_t)(n >> 4) * (ldb >> 5) + (r >> 5)) * 512u + ((r & 31u) >> 3) * 128u + (n & 15u) * 8u + (r & 7u);
}

// tix() of the lane's four results of MFMA tile (units 16 n16 .. + 15, rows 16
// r16 .. + 15, four rows of unit l % 16 a lane): the tile's part (uniform) and
// the lane's
__host__ __device__ __forceinline__ size_t tix_tile(uint32_t n16, uint32_t r16, uint32_t ldb)
{
  return ((size_t)n16 * (ldb >> 5) + (r16 >> 1)) * 512u + (r16 & 1u) * 256u;
}
__host__ __device__ __forceinline__ uint32_t tix_lane(uint32_t lane)
{
  return (lane >> 5) * 128u + (lane & 15u) * 8u + ((lane >> 4) & 1u) * 4u;
}

// Raw buffer resource word 3 of gfx9-family targets (32-bit data format,
// no swizzle); loads past the resource's byte count return zero.
constexpr int BUF_DWORD3 = 0x00020000;

// sum of the 8 BF16 values of a fragment, in element order
__device__ __forceinline__ float sum8bf(uint4 q)
{
  const uint32_t w[4] = {q.x, q.y, q.z, q.w};
  float a = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    a += bf2f((uint16_t)(w[j] & 0xffffu));
    a += bf2f((uint16_t)(w[j] >> 16));
  }
  return a;
}

__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff)
{
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, soff, 0));
}

__device__ __forceinline__ f32x4 mma(uint4 a, uint4 b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                 0, 0, 0);
}

constexpr float GELU_C = 0.7978845608028654f;   // sqrt(2 / pi)
constexpr float GELU_A = 0.044715f;

// tanh-form GELU through 0.5 (1 + tanh u) = 1 / (1 + 2^(-2u log2 e)), u =
// GELU_C (z + GELU_A z^3): the constants folded into one polynomial of z^2, one
// exp and one reciprocal, seven operations (the same function; FP32 rounding only)
constexpr float GELU_K1 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634);
constexpr float GELU_K3 = (float)(-2.0 * 0.7978845608028654 * 1.4426950408889634 * 0.044715);
__device__ __forceinline__ float gelu_sig(float z, float zz)
{
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * __builtin_fmaf(zz, GELU_K3, GELU_K1)));
}
// d gelu / dz = s + 2 z s (1 - s) u',  s = sigmoid(2u) = gelu_sig(z), h = z s, u' = c (1 + 3 a z^2)
// (u' kept finite: h (1 - s) is 0 long before z^2 overflows)
__device__ __forceinline__ float gelu_grad(float zz, float s, float h)
{
  const float du = __builtin_fmaf(fminf(zz, 1e30f), 6.0f * GELU_A * GELU_C, 2.0f * GELU_C);
  return __builtin_fmaf(h * (1.0f - s), du, s);
}

// two floats to packed BF16, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t cvt2bf(float lo, float hi)
{
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}

// device view of the packed weights
struct Weights {
  const uint16_t *W1;    // bf16, element (unit, input) at tix(unit, input, 32)
  const uint16_t *W2;    // at tix(unit, input, 256)
  const uint16_t *W3;
  const uint16_t *W2T;   // transposed: at tix(input, unit, 256)
  const uint16_t *W3T;
  const uint16_t *w4;    // [256]
  const float *theta;    // FP32 master (biases are read from it)
};

// Input features of one (node, candidate) row; the same normalisation for the
// records the plain trainer emits and for the rows the proposal scores.
//   hist[c] = n_c / n (c < 16), depth / 16, u, v scaled by the bound of each
//   component, threshold mapped from [lo, hi] to [-1, 1].
struct RowNorm {
  float inv_p[4];
  float thr_lo, thr_scale;   // thr_n = (thr - lo) * scale - 1, scale = 2 / (hi - lo)
};

__device__ __forceinline__ void cand_features(const RowNorm &nm, const float *p, float thr, float *out6,
                                              float depth)
{
  out6[0] = depth;
#pragma unroll
  for (int j = 0; j < 4; j++) out6[1 + j] = p[j] * nm.inv_p[j];
  out6[5] = (thr - nm.thr_lo) * nm.thr_scale - 1.0f;
}

// rows from memory: X bf16 [n][32]
struct RowsMem {
  const uint16_t *X;
  uint32_t n;
  __device__ __forceinline__ uint4 fill(uint32_t row, uint32_t q) const
  {
    if (row >= n) return make_uint4(0u, 0u, 0u, 0u);
    return *(const uint4 *)(X + (size_t)row * INP + q * 8);
  }
};

// training rows: row r of the batch is row perm[r] of X (perm null: row r)
struct RowsPerm {
  const uint16_t *X;
  const uint32_t *perm;
  uint32_t n;
  __device__ __forceinline__ uint4 fill(uint32_t row, uint32_t q) const
  {
    if (row >= n) return make_uint4(0u, 0u, 0u, 0u);
    return *(const uint4 *)(X + (size_t)(perm ? perm[row] : row) * INP + q * 8);
  }
};

__device__ __forceinline__ uint4 pack8(const float *v)
{
  return uint4{cvt2bf(v[0], v[1]), cvt2bf(v[2], v[3]), cvt2bf(v[4], v[5]), cvt2bf(v[6], v[7])};
}

// Matrix products of a tile of 16 RT rows: a wave owns 64 units (4 x RT MFMA
// 16x16 tiles).  MFMA fragments (16x16x32): lane l holds A[l % 16][8 (l / 16)
// .. +7], B[8 (l / 16) .. +7][l % 16]; the result C[4 (l / 16) + jj][l % 16] in
// acc[jj].  The activations are operand A and the lane's four results are four
// rows of one unit, or (UT) the weights are and they are four units of one row.
//
// The weights come from L2, a 32-deep step (4 fragments a wave) at a time and
// through a ring of registers WD steps ahead that runs on over the layers: the
// loads of a layer's first steps are in flight during the epilogue before it.
// A block of few rows has little work to hide them behind (RT = 2: 128 cycles of
// MFMA a step against ~1000 of latency) and the registers for a whole layer.
// The activations' fragments come from LDS two products ahead.  Left to the
// compiler, every step waited for its own loads.
template <int RT>
constexpr int weight_depth()
{
  return RT >= 8 ? 2 : RT == 4 ? 4 : 8;
}
constexpr int KS = HID / 32;   // steps of a hidden layer

// fragment of unit group cg (16 units), step s of a matrix with K columns (tix()
// order), through a buffer resource: the address costs one register, not two a
// fragment
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rsrc(const void *p, uint32_t bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, BUF_DWORD3);
}
__device__ __forceinline__ uint4 wfrag(__amdgpu_buffer_rsrc_t W, int K, uint32_t cg, int s, uint32_t lane)
{
  return buf_load16(W, lane * 16u, (int)((cg * (uint32_t)(K / 32) + (uint32_t)s) * 1024u));
}

// Steps [S0, S1) of the weight stream against the tile: acc = c0[ct] + ...;
// load(s) fetches step s into ring slot s % WD (nothing past the last step).
template <int S0, int S1, int RT, bool UT, int WD, class Load>
__device__ __forceinline__ void tile_gemm(const uint16_t *act, uint32_t lane, uint4 (&wb)[WD][4], const Load &load,
                                          const f32x4 (&c0)[4], f32x4 (&acc)[RT][4])
{
  constexpr int N = (S1 - S0) * RT, AD = N < 3 ? N : 3;
  const uint16_t *base = act + (lane & 15u) * LDA + (lane >> 4) * 8u;
  uint4 a[AD];
#pragma unroll
  for (int i = 0; i < AD - 1; i++) a[i] = *(const uint4 *)(base + (i % RT) * 16 * LDA + (i / RT) * 32);
#pragma unroll
  for (int i = 0; i < N; i++) {
    const int s = S0 + i / RT, rt = i % RT, j = i + AD - 1;
    if (j < N) a[j % AD] = *(const uint4 *)(base + (j % RT) * 16 * LDA + (j / RT) * 32);
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
      const f32x4 c = s == S0 ? c0[ct] : acc[rt][ct];
      acc[rt][ct] = UT ? mma(wb[s % WD][ct], a[i % AD], c) : mma(a[i % AD], wb[s % WD][ct], c);
    }
    if (rt == RT - 1) load(s + WD);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Forward.  Inference: y[row] for rows < n (grid = ceil(n / FR)).  Training
// (TRAIN): also G (gelu'(z) of the FP32 pre-activations z of layers 1..3,
// rounded to BF16 for the backward pass; element (256 l + unit, row) at
// tix()) and
// HT (BF16 activations, element (256 l + unit, row) at tix(): l = 0 is the
// input, 32 units; l = 1..3 the hidden layers); the grid covers ldb rows.
template <class Src, bool TRAIN, int FR = FWD_ROWS>
__global__ __launch_bounds__(THREADS, 2) void k_mlp_fwd(Src src, uint32_t n, Weights w, float *__restrict__ y,
                                                     uint16_t *__restrict__ G, uint16_t *__restrict__ HT, uint32_t ldb)
{
  static_assert(FR == 32 || FR == 64 || FR == 128, "32, 64 or 128 rows per block");
  constexpr int RT = FR / 16;
  __shared__ __align__(16) uint16_t act[FR * LDA];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t row0 = blockIdx.x * FR;
  constexpr int WD = weight_depth<RT>();
  const __amdgpu_buffer_rsrc_t r1 = weight_rsrc(w.W1, HID * INP * 2), r2 = weight_rsrc(w.W2, HID * HID * 2),
                               r3 = weight_rsrc(w.W3, HID * HID * 2), rth = weight_rsrc(w.theta, NPARAM * 4);
  uint4 wb[WD][4];
  const auto load = [&](int s) __attribute__((always_inline)) {
    if (s >= 1 + 2 * KS) return;
#pragma unroll
    for (int ct = 0; ct < 4; ct++)
      wb[s % WD][ct] = s == 0 ? wfrag(r1, INP, 4u * wave + ct, 0, lane)
                              : wfrag(s <= KS ? r2 : r3, HID, 4u * wave + ct, (s - 1) % KS, lane);
  };
  // bias of a layer in accumulator form
  f32x4 c0[4];
  const auto load_bias = [&](int off) __attribute__((always_inline)) {
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
      if constexpr (TRAIN) {
        const float b = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(rth, (lane & 15u) * 4u, (off + 64u * wave + 16u * ct) * 4u, 0));
        c0[ct] = f32x4{b, b, b, b};
      } else {
        c0[ct] = __builtin_bit_cast(f32x4, buf_load16(rth, (lane >> 4) * 16u, (off + 64u * wave + 16u * ct) * 4u));
      }
    }
  };
#pragma unroll
  for (int s = 0; s < WD; s++) load(s);
  load_bias(OFF_B1);
#pragma unroll
  for (uint32_t i = tid; i < FR * 4u; i += THREADS) {
    const uint32_t r = i >> 2, q = i & 3u;
    const uint4 v = src.fill(row0 + r, q);
    *(uint4 *)(act + r * LDA + q * 8) = v;
  }
  __syncthreads();
  if (TRAIN) {
    static_assert(INP == 32, "the input is two blocks of 16 units");
    // the input tile into HT's layer 0: 2 unit groups x FR / 32 row steps of
    // 1 KiB blocks, chunk c of a block = units 16 g + c % 16, rows 8 (c / 16) .. + 7
#pragma unroll
    for (uint32_t i = tid; i < (FR / 32u) * 2u * 64u; i += THREADS) {
      const uint32_t b = i >> 6, c = i & 63u;
      const uint32_t u = (b & 1u) * 16u + (c & 15u), r = (b >> 1) * 32u + (c >> 4) * 8u;
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; j++)
        w[j] = (uint32_t)act[(r + 2 * j) * LDA + u] | ((uint32_t)act[(r + 2 * j + 1) * LDA + u] << 16);
      *(uint4 *)(HT + tix(u, row0 + r, ldb)) = uint4{w[0], w[1], w[2], w[3]};
    }
  }
  f32x4 acc[RT][4];
  uint4 w4f[KS];
  const auto load_w4 = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < KS; s++) w4f[s] = *(const uint4 *)(w.w4 + 32 * s + 8u * (lane >> 4));
  };
  // the accumulators start from the bias; inference has a lane hold four units
  // of a row (one 8-byte LDS store), training four rows of a unit (the order G
  // and HT are stored in)
#pragma unroll
  for (int layer = 0; layer < 3; layer++) {
    if (layer == 0) tile_gemm<0, 1, RT, !TRAIN, WD>(act, lane, wb, load, c0, acc);
    else if (layer == 1) tile_gemm<1, 1 + KS, RT, !TRAIN, WD>(act, lane, wb, load, c0, acc);
    else tile_gemm<1 + KS, 1 + 2 * KS, RT, !TRAIN, WD>(act, lane, wb, load, c0, acc);
    if (layer < 2) {
      load_bias(layer == 0 ? OFF_B2 : OFF_B3);
    } else if (RT < 8) {
      load_w4();
    }
    __syncthreads();   // every wave has read the layer input
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
      for (int ct = 0; ct < 4; ct++) {
        float h[4], g[4];
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
          const float z = acc[rt][ct][jj], zz = z * z, sg = gelu_sig(z, zz);
          h[jj] = z * sg;
          if (TRAIN) g[jj] = gelu_grad(zz, sg, h[jj]);
        }
        const uint2 hb{cvt2bf(h[0], h[1]), cvt2bf(h[2], h[3])};
        if constexpr (TRAIN) {
          const uint32_t col = 64u * wave + 16u * ct + (lane & 15u), rb = 16u * rt + 4u * (lane >> 4);
          act[(rb + 0) * LDA + col] = (uint16_t)hb.x;
          act[(rb + 1) * LDA + col] = (uint16_t)(hb.x >> 16);
          act[(rb + 2) * LDA + col] = (uint16_t)hb.y;
          act[(rb + 3) * LDA + col] = (uint16_t)(hb.y >> 16);
          const uint32_t n16 = layer * (HID / 16) + 4u * wave + ct, r16 = row0 / 16u + rt;
          *(uint2 *)(HT + tix_tile(n16 + HID / 16, r16, ldb) + tix_lane(lane)) = hb;
          *(uint2 *)(G + tix_tile(n16, r16, ldb) + tix_lane(lane)) = uint2{cvt2bf(g[0], g[1]), cvt2bf(g[2], g[3])};
        } else {
          const uint32_t r = 16u * rt + (lane & 15u), ub = 64u * wave + 16u * ct + 4u * (lane >> 4);
          *(uint2 *)(act + r * LDA + ub) = hb;
        }
      }
    if (RT >= 8 && layer == 2) load_w4();   // (no registers for them before)
    __syncthreads();
  }
  // output layer: y = h3 . w4 + b4 on the matrix cores, w4 as every row of
  // operand A: lane l < 16 receives the sum of row 16 rt + l
  const float b4 = w.theta[OFF_B4];
#pragma unroll
  for (int i = 0; i < (RT + 3) / 4; i++) {
    const uint32_t rt = wave + 4u * i;
    if (RT % 4 != 0 && rt >= (uint32_t)RT) break;
    f32x4 s{b4, b4, b4, b4};
#pragma unroll
    for (int k = 0; k < KS; k++)
      s = mma(w4f[k], *(const uint4 *)(act + (16u * rt + (lane & 15u)) * LDA + 32 * k + 8u * (lane >> 4)), s);
    const uint32_t row = row0 + 16u * rt + lane;
    if (lane < 16u && row < (TRAIN ? ldb : n)) y[row] = s[0];
  }
}

// Backward of the mean squared error L = 1/n sum_r (y_r - t_r)^2 over the
// first n rows of the batch (rows n..ldb-1 are padding, dL/dy = 0 there), the
// target of row r being t[perm[r]] (perm null: t[r]).
// DZT receives dL/dZ_{l+1} (BF16, element (256 l + unit, row) at tix()),
// dy[ldb] FP32,
// lossp[block] the block's sum of squared errors.  TR rows per block (64 or
// 128: one or two waves hold the tile's rows in the loss reduction; 32: the
// first half of wave 0, the rest adding zeros).
template <int TR>
__global__ __launch_bounds__(THREADS, 2) void k_mlp_bwd(const float *__restrict__ y, const float *__restrict__ t,
                                                     const uint32_t *__restrict__ perm, uint32_t n, float inv_n, const uint16_t *__restrict__ G,
                                                     Weights w, uint16_t *__restrict__ DZT, float *__restrict__ dy,
                                                     float *__restrict__ lossp, uint32_t ldb)
{
  constexpr int ROWS = TR;
  constexpr int RT = ROWS / 16;
  static_assert(ROWS == 32 || ROWS == 64 || ROWS == 128, "up to two waves hold the tile's rows");
  constexpr int LW = ROWS < 64 ? 1 : ROWS / 64;   // waves of the loss reduction
  __shared__ __align__(16) uint16_t act[ROWS * LDA];
  __shared__ float dys[ROWS];
  __shared__ float wse[LW];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t row0 = blockIdx.x * ROWS;
  constexpr int WD = weight_depth<RT>();
  const __amdgpu_buffer_rsrc_t r3 = weight_rsrc(w.W3T, HID * HID * 2), r2 = weight_rsrc(w.W2T, HID * HID * 2);
  uint4 wb[WD][4];
  const auto load = [&](int s) __attribute__((always_inline)) {
    if (s >= 2 * KS) return;
#pragma unroll
    for (int ct = 0; ct < 4; ct++) wb[s % WD][ct] = wfrag(s < KS ? r3 : r2, HID, 4u * wave + ct, s % KS, lane);
  };
  // gelu' of the last layer for 64 (or ROWS) rows of the thread's unit
  constexpr int GB = ROWS < 64 ? ROWS / 8 : 8;
  uint4 g3[GB];
  const auto load_g3 = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < GB; i++) g3[i] = *(const uint4 *)(G + tix(2u * HID + tid, row0 + r0 + 8 * i, ldb));
  };
  load_g3(0);
  if (tid < 64u * LW) {
    const uint32_t row = row0 + tid;
    const bool live = tid < (uint32_t)ROWS && row < n;
    const float e = live ? y[row] - t[perm ? perm[row] : row] : 0.0f;
    const float d = live ? 2.0f * e * inv_n : 0.0f;
    if (tid < (uint32_t)ROWS) {
      dys[tid] = d;
      dy[row] = d;
    }
    float se = e * e;
    // fixed-order reduction: each wave over its 64 rows, then wave 0's sum + wave 1's
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) se += __shfl_xor(se, o);
    if (lane == 0) wse[wave] = se;
  }
  __syncthreads();
  if (tid == 0) lossp[blockIdx.x] = LW == 1 ? wse[0] : wse[0] + wse[LW - 1];
  // dZ3[r][k] = dy[r] * w4[k] * G3[r][k] (G = gelu'(z) from the forward); thread = column k
  {
    const uint32_t k = tid;
    const float wk = bf2f(w.w4[k]);
#pragma unroll
    for (int r0 = 0; r0 < ROWS; r0 += 8 * GB) {
      if (r0) load_g3(r0);
#pragma unroll
      for (int i = 0; i < GB; i++) {
        const int r8 = r0 + 8 * i;
        float v[8];
        const uint32_t gw[4] = {g3[i].x, g3[i].y, g3[i].z, g3[i].w};   // rows r8 .. r8 + 7
#pragma unroll
        for (int j = 0; j < 8; j++) {
          v[j] = dys[r8 + j] * wk * bf2f((uint16_t)(gw[j >> 1] >> (16 * (j & 1))));
        }
        const uint4 pk = pack8(v);
        *(uint4 *)(DZT + tix(2u * HID + k, row0 + r8, ldb)) = pk;
        const uint32_t pw[4] = {pk.x, pk.y, pk.z, pk.w};
#pragma unroll
        for (int j = 0; j < 8; j++) act[(r8 + j) * LDA + k] = (uint16_t)(pw[j >> 1] >> (16 * (j & 1)));
      }
    }
  }
#pragma unroll
  for (int s = 0; s < WD; s++) load(s);
  __syncthreads();
  f32x4 acc[RT][4];
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f}, c0[4] = {zero, zero, zero, zero};
  // gelu' of the tile's elements: fetched ahead of the product where registers are left
  constexpr bool G_AHEAD = RT <= 4;
  uint2 gp[G_AHEAD ? RT : 1][4];
#pragma unroll
  for (int layer = 2; layer >= 1; layer--) {
    const auto load_g = [&](int rt, int ct) __attribute__((always_inline)) {   // rows rb .. rb + 3
      return *(const uint2 *)(G + tix_tile((layer - 1) * (HID / 16) + 4u * wave + ct, row0 / 16u + rt, ldb) +
                              tix_lane(lane));
    };
    if constexpr (G_AHEAD) {
#pragma unroll
      for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int ct = 0; ct < 4; ct++) gp[rt][ct] = load_g(rt, ct);
    }
    // dH_{layer} = dZ_{layer+1} . W_{layer+1}: B[n][k] = W[n][k] = WT[k][n]
    if (layer == 2) tile_gemm<0, KS, RT, false, WD>(act, lane, wb, load, c0, acc);
    else tile_gemm<KS, 2 * KS, RT, false, WD>(act, lane, wb, load, c0, acc);
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
      for (int ct = 0; ct < 4; ct++) {
        const uint32_t col = 64u * wave + 16u * ct + (lane & 15u);
        const uint32_t rb = 16u * rt + 4u * (lane >> 4);
        uint2 gq;
        if constexpr (G_AHEAD) gq = gp[rt][ct];
        else gq = load_g(rt, ct);
        float d[4];
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
          const uint32_t gw = jj < 2 ? gq.x : gq.y;
          d[jj] = acc[rt][ct][jj] * __builtin_bit_cast(float, jj & 1 ? gw & 0xffff0000u : gw << 16);
        }
        const uint2 pk{cvt2bf(d[0], d[1]), cvt2bf(d[2], d[3])};
        act[(rb + 0) * LDA + col] = (uint16_t)pk.x;
        act[(rb + 1) * LDA + col] = (uint16_t)(pk.x >> 16);
        act[(rb + 2) * LDA + col] = (uint16_t)pk.y;
        act[(rb + 3) * LDA + col] = (uint16_t)(pk.y >> 16);
        *(uint2 *)(DZT + tix_tile((layer - 1) * (HID / 16) + 4u * wave + ct, row0 / 16u + rt, ldb) + tix_lane(lane)) = pk;
      }
    __syncthreads();
  }
}

// One block's share of the bias / output-layer partials of split s (`split`
// rows, a multiple of SPLIT), group g: g < 48 sums the 16 rows 16 g .. 16 g
// + 15 of DZT (db of hidden layer g / 16; training takes these from the
// weight-gradient blocks instead), 48 <= g < 64 the 16 rows 16 (g - 48) .. of
// H3 weighted by dy (dw4), g = 64 the output bias (db4, sum of dy).  Run by
// the extra blocks of k_mlp_wgrad; every thread of the block calls it.
// Wave w takes the 32-row steps w, w + 4, ... of the split; per step lane l
// reads the 16 bytes of the step's 1 KiB block that MFMA lane l would (row
// l % 16, batch rows 8 (l / 16) .. + 7) and adds them in order.  Then lanes
// l, l ^ 16, l ^ 32, l ^ 48 (the same row) are summed by a fixed butterfly
// and the four waves in order (deterministic).
static_assert(SPLIT % 512 == 0, "four waves take whole groups of four 32-row steps");
__device__ __forceinline__ void bgrad_group(const uint16_t *__restrict__ DZT, const uint16_t *__restrict__ HT3,
                                            const float *__restrict__ dy, uint32_t ldb, uint32_t split,
                                            float *__restrict__ part, size_t part_stride, uint32_t g, uint32_t s)
{
  __shared__ float red[4][64];
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t rb = s * split, steps = split / 32u;
  const uint32_t r8 = 8u * (lane >> 4);   // the lane's batch rows within a step
  float acc = 0.0f;
  if (g < 64u) {
    const uint16_t *blk = (g < 48u ? DZT + (size_t)g * 16u * ldb : HT3 + (size_t)(g - 48u) * 16u * ldb) + lane * 8u;
    // steps t, t + 4, t + 8, t + 12 loaded together (a split is a multiple
    // of 16 steps), added in increasing step order
    for (uint32_t t = wave; t < steps; t += 16u) {
      uint4 q[4];
#pragma unroll
      for (int u = 0; u < 4; u++) q[u] = *(const uint4 *)(blk + (size_t)((rb >> 5) + t + 4u * u) * 512u);
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const uint32_t r = rb + 32u * (t + 4u * u);
        const uint32_t w[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
        if (g < 48u) {
#pragma unroll
          for (int j = 0; j < 4; j++) {
            acc += bf2f((uint16_t)(w[j] & 0xffffu));
            acc += bf2f((uint16_t)(w[j] >> 16));
          }
        } else {
          const float4 d0 = *(const float4 *)(dy + r + r8), d1 = *(const float4 *)(dy + r + r8 + 4u);
          const float d[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
#pragma unroll
          for (int j = 0; j < 4; j++) {
            acc += d[2 * j] * bf2f((uint16_t)(w[j] & 0xffffu));
            acc += d[2 * j + 1] * bf2f((uint16_t)(w[j] >> 16));
          }
        }
      }
    }
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
  } else {
    for (uint32_t t = wave; t < steps; t += 4u) {
      const uint32_t r = rb + 32u * t;
      if (lane < 8u) {
        const float4 d = *(const float4 *)(dy + r + 4u * lane);
        acc += ((d.x + d.y) + d.z) + d.w;
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave != 0 || lane >= 16u) return;
  const float v = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
  float *out = part + (size_t)s * part_stride;
  if (g < 48u) {
    const uint32_t l = g / 16u;
    out[(l == 0 ? OFF_B1 : (l == 1 ? OFF_B2 : OFF_B3)) + (g % 16u) * 16u + lane] = v;
  } else if (g < 64u) {
    out[OFF_W4 + (g - 48u) * 16u + lane] = v;
  } else if (lane == 0) {
    out[OFF_B4] = v;
  }
}

// dW[n][k] of one layer over rows [s*split, (s+1)*split): DZ = dZ and H =
// the layer's input activations in the tix() block layout (a 16-row x
// 32-step MFMA operand is one contiguous 1 KiB block); out = partial of split s
// (row stride k_log; columns >= k_log are not stored).
// grid (4 n-tiles, k-tiles of 32, splits); wave w: rows n0 + 16 w .. +15.
// With hl != 0 one grid covers all three layers (hl elements apart in DZ and
// H, partials at OFF_W1 / OFF_W2 / OFF_W3 of part): k-tile 0 is layer 1's
// (32 inputs), 1..8 layer 2's and 9..16 layer 3's (k_log is not read).
// The blocks of k-tile 0 also sum the rows of DZ they load into the layer's
// bias partial (part - w_off + b_off, with hl the layer's OFF_B*): per lane
// its 8 values of each step in order, the steps in order, then lanes l,
// l ^ 16, l ^ 32, l ^ 48 (the same row) by a fixed butterfly.
// Rows blockIdx.y >= bg_y0 of the grid instead compute the output layer's
// partials: group 48 + (blockIdx.y - bg_y0) gridDim.x + blockIdx.x of
// bgrad_group() (HT3: the last hidden layer's activations, dy: dL/dy).
__global__ __launch_bounds__(THREADS) void k_mlp_wgrad(const uint16_t *__restrict__ DZ,
                                                       const uint16_t *__restrict__ H, uint32_t ldb, uint32_t k_log,
                                                       uint32_t split, float *__restrict__ part, size_t part_stride,
                                                       size_t hl, uint32_t w_off, uint32_t b_off,
                                                       const uint16_t *__restrict__ HT3, const float *__restrict__ dy,
                                                       uint32_t bg_y0)
{
  if (blockIdx.y >= bg_y0) {
    const uint32_t g = 48u + (blockIdx.y - bg_y0) * gridDim.x + blockIdx.x;
    if (g <= 64u) bgrad_group(DZ, HT3, dy, ldb, split, part, part_stride, g, blockIdx.z);
    return;
  }
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t kt = blockIdx.y;
  if (hl) {
    const uint32_t l = kt == 0 ? 0u : 1u + (kt - 1u) / 8u;
    kt = kt == 0 ? 0u : (kt - 1u) % 8u;
    k_log = l == 0 ? (uint32_t)IN : (uint32_t)HID;
    DZ += l * hl;
    H += l * hl;
    w_off = l == 0 ? OFF_W1 : (l == 1 ? OFF_W2 : OFF_W3);
    b_off = l == 0 ? OFF_B1 : (l == 1 ? OFF_B2 : OFF_B3);
  }
  const bool bias = kt == 0;
  float bs = 0.0f;
  const uint32_t n0 = blockIdx.x * 64u + 16u * wave, k0 = kt * 32u, s = blockIdx.z;
  const uint32_t r16 = lane & 15u;
  const uint32_t rb = s * split, re = min(ldb, rb + split);
  f32x4 acc[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
  // Two fragment sets in turn, as in k_mlp_wgrad64 below: the wave's 16 rows
  // of DZ and 32 rows of H as buffer resources, the loads of the next
  // 32-row step issued before the products of the current one.
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(DZ + (size_t)n0 * ldb), (short)0,
                                                                      (int)(16u * ldb * 2u), BUF_DWORD3);
  const __amdgpu_buffer_rsrc_t rbf = __builtin_amdgcn_make_buffer_rsrc((void *)(H + (size_t)k0 * ldb), (short)0,
                                                                       (int)(32u * ldb * 2u), BUF_DWORD3);
  const uint32_t o0 = lane * 16u, o1 = 16u * ldb * 2u + lane * 16u;   // rows +0 / +16: the next block row
  uint4 xa = buf_load16(ra, o0, (int)(rb * 32u));
  uint4 xb0 = buf_load16(rbf, o0, (int)(rb * 32u)), xb1 = buf_load16(rbf, o1, (int)(rb * 32u));
  for (uint32_t r = rb; r < re; r += 64u) {
    const int sy = (int)((r + 32u) * 32u);
    const uint4 ya = buf_load16(ra, o0, sy);
    const uint4 yb0 = buf_load16(rbf, o0, sy), yb1 = buf_load16(rbf, o1, sy);
    __builtin_amdgcn_sched_barrier(0);
    acc[0] = mma(xa, xb0, acc[0]);
    acc[1] = mma(xa, xb1, acc[1]);
    if (bias) bs += sum8bf(xa);
    __builtin_amdgcn_sched_barrier(0);
    const int sx = (int)((r + 64u < re ? r + 64u : r) * 32u);   // the last step reloads itself, unused
    xa = buf_load16(ra, o0, sx);
    xb0 = buf_load16(rbf, o0, sx);
    xb1 = buf_load16(rbf, o1, sx);
    __builtin_amdgcn_sched_barrier(0);
    acc[0] = mma(ya, yb0, acc[0]);
    acc[1] = mma(ya, yb1, acc[1]);
    if (bias) bs += sum8bf(ya);
  }
  float *out = part + (size_t)s * part_stride + w_off;
  if (bias) {
    bs += __shfl_xor(bs, 16, 64);
    bs += __shfl_xor(bs, 32, 64);
    if (lane < 16u) part[(size_t)s * part_stride + b_off + n0 + lane] = bs;
  }
#pragma unroll
  for (int ct = 0; ct < 2; ct++) {
    const uint32_t k = k0 + 16u * ct + r16;
    if (k >= k_log) continue;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) out[(size_t)(n0 + 4u * (lane >> 4) + jj) * k_log + k] = acc[ct][jj];
  }
}

// The same partials for a layer whose input width k_log is a multiple of
// 64, in 64 x 64 output tiles: wave w computes rows n0 + 32 (w % 2) .. +31
// and columns k0 + 32 (w / 2) .. +31 as 2 x 2 MFMA tiles, so each fragment
// loaded from L2 feeds two products (one in the kernel above).  The same
// fragments meet in the same order: the sums are the above kernel's.
// 1-D grid of T = (HID / 64) (k_log / 64) tiles per split times n_splits.
// Workgroup b runs on XCD b % n_xcc, and the T tiles of one split read the
// same rows of DZ and H: for every n_xcc splits, block b takes split
// n_xcc (b / (n_xcc T)) + b % n_xcc and tile (b / n_xcc) % T, which puts a
// split's tiles on one XCD (one L2).  Blocks past the last whole group of
// n_xcc splits take tile b % T of split b / T.
// The waves of k-tile 0 that load k-columns 0..31 also sum their DZ rows into
// the layer's bias partial at b_off, as k_mlp_wgrad does.
__global__ __launch_bounds__(THREADS) void k_mlp_wgrad64(const uint16_t *__restrict__ DZ,
                                                         const uint16_t *__restrict__ H, uint32_t ldb,
                                                         uint32_t k_log, uint32_t split, uint32_t n_splits,
                                                         uint32_t n_xcc, float *__restrict__ part, size_t part_stride,
                                                         uint32_t w_off, uint32_t b_off)
{
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t T = (HID / 64u) * (k_log / 64u), b = blockIdx.x, whole = n_splits / n_xcc * n_xcc * T;
  uint32_t tile, s;
  if (b < whole) {
    tile = (b / n_xcc) % T;
    s = b / (n_xcc * T) * n_xcc + b % n_xcc;
  } else {
    tile = b % T;
    s = b / T;
  }
  const uint32_t n0 = tile % (HID / 64u) * 64u + 32u * (wave & 1u);
  const uint32_t k0 = tile / (HID / 64u) * 64u + 32u * (wave >> 1);
  const bool bias = k0 == 0;
  float bs0 = 0.0f, bs1 = 0.0f;
  const uint32_t r16 = lane & 15u;
  const uint32_t rb = s * split, re = min(ldb, rb + split);
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // Two fragment sets in turn: the loads of the next 32-row step are issued
  // before the products of the current one, so each wave keeps a step of
  // loads in flight while its MFMAs run.  The split is a multiple of 512
  // rows (an even number of steps).  Buffer loads over the wave's 32 rows of
  // DZ and of H (ldb <= 2^20 rows: 64 MiB each), the row step in the scalar
  // offset.
  const int span = (int)(32u * ldb * 2u);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(DZ + (size_t)n0 * ldb), (short)0, span,
                                                                      BUF_DWORD3);
  const __amdgpu_buffer_rsrc_t rbf = __builtin_amdgcn_make_buffer_rsrc((void *)(H + (size_t)k0 * ldb), (short)0, span,
                                                                       BUF_DWORD3);
  const uint32_t o0 = lane * 16u, o1 = 16u * ldb * 2u + lane * 16u;   // rows +0 / +16: the next block row
  uint4 xa0 = buf_load16(ra, o0, (int)(rb * 32u)), xa1 = buf_load16(ra, o1, (int)(rb * 32u));
  uint4 xb0 = buf_load16(rbf, o0, (int)(rb * 32u)), xb1 = buf_load16(rbf, o1, (int)(rb * 32u));
  for (uint32_t r = rb; r < re; r += 64u) {
    const int sy = (int)((r + 32u) * 32u);
    const uint4 ya0 = buf_load16(ra, o0, sy), ya1 = buf_load16(ra, o1, sy);
    const uint4 yb0 = buf_load16(rbf, o0, sy), yb1 = buf_load16(rbf, o1, sy);
    __builtin_amdgcn_sched_barrier(0);   // keep each step's loads ahead of the other step's products
    acc[0][0] = mma(xa0, xb0, acc[0][0]);
    acc[0][1] = mma(xa0, xb1, acc[0][1]);
    acc[1][0] = mma(xa1, xb0, acc[1][0]);
    acc[1][1] = mma(xa1, xb1, acc[1][1]);
    if (bias) {
      bs0 += sum8bf(xa0);
      bs1 += sum8bf(xa1);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int sx = (int)((r + 64u < re ? r + 64u : r) * 32u);   // the last step reloads itself, unused
    xa0 = buf_load16(ra, o0, sx);
    xa1 = buf_load16(ra, o1, sx);
    xb0 = buf_load16(rbf, o0, sx);
    xb1 = buf_load16(rbf, o1, sx);
    __builtin_amdgcn_sched_barrier(0);
    acc[0][0] = mma(ya0, yb0, acc[0][0]);
    acc[0][1] = mma(ya0, yb1, acc[0][1]);
    acc[1][0] = mma(ya1, yb0, acc[1][0]);
    acc[1][1] = mma(ya1, yb1, acc[1][1]);
    if (bias) {
      bs0 += sum8bf(ya0);
      bs1 += sum8bf(ya1);
    }
  }
  float *out = part + (size_t)s * part_stride + w_off;
  if (bias) {
    bs0 += __shfl_xor(bs0, 16, 64);
    bs0 += __shfl_xor(bs0, 32, 64);
    bs1 += __shfl_xor(bs1, 16, 64);
    bs1 += __shfl_xor(bs1, 32, 64);
    if (lane < 16u) {
      part[(size_t)s * part_stride + b_off + n0 + lane] = bs0;
      part[(size_t)s * part_stride + b_off + n0 + 16u + lane] = bs1;
    }
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint32_t k = k0 + 16u * j + r16;
#pragma unroll
      for (int jj = 0; jj < 4; jj++) out[(size_t)(n0 + 16u * i + 4u * (lane >> 4) + jj) * k_log + k] = acc[i][j][jj];
    }
}


// g = sum of the split partials (fixed order); optional gradient output;
// Adam (bias-corrected, as Kingma & Ba 2015, Algorithm 1):
//   m = b1 m + (1 - b1) g;  v = b2 v + (1 - b2) g^2;
//   theta -= lr * (m * c1) / (sqrt(v * c2) + eps),  c1 = 1/(1-b1^t), c2 = 1/(1-b2^t)
// With update, the new weights also go to their BF16 copies (what k_mlp_pack
// writes, element for element).  With loss_out, the last block first sums
// the step's nblk loss partials: per thread in block order, then a fixed
// 256-way tree, times loss_scale.
// 256 threads per block.
struct Packed {
  uint16_t *W1, *W2, *W2T, *W3, *W3T, *w4;
};
__global__ __launch_bounds__(256) void k_mlp_adam(float *__restrict__ theta, float *__restrict__ m,
                                                  float *__restrict__ v, const float *__restrict__ part,
                                                  uint32_t n_split, size_t part_stride, float *__restrict__ grad_out,
                                                  int update, float lr, float b1, float b2, float eps, float c1,
                                                  float c2, Packed pk, const float *__restrict__ lossp, uint32_t nblk,
                                                  float loss_scale, float *__restrict__ loss_out)
{
  static_assert(IN == INP, "W1 rows have no padding columns");
  if (loss_out && blockIdx.x == gridDim.x - 1) {
    __shared__ float red[256];
    const uint32_t t = threadIdx.x;
    float s = 0.0f;
    for (uint32_t b = t; b < nblk; b += 256u) s += lossp[b];
    red[t] = s;
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
      if (t < h) red[t] += red[t + h];
      __syncthreads();
    }
    if (t == 0) *loss_out = red[0] * loss_scale;
  }
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint32_t)NPARAM) return;
  float g = 0.0f;
  // the partial loads issued eight at a time, added in split order
#pragma unroll 8
  for (uint32_t s = 0; s < n_split; s++) g += part[(size_t)s * part_stride + i];
  if (grad_out) grad_out[i] = g;
  if (!update) return;
  const float mi = b1 * m[i] + (1.0f - b1) * g;
  const float vi = b2 * v[i] + (1.0f - b2) * (g * g);
  m[i] = mi;
  v[i] = vi;
  const float th = theta[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  theta[i] = th;
  const uint16_t hb = f2bf(th);
  if (i < (uint32_t)OFF_B1) {
    pk.W1[tix((i - OFF_W1) / INP, (i - OFF_W1) % INP, INP)] = hb;
  } else if (i >= (uint32_t)OFF_W2 && i < (uint32_t)OFF_B2) {
    const uint32_t j = i - OFF_W2;
    pk.W2[tix(j / HID, j % HID, HID)] = hb;
    pk.W2T[tix(j % HID, j / HID, HID)] = hb;
  } else if (i >= (uint32_t)OFF_W3 && i < (uint32_t)OFF_B3) {
    const uint32_t j = i - OFF_W3;
    pk.W3[tix(j / HID, j % HID, HID)] = hb;
    pk.W3T[tix(j % HID, j / HID, HID)] = hb;
  } else if (i >= (uint32_t)OFF_W4 && i < (uint32_t)OFF_B4) {
    pk.w4[i - OFF_W4] = hb;
  }
}

// FP32 master -> BF16 working copies
__global__ void k_mlp_pack(const float *__restrict__ theta, uint16_t *__restrict__ W1, uint16_t *__restrict__ W2,
                           uint16_t *__restrict__ W2T, uint16_t *__restrict__ W3, uint16_t *__restrict__ W3T,
                           uint16_t *__restrict__ w4, float *__restrict__ m, float *__restrict__ v)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t j = i; j < (uint32_t)NPARAM; j += gridDim.x * blockDim.x) m[j] = v[j] = 0.0f;
  if (i < (uint32_t)(HID * HID)) {
    const uint32_t nn = i / HID, k = i % HID;
    const uint16_t a = f2bf(theta[OFF_W2 + i]), b = f2bf(theta[OFF_W3 + i]);
    W2[tix(nn, k, HID)] = a;
    W3[tix(nn, k, HID)] = b;
    W2T[tix(k, nn, HID)] = a;
    W3T[tix(k, nn, HID)] = b;
  }
  if (i < (uint32_t)(HID * INP)) {
    const uint32_t nn = i / INP, k = i % INP;
    W1[tix(nn, k, INP)] = k < (uint32_t)IN ? f2bf(theta[OFF_W1 + nn * IN + k]) : (uint16_t)0;
  }
  if (i < (uint32_t)HID) w4[i] = f2bf(theta[OFF_W4 + i]);
}

// ---------------------------------------------------------------------------
// Selection: scores [n_slots][K] -> sel [n_slots][keep].  The `screen`
// largest scores of a slot (ties: lower candidate index first) form its
// screened set; sel lists the first `keep` members of that set in increasing
// candidate index (screen == keep: the top keep).  Candidates are i.i.d.
// draws of the sampler, so with screen > keep the kept ones are a random
// subset of the screened set.  One 256-thread block per slot.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t order_key(float s)
{
  if (s != s) return 0u;   // NaN ranks last
  const uint32_t u = __builtin_bit_cast(uint32_t, s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__global__ __launch_bounds__(256) void k_topk(const float *__restrict__ scores, uint32_t K, uint32_t screen,
                                              uint32_t keep, uint32_t *__restrict__ sel)
{
  __shared__ uint32_t hist[256];
  __shared__ uint32_t sh_prefix, sh_need;
  __shared__ uint32_t wsum[2][4];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const float *s = scores + (size_t)blockIdx.x * K;
  uint32_t *out = sel + (size_t)blockIdx.x * keep;
  uint32_t prefix = 0u, mask = 0u, need = screen;
  for (int pass = 0; pass < 4; pass++) {
    const uint32_t shift = 24u - 8u * (uint32_t)pass;
    hist[tid] = 0u;
    __syncthreads();
    for (uint32_t i = tid; i < K; i += 256) {
      const uint32_t k = order_key(s[i]);
      if ((k & mask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (tid == 0) {
      // largest digit d with count(> d) < need <= count(>= d)
      uint32_t above = 0u, d = 255u;
      for (;; d--) {
        const uint32_t c = hist[d];
        if (above + c >= need || d == 0u) break;
        above += c;
      }
      sh_prefix = prefix | (d << shift);
      sh_need = need - above;
    }
    __syncthreads();
    prefix = sh_prefix;
    need = sh_need;
    mask |= 255u << shift;
  }
  // prefix = the screen-th largest key; the screened set is every key above
  // it and the first `need` keys equal to it; the first `keep` of the set in
  // index order are written
  uint32_t base_sel = 0u, base_eq = 0u;
  for (uint32_t c0 = 0; c0 < K; c0 += 256) {
    const uint32_t i = c0 + tid;
    const uint32_t k = i < K ? order_key(s[i]) : 0u;
    const bool gt = i < K && k > prefix, eq = i < K && k == prefix;
    const unsigned long long meq = __ballot(eq);
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64u - lane));
    if (lane == 0) wsum[0][wave] = (uint32_t)__popcll(meq);
    __syncthreads();
    uint32_t eq_before = base_eq;
    for (uint32_t w = 0; w < wave; w++) eq_before += wsum[0][w];
    eq_before += (uint32_t)__popcll(meq & lt);
    const bool take = gt || (eq && eq_before < need);
    const unsigned long long mt = __ballot(take);
    if (lane == 0) wsum[1][wave] = (uint32_t)__popcll(mt);
    __syncthreads();
    uint32_t pos = base_sel;
    for (uint32_t w = 0; w < wave; w++) pos += wsum[1][w];
    pos += (uint32_t)__popcll(mt & lt);
    if (take && pos < keep) out[pos] = i;
    for (uint32_t w = 0; w < 4; w++) {
      base_eq += wsum[0][w];
      base_sel += wsum[1][w];
    }
    __syncthreads();
  }
}

// single-wave layout probe of the MFMA fragments: C[16][16] = A[16][32] B[32][16]
// (A row-major bf16, B column-major bf16, i.e. Bt[16][32])
__global__ void k_mma_probe(const uint16_t *__restrict__ A, const uint16_t *__restrict__ Bt, float *__restrict__ C)
{
  const uint32_t lane = threadIdx.x;
  if (lane >= 64) return;
  const uint32_t r16 = lane & 15u, kg = (lane >> 4) * 8u;
  const uint4 a = *(const uint4 *)(A + r16 * 32 + kg);
  const uint4 b = *(const uint4 *)(Bt + r16 * 32 + kg);
  const f32x4 c = mma(a, b, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
  for (int jj = 0; jj < 4; jj++) C[(4u * (lane >> 4) + jj) * 16 + r16] = c[jj];
}

}  // namespace mlp
}  // namespace pd
