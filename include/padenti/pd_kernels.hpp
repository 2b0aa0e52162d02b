// gfx950 kernels of the random-forest hot path.
//
//  k_hist      (a) per-node class histograms H[slot][c][t][f]
//  k_split     (b) information-gain argmax with lowest-k tie-break
//  k_finalize      winner decode + left class counts
//  k_route         one tree level of sample routing + partition by child
//  k_predict   (c) per-pixel forest traversal (leaf ids / FP32 posteriors)
//
// Histogram design (replaces hist_update.cl:36-187 + the host SSE2
// accumulation cl_tree_trainer_impl_traverse_ts.hpp:518-617):
//  * one work item = (frontier slot, chunk of that node's samples, tile of 64
//    candidate features); a block of 4, 8 or 16 wave64s owns the item;
//  * lane l of every wave owns candidate f = perm[64*tile + l] (the node's
//    probe-coherent order, or f = 64*tile + l without one): its FeatDim
//    parameters and nT thresholds are derived by MD5 once per block (as the
//    reference derives them per (sample, feature)) and then held in VGPRs;
//  * the waves stride over the chunk's samples; a sample is wave-uniform, so
//    its record and image descriptor come through scalar loads;
//  * for each (sample, candidate) the lane counts r = #{t : !(v <= thr_t)}
//    and does ONE LDS add into rank bin [c][r] (a 32-bit or 16-bit count);
//  * at the end, count(c, t) = sum_{r <= L_t} bin[c][r] with
//    L_t = #{t' : thr_t' < thr_t}, which equals #{samples : v <= thr_t}
//    exactly (proof in the kernel comment), and is stored (single-chunk
//    node) or atomically added (multi-chunk node) to H in the reference's
//    [c][t][f] layout.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "pd_math.hpp"
#include "pd_features.hpp"
#include "pd_mlp.hpp"

#pragma clang fp contract(off)

namespace pd {

struct ImgDesc {
  uint64_t off;   // element offset of the image in the packed pixel buffer
  uint32_t w, h;
};

constexpr uint32_t NULL_SLOT = 0xffffffffu;   // padding item: the block exits at once

struct HistItem {
  uint32_t slot;    // slice-local frontier slot (NULL_SLOT: padding)
  uint32_t begin;   // first entry in the active sample list
  uint32_t count;   // number of samples (<= 65535)
  uint32_t ftile;   // candidate tile: features [64*ftile, 64*ftile+64)
};

template <class F>
struct Bounds {
  typename F::FeatType lo[F::FeatDim], hi[F::FeatDim];
  typename F::FeatType tlo, thi;
};

// sample record (16 B): x = image | class << 24, y = px_x | px_y << 16,
// (z, w) = the functor's prepared per-pixel state (Prep bits)
__device__ __forceinline__ uint32_t rec_img(uint4 r) { return r.x & 0xffffffu; }
__device__ __forceinline__ uint32_t rec_cls(uint4 r) { return r.x >> 24; }
__device__ __forceinline__ int rec_x(uint4 r) { return (int)(r.y & 0xffffu); }
__device__ __forceinline__ int rec_y(uint4 r) { return (int)(r.y >> 16); }

constexpr int HIST_THREADS = 512;   // 8 wave64s share one 64-candidate tile

// Rank bins [class][rank 0..NTP][lane] come in two layouts: 16-bit counts
// (two neighbouring lanes share a word) or, "wide", one 32-bit word per
// (rank, lane).  Either way the bin of rank r is found from the binary
// search's final threshold slot address (slot r of the lane's column) by a
// shift and a uniform offset, not by rank arithmetic.  The wide layout takes
// twice the LDS and needs 4-byte responses (slot and bin word then have the
// same stride); the trainer picks it where it still fits two blocks per CU
// (WIDE_LDS_MAX).
template <int NTP, bool WIDE>
constexpr int bin_rows() { return NTP + 1; }

// 32-bit words per rank row of one class (FPW candidate columns)
template <bool WIDE, int FPW = 64>
constexpr int bin_row_words() { return WIDE ? FPW : FPW / 2; }

constexpr size_t WIDE_LDS_MAX = 80u * 1024u;

// power-of-two slot count of the per-lane sorted threshold list
template <int NTP>
constexpr int sorted_slots() { return NTP <= 1 ? 1 : (NTP <= 8 ? 8 : (NTP <= 16 ? 16 : (NTP <= 32 ? 32 : 64))); }

// LDS words of the region shared by the rank bins and, before the bins are
// zeroed, the candidate staging (parameters + raw thresholds): the staging
// is dead once the thresholds are sorted, so the two alias.
template <class F, int NTP, bool WIDE = false, int FPW = 64>
constexpr size_t hist_front_words(uint32_t nC)
{
  const size_t bins = (size_t)nC * bin_rows<NTP, WIDE>() * bin_row_words<WIDE, FPW>();
  const size_t staging = ((size_t)(F::FeatDim + NTP) * FPW * sizeof(typename F::FeatType) + 3) / 4;
  return bins > staging ? bins : staging;
}

template <class F, int NTP, bool WIDE = false, int FPW = 64>
constexpr size_t hist_lds_bytes(uint32_t nC)
{
  return hist_front_words<F, NTP, WIDE, FPW>(nC) * 4 +                       // rank bins | staging
         (size_t)sorted_slots<NTP>() * FPW * sizeof(typename F::FeatType) + // sorted thresholds
         (size_t)NTP * FPW;                                                   // ranks L_t
}

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v)
{
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    uint64_t w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  return v;
}

// Fill the Prep words of every sample record.
template <class F>
__global__ void k_prepare(const typename F::ImgType *__restrict__ pixels, const ImgDesc *__restrict__ imgs,
                          uint4 *__restrict__ recs, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint4 r = recs[i];
  const ImgDesc d = imgs[rec_img(r)];
  ImageView<typename F::ImgType, F::nChannels> view{pixels + d.off, (int)d.w, (int)d.h};
  pack_prep<typename F::Prep>(F::prepare(view, rec_x(r), rec_y(r)), r.z, r.w);
  recs[i] = r;
}

// Response of one (sample, candidate) pair.
template <class F>
__device__ __forceinline__ typename F::FeatType hist_eval(const typename F::ImgType *__restrict__ pixels,
                                                          const ImgDesc *__restrict__ imgs, uint4 r,
                                                          const typename F::FeatType (&p)[F::FeatDim],
                                                          const AcArgs &ac)
{
  const ImgDesc d = imgs[rec_img(r)];
  ImageView<typename F::ImgType, F::nChannels> view{pixels + d.off, (int)d.w, (int)d.h};
  return eval_hook<F>(view, rec_x(r), rec_y(r), unpack_prep<typename F::Prep>(r.z, r.w), p, ac, rec_img(r));
}

// The same through the hook's fast form.
template <class F>
__device__ __forceinline__ typename F::FeatType hist_eval_fast(const typename F::ImgType *__restrict__ pixels,
                                                               const ImgDesc *__restrict__ imgs, uint4 r,
                                                               const FastParams &fp)
{
  const ImgDesc d = imgs[rec_img(r)];
  ImageView<typename F::ImgType, F::nChannels> view{pixels + d.off, (int)d.w, (int)d.h};
  return F::eval_fast(view, rec_x(r), rec_y(r), unpack_prep<typename F::Prep>(r.z, r.w), fp);
}

// Rank r = #{t : !(v <= thr_t)} of response v by a branch-free binary search
// over the column's sorted thresholds (the predicate is true exactly on a
// prefix of the sorted list; a NaN response makes it true everywhere), then
// one LDS add into bin [class][r] (ranks above nT count as nT).  crow: the
// byte offset of the sample's class row of the bins.
template <class F, int NTP, bool WIDE, int FPW = 64>
__device__ __forceinline__ void hist_add(typename F::FeatType v, uint32_t crow, const typename F::FeatType *sth,
                                         uint32_t nT, bool fv, uint32_t lane, uint32_t *bins)
{
  using T = typename F::FeatType;
  constexpr int NS = sorted_slots<NTP>();
  // binary search carried as the byte offset of slot `pos` in the lane's
  // column (slot stride FPW * sizeof(T)); the step offsets fold into the LDS
  // read's immediate
  constexpr uint32_t SB = (uint32_t)FPW * (uint32_t)sizeof(T);
  const char *col = (const char *)(sth + lane);
  const char *at = col;
#pragma unroll
  for (int step = NS / 2; step >= 1; step >>= 1) {
    const T s = *(const T *)(at + (uint32_t)(step - 1) * SB);
    at += (v <= s) ? 0u : (uint32_t)step * SB;
  }
  // the steps reach at most NS-1: one more test of slot `pos` (the first
  // slot whose predicate can be false) adds the last one when all NS are true
  if (NS == NTP) at += (v <= *(const T *)at) ? 0u : SB;
  const char *top = col + nT * SB;   // ranks above nT count as nT
  at = at < top ? at : top;
  if constexpr (WIDE) {
    static_assert(sizeof(T) == 4, "wide bins need 4-byte responses");
    // slot pos of the lane's threshold column and word [pos][lane] of a
    // class's bins are the same byte offset from their region's base
    const ptrdiff_t k = ((const char *)bins - (const char *)sth) + (ptrdiff_t)crow;   // uniform
    uint32_t *dst = (uint32_t *)(const_cast<char *>(at) + k);
    if (fv) atomicAdd(dst, 1u);
  } else {
    // the 16-bit count [pos][col] sits at byte 2 * (FPW pos + col): the
    // slot's byte offset (FPW pos + col) * sizeof(T) rescaled; its word is
    // shared with the neighbouring column (low half: even columns)
    const uint32_t off = (uint32_t)(at - (const char *)sth);
    const uint32_t hoff = sizeof(T) >= 2 ? off / (uint32_t)(sizeof(T) / 2) : off * 2u;
    uint32_t *dst = (uint32_t *)((char *)bins + crow + (hoff & ~3u));
    if (fv) atomicAdd(dst, 1u << ((lane & 1u) * 16u));
  }
}

// Class fraction p / d of a split side (counts, p <= d): the plain IEEE
// division, or (FAST, d < 2^21) the product with the side's correctly
// rounded reciprocal y = RN(1/d) and one FMA residual correction, which is
// already RN(p/d): with |p/d| in [2^e, 2^(e+1)) the corrected value is within
// 2^(e-46) of p/d, while p - m*d is a non-zero multiple of 2^(e-25) for every
// rounding midpoint m (p an integer, m an odd multiple of 2^(e-25) with a
// 25-bit numerator), so |p/d - m| >= 2^(e-25)/d > 2^(e-46).
constexpr int COUNT_RATIO_FAST_MAX = 1 << 21;
template <bool FAST>
__device__ __forceinline__ float count_ratio(uint32_t p, float fd, float y)
{
  const float fp = (float)p;
  if constexpr (FAST) {
    const float q = fp * y;
    const float r = __builtin_fmaf(-fd, q, fp);
    return __builtin_fmaf(r, y, q);
  } else {
    (void)y;
    return fp / fd;
  }
}

// k log2 k of a sample count, in FP32 (k = 0: 0): the hardware logarithm.
__device__ __forceinline__ float count_klogk(uint32_t k)
{
  return (float)k * __builtin_amdgcn_logf((float)(k > 1u ? k : 1u));
}

// Bound on |approximate gain - FP32 gain| of a pair of a node of at most 65535
// samples holding n classes (bits).  Approximate: h - (f(nL) + f(nR) - sum
// f(lc) - sum f(rc)) / N with f = count_klogk.  The counts of the four groups
// add up to 2N, and log2 k < 16: logarithms within 2^-20 (the hardware's over
// all k <= 65535; test_count_logarithm_bound) and the products' roundings (2^-24 of at most 16)
// add up to 2 * (2^-20 + 2^-20) = 4e-6, each of the 2n + 3 sums rounds by at
// most 16 * 2^-24 = 1e-6, the last three operations by 3e-6.  The FP32 gain: n
// terms a side, every partial sum at most log2 n <= 6, so n * 6 * 2^-24 =
// 4e-7 n, and 3e-6 for the roundings of the terms and the last products.  In all
// below 1.3e-5 + 2.4e-6 n.
__device__ __forceinline__ float gain_slack(uint32_t n) { return 2e-5f + 4e-6f * (float)n; }

// Per-slot mode bits of the histogram kernel.
constexpr uint8_t SLOT_ATOMIC = 1;   // several chunks add into H (else plain stores)
constexpr uint8_t SLOT_FUSED = 2;    // one chunk: evaluate the gains in-kernel, no H

// Gain of pair (t, f) read from the in-LDS prefix counts of this lane's
// candidate: left(c) = prefix_c[L_t].  Op order of learn_best_feature.cl:63-93
// (h: the node entropy, N: the node total, both computed per thread).
template <bool WIDE, int FPW = 64>
__device__ __forceinline__ uint32_t prefix_at(const uint32_t *bins, int RW, uint32_t c, uint32_t l, uint32_t col)
{
  if constexpr (WIDE) return bins[(c * RW + l) * (uint32_t)FPW + col];
  return ((const uint16_t *)bins)[(c * RW + l) * (uint32_t)FPW + col];
}

// ---------------------------------------------------------------------------
// Probe-coherent candidate order.  A functor may declare
//   static constexpr int kProbeRowA = a, kProbeRowB = b;
// when p[a] and p[b] are the row (y) offset numerators of its two texel
// probes (a == b for a one-probe feature).  The trainer then lays each node's
// candidates out along a Hilbert curve of (p[a], p[b]) before cutting them
// into 64-lane tiles.  Images are row-major and a 128-byte cache line is a
// strip of one row, so a tile whose probes share a narrow band of row
// offsets touches few lines per gather, and the samples that follow (sorted
// by pixel within an image) probe the same rows again while they are still
// in the L1.  The order only decides which lane evaluates which candidate;
// every count, key and output column stays that of the candidate's own index.
// ---------------------------------------------------------------------------
template <class F, class = void>
struct probe_rows {
  static constexpr bool on = false;
  static constexpr int a = 0, b = 0;
};
template <class F>
struct probe_rows<F, std::void_t<decltype(F::kProbeRowA), decltype(F::kProbeRowB)>> {
  static constexpr bool on = true;
  static constexpr int a = F::kProbeRowA, b = F::kProbeRowB;
};

constexpr uint32_t ORDER_MAX = 4096;   // candidates one order block sorts in LDS (a segment of a node)
constexpr uint32_t ORDER_THREADS = 1024;

// 10-bit grid coordinate of v in [lo, hi]
template <typename T>
__device__ __forceinline__ uint32_t order_coord(T v, T lo, T hi)
{
  const float span = (float)hi - (float)lo;
  float t = span > 0.0f ? ((float)v - (float)lo) / span : 0.0f;
  t = fminf(fmaxf(t, 0.0f), 1.0f);
  return (uint32_t)(t * 1023.0f);
}

// Position of cell (x, y) of the 1024 x 1024 grid along a Hilbert curve (the
// quadrant-by-quadrant xy -> d conversion with a rotation / reflection per
// level).  Consecutive positions are neighbouring cells, so any run of 64
// candidates covers a compact patch of the (row offset, row offset) plane.
PD_HD uint32_t hilbert_index(uint32_t x, uint32_t y)
{
  uint32_t d = 0;
  for (uint32_t s = 512u; s > 0u; s >>= 1) {
    const uint32_t rx = (x & s) ? 1u : 0u, ry = (y & s) ? 1u : 0u;
    d += s * s * ((3u * rx) ^ ry);
    if (ry == 0u) {
      if (rx == 1u) {
        x = 1023u - x;
        y = 1023u - y;
      }
      const uint32_t t = x;
      x = y;
      y = t;
    }
  }
  return d;
}

// One block per (slot q, segment g of ORDER_MAX candidates): perm[q][j] for
// j in the segment = the candidate (output column) at tile position j,
// the segment's candidates sorted by (Hilbert position of the probes' row
// offsets, column): a bitonic sort of <= ORDER_MAX 64-bit keys in LDS.
// Segments are whole tiles (ORDER_MAX is a multiple of 64) and perm holds
// 16-bit columns, so nF <= 65536.
template <class F>
__global__ __launch_bounds__(ORDER_THREADS) void k_cand_order(uint32_t tree, const int32_t *__restrict__ slot_node,
                                                              uint32_t nF, Bounds<F> bnd,
                                                              const uint32_t *__restrict__ cand_map,
                                                              uint16_t *__restrict__ perm)
{
  using T = typename F::FeatType;
  constexpr int A = probe_rows<F>::a, B = probe_rows<F>::b;
  static_assert(probe_rows<F>::on && A >= 0 && A < F::FeatDim && B >= 0 && B < F::FeatDim,
                "kProbeRowA / kProbeRowB name parameters of the feature");
  __shared__ unsigned long long key[ORDER_MAX];
  static_assert(ORDER_MAX % 64u == 0u && ORDER_MAX <= 65536u, "segments of whole tiles, 16-bit keys");
  const uint32_t q = blockIdx.x;
  const uint32_t base = blockIdx.y * ORDER_MAX;
  const uint32_t n = nF - base < ORDER_MAX ? nF - base : ORDER_MAX;   // the grid has base < nF
  const uint32_t node = (uint32_t)slot_node[q];
  uint32_t n2 = 1;
  while (n2 < n) n2 <<= 1;
  for (uint32_t f = threadIdx.x; f < n2; f += ORDER_THREADS) {
    unsigned long long k = ~0ull;   // padding sorts last
    if (f < n) {
      const uint32_t fs = cand_map ? cand_map[(size_t)q * nF + base + f] : base + f;
      T p[F::FeatDim];
      candidate_params<T, F::FeatDim>(tree, node, fs, bnd.lo, bnd.hi, p);
      const uint32_t qa = order_coord<T>(p[A], bnd.lo[A], bnd.hi[A]);
      const uint32_t m = A == B ? qa : hilbert_index(qa, order_coord<T>(p[B], bnd.lo[B], bnd.hi[B]));
      k = ((unsigned long long)m << 32) | f;
    }
    key[f] = k;
  }
  __syncthreads();
  for (uint32_t size = 2; size <= n2; size <<= 1) {
    for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
      for (uint32_t i = threadIdx.x; i < n2 / 2; i += ORDER_THREADS) {
        const uint32_t a = 2u * i - (i & (stride - 1u));   // partner a + stride, bit `stride` of a clear
        const unsigned long long x = key[a], y = key[a + stride];
        const bool up = (a & size) == 0u;
        if ((x > y) == up) {
          key[a] = y;
          key[a + stride] = x;
        }
      }
      __syncthreads();
    }
  }
  for (uint32_t j = threadIdx.x; j < n; j += ORDER_THREADS)
    perm[(size_t)q * nF + base + j] = (uint16_t)(base + (uint32_t)(key[j] & 0xffffu));
}

// SPW samples per wave step: a tile holds FPW = 64 / SPW candidates, lane l
// evaluates column l % FPW on sample l / FPW of the step.  SPW = 1 is the
// wave-uniform sample of the description above; SPW > 1 lets neighbouring
// samples of the chunk share the lines their probes touch in one gather.
//
// Candidate table (optional, ctab): the staging of every (slot q, tile,
// column) computed beforehand by k_cand_table -- the parameters and the raw
// thresholds the block would derive by MD5, laid out
// [q][tile][FD + nT][FPW] -- so that a block copies them (all its waves,
// coalesced) instead of one wave running the threshold chain (nT / 4
// dependent MD5s) while the others wait at the barrier.
template <class F>
__global__ __launch_bounds__(256) void k_cand_table(uint32_t tree, const int32_t *__restrict__ slot_node,
                                                    uint32_t n_slots, uint32_t nF, uint32_t nT, uint32_t fpw,
                                                    uint32_t ftiles, Bounds<F> bnd,
                                                    const uint32_t *__restrict__ cand_map,
                                                    const uint16_t *__restrict__ perm,
                                                    typename F::FeatType *__restrict__ ctab)
{
  using T = typename F::FeatType;
  constexpr int FD = F::FeatDim;
  const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
  const uint64_t per_slot = (uint64_t)ftiles * fpw;
  if (i >= (uint64_t)n_slots * per_slot) return;
  const uint32_t q = (uint32_t)(i / per_slot);
  const uint32_t tp = (uint32_t)(i % per_slot);
  const uint32_t tile = tp / fpw, col = tp % fpw;
  const bool fv = tp < nF;
  // the same column -> candidate mapping as the histogram kernel
  const uint32_t f = (perm && fv) ? (uint32_t)perm[(size_t)q * nF + tp] : tp;
  const uint32_t fs = (cand_map && fv) ? cand_map[(size_t)q * nF + f] : f;
  const uint32_t node = (uint32_t)slot_node[q];
  const uint32_t rec = (uint32_t)FD + nT;
  T *out = ctab + ((size_t)q * ftiles + tile) * rec * fpw + col;
  T p[FD];
  candidate_params<T, FD>(tree, node, fs, bnd.lo, bnd.hi, p);
#pragma unroll
  for (int j = 0; j < FD; j++) out[(size_t)j * fpw] = p[j];
  U4 s = {tree, node, fs, 1u};
  for (uint32_t t = 0; t < nT; t++) {
    if ((t & 3u) == 0u) s = md5rand(s);
    out[(size_t)(FD + t) * fpw] = sample_value<T>(u4_get(s, t & 3u), bnd.tlo, bnd.thi);
  }
}

// Eight waves a SIMD are asked for to bound the scalar registers: a SIMD has 800 and,
// with 16 a wave for the trap handler, a wave with more than 80 leaves room for
// seven; the pruned search's loops had taken some instantiations to 82.  Hooks whose
// tile leaves LDS for more blocks lose by it: the int16 demo hook, 300 images, 1000 x
// 20 candidates, 14.0 ms of histograms a tree at 74 registers (before the pruned
// search), 14.6 at 82, 12.6 at 78; the depth hooks are within 0.5% either way.
template <class F, int NTP, int NWAVES = HIST_THREADS / 64, bool WIDE = false, int SPW = 1>
__global__ __launch_bounds__(NWAVES * 64, 8) void k_hist(
    const typename F::ImgType *__restrict__ pixels, const ImgDesc *__restrict__ imgs,
    const uint4 *__restrict__ recs, const HistItem *__restrict__ items, uint32_t item_base,
    const int32_t *__restrict__ slot_node, const uint8_t *__restrict__ slot_mode,
    const int32_t *__restrict__ slot_hidx, const uint32_t *__restrict__ tot, const float *__restrict__ slot_h,
    Bounds<F> bnd, uint32_t tree,
    uint32_t nF, uint32_t nT, uint32_t nC, uint32_t *__restrict__ H, unsigned long long *__restrict__ cand_key,
    uint32_t *__restrict__ cand_left, const uint32_t *__restrict__ cand_map, const uint16_t *__restrict__ perm,
    const typename F::FeatType *__restrict__ ctab, uint32_t fast, AcArgs ac)
{
  using T = typename F::FeatType;
  constexpr int FD = F::FeatDim;
  constexpr int RW = bin_rows<NTP, WIDE>();   // rank rows per class
  constexpr uint32_t NW = NWAVES;
  constexpr uint32_t NTH = NWAVES * 64;
  constexpr uint32_t FPW = 64u / (uint32_t)SPW;   // candidate columns of the tile
  static_assert(SPW == 1 || SPW == 2 || SPW == 4, "1, 2 or 4 samples per wave step");
  static_assert(NWAVES >= 2, "candidate set-up uses two waves");
  constexpr int NS = sorted_slots<NTP>();
  constexpr uint32_t CROW = (uint32_t)(RW * bin_row_words<WIDE, (int)FPW>() * 4);   // class row of the bins, bytes
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t *bins = lds;           // [nC][RW][FPW] counts, zeroed once the staging is dead
  T *sp = (T *)lds;               // staging: parameters [FD][FPW] ...
  T *st = sp + FD * FPW;          // ... and raw thresholds [NTP][FPW]
  T *sth = (T *)(lds + hist_front_words<F, NTP, WIDE, (int)FPW>(nC));
  uint8_t *sl = (uint8_t *)(sth + NS * FPW);

  const HistItem it = items[item_base + blockIdx.x];
  if (it.slot == NULL_SLOT) return;   // whole block: no barrier reached
  const uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63u;
  const uint32_t col = lane % FPW;   // the lane's candidate column
  const uint32_t sub = lane / FPW;   // the lane's sample within a wave step
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // tile position tp; the column's candidate (output column) f is tp itself
  // or the slot's probe-coherent order at tp
  const uint32_t tp = it.ftile * FPW + col;
  const bool fv = tp < nF;
  const uint32_t f = (perm && fv) ? (uint32_t)perm[(size_t)it.slot * nF + tp] : tp;
  const uint32_t node = (uint32_t)slot_node[it.slot];
  // sampler index of the lane's candidate: f itself, or (proposal) the
  // f-th entry of the slot's selected candidate list
  const uint32_t fs = (cand_map && fv) ? cand_map[(size_t)it.slot * nF + f] : f;

  // candidate parameters and thresholds: copied from the candidate table, or
  // derived here by wave 0 (parameters) and wave 1 (thresholds), one MD5
  // chain each
  if (ctab) {
    const uint32_t ftiles = (nF + FPW - 1) / FPW;
    const uint32_t rec = (uint32_t)FD + nT;
    const T *src = ctab + ((size_t)it.slot * ftiles + it.ftile) * rec * FPW;
    for (uint32_t i = tid; i < (uint32_t)(FD + NTP) * FPW; i += NTH) {
      const uint32_t j = i / FPW;
      if (j < (uint32_t)FD) sp[i] = src[i];
      else st[i - FD * FPW] = (j - FD < nT) ? src[i] : pad_threshold<T>();
    }
  } else if (tid < FPW) {
    T p[FD];
    candidate_params<T, FD>(tree, node, fs, bnd.lo, bnd.hi, p);
#pragma unroll
    for (int j = 0; j < FD; j++) sp[j * FPW + col] = p[j];
  } else if (tid >= 64 && tid < 64 + FPW) {
    U4 s = {tree, node, fs, 1u};
#pragma unroll
    for (int t = 0; t < NTP; t++) {
      if ((t & 3) == 0 && (uint32_t)t < nT) s = md5rand(s);
      st[t * FPW + col] = ((uint32_t)t < nT) ? sample_value<T>(u4_get(s, t & 3), bnd.tlo, bnd.thi)
                                              : pad_threshold<T>();
    }
  }
  __syncthreads();
  // Per (t, f): the stable sort position (ties by index) that scatters the
  // column's thresholds into sorted order; slots nT..NS-1 hold the padding
  // value, which is below nothing.  A group of waves sorts the column's
  // thresholds TS at a time against one pass over all of them (one threshold a
  // pass with two compares each read the column TS times: histograms of a tree of
  // depth 20, 4000 x 32 candidates, 123 -> 119 ms).
  {
    constexpr uint32_t G = NW * SPW;                          // thresholds per step
    constexpr int TS = (NTP + (int)G - 1) / (int)G;           // thresholds per lane
    T th[TS];
    uint32_t P[TS];
#pragma unroll
    for (int i = 0; i < TS; i++) {
      const uint32_t t = (uint32_t)i * G + wave * SPW + sub;
      th[i] = st[(t < (uint32_t)NTP ? t : 0u) * FPW + col];
      P[i] = 0u;
    }
#pragma unroll 4
    for (int t2 = 0; t2 < NTP; t2++) {
      const T o = st[t2 * FPW + col];
#pragma unroll
      for (int i = 0; i < TS; i++) {
        const uint32_t t = (uint32_t)i * G + wave * SPW + sub;
        P[i] += ((uint32_t)t2 < t ? o <= th[i] : o < th[i]) ? 1u : 0u;
      }
    }
#pragma unroll
    for (int i = 0; i < TS; i++) {
      const uint32_t t = (uint32_t)i * G + wave * SPW + sub;
      if (t < nT) {
        sth[P[i] * FPW + col] = th[i];
        sl[t * FPW + col] = (uint8_t)P[i];   // L_t once equal thresholds are counted out, below
      }
    }
    for (uint32_t t = nT + wave * SPW + sub; t < (uint32_t)NS; t += G) sth[t * FPW + col] = pad_threshold<T>();
  }
  T p[FD];
#pragma unroll
  for (int j = 0; j < FD; j++) p[j] = sp[j * FPW + col];
  __syncthreads();   // staging read by every wave: the bins may now take its place
  // rank L_t = #{t' < nT : thr_t' < thr_t} (used by the flush): the sorted
  // position of the first threshold equal to thr_t
  for (uint32_t t = wave * SPW + sub; t < nT; t += NW * SPW) {
    uint32_t l = sl[t * FPW + col];
    const T th = sth[l * FPW + col];
    while (l > 0u && !(sth[(l - 1u) * FPW + col] < th)) l--;
    sl[t * FPW + col] = (uint8_t)l;
  }
  for (uint32_t i = tid; i < nC * (uint32_t)(RW * bin_row_words<WIDE, (int)FPW>()); i += NTH) bins[i] = 0u;
  __syncthreads();

  // Sample loop.  r(v) = #{t : !(v <= thr_t)} is #{t : thr_t < v} for a
  // finite v and >= nT for NaN (padded slots never count for finite v).
  // v <= thr_t  <=>  r(v) <= L_t:  if v <= thr_t every thr below v is below
  // thr_t; if v > thr_t then thr_t and every thr <= thr_t are below v, so
  // r(v) >= L_t + 1.
  const uint32_t end = it.begin + it.count;
  auto scan_samples = [&](auto eval) {
    if constexpr (SPW == 1) {
      // two samples per wave and step, each wave-uniform (scalar record loads).
      // (A variant with unpredicated probes that issued both samples' gathers
      // before either bin update measured slower: the gathers are bound by
      // throughput, not latency.)
      uint32_t i = it.begin + wave;
      for (; i + NW < end; i += 2 * NW) {
        const uint4 ra = recs[i];
        const uint4 rb = recs[i + NW];
        hist_add<F, NTP, WIDE>(eval(ra), __builtin_amdgcn_readfirstlane(rec_cls(ra) * CROW), sth, nT, fv, lane, bins);
        hist_add<F, NTP, WIDE>(eval(rb), __builtin_amdgcn_readfirstlane(rec_cls(rb) * CROW), sth, nT, fv, lane, bins);
      }
      if (i < end) {
        const uint4 ra = recs[i];
        hist_add<F, NTP, WIDE>(eval(ra), __builtin_amdgcn_readfirstlane(rec_cls(ra) * CROW), sth, nT, fv, lane, bins);
      }
    } else {
      // SPW consecutive samples per wave step, one per group of FPW lanes
      // (per-lane record loads; a lane past the chunk's end re-reads its first
      // record and adds nothing)
      for (uint32_t i = it.begin + wave * SPW; i < end; i += NW * SPW) {
        const uint32_t s = i + sub;
        const bool sv = s < end;
        const uint4 r = recs[sv ? s : it.begin];
        hist_add<F, NTP, WIDE, (int)FPW>(eval(r), rec_cls(r) * CROW, sth, nT, fv && sv, col, bins);
      }
    }
  };
  // the hook's fast form where the launch's feature bounds allow it
  if constexpr (has_fast<F>::value) {
    if (fast) {
      const FastParams fp = F::fast_params(p);
      scan_samples([&](const uint4 &r) { return hist_eval_fast<F>(pixels, imgs, r, fp); });
    } else {
      scan_samples([&](const uint4 &r) { return hist_eval<F>(pixels, imgs, r, p, ac); });
    }
  } else {
    scan_samples([&](const uint4 &r) { return hist_eval<F>(pixels, imgs, r, p, ac); });
  }
  __syncthreads();

  // Flush: per (class, column), classes strided over the waves and the
  // sample groups, turn the column's rank bins into prefix counts in place,
  // then count(c, t) = prefix[L_t].
  const uint8_t mode = slot_mode[it.slot];
  const int32_t hidx = slot_hidx[it.slot];
  const size_t per_class = (size_t)nT * nF;
  for (uint32_t c = wave * SPW + sub; c < nC; c += NW * SPW) {
    uint32_t run = 0;
    if constexpr (WIDE) {
      uint32_t *b = bins + (size_t)c * RW * FPW + col;
#pragma unroll
      for (int j = 0; j < RW; j++) {
        run += b[j * FPW];
        b[j * FPW] = run;
      }
    } else {
      uint16_t *b = (uint16_t *)bins + (size_t)c * RW * FPW + col;
#pragma unroll
      for (int j = 0; j < RW; j++) {
        run += b[j * FPW];
        b[j * FPW] = (uint16_t)run;
      }
    }
    if (!fv || hidx < 0) continue;
    uint32_t *out = H + ((size_t)hidx * nC + c) * per_class + f;
#pragma unroll
    for (int t = 0; t < NTP; t++) {
      if ((uint32_t)t >= nT) break;
      const uint32_t val = prefix_at<WIDE, (int)FPW>(bins, RW, c, sl[t * FPW + col], col);
      if (mode & SLOT_ATOMIC) {
        if (val) atomicAdd(out + (size_t)t * nF, val);
      } else {
        out[(size_t)t * nF] = val;
      }
    }
  }
  if (!(mode & SLOT_FUSED)) return;

  // Fused split search of this tile: the first maximum over k = t*nF + f of
  // the FP32 gain (keys: larger gain, then smaller k), then the winner's
  // left class counts.  Candidates of the other tiles of the node are merged
  // by the finalize kernel.
  __shared__ unsigned long long red[NW];
  __syncthreads();
  const uint32_t *tt = tot + (size_t)it.slot * nC;
  int N = 0;
  // classes the node holds (bit c): a class without a sample in the node
  // has zero counts on both sides of every split, its two entropy terms are
  // plogp(+0) = +0 and subtracting them leaves hL and hR unchanged, so the
  // scan skips it (the same floats; a wave-uniform loop over the set bits,
  // in increasing class order)
  uint64_t held = 0;
  for (uint32_t c = 0; c < nC; c++) {
    N += (int)tt[c];
    if (tt[c]) held |= 1ull << c;
  }
  const float fN = (float)N;
  // the node entropy -sum plogp(tot_c / N), computed once per slot by the
  // host with the same FP32 / log2 operations (slot_entropy)
  const float h = slot_h[it.slot];
  unsigned long long best = 0ull;
  // The FP32 gain of a pair costs an IEEE division and a 45-operation FP64
  // logarithm per class and side, and only the tile's largest is wanted.  So
  // every pair's gain is first approximated (gain_slack() bounds the error) and
  // only the pairs that can still be the largest, those within two error bounds
  // of the tile's largest approximation, are evaluated exactly: usually one or
  // two.  A wave with one pair evaluates it directly (nT == 1: the exact
  // evaluation of one lane costs as much as that of 64).  Levels of ~500 samples
  // a node, 4000 x 32 candidates, 16 classes: 9.8 -> 8.1 ms a level (every pair
  // exact -> this); 2000 x 20, 8 classes: 5.48 -> 5.24 ms.
  constexpr int PW = (NTP + (int)(NW * SPW) - 1) / (int)(NW * SPW);   // pairs per lane
  float approx[PW], limit = -INFINITY;
  if constexpr (NTP > 1) {
    float *red_approx = (float *)sth;   // (the sorted thresholds are done with)
    const float rN = 1.0f / fN;
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < PW; i++) {
      const uint32_t t = (uint32_t)i * (NW * SPW) + wave * SPW + sub;
      approx[i] = -INFINITY;
      if (t < nT && fv) {
        const uint32_t l = sl[t * FPW + col];
        uint32_t nL = 0;
        float s = 0.0f;
        for (uint64_t m = held; m; m &= m - 1) {
          const uint32_t c = (uint32_t)__builtin_ctzll(m);
          const uint32_t lc = prefix_at<WIDE, (int)FPW>(bins, RW, c, l, col);
          nL += lc;
          s += count_klogk(lc) + count_klogk(tt[c] - lc);
        }
        approx[i] = h - (count_klogk(nL) + count_klogk((uint32_t)N - nL) - s) * rN;
        top = fmaxf(top, approx[i]);
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) top = fmaxf(top, __shfl_xor(top, o, 64));
    if (lane == 0) red_approx[wave] = top;
    __syncthreads();
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) top = fmaxf(top, red_approx[w]);
    limit = top - 2.0f * gain_slack((uint32_t)__popcll(held));
  }
  if (fv) {
    auto scan = [&](auto fast) {
#pragma unroll
      for (int i = 0; i < PW; i++) {
        const uint32_t t = (uint32_t)i * (NW * SPW) + wave * SPW + sub;
        if (t >= nT) continue;
        if (NTP > 1 && !(approx[i] >= limit)) continue;
        const uint32_t l = sl[t * FPW + col];
        int nL = 0;
        for (uint64_t m = held; m; m &= m - 1)
          nL += (int)prefix_at<WIDE, (int)FPW>(bins, RW, (uint32_t)__builtin_ctzll(m), l, col);
        const int nR = N - nL;
        const float fL = (float)nL, fR = (float)nR;
        const float yL = 1.0f / fL, yR = 1.0f / fR;   // used by the fast form only
        float hL = 0.0f, hR = 0.0f;
        for (uint64_t m = held; m; m &= m - 1) {
          const uint32_t c = (uint32_t)__builtin_ctzll(m);
          const uint32_t lc = prefix_at<WIDE, (int)FPW>(bins, RW, c, l, col);
          float tmp = nL ? count_ratio<decltype(fast)::value>(lc, fL, yL) : 0.0f;
          hL -= plogp(tmp);
          tmp = nR ? count_ratio<decltype(fast)::value>(tt[c] - lc, fR, yR) : 0.0f;
          hR -= plogp(tmp);
        }
        const float a = fL / fN * hL;
        const float b = fR / fN * hR;
        const unsigned long long key = split_key(h - (a + b), t * nF + f);
        best = key > best ? key : best;
      }
    };
    if (N < COUNT_RATIO_FAST_MAX) scan(std::true_type{});
    else scan(std::false_type{});
  }
  best = wave_max_u64(best);
  if (lane == 0) red[wave] = best;
  __syncthreads();
  unsigned long long m = red[0];
#pragma unroll
  for (uint32_t w = 1; w < NW; w++) m = red[w] > m ? red[w] : m;
  const uint32_t ftiles = (nF + FPW - 1) / FPW;
  const size_t ci = (size_t)it.slot * ftiles + it.ftile;
  if (tid == 0) cand_key[ci] = m;
  // column of the winner (every wave holds the same lane -> column map; the
  // lowest such lane is the column itself)
  const uint64_t wmask = __ballot(fv && f == key_index(m) % nF);
  if (tid < nC) {
    uint32_t left = 0;
    if (m != 0ull) {   // (0: no pair was evaluated, see k_finalize)
      const uint32_t k = key_index(m);
      const uint32_t wl = (uint32_t)__builtin_ctzll(wmask) % FPW;
      const uint32_t l = sl[(k / nF) * FPW + wl];
      left = prefix_at<WIDE, (int)FPW>(bins, RW, tid, l, wl);
    }
    cand_left[ci * nC + tid] = left;
  }
}

// ---------------------------------------------------------------------------
// Split proposal: input rows of the network.
// slot_in[q][17] = the node's class histogram n_c / n (16, zero padded) and
// its depth feature; candidate c of node q is the sampler's candidate c
// (parameters from seed (tree, node, c, 0), the first threshold of seed
// (tree, node, c, 1)), so the pool of K candidates is exactly the plain
// trainer's candidate set with nF = K, nT = 1.
// ---------------------------------------------------------------------------
template <class F>
__device__ __forceinline__ uint4 candidate_row(const float *slot_in, uint32_t q4, uint32_t tree, uint32_t node,
                                               uint32_t cand, uint32_t t, const Bounds<F> &bnd,
                                               const mlp::RowNorm &nm, const float *stats = nullptr)
{
  using T = typename F::FeatType;
  float v[8];
  if (q4 < 2) {
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = slot_in[q4 * 8 + j];
  } else if (q4 == 2) {
    T p[F::FeatDim];
    candidate_params<T, F::FeatDim>(tree, node, cand, bnd.lo, bnd.hi, p);
    const T th = candidate_threshold<T>(tree, node, cand, t, bnd.tlo, bnd.thi);
    float pf[4];
#pragma unroll
    for (int j = 0; j < 4; j++) pf[j] = j < F::FeatDim ? (float)p[j] : 0.0f;
    mlp::cand_features(nm, pf, (float)th, v, slot_in[16]);
    v[6] = stats ? stats[0] : 0.0f;
    v[7] = stats ? stats[1] : 0.0f;
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = stats ? stats[2 + j] : 0.0f;
  }
  return mlp::pack8(v);
}

// Number of subsample statistics per candidate in a network row (columns
// 22..31): the estimated left fraction of classes 0..7, the estimated gain
// relative to the node's best estimate, the estimated overall left fraction.
constexpr int SUB_STATS = 10;
constexpr int SUB_CLASSES = 8;

// Rows of the screened candidates of the ranked slots with their stratified
// subsample statistics: row q * K + j is candidate map[q * K + j] (sampler
// index) of slot q; frac [q][K][9] holds its estimated class left fractions
// (8) and overall left fraction, est [q][K] its estimated gain, gmax [q] the
// slot's best estimate.
template <class F>
struct SubRows {
  const float *slot_in;       // [n_slots][17]
  const int32_t *slot_node;   // [n_slots]
  const uint32_t *map;        // [n_slots][K]
  const float *frac;          // [n_slots][K][9]
  const float *est;           // [n_slots][K]
  const float *gmax;          // [n_slots]
  uint32_t K, tree, n_rows;
  Bounds<F> bnd;
  mlp::RowNorm nm;
  __device__ __forceinline__ void stats(uint32_t row, float *st) const
  {
    const uint32_t q = row / K;
    const float *fr = frac + (size_t)row * (SUB_CLASSES + 1);
#pragma unroll
    for (int c = 0; c < SUB_CLASSES; c++) st[c] = fr[c];
    st[SUB_CLASSES] = gmax[q] > 0.0f ? est[row] / gmax[q] : 0.0f;
    st[SUB_CLASSES + 1] = fr[SUB_CLASSES];
  }
  __device__ __forceinline__ uint4 fill(uint32_t row, uint32_t q4) const
  {
    if (row >= n_rows) return make_uint4(0u, 0u, 0u, 0u);
    const uint32_t q = row / K;
    float st[SUB_STATS];
    if (q4 >= 2) stats(row, st);
    return candidate_row<F>(slot_in + (size_t)q * 17, q4, tree, (uint32_t)slot_node[q], map[row], 0u, bnd, nm,
                            q4 >= 2 ? st : nullptr);
  }
};

// The rows of SubRows whose candidates the correction network scores: for
// each slot the M positions sel[q][0..M) (the slot's best M by the estimate),
// row q * M + j standing for SubRows row q * K + sel[q][j].
template <class F>
struct SubRowsSel {
  SubRows<F> base;
  const uint32_t *sel;   // [n_slots][M]
  uint32_t M, n_rows;
  __device__ __forceinline__ uint4 fill(uint32_t row, uint32_t q4) const
  {
    if (row >= n_rows) return make_uint4(0u, 0u, 0u, 0u);
    return base.fill((row / M) * base.K + sel[row], q4);
  }
};

// Ranking score of the learned refinement: every pair -FLT_MAX, then the
// selected M of each slot (sel, as in SubRowsSel) get score + y, their
// estimate relative to the slot's best plus the network's correction, so the
// kept set comes from the candidates the network scored.
__global__ __launch_bounds__(256) void k_fill_f32(float *__restrict__ v, uint64_t n, float x)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = x;
}

__global__ __launch_bounds__(256) void k_sel_score(const float *__restrict__ score, const uint32_t *__restrict__ sel,
                                                   const float *__restrict__ y, uint32_t K, uint32_t M, uint64_t n,
                                                   float *__restrict__ out)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t pos = (i / M) * K + sel[i];
  out[pos] = score[pos] + y[i];
}

// Largest value of each slot's K scores (one block per slot).
__global__ __launch_bounds__(256) void k_slot_max(const float *__restrict__ v, uint32_t K, float *__restrict__ out)
{
  __shared__ float red[256];
  const float *x = v + (size_t)blockIdx.x * K;
  float m = -INFINITY;
  for (uint32_t j = threadIdx.x; j < K; j += 256) m = fmaxf(m, x[j]);
  red[threadIdx.x] = m;
  __syncthreads();
  for (uint32_t s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// Ranking score of the stratified refinement: the estimated gain relative to
// the slot's best estimate, plus (when y is given) the network's correction
// (a network with every weight zero outputs 0 and ranks exactly as the
// estimate alone).
__global__ __launch_bounds__(256) void k_residual_score(const float *__restrict__ est, const float *__restrict__ gmax,
                                                        const float *__restrict__ y, uint32_t K, uint64_t n,
                                                        float *__restrict__ score)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = gmax[i / K];
  const float r = g > 0.0f ? est[i] / g : 0.0f;
  score[i] = y ? r + y[i] : r;
}

// Records of the learned refinement (pool runs with the exact gains of every
// screened candidate, `full` [q][K], best exact gain `gbest` [q]): for slot e
// of the emit list, R rows, half of them the first R/2 of its best-estimated
// candidates (top [e][R/2], positions in 0..K) and half drawn by MD5 of
// (tree, node, j, 11); input row as SubRows, target t = the exact gain,
// rel = its value relative to the slot's best exact gain minus the estimated
// relative gain (what the network's correction should add).
template <class F>
__global__ void k_emit_sub(SubRows<F> rows, const float *__restrict__ full, const float *__restrict__ gbest,
                           const uint32_t *__restrict__ top, const uint32_t *__restrict__ emit_slots,
                           const uint64_t *__restrict__ out_base, uint32_t ne, uint32_t R,
                           uint16_t *__restrict__ out_x, float *__restrict__ out_t, float *__restrict__ out_rel)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t e = (uint32_t)(i / R), j = (uint32_t)(i % R);
  if (e >= ne) return;
  const uint32_t q = emit_slots[e];
  const uint32_t node = (uint32_t)rows.slot_node[q];
  const uint32_t pos = j < R / 2 ? top[(size_t)e * (R / 2) + j] : md5rand(U4{rows.tree, node, j, 11u}).x % rows.K;
  const uint32_t row = q * rows.K + pos;
  const uint64_t o = out_base[e] + j;
#pragma unroll
  for (uint32_t q4 = 0; q4 < 4; q4++) *(uint4 *)(out_x + o * mlp::INP + q4 * 8) = rows.fill(row, q4);
  const float g = full[row];
  out_t[o] = g;
  const float ge = rows.gmax[q] > 0.0f ? rows.est[row] / rows.gmax[q] : 0.0f;
  if (out_rel) out_rel[o] = (gbest[q] > 0.0f ? g / gbest[q] : 0.0f) - ge;
}

template <class F>
struct PoolRows {
  const float *slot_in;       // [n_slots][17]
  const int32_t *slot_node;   // [n_slots]
  uint32_t K, tree, n_rows;
  Bounds<F> bnd;
  mlp::RowNorm nm;
  __device__ __forceinline__ uint4 fill(uint32_t row, uint32_t q4) const
  {
    if (row >= n_rows) return make_uint4(0u, 0u, 0u, 0u);
    const uint32_t q = row / K, cand = row % K;
    return candidate_row<F>(slot_in + (size_t)q * 17, q4, tree, (uint32_t)slot_node[q], cand, 0u, bnd, nm);
  }
};

// Record emitter of the plain trainer: for emitting slot e (slice-local slot
// emit_slots[e]), R records (input row, measured FP32 gain) of pairs
// k = t*nF + f drawn by MD5 of (tree, node, j, 7) (all pairs in order when
// R >= nT*nF), written at out_base[e] + j; out_rel (optional) receives the
// gain relative to the node's best gain over all pairs, best[e].
template <class F>
__global__ void k_emit(const float *__restrict__ gains, const uint32_t *__restrict__ emit_slots,
                       const uint64_t *__restrict__ out_base, const float *__restrict__ best, uint32_t ne, uint32_t R,
                       const float *__restrict__ slot_in, const int32_t *__restrict__ slot_node, uint32_t nF,
                       uint32_t nT, uint32_t tree, Bounds<F> bnd, mlp::RowNorm nm, uint16_t *__restrict__ out_x,
                       float *__restrict__ out_t, float *__restrict__ out_rel)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t e = (uint32_t)(i / R), j = (uint32_t)(i % R);
  if (e >= ne) return;
  const uint32_t q = emit_slots[e];
  const uint32_t node = (uint32_t)slot_node[q];
  const uint32_t npairs = nF * nT;
  uint32_t k = j;
  if (R < npairs) k = md5rand(U4{tree, node, j, 7u}).x % npairs;
  const uint32_t f = k % nF, t = k / nF;
  const uint64_t o = out_base[e] + j;
#pragma unroll
  for (uint32_t q4 = 0; q4 < 4; q4++)
    *(uint4 *)(out_x + o * mlp::INP + q4 * 8) = candidate_row<F>(slot_in + (size_t)q * 17, q4, tree, node, f, t,
                                                                 bnd, nm);
  const float g = gains[(size_t)q * npairs + k];
  out_t[o] = g;
  if (out_rel) out_rel[o] = best[e] > 0.0f ? g / best[e] : 0.0f;
}

// Zero the H region of every slot that several chunks add into.
__global__ void k_zero_slots(uint32_t *__restrict__ H, const uint32_t *__restrict__ slots, uint32_t n_slots,
                             size_t per_slot)
{
  const size_t total = (size_t)n_slots * per_slot;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const size_t s = i / per_slot, o = i % per_slot;
    H[(size_t)slots[s] * per_slot + o] = 0u;
  }
}

// ---------------------------------------------------------------------------
// (b) split search.  Every thread scans pairs k = t*nF + f in increasing
// order keeping the first maximum (strict >), then (gain, k) keys are
// max-reduced over the wave, the block and (atomically) over the blocks of
// the slot: the larger key is the larger gain, then the smaller k — the
// reference's first maximum (learn_best_feature.cl:96-101 together with
// std::max_element, cl_tree_trainer_impl_learn_best_featthr.hpp:111-112).
// ---------------------------------------------------------------------------
constexpr int SPLIT_THREADS = 256;

template <int NCM>
__device__ __forceinline__ float node_entropy(const uint32_t *tot, uint32_t nC, int &N)
{
  int n = 0;
#pragma unroll
  for (int l = 0; l < NCM; l++)
    if ((uint32_t)l < nC) n += (int)tot[l];
  N = n;
  const float fN = (float)n;
  float h = 0.0f;
#pragma unroll
  for (int l = 0; l < NCM; l++)
    if ((uint32_t)l < nC) h -= plogp((float)tot[l] / fN);
  return h;
}

// Gain of one pair given left counts; op order of learn_best_feature.cl:63-93
// (h is the node entropy, the same value the kernel recomputes per pair).
template <int NCM, bool FAST>
__device__ __forceinline__ float pair_gain(const uint32_t *left, const uint32_t *tot, uint32_t nC, float h, int N)
{
  int nL = 0;
#pragma unroll
  for (int l = 0; l < NCM; l++)
    if ((uint32_t)l < nC) nL += (int)left[l];
  const int nR = N - nL;
  const float fN = (float)N, fL = (float)nL, fR = (float)nR;
  const float yL = 1.0f / fL, yR = 1.0f / fR;   // used by the fast form only
  float hL = 0.0f, hR = 0.0f;
#pragma unroll
  for (int l = 0; l < NCM; l++) {
    if ((uint32_t)l < nC) {
      float tmp = nL ? count_ratio<FAST>(left[l], fL, yL) : 0.0f;
      hL -= plogp(tmp);
      tmp = nR ? count_ratio<FAST>(tot[l] - left[l], fR, yR) : 0.0f;
      hR -= plogp(tmp);
    }
  }
  const float a = fL / fN * hL;
  const float b = fR / fN * hR;
  return h - (a + b);
}


// slot_list (may be NULL): the slots to search, in H order (slot_list[i] is
// the slot of H block i); NULL searches slots 0.. with H block = slot.
template <int NCM>
__global__ __launch_bounds__(SPLIT_THREADS) void k_split(const uint32_t *__restrict__ H,
                                                         const uint32_t *__restrict__ tot, uint32_t nC,
                                                         uint32_t nT, uint32_t nF, uint32_t blocks_per_slot,
                                                         uint32_t pairs_per_block,
                                                         unsigned long long *__restrict__ best,
                                                         float *__restrict__ all_gains,
                                                         const uint32_t *__restrict__ slot_list)
{
  __shared__ uint64_t red[SPLIT_THREADS / 64];
  const uint32_t hblk = blockIdx.x / blocks_per_slot;
  const uint32_t slot = slot_list ? slot_list[hblk] : hblk;
  const uint32_t part = blockIdx.x % blocks_per_slot;
  const uint32_t npairs = nT * nF;
  uint32_t tv[NCM];
#pragma unroll
  for (int l = 0; l < NCM; l++) tv[l] = ((uint32_t)l < nC) ? tot[(size_t)slot * nC + l] : 0u;
  int N;
  const float h = node_entropy<NCM>(tv, nC, N);
  const uint32_t *Hs = H + (size_t)hblk * nC * npairs;
  const uint32_t k0 = part * pairs_per_block;
  const uint32_t k1 = min(npairs, k0 + pairs_per_block);
  uint64_t key = 0;
  auto scan = [&](auto fast) {
    for (uint32_t k = k0 + threadIdx.x; k < k1; k += SPLIT_THREADS) {
      uint32_t left[NCM];
#pragma unroll
      for (int l = 0; l < NCM; l++) left[l] = ((uint32_t)l < nC) ? Hs[(size_t)l * npairs + k] : 0u;
      const float g = pair_gain<NCM, decltype(fast)::value>(left, tv, nC, h, N);
      if (all_gains) all_gains[(size_t)slot * npairs + k] = g;
      const uint64_t kk = split_key(g, k);
      key = kk > key ? kk : key;
    }
  };
  if (N < COUNT_RATIO_FAST_MAX) scan(std::true_type{});
  else scan(std::false_type{});
  key = wave_max_u64(key);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = key;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t m = red[0];
#pragma unroll
    for (int w = 1; w < SPLIT_THREADS / 64; w++) m = red[w] > m ? red[w] : m;
    atomicMax(best + slot, (unsigned long long)m);
  }
}

// Winner of each slot: res[slot] = {k, gain bits, left[0..nC)}.  A fused
// slot takes the largest key over its tiles' candidates (larger gain, then
// smaller k) and that tile's left counts; any other slot its searched key
// and the counts of H block slot_hidx[slot].  With par / thr, also the winner's
// feature parameters and threshold, re-derived from the sampler for the tree
// arrays (f mapped through cand_map when given; the reference re-derives them
// on the host, cl_tree_trainer_impl_learn_best_featthr.hpp:183-222).
template <class F>
__global__ void k_finalize(const uint32_t *__restrict__ H, const unsigned long long *__restrict__ best,
                           const uint8_t *__restrict__ slot_mode, const int32_t *__restrict__ slot_hidx,
                           const unsigned long long *__restrict__ cand_key, const uint32_t *__restrict__ cand_left,
                           uint32_t n_slots, uint32_t nC, uint32_t nT, uint32_t nF, uint32_t fpw,
                           uint32_t *__restrict__ res, uint32_t tree, const int32_t *__restrict__ slot_node,
                           const uint32_t *__restrict__ cand_map, Bounds<F> bnd,
                           typename F::FeatType *__restrict__ par, typename F::FeatType *__restrict__ thr)
{
  using T = typename F::FeatType;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t slot = i / (nC + 2), c = i % (nC + 2);
  if (slot >= n_slots) return;
  uint64_t key;
  size_t ci = 0;
  const bool fused = (slot_mode[slot] & SLOT_FUSED) != 0;
  if (fused) {
    const uint32_t ftiles = (nF + fpw - 1) / fpw;
    key = 0;
    for (uint32_t ft = 0; ft < ftiles; ft++) {
      const uint64_t kk = cand_key[(size_t)slot * ftiles + ft];
      if (kk > key) {
        key = kk;
        ci = (size_t)slot * ftiles + ft;
      }
    }
  } else {
    key = best[slot];
  }
  uint32_t k = key_index(key);
  // A search of a slot that holds samples evaluates some pair: k_split all of them,
  // the fused search at least the one with the tile's largest approximation, which
  // is finite.  (An empty fused slot, N = 0, would evaluate none: key 0, pair 0, no
  // left samples.  Frontier nodes hold samples and train() refuses an empty set.)
  if (k >= nT * nF) k = 0;
  uint32_t *r = res + (size_t)slot * (nC + 2);
  if (c == 0) {
    r[0] = k;
    if (par) {
      const uint32_t f = k % nF;
      const uint32_t fs = cand_map ? cand_map[(size_t)slot * nF + f] : f;
      const uint32_t node = (uint32_t)slot_node[slot];
      T p[F::FeatDim];
      candidate_params<T, F::FeatDim>(tree, node, fs, bnd.lo, bnd.hi, p);
      for (int j = 0; j < F::FeatDim; j++) par[(size_t)slot * F::FeatDim + j] = p[j];
      thr[slot] = candidate_threshold<T>(tree, node, fs, k / nF, bnd.tlo, bnd.thi);
    }
  } else if (c == 1) {
    const float g = key_gain(key);
    r[1] = __float_as_uint(g);
  } else if (fused) {
    r[c] = cand_left[ci * nC + (c - 2)];
  } else {
    r[c] = H[((size_t)slot_hidx[slot] * nC + (c - 2)) * nT * nF + k];
  }
}

// ---------------------------------------------------------------------------
// Routing of one level (replaces re-running predict.cl from the root at
// every level, cl_tree_trainer_impl_traverse_ts.hpp:211-244).  Order
// preserving: k_route_flags evaluates each active sample of a split node
// and writes a left/right flag pair; an exclusive scan of the pairs gives
// every sample its rank among the samples of its node going the same way;
// k_route_scatter appends it to its child's run of the next active list.
// A node's samples therefore stay in (image, pixel) order at every level.
// ---------------------------------------------------------------------------
template <class F>
__global__ __launch_bounds__(256) void k_route_flags(const typename F::ImgType *__restrict__ pixels,
                                                     const ImgDesc *__restrict__ imgs, const uint4 *__restrict__ recs,
                                                     const uint32_t *__restrict__ rec_slot, uint32_t n,
                                                     const uint8_t *__restrict__ slot_split,
                                                     const typename F::FeatType *__restrict__ slot_feat,
                                                     const typename F::FeatType *__restrict__ slot_thr,
                                                     unsigned long long *__restrict__ flags, AcArgs ac)
{
  using T = typename F::FeatType;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  unsigned long long fl = 0ull;   // (left) | (right << 32); entry n is the scan's total
  if (i < n) {
    const uint32_t slot = rec_slot[i];
    if (slot_split[slot]) {
      const uint4 r = recs[i];
      const ImgDesc d = imgs[rec_img(r)];
      ImageView<typename F::ImgType, F::nChannels> view{pixels + d.off, (int)d.w, (int)d.h};
      T p[F::FeatDim];
#pragma unroll
      for (int j = 0; j < F::FeatDim; j++) p[j] = slot_feat[(size_t)slot * F::FeatDim + j];
      const T v = eval_hook<F>(view, rec_x(r), rec_y(r), unpack_prep<typename F::Prep>(r.z, r.w), p, ac, rec_img(r));
      fl = (v <= slot_thr[slot]) ? 1ull : (1ull << 32);
    }
  }
  flags[i] = fl;
}

// rank[i] = exclusive prefix of the flag pairs; slot q spans
// [slot_begin[q], slot_begin[q+1]) of the active list.
__global__ __launch_bounds__(256) void k_route_scatter(const uint4 *__restrict__ recs,
                                                       const uint32_t *__restrict__ rec_slot, uint32_t n,
                                                       const unsigned long long *__restrict__ flags,
                                                       const unsigned long long *__restrict__ rank,
                                                       const uint32_t *__restrict__ slot_begin,
                                                       const int32_t *__restrict__ slot_next,
                                                       const uint32_t *__restrict__ next_begin, uint4 *__restrict__ out_recs,
                                                       uint32_t *__restrict__ out_slot, uint32_t out_cap,
                                                       uint32_t n_slots, uint32_t *__restrict__ ccount)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_slots) {
    const unsigned long long a = rank[slot_begin[i]], b = rank[slot_begin[i + 1]];
    ccount[2 * i] = (uint32_t)b - (uint32_t)a;
    ccount[2 * i + 1] = (uint32_t)(b >> 32) - (uint32_t)(a >> 32);
  }
  if (i >= n) return;
  const unsigned long long fl = flags[i];
  if (!fl) return;
  const uint32_t slot = rec_slot[i];
  const uint32_t side = (uint32_t)(fl >> 32) ? 1u : 0u;
  const int32_t ns = slot_next[2 * slot + side];
  if (ns < 0) return;
  const unsigned long long r0 = rank[slot_begin[slot]], ri = rank[i];
  const uint32_t k = side ? (uint32_t)(ri >> 32) - (uint32_t)(r0 >> 32) : (uint32_t)ri - (uint32_t)r0;
  const uint32_t pos = next_begin[ns] + k;
  // out_cap bounds the write even if routing disagreed with the split counts
  // (the host compares the per-child totals with them and reports it)
  if (pos < out_cap) {
    out_recs[pos] = recs[i];
    out_slot[pos] = (uint32_t)ns;
  }
}

// ---------------------------------------------------------------------------
// (c) forest prediction.  Node records are packed breadth-first per tree
// (one aligned load per visited node).  A block covers 256 consecutive
// pixels of one frame; blocks map to frames through a prefix table.
// Posteriors are summed in tree order in FP32 and divided by nTrees
// (cl_classifier_impl.hpp:533-552); output is planar [c][y][x] per frame.
// Masked-out pixels get posterior 0 and leaf id -1.
// ---------------------------------------------------------------------------
// Compact forest node: the tree's existing nodes in breadth-first order,
// children adjacent.  left >= 0: compact index of the left child (the right
// child follows it); left < 0: leaf number -1 - left in the tree's leaf
// table (original node id + posterior row).
template <typename T, int FD>
struct alignas(FD * sizeof(T) + 8 <= 16 ? 16 : 32) NodeRec {
  int32_t left;
  T thr;
  T p[FD];
};

// A node record at a wave-uniform address, read through the scalar cache
// (one s_load for the wave instead of one texture-path load per lane).  The
// load and its wait are one asm block, so the registers are written before
// the block ends.  Records of other sizes take the vector path.
template <class Rec>
__device__ __forceinline__ Rec load_node_uniform(const Rec *p)
{
  Rec r;
  if constexpr (sizeof(Rec) == 16) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 v;
    asm volatile("s_load_dwordx4 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
    __builtin_memcpy(&r, &v, sizeof(Rec));
  } else if constexpr (sizeof(Rec) == 32) {
    typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
    u32x8 v;
    asm volatile("s_load_dwordx8 %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
    __builtin_memcpy(&r, &v, sizeof(Rec));
  } else {
    r = *p;
  }
  return r;
}

struct FrameDesc {
  uint64_t img_off;    // element offset of the frame's pixels
  uint64_t post_off;   // element offset of the frame's posterior [nC][h][w]
  uint64_t leaf_off;   // element offset of the frame's leaf ids [tree][h][w]
  uint64_t mask_off;   // byte offset of the frame's mask (if masks given)
  uint32_t w, h;
  uint32_t block0;     // first block of the frame
  uint32_t pad;
};
static_assert(sizeof(FrameDesc) == 48, "frame table entries are 48 bytes");

// XCD-aware block order: workgroup b runs on XCD b % n_xcc, so it takes
// pixel block (b % n_xcc) * per_xcc + b / n_xcc: each XCD walks one
// contiguous stretch of the frames, whose texels and rows then stay in that
// XCD's L2 (the grid is n_xcc * per_xcc blocks; those past n_blocks exit).
// Node records: while every active lane of a wave is at one node (the top
// levels of a spatially coherent block) the record is read once through the
// scalar cache instead of 64 lanes through the texture path.
// FAST: every node's offset parameters allow the hook's fast form.
template <class F, int NCM, bool FAST>
__global__ __launch_bounds__(256) void k_predict(
    const typename F::ImgType *__restrict__ pixels, const FrameDesc *__restrict__ frames, uint32_t n_frames,
    uint32_t n_blocks, uint32_t n_xcc, uint32_t per_xcc, const uint8_t *__restrict__ masks,
    const NodeRec<typename F::FeatType, F::FeatDim> *__restrict__ nodes,
    const uint32_t *__restrict__ tree_off, uint32_t n_trees, uint32_t max_steps,
    const float *__restrict__ leaf_post, const int32_t *__restrict__ leaf_id, const uint32_t *__restrict__ leaf_off,
    uint32_t nC, float *__restrict__ out_post, int32_t *__restrict__ out_leaf)
{
  using T = typename F::FeatType;
  const uint32_t blk = (blockIdx.x % n_xcc) * per_xcc + blockIdx.x / n_xcc;
  if (blk >= n_blocks) return;
  // frame of this block: last frame with block0 <= blk (uniform)
  uint32_t lo = 0, hi = n_frames;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (frames[mid].block0 <= blk) lo = mid; else hi = mid;
  }
  const FrameDesc fd = frames[lo];
  const uint32_t npx = fd.w * fd.h;
  const uint32_t px = (blk - fd.block0) * 256u + threadIdx.x;
  if (px >= npx) return;
  const int x = (int)(px % fd.w), y = (int)(px / fd.w);
  const bool on = masks ? masks[fd.mask_off + px] != 0 : true;
  ImageView<typename F::ImgType, F::nChannels> view{pixels + fd.img_off, (int)fd.w, (int)fd.h};
  const typename F::Prep prep = F::prepare(view, x, y);
  float acc[NCM];
#pragma unroll
  for (int c = 0; c < NCM; c++) acc[c] = 0.0f;
  for (uint32_t t = 0; t < n_trees; t++) {
    int32_t id = -1;
    if (on) {
      const NodeRec<T, F::FeatDim> *tr = nodes + tree_off[t];
      int32_t n = 0, leaf = 0;
      // max_steps splits at most, then the leaf (every node of a tree's
      // last level is a leaf)
      for (uint32_t s = 0; s <= max_steps; s++) {
        const int32_t n0 = __builtin_amdgcn_readfirstlane(n);
        NodeRec<T, F::FeatDim> rec;
        if (__builtin_amdgcn_ballot_w64(n != n0) == 0) rec = load_node_uniform(tr + n0);
        else rec = tr[n];
        if (rec.left < 0) {
          leaf = -1 - rec.left;
          break;
        }
        // (auto-context hooks never come here: they predict through node maps)
        T v;
        if constexpr (FAST) v = F::eval_fast(view, x, y, prep, F::fast_params(rec.p));
        else v = eval_hook<F>(view, x, y, prep, rec.p, AcArgs{}, 0u);
        n = rec.left + ((v <= rec.thr) ? 0 : 1);
      }
      const uint32_t li = leaf_off[t] + (uint32_t)leaf;
      id = leaf_id[li];
      if (out_post) {
        // leaf rows padded to a multiple of 4 floats: 16-byte loads (the
        // gather of a scattered leaf row costs per load instruction)
        const float4 *pp = (const float4 *)(leaf_post + (size_t)li * ((nC + 3u) & ~3u));
#pragma unroll
        for (int c4 = 0; c4 < NCM / 4; c4++) {
          if ((uint32_t)(4 * c4) >= nC) break;
          const float4 q = pp[c4];
          acc[4 * c4 + 0] += q.x;
          acc[4 * c4 + 1] += q.y;
          acc[4 * c4 + 2] += q.z;
          acc[4 * c4 + 3] += q.w;
        }
      }
    }
    if (out_leaf) out_leaf[fd.leaf_off + (size_t)t * npx + px] = id;
  }
  if (out_post) {
    const float nt = (float)n_trees;
#pragma unroll
    for (int c = 0; c < NCM; c++)
      if ((uint32_t)c < nC) out_post[fd.post_off + (size_t)c * npx + px] = on ? acc[c] / nt : 0.0f;
  }
}

// ---------------------------------------------------------------------------
// Node-id maps of auto-context hooks.  One pass moves every routed pixel of
// a node that has children one level down: map_out = child by the hook
// evaluated with the context of map_in (the maps of all images packed,
// image i at ac.map_off[i]; a block per 256 pixels of one image, block0[i] =
// first block of image i).  Pixels at -1 or at a leaf keep their value.
// ---------------------------------------------------------------------------
template <class F>
__global__ __launch_bounds__(256) void k_ac_route_map(const typename F::ImgType *__restrict__ pixels,
                                                      const ImgDesc *__restrict__ imgs, uint32_t n_images,
                                                      const uint32_t *__restrict__ block0,
                                                      const typename F::FeatType *__restrict__ tree_feat,
                                                      const typename F::FeatType *__restrict__ tree_thr, AcArgs ac,
                                                      int32_t *__restrict__ map_out)
{
  using T = typename F::FeatType;
  uint32_t lo = 0, hi = n_images;  // image of this block: last with block0 <= blockIdx.x (uniform)
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (block0[mid] <= blockIdx.x) lo = mid;
    else hi = mid;
  }
  const ImgDesc d = imgs[lo];
  const uint32_t npx = d.w * d.h;
  const uint32_t px = (blockIdx.x - block0[lo]) * 256u + threadIdx.x;
  if (px >= npx) return;
  const uint64_t mo = ac.map_off[lo];
  const int32_t n = ac.maps[mo + px];
  int32_t out = n;
  if (n >= 0) {
    const int32_t lc = ac.left[n];
    if (lc >= 0) {
      const int x = (int)(px % d.w), y = (int)(px / d.w);
      ImageView<typename F::ImgType, F::nChannels> view{pixels + d.off, (int)d.w, (int)d.h};
      T p[F::FeatDim];
#pragma unroll
      for (int j = 0; j < F::FeatDim; j++) p[j] = tree_feat[(size_t)n * F::FeatDim + j];
      const T v = eval_hook<F>(view, x, y, F::prepare(view, x, y), p, ac, lo);
      out = lc + ((v <= tree_thr[n]) ? 0 : 1);
    }
  }
  map_out[mo + px] = out;
}

// map[i] = 0 (the root) where the pixel is routed (labels[i] != 0 or mask[i]
// != 0; every pixel when sel is null), else -1.
__global__ __launch_bounds__(256) void k_ac_map_init(const uint8_t *__restrict__ sel, uint64_t n,
                                                     int32_t *__restrict__ map)
{
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u)
    map[i] = (sel && !sel[i]) ? -1 : 0;
}

// Forest posterior over node maps: out[c][i] (+)= post[map[i]][c] in tree
// order (first: assign), then k_ac_post_finish divides by the tree count
// (masked-out pixels: 0), the order of k_predict's sum.
__global__ __launch_bounds__(256) void k_ac_post_add(const int32_t *__restrict__ map, uint32_t npx,
                                                     const float *__restrict__ post, uint32_t nC, int first,
                                                     float *__restrict__ out)
{
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= npx) return;
  const int32_t n = map[i];
  for (uint32_t c = 0; c < nC; c++) {
    const float v = n >= 0 ? post[(size_t)n * nC + c] : 0.0f;
    out[(size_t)c * npx + i] = first ? v : out[(size_t)c * npx + i] + v;
  }
}

__global__ __launch_bounds__(256) void k_ac_post_finish(const int32_t *__restrict__ map, uint32_t npx, uint32_t nC,
                                                        float n_trees, float *__restrict__ out)
{
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= npx) return;
  const bool on = map[i] >= 0;
  for (uint32_t c = 0; c < nC; c++) out[(size_t)c * npx + i] = on ? out[(size_t)c * npx + i] / n_trees : 0.0f;
}

__global__ __launch_bounds__(256) void k_fill_i32(int32_t *__restrict__ p, uint64_t n, int32_t v)
{
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) p[i] = v;
}

// Evenly spaced subsample of every slot's records (the refinement stage of
// the split proposal): slot q's dst_count[q] records at dst_begin[q] are
// src[src_begin[q] + floor(j * src_count[q] / dst_count[q])], j < dst_count[q]
// (dst_begin has n_slots + 1 entries, the last = total); their classes are
// counted into cls[q][nC] (zeroed by the caller).
__global__ __launch_bounds__(256) void k_subsample(const uint4 *__restrict__ src, const uint32_t *__restrict__ src_begin,
                                                   const uint32_t *__restrict__ src_count,
                                                   const uint32_t *__restrict__ dst_begin,
                                                   const uint32_t *__restrict__ dst_count, uint32_t n_slots,
                                                   uint32_t total, uint32_t nC, uint4 *__restrict__ dst,
                                                   uint32_t *__restrict__ cls)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  // the slot: dst_begin[lo] <= i < dst_begin[lo + 1]
  uint32_t lo = 0, hi = n_slots;
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    if (dst_begin[mid] <= i) lo = mid;
    else hi = mid;
  }
  const uint32_t j = i - dst_begin[lo];
  const uint4 r = src[src_begin[lo] + (uint32_t)(((uint64_t)j * src_count[lo]) / dst_count[lo])];
  dst[i] = r;
  atomicAdd(&cls[(size_t)lo * nC + rec_cls(r)], 1u);
}

// Class-stratified subsample of the ranked slots (split proposal).  A
// record of class c in slot g is kept when a hash of (its image and pixel,
// the node) falls below rate[g][c] (a fraction of 2^32; 0xffffffff keeps the
// whole class), so rare classes can be kept at higher rates than common ones.
// The selected set depends only on the records, not on their order; the
// scatter keeps the node's (image, pixel) order.  Ranges: slot g's records
// are src[src_begin[g] ...] and occupy [cat_begin[g], cat_begin[g + 1]) of
// the concatenation the flags are indexed by.
__device__ __forceinline__ uint32_t strat_hash(uint32_t a, uint32_t b, uint32_t c)
{
  uint32_t h = a * 0x9e3779b1u ^ (b + 0x7f4a7c15u) * 0x85ebca77u ^ (c + 0x165667b1u) * 0xc2b2ae3du;
  h ^= h >> 16;
  h *= 0x7feb352du;
  h ^= h >> 15;
  h *= 0x846ca68bu;
  h ^= h >> 16;
  return h;
}

__device__ __forceinline__ uint32_t cat_slot(const uint32_t *__restrict__ cat_begin, uint32_t n_slots, uint32_t i)
{
  uint32_t lo = 0, hi = n_slots;
  while (hi - lo > 1u) {
    const uint32_t mid = (lo + hi) >> 1;
    if (cat_begin[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(256) void k_strat_flags(const uint4 *__restrict__ src,
                                                     const uint32_t *__restrict__ src_begin,
                                                     const uint32_t *__restrict__ cat_begin, uint32_t n_slots,
                                                     uint32_t total, uint32_t nC, const int32_t *__restrict__ node,
                                                     const uint32_t *__restrict__ rate,
                                                     unsigned long long *__restrict__ flags,
                                                     uint32_t *__restrict__ cls)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > total) return;
  if (i == total) {   // the scan's extra element: its prefix is the subsample size
    flags[i] = 0ull;
    return;
  }
  const uint32_t g = cat_slot(cat_begin, n_slots, i);
  const uint4 r = src[src_begin[g] + (i - cat_begin[g])];
  const uint32_t c = rec_cls(r);
  const uint32_t lim = rate[(size_t)g * nC + c];
  const bool keep = lim == 0xffffffffu || strat_hash(r.x & 0xffffffu, r.y, (uint32_t)node[g]) < lim;
  flags[i] = keep ? 1ull : 0ull;
  if (keep) atomicAdd(&cls[(size_t)g * nC + c], 1u);
}

__global__ __launch_bounds__(256) void k_strat_scatter(const uint4 *__restrict__ src,
                                                       const uint32_t *__restrict__ src_begin,
                                                       const uint32_t *__restrict__ cat_begin, uint32_t n_slots,
                                                       uint32_t total, const unsigned long long *__restrict__ flags,
                                                       const unsigned long long *__restrict__ pos,
                                                       uint4 *__restrict__ dst)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total || !flags[i]) return;
  const uint32_t g = cat_slot(cat_begin, n_slots, i);
  dst[pos[i]] = src[src_begin[g] + (i - cat_begin[g])];
}

// Estimated gain of every candidate of a stratified subsample over the
// whole node: class c's left count on the subsample, H[q][c][f], scaled by
// T[q][c] / S[q][c] (node over subsample class count; a class the subsample
// missed takes the subsample's overall left fraction), then the node's
// information gain in FP32.  Used only to rank candidates, never to choose a
// split: the kept candidates are histogrammed exactly on all samples.
template <int NCM>
__global__ __launch_bounds__(256) void k_est_gain(const uint32_t *__restrict__ H, uint32_t n_slots, uint32_t K,
                                                  uint32_t nC, const uint32_t *__restrict__ T,
                                                  const uint32_t *__restrict__ S, float *__restrict__ gains,
                                                  float *__restrict__ frac)
{
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint64_t)n_slots * K) return;
  const uint32_t q = (uint32_t)(i / K), f = (uint32_t)(i % K);
  const uint32_t *h = H + (size_t)q * nC * K + f;
  const uint32_t *t = T + (size_t)q * nC, *sc = S + (size_t)q * nC;
  float L[NCM];
  float hs = 0.0f, ss = 0.0f;
  for (uint32_t c = 0; c < nC; c++) {
    hs += (float)h[(size_t)c * K];
    ss += (float)sc[c];
  }
  const float fall = ss > 0.0f ? hs / ss : 0.5f;
  float nL = 0.0f, N = 0.0f;
  for (uint32_t c = 0; c < nC; c++) {
    const float tc = (float)t[c];
    L[c] = sc[c] ? (float)h[(size_t)c * K] * (tc / (float)sc[c]) : tc * fall;
    nL += L[c];
    N += tc;
  }
  const float nR = N - nL;
  float hP = 0.0f, hL = 0.0f, hR = 0.0f;
  for (uint32_t c = 0; c < nC; c++) {
    const float tc = (float)t[c], rc = tc - L[c];
    if (tc > 0.0f) hP -= (tc / N) * __log2f(tc / N);
    if (L[c] > 0.0f && nL > 0.0f) hL -= (L[c] / nL) * __log2f(L[c] / nL);
    if (rc > 0.0f && nR > 0.0f) hR -= (rc / nR) * __log2f(rc / nR);
  }
  gains[i] = N > 0.0f ? hP - (nL / N * hL + nR / N * hR) : 0.0f;
  if (frac) {
    // estimated left fraction of classes 0..7 and overall (network inputs)
    float *o = frac + i * 9;
    for (uint32_t c = 0; c < 8; c++) o[c] = (c < nC && t[c] > 0u) ? L[c] / (float)t[c] : 0.0f;
    o[8] = N > 0.0f ? nL / N : 0.0f;
  }
}

// ---------------------------------------------------------------------------
// Small unit kernels used by the parity tests of the individual steps.
// ---------------------------------------------------------------------------
template <class F>
__global__ void k_candidates(uint32_t tree, const int32_t *__restrict__ nodes, uint32_t n_nodes, uint32_t nF,
                             uint32_t nT, Bounds<F> bnd, typename F::FeatType *__restrict__ params,
                             typename F::FeatType *__restrict__ thrs)
{
  using T = typename F::FeatType;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_nodes * nF) return;
  const uint32_t nd = (uint32_t)nodes[i / nF], f = i % nF;
  T p[F::FeatDim];
  candidate_params<T, F::FeatDim>(tree, nd, f, bnd.lo, bnd.hi, p);
  for (int j = 0; j < F::FeatDim; j++) params[(size_t)i * F::FeatDim + j] = p[j];
  U4 s = {tree, nd, f, 1u};
  for (uint32_t t = 0; t < nT; t++) {
    if ((t & 3) == 0) s = md5rand(s);
    thrs[(size_t)i * nT + t] = sample_value<T>(u4_get(s, t & 3), bnd.tlo, bnd.thi);
  }
}

template <class F>
__global__ void k_feature_eval(const typename F::ImgType *__restrict__ pixels, uint32_t w, uint32_t h,
                               const int32_t *__restrict__ xy, const typename F::FeatType *__restrict__ params,
                               uint32_t n, typename F::FeatType *__restrict__ out)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  ImageView<typename F::ImgType, F::nChannels> view{pixels, (int)w, (int)h};
  out[i] = F::eval(view, xy[2 * i], xy[2 * i + 1], params + (size_t)i * F::FeatDim);
}

__global__ void k_div(const float *__restrict__ p, const float *__restrict__ d, float *__restrict__ q, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const DivPrep dp = div_prep(d[i]);
  q[i] = div_by(p[i], dp, div_fast_ok(dp));
}

__global__ void k_div_int(const float *__restrict__ p, const float *__restrict__ d, float *__restrict__ q, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  q[i] = int_div(p[i], int_div_prep(d[i]));
}

__global__ void k_count_klogk(const uint32_t *__restrict__ k, float *__restrict__ out, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = count_klogk(k[i]);
}

// Plain streaming copy (16 B per lane per step): HBM bandwidth probe and the
// reference point that scales the FETCH_SIZE / WRITE_SIZE counters.
__global__ __launch_bounds__(256) void k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n)
{
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// LDS atomic-add probe: every lane of a 512-thread block adds into its own
// column of a [64][64] u32 table, rows rotating per step, as the histogram
// kernel adds into its rank bins (one conflict-free ds_add_u32 per lane per
// step).  Measures the sustained LDS-atomic rate that bounds the histogram.
// out: gridDim.x * 512 words (the final table rows, so nothing is dead code).
__global__ __launch_bounds__(512) void k_lds_add(uint32_t iters, uint32_t *__restrict__ out)
{
  __shared__ uint32_t bins[64 * 64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (uint32_t i = threadIdx.x; i < 64u * 64u; i += blockDim.x) bins[i] = 0u;
  __syncthreads();
  uint32_t row = wave * 8u;
  for (uint32_t it = 0; it < iters; it++) {
#pragma unroll
    for (int u = 0; u < 8; u++) atomicAdd(&bins[((row + 5u * (uint32_t)u) & 63u) * 64u + lane], 1u);
    row += 3u;
  }
  __syncthreads();
  out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = bins[threadIdx.x];
}

// Texel-gather probe: every wave issues `iters` 64-lane uint16 loads whose
// lanes fall into 64 / g distinct 128-byte lines (lanes grouped g by g),
// the lines drawn at random from the first `lines` lines of `buf` (which
// must hold lines * 128 bytes).  With the window inside the vector L1 it
// times the L1-hit path, with a window of a few MiB the L1-miss (L2 fill)
// path: the two ceilings of the histogram kernel's scattered gathers.
// out: one word per thread (the sums, so no load is dead).
__device__ __forceinline__ uint32_t probe_hash(uint32_t x)
{
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

__global__ __launch_bounds__(256) void k_gather_probe(const uint16_t *__restrict__ buf, uint32_t lines, uint32_t g,
                                                      uint32_t iters, uint32_t *__restrict__ out)
{
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t grp = lane / g;
  uint32_t acc = 0;
  for (uint32_t it = 0; it < iters; it++) {
    const uint32_t line = probe_hash(wave * 7919u + it * 104729u + grp * 31u) % lines;
    acc += buf[line * 64u + ((lane * 5u + it) & 63u)];
  }
  out[blockIdx.x * blockDim.x + threadIdx.x] = acc;
}

__global__ void k_log2_det(const float *__restrict__ x, float *__restrict__ y, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = log2_det(x[i]);
}

__global__ void k_md5(const uint4 *__restrict__ in, uint4 *__restrict__ out, uint32_t n)
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint4 a = in[i];
  const U4 r = md5rand(U4{a.x, a.y, a.z, a.w});
  out[i] = make_uint4(r.x, r.y, r.z, r.w);
}

}  // namespace pd
