// Dataset ingestion on the device: the two pixel samplers of the reference
// (UniformImageSampler, src/padenti/uniform_image_sampler_impl.hpp:34-63;
// ClassWeightedImageSampler, src/padenti/classweighted_image_sampler_impl.hpp:
// 57-123), the CRC-32 of each image's bytes that seeds them, and the RGB ->
// label mapping of the labels loader (src/padenti/cv_image_loader_impl.hpp:
// 235-267).
//
// Both samplers seed a Mersenne twister MT19937 per image with
// crc32(image bytes) ^ seed and draw from it in pixel-scan order; the device
// path reproduces every draw, so the sample lists equal the reference's.
//   uniform:        labelled pixels L (label != 0) in scan order; n_samples
//                   times r = uniform_int(0, |L|-1) (Boost's rejection form:
//                   bucket = floor(2^32 / |L|), accept x / bucket <= |L| - 1),
//                   sample L[r]; sort ascending (duplicates kept).
//   class-weighted: bucket size B_c = ceilf(w_c * (float)n_samples); per
//                   labelled pixel i of class c with class ordinal k: k < B_c
//                   fills slot k; otherwise one draw u = x * 2^-32 (double)
//                   and j = roundf((float)(u * k)), slot j <- i when j < B_c;
//                   output the filled slots of every class, sorted.
// The reservoir's last-writer-wins rule becomes a max over pixel indices,
// which is what makes the scan parallel: the draw index of a pixel is the
// number of earlier labelled pixels whose class ordinal is past its bucket.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pd {
namespace ingest {

// ---- CRC-32 (ISO-HDLC: reflected polynomial 0x04C11DB7, init and final xor
// 0xFFFFFFFF; the check value of "123456789" is 0xCBF43926).  Polynomials are
// held bit-reflected: bit 31 is the coefficient of x^0.
constexpr uint32_t CRC_POLY = 0xEDB88320u;
constexpr uint32_t CRC_ONE = 0x80000000u;  // the polynomial 1

// a * b mod P
__host__ __device__ constexpr uint32_t gf2_mul(uint32_t a, uint32_t b)
{
  uint32_t p = 0;
  for (int i = 0; i < 32; i++) {
    p ^= b & (0u - ((a >> (31 - i)) & 1u));
    b = (b >> 1) ^ (CRC_POLY & (0u - (b & 1u)));  // b *= x
  }
  return p;
}

struct CrcTables {
  uint32_t t[4][256];  // t[0]: one byte; t[s]: a byte followed by s zero bytes
  uint32_t x2k[72];    // x^(2^k) mod P
  uint32_t w64[64];    // x^(8 * 64 * j) mod P: j segments of 64 bytes
};

constexpr CrcTables make_crc_tables()
{
  CrcTables T{};
  for (uint32_t i = 0; i < 256; i++) {
    uint32_t c = i;
    for (int k = 0; k < 8; k++) c = (c >> 1) ^ (CRC_POLY & (0u - (c & 1u)));
    T.t[0][i] = c;
  }
  for (int s = 1; s < 4; s++)
    for (uint32_t i = 0; i < 256; i++) T.t[s][i] = (T.t[s - 1][i] >> 8) ^ T.t[0][T.t[s - 1][i] & 0xFFu];
  T.x2k[0] = CRC_ONE >> 1;  // x
  for (int k = 1; k < 72; k++) T.x2k[k] = gf2_mul(T.x2k[k - 1], T.x2k[k - 1]);
  T.w64[0] = CRC_ONE;
  for (int j = 1; j < 64; j++) T.w64[j] = gf2_mul(T.w64[j - 1], T.x2k[9]);  // * x^512
  return T;
}

__constant__ const CrcTables c_crc = make_crc_tables();

// x^(8n) mod P: the effect of n zero bytes on a CRC register
__host__ __device__ inline uint32_t crc_x8n(const CrcTables &T, uint64_t n)
{
  uint32_t r = CRC_ONE;
  for (int k = 3; n; n >>= 1, k++)
    if (n & 1u) r = gf2_mul(r, T.x2k[k]);
  return r;
}

// register form with zero initial value ("pure" CRC), four bytes at once
__device__ __forceinline__ uint32_t crc_word(const uint32_t (*T)[256], uint32_t crc, uint32_t w)
{
  crc ^= w;
  return T[3][crc & 0xFFu] ^ T[2][(crc >> 8) & 0xFFu] ^ T[1][(crc >> 16) & 0xFFu] ^ T[0][crc >> 24];
}

__device__ __forceinline__ uint32_t crc_byte(const uint32_t (*T)[256], uint32_t crc, uint32_t b)
{
  return T[0][(crc ^ b) & 0xFFu] ^ (crc >> 8);
}

// One image's byte range [start, end) (absolute addresses) cut into 4 KiB
// blocks from a0 = start & ~63; block m covers [a0 + 4096 m, a0 + 4096 (m+1)).
// A wave hashes a chunk of up to CRC_CHUNK consecutive blocks.
constexpr uint32_t CRC_CHUNK = 8;
constexpr uint32_t CRC_GAP = 4096 - 64;  // bytes between a lane's segments in consecutive blocks

struct CrcJob {
  uint64_t start, end, a0;
  uint32_t first_chunk, n_blocks;
};

// Largest i < n with first[i] <= v (first ascending, first[0] = 0).
__device__ __forceinline__ uint32_t find_owner(const uint32_t *__restrict__ first, uint32_t n, uint32_t v)
{
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (first[mid] <= v) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint32_t crc_seg(const uint32_t (*T)[256], uint32_t crc, const uint4 (&v)[4])
{
#pragma unroll
  for (int q = 0; q < 4; q++) {
    crc = crc_word(T, crc, v[q].x);
    crc = crc_word(T, crc, v[q].y);
    crc = crc_word(T, crc, v[q].z);
    crc = crc_word(T, crc, v[q].w);
  }
  return crc;
}

// a * x^(8 CRC_GAP) mod P from G[k][v] = (v at byte k) * x^(8 CRC_GAP)
__device__ __forceinline__ uint32_t mul_gap(const uint32_t (*G)[256], uint32_t a)
{
  return G[0][a & 0xFFu] ^ G[1][(a >> 8) & 0xFFu] ^ G[2][(a >> 16) & 0xFFu] ^ G[3][a >> 24];
}

// Wave per chunk, lane per 64-byte segment of every block (four 16-byte
// loads, the next block's prefetched while the current one is hashed).  A
// lane carries one register across the chunk's whole blocks: before each
// new segment it is shifted over the 4032 bytes of the other lanes (table
// multiply).  At the end of the whole blocks the lane registers are shifted
// to the block end (x^(8 * 64 * j)), xor-reduced, and shifted by
// P[n_blocks - 1 - e] = x^(8 * 4096 (n_blocks - 1 - e)) (e = the chunk's end
// block) into acc_a; the image's last block (lanes whose segment ends in the
// image, then the tail bytes) goes to acc_b.  k_crc_final applies the last
// block's length.  xor is order free, so the result is deterministic.
__global__ __launch_bounds__(256) void k_crc32(const CrcJob *__restrict__ jobs, const uint32_t *__restrict__ chunk0,
                                               uint32_t n_images, uint32_t n_chunks, const uint32_t *__restrict__ P,
                                               const uint32_t *__restrict__ gap, uint32_t *acc_a, uint32_t *acc_b)
{
  __shared__ uint32_t T[4][256], G[4][256];
  for (uint32_t i = threadIdx.x; i < 1024; i += 256) {
    T[i >> 8][i & 255] = c_crc.t[i >> 8][i & 255];
    G[i >> 8][i & 255] = gap[i];
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t ch = blockIdx.x * 4u + (threadIdx.x >> 6); ch < n_chunks; ch += gridDim.x * 4u) {
    const uint32_t im = find_owner(chunk0, n_images, ch);
    const CrcJob J = jobs[im];
    const uint32_t m0 = (ch - J.first_chunk) * CRC_CHUNK;
    const uint32_t m1 = (m0 + CRC_CHUNK < J.n_blocks) ? m0 + CRC_CHUNK : J.n_blocks;
    const bool has_last = (m1 == J.n_blocks);
    const uint32_t mf = has_last ? J.n_blocks - 1u : m1;  // whole blocks [m0, mf)
    const bool head = (J.start > J.a0) && lane == 0;        // lane 0 of block 0 starts inside its segment
    if (m0 < mf) {
      uint4 v[4] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
      if (!(m0 == 0 && head)) {
        const uint4 *p = reinterpret_cast<const uint4 *>(J.a0 + (uint64_t)m0 * 4096u + 64ull * lane);
        v[0] = p[0]; v[1] = p[1]; v[2] = p[2]; v[3] = p[3];
      }
      uint32_t reg = 0;
      for (uint32_t m = m0; m < mf; m++) {
        const uint4 cur[4] = {v[0], v[1], v[2], v[3]};
        if (m + 1u < mf) {
          const uint4 *p = reinterpret_cast<const uint4 *>(J.a0 + (uint64_t)(m + 1u) * 4096u + 64ull * lane);
          v[0] = p[0]; v[1] = p[1]; v[2] = p[2]; v[3] = p[3];
        }
        if (m > m0) reg = mul_gap(G, reg);
        if (m == 0 && head) {
          for (uint64_t a = J.start; a < J.a0 + 64u; a++) reg = crc_byte(T, reg, *reinterpret_cast<const uint8_t *>(a));
        } else {
          reg = crc_seg(T, reg, cur);
        }
      }
      reg = gf2_mul(reg, c_crc.w64[63u - lane]);
      for (int o = 32; o >= 1; o >>= 1) reg ^= __shfl_xor(reg, o);
      if (lane == 0) atomicXor(&acc_a[im], gf2_mul(reg, P[J.n_blocks - 1u - mf]));
    }
    if (has_last) {
      const uint32_t m = J.n_blocks - 1u;
      const uint64_t blo = J.a0 + (uint64_t)m * 4096u;
      const uint32_t L = (uint32_t)((J.end - blo) >> 6);  // lanes whose segment ends in the image
      uint32_t crc = 0;
      if (lane < L) {
        const uint64_t lo = blo + 64ull * lane;
        if (lo >= J.start) {
          const uint4 *p = reinterpret_cast<const uint4 *>(lo);
          const uint4 w[4] = {p[0], p[1], p[2], p[3]};
          crc = crc_seg(T, crc, w);
        } else {  // the image's first segment starts inside it
          for (uint64_t a = J.start; a < lo + 64u; a++) crc = crc_byte(T, crc, *reinterpret_cast<const uint8_t *>(a));
        }
        crc = gf2_mul(crc, c_crc.w64[L - 1u - lane]);
      }
      for (int o = 32; o >= 1; o >>= 1) crc ^= __shfl_xor(crc, o);
      const uint64_t t0 = blo + 64ull * L;
      for (uint64_t a = (t0 > J.start ? t0 : J.start); a < J.end; a++)
        crc = crc_byte(T, crc, *reinterpret_cast<const uint8_t *>(a));
      if (lane == 0) atomicXor(&acc_b[im], crc);
    }
  }
}

// crc32 = pure ^ (0xFFFFFFFF * x^(8 len)) ^ 0xFFFFFFFF, pure = acc_a * x^(8 q) ^ acc_b
// with q the length of the last block from a0 (at most 4096).
__device__ __forceinline__ uint32_t crc_join(const CrcJob &J, uint32_t a, uint32_t b, uint32_t xq, uint32_t xlen)
{
  const uint32_t pure = J.n_blocks ? gf2_mul(a, xq) ^ b : 0u;
  return pure ^ gf2_mul(0xFFFFFFFFu, xlen) ^ 0xFFFFFFFFu;
}
__device__ __forceinline__ uint64_t crc_tail(const CrcJob &J)
{
  return J.n_blocks ? J.end - J.a0 - 4096ull * (J.n_blocks - 1u) : 0ull;
}

// Up to CRC_WAVES images: one wave per image, lane k < 16 holding the factor of
// bit k of q, lane 16 + k that of bit k of len (below 2^44), multiplied in a tree
// (a thread walking the bits: 11.5 us for 150 images, the wave 8.2).  A wave does
// all 1300 operations of the tree whatever the bits, so beyond a wave a SIMD the
// images add up (5000 of them 20 us, 100000 0.4 ms) and a thread an image is the
// faster form again (7 us, and 1.16 instead of 1.56 ms for the whole CRC of 100000
// images of 3000 bytes).  The grids are bounded; they go on by their size.
constexpr uint32_t CRC_WAVES = 1024;
__global__ __launch_bounds__(256) void k_crc_final_wave(const CrcJob *__restrict__ jobs, uint32_t n_images,
                                                        const uint32_t *__restrict__ acc_a,
                                                        const uint32_t *__restrict__ acc_b, uint32_t *crc_out)
{
  const uint32_t lane = threadIdx.x & 63u;
  for (uint64_t i = blockIdx.x * 4u + (threadIdx.x >> 6); i < n_images; i += gridDim.x * 4u) {
    const CrcJob J = jobs[i];
    const uint64_t n = lane < 16u ? crc_tail(J) : J.end - J.start;
    const uint32_t bit = lane < 16u ? lane : lane - 16u;
    uint32_t f = (n >> bit) & 1u ? c_crc.x2k[bit + 3u] : CRC_ONE;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) f = gf2_mul(f, __shfl_xor(f, o));
    const uint32_t a = gf2_mul(f, __shfl_xor(f, 16));   // lanes 32..: bits 16..47 of len
    const uint32_t l = gf2_mul(__shfl(a, 32), __shfl(f, 16));
    const uint32_t fq = __shfl(f, 0);
    if (lane == 0u) crc_out[i] = crc_join(J, acc_a[i], acc_b[i], fq, l);
  }
}
__global__ __launch_bounds__(64) void k_crc_final(const CrcJob *__restrict__ jobs, uint32_t n_images,
                                                  const uint32_t *__restrict__ acc_a,
                                                  const uint32_t *__restrict__ acc_b, uint32_t *crc_out)
{
  for (uint64_t i = blockIdx.x * 64u + threadIdx.x; i < n_images; i += gridDim.x * 64u) {
    const CrcJob J = jobs[i];
    crc_out[i] = crc_join(J, acc_a[i], acc_b[i], crc_x8n(c_crc, crc_tail(J)), crc_x8n(c_crc, J.end - J.start));
  }
}

// ---- MT19937 (Matsumoto & Nishimura 1998), 256 threads share one state ----
constexpr uint32_t MT_N = 624, MT_M = 397;

__device__ __forceinline__ uint32_t mt_mix(uint32_t u, uint32_t v)
{
  const uint32_t y = (u & 0x80000000u) | (v & 0x7FFFFFFFu);
  return (y >> 1) ^ (0x9908B0DFu & (0u - (y & 1u)));
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
  y ^= y >> 11;
  y ^= (y << 7) & 0x9D2C5680u;
  y ^= (y << 15) & 0xEFC60000u;
  return y ^ (y >> 18);
}

// init_genrand(s): one thread (the recurrence is serial)
__device__ inline void mt_seed(uint32_t *mt, uint32_t s)
{
  mt[0] = s;
  for (uint32_t i = 1; i < MT_N; i++) {
    s = 1812433253u * (s ^ (s >> 30)) + i;
    mt[i] = s;
  }
}

// One twist of the whole state by the block (>= 256 threads, every thread
// calls it), then the 624 tempered outputs into out[0..623].  The serial
// recurrence new[i] = new/old[i+397 mod 624] ^ mix(old[i], old/new[i+1]) runs
// in three dependent ranges: [0,227) reads old words only, [227,454) and
// [454,624) read new[i-227] of the range before (i = 623 reads new[0]).
__device__ inline void mt_twist(uint32_t *mt, uint32_t *out, uint32_t tid)
{
  uint32_t a1 = 0, a2 = 0, a3 = 0, last_old = 0;
  if (tid < 227) {
    a1 = mt[tid + MT_M] ^ mt_mix(mt[tid], mt[tid + 1]);
    a2 = mt_mix(mt[227 + tid], mt[228 + tid]);
  }
  if (tid < 169) a3 = mt_mix(mt[454 + tid], mt[455 + tid]);
  if (tid == 169) last_old = mt[623];
  __syncthreads();
  if (tid < 227) mt[tid] = a1;
  __syncthreads();
  if (tid < 227) mt[227 + tid] = mt[tid] ^ a2;
  __syncthreads();
  if (tid < 169) mt[454 + tid] = mt[227 + tid] ^ a3;
  if (tid == 169) mt[623] = mt[396] ^ mt_mix(last_old, mt[0]);
  __syncthreads();
  for (uint32_t i = tid; i < MT_N; i += blockDim.x) out[i] = mt_temper(mt[i]);
  __syncthreads();
}

// ---- labelled-pixel rank index (uniform sampler) --------------------------
struct SampleJob {
  uint64_t lab_off;   // byte offset of the image's labels (16-byte aligned)
  uint32_t n_px;      // width * height
  uint32_t word0;     // first 32-pixel word of the image in the bitmask
  uint32_t out_base;  // first output slot of the image (image * capacity)
  uint32_t pad;
};

__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t *ws, uint32_t &total)
{
  // 256 threads: inclusive wave scan, wave totals in ws[0..3]
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t s = v;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(s, o);
    if (lane >= (uint32_t)o) s += t;
  }
  if (lane == 63) ws[wave] = s;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for (uint32_t w = 0; w < 4; w++) {
    const uint32_t x = ws[w];
    if (w < wave) before += x;
    total += x;
  }
  __syncthreads();
  return before + s - v;
}

// bits[word0 + w] = labelled-pixel mask of pixels [32 w, 32 w + 32); pre = the
// labelled pixels before it in its tile; tile_cnt = the tile's labelled pixels.
// A block per tile of 256 words of one image; tile0[i] = first tile of image i
// (binary search, n_images entries).
__global__ __launch_bounds__(256) void k_label_bits(const uint8_t *__restrict__ labels,
                                                    const SampleJob *__restrict__ jobs,
                                                    const uint32_t *__restrict__ tile0, uint32_t n_images,
                                                    uint32_t *bits, uint16_t *pre, uint32_t *tile_cnt)
{
  __shared__ uint32_t s_im, ws[4];
  if (threadIdx.x == 0) s_im = find_owner(tile0, n_images, blockIdx.x);
  __syncthreads();
  const uint32_t im = s_im;
  const SampleJob J = jobs[im];
  const uint32_t w = (blockIdx.x - tile0[im]) * 256u + threadIdx.x;
  const uint8_t *lab = labels + J.lab_off + 32ull * w;
  uint32_t m = 0;
  if (32ull * w + 32u <= J.n_px) {
    const uint4 a = reinterpret_cast<const uint4 *>(lab)[0], b = reinterpret_cast<const uint4 *>(lab)[1];
    const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) m |= (((v[k] >> (8 * j)) & 0xFFu) != 0u ? 1u : 0u) << (4 * k + j);
  } else {
    for (uint32_t j = 0; 32ull * w + j < J.n_px; j++) m |= (lab[j] != 0u ? 1u : 0u) << j;
  }
  uint32_t total;
  const uint32_t before = block_excl_scan(__popc(m), ws, total);
  if (32ull * w < J.n_px) {
    bits[J.word0 + w] = m;
    pre[J.word0 + w] = (uint16_t)before;
  }
  if (threadIdx.x == 0) tile_cnt[blockIdx.x] = total;
}

constexpr uint32_t COARSE = 1024;   // entries of the tile prefix kept in LDS

// Rank index of one image: labelled pixels before its tiles (tile, in LDS every
// `stride` tiles: coarse), before a word in its tile (pre), and the words.
struct RankIndex {
  const uint32_t *bits, *tile;
  const uint16_t *pre;
  const uint32_t *coarse;
  uint32_t n_words, n_tiles, n_coarse, stride;
};

// Pixels of NR labelled ranks, searched in step (the chains of dependent loads
// overlap): largest tile, then word, with a prefix <= r, then the bit.
template <int NR>
__device__ __forceinline__ void select_ranks(const RankIndex &ix, const uint32_t (&r)[NR], uint32_t (&px)[NR])
{
  uint32_t lo[NR], hi[NR], rem[NR];
#pragma unroll
  for (int k = 0; k < NR; k++) lo[k] = 0u, hi[k] = ix.n_coarse;
  for (uint32_t span = ix.n_coarse; span > 1u; span = (span + 1u) >> 1)
#pragma unroll
    for (int k = 0; k < NR; k++) {
      const uint32_t mid = (lo[k] + hi[k]) >> 1;   // (lo once the range is one entry)
      if (ix.coarse[mid] <= r[k]) lo[k] = mid;
      else hi[k] = mid;
    }
#pragma unroll
  for (int k = 0; k < NR; k++) {
    lo[k] *= ix.stride;
    hi[k] = lo[k] + ix.stride < ix.n_tiles ? lo[k] + ix.stride : ix.n_tiles;
  }
  for (uint32_t span = ix.stride; span > 1u; span = (span + 1u) >> 1)
#pragma unroll
    for (int k = 0; k < NR; k++) {
      const uint32_t mid = (lo[k] + hi[k]) >> 1;
      if (ix.tile[mid] <= r[k]) lo[k] = mid;
      else hi[k] = mid;
    }
#pragma unroll
  for (int k = 0; k < NR; k++) {
    rem[k] = r[k] - (ix.stride == 1u ? ix.coarse[lo[k]] : ix.tile[lo[k]]);
    lo[k] *= 256u;
    hi[k] = lo[k] + 256u < ix.n_words ? lo[k] + 256u : ix.n_words;
  }
#pragma unroll 1
  for (int step = 0; step < 8; step++)
#pragma unroll
    for (int k = 0; k < NR; k++) {
      const uint32_t mid = (lo[k] + hi[k]) >> 1;
      if (ix.pre[mid] <= rem[k]) lo[k] = mid;
      else hi[k] = mid;
    }
#pragma unroll
  for (int k = 0; k < NR; k++) {
    uint32_t b = ix.bits[lo[k]], n = rem[k] - ix.pre[lo[k]], at = 0;   // the n-th set bit
#pragma unroll
    for (uint32_t h = 16; h; h >>= 1) {
      const uint32_t c = __popc(b & ((1u << h) - 1u));
      if (n >= c) {
        n -= c;
        b >>= h;
        at += h;
      }
    }
    px[k] = 32u * lo[k] + at;
  }
}

// One block of 256 threads per image.  tile_pre: the tiles' counts in, their
// exclusive prefix within the image out.  Writes the unsorted samples and the
// segment end for the sort.  Bound by latency: the seeding of the state (624
// dependent steps), a twist per 624 draws and the rank searches.  400 images of
// 640 x 480, 2000 samples: 73 us with one search at a time over a prefix of the
// whole batch (and a 28 us scan for it), now 43 us without the scan.
__global__ __launch_bounds__(256) void k_sample_uniform(const SampleJob *__restrict__ jobs,
                                                        const uint32_t *__restrict__ tile0, uint32_t n_images,
                                                        uint32_t n_tiles, const uint32_t *__restrict__ bits,
                                                        const uint16_t *__restrict__ pre, uint32_t *tile_pre,
                                                        const uint32_t *__restrict__ crc, uint32_t seed,
                                                        uint32_t n_samples, uint32_t *out, uint32_t *n_out,
                                                        uint32_t *seg_end)
{
  __shared__ uint32_t mt[MT_N], y[MT_N], ws[4], coarse[COARSE];
  const uint32_t im = blockIdx.x, tid = threadIdx.x;
  const SampleJob J = jobs[im];
  const uint32_t t0 = tile0[im], nt = (im + 1u < n_images ? tile0[im + 1u] : n_tiles) - t0;
  RankIndex ix{bits + J.word0, tile_pre + t0, pre + J.word0, coarse, (J.n_px + 31u) >> 5, nt, 0u, 1u};
  while ((nt + ix.stride - 1u) / ix.stride > COARSE) ix.stride *= 2u;
  ix.n_coarse = (nt + ix.stride - 1u) / ix.stride;
  uint32_t n_lab = 0;
  for (uint32_t b = 0; b < nt; b += 256u) {
    const uint32_t t = b + tid, v = t < nt ? tile_pre[t0 + t] : 0u;
    uint32_t total;
    const uint32_t before = n_lab + block_excl_scan(v, ws, total);
    if (t < nt) {
      if (ix.stride > 1u) tile_pre[t0 + t] = before;
      if (t % ix.stride == 0u) coarse[t / ix.stride] = before;
    }
    n_lab += total;
  }
  uint32_t *o = out + J.out_base;
  if (n_lab == 0u) {  // no labelled pixel: no sample (the reference's range would be empty)
    if (tid == 0) { n_out[im] = 0; seg_end[im] = J.out_base; }
    return;
  }
  __syncthreads();
  if (n_lab == 1u) {  // uniform_int over one value draws nothing
    const uint32_t r[1] = {0u};
    uint32_t px[1];
    select_ranks(ix, r, px);
    for (uint32_t s = tid; s < n_samples; s += 256u) o[s] = px[0];
    if (tid == 0) { n_out[im] = n_samples; seg_end[im] = J.out_base + n_samples; }
    return;
  }
  const uint32_t range = n_lab - 1u;
  const uint32_t bucket = (uint32_t)(0x100000000ull / n_lab);
  if (tid == 0) mt_seed(mt, crc[im] ^ seed);
  __syncthreads();
  uint32_t filled = 0;
  while (filled < n_samples) {
    mt_twist(mt, y, tid);
    uint32_t r[3], q[3], px[3], acc = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const uint32_t i = 3u * tid + k;
      r[k] = (i < MT_N) ? y[i] / bucket : 0xFFFFFFFFu;
      q[k] = r[k] <= range ? r[k] : 0u;
      acc += (r[k] <= range) ? 1u : 0u;
    }
    uint32_t total;
    uint32_t slot = filled + block_excl_scan(acc, ws, total);
    select_ranks(ix, q, px);
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (r[k] <= range) {
        if (slot < n_samples) o[slot] = px[k];
        slot++;
      }
    filled += total;
  }
  if (tid == 0) { n_out[im] = n_samples; seg_end[im] = J.out_base + n_samples; }
}

// ---- class-weighted reservoir --------------------------------------------
// The serial loop walks the pixels in scan order: pixel p of class c with class
// ordinal k goes to slot k while k < B_c, afterwards it draws from the image's
// MT19937 stream and may replace a slot.  Neither the ordinals nor the draw
// indices depend on what was drawn, so the loop is three parallel steps:
//   k_weighted_count  class counts of every segment (seg_len pixels, one wave
//                     each) and, in its first blocks, the tempered outputs of
//                     every image's stream;
//   k_weighted_scan   per image: class ordinals and draw index at the start of
//                     every segment;
//   k_weighted_draw   the segments' pixels, one wave a segment.
// Only the stream is serial (454 words a step, below).  150 images of 321 x 243,
// 16 classes: 846 us with one wave an image walking all of it, 102 us now.  The
// labels are read and ranked twice, so a batch that keeps a wave on every SIMD for
// as long as its largest image takes (1024 images of one size) keeps the walk,
// k_sample_weighted (images of 640 x 480, walk
// -> segments: 250 images 2.75 -> 0.70 ms, 500 2.81 -> 1.23, 1000 2.82 -> 2.71; 5000
// 4.3 -> 8.8).
//
// The streams are generated for draws [w0, w0 + win) of every image of a group
// at a time (win * n_images words of scratch, which bounds the group); an image
// larger than the scratch takes several windows, and a segment's draws may lie in
// two of them and more.
constexpr uint32_t MT_LAG = MT_N - MT_M;     // 227
constexpr uint32_t MT_STEP = 2 * MT_LAG;     // words a step computes from the last 624

// Ordering inside one wave: LDS operations of a wave execute in issue order,
// so a fence + wave barrier is all the synchronisation lanes of one wave need.
__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of the block is in order for its waves (no wait for global memory)
__device__ __forceinline__ void lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Ordinals of the wave's 64 labels: calls f(class, mask of its lanes) for every
// distinct class of the lanes with l != 0.
template <class Fn>
__device__ __forceinline__ void each_class(uint32_t l, const Fn &f)
{
  uint64_t pending = __ballot(l != 0u);
  while (pending) {
    const uint32_t lead = (uint32_t)__builtin_ctzll(pending);
    const uint32_t cl = __builtin_amdgcn_readlane(l, lead);
    const uint64_t mm = __ballot(l == cl);
    f(cl - 1u, mm);
    pending &= ~mm;
  }
}

// Blocks [0, n_images): the stream of image blockIdx.x, draws [w0, w0 + win)
// into draws[image * win ..] (images and seg0 are a group's, segments [seg_base,
// seg_end)); `state` carries the last 624 words to the next
// window.  The other blocks (w0 = 0 only): class counts of four segments.
// Labels above n_classes set *bad and count as unlabelled.
//
// x[k + 624] = x[k + 397] ^ mix(x[k], x[k + 1]): thread i computes words k + 624
// + i and k + 851 + i of a step of 454; the x[k + 397] of each is the word it
// computed before, so only old words come from LDS, a ring of 2048 (a step writes
// words k + 624 .. k + 1077 and reads k .. k + 454; its barrier keeps later writes
// to their slots behind the reads).  Bound by a step's latency: 227 words a step
// and x[k + 397] from LDS took the kernel 72 us for 78003 draws an image, this
// one 56 us.
__global__ __launch_bounds__(256) void k_weighted_count(const uint8_t *__restrict__ labels,
                                                        const SampleJob *__restrict__ jobs, uint32_t n_images,
                                                        const uint32_t *__restrict__ seg0, uint32_t seg_base,
                                                        uint32_t seg_end,
                                                        uint32_t seg_len, const uint32_t *__restrict__ crc,
                                                        uint32_t seed, uint32_t n_classes, uint32_t w0, uint32_t win,
                                                        uint32_t *__restrict__ draws, uint32_t *__restrict__ state,
                                                        uint32_t *__restrict__ counts, uint32_t *bad)
{
  __shared__ uint32_t sh[2048];
  const uint32_t tid = threadIdx.x;
  if (blockIdx.x < n_images) {
    const uint32_t im = blockIdx.x, n_px = jobs[im].n_px;
    if (n_px <= w0) return;
    if (w0 == 0u) {
      if (tid == 0) mt_seed(sh, crc[im] ^ seed);
    } else {
      for (uint32_t i = tid; i < MT_N; i += 256u) sh[i] = state[(size_t)im * MT_N + i];
    }
    lds_sync();
    const uint32_t n = n_px - w0 < win ? n_px - w0 : win;   // (an image draws at most once a pixel)
    uint32_t *o = draws + (size_t)im * win;
    uint32_t k = 0, x = tid < MT_LAG ? sh[MT_M + tid] : 0u;
    for (; k < n; k += MT_STEP) {
      if (tid < MT_LAG) {
        const uint32_t i = k + tid;
        const uint32_t m0 = mt_mix(sh[i & 2047u], sh[(i + 1u) & 2047u]);
        const uint32_t m1 = mt_mix(sh[(i + MT_LAG) & 2047u], sh[(i + MT_LAG + 1u) & 2047u]);
        const uint32_t y = x ^ m0;
        x = y ^ m1;
        sh[(i + MT_N) & 2047u] = y;
        sh[(i + MT_N + MT_LAG) & 2047u] = x;
        if (i < n) o[i] = mt_temper(y);
        if (i + MT_LAG < n) o[i + MT_LAG] = mt_temper(x);
      }
      lds_sync();
    }
    if (n_px - w0 > win)   // (win is a multiple of MT_STEP)
      for (uint32_t i = tid; i < MT_N; i += 256u) state[(size_t)im * MT_N + i] = sh[(k + i) & 2047u];
    return;
  }
  const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t seg = seg_base + (blockIdx.x - n_images) * 4u + wave;
  if (seg >= seg_end) return;
  uint32_t *cnt = sh + 256u * wave;
  for (uint32_t c = lane; c < 256u; c += 64u) cnt[c] = 0;
  wave_sync();
  const uint32_t im = find_owner(seg0, n_images, seg);
  const SampleJob J = jobs[im];
  const uint8_t *lab = labels + J.lab_off;
  const uint32_t p0 = (seg - seg0[im]) * seg_len, p1 = J.n_px - p0 < seg_len ? J.n_px : p0 + seg_len;
  for (uint32_t t = p0; t < p1; t += 1024u) {
    uint32_t cur[16];
#pragma unroll
    for (uint32_t s = 0; s < 16u; s++) cur[s] = t + 64u * s + lane < p1 ? lab[t + 64u * s + lane] : 0u;
#pragma unroll
    for (uint32_t s = 0; s < 16u; s++) {
      if (t + 64u * s >= p1) break;
      uint32_t l = cur[s];
      if (l > n_classes) {
        atomicOr(bad, 1u);
        l = 0;
      }
      each_class(l, [&](uint32_t c, uint64_t mm) {
        if (lane == 0) cnt[c] += (uint32_t)__popcll(mm);
      });
    }
  }
  wave_sync();
  for (uint32_t c = lane; c < n_classes; c += 64u) counts[(size_t)seg * n_classes + c] = cnt[c];
}

// One block of 1024 threads per image.  counts[seg][c]: class counts of a
// segment in, class ordinal at its start out; seg_draw[seg] = (draw index at its
// start, number of draws); class_count[image][c] the totals.
__global__ __launch_bounds__(1024) void k_weighted_scan(const uint32_t *__restrict__ seg0, uint32_t n_images,
                                                        uint32_t seg_end, uint32_t n_classes,
                                                        const uint32_t *__restrict__ B, uint32_t *counts,
                                                        uint2 *__restrict__ seg_draw,
                                                        uint32_t *__restrict__ class_count)
{
  __shared__ uint32_t sB[256], tot[256], ws[16];
  const uint32_t im = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t s0 = seg0[im], ns = (im + 1u < n_images ? seg0[im + 1u] : seg_end) - s0;
  uint32_t *ct = counts + (size_t)s0 * n_classes;
  if (tid < n_classes) sB[tid] = B[tid];
  for (uint32_t c = wave; c < n_classes; c += 16u) {
    uint32_t run = 0;
    for (uint32_t s = 0; s < ns; s += 64u) {
      const uint32_t v = s + lane < ns ? ct[(size_t)(s + lane) * n_classes + c] : 0u;
      uint32_t x = v;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(x, o);
        if (lane >= (uint32_t)o) x += t;
      }
      if (s + lane < ns) ct[(size_t)(s + lane) * n_classes + c] = run + x - v;
      run += __shfl(x, 63);
    }
    if (lane == 0) {
      tot[c] = run;
      class_count[(size_t)im * n_classes + c] = run;
    }
  }
  __syncthreads();
  uint32_t carry = 0;
  for (uint32_t s1 = 0; s1 < ns; s1 += 1024u) {
    const uint32_t s = s1 + tid;
    uint32_t d = 0;
    if (s < ns)
      for (uint32_t c = 0; c < n_classes; c++) {
        const uint32_t st = ct[(size_t)s * n_classes + c];
        const uint32_t en = s + 1u < ns ? ct[(size_t)(s + 1u) * n_classes + c] : tot[c];
        const uint32_t from = st > sB[c] ? st : sB[c];
        d += en > from ? en - from : 0u;
      }
    uint32_t x = d;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += t;
    }
    if (lane == 63u) ws[wave] = x;
    __syncthreads();
    uint32_t before = carry;
    for (uint32_t w = 0; w < 16u; w++) {
      const uint32_t t = ws[w];
      if (w < wave) before += t;
      carry += t;
    }
    if (s < ns) seg_draw[s0 + s] = uint2{before + x - d, d};
    __syncthreads();
  }
}

// One wave per segment, 64 pixels per step in scan order.  A pixel's class
// ordinal is the count so far (LDS, from the segment's start) plus its rank
// among the wave's lanes of that class; it draws iff the ordinal is at least
// B_c, and its draw index is the wave prefix of those flags.  bucket:
// zero-initialised slots [image][sum B] (class c at boff[c]) filled with
// atomicMax (the last writer in scan order has the largest pixel index).  Draws
// outside the window [w0, w0 + win) are another launch's; pixels that do not
// draw belong to the first one's.  Bound by VALU issue (about 90 operations a
// step).
__global__ __launch_bounds__(256) void k_weighted_draw(const uint8_t *__restrict__ labels,
                                                       const SampleJob *__restrict__ jobs, uint32_t n_images,
                                                       const uint32_t *__restrict__ seg0, uint32_t seg_base,
                                                       uint32_t seg_end, uint32_t seg_len, uint32_t n_classes,
                                                       const uint32_t *__restrict__ B,
                                                       const uint32_t *__restrict__ boff, uint32_t w0, uint32_t win,
                                                       const uint32_t *__restrict__ draws,
                                                       const uint32_t *__restrict__ counts,
                                                       const uint2 *__restrict__ seg_draw, uint32_t *bucket)
{
  __shared__ uint32_t sB[256], sO[256], cnt_all[4][256];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  sB[tid] = tid < n_classes ? B[tid] : 0u;
  sO[tid] = tid < n_classes ? boff[tid] : 0u;
  __syncthreads();  // the only block-wide barrier: from here on the waves are independent
  const uint32_t seg = seg_base + blockIdx.x * 4u + wave;
  if (seg >= seg_end) return;
  const uint2 sd = seg_draw[seg];
  // no draw of the segment is in the window: it ends before it or begins behind it
  // (one that begins before it and ends inside draws its last ones here)
  if (w0 != 0u && (sd.x + sd.y <= w0 || (sd.x >= w0 && sd.x - w0 >= win))) return;
  uint32_t *cnt = cnt_all[wave];
  for (uint32_t c = lane; c < n_classes; c += 64u) cnt[c] = counts[(size_t)seg * n_classes + c];
  const uint32_t im = find_owner(seg0, n_images, seg);
  const SampleJob J = jobs[im];
  const uint8_t *lab = labels + J.lab_off;
  const uint32_t *x = draws + (size_t)im * win;
  uint32_t *bk = bucket + J.out_base;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64u - lane));
  const uint32_t p0 = (seg - seg0[im]) * seg_len, p1 = J.n_px - p0 < seg_len ? J.n_px : p0 + seg_len;
  uint32_t D = sd.x;
  wave_sync();
  for (uint32_t t = p0; t < p1; t += 1024u) {
    uint32_t cur[16];
#pragma unroll
    for (uint32_t s = 0; s < 16u; s++) cur[s] = t + 64u * s + lane < p1 ? lab[t + 64u * s + lane] : 0u;
#pragma unroll
    for (uint32_t s = 0; s < 16u; s++) {
      if (t + 64u * s >= p1) break;
      const uint32_t p = t + 64u * s + lane;
      const uint32_t l = cur[s] <= n_classes ? cur[s] : 0u;
      uint32_t k = 0, Bc = 0, Oc = 0;
      each_class(l, [&](uint32_t c, uint64_t mm) {
        const uint32_t before = cnt[c], b = sB[c], o = sO[c];
        if (l == c + 1u) {
          k = before + (uint32_t)__popcll(mm & lt);
          Bc = b;
          Oc = o;
        }
        if (lane == 0) cnt[c] = before + (uint32_t)__popcll(mm);
      });
      const bool draw = l != 0u && k >= Bc;
      const uint64_t dm = __ballot(draw);
      const uint32_t d = D + (uint32_t)__popcll(dm & lt) - w0;   // (wraps below the window)
      D += (uint32_t)__popcll(dm);
      if (draw) {
        if (d < win) {
          const double u = (double)x[d] * 2.3283064365386962890625e-10;  // x / 2^32
          const uint32_t j = (uint32_t)roundf((float)(u * (double)k));
          if (j < Bc) atomicMax(&bk[Oc + j], p);
        }
      } else if (l != 0u && w0 == 0u) {
        atomicMax(&bk[Oc + k], p);
      }
    }
  }
}

// One twist of a state by one wave (no tempering: outputs are tempered when
// drawn).  Same three dependent ranges as mt_twist.
__device__ inline void mt_twist_wave(uint32_t *mt, uint32_t lane)
{
  uint32_t a1[4], a2[4], a3[3];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const uint32_t i = lane + 64u * r;
    a1[r] = a2[r] = 0;
    if (i < 227) {
      a1[r] = mt[i + MT_M] ^ mt_mix(mt[i], mt[i + 1]);
      a2[r] = mt_mix(mt[227 + i], mt[228 + i]);
    }
  }
#pragma unroll
  for (int r = 0; r < 3; r++) {
    const uint32_t i = lane + 64u * r;
    a3[r] = (i < 169) ? mt_mix(mt[454 + i], mt[455 + i]) : 0u;
  }
  const uint32_t last_old = mt[623];
  wave_sync();
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (lane + 64u * r < 227) mt[lane + 64u * r] = a1[r];
  wave_sync();
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (lane + 64u * r < 227) mt[227 + lane + 64u * r] = mt[lane + 64u * r] ^ a2[r];
  wave_sync();
#pragma unroll
  for (int r = 0; r < 3; r++)
    if (lane + 64u * r < 169) mt[454 + lane + 64u * r] = mt[227 + lane + 64u * r] ^ a3[r];
  if (lane == 0) mt[623] = mt[396] ^ mt_mix(last_old, mt[0]);
  wave_sync();
}

// Large batches, and batches without scratch: one wave per image (four images
// per block), 64 pixels per step in scan
// order (lane l: pixel t0 + 64 s + l); the label bytes of the next 16 steps
// are prefetched from global memory.  A pixel's class ordinal k is the class
// count so far (LDS) plus its rank among the wave's lanes of that class (one
// ballot per distinct class, the class read with readlane); it draws iff
// k >= B_c, and its draw index is the wave prefix of those flags, so the MT
// stream is consumed in the serial loop's order.  bucket: zero-initialised
// slots [image][sum B] (class c at boff[c]) filled with atomicMax (the last
// writer in scan order has the largest pixel index).  Labels above
// n_classes set *bad.
//
// Bound by VALU issue: about 85 VALU + 43 SALU instructions per 64-pixel step
// (class ranks, the draw's FP64 product and roundf, tempering, a twist per
// 624 draws).  Keeping the slots in LDS instead of global atomics cut the
// occupancy and ran slower.
__global__ __launch_bounds__(256) void k_sample_weighted(const uint8_t *__restrict__ labels,
                                                         const SampleJob *__restrict__ jobs, uint32_t n_images,
                                                         const uint32_t *__restrict__ crc, uint32_t seed,
                                                         uint32_t n_classes, const uint32_t *__restrict__ B,
                                                         const uint32_t *__restrict__ boff, uint32_t *bucket,
                                                         uint32_t *class_count, uint32_t *bad)
{
  __shared__ uint32_t sB[256], sO[256];
  __shared__ uint32_t mt_all[4][MT_N], cnt_all[4][256];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  sB[threadIdx.x] = threadIdx.x < n_classes ? B[threadIdx.x] : 0u;
  sO[threadIdx.x] = threadIdx.x < n_classes ? boff[threadIdx.x] : 0u;
  __syncthreads();  // the only block-wide barrier: from here on the waves are independent
  const uint32_t im = blockIdx.x * 4u + wave;
  if (im >= n_images) return;
  uint32_t *mt = mt_all[wave], *cnt = cnt_all[wave];
  for (uint32_t c = lane; c < 256u; c += 64u) cnt[c] = 0;
  const SampleJob J = jobs[im];
  const uint8_t *lab = labels + J.lab_off;
  uint32_t *bk = bucket + J.out_base;
  if (lane == 0) mt_seed(mt, crc[im] ^ seed);
  wave_sync();
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64u - lane));
  uint32_t D = 0, gen = 0;  // draws consumed; outputs generated ([gen - 624, gen) are in mt)
  uint32_t nx[16];
#pragma unroll
  for (int s = 0; s < 16; s++) nx[s] = (64u * s + lane < J.n_px) ? lab[64u * s + lane] : 0u;
  for (uint32_t t0 = 0; t0 < J.n_px; t0 += 1024u) {
    uint32_t cur[16];
#pragma unroll
    for (int s = 0; s < 16; s++) {
      cur[s] = nx[s];
      const uint32_t q = t0 + 1024u + 64u * s + lane;
      nx[s] = (q < J.n_px) ? lab[q] : 0u;  // prefetch the next tile
    }
#pragma unroll
    for (int s = 0; s < 16; s++) {
      if (t0 + 64u * s >= J.n_px) break;
      const uint32_t p = t0 + 64u * s + lane;
      uint32_t l = cur[s];
      if (l > n_classes) { atomicOr(bad, 1u); l = 0; }
      const bool valid = l != 0u;
      const uint32_t c = l - 1u;
      uint32_t k = 0, Bc = 0, Oc = 0;
      uint64_t pending = __ballot(valid);
      while (pending) {
        const uint32_t lead = (uint32_t)__builtin_ctzll(pending);
        const uint32_t cl = __builtin_amdgcn_readlane(c, lead);
        const uint64_t mm = __ballot(valid && c == cl);
        const uint32_t before = cnt[cl], bcl = sB[cl], ocl = sO[cl];
        if (valid && c == cl) {
          k = before + (uint32_t)__popcll(mm & lt);
          Bc = bcl;
          Oc = ocl;
        }
        if (lane == lead) cnt[cl] = before + (uint32_t)__popcll(mm);
        pending &= ~mm;
      }
      const bool draw = valid && k >= Bc;
      const uint64_t dm = __ballot(draw);
      const uint32_t d = D + (uint32_t)__popcll(dm & lt);
      D += (uint32_t)__popcll(dm);
      uint32_t x = 0;
      if (D > gen) {  // wave-uniform: this step crosses into the next twist
        if (draw && d < gen) x = mt[d + MT_N - gen];
        mt_twist_wave(mt, lane);
        gen += MT_N;
        if (draw && d + MT_N >= gen) x = mt[d + MT_N - gen];
      } else if (draw) {
        x = mt[d + MT_N - gen];
      }
      if (draw) {
        const double u = (double)mt_temper(x) * 2.3283064365386962890625e-10;  // x / 2^32
        const uint32_t j = (uint32_t)roundf((float)(u * (double)k));
        if (j < Bc) atomicMax(&bk[Oc + j], p);
      } else if (valid) {
        atomicMax(&bk[Oc + k], p);
      }
    }
  }
  wave_sync();
  for (uint32_t c = lane; c < n_classes; c += 64u) class_count[(uint64_t)im * n_classes + c] = cnt[c];
}

// filled slots of every class -> contiguous unsorted samples; segment end
__global__ __launch_bounds__(256) void k_compact_buckets(const SampleJob *__restrict__ jobs, uint32_t n_classes,
                                                         const uint32_t *__restrict__ B,
                                                         const uint32_t *__restrict__ boff,
                                                         const uint32_t *__restrict__ class_count,
                                                         const uint32_t *__restrict__ bucket, uint32_t *out,
                                                         uint32_t *n_out, uint32_t *seg_end)
{
  const uint32_t im = blockIdx.x, tid = threadIdx.x;
  const SampleJob J = jobs[im];
  uint32_t dst = 0;
  for (uint32_t c = 0; c < n_classes; c++) {
    const uint32_t cc = class_count[(uint64_t)im * n_classes + c];
    const uint32_t n = cc < B[c] ? cc : B[c];
    for (uint32_t j = tid; j < n; j += 256u) out[J.out_base + dst + j] = bucket[J.out_base + boff[c] + j];
    dst += n;
  }
  if (tid == 0) { n_out[im] = dst; seg_end[im] = J.out_base + dst; }
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t *p, uint64_t n, uint32_t v)
{
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) p[i] = v;
}

// ---- RGB(A) -> label: the first class whose colour equals the pixel's RGB
// (alpha ignored) gives label class + 1, no match gives 0.  keys: the map's
// distinct colours (r << 16 | g << 8 | b) ascending with the first class of
// each, so a binary search finds the first match.
__global__ __launch_bounds__(256) void k_rgb_labels(const uint8_t *__restrict__ rgb, uint64_t n_px, uint32_t ch,
                                                    const uint32_t *__restrict__ keys,
                                                    const uint8_t *__restrict__ cls, uint32_t n_keys,
                                                    uint8_t *__restrict__ out)
{
  __shared__ uint32_t sk[256];
  __shared__ uint8_t sc[256];
  if (threadIdx.x < n_keys) { sk[threadIdx.x] = keys[threadIdx.x]; sc[threadIdx.x] = cls[threadIdx.x]; }
  __syncthreads();
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n_px; i += (uint64_t)gridDim.x * 256u) {
    const uint8_t *p = rgb + i * ch;
    const uint32_t key = ((uint32_t)p[0] << 16) | ((uint32_t)p[1] << 8) | p[2];
    uint32_t lo = 0, hi = n_keys;  // first key >= key
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (sk[mid] < key) lo = mid + 1;
      else hi = mid;
    }
    out[i] = (lo < n_keys && sk[lo] == key) ? (uint8_t)(sc[lo] + 1u) : (uint8_t)0;
  }
}

}  // namespace ingest
}  // namespace pd
