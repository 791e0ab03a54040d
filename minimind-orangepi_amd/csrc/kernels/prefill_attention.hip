// prefill_attention.hip -- causal attention of many prompt rows on gfx950's
// matrix cores (the reference's device_prefill_attention,
// ascend_custom_ops.h:122-130; per token decoder_layer.cpp:184-234): `tokens`
// queries at positions start .. start + tokens - 1 attend cache keys 0 ..
// their own position.  One kernel for an fp16 cache and one for an fp32 one;
// prefill.hip has the kernel for fewer rows and the other head shapes.
#include "device_common.h"
#include "kernels.h"

#include <type_traits>

namespace mmr {
namespace {

using f32x4 = float __attribute__((ext_vector_type(4)));
using f32x16 = float __attribute__((ext_vector_type(16)));
using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
using f16x4 = _Float16 __attribute__((ext_vector_type(4)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
using i16x4 = short __attribute__((ext_vector_type(4)));

constexpr int kQueryTile = 32;
constexpr int kKeyTile = 32;  // a tile's keys lie in one KV page
constexpr int kWaves = 8;
constexpr int kHeads = 2;  // query heads per block
constexpr int kThreads = kWaves * kWave;

// 16-byte chunk position of (row, chunk) in an LDS tile [32 rows][D / 8
// chunks] of fp16: chunks of a row are permuted by an exclusive or with a
// function of the row, chosen so that both readers touch 256 contiguous-bank
// bytes per pass without padding: the K fragments (16 rows at one chunk: 16
// distinct 16-byte bank groups) and the transposing V reads (4 consecutive
// rows x 64 bytes: 4 distinct 64-byte bank groups).
template <int D>
__device__ __forceinline__ int tile_chunk(int row, int chunk) {
  constexpr int kRow = D / 8;
  int x;
  if constexpr (D == 64) {
    x = ((row & 2) << 1) | ((row >> 2) & 3);
  } else {
    x = (row >> 2) & 3;
  }
  return row * kRow + (chunk ^ x);
}

// Maximum (sum) over the two 32-lane halves of the wave.
__device__ __forceinline__ float half_swap_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_swap_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Eight values split hi + lo (split2).
__device__ __forceinline__ void split8(const float* x, f16x8& hi, f16x8& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) split2(x[2 * e], x[2 * e + 1], h[e], l[e]);
  hi = __builtin_bit_cast(f16x8, u32x4{h[0], h[1], h[2], h[3]});
  lo = __builtin_bit_cast(f16x8, u32x4{l[0], l[1], l[2], l[3]});
}

// Sum of a tile's 16 probabilities in a tree: added one by one to the running
// sum, thousands of keys cost it several units in the last place.
__device__ __forceinline__ float sum16(const float (&p)[16]) {
  float s[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) s[q] = (p[4 * q] + p[4 * q + 1]) + (p[4 * q + 2] + p[4 * q + 3]);
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// The end of a block: the key ranges' (m, l) per query and O^T, as the lanes
// of wave (s, hb) hold them, merge pairwise through `mrg`, and range 0's waves
// write the rows.
template <int D, int HB>
__device__ __forceinline__ void merge_and_write(const PrefillAttnArgs& a, f32x16 (&ot)[D / 32], float m_run,
                                                float l_part, float* mrg, int s, int hb, int lane, int h, int b,
                                                int q0) {
  constexpr int S = kWaves / HB, DT = D / 32;
  constexpr int kMergeFloats = (D / 2 + 2) * kWave;
  const int qi = lane % 32, half = lane / 32;
#pragma unroll
  for (int step = S / 2; step >= 1; step /= 2) {
    __syncthreads();  // the stages (or the previous round's values) have been read
    if (s >= step && s < 2 * step) {
      float* dst = mrg + ((s - step) * HB + hb) * kMergeFloats;
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(dst + ((j * 4 + q) * kWave + lane) * 4) =
              make_float4(ot[j][4 * q], ot[j][4 * q + 1], ot[j][4 * q + 2], ot[j][4 * q + 3]);
      dst[D / 2 * kWave + lane] = m_run;
      dst[D / 2 * kWave + kWave + lane] = l_part;
    }
    __syncthreads();
    if (s < step) {
      const float* src = mrg + (s * HB + hb) * kMergeFloats;
      const float m_b = src[D / 2 * kWave + lane], l_b = src[D / 2 * kWave + kWave + lane];
      const float m_new = fmaxf(m_run, m_b);
      const float m_use = m_new == -INFINITY ? 0.0f : m_new;
      const float ea = __builtin_amdgcn_exp2f(m_run - m_use), eb = __builtin_amdgcn_exp2f(m_b - m_use);
      l_part = l_part * ea + l_b * eb;
      m_run = m_new;
#pragma unroll
      for (int j = 0; j < DT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 v = *reinterpret_cast<const float4*>(src + ((j * 4 + q) * kWave + lane) * 4);
          ot[j][4 * q] = fmaf(v.x, eb, ot[j][4 * q] * ea);
          ot[j][4 * q + 1] = fmaf(v.y, eb, ot[j][4 * q + 1] * ea);
          ot[j][4 * q + 2] = fmaf(v.z, eb, ot[j][4 * q + 2] * ea);
          ot[j][4 * q + 3] = fmaf(v.w, eb, ot[j][4 * q + 3] * ea);
        }
    }
  }
  if (s > 0) return;
  const float inv = 1.0f / half_swap_sum(l_part);
  const bool live = q0 + qi < a.tokens;
  const int64_t orow = static_cast<int64_t>(b) * a.tokens + q0 + qi;
  const int64_t row = orow * a.out_stride + h * D + 4 * half;
#pragma unroll
  for (int j = 0; j < DT; ++j) {
    ot[j] *= inv;
    if (a.out && live) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(a.out + row + 32 * j + 8 * q) =
            make_float4(ot[j][4 * q], ot[j][4 * q + 1], ot[j][4 * q + 2], ot[j][4 * q + 3]);
    }
    if (a.out_split.hi) {  // the 32 dims of slice j are one chunk: 16 here, 16 in the other half
      float mx = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(ot[j][i]));
      mx = half_swap_max(mx);
      int e = 0;
      frexpf(mx, &e);  // e = 0 for a zero chunk
      e = max(e, -100);
      const float sc = ldexpf(1.0f, 15 - e);
      if (live) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f16x4 hi, lo;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = ot[j][4 * q + i] * sc;
            hi[i] = static_cast<_Float16>(x);
            lo[i] = static_cast<_Float16>(x - static_cast<float>(hi[i]));
          }
          *reinterpret_cast<f16x4*>(a.out_split.hi + row + 32 * j + 8 * q) = hi;
          *reinterpret_cast<f16x4*>(a.out_split.lo + row + 32 * j + 8 * q) = lo;
        }
        if (half == 0)
          a.out_split.inv[orow * (a.hq * D / kSplitChunkFine) + h * DT + j] = ldexpf(1.0f, e - 15);
      }
    }
  }
}

// Whether any wave of the block holds an infinity or a NaN (`bad` is LDS of its
// own; the waves meet here).
template <int DT>
__device__ __forceinline__ bool block_not_finite(const f32x16 (&ot)[DT], float l_part, int (&bad)[kWaves], int wave,
                                                 int lane) {
  float z = l_part * 0.0f;
#pragma unroll
  for (int j = 0; j < DT; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) z = fmaf(ot[j][i], 0.0f, z);
  const bool mine = __any(z != 0.0f);
  if (lane == 0) bad[wave] = mine;
  __syncthreads();
  int any = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) any |= bad[w];
  return __builtin_amdgcn_readfirstlane(any) != 0;
}

// The block's rows once more, in plain fp32 and over each query's own keys
// only.  An infinite or NaN key or value reaches, on the matrix cores, every
// query of its tile (0 times it is NaN, also where the key is masked), and with
// split operands every value under its scale.  Here it reaches what the formula
// says: scores of -inf count for nothing, a value touches its own dim, and
// queries before it stay as they are.  It takes some 50 to 100 times as long (6,000
// rows with a NaN in key 0's value: fp16 0.16 -> 14 ms, fp32 0.31 -> 32).  Wave: HB heads x queries s, s + S, ...;
// lane: a key of 64 for the scores, dims lane and lane + 64 for the values.
template <typename KV, int D, int HB, bool kPool>
__device__ void attend_rows_plainly(const PrefillAttnArgs& a, int s, int lane, int h, int b, int q0) {
  constexpr int S = kWaves / HB;
  static_assert(D <= 2 * kWave && kKvPage == kWave, "two dims a lane, a page of keys a step");
  const int g = h / (a.hq / a.hkv);
  const float qscale = 1.4426950408889634f / sqrtf(static_cast<float>(D));
  const int rows = min(kQueryTile, a.tokens - q0);
  for (int qi = s; qi < rows; qi += S) {
    const int qpos = a.start + q0 + qi;
    const int64_t row = static_cast<int64_t>(b) * a.tokens + q0 + qi;
    const float* q = a.query + row * a.query_stride + h * D;
    float m_run = -INFINITY, l = 0.0f, o[2] = {0.0f, 0.0f};
    for (int t0 = 0; t0 <= qpos; t0 += kWave) {
      const KV *k, *v;
      if constexpr (kPool) {
        const int64_t off = kv_pool_offset(a.pool.interleave, b, t0, g, a.hkv, D);
        k = static_cast<const KV*>(a.pool.k) + off;
        v = static_cast<const KV*>(a.pool.v) + off;
      } else {
        const int seg = kv_segment(t0);
        const int64_t off = kv_segment_offset(seg, t0, g, a.hkv, D);
        k = static_cast<const KV*>(a.seg.s[seg].k) + off;
        v = static_cast<const KV*>(a.seg.s[seg].v) + off;
      }
      const int keys = min(kWave, qpos + 1 - t0);
      const KV* key = k + min(lane, keys - 1) * D;
      float dot = 0.0f;
      for (int i = 0; i < D; ++i) dot = fmaf(q[i], to_float<KV>(key[i]), dot);
      const float score = lane < keys ? dot * qscale : -INFINITY;
      const float m_new = fmaxf(m_run, group_max<kWave>(score));
      const float m_use = m_new == -INFINITY ? 0.0f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_use), p = __builtin_amdgcn_exp2f(score - m_use);
      m_run = m_new;
      l = l * alpha + group_sum<kWave>(p);
      o[0] *= alpha;
      o[1] *= alpha;
      for (int j = 0; j < keys; ++j) {
        const float pj = read_lane(p, j);
#pragma unroll
        for (int c = 0; c < 2; ++c)
          if (lane + c * kWave < D) o[c] = fmaf(pj, to_float<KV>(v[j * D + lane + c * kWave]), o[c]);
      }
    }
    const float inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int dim = lane + c * kWave;
      const float x = o[c] * inv;
      const int64_t off = row * a.out_stride + h * D + dim;
      if (a.out && dim < D) a.out[off] = x;
      if (a.out_split.hi) {
        const float mx = group_max<kSplitChunkFine>(dim < D ? fabsf(x) : 0.0f);
        int e = 0;
        frexpf(mx, &e);  // e = 0 for a zero chunk
        e = max(e, -100);
        const float xs = x * ldexpf(1.0f, 15 - e);
        const _Float16 hi = static_cast<_Float16>(xs), lo = static_cast<_Float16>(xs - static_cast<float>(hi));
        if (dim < D) {
          __builtin_memcpy(a.out_split.hi + off, &hi, 2);
          __builtin_memcpy(a.out_split.lo + off, &lo, 2);
          if (dim % kSplitChunkFine == 0)
            a.out_split.inv[row * (a.hq * D / kSplitChunkFine) + (h * D + dim) / kSplitChunkFine] = ldexpf(1.0f, e - 15);
        }
      }
    }
  }
}

// Block = 32 queries x kHeads query heads of one KV group; its 8 waves are 2
// heads x S = 4 key ranges, wave (s, hb) taking the 32-key tiles s, s + S, ...
// of the block's causal range for head hb with its own online softmax.  The
// two waves of a key range share one LDS stage, which direct loads
// (global_load_lds) fill, double buffered, without passing registers.
//
// Per tile S^T = K Q^T and O^T += V^T P^T, both on v_mfma_f32_32x32x16_f16
// with q and p split hi + lo (K and V are exact in fp16).  Lane l holds
// S^T[key 8 (i / 4) + 4 (l / 32) + i % 4][query l % 32], i = 0..15, and the
// second product sums over the keys in that order, so the probabilities are
// its B operand as they are; the A operand V^T comes from two transposing LDS
// reads (ds_read_b64_tr_b16) of 4 consecutive keys each.  Scores carry
// log2(e) / sqrt(d) (folded into q), the softmax is base 2.
//
// What bounds it: the matrix cores (24 products of 32 cycles a tile and head
// for d = 96; 46% of the time a CU holds a block) and, beside them, the softmax's
// vector instructions (55%; LDS 13%).  A wave
// alone leaves the matrix cores idle through its LDS reads, loads and
// bookkeeping, so the products of tile i + 1's scores and tile i - 1's values
// are formed while tile i's scores become probabilities, and the two waves of
// a SIMD run half a step apart, one in the loads while the other has the
// matrix cores (1.33 -> 1.03 us per step of two tiles).  32-query tiles read a
// quarter of the K and V bytes per product of the 16-query kernel in
// prefill.hip (two heads share what there one head of half the queries
// reads), which is what that kernel waits for on long prompts.  8 query heads
// on 2, 3,000 rows from position 1,111: d 96 142.7 -> 72.6 us, d 64 95.4 ->
// 56.2, d 32 69.6 -> 40.9; 4,096 rows from 0, d 96: 163.8 -> 78.3 us.
template <int D, bool kPool>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attention_f16_kernel(
    PrefillAttnArgs a) {
  constexpr int HB = kHeads, S = kWaves / HB;
  constexpr int kGroupThreads = HB * kWave;
  constexpr int kRow = D / 8;                       // 16-byte chunks per row
  constexpr int kTileChunks = kKeyTile * kRow;      // of K or of V
  constexpr int kPer = 2 * kTileChunks / kGroupThreads;
  constexpr int kBuffers = 2;
  constexpr int kTileBytes = kTileChunks * 16;
  constexpr int kStageBytes = 2 * kTileBytes;        // K, then V
  constexpr int kMergeFloats = (D / 2 + 2) * kWave;  // one wave's O^T, m and l
  constexpr int kLdsBytes = kStageBytes * kBuffers * S > kMergeFloats * 4 * kWaves / 2
                                ? kStageBytes * kBuffers * S
                                : kMergeFloats * 4 * kWaves / 2;
  constexpr int DJ = D / 16, DT = D / 32;
  static_assert(2 * kTileChunks % kGroupThreads == 0 && kTileChunks % kWave == 0, "tile split over the group");
  __shared__ __align__(16) char lds[kLdsBytes];
  __shared__ int bad[kWaves];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int s = wave / HB, hb = wave % HB;
  const int gtid = threadIdx.x % kGroupThreads;
  const int h = blockIdx.y * HB + hb;
  const int g = h / (a.hq / a.hkv);
  // The query tiles with the longest key ranges start first.
  const int q0 = (gridDim.x - 1 - blockIdx.x) * kQueryTile;
  const int qi = lane % 32, half = lane / 32;
  const int qpos = a.start + q0 + qi;

  const int b = blockIdx.z;
  const int last_key = a.start + min(q0 + kQueryTile, a.tokens) - 1;
  const int n_tiles = last_key / kKeyTile + 1;
  const int n_iter = (n_tiles + S - 1) / S;

  // Direct loads of a tile: wave-wide load i of the group's wave hb fills
  // chunks 64 (hb + HB i) .. + 63 of [K tile | V tile]; the lane's source row
  // and column (bytes) follow from the chunk's place in the swizzled tile.
  uint32_t whole[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = (gtid + i * kGroupThreads) % kTileChunks, row = c / kRow;
    whole[i] = static_cast<uint32_t>(row * D * 2 + (tile_chunk<D>(row, c % kRow) - row * kRow) * 16);
  }
  struct Tile {
    const char *k, *v;
    int limit;  // last row that may be read: rows past the last key are masked, any key's row will do
  };
  auto locate = [&](int i) {
    const int t0 = min(s + i * S, n_tiles - 1) * kKeyTile;
    if constexpr (kPool) {
      const int64_t off = kv_pool_offset(a.pool.interleave, b, t0, g, a.hkv, D) * 2;
      return Tile{static_cast<const char*>(a.pool.k) + off, static_cast<const char*>(a.pool.v) + off, last_key - t0};
    }
    const int seg = kv_segment(t0);
    const int64_t off = kv_segment_offset(seg, t0, g, a.hkv, D) * 2;
    return Tile{static_cast<const char*>(a.seg.s[seg].k) + off, static_cast<const char*>(a.seg.s[seg].v) + off,
                last_key - t0};
  };
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds)) + s * kBuffers * kStageBytes;
  auto k_buf = [&](int i) { return (i % kBuffers) * kStageBytes; };
  auto v_buf = [&](int i) { return (i % kBuffers) * kStageBytes + kTileBytes; };
  // K of tile ik (and V of tile iv, if want_v) of key range s.
  auto issue = [&](int ik, const Tile& tk, auto want_v, int iv, const Tile& tv) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int first = (hb + i * HB) * kWave;  // wave-uniform
      const bool is_k = first < kTileChunks;
      if (!is_k && !decltype(want_v)::value) continue;
      const int limit = is_k ? tk.limit : tv.limit;
      uint32_t off = whole[i];
      if (limit < kKeyTile - 1) {  // wave-uniform: the last tile, partly past the last key
        const int row = (gtid + i * kGroupThreads) % kTileChunks / kRow;
        off -= static_cast<uint32_t>(max(row - limit, 0) * (D * 2));
      }
      dma_load<16>(is_k ? tk.k : tv.v, off, lds0 + first * 16 + (is_k ? k_buf(ik) : v_buf(iv) - kTileBytes));
    }
  };
  // This wave's loads so far are in LDS and its reads of LDS are done; the
  // barrier then says so to the wave that shares the stage.
  auto landed = [&] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto barrier = [&] { asm volatile("s_barrier" ::: "memory"); };
  const std::true_type yes;
  const std::false_type no;
  const Tile tile0 = locate(0), tile1 = locate(1);
  issue(0, tile0, no, 0, tile0);
  issue(1, tile1, no, 0, tile0);

  // Q^T: dims 16 j + 8 half + {0..7} of query qi, scaled, split hi + lo.
  f16x8 qh[DJ], ql[DJ];
  {
    const float qscale = 1.4426950408889634f / sqrtf(static_cast<float>(D));
    const int64_t qrow = static_cast<int64_t>(b) * a.tokens + min(q0 + qi, a.tokens - 1);
    const float* qsrc = a.query + qrow * a.query_stride + h * D + 8 * half;
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      const float4 x0 = *reinterpret_cast<const float4*>(qsrc + 16 * j);
      const float4 x1 = *reinterpret_cast<const float4*>(qsrc + 16 * j + 4);
      const float x[8] = {x0.x * qscale, x0.y * qscale, x0.z * qscale, x0.w * qscale,
                          x1.x * qscale, x1.y * qscale, x1.z * qscale, x1.w * qscale};
      split8(x, qh[j], ql[j]);
    }
  }

  f32x16 ot[DT];  // O^T[dim 32 jt + 8 (i / 4) + 4 half + i % 4][query qi]
#pragma unroll
  for (int j = 0; j < DT; ++j) ot[j] = f32x16{};
  float m_run = -INFINITY, l_part = 0.0f, alpha = 1.0f;
  bool grew = false;  // wave-uniform

  const char* stage = lds + s * kBuffers * kStageBytes;
  f16x8 kf[DJ], va[2][DT];
  auto read_k = [&](int i) {
    const char* src = stage + k_buf(i);
#pragma unroll
    for (int j = 0; j < DJ; ++j) kf[j] = *reinterpret_cast<const f16x8*>(src + tile_chunk<D>(qi, 2 * j + half) * 16);
  };
  auto read_v = [&](int i) {
    const char* src = stage + v_buf(i) + lane % 2 * 8;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jt = 0; jt < DT; ++jt) {
        const int row = 16 * t + 4 * half + lane % 16 / 4;
        const int chunk = 4 * jt + lane / 16 % 2 * 2 + lane % 4 / 2;
        const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(src + tile_chunk<D>(row, chunk) * 16));
        const i16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(src + tile_chunk<D>(row + 8, chunk) * 16));
        va[t][jt] = __builtin_bit_cast(f16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  };
  auto scores = [&] {
    f32x16 st{};
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j], qh[j], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j], ql[j], st, 0, 0, 0);
    }
    return st;
  };
  f16x8 ph[2], pl[2];
  auto add_pv = [&] {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int jt = 0; jt < DT; ++jt) {
        ot[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[t][jt], ph[t], ot[jt], 0, 0, 0);
        ot[jt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[t][jt], pl[t], ot[jt], 0, 0, 0);
      }
  };

  landed();
  read_k(0);
  f32x16 st = scores();
#pragma unroll
  for (int t = 0; t < 2; ++t) ph[t] = pl[t] = f16x8{};
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int jt = 0; jt < DT; ++jt) va[t][jt] = f16x8{};

  // Step i: the scores of tile i become probabilities while the matrix cores
  // form tile i + 1's scores and add tile i - 1's values.  Waves 0-3 and 4-7
  // (one of each per SIMD) run half a step apart: while one half is between
  // its barriers in the loads and the maximum, the other has the matrix cores.
  Tile tv = tile0, tv1 = tile1, tk = locate(2);
  auto step = [&](int i, auto parity) {
    constexpr int kParity = decltype(parity)::value;  // i % 2
    landed();
    read_k(kParity ^ 1);
    if (i > 0) read_v(kParity ^ 1);
    issue(kParity, tk, yes, kParity, tv);
    const int t0 = (s + i * S) * kKeyTile;
    if (t0 + kKeyTile - 1 > a.start + q0) {  // wave-uniform: the tile reaches past the first query
#pragma unroll
      for (int e = 0; e < 16; ++e) st[e] = t0 + 8 * (e / 4) + 4 * half + e % 4 <= qpos ? st[e] : -INFINITY;
    }
    float mx = st[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, st[e]);
    mx = half_swap_max(mx);
    // Tile i - 1's rise of the maximum reaches O^T before its values do.
    if (grew) {
#pragma unroll
      for (int j = 0; j < DT; ++j) ot[j] *= alpha;
    }
    const float m_new = fmaxf(m_run, mx);
    grew = __any(m_new > m_run);
    // No key of this query yet: the exponents below are of -inf - 0.
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    l_part *= alpha;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_s_setprio(1);
    // One basic block: 24 (d = 96) matrix products with the softmax's vector
    // instructions spread between them.
    const f32x16 st_next = scores();
    add_pv();
    tv = tv1;
    tv1 = tk;
    tk = locate(i + 3);
    float p[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      p[e] = __builtin_amdgcn_exp2f(st[e] - m_use);
      l_part += p[e];
    }
    f16x8 nh[2], nl[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) split8(p + 8 * t, nh[t], nl[t]);
#pragma unroll
    for (int e = 0; e < 2 * DJ + 4 * DT; ++e) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (72 + 2 * DJ + 4 * DT - 1) / (2 * DJ + 4 * DT), 0);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      ph[t] = nh[t];
      pl[t] = nl[t];
    }
    st = st_next;
    __builtin_amdgcn_s_setprio(0);
  };
  if (wave >= kWaves / 2) barrier();
  for (int i = 0; i < n_iter; i += 2) {
    step(i, std::integral_constant<int, 0>{});
    if (i + 1 < n_iter) step(i + 1, std::integral_constant<int, 1>{});
  }
  if (wave < kWaves / 2) barrier();
  landed();
  read_v(n_iter - 1);
  if (grew) {
#pragma unroll
    for (int j = 0; j < DT; ++j) ot[j] *= alpha;
  }
  add_pv();

  if (block_not_finite(ot, l_part, bad, wave, lane)) {
    attend_rows_plainly<__half, D, HB, kPool>(a, s, lane, h, b, q0);
    return;
  }
  merge_and_write<D, HB>(a, ot, m_run, l_part, reinterpret_cast<float*>(lds), s, hb, lane, h, b, q0);
}

// The same over an fp32 cache, D = 64 or 96: block = 32 queries
// x 4 query heads of one KV group, its 8 waves 4 heads x 2 key ranges.  K, V,
// q and p all go to the matrix cores as hi + lo fp16 planes (22 bits; the lo x
// lo products, 2^-22 of the others, are left out), with power-of-two scales
// that keep every plane below 2^15: q per query; K per 8 keys, four of a lane's
// 16 scores; V per tile of 32 keys and D / 4 dims, whose products are summed
// before they meet O^T, so that O^T has no scale; p a fixed 2^15.  A value
// keeps the 22 bits down to 2^-17 of the largest under its scale, below that
// 2^-40 of the largest.  K and V pass through registers, where they are split,
// into the stage that the four heads share: a wave stages 8 rows of K and D / 4
// dims of all 32 rows of V, so that each scale is its own to find.
//
// What bounds it: the splits' and the softmax's vector instructions (67% of the
// time a CU holds a block, d = 96) beside 36 products of 32 cycles a tile and
// head (37%; 1,152 cycles, where products of fp32 operands would take 6,144).  prefill.hip's kernel / this
// one, 8 query heads on 2: d 96, 2,000 rows 118.9 / 89.3 us, 4,096 rows 398.1 /
// 170.5, 3,000 rows after 1,111 keys 349.8 / 171.3; d 64 77.6 / 71.5, 248.3 /
// 136.5, 222.4 / 137.6.  Error against 64 bits of each dimension, of its own
// largest value (d 96, 2,000 rows after 2,000 keys): 2.0e-6 / 1.1e-6; with V's
// dimensions spread over 2^16 1.9e-6 / 1.1e-6, its keys over 2^20 2.2e-6 /
// 1.8e-6, q's dimensions and (inversely) k's over 2^8 1.9e-6 / 1.2e-6, over 2^20
// 1.9e-6 / 1.3e-6, but over 2^24 1.8e-6 / 1.9e-5.  (A tile's values are
// summed before they meet the long sums: added product by product, 3,000 rows
// after 3,000 keys had 5.9e-7 of the largest value against 3.4e-7.  Under one V
// scale per 8 keys and all dims, dimensions 2^-20 of the others' size had 8.7e-6
// of their own; they still do where they share their D / 4 with large ones.
// Scales per 8 dims: 173 -> 198 us, for their maxima over the wave; per 32 dims
// and 8 rows a wave, exchanged through LDS: 195 us.)
constexpr int kHeads32 = 4;
template <int D, bool kPool>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attention_f32_kernel(
    PrefillAttnArgs a) {
  constexpr int HB = kHeads32, S = kWaves / HB;
  constexpr int kRow = D / 8;
  constexpr int kPlaneBytes = kKeyTile * kRow * 16;
  constexpr int kStageBytes = 4 * kPlaneBytes;  // K hi, K lo, V hi, V lo
  constexpr int kMergeFloats = (D / 2 + 2) * kWave;
  constexpr int kStages = 2 * S * kStageBytes;
  constexpr int kLdsBytes = kStages > kMergeFloats * 4 * kWaves / 2 ? kStages : kMergeFloats * 4 * kWaves / 2;
  constexpr int DJ = D / 16, DT = D / 32;
  constexpr int C = D / HB;           // dims of V under one scale
  constexpr int kPer = D / 32;        // float4s of K (and of V) that a thread stages per tile
  // Rows of q and k are scaled as at least 2^-40, so that a masked score's -inf
  // never meets a factor of 0; below 2^-57 they keep fewer than 22 bits.
  constexpr int kMinScoreExp = -40;
  constexpr int kMinValueExp = -100;
  __shared__ __align__(16) char lds[kLdsBytes];
  __shared__ int bad[kWaves];
  __shared__ __align__(16) int k_exp[2][S][HB], v_exp[2][S][HB];

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int s = wave / HB, hb = wave % HB;
  const int h = blockIdx.y * HB + hb;
  const int g = h / (a.hq / a.hkv);
  const int q0 = (gridDim.x - 1 - blockIdx.x) * kQueryTile;
  const int qi = lane % 32, half = lane / 32;
  const int qpos = a.start + q0 + qi;
  const int b = blockIdx.z;
  const int last_key = a.start + min(q0 + kQueryTile, a.tokens) - 1;
  const int n_tiles = last_key / kKeyTile + 1;
  const int n_iter = (n_tiles + S - 1) / S;

  // This wave stages rows 8 hb .. + 7 of a K tile, eight lanes a row, and dims
  // C hb .. + C - 1 of a V tile's 32 rows.
  static_assert(8 * HB == kKeyTile && kPer * kWave * 4 == kKeyTile * C, "tile split over the waves");
  const int krow = 8 * hb + lane / 8;
  auto vrow = [&](int u) { return (lane + u * kWave) / (C / 4); };
  int koff[kPer], kpos[kPer], voff[kPer], vpos[kPer];  // elements from the tile in memory, bytes from its plane
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int kcol = 32 * u + lane % 8 * 4, vcol = C * hb + (lane + u * kWave) % (C / 4) * 4;
    // (Of d 96 the swizzle permutes groups of 4 chunks: each piece alike.)
    koff[u] = u > 0 ? koff[0] + 32 * u : krow * D + kcol;
    kpos[u] = D == 96 && u > 0 ? kpos[0] + 64 * u : tile_chunk<D>(krow, kcol / 8) * 16 + kcol % 8 * 2;
    voff[u] = vrow(u) * D + vcol;
    vpos[u] = tile_chunk<D>(vrow(u), vcol / 8) * 16 + vcol % 8 * 2;
  }
  f32x4 kreg[kPer], vreg[kPer];
  auto load = [&](f32x4 (&r)[kPer], const int (&whole)[kPer], auto row, void* const* seg_base, const void* pool, int i) {
    const int t0 = min(s + i * S, n_tiles - 1) * kKeyTile;
    const float* base;
    if constexpr (kPool) {
      base = static_cast<const float*>(pool) + kv_pool_offset(a.pool.interleave, b, t0, g, a.hkv, D);
    } else {
      const int seg = kv_segment(t0);
      base = static_cast<const float*>(seg_base[2 * seg]) + kv_segment_offset(seg, t0, g, a.hkv, D);
    }
    const int limit = last_key - t0;  // rows past the last key are masked, any key's row will do
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      int off = whole[u];
      if (limit < kKeyTile - 1) off -= max(row(u) - limit, 0) * D;  // wave-uniform branch
      r[u] = *reinterpret_cast<const f32x4*>(base + off);
    }
  };
  static_assert(sizeof(KvSeg) == 2 * sizeof(void*), "segments are (k, v) pairs");
  auto load_k = [&](int i) { load(kreg, koff, [&](int) { return krow; }, &a.seg.s[0].k, a.pool.k, i); };
  auto load_v = [&](int i) { load(vreg, voff, vrow, &a.seg.s[0].v, a.pool.v, i); };
  char* stage0 = lds + s * kStageBytes;
  auto stage = [&](int parity) { return stage0 + parity * S * kStageBytes; };
  static_assert(C % 8 == 0, "a scale for whole runs of 8 dims");
  auto largest = [](const f32x4& r) {
    return fmaxf(fmaxf(fabsf(r[0]), fabsf(r[1])), fmaxf(fabsf(r[2]), fabsf(r[3])));
  };
  // The wave's share of a tile to one exponent (at least `least`) and two planes.
  auto store = [&](const f32x4 (&r)[kPer], const int (&pos)[kPer], char* hi_plane, int* exponent, int least) {
    float mx = 0.0f;
#pragma unroll
    for (int u = 0; u < kPer; ++u) mx = fmaxf(mx, largest(r[u]));
    mx = group_max<kWave>(mx);
    const int e = mx > 0.0f ? max(__builtin_amdgcn_frexp_expf(mx), least) : least;
    const float sc = ldexpf(1.0f, 15 - e);
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      uint32_t hw[2], lw[2];
#pragma unroll
      for (int w = 0; w < 2; ++w) split2(r[u][2 * w] * sc, r[u][2 * w + 1] * sc, hw[w], lw[w]);
      *reinterpret_cast<uint2*>(hi_plane + pos[u]) = make_uint2(hw[0], hw[1]);
      *reinterpret_cast<uint2*>(hi_plane + kPlaneBytes + pos[u]) = make_uint2(lw[0], lw[1]);
    }
    if (lane == 0) exponent[hb] = e;
  };
  auto store_k = [&](int parity) { store(kreg, kpos, stage(parity), k_exp[parity][s], kMinScoreExp); };
  auto store_v = [&](int parity) { store(vreg, vpos, stage(parity) + 2 * kPlaneBytes, v_exp[parity][s], kMinValueExp); };
  auto barrier = [&] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  load_k(0);
  load_v(0);

  // Q^T: dims 16 j + 8 half + {0..7} of query qi times log2(e) / sqrt(d) and
  // the query's scale 2^(15 - e_q), split hi + lo.
  f16x8 qh[DJ], ql[DJ];
  int e_q = kMinScoreExp;
  {
    const float qscale = 1.4426950408889634f / sqrtf(static_cast<float>(D));
    const int64_t qrow = static_cast<int64_t>(b) * a.tokens + min(q0 + qi, a.tokens - 1);
    const float* qsrc = a.query + qrow * a.query_stride + h * D + 8 * half;
    float x[DJ][8];
    float mx = 0.0f;
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      const float4 x0 = *reinterpret_cast<const float4*>(qsrc + 16 * j);
      const float4 x1 = *reinterpret_cast<const float4*>(qsrc + 16 * j + 4);
      const float y[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[j][e] = y[e] * qscale;
        mx = fmaxf(mx, fabsf(x[j][e]));
      }
    }
    mx = half_swap_max(mx);
    if (mx > 0.0f) e_q = max(__builtin_amdgcn_frexp_expf(mx), kMinScoreExp);
    const float sc = ldexpf(1.0f, 15 - e_q);
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] *= sc;
      split8(x[j], qh[j], ql[j]);
    }
  }

  f32x16 ot[DT];  // O^T[dim 32 jt + 8 (i / 4) + 4 half + i % 4][query qi]
#pragma unroll
  for (int j = 0; j < DT; ++j) ot[j] = f32x16{};
  float m_run = -INFINITY, l_part = 0.0f, alpha = 1.0f;
  float v_unit[HB];  // 2^(e - 30) of the V tile whose values come next, e its exponents
#pragma unroll
  for (int j = 0; j < HB; ++j) v_unit[j] = 0.0f;
  bool grew = false;  // wave-uniform

  auto scores = [&](int parity) {
    const char* kst = stage(parity);
    f32x16 st{};
#pragma unroll
    for (int j = 0; j < DJ; ++j) {
      const int pos = tile_chunk<D>(qi, 2 * j + half) * 16;
      const f16x8 kh = *reinterpret_cast<const f16x8*>(kst + pos);
      const f16x8 kl = *reinterpret_cast<const f16x8*>(kst + pos + kPlaneBytes);
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[j], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[j], st, 0, 0, 0);
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[j], st, 0, 0, 0);
    }
    return st;
  };
  f16x8 ph[2], pl[2];
  auto add_pv = [&](int parity) {
    const char* vst = stage(parity) + 2 * kPlaneBytes + lane % 2 * 8;
#pragma unroll
    for (int jt = 0; jt < DT; ++jt) {
      f32x16 sum{};  // the tile's, 2^(30 - e) times: a sixth of the roundings at O^T's size
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int row = 16 * t + 4 * half + lane % 16 / 4;
        const int chunk = 4 * jt + lane / 16 % 2 * 2 + lane % 4 / 2;
        auto column = [&](int plane) {
          const char* src = vst + plane * kPlaneBytes;
          const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(src + tile_chunk<D>(row, chunk) * 16));
          const i16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(src + tile_chunk<D>(row + 8, chunk) * 16));
          return __builtin_bit_cast(f16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        const f16x8 vh = column(0), vl = column(1);
        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph[t], sum, 0, 0, 0);
        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl[t], sum, 0, 0, 0);
        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph[t], sum, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 16; ++e) ot[jt][e] = fmaf(sum[e], v_unit[(32 * jt + 8 * (e / 4)) / C], ot[jt][e]);
    }
  };

  // Steps as in the fp16 kernel: K is staged two tiles ahead and V with its
  // tile, each from registers that were loaded a step earlier.
  store_k(0);
  load_k(1);
  store_k(1);
  load_k(2);
  barrier();
  f32x16 st = scores(0);
  int4 kx = *reinterpret_cast<const int4*>(&k_exp[0][s][0]);
#pragma unroll
  for (int t = 0; t < 2; ++t) ph[t] = pl[t] = f16x8{};

  auto step = [&](int i, auto parity) {
    constexpr int kParity = decltype(parity)::value;  // i % 2
    barrier();
    store_k(kParity);
    store_v(kParity);
    load_k(i + 3);
    load_v(i + 1);
    const int t0 = (s + i * S) * kKeyTile;
    if (t0 + kKeyTile - 1 > a.start + q0) {  // wave-uniform: the tile reaches past the first query
#pragma unroll
      for (int e = 0; e < 16; ++e) st[e] = t0 + 8 * (e / 4) + 4 * half + e % 4 <= qpos ? st[e] : -INFINITY;
    }
    const float inv[4] = {ldexpf(1.0f, e_q + kx.x - 30), ldexpf(1.0f, e_q + kx.y - 30), ldexpf(1.0f, e_q + kx.z - 30),
                          ldexpf(1.0f, e_q + kx.w - 30)};
    float mx = -INFINITY;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      mx = fmaxf(mx, fmaxf(fmaxf(st[4 * q], st[4 * q + 1]), fmaxf(st[4 * q + 2], st[4 * q + 3])) * inv[q]);
    mx = half_swap_max(mx);
    // Tile i - 1's rise of the maximum reaches O^T before its values do.
    if (grew) {
#pragma unroll
      for (int j = 0; j < DT; ++j) ot[j] *= alpha;
    }
    const float m_new = fmaxf(m_run, mx);
    grew = __any(m_new > m_run);
    // No key of this query yet: the exponents below are of -inf - 0.
    const float m_use = m_new == -INFINITY ? 0.0f : m_new;
    alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    l_part *= alpha;
    barrier();
    __builtin_amdgcn_s_setprio(1);
    const f32x16 st_next = scores(kParity ^ 1);
    kx = *reinterpret_cast<const int4*>(&k_exp[kParity ^ 1][s][0]);
    if (i > 0) add_pv(kParity ^ 1);
    const int4 vx = *reinterpret_cast<const int4*>(&v_exp[kParity][s][0]);
    const int ve[HB] = {vx.x, vx.y, vx.z, vx.w};
#pragma unroll
    for (int j = 0; j < HB; ++j) v_unit[j] = ldexpf(1.0f, __builtin_amdgcn_readfirstlane(ve[j]) - 30);
    float p[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) p[e] = __builtin_amdgcn_exp2f(fmaf(st[e], inv[e / 4], -m_use));
    l_part += sum16(p);
#pragma unroll
    for (int e = 0; e < 16; ++e) p[e] *= 32768.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t) split8(p + 8 * t, ph[t], pl[t]);
    st = st_next;
    __builtin_amdgcn_s_setprio(0);
  };
  if (wave >= kWaves / 2) barrier();
  for (int i = 0; i < n_iter; i += 2) {
    step(i, std::integral_constant<int, 0>{});
    if (i + 1 < n_iter) step(i + 1, std::integral_constant<int, 1>{});
  }
  if (wave < kWaves / 2) barrier();
  if (grew) {
#pragma unroll
    for (int j = 0; j < DT; ++j) ot[j] *= alpha;
  }
  add_pv((n_iter - 1) & 1);
  if (block_not_finite(ot, l_part, bad, wave, lane)) {
    attend_rows_plainly<float, D, HB, kPool>(a, s, lane, h, b, q0);
    return;
  }
  merge_and_write<D, HB>(a, ot, m_run, l_part, reinterpret_cast<float*>(lds), s, hb, lane, h, b, q0);
}

}  // namespace

// What both kernels need: rows are read and written 16 bytes at a time, and a
// block's heads are of one KV group.
static bool many_rows_shape(const PrefillAttnArgs& a, int heads) {
  if ((reinterpret_cast<uintptr_t>(a.query) | reinterpret_cast<uintptr_t>(a.out)) % 16 != 0 ||
      (a.query_stride | a.out_stride) % 4 != 0)
    return false;
  return a.hkv > 0 && a.hq % a.hkv == 0 && a.hq / a.hkv % heads == 0;
}

// The time of a launch as its blocks' rounds (one block per CU) times a block's
// start and end and its keys.
struct AttnCost {
  float base, round, key;  // us
  float us(int64_t blocks, float keys) const {
    constexpr int64_t kCus = 256;
    return base + static_cast<float>((blocks + kCus - 1) / kCus) * (round + key * keys);
  }
};

// These kernels against prefill.hip's, whose blocks are 16 queries x 1 head: an
// eighth (fp32 cache) or a quarter as many blocks here, with a longer start and
// end.  Either time steps up when the blocks pass a multiple of the 256 CUs,
// for one sequence as for a batch of short ones.  The costs are fitted to kernel
// times of 93 launches per row of the table, 8 query heads on 2, one sequence of
// 64-4,096 rows after 0-6,000 keys and batches of 2-128 sequences of 8-1,500
// rows; the choice by them takes 0.1% (d 32: 0.4, fp32 d 64: 0.3) more than the better
// kernel of each, where a count of this kernel's blocks took 1.6-5.2%.  Some of
// them (prefill.hip / this one), fp16 d 96: 64 sequences of 16 rows 10.2 / 11.1
// us, of 24 19.6 / 12.1; 16 of 64 10.6 / 12.3, of 100 20.1 / 13.4; one of 512 rows
// 8.9 / 13.3, of 700 after 2,000 keys 43.7 / 32.5; d 64: 64 of 33 14.5 / 18.4, 16 of
// 160 14.8 / 18.2, of 255 24.8 / 21.4.  fp32 d 96: 64 of 16 11.7 / 13.4, of 24 21.5 /
// 14.6; 8 of 200 28.3 / 21.6; one of 1,000 43.8 / 49.8, of 2,000 118.9 / 89.3; d 64:
// 32 of 48 9.8 / 11.7, 16 of 255 38.8 / 22.1.  (fp16 d 128 does not fit the
// registers of two waves per SIMD; d 32 on an fp32 cache, with a third of d 96's
// products to the same softmax and splits, measured slower at all but 4,096 rows.)
bool prefill_attention_many_rows(const PrefillAttnArgs& a, KvDtype kv) {
  const bool f16 = kv == kKvF16;
  const int heads = f16 ? kHeads : kHeads32;
  if (!(f16 || kv == kKvF32) || !many_rows_shape(a, heads)) return false;
  AttnCost few, many;
  switch (a.d) {
    case 32:
      if (!f16) return false;
      few = {3.0f, 0.9f, 0.0046f}, many = {5.0f, 2.0f, 0.0055f};
      break;
    case 64:
      if (f16) {
        few = {3.4f, 1.85f, 0.0055f}, many = {0.0f, 9.5f, 0.0068f};
      } else {
        few = {3.9f, 1.95f, 0.0152f}, many = {0.0f, 11.6f, 0.0370f};
      }
      break;
    case 96:
      if (f16) {
        few = {2.2f, 4.2f, 0.0076f}, many = {0.0f, 11.8f, 0.0082f};
      } else {
        few = {2.9f, 4.7f, 0.0220f}, many = {0.0f, 15.6f, 0.0450f};
      }
      break;
    default: return false;
  }
  const int64_t row_heads = static_cast<int64_t>(a.hq) * a.seqs;
  const float start = static_cast<float>(a.start), tokens = static_cast<float>(a.tokens);
  const int64_t few_blocks = (a.tokens + int64_t{15}) / 16 * row_heads;
  const int64_t many_blocks = (a.tokens + int64_t{kQueryTile} - 1) / kQueryTile * (row_heads / heads);
  // Keys of a block: the mean where there are many rounds, nearer the longest in one.
  return many.us(many_blocks, start + 0.75f * tokens) < few.us(few_blocks, start + 0.5f * tokens);
}

namespace {
// The page lookup is a compile-time choice: a branch there would cut the
// step's matrix products into two blocks (82 -> 93 us a pass, fp16, 3,000 rows).
template <int D>
void launch_f16(const PrefillAttnArgs& a, hipStream_t stream) {
  const dim3 grid((a.tokens + kQueryTile - 1) / kQueryTile, a.hq / kHeads, a.seqs);
  if (a.pool.k) {
    prefill_attention_f16_kernel<D, true><<<grid, kThreads, 0, stream>>>(a);
  } else {
    prefill_attention_f16_kernel<D, false><<<grid, kThreads, 0, stream>>>(a);
  }
}
template <int D>
void launch_f32(const PrefillAttnArgs& a, hipStream_t stream) {
  const dim3 grid((a.tokens + kQueryTile - 1) / kQueryTile, a.hq / kHeads32, a.seqs);
  if (a.pool.k) {
    prefill_attention_f32_kernel<D, true><<<grid, kThreads, 0, stream>>>(a);
  } else {
    prefill_attention_f32_kernel<D, false><<<grid, kThreads, 0, stream>>>(a);
  }
}
}  // namespace

hipError_t launch_prefill_attention_many_rows(const PrefillAttnArgs& a, KvDtype kv, hipStream_t stream) {
  if (kv == kKvF32) {
    switch (a.d) {
      case 64: launch_f32<64>(a, stream); break;
      case 96: launch_f32<96>(a, stream); break;
      default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
  }
  switch (a.d) {
    case 32: launch_f16<32>(a, stream); break;
    case 64: launch_f16<64>(a, stream); break;
    case 96: launch_f16<96>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mmr
