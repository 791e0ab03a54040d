// prefill_attention.hip -- causal attention of many prompt rows over an fp16
// KV cache on gfx950's matrix cores (the reference's device_prefill_attention,
// ascend_custom_ops.h:122-130; per token decoder_layer.cpp:184-234): `tokens`
// queries at positions start .. start + tokens - 1 attend cache keys 0 ..
// their own position.  prefill.hip has the kernel for fewer rows, an fp32
// cache and the other head shapes, and the rule that chooses.
#include "device_common.h"
#include "kernels.h"

#include <type_traits>

namespace mmr {
namespace {

using f32x2 = float __attribute__((ext_vector_type(2)));
using f16x2 = _Float16 __attribute__((ext_vector_type(2)));
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

// x = hi + lo in fp16, each rounded to nearest: 22 significant bits.  lo =
// fp16(x - hi) is one instruction per value: hi * -1 + x, exact in fp32,
// converted by v_fma_mix as it is written.
__device__ __forceinline__ void split8(const float* x, f16x8& hi, f16x8& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x[2 * e], x[2 * e + 1]}, f16x2));
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l[e]) : "v"(h[e]), "v"(x[2 * e]));
    asm("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(l[e]) : "v"(h[e]), "v"(x[2 * e + 1]));
  }
  hi = __builtin_bit_cast(f16x8, u32x4{h[0], h[1], h[2], h[3]});
  lo = __builtin_bit_cast(f16x8, u32x4{l[0], l[1], l[2], l[3]});
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
// for d = 96) and, beside them, the softmax's vector instructions.  A wave
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

  // Merge the key ranges pairwise: (m, l) per query, O^T as the lanes hold it.
  float* mrg = reinterpret_cast<float*>(lds);
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

}  // namespace

// Enough rows for this kernel, against prefill.hip's, whose blocks are 16
// queries x 1 head, one per CU.  That one's time steps up when its blocks
// pass 256, the CUs (512 rows for 8 heads); this one has a quarter as many
// blocks, with a longer start and end, and wins once they fill about half the
// CUs, or sooner after a long cached context, where the key loop is most of
// the time.  d 96 (16-query kernel / this one): 512 rows 8.9 / 13.3 us, 700
// rows 15.2 / 15.7, 1,000 rows 22.2 / 18.0; after 2,000 cached keys 300 rows
// 21.9 / 28.3, 700 rows 43.7 / 32.5.  d 64: 700 rows 11.4 / 12.5, 1,000 rows
// 15.1 / 14.6; after 2,000 keys 700 rows 30.2 / 26.3.  (d 128 does not fit
// the registers of two waves per SIMD.)
bool prefill_attention_many_rows(const PrefillAttnArgs& a) {
  if (a.d != 32 && a.d != 64 && a.d != 96) return false;
  if ((reinterpret_cast<uintptr_t>(a.query) | reinterpret_cast<uintptr_t>(a.out)) % 16 != 0 ||
      (a.query_stride | a.out_stride) % 4 != 0)
    return false;  // rows are read and written 16 bytes at a time
  if (a.hkv <= 0 || a.hq % a.hkv != 0 || a.hq / a.hkv % kHeads != 0) return false;
  const int64_t blocks = int64_t{(a.tokens + kQueryTile - 1) / kQueryTile} * (a.hq / kHeads) * a.seqs;
  return blocks >= 112 || (blocks >= 80 && a.start >= a.tokens);
}

namespace {
template <int D>
void launch_many_rows(const PrefillAttnArgs& a, hipStream_t stream) {
  const dim3 grid((a.tokens + kQueryTile - 1) / kQueryTile, a.hq / kHeads, a.seqs);
  // The page lookup is a compile-time choice: a branch there would cut the
  // step's matrix products into two blocks (82 -> 93 us a pass, 3,000 rows).
  if (a.pool.k) {
    prefill_attention_f16_kernel<D, true><<<grid, kThreads, 0, stream>>>(a);
  } else {
    prefill_attention_f16_kernel<D, false><<<grid, kThreads, 0, stream>>>(a);
  }
}
}  // namespace

hipError_t launch_prefill_attention_many_rows(const PrefillAttnArgs& a, hipStream_t stream) {
  switch (a.d) {
    case 32: launch_many_rows<32>(a, stream); break;
    case 64: launch_many_rows<64>(a, stream); break;
    case 96: launch_many_rows<96>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace mmr
