// gemm_rows.hip -- the prompt projection for many rows: C[m][n] = sum_k
// A[m][k] * W[n][k] on 128 x 256 tiles of gfx950's fp16 matrix cores
// (device_matmul / device_matmul_add with batch = seq_len, ascend_matmul.h:
// 102-107).  prefill.hip has the kernels for fewer rows and other K, and the
// rule that chooses.
#include "device_common.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace mmr {
namespace {

using f32x16 = float __attribute__((ext_vector_type(16)));
using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
using f16x4 = _Float16 __attribute__((ext_vector_type(4)));

constexpr int kBM = 128, kBN = 256, kBK = 64;
constexpr int kWaves = 8, kThreads = kWaves * kWave;
constexpr int kStages = 2;
constexpr int kRowChunks = kBK / 8;
constexpr int kPlaneBytes = kBM * kBK * 2;                     // one fp16 plane of A, one stage
constexpr int kStageBytes = 2 * kPlaneBytes + kBN * kBK * 2;   // A hi, A lo, W
constexpr int kActLd = kBN / 2 + 4;                            // floats per row of the act tile
static_assert(kBM * kActLd * 4 <= kStages * kStageBytes, "act tile exceeds the stages");

enum : int { kA32, kAPlanes };  // fp32 rows; fp16 planes with one scale per row and 128 columns
enum : int { kStore, kStoreSplit, kResidual, kSwiGlu };  // kStoreSplit: K split over gridDim.z

// 16-byte chunk position of (row, chunk) in a stage [rows][8 chunks]: the 16
// rows that a fragment read takes at one chunk lie in 16 distinct 16-byte
// bank groups.
__device__ __forceinline__ int chunk_pos(int row, int chunk) { return row * kRowChunks + (chunk ^ ((row >> 1) & 7)); }

// Block = 128 x 256 of C, 8 waves of 64 x 64 (2 x 2 fragments of 32 x 32), K
// in stages of 64: W and pre-split A by direct loads (whole 128-byte lines),
// fp32 A through registers, where it is split hi + lo under a scale per row and 64
// columns (32 in K splits, whose A the layers would otherwise split per 32).  Per
// k step of 16 the products are v_mfma_f32_32x32x16_f16 of the hi and the lo plane.
//
// What bounds it: no unit alone.  While a CU holds a block the matrix cores work
// 40% of the time on fp32 A (51% on planes with SwiGLU), the vector unit 49%
// (25%), LDS 27% (25%), and waves wait a third of theirs, most of it at the
// stages' barriers; on fp32 A the split of A is done again by every column tile.
// On real data the products also pull the clock down (the same launch on
// degenerate data ran 10% faster).  The 64 x 64 tiles of prefill.hip bring twice
// the bytes per product into LDS, and read twice as many from it.  2,048 rows of
// fp32 A, W 4096 x 768: 55.6 us there, 33.8 here (463 -> 762 TFLOP/s of
// products).  Tried before the scales per 64 and 128 columns, pre-split A, 6,000
// rows (gate_up + SwiGLU 85 us, QKV 29; prefill.hip 109 and 39): 128 x 128 tiles
// of 4 waves, two blocks per CU, 101 and 36; 64 x 128 per wave with one level of
// sums, 96 and twice the error.  One scale for a whole row, or one that follows
// its largest value so far, was no faster (2,048 rows 34.2 us) and lost the bits
// of columns far smaller than others.  K may be split over gridDim.z
// (gemm_rows_splits).
template <int kA, int kEpi>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_rows_kernel(GemmArgs g) {
  __shared__ __align__(16) char lds[kStages * kStageBytes];
  // The rows' 1 / s.  Planes: of a pair of stages (128 columns), two pairs in
  // turn.  fp32 A: of a stage's kScaleCols columns each, four stages in turn (a
  // wave may be staging t + 2 while another still adds up t).
  constexpr int kScaleCols = kEpi == kStoreSplit ? kSplitChunkFine : kBK;
  constexpr int kStageScales = kA == kA32 ? kBK / kScaleCols : 1;
  __shared__ __align__(16) float scale[kA == kA32 ? 4 * kStageScales : 2][kBM];

  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 4, wn = wave % 4;
  // Block id i runs on XCD i % 8: each XCD takes a contiguous run of tiles,
  // ordered so that a run covers squares of up to 8 x 8 tiles, whose A rows and
  // W rows its L2 holds.
  const int mt = (g.m + kBM - 1) / kBM, nt = (g.n + kBN - 1) / kBN;
  const int tiles = mt * nt, per_xcd = (tiles + kXcds - 1) / kXcds;
  const int tile = static_cast<int>(blockIdx.x % kXcds) * per_xcd + static_cast<int>(blockIdx.x / kXcds);
  if (tile >= tiles || static_cast<int>(blockIdx.x / kXcds) >= per_xcd) return;  // block-uniform
  const int band = tile / (8 * nt), in_band = tile % (8 * nt);
  const int band_rows = min(8, mt - band * 8);
  const int m0 = (band * 8 + in_band % band_rows) * kBM, n0 = in_band / band_rows * kBN;
  int nk = g.k / kBK;  // even
  if constexpr (kEpi == kStoreSplit) {
    // Split z of S takes pairs of stages z P / S .. (z + 1) P / S of the P =
    // K / 128, at least one; the operands and the output start there.
    const int pairs = nk / 2, split = static_cast<int>(blockIdx.z), splits = static_cast<int>(gridDim.z);
    const int first = pairs * split / splits;
    nk = 2 * (pairs * (split + 1) / splits - first);
    g.w += first * 2 * kBK;
    if constexpr (kA == kA32) {
      g.a += first * 2 * kBK;
    } else {
      g.a_hi += first * 2 * kBK;
      g.a_lo += first * 2 * kBK;
      g.a_inv += first;
    }
    g.c += split * g.split_stride;
  }

  // Direct loads: wave-wide load i fills rows 8 i .. + 7 of a plane (128 bytes
  // each: whole cache lines); this wave takes loads wave, wave + 8, ...
  constexpr int kALoads = kBM / 8 / kWaves, kWLoads = kBN / 8 / kWaves;
  auto source = [&](int j, int r0, int rows, int64_t stride) {
    const int row = (wave + kWaves * j) * 8 + lane / 8;
    return static_cast<uint32_t>((min(r0 + row, rows - 1) * stride + ((lane % 8) ^ ((row >> 1) & 7)) * 8) * 2);
  };
  uint32_t a_off[kALoads], w_off[kWLoads];
#pragma unroll
  for (int j = 0; j < kALoads; ++j) a_off[j] = kA == kA32 ? 0 : source(j, m0, g.m, g.lda);
#pragma unroll
  for (int j = 0; j < kWLoads; ++j) w_off[j] = source(j, n0, g.n, g.k);
  // Planes: waves 0 and 1 bring the scales of 64 rows each.
  const uint32_t s_off = static_cast<uint32_t>(
      min(m0 + wave * kWave + lane, g.m - 1) * static_cast<int64_t>(g.k / kSplitChunk) * 4);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
  const uint32_t scale0 = __builtin_amdgcn_readfirstlane(lds_address(scale)) + wave * kWave * 4;
  auto issue = [&](int t, int buf) {
    const int64_t kb = static_cast<int64_t>(t) * kBK * 2;
    const uint32_t dst = lds0 + buf * kStageBytes + wave * 1024;
    if constexpr (kA != kA32) {
      if (buf == 0 && wave < kBM / kWave)
        dma_load<4>(g.a_inv + t / 2, s_off, scale0 + (t / 2) % 2 * (kBM * 4));
#pragma unroll
      for (int j = 0; j < kALoads; ++j) {
        dma_load<16>(reinterpret_cast<const char*>(g.a_hi) + kb, a_off[j], dst + j * kWaves * 1024);
        dma_load<16>(reinterpret_cast<const char*>(g.a_lo) + kb, a_off[j], dst + j * kWaves * 1024 + kPlaneBytes);
      }
    }
#pragma unroll
    for (int j = 0; j < kWLoads; ++j)
      dma_load<16>(reinterpret_cast<const char*>(g.w) + kb, w_off[j], dst + j * kWaves * 1024 + 2 * kPlaneBytes);
  };

  // fp32 A: this thread's four 4-column pieces of a stage, row (tid + 512 u)
  // / 16, columns 4 (tid % 16).  The lanes of a row's kScaleCols columns find
  // their maximum together, and with it the scale s = 2^(15 - e).
  constexpr int kPieces = kBM * kBK / 4 / kThreads, kPieceRows = kThreads / 16;
  const int a_row = tid / 16, a_col = tid % 16;
  float4 areg[kA == kA32 ? kPieces : 1];
  const float* a_rows = kA == kA32 ? g.a + static_cast<int64_t>(m0) * g.lda : nullptr;
  uint32_t a_src[kPieces];  // bytes from there: under 128 rows of lda < 2^23
#pragma unroll
  for (int u = 0; u < kPieces; ++u)
    a_src[u] = static_cast<uint32_t>(min(a_row + u * kPieceRows, g.m - 1 - m0) * (g.lda * int64_t{4}) + a_col * 16);
  auto load_a = [&](int t) {
    const char* base = reinterpret_cast<const char*>(a_rows + t * kBK);
#pragma unroll
    for (int u = 0; u < kPieces; ++u) areg[u] = *reinterpret_cast<const float4*>(base + a_src[u]);
  };
  // Rows 32 on, a piece's chunk keeps its place in the row.
  static_assert(kPieceRows % 16 == 0, "chunk_pos repeats every 16 rows");
  char* const a_dst = lds + chunk_pos(a_row, a_col / 2) * 16 + a_col % 2 * 8;
  float* const s_dst = &scale[a_col / (kScaleCols / 4)][a_row];
  auto store_a = [&](int t, int buf, int u0, int u1) {
#pragma unroll
    for (int u = u0; u < u1; ++u) {
      const float4 v = areg[u];
      const float mx = group_max<kScaleCols / 4>(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
      const int e = max(__builtin_amdgcn_frexp_expf(mx), -100);  // 0 for a zero chunk
      const float sc = ldexpf(1.0f, 15 - e);
      const float x[4] = {v.x * sc, v.y * sc, v.z * sc, v.w * sc};
      f16x4 hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hi[j] = static_cast<_Float16>(x[j]);
        lo[j] = static_cast<_Float16>(x[j] - static_cast<float>(hi[j]));
      }
      char* dst = a_dst + buf * kStageBytes + u * kPieceRows * kRowChunks * 16;
      *reinterpret_cast<f16x4*>(dst) = hi;
      *reinterpret_cast<f16x4*>(dst + kPlaneBytes) = lo;
      // The lanes of a group write the same value to the same place.
      s_dst[t % 4 * kStageScales * kBM + u * kPieceRows] = ldexpf(1.0f, e - 15);
    }
  };

  const int half = lane / 32, l32 = lane % 32;
  // Fragment addresses within a stage; the next 32 rows (columns) are 4 KB on.
  int a_rd[4], w_rd[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    a_rd[ks] = chunk_pos(wm * 64 + l32, 2 * ks + half) * 16;
    w_rd[ks] = chunk_pos(wn * 64 + l32, 2 * ks + half) * 16 + 2 * kPlaneBytes;
  }
  f32x16 acc[2][2], part[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  struct Frags {
    f16x8 ah[2], al[2], w[2];
  };
  auto read = [&](Frags& f, int buf, int ks) {
    const char* st = lds + buf * kStageBytes;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      f.ah[i] = *reinterpret_cast<const f16x8*>(st + a_rd[ks] + i * 4096);
      f.al[i] = *reinterpret_cast<const f16x8*>(st + a_rd[ks] + i * 4096 + kPlaneBytes);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) f.w[j] = *reinterpret_cast<const f16x8*>(st + w_rd[ks] + j * 4096);
  };
  // Sums run in two levels: the products of the columns under one scale in
  // `part`, then, each row's times its 1 / s, into `acc`; a single chain of K / 16
  // additions doubled the error against 64 bits.
  auto multiply = [&](const Frags& f, bool fresh) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.w[j], fresh ? f32x16{} : part[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.w[j], part[i][j], 0, 0, 0);
  };
  auto flush = [&](const float* inv) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 sv = *reinterpret_cast<const float4*>(inv + wm * 64 + i * 32 + 8 * q + 4 * half);
        const float s4[4] = {sv.x, sv.y, sv.z, sv.w};
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[i][j][4 * q + r] = fmaf(part[i][j][4 * q + r], s4[r], acc[i][j][4 * q + r]);
      }
    if constexpr (kA == kA32) {
      // Here, and not sunk to the next use of acc past store_a's branch: both
      // sums and the next products' would be live at once and spill.
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) asm volatile("" : "+v"(acc[i][j]));
    }
  };

  // Each k step's fragments are read while the one before is multiplied,
  // across stages too.  Stage t + 1 has to be in LDS, and stage t's last
  // fragments in registers, before stage t's last products; then stage t's
  // buffer takes stage t + 2.
  {
    issue(0, 0);
    if constexpr (kA == kA32) {
      load_a(0);
      store_a(0, 0, 0, kPieces);
    }
    issue(1, 1);
    if constexpr (kA == kA32) load_a(1);
    // Stage 0 has landed (fp32 A: its W, waited for with A).
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                 :
                 : "n"((kA == kA32 ? kPieces : 2 * kALoads) + kWLoads)
                 : "memory");
    Frags f0, f1;
    read(f0, 0, 0);
    constexpr bool kHalves = kA == kA32 && kStageScales == 2;  // a scale per two k steps
    auto step = [&](int t, int buf, bool fresh, bool last) {
      read(f1, buf, 1);
      multiply(f0, fresh);
      if constexpr (kA == kA32) {
        if (t + 1 < nk) store_a(t + 1, buf ^ 1, 0, kPieces / 2);
      }
      read(f0, buf, 2);
      multiply(f1, false);
      if constexpr (kHalves) flush(&scale[t % 4 * kStageScales][0]);
      if constexpr (kA == kA32) {
        if (t + 1 < nk) store_a(t + 1, buf ^ 1, kPieces / 2, kPieces);
      }
      read(f1, buf, 3);
      multiply(f0, kHalves);
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (t + 2 < nk) {
        issue(t + 2, buf);
        if constexpr (kA == kA32) load_a(t + 2);
      }
      read(f0, buf ^ 1, 0);  // past the last stage: stale, not used
      multiply(f1, false);
      if (last) flush(&scale[kA == kA32 ? t % 4 * kStageScales + kStageScales - 1 : t / 2 % 2][0]);
    };
    for (int t = 0; t < nk; t += 2) {
      step(t, 0, true, kA == kA32);
      step(t + 1, 1, kA == kA32, true);
    }
  }

  // Lane: column l32 of each 32 x 32 fragment, rows 8 q + 4 half + r.
  if constexpr (kEpi == kSwiGlu) {
    // Gate column 2c in lane 2c, up column in lane 2c + 1: after one exchange
    // the even lane forms act for rows r = 0, 1 and the odd lane for 2, 3;
    // act goes through LDS so that a thread writes 4 columns of a row.
    __syncthreads();
    float* act = reinterpret_cast<float*>(lds);
    const bool odd = (lane & 1) != 0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[4], x[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = acc[i][j][4 * q + r];
            x[r] = dpp_move<dpp::kQuadXor1>(v[r]);
          }
          const float gate[2] = {odd ? x[2] : v[0], odd ? x[3] : v[1]};
          const float up[2] = {odd ? v[2] : x[0], odd ? v[3] : x[1]};
          const int row = wm * 64 + i * 32 + 8 * q + 4 * half + (odd ? 2 : 0), col = (wn * 64 + j * 32 + l32) / 2;
#pragma unroll
          for (int r = 0; r < 2; ++r) act[(row + r) * kActLd + col] = silu_fast(gate[r]) * up[r];
        }
    __syncthreads();
    const int nkc = g.n / 2 / kSplitChunkFine;
#pragma unroll
    for (int p = 0; p < kBM * kBN / 8 / kThreads; ++p) {
      const int idx = tid + p * kThreads, r = idx / (kBN / 8), c4 = idx % (kBN / 8);
      const int row = m0 + r, col = n0 / 2 + c4 * 4;
      const bool ok = row < g.m && col < g.n / 2;
      const float4 v = *reinterpret_cast<const float4*>(&act[r * kActLd + c4 * 4]);
      const int64_t off = static_cast<int64_t>(row) * g.ldc + col;
      if (!g.act_split.hi) {
        if (ok) *reinterpret_cast<float4*>(g.c + off) = v;
        continue;
      }
      const float top = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
      const float mx = group_max<kSplitChunkFine / 4>(ok ? top : 0.0f);
      int e = 0;
      frexpf(mx, &e);  // e = 0 for a zero chunk
      e = max(e, -100);
      const float sc = ldexpf(1.0f, 15 - e);
      const float x[4] = {v.x * sc, v.y * sc, v.z * sc, v.w * sc};
      f16x4 hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hi[j] = static_cast<_Float16>(x[j]);
        lo[j] = static_cast<_Float16>(x[j] - static_cast<float>(hi[j]));
      }
      if (ok) {
        *reinterpret_cast<f16x4*>(g.act_split.hi + off) = hi;
        *reinterpret_cast<f16x4*>(g.act_split.lo + off) = lo;
        if (c4 % (kSplitChunkFine / 4) == 0)
          g.act_split.inv[static_cast<int64_t>(row) * nkc + col / kSplitChunkFine] = ldexpf(1.0f, e - 15);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn * 64 + j * 32 + l32;
        const int base = m0 + wm * 64 + i * 32 + 4 * half;
        float res[16];
        if constexpr (kEpi == kResidual) {
#pragma unroll
          for (int e = 0; e < 16; ++e)
            res[e] = g.residual[static_cast<int64_t>(min(base + 8 * (e / 4) + e % 4, g.m - 1)) * g.ldc + min(col, g.n - 1)];
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = base + 8 * (e / 4) + e % 4;
          if (row < g.m && col < g.n)
            g.c[static_cast<int64_t>(row) * g.ldc + col] = kEpi == kResidual ? res[e] + acc[i][j][e] : acc[i][j][e];
        }
      }
  }
}

template <int kA>
void launch(const GemmArgs& g, hipStream_t s) {
  const int tiles = ((g.m + kBM - 1) / kBM) * ((g.n + kBN - 1) / kBN);
  const dim3 grid((tiles + kXcds - 1) / kXcds * kXcds, 1, g.k_splits);  // x % 8 == 0: a tile's splits share an XCD
  if (g.k_splits > 1) {
    gemm_rows_kernel<kA, kStoreSplit><<<grid, kThreads, 0, s>>>(g);
  } else if (g.swiglu || g.residual) {
    // Of planes, as the layers call it, or onto a caller's fp32 rows.
    constexpr int kEpi = kA == kAPlanes ? kSwiGlu : kResidual;
    gemm_rows_kernel<kA, kEpi><<<grid, kThreads, 0, s>>>(g);
  } else {
    gemm_rows_kernel<kA, kStore><<<grid, kThreads, 0, s>>>(g);
  }
}

}  // namespace

// K splits for a launch of too few tiles for the chip (the plain products of
// the prefill layers, whose consumers add the partials): up to 3, as many as
// keep the blocks to one round, each XCD's 32 CUs taking its share of the tiles
// times the splits.  Whole prompts (fp16 cache, MiniMind2, tiles of O and down
// / of QKV; before: 64 x 64 tiles for O and down, QKV unsplit): 2,500 tokens,
// 60 / 100 tiles, 3 and 2 splits, 3.79 -> 3.57 ms (QKV unsplit 3.64); 3,000
// tokens, 72 / 120, 4.33 -> 3.93 (2 and 2 splits: 4.12); 3,500 tokens, 84, 2
// splits, 4.62 -> 4.51 (3, whose 33 blocks an XCD are two rounds: 4.77); 4,096
// tokens, 96, 2 splits, 5.20 -> 5.01; 2,300 tokens, 54, 3.47 -> 3.34; but 2,048
// tokens, 48 tiles, 2.88 -> 2.94.  4 splits (60 tiles) equal 3; fewer rows are
// not worth it (900 rows, 24 tiles, 8 splits: 1.90 -> 2.01 ms), nor is a short
// K (QKV of 2,500 x 768 x 512 in 3 splits: small model 1.25 -> 1.28 ms).
int gemm_rows_splits(int m, int n, int k) {
  constexpr int kMinRows = 1024, kMinTiles = 54, kMinK = 768, kMaxSplits = 3, kXcdCus = 32;
  if (m < kMinRows || k < kMinK || k % (2 * kBK) != 0) return 0;
  const int64_t tiles = static_cast<int64_t>((m + kBM - 1) / kBM) * ((n + kBN - 1) / kBN);
  const int64_t per_xcd = (tiles + kXcds - 1) / kXcds;
  const int64_t splits = std::min<int64_t>(kMaxSplits, kXcdCus / per_xcd);
  return tiles >= kMinTiles && splits > 1 ? static_cast<int>(splits) : 0;
}

// The unsplit launch against prefill.hip's kernels: a block takes a CU to
// itself, so a launch takes as long as one block per round of 256, and from 96
// tiles on that is the shorter (fp32 A, prefill.hip / this one: 88 tiles, 1,000
// rows of 2816 x 512, 24.4 / 22.3 us; 96 tiles, 4,096 rows of 768 x 2048, 77.0 /
// 72.2; 80 tiles, 2,048 rows of 1152 x 768, 32.1 / 30.3; 64 tiles, 4,096 rows of
// 512 x 1408, 46.2 / 51.9; 128 tiles, 1,000 rows of 4096 x 768, 33.3 / 33.3; 352
// tiles, 4,096 rows of 2816 x 512, 59.9 / 44.8).  A tile's rows must be there:
// up to 64, one row of 64-row tiles does the same product on finer blocks (64
// rows of 24576 x 768 20.3 / 27.5 us, of 24576 x 2048 42.4 / 64.1, of 32768 x
// 768 25.4 / 28.4; 65 rows of 24576 x 256, 768, 2048 and 4096 15.6 / 12.8, 30.9 /
// 27.7, 68.8 / 64.0 and 128.4 / 122.8).  Of the few-rows kernel's range (up to
// 32 rows, K >= 256) that one keeps up to 16 rows (8 rows of 32768 x 768 18.7 /
// 27.0) and, for 17-32, launches below 160 tiles (17 rows of 24576 x 768 21.9 /
// 26.3, of 24576 x 4096 79.8 / 121.6; but of 49152 x 512, 192 tiles, 39.4 /
// 21.9, of 65536 x 768, 256 tiles, 52.5 / 32.4 and of 151936 x 1024, 594 tiles,
// 128.3 / 115.4).
bool gemm_rows_unsplit(int m, int n, int k) {
  constexpr int kMinTiles = 96, kMinRows = 65, kFewRows = 17, kFewRowsEnd = 32, kFewRowsTiles = 160, kFewRowsK = 256;
  const int64_t tiles = static_cast<int64_t>((m + kBM - 1) / kBM) * ((n + kBN - 1) / kBN);
  if (k % (2 * kBK) != 0) return false;
  if (m >= kFewRows && m <= kFewRowsEnd) return k >= kFewRowsK && tiles >= kFewRowsTiles;
  return m >= kMinRows && tiles >= kMinTiles;
}

bool gemm_many_rows(const GemmArgs& g) {
  const int64_t a_bytes = static_cast<int64_t>(g.m) * g.lda * 2, w_bytes = static_cast<int64_t>(g.n) * g.k * 2;
  const int64_t tiles = static_cast<int64_t>((g.m + kBM - 1) / kBM) * ((g.n + kBN - 1) / kBN);
  const bool enough = g.k_splits == 1 ? gemm_rows_unsplit(g.m, g.n, g.k) : g.k_splits == gemm_rows_splits(g.m, g.n, g.k);
  return enough && tiles < (1 << 30) && !g.register_staged && g.k % (2 * kBK) == 0 &&
         (!g.a_hi || (g.a_chunk == kSplitChunk && !g.residual)) &&
         (!g.swiglu || (g.a_hi && g.n % 8 == 0 && g.ldc % 4 == 0)) &&
         (reinterpret_cast<uintptr_t>(g.a) | reinterpret_cast<uintptr_t>(g.a_hi) | reinterpret_cast<uintptr_t>(g.a_lo) |
          reinterpret_cast<uintptr_t>(g.w)) % 16 == 0 &&
         a_bytes < (int64_t{1} << 32) && w_bytes < (int64_t{1} << 32) && g.lda < (1 << 23);
}

hipError_t launch_gemm_many_rows(const GemmArgs& g, hipStream_t stream) {
  if (g.a_hi) {
    launch<kAPlanes>(g, stream);
  } else {
    launch<kA32>(g, stream);
  }
  return hipGetLastError();
}

}  // namespace mmr
