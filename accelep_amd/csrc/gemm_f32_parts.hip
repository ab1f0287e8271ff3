// fp32 GEMM on the bf16 matrix cores with fp32 results: C[m, n] = A[m, k] @ B[k, n] for any
// m, n >= 1 and k >= 32, of any alignment (Device::MatMul, src/sim_device.cc:185-196).
//
// Both operands are split exactly into three bf16 parts and a product takes six part products, as
// GemmF32SplitBf16Kernel does (gemm_f32.hip has the bound): hi*hi' in one accumulator, the five
// cross terms in another, added once at the end. Six bf16 passes are 2.7 times the rate of one
// fp32 pass.
//  * Workgroup tile 128 x 128 (8 waves: 2 x 2 of 64 x 64, two of each over 16 of a chunk's 32 k) or
//    64 x 64 (4 waves of 32 x 32), K step 32. A chunk's six planes sit in LDS as [part][row or
//    column][k], 16-byte k groups swizzled, double buffered: an MFMA operand is one 16-byte read.
//  * The split happens once per workgroup on the way into LDS. A thread takes 8 k of one A row
//    (two 16-byte loads) and 8 k of one B column (eight dword loads, a wave reads 64 neighbouring
//    columns): both give whole 16-byte LDS pieces with no exchange between lanes, and neither
//    needs an alignment. Two register sets: chunk c + 2 is requested while chunk c is multiplied.
//  * A ragged k puts its short chunk first and zeroes A's part of it in the prologue; rows and
//    columns past the matrix read a clamped one and are not stored.
// Bound: the matrix cores at the chip's power limit. 1000 x 4096 x 4096: 350 us on the fp32 matrix
// cores (96 TFLOP/s) -> 168 to 173 us = 199 TFLOP/s = 1195 TFLOP/s
// of bf16 products, what a large bf16 library product reaches (1160 to 1290); 181 us with the
// compiler's own order of a chunk. 2000 x 1023 x 2047: 136 -> 54 us; 333 x 2048 x 3000: 109 -> 38; 100
// x 777 x 1001: 19.9 -> 10.4. Error against float64 at k = 4096: 1.15e-6 -> 2.7e-7.
//  * The parts carry an operand whole from 2^-110 up to the last binade below the fp32 limit; of a
//    smaller one up to 2^-134 is lost. A wave sums a 32 x 32 tile again on the fp32 matrix cores where
//    a sum is not finite, or not zero and below 2^-110. Two more cases need a look at the operands: a
//    sum of zero (all of its products may be lost) or below 2^-64, and an operand of 2^32 or more (times
//    the loss it can reach larger sums; without one, a sum of 2^-64 or more loses at most k 2^-102,
//    k 2^-38 of it). There the workgroup reads its operands again, and the tile is summed again if one
//    of them is not zero and below 2^-110. 1000 x 4096 x 4096: following the largest operand takes 1.4
//    to 4 us (2 % on the slower of two cards; 9 us more with the lowest exponent followed too), the
//    second reading 30 us, one infinity in A 130, a row of 1e-37 200 (349 us in all on the fp32 matrix
//    cores alone; 64 x 64 tiles summed again one k pair after the other: 440 and 620).
#include "device_common.h"

#include <algorithm>

namespace accel_hip {
namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBK = 32;
constexpr int kXcds = 8;
constexpr int kBand = 4;  // row tiles per band of the tile order

template <int BM>
struct Shape {
  static constexpr int kThreads = 4 * BM;       // one 8-k group of a row and of a column each
  static constexpr int kGroups = BM == 128 ? 2 : 1;  // waves over the k of a chunk
  static constexpr int kS = BM / 64;            // MFMA tiles per wave along each side
  static constexpr int kPlaneVecs = BM * 4;     // 16-byte pieces of one plane
  static constexpr int kBufVecs = 6 * kPlaneVecs;
};

struct PartsArgs {
  const float* a;
  const float* b;
  float* c;
  int64_t m, k, n;
  int32_t tiles_m, tiles_n, tiles, tiles_per_xcd;
  int64_t chunks_per_split;
  float* partials;  // [splits][m][n] when the K range is split, else nullptr
  Epilogue epi;
};

struct Raw {
  v4f a[2];
  float b[8];
};

// First k of chunk ch: chunk 0 reads k 0 .. 31 and keeps 32 - pad of them.
__device__ __forceinline__ int64_t ChunkK(int64_t ch, int pad) { return ch == 0 ? 0 : ch * kBK - pad; }

// Piece of k group g (0..3) of plane row `row`: rows 4 apart share LDS banks, so they take
// different slots.
__device__ __forceinline__ int Piece(int row, int g) { return row * 4 + (g ^ (((row >> 1) ^ (row >> 2)) & 3)); }

__device__ __forceinline__ void LoadRaw(const float* a, const float* b, int64_t n, Raw& r) {
  __builtin_memcpy(&r.a[0], a, sizeof(v4f));
  __builtin_memcpy(&r.a[1], a + 4, sizeof(v4f));
#pragma unroll
  for (int t = 0; t < 8; ++t) r.b[t] = b[t * n];
}

// Operands of this size and more may lift what the parts lose of a tiny one over 2^-64.
constexpr float kHuge = 0x1p32f;
// A workgroup met such an operand; it has a sum below 2^-64 (zero too).
constexpr uint32_t kSeenHuge = 1, kSeenSmall = 2;

// largest = max(largest, |x0|, |x1|) in one instruction (NaNs, which the sums show, are left out).
__device__ __forceinline__ void KeepLargest(float& largest, float x0, float x1) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(largest) : "v"(x0), "v"(x1));
}

// Eight floats (k ascending) to the pieces of the three planes.
template <int BM>
__device__ __forceinline__ void StoreParts(u32x4* planes, int piece, const float (&x)[8], float& largest) {
  uint32_t w[3][4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    SplitBf16Pair(x[2 * v], x[2 * v + 1], w[0][v], w[1][v], w[2][v]);
    KeepLargest(largest, x[2 * v], x[2 * v + 1]);
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) planes[q * Shape<BM>::kPlaneVecs + piece] = u32x4{w[q][0], w[q][1], w[q][2], w[q][3]};
}

template <int BM>
__device__ __forceinline__ void StoreRaw(u32x4* buf, int a_piece, int b_piece, const Raw& r, float& largest) {
  const float xa[8] = {r.a[0][0], r.a[0][1], r.a[0][2], r.a[0][3], r.a[1][0], r.a[1][1], r.a[1][2], r.a[1][3]};
  StoreParts<BM>(buf, a_piece, xa, largest);
  StoreParts<BM>(buf + 3 * Shape<BM>::kPlaneVecs, b_piece, r.b, largest);
}

__device__ __forceinline__ v16f Mfma(const u32x4& a, const u32x4& b, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 16 k of a wave's tile: k groups g0 and g0 + 1 of the chunk.
template <int BM>
__device__ __forceinline__ void MultiplyStep(const u32x4* buf, int lane, int wm, int wn, int g0,
                                             v16f (&hh)[Shape<BM>::kS][Shape<BM>::kS],
                                             v16f (&cross)[Shape<BM>::kS][Shape<BM>::kS]) {
  constexpr int S = Shape<BM>::kS;
  constexpr int P = Shape<BM>::kPlaneVecs;
  const int g = g0 + (lane >> 5);
  u32x4 av[S][3], bv[S][3];
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int i = 0; i < S; ++i) {
      av[i][q] = buf[q * P + Piece((wm * S + i) * 32 + (lane & 31), g)];
      bv[i][q] = buf[(3 + q) * P + Piece((wn * S + i) * 32 + (lane & 31), g)];
    }
  // hi*hi', then hi*mid', mid*hi', mid*mid', hi*lo', lo*hi' (part 0 hi, 1 mid, 2 lo)
  constexpr int kPa[6] = {0, 0, 1, 1, 0, 2};
  constexpr int kPb[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
  for (int q = 0; q < 6; ++q)
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int j = 0; j < S; ++j) {
        v16f& acc = q == 0 ? hh[i][j] : cross[i][j];
        acc = Mfma(av[i][kPa[q]], bv[j][kPb[q]], acc);
      }
}

// Whether some operand that the thread splits in chunks [c0, c1) is not zero and below 2^-110.
__device__ bool TinyOperand(const float* asrc, const float* bsrc, int64_t n, int64_t c0, int64_t c1, int pad) {
  uint32_t low = 0xffffffffu;  // of the bits without the sign, less 1
#pragma unroll 4
  for (int64_t ch = c0; ch < c1; ++ch) {
    Raw r;
    LoadRaw(asrc + ChunkK(ch, pad), bsrc + ChunkK(ch, pad) * n, n, r);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      low = min(low, (__float_as_uint(r.a[e >> 2][e & 3]) << 1) - 1);
      low = min(low, (__float_as_uint(r.b[e]) << 1) - 1);
    }
  }
  return low < (uint32_t(127 - 110) << 24) - 1;
}

// A 32 x 32 tile's sums over the wave's k of chunks [c0, c1) in plain fp32: rows from m0, columns from n0.
template <int BM>
__device__ void PlainSums(const PartsArgs& p, int64_t m0, int64_t n0, int64_t c0, int64_t c1, int pad, int lane, int kg,
                          v16f& acc) {
  constexpr int kPer = 2 / Shape<BM>::kGroups;  // groups of 16 k of a chunk
  const float* arow = p.a + min(m0 + (lane & 31), p.m - 1) * p.k;
  const float* bcol = p.b + min(n0 + (lane & 31), p.n - 1);
  const auto first_k = [&](int g) { return 16 * (kPer == 1 ? kg : g % kPer) + 8 * (lane >> 5); };
  PlainTileSums<Raw, 4>(
      static_cast<int>(c1 - c0) * kPer,
      [&](int g, Raw& r) {
        const int64_t gk = ChunkK(c0 + g / kPer, pad) + first_k(g);
        LoadRaw(arow + gk, bcol + gk * p.n, p.n, r);
      },
      [&](int g, const Raw& r, float (&x)[8], float (&y)[8]) {
        const int keep = c0 + g / kPer == 0 ? kBK - pad : kBK;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const bool in = first_k(g) + s < keep;
          x[s] = in ? r.a[s >> 2][s & 3] : 0.f;
          y[s] = in ? r.b[s] : 0.f;
        }
      },
      acc);
}

template <int BM>
__global__ __launch_bounds__(Shape<BM>::kThreads) __attribute__((amdgpu_waves_per_eu(BM == 128 ? 2 : 3))) void
GemmF32PartsKernel(PartsArgs p) {
  constexpr int S = Shape<BM>::kS;
  constexpr int kGroups = Shape<BM>::kGroups;
  __shared__ u32x4 lds[2 * Shape<BM>::kBufVecs];
  __shared__ uint32_t seen;  // kSeenHuge, kSeenSmall: over the workgroup
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1;
  const int wm = (wave >> 1) & 1;
  const int kg = wave >> 2;
  // Contiguous runs of tiles per XCD (workgroup b runs on XCD b % 8), in bands of kBand row tiles
  // walked column by column.
  const int t = (blockIdx.x % kXcds) * p.tiles_per_xcd + blockIdx.x / kXcds;
  if (t >= p.tiles) return;
  const int band_tiles = kBand * p.tiles_n;
  const int band = t / band_tiles;
  const int in_band = t % band_tiles;
  const int rows_in_band = min(kBand, p.tiles_m - band * kBand);
  const int64_t m0 = static_cast<int64_t>(band * kBand + in_band % rows_in_band) * BM;
  const int64_t n0 = static_cast<int64_t>(in_band / rows_in_band) * BM;
  const int64_t c0 = static_cast<int64_t>(blockIdx.y) * p.chunks_per_split;
  const int64_t k_chunks = (p.k + kBK - 1) / kBK;
  const int chunks = static_cast<int>(min(k_chunks, c0 + p.chunks_per_split) - c0);
  const int pad = static_cast<int>(k_chunks * kBK - p.k);

  // This thread's 8-k group of an A row (4 lanes read a row's 128 bytes) and of a B column.
  const int ar = tid >> 2, ag = tid & 3;
  const int bc = tid % BM, bg = tid / BM;
  const float* asrc = p.a + min(m0 + ar, p.m - 1) * p.k + 8 * ag;
  const float* bsrc = p.b + 8 * bg * p.n + min(n0 + bc, p.n - 1);
  const int a_piece = Piece(ar, ag), b_piece = Piece(bc, bg);

  v16f hh[S][S], cross[S][S];
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int j = 0; j < S; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        hh[i][j][r] = 0.f;
        cross[i][j][r] = 0.f;
      }

  Raw raw[2];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const int64_t k0 = ChunkK(c0 + min(st, chunks - 1), pad);
    LoadRaw(asrc + k0, bsrc + k0 * p.n, p.n, raw[st]);
  }
  if (c0 == 0 && pad != 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (8 * ag + e >= kBK - pad) raw[0].a[e >> 2][e & 3] = 0.f;
  }
  if (tid == 0) seen = 0;
  float largest = 0.f;  // of the operands this thread splits, without the sign
  StoreRaw<BM>(lds, a_piece, b_piece, raw[0], largest);
  __syncthreads();
  for (int base = 0; base < chunks; base += 2) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int ch = base + st;
      if (ch >= chunks) break;  // workgroup-uniform
      // Past the end the loads repeat the last chunk and the store goes to the idle buffer.
      const int64_t k0 = ChunkK(c0 + min(ch + 2, chunks - 1), pad);
      LoadRaw(asrc + k0, bsrc + k0 * p.n, p.n, raw[st]);
      const u32x4* buf = lds + (ch & 1) * Shape<BM>::kBufVecs;
      if constexpr (kGroups == 2) {
        MultiplyStep<BM>(buf, lane, wm, wn, 2 * kg, hh, cross);
      } else {
        MultiplyStep<BM>(buf, lane, wm, wn, 0, hh, cross);
        MultiplyStep<BM>(buf, lane, wm, wn, 2, hh, cross);
      }
      StoreRaw<BM>(lds + ((ch + 1) & 1) * Shape<BM>::kBufVecs, a_piece, b_piece, raw[st ^ 1], largest);
      if constexpr (kGroups == 2) {
        // The operand reads first, then one MFMA, a share of the split and of its stores in turn.
        __builtin_amdgcn_sched_group_barrier(0x100, 12, 0);  // LDS read
#pragma unroll
        for (int q = 0; q < 24; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // VALU
          __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
        }
      }
      LdsBarrier();  // the loads in flight for later chunks stay in flight
    }
  }

  uint32_t top = 0, low = 0xffffffffu;  // of the sums' bits without the sign
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int j = 0; j < S; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        hh[i][j][r] = hh[i][j][r] + cross[i][j][r];
        const uint32_t u = __float_as_uint(hh[i][j][r]) << 1;
        top = max(top, u);
        low = min(low, u);
      }
  constexpr uint32_t kInf = 0xff000000u, k2m64 = uint32_t(127 - 64) << 24, k2m110 = uint32_t(127 - 110) << 24;
  const uint32_t look = (__any(largest >= kHuge) ? kSeenHuge : 0u) | (__any(low < k2m64) ? kSeenSmall : 0u);
  if (lane == 0 && look != 0) atomicOr(&seen, look);
  __syncthreads();
  const bool huge = (seen & kSeenHuge) != 0;
  const bool tiny = seen != 0 && __syncthreads_or(TinyOperand(asrc, bsrc, p.n, c0, c0 + chunks, pad));
  if (__any(top >= kInf || low < k2m64) || (tiny && huge)) {
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int j = 0; j < S; ++j) {
        bool again = tiny && huge;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t u = __float_as_uint(hh[i][j][r]) << 1;
          again |= u >= kInf || u - 1 < k2m110 - 1 || (tiny && u < k2m64);
        }
        if (__any(again))
          PlainSums<BM>(p, m0 + (wm * S + i) * 32, n0 + (wn * S + j) * 32, c0, c0 + chunks, pad, lane, kg, hh[i][j]);
      }
  }

  // Two waves hold a 64 x 64 tile's sums over the two halves of each chunk: wave kg finishes column
  // tile kg and gives its sums of the other one away through LDS.
  constexpr int kCols = S / kGroups == 0 ? 1 : S / kGroups;  // column tiles a wave finishes
  v16f sum[S][kCols];
  if constexpr (kGroups == 2) {
    float* stage = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        stage[((wave * S + i) * 16 + r) * 64 + lane] = kg == 0 ? hh[i][1][r] : hh[i][0][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float other = stage[(((wave ^ 4) * S + i) * 16 + r) * 64 + lane];
        sum[i][0][r] = kg == 0 ? hh[i][0][r] + other : other + hh[i][1][r];
      }
  } else {
#pragma unroll
    for (int i = 0; i < S; ++i) sum[i][0] = hh[i][0];
  }

  // Element r of a 32 x 32 tile sits at row 8 * (r / 4) + 4 * (lane / 32) + r % 4, column lane % 32.
  const int64_t col = n0 + (wn * S + (kGroups == 2 ? kg : 0)) * 32 + (lane & 31);
  if (col >= p.n) return;
  const int64_t row0 = m0 + wm * S * 32 + 4 * (lane >> 5);
  if (p.partials != nullptr) {  // SplitReduceKernel adds the splits in order and applies the epilogue
    float* part = p.partials + static_cast<int64_t>(blockIdx.y) * p.m * p.n + col;
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = row0 + i * 32 + 8 * (r >> 2) + (r & 3);
        if (row < p.m) part[row * p.n] = sum[i][0][r];
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = row0 + i * 32 + 8 * (r >> 2) + (r & 3);
      if (row < p.m) StoreC(p.c, row, col, p.n, p.epi, ApplyEpilogue(sum[i][0][r], row, col, p.n, p.epi));
    }
}

// Tile side and K splits: the cheapest by this estimate (us). A workgroup's chunk takes kChunk64[w]
// with w workgroups on its CU (at most 3 at once), or kChunk128 (96 KB of LDS: one at a time); a
// split adds a launch and the partial sums' way through memory. Measured at k = 4096: 128 tiles
// 1.3 us a chunk (1000 x 4096 x 4096, one tile a CU, 168 us; 207 in two splits); 64 tiles 0.65 / 1.0
// / 1.28 us (33, 512 and 1000 rows, n = 4096: 84, 129 and 247 us). 333 x 2048 x 3000: 83 / 50 / 57
// us with 128 tiles in 1 / 2 / 4 splits, 62 / 50 / 47 with 64 tiles; 64 x 1536 x 576: 35 / 21 / 14
// / 10 us with 64 tiles in 1 / 2 / 4 / 8 splits.
struct Plan {
  int bm;
  int64_t splits;
};

Plan PlanParts(int64_t m, int64_t n, int64_t chunks, int64_t cus, int64_t max_splits) {
  constexpr double kChunk128[2] = {0, 1.3};
  constexpr double kChunk64[4] = {0, 0.65, 1.0, 1.28};
  Plan best{128, 1};
  double best_us = 0;
  for (const int bm : {128, 64}) {
    const int64_t tiles = ((m + bm - 1) / bm) * ((n + bm - 1) / bm);
    const int64_t cap = bm == 128 ? 1 : 3;
    const double* us = bm == 128 ? kChunk128 : kChunk64;
    for (int64_t s = 1; s <= std::max<int64_t>(1, std::min(max_splits, chunks / 2)); ++s) {
      if (s > 1 && tiles * (s - 1) >= cap * cus) break;  // the CUs are full with fewer splits
      const int64_t per_cu = (tiles * s + cus - 1) / cus;
      double t = ((per_cu / cap) * us[cap] + us[per_cu % cap]) * static_cast<double>((chunks + s - 1) / s);
      if (s > 1) t += 3.0 + static_cast<double>((2 * s + 1) * m * n) * 4e-6 / 4.0;
      if (best_us == 0 || t < best_us) {
        best_us = t;
        best = Plan{bm, s};
      }
    }
  }
  return best;
}

}  // namespace

bool LaunchGemmF32Parts(const float* a, const float* b, float* c, int64_t m, int64_t k, int64_t n, const Epilogue& epi,
                        hipStream_t stream) {
  if (m < 1 || n < 1 || k < kBK) return false;
  const int64_t cus = Ctx().cu_count > 0 ? Ctx().cu_count : 256;
  const int64_t chunks = (k + kBK - 1) / kBK;
  // With a split K (ranges of whole chunks) a second kernel adds the partial sums in split order.
  // Where the partial sums have no room (inside a capture, or the no-allocation scratch) the tiles are
  // those of the best plan that keeps K whole.
  constexpr int64_t kMaxSplits = 16;
  Plan plan = PlanParts(m, n, chunks, cus, kMaxSplits);
  int64_t cper = (chunks + plan.splits - 1) / plan.splits;
  int64_t splits = (chunks + cper - 1) / cper;
  if (splits > 1 && !ScratchReady(static_cast<size_t>(splits * m * n) * sizeof(float), kTempFlags, 0)) {
    plan = PlanParts(m, n, chunks, cus, 1);
    splits = 1;
    cper = chunks;
  }
  const int bm = plan.bm;
  const int64_t tiles_m = (m + bm - 1) / bm;
  const int64_t tiles_n = (n + bm - 1) / bm;
  const int64_t tiles = tiles_m * tiles_n;
  if (tiles * kBand > 0x7fffffff) return false;
  PartsArgs args;
  args.a = a;
  args.b = b;
  args.c = c;
  args.m = m;
  args.k = k;
  args.n = n;
  args.tiles_m = static_cast<int32_t>(tiles_m);
  args.tiles_n = static_cast<int32_t>(tiles_n);
  args.tiles = static_cast<int32_t>(tiles);
  args.tiles_per_xcd = static_cast<int32_t>((tiles + kXcds - 1) / kXcds);
  args.chunks_per_split = cper;
  args.partials = splits > 1 ? static_cast<float*>(Workspace(static_cast<size_t>(splits * m * n) * sizeof(float))) : nullptr;
  args.epi = epi;
  const dim3 grid(static_cast<uint32_t>(args.tiles_per_xcd * kXcds), static_cast<uint32_t>(splits));
  if (bm == 128) hipLaunchKernelGGL(GemmF32PartsKernel<128>, grid, dim3(Shape<128>::kThreads), 0, stream, args);
  else hipLaunchKernelGGL(GemmF32PartsKernel<64>, grid, dim3(Shape<64>::kThreads), 0, stream, args);
  Check(hipGetLastError(), "GemmF32PartsKernel launch");
  if (splits > 1) LaunchSplitReduce(args.partials, static_cast<int32_t>(splits), m, n, c, kScalePerRow, nullptr, 0, epi, stream);
  return true;
}

}  // namespace accel_hip
