// int8-weight GEMV that reads W in place: C[m, n] = A[m, k] @ dequant(q[k, n]) for m <= 16 and any
// plane accel::MatMulQuantized takes (src/sim_device.cc:541-602): zero points, a per-row scale, any
// k, n and alignment, no staged copy.
//
// Exact products on v_mfma_f32_16x16x32_bf16 (A: 16 rows x 32 k, B: 32 k x 16 columns):
//  * q - z is an integer in [-255, 255], which bf16 holds exactly;
//  * an activation x (times the row's scale where it has one: fl(x * s), one rounding where the
//    reference rounds (q - z) * s) is the sum of three bf16 parts, which carry its 24 bits.
// Only the fp32 accumulation rounds. The parts carry an activation whole from 2^-110 up to the last
// binade below the fp32 limit; of a smaller one up to 2^-134 is lost, which reaches no sum of 2^-64 or
// more. A workgroup takes its products again on v_mfma_f32_16x16x4f32 for the rows where a sum is not
// finite, or not zero and below 2^-110, or below 2^-64 (zero too) beside an activation below 2^-110, which
// it looks for in those rows then. With zero points, 4096 x 4096, m = 8: 9.6 us, one infinity 16.4, a row of
// zeros 13.3; 4096 x 14336, m = 16: 19.9, 45.7 and 24.0 (with the elements of a workgroup summed one weight
// after the other 59 and 1200 us for the infinity). Following the lowest activation in the loop
// instead of looking for it costs ordinary calls 0.2 to 0.6 us.
//
//  * A workgroup owns 16 * V columns over one split of K. Its waves take 32-row blocks in turn;
//    lane l reads V consecutive bytes (slot l % 16) of rows 8g .. 8g + 7, g = l / 16, of the block,
//    so one load of the wave covers four row runs of 16 * V bytes, and byte j of its 8 rows is the
//    lane's B operand of the MFMA for column j: no LDS stage and no lane exchange.
//  * The A operand is 8 consecutive floats of row l % 16, read straight from A (rows past m repeat
//    row m - 1; their sums are not stored).
//  * The next block's loads are issued before the current one is converted and multiplied.
//  * The waves' sums meet in LDS in wave order; with a split K each workgroup stores its partial
//    sums and the last one of a column group to arrive adds them in split order.
//
// Bound: HBM, k * n bytes, read in runs of 16 * V bytes a row (about 3.7 TB/s), and about 5 us of
// entry, exchange and store. Loads are plain ones: neighbouring groups share the lines of unaligned
// rows in L2 (3001 x 10001, m = 16: 13.3 us, 15.1 with nontemporal loads). The kernel before it
// multiplied on v_mfma_f32_16x16x4f32 from an LDS stage of A and split K into a second kernel:
// m = 16 with zero points 4096 x 14336 36 -> 19.4 us, 4096 x 4096 17.2 -> 9.3 (m = 8), 3001 x 10001
// 63 -> 15.1, 576 x 3072 14.6 -> 5.0. The hi parts and the rest have accumulators of their own:
// error against float64 at 4096 x 4096 1.3e-7 with one set, 9.3e-8 with two (1.7e-7 before).
#include "device_common.h"

#include <algorithm>

namespace accel_hip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kXcds = 8;
constexpr int kBlockRows = 32;
constexpr int kWaves = 8;  // waves of a workgroup

// What the plane brings: kNone per-column or whole-tensor scale, no zero points; kZero the same
// with zero points; kRow a per-row scale; kRowZero the same with zero points.
enum Form : int { kNone = 0, kZero = 1, kRow = 2, kRowZero = 3 };

// V consecutive bytes at any address.
template <int V>
struct Run;
template <>
struct Run<1> {
  typedef uint8_t type;
};
template <>
struct Run<2> {
  typedef uint16_t type __attribute__((aligned(1)));
};
template <>
struct Run<4> {
  typedef uint32_t type __attribute__((aligned(1)));
};
template <>
struct Run<8> {
  typedef uint32_t type __attribute__((ext_vector_type(2), aligned(1)));
};
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));

struct Q8InPlaceArgs {
  const float* scale;
  const int8_t* zero;
  int32_t mode;
  int64_t const_index;
  float* c;
  Epilogue epi;
};

template <int V>
constexpr int Words() {
  return V < 4 ? 1 : V / 4;
}

// One 32-row block of a lane: V bytes of its 8 rows, the 8 activations, and with a per-row scale
// the rows' scales and zero points.
template <int V, int kForm>
struct Block {
  uint32_t w[8][Words<V>()];
  float x[8];
  float s[kForm >= kRow ? 8 : 1];
  int8_t z[kForm == kRowZero ? 8 : 1];
};

template <int V, int kForm>
__device__ __forceinline__ void LoadBlock(const int8_t* qcol, const float* arow, const Q8InPlaceArgs& p, int32_t kb,
                                          int64_t n, int32_t row, Block<V, kForm>& t) {
  using R = typename Run<V>::type;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const R* src = reinterpret_cast<const R*>(qcol + (row + u) * n);
    const R v = *src;
    if constexpr (V <= 4) {
      t.w[u][0] = v;
    } else {
#pragma unroll
      for (int i = 0; i < Words<V>(); ++i) t.w[u][i] = v[i];
    }
  }
#pragma unroll
  for (int u = 0; u < 8; u += 4) {
    const v4f_any v = *reinterpret_cast<const v4f_any*>(arow + row + u);
#pragma unroll
    for (int i = 0; i < 4; ++i) t.x[u + i] = v[i];
  }
  if constexpr (kForm >= kRow) {
#pragma unroll
    for (int u = 0; u < 8; u += 4) {
      const v4f_any v = *reinterpret_cast<const v4f_any*>(p.scale + kb + row + u);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.s[u + i] = v[i];
    }
  }
  if constexpr (kForm == kRowZero) __builtin_memcpy(t.z, p.zero + kb + row, 8);
}

// The last, short block of a split: rows past its end read its last row and enter as 0.
template <int V, int kForm>
__device__ __forceinline__ void LoadTail(const int8_t* qcol, const float* arow, const Q8InPlaceArgs& p, int32_t kb,
                                         int64_t n, int32_t row, int32_t rows, Block<V, kForm>& t) {
  using R = typename Run<V>::type;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int32_t r = min(row + u, rows - 1);
    const R v = *reinterpret_cast<const R*>(qcol + r * n);
    if constexpr (V <= 4) {
      t.w[u][0] = v;
    } else {
#pragma unroll
      for (int i = 0; i < Words<V>(); ++i) t.w[u][i] = v[i];
    }
    const float x = arow[r];
    t.x[u] = row + u < rows ? x : 0.f;
    if constexpr (kForm >= kRow) {
      const float sc = p.scale[kb + r];
      t.s[u] = row + u < rows ? sc : 0.f;
    }
    if constexpr (kForm == kRowZero) t.z[u] = p.zero[kb + r];
  }
}

template <int V, int kForm>
__device__ __forceinline__ void Multiply(const Block<V, kForm>& t, const float (&zc)[V], v4f (&acc)[V],
                                         v4f (&rest)[V]) {
  u32x4 ah, am, al;
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    float x0 = t.x[2 * h], x1 = t.x[2 * h + 1];
    if constexpr (kForm >= kRow) {
      x0 = __fmul_rn(x0, t.s[2 * h]);
      x1 = __fmul_rn(x1, t.s[2 * h + 1]);
    }
    uint32_t hi, mid, lo;
    SplitBf16Pair(x0, x1, hi, mid, lo);
    ah[h] = hi;
    am[h] = mid;
    al[h] = lo;
  }
  u32x4 bw[V];
#pragma unroll
  for (int c = 0; c < V; ++c)
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float w0 = ByteToFloat(t.w[2 * h][c >> 2], c & 3), w1 = ByteToFloat(t.w[2 * h + 1][c >> 2], c & 3);
      if constexpr (kForm == kZero) {
        w0 -= zc[c];
        w1 -= zc[c];
      } else if constexpr (kForm == kRowZero) {
        w0 -= static_cast<float>(t.z[2 * h]);
        w1 -= static_cast<float>(t.z[2 * h + 1]);
      }
      bw[c][h] = PackBf16(w0, w1);
    }
#pragma unroll
  for (int c = 0; c < V; ++c)
    acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ah), __builtin_bit_cast(bf16x8, bw[c]),
                                                     acc[c], 0, 0, 0);
#pragma unroll
  for (int c = 0; c < V; ++c)
    rest[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, am), __builtin_bit_cast(bf16x8, bw[c]),
                                                      rest[c], 0, 0, 0);
#pragma unroll
  for (int c = 0; c < V; ++c)
    rest[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, al), __builtin_bit_cast(bf16x8, bw[c]),
                                                      rest[c], 0, 0, 0);
}

// The same block in plain fp32: row 8g + u of it is k slot g of MFMA u.
template <int V, int kForm>
__device__ __forceinline__ void MultiplyPlain(const Block<V, kForm>& t, const float (&zc)[V], v4f (&acc)[V]) {
#pragma unroll
  for (int u = 0; u < 8; ++u)
#pragma unroll
    for (int c = 0; c < V; ++c) {
      float w = ByteToFloat(t.w[u][c >> 2], c & 3);
      if constexpr (kForm == kZero) w -= zc[c];
      if constexpr (kForm == kRowZero) w -= static_cast<float>(t.z[u]);
      if constexpr (kForm >= kRow) w = __fmul_rn(w, t.s[u]);
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.x[u], w, acc[c], 0, 0, 0);
    }
}

// The wave's sums over its blocks of the split in plain fp32, for the group of columns from col0.
template <int V, int kForm>
__device__ void PlainSums(const int8_t* q, const float* a, const Q8InPlaceArgs& p, int32_t m, int32_t k, int32_t kb,
                          int64_t n, int64_t col0, int rows, int wave, int lane, v4f (&acc)[V]) {
  const int slot = lane & 15, g = lane >> 4;
  const int64_t col = min(col0 + V * slot, n - V);
  const int8_t* qcol = q + kb * n + col;
  const float* arow = a + static_cast<int64_t>(slot < m ? slot : m - 1) * k + kb;
  float zc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    zc[j] = kForm == kZero ? static_cast<float>(p.zero[p.mode == kScalePerCol ? col + j : p.const_index]) : 0.f;
  }
  const int whole = rows / kBlockRows;
  for (int i = wave; i < whole; i += kWaves) {
    Block<V, kForm> t;
    LoadBlock<V, kForm>(qcol, arow, p, kb, n, i * kBlockRows + 8 * g, t);
    MultiplyPlain<V, kForm>(t, zc, acc);
  }
  if (rows % kBlockRows != 0 && wave == whole % kWaves) {
    Block<V, kForm> t;
    LoadTail<V, kForm>(qcol, arow, p, kb, n, whole * kBlockRows + 8 * g, rows, t);
    MultiplyPlain<V, kForm>(t, zc, acc);
  }
}

// The rows (bit i) of A[m, k] at `a` that hold an activation in this thread's k of [kb, kb + rows) which is
// not zero and, times its row scale where there is one, below 2^-110.
template <int kForm>
__device__ uint32_t TinyRows(const float* a, const Q8InPlaceArgs& p, int32_t m, int32_t k, int32_t kb, int32_t rows,
                             int tid) {
  uint32_t tiny = 0;
#pragma unroll 1
  for (int r = kb + tid; r < kb + rows; r += 64 * kWaves) {
    const float s = kForm >= kRow ? p.scale[r] : 1.f;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = a[static_cast<int64_t>(min(i, m - 1)) * k + r];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      uint32_t u = __float_as_uint(x[i]) << 1;
      if constexpr (kForm >= kRow) u = u == 0 || s == 0.f ? 0 : max(__float_as_uint(__fmul_rn(x[i], s)) << 1, 1u);
      if (u - 1 < (uint32_t(127 - 110) << 24) - 1) tiny |= 1u << i;
    }
  }
  return tiny;
}

// Workgroups of a grid's first dimension at most: a dimension holds less than 2^32 threads.
constexpr uint32_t kGridX = uint32_t(1) << 22;

// What the first loads need leads the arguments (preloaded into SGPRs at wave launch). Grid: a
// multiple of 8 workgroups; those of one XCD (blockIdx.x % 8) take consecutive
// (column group, split) pairs, so the splits of a group meet in one L2. Up to V = 4 two workgroups
// share a CU (at most 128 VGPRs; the compiler would take 132 to 152).
template <int V, int kForm>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(V <= 4 ? 4 : 2))) void GemvQ8InPlaceKernel(const int8_t* q, const float* a, float* partials,
                                                              uint32_t* arrivals, int32_t m, int32_t k, int32_t rows_per_split,
                                                              int32_t splits, int32_t pairs, int64_t n, Q8InPlaceArgs p) {
  constexpr int kCols = 16 * V;
  constexpr int kThreads = 64 * kWaves;
  __shared__ float red[kWaves][16][17 * V];  // column V * slot + j of a group at 17 * j + slot
  __shared__ bool is_last;
  __shared__ uint32_t again[2];  // rows to sum again; rows with a sum below 2^-64
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = lane & 15;
  const int g = lane >> 4;
  if (tid == 0) again[0] = again[1] = 0;
  const uint32_t per_xcd = (static_cast<uint32_t>(pairs) + kXcds - 1) / kXcds;
  const uint32_t b = blockIdx.y * kGridX + blockIdx.x;  // one row of workgroups, but for huge n
  const int pair = static_cast<int>(b % kXcds * per_xcd + b / kXcds);
  if (b / kXcds >= per_xcd || pair >= pairs) return;
  const int group = pair / splits;
  const int split = pair - group * splits;
  const int kb = split * rows_per_split;
  const int rows = min(k, kb + rows_per_split) - kb;
  // A run past the last column reads the last V columns instead; the store leaves the columns
  // before its own start to the lanes that own them.
  const int64_t col = min(static_cast<int64_t>(group) * kCols + V * slot, n - V);
  const int8_t* qcol = q + kb * n + col;
  const float* arow = a + static_cast<int64_t>(slot < m ? slot : m - 1) * k + kb;

  v4f acc[V], rest[V];  // sums of the hi parts, and of the mid and lo parts
  float zc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    acc[j] = rest[j] = v4f{0.f, 0.f, 0.f, 0.f};
    zc[j] = 0.f;
  }
  const int whole = rows / kBlockRows;  // whole blocks of the split; the wave takes wave, wave + W, ...
  if (wave < whole) {
    Block<V, kForm> t[2];
    LoadBlock<V, kForm>(qcol, arow, p, kb, n, wave * kBlockRows + 8 * g, t[0]);
    if constexpr (kForm == kZero) {
#pragma unroll
      for (int j = 0; j < V; ++j) zc[j] = static_cast<float>(p.zero[p.mode == kScalePerCol ? col + j : p.const_index]);
    }
    for (int i = wave;;) {
      if (i + kWaves < whole) LoadBlock<V, kForm>(qcol, arow, p, kb, n, (i + kWaves) * kBlockRows + 8 * g, t[1]);
      __builtin_amdgcn_sched_barrier(0);
      Multiply<V, kForm>(t[0], zc, acc, rest);
      i += kWaves;
      if (i >= whole) break;
      if (i + kWaves < whole) LoadBlock<V, kForm>(qcol, arow, p, kb, n, (i + kWaves) * kBlockRows + 8 * g, t[0]);
      __builtin_amdgcn_sched_barrier(0);
      Multiply<V, kForm>(t[1], zc, acc, rest);
      i += kWaves;
      if (i >= whole) break;
    }
  }
  if (rows % kBlockRows != 0 && wave == whole % kWaves) {
    Block<V, kForm> t;
    LoadTail<V, kForm>(qcol, arow, p, kb, n, whole * kBlockRows + 8 * g, rows, t);
    if constexpr (kForm == kZero) {
#pragma unroll
      for (int j = 0; j < V; ++j) zc[j] = static_cast<float>(p.zero[p.mode == kScalePerCol ? col + j : p.const_index]);
    }
    Multiply<V, kForm>(t, zc, acc, rest);
  }
  // Element r of MFMA j in lane l: row 4 * (l / 16) + r, column j of the lane's run.
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < V; ++j) red[wave][4 * g + r][17 * j + slot] = acc[j][r] + rest[j][r];
  __syncthreads();

  // Thread: one column of the group, rows tid / kCols + e * kStep. Column c of the group is matrix
  // column min(run start, n - V) + c % V, stored here when it is not before the run's own start.
  constexpr int kStep = kThreads / kCols < 16 ? kThreads / kCols : 16;
  constexpr int kPer = 16 / kStep;
  const int c = tid % kCols;
  const int i0 = min(tid / kCols, 15);
  const int64_t own = static_cast<int64_t>(group) * kCols + c / V * V;
  const int64_t out_col = min(own, n - V) + c % V;
  const bool live_col = out_col >= own && tid / kCols < 16;
  float sum[kPer];
  const auto wave_sum = [&](int e) {
    const int at = 17 * (c % V) + c / V;
    float s = red[0][i0 + e * kStep][at];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) s = s + red[v][i0 + e * kStep][at];
    return s;
  };
  uint32_t bad = 0, small = 0;  // rows of A
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int i = i0 + e * kStep;
    sum[e] = wave_sum(e);
    const uint32_t u = __float_as_uint(sum[e]) << 1;
    if (!live_col || i >= m) continue;
    if (u >= 0xff000000u || u - 1 < (uint32_t(127 - 110) << 24) - 1) bad |= 1u << i;
    if (u < uint32_t(127 - 64) << 24) small |= 1u << i;
  }
  if (bad != 0) atomicOr(&again[0], bad);
  if (small != 0) atomicOr(&again[1], small);
  __syncthreads();
  if ((again[0] | again[1]) != 0) {
    if (again[1] != 0) {
      const uint32_t tiny = TinyRows<kForm>(a, p, m, k, kb, rows, tid) & again[1];
      if (tiny != 0) atomicOr(&again[0], tiny);
      __syncthreads();
    }
    const uint32_t redo = again[0];
    if (redo != 0) {
      int tail = lane;
      // addresses made from it are not formed before the loop and kept through it
      if constexpr (kForm == kRowZero) asm("" : "+v"(tail));
      PlainSums<V, kForm>(q, a, p, m, k, kb, n, static_cast<int64_t>(group) * kCols, rows, wave, tail, acc);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < V; ++j) red[wave][4 * g + r][17 * j + slot] = acc[j][r];
      __syncthreads();
#pragma unroll
      for (int e = 0; e < kPer; ++e)
        if (redo >> (i0 + e * kStep) & 1u) sum[e] = wave_sum(e);
    }
  }
  if (splits > 1) {
    const int64_t block = static_cast<int64_t>(m) * n;
    float* mine = partials + split * block + out_col;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      const int i = i0 + e * kStep;
      if (live_col && i < m)
        __hip_atomic_store(&mine[i * n], sum[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) is_last = atomicAdd(&arrivals[group], 1u) == static_cast<uint32_t>(splits - 1);
    __syncthreads();
    if (!is_last) return;
    if (tid == 0) atomicExch(&arrivals[group], 0u);  // ready for the next launch
    // kChunk splits of all the thread's rows are requested at once (clamped to valid rows and
    // splits; the extra values are not used).
    constexpr int kChunk = kPer >= 8 ? 4 : 8;
    const float* part = partials + out_col;
    for (int sp0 = 0; sp0 < splits; sp0 += kChunk) {
      float v[kChunk][kPer];
#pragma unroll
      for (int f = 0; f < kChunk; ++f)
#pragma unroll
        for (int e = 0; e < kPer; ++e)
          v[f][e] = __hip_atomic_load(&part[min(sp0 + f, splits - 1) * block + min(i0 + e * kStep, m - 1) * n],
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int f = 0; f < kChunk; ++f)
#pragma unroll
        for (int e = 0; e < kPer; ++e)
          if (sp0 + f < splits) sum[e] = sp0 + f == 0 ? v[f][e] : sum[e] + v[f][e];
    }
  }
  if (!live_col) return;
  float cs = 1.f;
  if constexpr (kForm < kRow) cs = p.scale[p.mode == kScalePerCol ? out_col : p.const_index];
  // The residual and bias values of all the thread's rows are requested before the first store.
  float bias[kPer], res[kPer];
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int64_t i = min(i0 + e * kStep, m - 1);
    bias[e] = p.epi.bias != nullptr ? p.epi.bias[BiasIndex(p.epi, i, out_col)] : 0.f;
    res[e] = p.epi.residual != nullptr ? p.epi.residual[i * n + out_col] : 0.f;
  }
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int i = i0 + e * kStep;
    if (i < m)
      StoreC(p.c, i, out_col, n, p.epi,
             ApplyEpilogueLoaded(kForm < kRow ? __fmul_rn(sum[e], cs) : sum[e], p.epi, bias[e], res[e]));
  }
}

template <int V>
void LaunchForm(int form, dim3 grid, hipStream_t stream, const int8_t* q, const float* a, float* partials,
                uint32_t* arrivals, int32_t m, int32_t k, int32_t rows, int32_t splits, int32_t pairs, int64_t n,
                const Q8InPlaceArgs& args) {
  switch (form) {
#define ACCEL_Q8_INPLACE(F)                                                                                      \
  case F:                                                                                                        \
    hipLaunchKernelGGL((GemvQ8InPlaceKernel<V, F>), grid, dim3(64 * kWaves), 0, stream, q, a, partials, arrivals, \
                       m, k, rows, splits, pairs, n, args);                                                      \
    break;
    ACCEL_Q8_INPLACE(kNone) ACCEL_Q8_INPLACE(kZero) ACCEL_Q8_INPLACE(kRow) ACCEL_Q8_INPLACE(kRowZero)
#undef ACCEL_Q8_INPLACE
  }
}

}  // namespace

void LaunchGemvQ8InPlace(const float* a, const Q8View& b, float* c, int64_t m, int64_t k, int64_t n,
                         const Epilogue& epi, hipStream_t stream) {
  const Context& ctx = Ctx();
  const int64_t cus = ctx.cu_count > 0 ? ctx.cu_count : 256;
  if (m < 1 || m > 16 || k < 1 || n < 1 || k >= (int64_t(1) << 28) || n >= (int64_t(1) << 34))
    Fail(ACCEL_HIP_INVALID_ARGUMENT, "GEMV too large");
  // Bytes of a row a lane reads. Long runs use whole cache lines, short ones give a small matrix
  // enough workgroups without a split of K (m = 16: 576 x 3072 4.8 us at 2, 5.5 at 4, 7.6 at 8;
  // 4096 x 4096 9.4 at 4, 10.2 at 8; 3000 x 11000 15.8 at 4, 14.6 at 8; 4096 x 14336 20.3 at 4,
  // 17.7 at 8, 19.7 at 16).
  const int64_t elems = k * n;
  int v = elems >= (int64_t(27) << 20) ? 8 : elems >= (int64_t(4) << 20) ? 4 : 2;
  while (v > n) v /= 2;
  const int64_t groups = (n + 16 * v - 1) / (16 * v);
  // Workgroups in whole rounds: one a CU, two with the 64-column groups of a large matrix
  // (4096 x 4096 the same either way, 2048 x 4096 7.6 us with one, 8.3 with two; 2500 x 9000 13.6
  // with one, 11.1 with two); a few more than a round cost as much as another (128 columns, 3001 x
  // 10001: 13.3 us in 3 splits = 237 workgroups, 18.5 in 4). A split of fewer than 512 (256) rows
  // costs more in its exchange (about 1.5 us) than it saves (768 x 2048 5.0 us whole, 5.8 in two).
  const int64_t target = v == 4 && elems >= (int64_t(16) << 20) ? 2 * cus : cus;
  int64_t splits = std::max<int64_t>(1, std::min<int64_t>(target / groups, k / (v <= 2 ? 512 : 256)));
  const auto part_bytes = [&](int64_t s) { return static_cast<size_t>(s * m * n) * sizeof(float); };
  const size_t count_bytes = static_cast<size_t>(groups) * sizeof(uint32_t);
  if (splits > 1 && !ScratchReady(part_bytes(splits), kTempArrivals, count_bytes)) splits = 1;
  int64_t rows = (k + splits - 1) / splits;
  rows = (rows + kBlockRows - 1) / kBlockRows * kBlockRows;
  splits = (k + rows - 1) / rows;
  const int64_t pairs = groups * splits;
  if (pairs > 0x7ffffff0) Fail(ACCEL_HIP_INVALID_ARGUMENT, "GEMV too large");
  Q8InPlaceArgs args;
  args.scale = b.scale;
  args.zero = b.zero;
  args.mode = b.mode;
  args.const_index = b.const_index;
  args.c = c;
  args.epi = epi;
  float* partials = nullptr;
  uint32_t* arrivals = nullptr;
  if (splits > 1) {
    partials = static_cast<float*>(Workspace(part_bytes(splits)));
    arrivals = static_cast<uint32_t*>(Temp(kTempArrivals, count_bytes));
  }
  const uint32_t blocks = static_cast<uint32_t>((pairs + kXcds - 1) / kXcds * kXcds);
  const dim3 grid(std::min(blocks, kGridX), (blocks + kGridX - 1) / kGridX);
  const int form = b.mode == kScalePerRow ? (b.zero != nullptr ? kRowZero : kRow) : (b.zero != nullptr ? kZero : kNone);
  const int32_t m32 = static_cast<int32_t>(m), k32 = static_cast<int32_t>(k), rows32 = static_cast<int32_t>(rows);
  const int32_t splits32 = static_cast<int32_t>(splits), pairs32 = static_cast<int32_t>(pairs);
  const auto launch = v == 8 ? LaunchForm<8> : v == 4 ? LaunchForm<4> : v == 2 ? LaunchForm<2> : LaunchForm<1>;
  launch(form, grid, stream, b.q, a, partials, arrivals, m32, k32, rows32, splits32, pairs32, n, args);
  Check(hipGetLastError(), "GemvQ8InPlaceKernel launch");
}

}  // namespace accel_hip
