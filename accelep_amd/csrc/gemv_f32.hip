// fp32-weight GEMV: C[m, n] = A[m, k] @ B[k, n] (+ fused epilogue) for m <= 16, B fp32 row-major
// as Device::MatMul receives it (src/sim_device.cc:185-196): a decode step or batch on a model
// whose weights are not quantized.
//
// Bound: HBM. Algorithmic bytes per call = 4*(k*n + m*k + m*n); B is read once, in place.
//
//  * A workgroup owns 16 * V columns over one split of K; its waves take batches of 4 * U rows in
//    turn. Lane l reads V consecutive columns (slot l % 16) of U rows (group l / 16), so one
//    load of the wave covers four runs of 16 * V floats, and multiplies them with
//    v_mfma_f32_16x16x4f32: V MFMAs per load, whose k slot g is row U*g + u of the batch and
//    whose column l % 16 is the lane's own column j. The A operand of the U MFMA steps is
//    then U consecutive floats of row l % 16, read straight from A: no LDS stage, no lane
//    exchange, and the same work for any m <= 16 (rows past m repeat row m - 1; their sums
//    are not stored). On the VALU a 16-row product took 23 us for 4096 x 4096 (m * 4
//    multiply-adds per 16 bytes and the lanes' sums exchanged), here as long as a 1-row one.
//  * The next batch's loads are issued before the current batch is multiplied.
//  * The waves' sums are added through LDS in wave order. Where the columns alone leave CUs
//    idle, K is split: each workgroup stores its partial sums and the last one of a column
//    group to arrive adds them in split order (no second kernel).
//  * A decode row's RMSNorm or product with `up` may come in with it (F32Prologue): the row is
//    multiplied by the norm's weight (or by `up`) as it is read, every workgroup takes the row's
//    sum of squares again behind its first loads, and 1 / rms (and the gate's SiLU) is applied at
//    the store. A SmolLM2-135M layer's four products take 22.4 us so, 21.2 before beside 9.5 us of
//    norm and SiLU passes; 64-id prompt and 16 tokens 18.9 -> 15.7 ms.
#include "device_common.h"

#include <algorithm>

namespace accel_hip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kXcds = 8;

// V consecutive floats at a 4-byte aligned address (rows of an odd n start anywhere).
template <int V>
struct Run;
template <>
struct Run<1> {
  typedef float type __attribute__((ext_vector_type(1)));
};
template <>
struct Run<2> {
  typedef float type __attribute__((ext_vector_type(2), aligned(4)));
};
template <>
struct Run<4> {
  typedef float type __attribute__((ext_vector_type(4), aligned(4)));
};

// What a decode row (m = 1) has done to it on the way in (F32Prologue): nothing, the RMSNorm (times
// the norm's weight here, 1 / rms at the store), or the product with `up`.
enum In : int { kInNone = 0, kInRms = 1, kInMul = 2 };

struct GemvF32Args {
  float* c;
  Epilogue epi;
  float rms_eps;
  bool silu_split0;
};

// One batch of a wave: U rows of B per lane and the lane's U values of A (and of the operand they
// are multiplied by).
template <int V, int U, int kIn>
struct F32Batch {
  float w[U][V];
  float x[U];
  float y[kIn != kInNone ? U : 1];
};

template <int V, int U, bool kStream, int kIn>
__device__ __forceinline__ void LoadF32Batch(const float* bcol, const float* arow, const float* second, int32_t n,
                                             int32_t row, F32Batch<V, U, kIn>& t) {
  using R = typename Run<V>::type;
  using A4 = typename Run<4>::type;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const R* src = reinterpret_cast<const R*>(bcol + static_cast<int64_t>(row + u) * n);
    R v;
    if constexpr (kStream) v = __builtin_nontemporal_load(src);
    else v = *src;
#pragma unroll
    for (int j = 0; j < V; ++j) t.w[u][j] = v[j];
  }
#pragma unroll
  for (int u = 0; u < U; u += 4) {
    const A4 v = *reinterpret_cast<const A4*>(arow + row + u);
#pragma unroll
    for (int i = 0; i < 4; ++i) t.x[u + i] = v[i];
  }
  if constexpr (kIn != kInNone) {
#pragma unroll
    for (int u = 0; u < U; u += 4) {
      const A4 v = *reinterpret_cast<const A4*>(second + row + u);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.y[u + i] = v[i];
    }
  }
}

template <int V, int U, int kIn>
__device__ __forceinline__ void MultiplyF32Batch(const F32Batch<V, U, kIn>& t, v4f (&acc)[V]) {
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float x = kIn != kInNone ? __fmul_rn(t.x[u], t.y[u]) : t.x[u];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, t.w[u][j], acc[j], 0, 0, 0);
  }
}

// What the first loads need leads the arguments (preloaded into SGPRs at wave launch). Grid: one
// dimension, a multiple of 8 workgroups; those of one XCD (blockIdx.x % 8) take consecutive
// (column group, split) pairs, so the splits of a group meet in one L2.
template <int V, int W, int U, bool kStream, int kIn>
__global__ __launch_bounds__(64 * W) void GemvF32Kernel(const float* b, const float* a, float* partials,
                                                        uint32_t* arrivals, int32_t m, int32_t k, int32_t n,
                                                        int32_t rows_per_split, int32_t splits, int32_t pairs,
                                                        const float* second, GemvF32Args p) {
  constexpr int kCols = 16 * V;
  constexpr int kRows = 4 * U;  // rows of a batch
  __shared__ __align__(16) float red[W][16][kCols];
  __shared__ bool is_last;
  __shared__ double squares[kIn == kInRms ? W : 1];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = lane & 15;
  const int g = lane >> 4;
  const int per_xcd = static_cast<int>(gridDim.x / kXcds);
  const int pair = static_cast<int>(blockIdx.x % kXcds) * per_xcd + static_cast<int>(blockIdx.x / kXcds);
  if (pair >= pairs) return;
  const int group = pair / splits;
  const int split = pair - group * splits;
  const int kb = split * rows_per_split;
  const int rows = min(k, kb + rows_per_split) - kb;
  // A run past the last column reads the last V columns instead; the store leaves the columns
  // before its own start to the lanes that own them.
  const int col = group * kCols + V * slot;
  const int colc = min(col, n - V);
  const float* bcol = b + static_cast<int64_t>(kb) * n + colc;
  const float* arow = a + static_cast<int64_t>(slot < m ? slot : m - 1) * k + kb;
  const float* yrow = kIn != kInNone ? second + kb : nullptr;

  // The whole row's values of this thread, for its sum of squares: every workgroup takes it again,
  // behind the loads of its first batch.
  constexpr int kSquares = kIn == kInRms ? static_cast<int>(kGemvPrologueMaxK) / (64 * W) : 1;
  float xs[kSquares];
  const auto load_row = [&] {
    if constexpr (kIn == kInRms) {
#pragma unroll
      for (int j = 0; j < kSquares; ++j) {
        const int i = tid + j * 64 * W;
        xs[j] = i < k ? a[i] : 0.f;
      }
    }
  };
  v4f acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
  const int whole = rows / kRows;  // whole batches of the split; the wave takes wave, wave + W, ...
  if (wave < whole) {
    F32Batch<V, U, kIn> t[2];
    LoadF32Batch<V, U, kStream, kIn>(bcol, arow, yrow, n, wave * kRows + U * g, t[0]);
    load_row();
    for (int i = wave;;) {
      if (i + W < whole) LoadF32Batch<V, U, kStream, kIn>(bcol, arow, yrow, n, (i + W) * kRows + U * g, t[1]);
      __builtin_amdgcn_sched_barrier(0);
      MultiplyF32Batch<V, U, kIn>(t[0], acc);
      i += W;
      if (i >= whole) break;
      if (i + W < whole) LoadF32Batch<V, U, kStream, kIn>(bcol, arow, yrow, n, (i + W) * kRows + U * g, t[0]);
      __builtin_amdgcn_sched_barrier(0);
      MultiplyF32Batch<V, U, kIn>(t[1], acc);
      i += W;
      if (i >= whole) break;
    }
  } else {
    load_row();
  }
  // The rows past the last whole batch, four at a time, by the waves that come next in turn. A
  // row past the end enters as 0 * 0.
  for (int r0 = whole * kRows + 4 * ((wave + W - whole % W) % W); r0 < rows; r0 += 4 * W) {
    const int r = r0 + g;
    float x = 0.f;
    float w[V];
#pragma unroll
    for (int j = 0; j < V; ++j) w[j] = 0.f;
    if (r < rows) {
      const typename Run<V>::type v = *reinterpret_cast<const typename Run<V>::type*>(bcol + static_cast<int64_t>(r) * n);
#pragma unroll
      for (int j = 0; j < V; ++j) w[j] = v[j];
      x = arow[r];
      if constexpr (kIn != kInNone) x = __fmul_rn(x, yrow[r]);
    }
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, w[j], acc[j], 0, 0, 0);
  }
  // Element r of MFMA j in lane l: row 4 * (l / 16) + r, column j of the lane's run.
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int j = 0; j < V; ++j) red[wave][4 * g + r][V * slot + j] = acc[j][r];
  if constexpr (kIn == kInRms) {
    double ss = 0;
#pragma unroll
    for (int j = 0; j < kSquares; ++j) ss += static_cast<double>(xs[j]) * static_cast<double>(xs[j]);
    ss = WaveButterfly(ss, [](double u, double v) { return u + v; });
    if (lane == 0) squares[wave] = ss;
  }
  __syncthreads();

  constexpr int kThreads = 64 * W;
  constexpr int kPer = (16 * kCols + kThreads - 1) / kThreads;  // outputs of a thread at m = 16
  float sum[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int t = tid + q * kThreads;
    sum[q] = 0.f;
    if (t < m * kCols) {
      const int i = t / kCols, c = t % kCols;
      float s = red[0][i][c];
#pragma unroll
      for (int v = 1; v < W; ++v) s = s + red[v][i][c];
      sum[q] = s;
    }
  }
  // Position c of the group's columns holds matrix column min(run start, n - V) + c % V, stored
  // here when it is not before the run's own start.
  const auto column = [&](int c) {
    const int own = group * kCols + c / V * V;
    const int at = min(own, n - V) + c % V;
    return at >= own ? at : -1;
  };
  if (splits > 1) {
    const int64_t block = static_cast<int64_t>(m) * n;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int t = tid + q * kThreads;
      const int at = column(t % kCols);
      if (t < m * kCols && at >= 0)
        __hip_atomic_store(&partials[split * block + static_cast<int64_t>(t / kCols) * n + at], sum[q],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) is_last = atomicAdd(&arrivals[group], 1u) == static_cast<uint32_t>(splits - 1);
    __syncthreads();
    if (!is_last) return;
    if (tid == 0) atomicExch(&arrivals[group], 0u);  // ready for the next launch
    constexpr int kChunk = 8;  // splits requested at once
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int t = tid + q * kThreads;
      const int at = column(t % kCols);
      if (t >= m * kCols || at < 0) continue;
      const float* src = partials + static_cast<int64_t>(t / kCols) * n + at;
      float s = 0.f;
      for (int sp0 = 0; sp0 < splits; sp0 += kChunk) {
        float v[kChunk];
#pragma unroll
        for (int e = 0; e < kChunk; ++e)
          v[e] = __hip_atomic_load(&src[min(sp0 + e, splits - 1) * block], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int e = 0; e < kChunk; ++e)
          if (sp0 + e < splits) s = sp0 + e == 0 ? v[e] : s + v[e];
      }
      sum[q] = s;
    }
  }
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int t = tid + q * kThreads;
    const int at = column(t % kCols);
    if (t >= m * kCols || at < 0) continue;
    float v = sum[q];
    if constexpr (kIn == kInRms) {
      double total = squares[0];
#pragma unroll
      for (int w = 1; w < W; ++w) total += squares[w];
      v = __fmul_rn(v, static_cast<float>(1.0 / sqrt(total / static_cast<double>(k) + static_cast<double>(p.rms_eps))));
    }
    v = ApplyEpilogue(v, t / kCols, at, n, p.epi);
    if constexpr (kIn == kInRms) {
      if (p.silu_split0 && at < p.epi.split[0]) v = __fdiv_rn(v, __fadd_rn(1.f, expf(-v)));
    }
    StoreC(p.c, t / kCols, at, n, p.epi, v);
  }
}

}  // namespace

namespace {

template <int V, int W, int U, int kIn>
void LaunchForm(bool stream_b, uint32_t grid, hipStream_t stream, const float* b, const float* a, float* partials,
                uint32_t* arrivals, int32_t m, int32_t k, int32_t n, int32_t rows, int32_t splits, int32_t pairs,
                const float* second, const GemvF32Args& args) {
  if (stream_b)
    hipLaunchKernelGGL((GemvF32Kernel<V, W, U, true, kIn>), dim3(grid), dim3(64 * W), 0, stream, b, a, partials,
                       arrivals, m, k, n, rows, splits, pairs, second, args);
  else
    hipLaunchKernelGGL((GemvF32Kernel<V, W, U, false, kIn>), dim3(grid), dim3(64 * W), 0, stream, b, a, partials,
                       arrivals, m, k, n, rows, splits, pairs, second, args);
}

}  // namespace

bool LaunchGemvF32(const float* a, const float* b, float* c, int64_t m, int64_t k, int64_t n, const Epilogue& epi,
                   hipStream_t stream, const F32Prologue* prologue) {
  // 32-bit rows and columns; a column run of up to 4 lies inside a row.
  if (m < 1 || m > 16 || n < 4 || k < 1 || k >= (int64_t(1) << 28) || n >= (int64_t(1) << 28)) return false;
  const Context& ctx = Ctx();
  const int64_t cus = ctx.cu_count > 0 ? ctx.cu_count : 256;
  // Columns a lane reads per row: long runs stream best where the matrix is large (4096 x 4096:
  // 15.9 us at 4, 15.8 at 2 with twice the partial sums at m = 16, 17.3 against 18.5 us), short
  // ones give a small matrix enough workgroups without a split of K (576 x 960: 3.9 us at 1,
  // 4.9 at 2, 6.1 at 4; 2048 x 2048 in splits: 7.2 / 7.4 / 8.0 us).
  const int64_t elems = k * n;
  const int v = elems >= (int64_t(12) << 20) ? 4 : elems >= (int64_t(6) << 20) ? 2 : 1;
  const int64_t groups = (n + 16 * v - 1) / (16 * v);
  // One workgroup per CU; a split of fewer than 384 rows costs more in its exchange (about 2 us)
  // than it saves (576 x 576: 4.1 us whole, 4.4 in two; 1536 x 576: 6.6 whole, 4.9 in four).
  int64_t splits = std::max<int64_t>(1, std::min<int64_t>((cus + groups - 1) / groups, k / 384));
  const auto part_bytes = [&](int64_t s) { return static_cast<size_t>(s * m * n) * sizeof(float); };
  const size_t count_bytes = static_cast<size_t>(groups) * sizeof(uint32_t);
  if (splits > 1 && !ScratchReady(part_bytes(splits), kTempArrivals, count_bytes)) splits = 1;
  int64_t rows = (k + splits - 1) / splits;
  rows = (rows + 15) / 16 * 16;
  splits = (k + rows - 1) / rows;
  const int64_t pairs = groups * splits;
  if (pairs > 0x7ffffff0) return false;
  GemvF32Args args;
  args.c = c;
  args.epi = epi;
  args.rms_eps = 0.f;
  args.silu_split0 = false;
  const float* second = nullptr;
  int in = kInNone;
  if (prologue != nullptr) {
    if (m != 1 || k > kGemvPrologueMaxK || (prologue->rms_weight == nullptr) == (prologue->mul_up == nullptr) ||
        (prologue->silu_split0 && (prologue->rms_weight == nullptr || epi.split[0] <= 0)))
      Fail(ACCEL_HIP_INVALID_ARGUMENT, "fp32 GEMV prologue needs m = 1, k <= 4096 and one input transform");
    in = prologue->rms_weight != nullptr ? kInRms : kInMul;
    second = in == kInRms ? prologue->rms_weight : prologue->mul_up;
    args.rms_eps = prologue->rms_eps;
    args.silu_split0 = prologue->silu_split0;
  }
  float* partials = nullptr;
  uint32_t* arrivals = nullptr;
  if (splits > 1) {
    partials = static_cast<float*>(Workspace(part_bytes(splits)));
    arrivals = static_cast<uint32_t*>(Temp(kTempArrivals, count_bytes));
  }
  const uint32_t grid = static_cast<uint32_t>((pairs + kXcds - 1) / kXcds * kXcds);
  // Streaming (nontemporal) loads of a matrix too large to stay in an XCD's 4 MB L2 beside others
  // (4096 x 4096: 15.9 us against 17.3 with plain loads; 576 x 576 repeated: 3.5 plain, 3.9).
  const bool stream_b = elems >= (int64_t(2) << 20);
  const int32_t m32 = static_cast<int32_t>(m), k32 = static_cast<int32_t>(k), n32 = static_cast<int32_t>(n);
  const int32_t r32 = static_cast<int32_t>(rows), s32 = static_cast<int32_t>(splits), p32 = static_cast<int32_t>(pairs);
#define ACCEL_GEMV_F32(V, U)                                                                                          \
  (in == kInRms ? LaunchForm<V, 8, U, kInRms> : in == kInMul ? LaunchForm<V, 8, U, kInMul> : LaunchForm<V, 8, U, kInNone>) \
  (stream_b, grid, stream, b, a, partials, arrivals, m32, k32, n32, r32, s32, p32, second, args)
  if (v == 4) ACCEL_GEMV_F32(4, 4);
  else if (v == 2) ACCEL_GEMV_F32(2, 4);
  else ACCEL_GEMV_F32(1, 8);
#undef ACCEL_GEMV_F32
  Check(hipGetLastError(), "GemvF32Kernel launch");
  return true;
}

}  // namespace accel_hip
