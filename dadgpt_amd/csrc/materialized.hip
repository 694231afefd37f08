// Row kernels of the materialized attention path (the [BH, S, S] probability matrix in HBM):
// the reference's own elementwise operators, and one-pass fusions of the chains it runs
// between its batched GEMMs (src/model.cpp:395-420 forward, :575-616 backward, :765-790
// decode).
//
// Every kernel works on whole rows, one wave per row at a time; a lane holds 4 consecutive
// columns of every 256 (one 16-byte piece), so each load instruction of a wave covers 1024
// contiguous bytes. Row maxima and sums are wave reductions on DPP. The matrices are fp32, as
// the reference's. Bound: HBM. Rows of up to 1,024 columns are read once into registers
// (kMaxPieces pieces a lane, or one column a lane up to kNarrow columns), several rows per wave
// so that enough bytes are in flight, and the causal kernels never read what lies past the
// diagonal; longer rows take the loop kernels, which pass over the row again for each reduction.
//
// Arithmetic order per element follows the reference's operators: scores are multiplied by
// the scale, then masked to -1e9 (src/model.cpp:407-408; cuda/gpu_ops.cu:476-525), the
// softmax subtracts the row max, exponentiates with expf and divides by the row sum
// (cuda/gpu_ops.cu:147-193), and the softmax backward is p * (dp - sum(dp * p))
// (cuda/gpu_ops.cu:542-563), masked, then scaled (src/model.cpp:601-607). Only the order of
// the row sums differs (a wave tree instead of a block tree).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "dropout.hpp"
#include "lanes.hpp"
#include "kernels.hpp"

namespace dadgpt {
namespace {

constexpr int kRowsPerBlock = 4;
constexpr float kMaskValue = -1e9f;  // cuda/gpu_ops.cu:482

// The wave's first row (a scalar; the host keeps row counts below 2^26), RPW rows per wave.
template <int RPW = 1>
__device__ __forceinline__ unsigned wave_row0() {
  return (blockIdx.x * kRowsPerBlock + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * RPW;
}

__device__ __forceinline__ float wave_max(float x) { return lanes::group_max<64>(x); }
__device__ __forceinline__ float wave_sum(float x) { return lanes::group_sum<64>(x); }
// The same for several rows side by side, step by step.
template <int N, typename F>
__device__ __forceinline__ void each(float (&x)[N], F f) {
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = f(x[i]);
}
template <int N>
__device__ __forceinline__ void wave_max_of(float (&x)[N]) {
  each(x, [](float v) { return fmaxf(v, lanes::dpp<lanes::kQuadXor1>(v)); });
  each(x, [](float v) { return fmaxf(v, lanes::dpp<lanes::kQuadXor2>(v)); });
  each(x, [](float v) { return fmaxf(v, lanes::dpp<lanes::kHalfMirror>(v)); });
  each(x, [](float v) { return fmaxf(v, lanes::dpp<lanes::kMirror>(v)); });
  each(x, [](float v) { return lanes::max_xor16(v); });
  each(x, [](float v) { return lanes::max_xor32(v); });
}
template <int N>
__device__ __forceinline__ void wave_sum_of(float (&x)[N]) {
  each(x, [](float v) { return v + lanes::dpp<lanes::kQuadXor1>(v); });
  each(x, [](float v) { return v + lanes::dpp<lanes::kQuadXor2>(v); });
  each(x, [](float v) { return v + lanes::dpp<lanes::kHalfMirror>(v); });
  each(x, [](float v) { return v + lanes::dpp<lanes::kMirror>(v); });
  each(x, [](float v) { return lanes::sum_xor16(v); });
  each(x, [](float v) { return lanes::sum_xor32(v); });
}

// Four floats at any 4-byte address: gfx950 loads and stores 16 bytes at dword alignment in one
// instruction, so rows of any length and offset move in the same pieces as aligned ones.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Columns c .. c+3 of a row of `cols` >= 4 columns (0 past the end), in two steps so that a
// kernel issues all its loads before it waits for one. load_raw never branches: the piece that
// crosses the row's end loads its last four columns instead (whole_piece moves those into
// place), and pieces past the one that holds column `last` load that one again.
__device__ __forceinline__ f32x4 load_raw(const float* row, int c, int last, int cols) {
  return *reinterpret_cast<const f32x4u*>(row + min(c, min(last & ~3, cols - 4)));
}
__device__ __forceinline__ f32x4 whole_piece(f32x4 v, int c, int cols) {
  if (cols % 4 != 0) {  // wave-uniform
    const int shift = c + 4 - cols;  // 1 to 3 for the piece that crosses the end
    if (shift > 0) {
      if (shift & 2) v = f32x4{v[2], v[3], 0.f, 0.f};
      if (shift & 1) v = f32x4{v[1], v[2], v[3], 0.f};
    }
  }
  return c < cols ? v : f32x4{0.f, 0.f, 0.f, 0.f};
}
// The same in one step, for any number of columns.
__device__ __forceinline__ f32x4 load_piece(const float* row, int c, int cols) {
  if (cols >= 4) return whole_piece(load_raw(row, c, cols - 1, cols), c, cols);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  for (int e = 0; e < 3; ++e)
    if (c + e < cols) v[e] = row[c + e];
  return v;
}
// load_piece and store_piece of rows without a crossing piece (WHOLE: the columns are a multiple
// of four), or of any row of at least four columns.
template <bool WHOLE>
__device__ __forceinline__ f32x4 load_cols(const float* row, int c, int cols) {
  if constexpr (WHOLE) return *reinterpret_cast<const f32x4u*>(row + c);
  return whole_piece(load_raw(row, c, cols - 1, cols), c, cols);
}
__device__ __forceinline__ void store_piece(float* row, int c, int cols, const f32x4& v) {
  if (c + 4 <= cols) {
    *reinterpret_cast<f32x4u*>(row + c) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 3; ++e)
    if (c + e < cols) row[c + e] = v[e];
}

template <bool WHOLE>
__device__ __forceinline__ void store_cols(float* row, int c, int cols, const f32x4& v) {
  if constexpr (WHOLE)
    *reinterpret_cast<f32x4u*>(row + c) = v;
  else
    store_piece(row, c, cols, v);
}

// What a softmax row sees of its input: the raw value (kPlain), scale then causal mask
// (kCausal: row r of a head is query r % S), or scale then a length mask (kLength: keys at or
// past lens[r / H] are masked; an empty cache gives a zero row). Columns at or past the row's
// limit hold kMaskValue whatever the input holds there, so they are not read.
enum RowMode { kPlain, kCausal, kLength };

template <int MODE>
__device__ __forceinline__ int row_limit(unsigned r, int cols, int S, const int* lens, int H) {
  if constexpr (MODE == kCausal) return (int)(r % (unsigned)S) + 1;
  if constexpr (MODE == kLength) {
    const int L = lens[r / (unsigned)H];
    return L < 0 ? 0 : (L > cols ? cols : L);
  }
  return cols;
}

// The maximum a row starts from: the reference's initial one (cuda/gpu_ops.cu:156), and the
// masked columns' value where there are any.
__device__ __forceinline__ float initial_max(int limit, int cols) {
  return limit < cols ? kMaskValue : -1e30f;
}

// The weight of a masked column: 0 unless every visible score lies at the mask value's level
// (mx is the same in every lane).
__device__ __forceinline__ float masked_weight(float mx) {
  if (__builtin_amdgcn_readfirstlane(mx > 0.5f * kMaskValue)) return 0.f;
  return expf(kMaskValue - mx);
}

// x / sum as q = x inv, corrected once by its remainder (Markstein's division by a reciprocal;
// inv = 1 / sum): the quotient IEEE division gives wherever it and the remainder are normal, and
// within a unit in the last place of it below, in three operations per element. sum >= 1 or the
// row is degenerate (0 or NaN, which stays NaN).
__device__ __forceinline__ float divide(float x, float sum, float inv) {
  const float q = x * inv;
  return fmaf(fmaf(-q, sum, x), inv, q);
}

constexpr int kMaxPieces = 4;  // 16-byte pieces a lane holds of a register row (1,024 columns)

// Rows per wave of the register kernels: four pieces a lane in flight, fewer where that would
// leave CUs idle (the grid then has fewer than four waves for each of the 1,024 SIMDs).
int rows_per_wave(long long rows, int pieces) {
  int n = 4 / pieces;
  while (n > 1 && rows < 4096LL * n) n >>= 1;
  return n;
}

// Softmax of rows of at most 256 NP columns, RPW rows per wave, each read once. WHOLE: the
// columns are a multiple of four, so no piece crosses a row's end.
// [BH 192, S 256] (50 MB) causal, in place: 24-27 us with the looping kernel below (three
// passes, two exponentials per element), 17.7 us read once but reduced row after row (each
// reduction's twelve dependent steps waited out, every element selected three times), 16.4 us
// here; its 75 MB take 15 at the rate of a copy.
template <int MODE, int NP, int RPW, bool WHOLE>
__global__ __launch_bounds__(64 * kRowsPerBlock) void softmax_rows_reg_kernel(
    float* out, const float* in, unsigned rows, int cols, int S, float scale,
    const int* __restrict__ lens, int H) {
  const int c0 = 4 * (threadIdx.x & 63);
  const unsigned r0 = wave_row0<RPW>();
  if (r0 >= rows) return;
  f32x4 x[RPW][NP];
  int limit[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const unsigned r = min(r0 + i, rows - 1);
    limit[i] = row_limit<MODE>(r, cols, S, lens, H);
#pragma unroll
    for (int n = 0; n < NP; ++n)
      x[i][n] = load_raw(in + (size_t)r * cols, c0 + 256 * n, max(limit[i] - 1, 0), cols);
  }
  // Masked columns become -inf, which exponentiates to 0; whatever a piece's other columns hold
  // (past the row's end, or past the last visible piece) does too. The rows' reductions run side
  // by side: a single one waits out each of its twelve dependent steps.
  float mx[RPW], sum[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    mx[i] = initial_max(limit[i], cols);
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int c = c0 + 256 * n;
      if constexpr (!WHOLE) x[i][n] = whole_piece(x[i][n], c, cols);
      if constexpr (MODE != kPlain) x[i][n] *= scale;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[i][n][e] = c + e < limit[i] ? x[i][n][e] : neg_inf();
        mx[i] = fmaxf(mx[i], x[i][n][e]);
      }
    }
  }
  wave_max_of(mx);
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    sum[i] = 0.f;
#pragma unroll
    for (int n = 0; n < NP; ++n)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[i] += x[i][n][e] = expf(x[i][n][e] - mx[i]);
  }
  wave_sum_of(sum);
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (r0 + i >= rows) return;
    float* dst = out + (size_t)(r0 + i) * cols;
    const float masked = masked_weight(mx[i]);
    if (limit[i] < cols) sum[i] += (float)(cols - limit[i]) * masked;
    // no keys: a zero row (0 times a finite reciprocal)
    const float d = MODE == kLength && limit[i] == 0 ? 1.0f : sum[i], inv = 1.0f / d;
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      const int c = c0 + 256 * n;
      f32x4 v = x[i][n];
      if (masked != 0.f && limit[i] > 0) {  // wave-uniform, see masked_weight
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = c + e < limit[i] ? v[e] : masked;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = divide(v[e], d, inv);
      if (c < cols) store_cols<WHOLE>(dst, c, cols, v);
    }
  }
}

// Softmax of rows of at most kNarrow columns, one column a lane, RPW rows per wave: a 16-byte
// piece would leave most lanes without columns and cost every lane four exponentials. Bound: the
// instructions per row. 49,152 rows of 3 / 17 / 64 columns: 21.0 / 14.7 / 15.0 us in pieces,
// 7.4 / 7.6 / 8.7 us here.
constexpr int kNarrow = 64;
template <int MODE, int RPW>
__global__ __launch_bounds__(64 * kRowsPerBlock) void softmax_rows_narrow_kernel(
    float* out, const float* in, unsigned rows, int cols, int S, float scale,
    const int* __restrict__ lens, int H) {
  const int c = threadIdx.x & 63;
  const unsigned r0 = wave_row0<RPW>();
  if (r0 >= rows) return;
  float x[RPW], mx[RPW], sum[RPW];
  int limit[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const unsigned r = min(r0 + i, rows - 1);
    limit[i] = row_limit<MODE>(r, cols, S, lens, H);
    x[i] = in[(size_t)r * cols + min(c, max(limit[i] - 1, 0))];
  }
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if constexpr (MODE != kPlain) x[i] *= scale;
    x[i] = c < limit[i] ? x[i] : neg_inf();
    mx[i] = fmaxf(initial_max(limit[i], cols), x[i]);
  }
  wave_max_of(mx);
#pragma unroll
  for (int i = 0; i < RPW; ++i) sum[i] = x[i] = expf(x[i] - mx[i]);
  wave_sum_of(sum);
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (r0 + i >= rows) return;
    const float masked = masked_weight(mx[i]);
    if (limit[i] < cols) sum[i] += (float)(cols - limit[i]) * masked;
    // no keys: a zero row
    const float d = MODE == kLength && limit[i] == 0 ? 1.0f : sum[i];
    const float w = c < limit[i] || limit[i] == 0 ? x[i] : masked;
    if (c < cols) out[(size_t)(r0 + i) * cols + c] = divide(w, d, 1.0f / d);
  }
}

// Softmax of rows of any length: one row per wave, read again for each reduction.
template <int MODE, bool WHOLE>
__global__ __launch_bounds__(64 * kRowsPerBlock) void softmax_rows_kernel(
    float* out, const float* in, unsigned rows, int cols, int S,
    float scale, const int* __restrict__ lens, int H) {
  const int c0 = 4 * (threadIdx.x & 63);
  const unsigned r = wave_row0();
  if (r >= rows) return;
  const float* src = in + (size_t)r * cols;
  float* dst = out + (size_t)r * cols;
  const int limit = row_limit<MODE>(r, cols, S, lens, H);
  auto visible = [&](auto f) {  // f(piece of scaled values, its first column)
    for (int c = c0; c < limit; c += 256) {
      f32x4 v = load_cols<WHOLE>(src, c, cols);
      if constexpr (MODE != kPlain) v *= scale;
      f(v, c);
    }
  };
  float mx = initial_max(limit, cols);
  visible([&](const f32x4& v, int c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < limit) mx = fmaxf(mx, v[e]);
  });
  mx = wave_max(mx);
  float sum = 0.f;
  visible([&](const f32x4& v, int c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < limit) sum += expf(v[e] - mx);
  });
  const float masked = masked_weight(mx);
  sum = wave_sum(sum) + (limit < cols ? (float)(cols - limit) * masked : 0.f);
  const float inv = 1.0f / sum;
  const bool empty = MODE == kLength && limit == 0;
  // in == out is allowed: each lane writes exactly the columns it reads, after reading them
  for (int c = c0; c < cols; c += 256) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (c < limit) v = load_cols<WHOLE>(src, c, cols);
    if constexpr (MODE != kPlain) v *= scale;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = empty ? 0.f : divide(c + e < limit ? expf(v[e] - mx) : masked, sum, inv);
    store_cols<WHOLE>(dst, c, cols, v);
  }
}

// Softmax backward per row: g = p * (dp - sum_j dp_j p_j). ACCUMULATE: din += g (the
// reference's operator). Otherwise the attention form: din = g, zero past the causal
// diagonal, times scale (din may be dout). The sum runs over whole rows, whatever p holds past
// the diagonal. REG: rows of at most 256 NP columns, RPW rows per wave, each read once;
// otherwise (NP = RPW = 1) any length, the row read twice. WHOLE (read by the loop only): the
// columns are a multiple of four.
// [BH 192, S 256], 3 x 50 MB: 36 us with 4-byte loads in two passes, 24.5 us here
// (6.1 TB/s).
template <bool ACCUMULATE, bool REG, int NP, int RPW, bool WHOLE>
__global__ __launch_bounds__(64 * kRowsPerBlock) void softmax_backward_rows_kernel(
    float* din, const float* dout, const float* __restrict__ p, unsigned rows, int cols, int S,
    float scale) {
  const int c0 = 4 * (threadIdx.x & 63);
  const unsigned r0 = wave_row0<RPW>();
  if (r0 >= rows) return;
  auto row_dot = [](const f32x4& g, const f32x4& pr, float dot) {
#pragma unroll
    for (int e = 0; e < 4; ++e) dot += g[e] * pr[e];
    return dot;
  };
  auto finish = [&](unsigned r, int c, const f32x4& g, const f32x4& pr, float dot) {
    const int limit = ACCUMULATE ? cols : (int)(r % (unsigned)S) + 1;
    float* d = din + (size_t)r * cols;
    f32x4 v;
    if constexpr (ACCUMULATE) v = load_cols<WHOLE>(d, c, cols);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = pr[e] * (g[e] - dot);
      if constexpr (ACCUMULATE)
        v[e] += t;
      else
        v[e] = c + e < limit ? t * scale : 0.0f;
    }
    store_cols<WHOLE>(d, c, cols, v);
  };
  if constexpr (REG) {
    f32x4 g[RPW][NP], pr[RPW][NP];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const unsigned r = min(r0 + i, rows - 1);
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        g[i][n] = load_raw(dout + (size_t)r * cols, c0 + 256 * n, cols - 1, cols);
        pr[i][n] = load_raw(p + (size_t)r * cols, c0 + 256 * n, cols - 1, cols);
      }
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      if (r0 + i >= rows) return;
      float dot = 0.f;
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        g[i][n] = whole_piece(g[i][n], c0 + 256 * n, cols);
        pr[i][n] = whole_piece(pr[i][n], c0 + 256 * n, cols);
        dot = row_dot(g[i][n], pr[i][n], dot);
      }
      dot = wave_sum(dot);
#pragma unroll
      for (int n = 0; n < NP; ++n)
        if (c0 + 256 * n < cols) finish(r0 + i, c0 + 256 * n, g[i][n], pr[i][n], dot);
    }
  } else {
    const float *gr = dout + (size_t)r0 * cols, *prow = p + (size_t)r0 * cols;
    float dot = 0.f;
    for (int c = c0; c < cols; c += 256)
      dot = row_dot(load_cols<WHOLE>(gr, c, cols), load_cols<WHOLE>(prow, c, cols), dot);
    dot = wave_sum(dot);
    for (int c = c0; c < cols; c += 256)
      finish(r0, c, load_cols<WHOLE>(gr, c, cols), load_cols<WHOLE>(prow, c, cols), dot);
  }
}

// The same for rows of at most kNarrow columns, one column a lane.
template <bool ACCUMULATE, int RPW>
__global__ __launch_bounds__(64 * kRowsPerBlock) void softmax_backward_narrow_kernel(
    float* din, const float* dout, const float* __restrict__ p, unsigned rows, int cols, int S,
    float scale) {
  const int c = threadIdx.x & 63;
  const unsigned r0 = wave_row0<RPW>();
  if (r0 >= rows) return;
  float g[RPW], pr[RPW], dot[RPW];
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const size_t at = (size_t)min(r0 + i, rows - 1) * cols + min(c, cols - 1);
    g[i] = dout[at];
    pr[i] = p[at];
  }
#pragma unroll
  for (int i = 0; i < RPW; ++i) dot[i] = c < cols ? g[i] * pr[i] : 0.f;
  wave_sum_of(dot);
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    if (r0 + i >= rows) return;
    const int limit = ACCUMULATE ? cols : (int)((r0 + i) % (unsigned)S) + 1;
    float* d = din + (size_t)(r0 + i) * cols + c;
    const float t = pr[i] * (g[i] - dot[i]);
    if constexpr (ACCUMULATE) {
      if (c < cols) *d += t;
    } else {
      if (c < cols) *d = c < limit ? t * scale : 0.0f;
    }
  }
}

// scores[h][i][j] = value for j > i over n_blocks blocks of S x S.
__global__ void causal_fill_kernel(float* __restrict__ m, long long rows, int S, float value) {
  const long long r = (long long)blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (r >= rows) return;
  float* row = m + r * S;
  for (int c = (int)(r % S) + 1 + (threadIdx.x & 63); c < S; c += 64) row[c] = value;
}

__global__ void scale_kernel(float* __restrict__ x, long long n, float scale) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    x[i] *= scale;
}

// Attention-probability dropout on the materialized path, with the flash kernels' mask
// (dropout.hpp): element (r, c) of the [BH*S, S] probabilities is row r = bh*S + query and key
// c. Each lane owns 8 consecutive columns per step, whose keep bits are one Philox block.
struct Group8 {
  float v[8];
  __device__ __forceinline__ float& operator[](int e) { return v[e]; }
};
// WHOLE: the columns are a multiple of eight, so every group is whole.
template <bool WHOLE>
__device__ __forceinline__ Group8 load_group(const float* row, int c, int cols) {
  f32x4 a, b;
  if constexpr (WHOLE)
    a = load_cols<true>(row, c, cols), b = load_cols<true>(row, c + 4, cols);
  else
    a = load_piece(row, c, cols), b = load_piece(row, c + 4, cols);
  return Group8{{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}};
}
template <bool WHOLE>
__device__ __forceinline__ void store_group(float* row, int c, int cols, Group8& g) {
  store_cols<WHOLE>(row, c, cols, f32x4{g[0], g[1], g[2], g[3]});
  if (WHOLE || c + 4 < cols) store_cols<WHOLE>(row, c + 4, cols, f32x4{g[4], g[5], g[6], g[7]});
}

// out = p * keep / (1 - p_drop) (the reference's gpu_dropout_forward, cuda/gpu_ops.cu:712-733,
// with this mask). out may be p.
template <bool WHOLE>
__global__ __launch_bounds__(64 * kRowsPerBlock) void dropout_rows_kernel(
    float* out, const float* p, unsigned rows, int cols, DropParams dr) {
  const unsigned r = wave_row0();
  if (r >= rows) return;
  for (int c = 8 * (threadIdx.x & 63); c < cols; c += 512) {
    Group8 g = load_group<WHOLE>(p + (size_t)r * cols, c, cols);
    const uint32_t bits = keep8(dr, (uint64_t)r, (uint32_t)c >> 3);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] *= keep_factor(bits, e, dr.scale);
    store_group<WHOLE>(out + (size_t)r * cols, c, cols, g);
  }
}

// The attention backward's row pass with dropout (src/model.cpp:594-607): dP = dPd * keep /
// (1 - p_drop) (gpu_dropout_backward, cuda/gpu_ops.cu:736-749), then the softmax backward
// against the undropped P, zero past the causal diagonal, times scale. ds may be dpd. NG > 0:
// rows of at most 512 NG columns, read and their keep bits generated once; NG = 0: any length,
// both done again for the second pass.
template <int NG, bool WHOLE>
__global__ __launch_bounds__(64 * kRowsPerBlock) void attn_probs_backward_dropout_kernel(
    float* ds, const float* dpd, const float* __restrict__ p, unsigned rows, int S,
    float scale, DropParams dr) {
  const int c0 = 8 * (threadIdx.x & 63);
  const unsigned r = wave_row0();
  if (r >= rows) return;
  const float *gr = dpd + (size_t)r * S, *pr = p + (size_t)r * S;
  const int limit = (int)(r % (unsigned)S) + 1;
  auto undrop = [&](int c) {  // dP of the undropped probabilities
    Group8 g = load_group<WHOLE>(gr, c, S);
    const uint32_t bits = keep8(dr, (uint64_t)r, (uint32_t)c >> 3);
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] *= keep_factor(bits, e, dr.scale);
    return g;
  };
  auto row_dot = [](Group8& g, Group8& q, float dot) {
#pragma unroll
    for (int e = 0; e < 8; ++e) dot += g[e] * q[e];
    return dot;
  };
  auto finish = [&](int c, Group8& g, Group8& q, float dot) {
#pragma unroll
    for (int e = 0; e < 8; ++e) g[e] = c + e < limit ? q[e] * (g[e] - dot) * scale : 0.f;
    store_group<WHOLE>(ds + (size_t)r * S, c, S, g);
  };
  float dot = 0.f;
  if constexpr (NG > 0) {
    Group8 g[NG], q[NG];
#pragma unroll
    for (int n = 0; n < NG; ++n)
      if (c0 + 512 * n < S) {
        q[n] = load_group<WHOLE>(pr, c0 + 512 * n, S);
        g[n] = undrop(c0 + 512 * n);
        dot = row_dot(g[n], q[n], dot);
      }
    dot = wave_sum(dot);
#pragma unroll
    for (int n = 0; n < NG; ++n)
      if (c0 + 512 * n < S) finish(c0 + 512 * n, g[n], q[n], dot);
  } else {
    for (int c = c0; c < S; c += 512) {
      Group8 g = undrop(c), q = load_group<WHOLE>(pr, c, S);
      dot = row_dot(g, q, dot);
    }
    dot = wave_sum(dot);
    for (int c = c0; c < S; c += 512) {
      Group8 g = undrop(c), q = load_group<WHOLE>(pr, c, S);
      finish(c, g, q, dot);
    }
  }
}

// The head split and merge (cuda/gpu_ops.cu:426-474), a pure permutation between the
// token-major [B*S, H*dh] layout and [B*H, S, dh]. One workgroup per token row (b, s): its
// threads walk the row in W-float pieces (16 bytes when dh and both buffers allow), so the
// token-major side is one contiguous run and the head-major side one contiguous run of dh
// floats per head. MERGE runs the other direction.
template <bool MERGE, int W>
__global__ __launch_bounds__(256) void heads_kernel(float* __restrict__ out,
                                                    const float* __restrict__ in, int S, int H,
                                                    int dh) {
  using V = std::conditional_t<W == 4, f32x4, float>;
  const int row = blockIdx.x;  // b * S + s
  const int b = row / S, s = row - b * S;
  const int D = H * dh;
  const size_t tok = (size_t)row * D;
  for (int c = W * threadIdx.x; c < D; c += W * blockDim.x) {
    const int h = c / dh, x = c - h * dh;
    const size_t head = (((size_t)b * H + h) * S + s) * dh + x;
    const size_t src = MERGE ? head : tok + c, dst = MERGE ? tok + c : head;
    *reinterpret_cast<V*>(out + dst) = *reinterpret_cast<const V*>(in + src);
  }
}

template <bool MERGE>
hipError_t launch_heads(float* out, const float* in, int B, int S, int H, int dh,
                        hipStream_t stream) {
  const bool wide = dh % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(in) % 16 == 0;
  const int pieces = wide ? H * dh / 4 : H * dh;
  const int threads = std::min(256, (pieces + 63) / 64 * 64);
  const unsigned rows = (unsigned)((long long)B * S);
  if (wide)
    heads_kernel<MERGE, 4><<<rows, threads, 0, stream>>>(out, in, S, H, dh);
  else
    heads_kernel<MERGE, 1><<<rows, threads, 0, stream>>>(out, in, S, H, dh);
  return hipGetLastError();
}

unsigned row_blocks(long long rows) {
  return (unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock);
}

// f(pieces, rows per wave) as compile-time constants for rows of 4 to 1,024 columns.
template <typename F>
void with_row_shape(long long rows, int cols, F f) {
  using std::integral_constant;
  if (cols <= 256) {
    switch (rows_per_wave(rows, 1)) {
      case 4: return f(integral_constant<int, 1>{}, integral_constant<int, 4>{});
      case 2: return f(integral_constant<int, 1>{}, integral_constant<int, 2>{});
      default: return f(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    }
  }
  if (cols <= 512) {
    if (rows_per_wave(rows, 2) == 2)
      return f(integral_constant<int, 2>{}, integral_constant<int, 2>{});
    return f(integral_constant<int, 2>{}, integral_constant<int, 1>{});
  }
  return f(integral_constant<int, 4>{}, integral_constant<int, 1>{});
}

// f(rows per wave) as a compile-time constant for rows of at most kNarrow columns.
template <typename F>
void with_narrow_rows(long long rows, F f) {
  using std::integral_constant;
  switch (rows_per_wave(rows, 1)) {
    case 4: return f(integral_constant<int, 4>{});
    case 2: return f(integral_constant<int, 2>{});
    default: return f(integral_constant<int, 1>{});
  }
}

template <int MODE>
hipError_t launch_softmax(float* out, const float* in, long long rows, int cols, int S,
                          float scale, const int* lens, int H, hipStream_t stream) {
  auto run = [&](auto kernel, int rpw) {
    kernel<<<row_blocks((rows + rpw - 1) / rpw), 64 * kRowsPerBlock, 0, stream>>>(
        out, in, (unsigned)rows, cols, S, scale, lens, H);
  };
  const bool whole = cols % 4 == 0;
  if (cols <= kNarrow)
    with_narrow_rows(rows, [&](auto rpw) { run(softmax_rows_narrow_kernel<MODE, rpw()>, rpw()); });
  else if (cols > 256 * kMaxPieces)
    run(whole ? softmax_rows_kernel<MODE, true> : softmax_rows_kernel<MODE, false>, 1);
  else
    with_row_shape(rows, cols, [&](auto np, auto rpw) {
      run(whole ? softmax_rows_reg_kernel<MODE, np(), rpw(), true>
                : softmax_rows_reg_kernel<MODE, np(), rpw(), false>,
          rpw());
    });
  return hipGetLastError();
}

template <bool ACCUMULATE>
hipError_t launch_softmax_backward(float* din, const float* dout, const float* p, long long rows,
                                   int cols, int S, float scale, hipStream_t stream) {
  auto run = [&](auto kernel, int rpw) {
    kernel<<<row_blocks((rows + rpw - 1) / rpw), 64 * kRowsPerBlock, 0, stream>>>(
        din, dout, p, (unsigned)rows, cols, S, scale);
  };
  if (cols <= kNarrow)
    with_narrow_rows(rows, [&](auto rpw) {
      run(softmax_backward_narrow_kernel<ACCUMULATE, rpw()>, rpw());
    });
  else if (cols > 256 * kMaxPieces)
    run(cols % 4 == 0 ? softmax_backward_rows_kernel<ACCUMULATE, false, 1, 1, true>
                      : softmax_backward_rows_kernel<ACCUMULATE, false, 1, 1, false>,
        1);
  else
    with_row_shape(rows, cols, [&](auto np, auto rpw) {
      run(softmax_backward_rows_kernel<ACCUMULATE, true, np(), rpw(), false>, rpw());
    });
  return hipGetLastError();
}

}  // namespace

hipError_t launch_softmax_rows(float* out, const float* in, long long rows, int cols,
                               hipStream_t stream) {
  return launch_softmax<kPlain>(out, in, rows, cols, 1, 1.0f, nullptr, 1, stream);
}

hipError_t launch_softmax_backward_rows(float* din, const float* dout, const float* p,
                                        long long rows, int cols, hipStream_t stream) {
  return launch_softmax_backward<true>(din, dout, p, rows, cols, 1, 1.0f, stream);
}

hipError_t launch_causal_fill(float* m, int n_blocks, int S, float value, hipStream_t stream) {
  const long long rows = (long long)n_blocks * S;
  causal_fill_kernel<<<row_blocks(rows), 64 * kRowsPerBlock, 0, stream>>>(m, rows, S, value);
  return hipGetLastError();
}

hipError_t launch_scale(float* x, long long n, float scale, hipStream_t stream) {
  const long long blocks = (n + 255) / 256;
  scale_kernel<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, stream>>>(x, n, scale);
  return hipGetLastError();
}

hipError_t launch_attention_probs(float* p, int BH, int S, float scale, hipStream_t stream) {
  return launch_softmax<kCausal>(p, p, (long long)BH * S, S, S, scale, nullptr, 1, stream);
}

hipError_t launch_attention_probs_backward(float* ds, const float* dp, const float* p, int BH,
                                           int S, float scale, hipStream_t stream) {
  return launch_softmax_backward<false>(ds, dp, p, (long long)BH * S, S, S, scale, stream);
}

hipError_t launch_decode_probs(float* p, const int* lens, int n_seq, int H, int max_len,
                               float scale, hipStream_t stream) {
  return launch_softmax<kLength>(p, p, (long long)n_seq * H, max_len, 1, scale, lens, H,
                                 stream);
}

hipError_t launch_attention_dropout(float* out, const float* p, int BH, int S,
                                   const Dropout& drop, hipStream_t stream) {
  const long long rows = (long long)BH * S;
  const DropParams dr = drop_params(&drop);
  auto kernel = S % 8 == 0 ? dropout_rows_kernel<true> : dropout_rows_kernel<false>;
  kernel<<<row_blocks(rows), 64 * kRowsPerBlock, 0, stream>>>(out, p, (unsigned)rows, S, dr);
  return hipGetLastError();
}

hipError_t launch_attention_probs_backward_dropout(float* ds, const float* dpd, const float* p,
                                                   int BH, int S, float scale,
                                                   const Dropout& drop, hipStream_t stream) {
  const long long rows = (long long)BH * S;
  const DropParams dr = drop_params(&drop);
  auto run = [&](auto whole) {
    auto kernel = S <= 512    ? attn_probs_backward_dropout_kernel<1, whole()>
                  : S <= 1024 ? attn_probs_backward_dropout_kernel<2, whole()>
                              : attn_probs_backward_dropout_kernel<0, whole()>;
    kernel<<<row_blocks(rows), 64 * kRowsPerBlock, 0, stream>>>(ds, dpd, p, (unsigned)rows, S,
                                                                scale, dr);
  };
  if (S % 8 == 0)
    run(std::true_type{});
  else
    run(std::false_type{});
  return hipGetLastError();
}

hipError_t launch_split_heads(float* out, const float* in, int B, int S, int H, int dh,
                              hipStream_t stream) {
  return launch_heads<false>(out, in, B, S, H, dh, stream);
}

hipError_t launch_merge_heads(float* out, const float* in, int B, int S, int H, int dh,
                              hipStream_t stream) {
  return launch_heads<true>(out, in, B, S, H, dh, stream);
}

}  // namespace dadgpt
