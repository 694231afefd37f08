// fp32 causal flash attention at fp32 accuracy on gfx950. This is the reference's precision
// (cuda/attention.cu:1): forward with online softmax and a saved natural-log logsumexp, backward
// recomputing the probabilities from it. Every fp32 product runs on the bf16 matrix cores,
// each float split into three bf16 values and each product formed from the six cross terms
// that matter (see X3 below: as accurate as the fp32 MFMA, in 37% of its matrix time, and
// beside the VALU, which the fp32 MFMA of gfx950 does not run beside). The softmax
// exponentials are exp_acc (below: 1.24 ulp in six VALU operations, the library expf 0.85 in
// thirteen) and the logsumexp's logarithm is logf; results match float64 to ~1e-6 (O, lse)
// and the fp32 CPU path within its own rounding. The forward moves its running maximum lazily
// (as the bf16 forward does) and masking runs only where a chunk needs it.
//
// Work decomposition (every product a 32 x 32 MFMA tile, one wave per 32 rows):
//  forward  a wave owns 32 queries (lane l holds query l % 32): S^T = K Q^T over each 32-key
//           chunk with Q in registers (split once), the online softmax per lane, O^T += V^T P^T
//           with P split from the score registers (the K rows are read through sigma32, so
//           score registers 8j..8j+7 of lane half h are the MFMA k-slice of that half: no lane
//           exchange). K and V tiles are split once per workgroup as they are staged, into
//           three bf16 planes each in the bf16 kernels' swizzled layout, read with
//           ds_read_b128 (K rows) and ds_read_b64_tr_b16 (V^T);
//  dK/dV    a wave owns 32 keys (lane l holds key l % 32) and walks the later query chunks:
//           S = Q K^T and dP = dO V^T with K and V split once (in registers; at d_head 64 V's two
//           lower planes in LDS), Q and dO as bf16 planes, P and dS in registers, dV^T += dO^T P
//           and dK^T += Q^T dS (no atomics);
//  dQ       a wave owns 32 queries again: S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T, with
//           Q and dO split once and K, V as bf16 planes;
//  delta    rowsum(dO * O), computed by the backward's workgroups or, for long rows, by a pass of
//           its own.
// dK/dV and dQ are workgroups of one launch. One or two waves share a row group's chunks, by the
// size of the grid (fwd_waves_per_group, bwd_waves_per_group).
// The next tile is loaded while the current one is on the matrix cores and split into planes as
// it is stored: through registers in the forward; in dK/dV and dQ by direct loads into LDS,
// which leaves the registers to the split operands (splitting dO, K and V once instead of at
// each use: B16 H12 S1024 backward 606 -> 528 us, bit-identical).
//
// The DROP instantiations apply attention-probability dropout with the keep bits of
// dropout.hpp: the forward and dQ hold keys along registers (keep_words16), dK/dV holds queries
// along registers (keep_col16).
#include <type_traits>

#include "common.hpp"
#include "dropout.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include "tiles.hpp"

namespace dadgpt {
namespace {

// A workgroup is KG x KS waves: KG row groups of 32 rows (queries, or keys in dK/dV) it owns,
// and KS waves per group that share its chunks of the other dimension. The staged tile has
// 32 KS rows; wave (g, s) of a workgroup computes group g against the tile's chunk s, and the KS
// partial results are merged through LDS at the end.
constexpr int kGroups = 4;
constexpr int kRows = 32 * kGroups;  // rows a workgroup owns
// At most 256 registers a lane (two waves per SIMD; one runs the backward ~15% slower).
constexpr int wgs_per_cu(int ks) { return 2 / ks; }

// Row (within a 32-row chunk) that score register u of lane half h stands for, when the A
// operand rows were read through sigma32: 16 * (u / 8) + 8 * h + u % 8.
__device__ __forceinline__ constexpr int reg_row(int u, int h) {
  return 16 * (u >> 3) + 8 * h + (u & 7);
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.f;
  return z;
}

// e^x to ~1.3 ulp (measured over [-87, 44] against double exp: 1.24 ulp, the library expf
// 0.85) in six VALU operations instead of the library's thirteen: x log2(e) as a rounded
// product e plus its exact remainder r (an FMA, with log2(e) split into two floats), then
// 2^e on the hardware exp2 and the first-order correction 2^(e+r) = 2^e (1 + r ln 2). Results
// below 2^-126 flush to zero and above 2^128 are +inf (no range reduction): the softmax
// weights these kernels exponentiate are either negligible there or take the rescaling path.
// An infinite x gives NaN (its remainder is inf - inf): callers keep -inf out.
__device__ __forceinline__ float exp_acc(float x) {
  constexpr float kL1 = 1.44269502162933349609375f;  // log2(e) rounded to float
  constexpr float kL2 = 1.925963033500011079e-08f;   // log2(e) - kL1
  const float e = x * kL1;
  const float r = fmaf(x, kL2, fmaf(x, kL1, -e));
  const float p = __builtin_amdgcn_exp2f(e);
  return fmaf(p, r * kLn2, p);
}

// A chunk whose weights reach this in some row moves that row's running maximum: with
// weights below 2^64, the running sums stay far inside fp32 range over any sequence length.
constexpr float kMaxW = 0x1p64f;

constexpr int kPitchPad = 4;  // epilogues stage rows of D floats at a pitch of D + 4

// A TR-row fp32 tile and its register prefetch by NT threads, TR*D/(4 NT) 16-byte pieces each;
// rows at or past S read as zeros.
template <int D, int TR, int NT>
struct Tile {
  static constexpr int kPieces = TR * D / 4 / NT;
  static constexpr int kThreads = NT;
  f32x4 r[kPieces];

  __device__ __forceinline__ void load(const float* src, int row0, int S) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int u = threadIdx.x + NT * i, row = u / (D / 4), c = u % (D / 4);
      r[i] = row0 + row < S ? *reinterpret_cast<const f32x4*>(src + (size_t)(row0 + row) * D +
                                                              4 * c)
                            : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ f32x4 piece(int i) const { return r[i]; }
};

// The same tile prefetched through LDS instead of registers: each lane's pieces travel by direct
// global -> LDS loads into the lane's own 16-byte slots, so a wave reads back only what it
// loaded itself and needs no barrier, just its own wait. Rows at or past S read row S-1.
template <int D, int TR, int NT>
struct RawTile {
  static constexpr int kPieces = TR * D / 4 / NT;
  static constexpr int kThreads = NT;
  const float* src;
  float* lds;  // TR * D floats
  int S, wave, lane;
  __device__ __forceinline__ void issue(int row0) const {
    const int left = S - 1 - row0;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int u = NT * i + 64 * wave + lane, row = u / (D / 4), c = u % (D / 4);
      dma_lds16_sbase(src + (size_t)row0 * D, (uint32_t)(min(row, left) * D + 4 * c) * 4u,
                      lds + 4 * (NT * i + 64 * wave));
    }
  }
  __device__ __forceinline__ f32x4 piece(int i) const {
    return *reinterpret_cast<const f32x4*>(lds + 4 * (NT * i + 64 * wave + lane));
  }
};

// fp32 products on the bf16 matrix cores. A float x is split into three bf16 values
// x = x1 + x2 + x3 (each the round-to-nearest of what the previous ones leave, so the three
// carry 24 significant bits and the rest is below 2^-27 |x|); a product x y is then the six
// cross terms whose weight is at least 2^-18 (x1y1, x1y2, x2y1, x1y3, x3y1, x2y2), each exact
// in fp32 and summed by the MFMA in fp32. Six v_mfma_f32_32x32x16_bf16 (32 cycles each) do
// the work of eight v_mfma_f32_32x32x2_f32 (64 cycles each), and, unlike the fp32 MFMA, they
// run beside the VALU. Measured over random 32x32x64 products: largest error 2.5e-7 of
// sum |x_k y_k|, against 3.5e-7 for the fp32 MFMA.
struct X3 {
  bf16x8 v[3];
};

// pack_bf16x2 for a word whose halves are taken apart again: opaque, because the compiler would
// otherwise convert the low half a second time instead of shifting it out of the word (48 of
// dK/dV's 576 VALU instructions per chunk). ONCE = false leaves the compiler the second
// conversion, which does not wait for the first: shorter for a wave that has its SIMD to itself.
template <bool ONCE = true>
__device__ __forceinline__ uint32_t pack_once(float lo, float hi) {
  uint32_t w = pack_bf16x2(lo, hi);
  if constexpr (ONCE) asm("" : "+v"(w));
  return w;
}

template <bool ONCE = true>
__device__ __forceinline__ X3 split3(const float (&x)[8]) {
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a0 = x[2 * i], a1 = x[2 * i + 1];
    const uint32_t p = pack_once<ONCE>(a0, a1);
    const float b0 = a0 - bf16_lo(p), b1 = a1 - bf16_hi(p);  // exact
    const uint32_t q = pack_once<ONCE>(b0, b1);
    const float c0 = b0 - bf16_lo(q), c1 = b1 - bf16_hi(q);  // exact
    w[0][i] = p;
    w[1][i] = q;
    w[2][i] = pack_bf16x2(c0, c1);
  }
  return X3{{as_bf16x8(w[0]), as_bf16x8(w[1]), as_bf16x8(w[2])}};
}

// acc += A B over a 16-deep slice, A and B as X3 (smallest terms first).
__device__ __forceinline__ f32x16 mfma_x6(const X3& a, const X3& b, f32x16 acc) {
  acc = mfma32(a.v[1], b.v[1], acc);
  acc = mfma32(a.v[2], b.v[0], acc);
  acc = mfma32(a.v[0], b.v[2], acc);
  acc = mfma32(a.v[1], b.v[0], acc);
  acc = mfma32(a.v[0], b.v[1], acc);
  return mfma32(a.v[0], b.v[0], acc);
}

// A 64-row tile split into three bf16 planes in LDS, each in the row-major swizzled layout of
// the bf16 kernels (tiles.hpp), so the score operands are ds_read_b128 and the transposed
// ones ds_read_b64_tr_b16 reads. Each float is split once per workgroup, when the tile is
// staged, instead of once per wave that reads it.
template <int D, int TR, typename T>
__device__ __forceinline__ void store_x3(const T& t, bf16* planes) {
#pragma unroll
  for (int i = 0; i < T::kPieces; ++i) {
    const int u = threadIdx.x + T::kThreads * i, row = u / (D / 4), c = u % (D / 4);
    const int off = rm_off<D>(row, c >> 1) + 4 * (c & 1);  // 4 floats: half a 16-byte chunk
    const f32x4 x = t.piece(i);
    uint32_t w[3][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float a0 = x[2 * k], a1 = x[2 * k + 1];
      const uint32_t p = pack_once(a0, a1);
      const float b0 = a0 - bf16_lo(p), b1 = a1 - bf16_hi(p);
      const uint32_t q = pack_once(b0, b1);
      w[0][k] = p;
      w[1][k] = q;
      w[2][k] = pack_bf16x2(b0 - bf16_lo(q), b1 - bf16_hi(q));
    }
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
      *reinterpret_cast<u32x2*>(planes + pl * TR * D + off) = u32x2{w[pl][0], w[pl][1]};
  }
}

// The B operand of a score product from a global row: lane half h supplies columns
// 16 ds + 8 h + 0..7 of `row`, split into three bf16 planes.
template <int D, bool ONCE = true>
__device__ __forceinline__ void load_split_row(X3 (&x)[D / 16], const float* row, int h) {
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) {
    float a[8];
    const f32x4 v0 = *reinterpret_cast<const f32x4*>(row + 16 * ds + 8 * h);
    const f32x4 v1 = *reinterpret_cast<const f32x4*>(row + 16 * ds + 8 * h + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = v0[e], a[4 + e] = v1[e];
    x[ds] = split3<ONCE>(a);
  }
}

template <int D, int TR>
__device__ __forceinline__ f32x16 score_tile_p(const bf16* planes, int chunk_row0,
                                               const X3 (&qb)[D / 16], int lane) {
  const int krow = chunk_row0 + sigma32(lane & 31), hi = lane >> 5;
  f32x16 acc = zero16();
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) {
    X3 a;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl)
      a.v[pl] = lds_op(planes + pl * TR * D, rm_off<D>(krow, 2 * ds + hi));
    acc = mfma_x6(a, qb[ds], acc);
  }
  return acc;
}

template <int D, int TR, bool ONCE = true>
__device__ __forceinline__ void accumulate_t_p(f32x16 (&acc)[D / 32], const bf16* planes,
                                               int chunk_row0, const f32x16& p, int lane) {
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = p[8 * j + e];
    const X3 pb = split3<ONCE>(x);
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      X3 a;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        a.v[pl] = lds_tr_op<D>(planes + pl * TR * D, chunk_row0 + 16 * j, 32 * db, lane);
      acc[db] = mfma_x6(a, pb, acc[db]);
    }
  }
}

// score_tile_p and accumulate_t_p at the start of `planes`, with the addresses from
// LaneLds (tiles.hpp): the dK/dV kernel's register relief. At D = 64 the kernel uses all 256: the
// one-wave instances without dropout and the two-wave ones with it keep one or two registers in
// scratch, the others none.
template <int D, int TR>
__device__ __forceinline__ f32x16 score_tile_px(const bf16* planes, const X3 (&b)[D / 16],
                                                const LaneLds& lo) {
  uint32_t ra[D / 16];
  row_addr_xor<D>(ra, lo.ro);
  f32x16 acc = zero16();
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) {
    X3 a;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) a.v[pl] = lds_row_at(planes + pl * TR * D, ra[ds]);
    acc = mfma_x6(a, b[ds], acc);
  }
  return acc;
}
// score_tile_px with the lower planes of the B operand in LDS (`blo`, by lane).
template <int D, int TR>
__device__ __forceinline__ f32x16 score_tile_pxl(const bf16* planes, const bf16x8 (&b0)[D / 16],
                                                 const bf16x8 (*blo)[2][64], int lane,
                                                 const LaneLds& lo) {
  uint32_t ra[D / 16];
  row_addr_xor<D>(ra, lo.ro);
  f32x16 acc = zero16();
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) {
    X3 a;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) a.v[pl] = lds_row_at(planes + pl * TR * D, ra[ds]);
    acc = mfma_x6(a, X3{{b0[ds], blo[ds][0][lane], blo[ds][1][lane]}}, acc);
  }
  return acc;
}
template <int D, int TR>
__device__ __forceinline__ void accumulate_t_px(f32x16 (&acc)[D / 32], const bf16* planes,
                                                const f32x16& p, const LaneLds& lo) {
  uint32_t ta[2][D / 32];
  tr_addr_xor<D>(ta, lo.tr);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = p[8 * j + e];
    const X3 pb = split3(x);
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      X3 a;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        a.v[pl] = lds_tr_at(planes + pl * TR * D + 16 * j * D, ta[0][db], ta[1][db]);
      acc[db] = mfma_x6(a, pb, acc[db]);
    }
  }
}

// Writes a wave's transposed accumulators (element r of lane (l32, h), block db: row l32 of
// the wave, column 32 db + c32_row(r, h)) as 32 contiguous rows of D floats through the wave's
// LDS slot `stage` (32 x (D + 4) floats), times `mul` (per lane).
template <int D>
__device__ __forceinline__ void store_rows_t(float* dst, int row0, int S,
                                             const f32x16 (&acc)[D / 32], float mul,
                                             float* stage, int lane) {
  const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      stage[l32 * (D + kPitchPad) + 32 * db + c32_row(r, h)] = acc[db][r] * mul;
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own LDS writes are done
  __builtin_amdgcn_wave_barrier();
  constexpr int kPieces = 32 * D / 4 / 64;
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const int u = lane + 64 * i, row = u / (D / 4), c = u % (D / 4);
    if (row0 + row < S)
      *reinterpret_cast<f32x4*>(dst + (size_t)(row0 + row) * D + 4 * c) =
          *reinterpret_cast<const f32x4*>(stage + row * (D + kPitchPad) + 4 * c);
  }
}

// ------------------------------------------------------------------------------ forward

// ONCE: the conversions of Q's and the weights' splits forced to happen once (pack_once).
template <int D, bool DROP, int KS, bool ONCE>
__global__ __launch_bounds__(64 * kGroups * KS, wgs_per_cu(KS)) void fwd_f32_kernel(
    float* __restrict__ out, float* __restrict__ lse, const float* __restrict__ q,
    const float* __restrict__ k, const float* __restrict__ v, int S, float scale,
    const DropParams dr) {
  constexpr int NT = 64 * kGroups * KS, TR = 64, CPT = 2 / KS;  // chunks per tile and wave
  // K and V tiles as three bf16 planes each; after the tile loop they hold the second waves'
  // partial results, then the epilogue's fp32 staging rows. With two waves per group there are
  // two sets (one workgroup has the CU's LDS to itself), see the tile loop.
  constexpr int kPlane = 3 * TR * D;
  __shared__ __attribute__((aligned(16))) bf16 planes[KS * 2 * kPlane];
  constexpr int kPart = (D / 32) * 1024 + 128;  // a partial: O, m and l (floats)
  constexpr int kStage = 32 * (D + kPitchPad);  // a wave's staged rows (floats)
  static_assert(4 * kPlane >= 4 * kGroups * (KS > 1 && kPart > kStage ? kPart : kStage),
                "partials and staging fit");
  const int bh = blockIdx.x;
  const int blk = gridDim.y - 1 - blockIdx.y;  // longest query blocks first
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar
  const int grp = wave % kGroups, sub = wave / kGroups;
  const size_t base = (size_t)bh * S * D;
  const int q0 = blk * kRows + 32 * grp;  // the wave's first query
  const int qi = q0 + l32;                // this lane's query
  const int last = min(S, (blk + 1) * kRows) - 1;  // the workgroup's last query
  const int n_tiles = last / TR + 1;

  X3 qb[D / 16];  // the lane's query row, split
  load_split_row<D, ONCE>(qb, q + base + (size_t)min(qi, S - 1) * D, h);
  f32x16 o[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) o[db] = zero16();
  float m = neg_inf(), lh = 0.f;  // running maximum; this lane half's sum of weights

  Tile<D, TR, NT> tk, tv;
  tk.load(k + base, 0, S);
  tv.load(v + base, 0, S);
  // Splits the loaded tile t into `to` and loads tile t + 1.
  auto stage = [&](int t, bf16* to) {
    store_x3<D, TR>(tk, to);
    store_x3<D, TR>(tv, to + kPlane);
    if (t + 1 < n_tiles) {
      tk.load(k + base, (t + 1) * TR, S);
      tv.load(v + base, (t + 1) * TR, S);
    }
  };
  auto compute = [&](int t, const bf16* skp) {
    const bf16* svp = skp + kPlane;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = KS == 1 ? i : sub;
      const int key0 = t * TR + 32 * c;
      if (key0 > q0 + 31) continue;  // wave-uniform: the whole chunk is in the future
      f32x16 s = score_tile_p<D, TR>(skp, 32 * c, qb, lane);
      // only the chunk whose first key is the wave's first query holds keys after a query
      // (or past S); waves are 32-query aligned, so it is the one with key0 == q0
      const bool diag = key0 == q0;
      // weights against the running maximum m as it stands (natural-log units)
      float w[16], ps;
      auto weights = [&](float mref) {
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = exp_acc(fmaf(s[u], scale, -mref));
        if (diag) {
#pragma unroll
          for (int u = 0; u < 16; ++u)
            if (key0 + reg_row(u, h) > qi) w[u] = 0.f;
        }
        ps = w[0];  // (0 + w[0] could not be folded: it maps -0 to +0)
#pragma unroll
        for (int u = 1; u < 16; ++u) ps += w[u];
      };
      weights(m);
      // The maximum moves only when a row's weights would reach 2^64 (or are inf/NaN: m is
      // -inf before a row's first chunk), compared on the bits (ps is +0, positive or NaN).
      // Both lane halves of a row take the row's decision, and only the rows that need it
      // move: the others rescale by exp(0) = 1 and recompute the same weights, so no row's
      // bits depend on another row.
      const bool need = __float_as_uint(ps) >= __float_as_uint(kMaxW);
      if (__builtin_amdgcn_ballot_w64(need) != 0) {  // wave-uniform
        float cm = neg_inf();
#pragma unroll
        for (int u = 0; u < 16; ++u)
          if (!(diag && key0 + reg_row(u, h) > qi)) cm = fmaxf(cm, s[u] * scale);
        // every row of a chunk the wave computes has a visible key: the row maximum is finite
        const float mn = or_halves(need) ? fmaxf(m, max_halves(cm)) : m;
        // 0 on a row's first chunk (exp_acc has no -inf input path)
        const float alpha = m == neg_inf() ? 0.f : exp_acc(m - mn);
        m = mn;
        lh *= alpha;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
        weights(m);
      }
      lh += ps;
      KeepWords16 keep = {};
      if constexpr (DROP) keep = keep_words16(dr, (uint64_t)bh * S + qi, key0, h);
#pragma unroll
      for (int u = 0; u < 16; ++u) s[u] = DROP ? w[u] * keep_factor(keep, u, dr) : w[u];
      accumulate_t_p<D, TR, ONCE>(o, svp, 32 * c, s, lane);
    }
  };
  if constexpr (KS == 1) {
    for (int t = 0; t < n_tiles; ++t) {
      __syncthreads();  // the previous tile's reads are done
      stage(t, planes);
      __syncthreads();
      compute(t, planes);
    }
  } else {
    // One barrier per tile: tile t is computed from one set while t + 1 is split into the other.
    // A SIMD holds one wave of each half, and the halves do the two in opposite order: in step,
    // both would be on the matrix cores and then both on the VALU.
    bf16 *set0 = planes, *set1 = planes + 2 * kPlane;
    stage(0, set0);
    __syncthreads();
    auto tile = [&](int t, bf16* cur, bf16* next) {
      if (sub == 1 && t + 1 < n_tiles) stage(t + 1, next);
      compute(t, cur);
      if (sub == 0 && t + 1 < n_tiles) stage(t + 1, next);
      __syncthreads();
    };
    for (int t = 0; t < n_tiles; t += 2) {
      tile(t, set0, set1);
      if (t + 1 < n_tiles) tile(t + 1, set1, set0);
    }
  }
  __syncthreads();  // every wave is done with the tiles: they hold partials and staging now
  constexpr int kSlot = KS > 1 && kPart > kStage ? kPart : kStage;
  float* slot = reinterpret_cast<float*>(planes) + grp * kSlot;
  if constexpr (KS == 2) {
    // (m, l, O) of the group's second wave: rescaled to the larger maximum and added. A wave
    // that saw no chunk has m = -inf and zeros, which get weight 0.
    float* ml = slot + (D / 32) * 1024;
    if (sub == 1) {
      put_acc(o, reinterpret_cast<AccLds*>(slot), lane);
      ml[lane] = m;
      ml[64 + lane] = lh;
    }
    __syncthreads();
    if (sub == 1) return;
    const float m1 = ml[lane], mn = fmaxf(m, m1);
    const float a0 = m == neg_inf() ? 0.f : exp_acc(m - mn);
    const float a1 = m1 == neg_inf() ? 0.f : exp_acc(m1 - mn);
    m = mn;
    lh = lh * a0 + ml[64 + lane] * a1;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] *= a0;
    add_acc(o, reinterpret_cast<const AccLds*>(slot), lane, a1);
    __builtin_amdgcn_wave_barrier();
  }
  const float l = sum_halves(lh);
  if (h == 0 && qi < S) lse[(size_t)bh * S + qi] = m + logf(l);
  store_rows_t<D>(out + base, q0, S, o, 1.0f / l, slot, lane);
}

// ----------------------------------------------------------------------------- backward

// delta[row] = sum_d dout[row][d] * out[row][d]: D/4 lanes per row, one 16-byte piece each;
// a grid-stride loop over rows (the lanes of a row share every trip, so the row's shuffles
// always see all of its lanes).
template <int D>
__global__ __launch_bounds__(256) void delta_f32_kernel(float* __restrict__ delta,
                                                        const float* __restrict__ dout,
                                                        const float* __restrict__ out,
                                                        long long rows) {
  constexpr int LPR = D / 4;
  const int c = threadIdx.x % LPR;
  const long long stride = (long long)gridDim.x * (256 / LPR);
  for (long long row = ((long long)blockIdx.x * 256 + threadIdx.x) / LPR; row < rows;
       row += stride) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(dout + row * D + 4 * c);
    const f32x4 b = *reinterpret_cast<const f32x4*>(out + row * D + 4 * c);
    float acc = a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3];
    acc = lanes::group_sum<LPR>(acc);
    if (c == 0) delta[row] = acc;
  }
}

// LDS of the backward kernels (bytes): two streamed tiles of 32 KS rows as three bf16 planes
// each, and raw; afterwards the partials and staging of the epilogue (`acc` accumulators a wave).
template <int D, int KS>
struct BwdLds {
  static constexpr int TR = 32 * KS, kPlane = 3 * TR * D;
  static constexpr int kBytes = 2 * kPlane * 2 + 2 * TR * D * 4;
  static constexpr int slot_floats(int acc) {
    const int stage = 32 * (D + kPitchPad), part = acc * 1024;
    return KS > 1 && part > stage ? part : stage;
  }
};

// What a backward kernel works on.
struct F32BwdArgs {
  float *dq, *dk, *dv, *delta;
  const float *q, *k, *v, *dout, *out, *lse;
  int S;
  float scale;
  DropParams dr;
};
// LDS of a workgroup: the tiles, and per query row of a dK/dV tile lse and delta * scale.
template <int D, int KS>
struct F32BwdShared {
  __attribute__((aligned(16))) char tiles[BwdLds<D, KS>::kBytes];
  __attribute__((aligned(16))) float sl[32 * KS], sd[32 * KS];
  // dK/dV at D = 64: the lower planes of the groups' V rows, by lane
  bf16x8 vlo[kGroups][D == 64 ? D / 16 : 1][2][64];
};

// delta of rows row0 .. S-1 into LDS, by the whole workgroup: D/4 lanes per row, one 16-byte
// piece each, four groups of rows in flight.
template <int D, int NT>
__device__ __forceinline__ void delta_rows(float* delta, const float* dout, const float* out,
                                           int row0, int S) {
  constexpr int LPR = D / 4, ROWS = NT / LPR, N = 4;
  const int c = threadIdx.x % LPR, lr = threadIdx.x / LPR;
  for (int b0 = row0; b0 < S; b0 += N * ROWS) {
    f32x4 g[N], o[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const size_t r = min(b0 + i * ROWS + lr, S - 1);
      g[i] = *reinterpret_cast<const f32x4*>(dout + r * D + 4 * c);
      o[i] = *reinterpret_cast<const f32x4*>(out + r * D + 4 * c);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float acc = g[i][0] * o[i][0] + g[i][1] * o[i][1] + g[i][2] * o[i][2] + g[i][3] * o[i][3];
      acc = lanes::group_sum<LPR>(acc);
      const int r = b0 + i * ROWS + lr;
      if (c == 0 && r < S) delta[r - row0] = acc;
    }
  }
}

// One workgroup's dK and dV. OWN_DELTA: delta is computed here, into own_delta (a float for each
// row from the first tile on); otherwise it is read from a.delta.
template <int D, bool DROP, int KS, bool OWN_DELTA>
__device__ __forceinline__ void dkdv_f32_workgroup(const F32BwdArgs& a, int bh, int blk,
                                                   F32BwdShared<D, KS>& sm, float* own_delta) {
  // Q and dO tiles: planes and raw
  using Lds = BwdLds<D, KS>;
  constexpr int TR = Lds::TR, NT = 64 * kGroups * KS;
  char* smem = sm.tiles;
  bf16 *sqp = reinterpret_cast<bf16*>(smem), *sgp = sqp + Lds::kPlane;
  float* raw = reinterpret_cast<float*>(sgp + Lds::kPlane);
  constexpr int kSlot = Lds::slot_floats(2 * (D / 32));
  static_assert(kGroups * kSlot * 4 <= Lds::kBytes, "partials and staging fit");
  float *sl = sm.sl, *sd = sm.sd;
  const float *q = a.q, *k = a.k, *v = a.v, *dout = a.dout, *lse = a.lse, *delta = a.delta;
  float *dk = a.dk, *dv = a.dv;
  const int S = a.S;
  const float scale = a.scale;
  const DropParams& dr = a.dr;
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar
  const int grp = wave % kGroups, sub = wave / kGroups;
  const size_t base = (size_t)bh * S * D;
  const int k0 = blk * kRows + 32 * grp;  // the wave's first key
  const int kj = k0 + l32;                // this lane's key
  const int t0 = (blk * kRows) / TR;  // first query tile with a query >= the first key
  const int n_tiles = (S + TR - 1) / TR;

  // The lane's K and V rows (score-product B layout), split. At D = 64 V's lower planes go to LDS,
  // which the two waves of a group share (published by the first barrier): with all six planes
  // in registers (96 of 256) the loop spilled and the compiler could not move the softmax under
  // the dP products (B16 H12 S1024 513 -> 498 us, with dropout B4 180 -> 153; at D = 32, where
  // they fit, the LDS reads cost 4%).
  constexpr bool kVLds = D == 64;
  X3 kb[D / 16], vb[D / 16];
  load_split_row<D>(kb, k + base + (size_t)min(kj, S - 1) * D, h);
  load_split_row<D>(vb, v + base + (size_t)min(kj, S - 1) * D, h);
  bf16x8 vb0[D / 16];
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) {
    vb0[ds] = vb[ds].v[0];
    if constexpr (kVLds) {
      if (sub == 0) sm.vlo[grp][ds][0][lane] = vb[ds].v[1], sm.vlo[grp][ds][1][lane] = vb[ds].v[2];
      asm volatile("" : "+v"(vb0[ds]));
    }
    // not to be split again inside the loop
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      asm volatile("" : "+v"(kb[ds].v[pl]));
      if constexpr (!kVLds) asm volatile("" : "+v"(vb[ds].v[pl]));
    }
  }
  f32x16 da[2 * (D / 32)];  // dV^T, then dK^T
  f32x16(&dva)[D / 32] = reinterpret_cast<f32x16(&)[D / 32]>(da[0]);
  f32x16(&dka)[D / 32] = reinterpret_cast<f32x16(&)[D / 32]>(da[D / 32]);
#pragma unroll
  for (int i = 0; i < 2 * (D / 32); ++i) da[i] = zero16();

  const LaneLds lo = lane_lds<D>(lane);
  const RawTile<D, TR, NT> tq{q + base, raw, S, wave, lane},
      tg{dout + base, raw + TR * D, S, wave, lane};
  float pl = 0.f, pd = 0.f;
  auto load_stats = [&](int row0) {
    const int r = row0 + (threadIdx.x & (TR - 1));
    pl = r < S ? lse[(size_t)bh * S + r] : 0.f;
    if constexpr (OWN_DELTA)
      pd = 0.f;  // read from own_delta as the tile is staged
    else
      pd = r < S ? delta[(size_t)bh * S + r] : 0.f;
  };
  tq.issue(t0 * TR);
  tg.issue(t0 * TR);
  load_stats(t0 * TR);
  if constexpr (OWN_DELTA)
    delta_rows<D, NT>(own_delta, dout + base, a.out + base, t0 * TR, S);
  for (int t = t0; t < n_tiles; ++t) {
    wait_vm_lds<0>();  // this wave's pieces of the tile
    __syncthreads();   // every wave is done with the previous tile's planes
    store_x3<D, TR>(tq, sqp);
    store_x3<D, TR>(tg, sgp);
    if (threadIdx.x < TR) {
      if constexpr (OWN_DELTA) pd = own_delta[min(t * TR + (int)threadIdx.x, S - 1) - t0 * TR];
      sl[threadIdx.x] = pl, sd[threadIdx.x] = pd * scale;
    }
    __syncthreads();
    if (t + 1 < n_tiles) {
      tq.issue((t + 1) * TR);
      tg.issue((t + 1) * TR);
      load_stats((t + 1) * TR);
    }
    const int qrow0 = t * TR + 32 * sub;
    // wave-uniform: every query of the chunk precedes every key, or lies past S
    if (qrow0 + 31 < k0 || (KS > 1 && qrow0 >= S)) continue;
    const bf16 *qc = sqp + 32 * sub * D, *gc = sgp + 32 * sub * D;
    // lane (l32, h), register u: query qrow0 + reg_row(u, h), key kj
    f32x16 s = score_tile_px<D, TR>(qc, kb, lo);   // Q K^T
    f32x16 dp;  // dO V^T
    if constexpr (kVLds)
      dp = score_tile_pxl<D, TR>(gc, vb0, sm.vlo[grp], lane, lo);
    else
      dp = score_tile_px<D, TR>(gc, vb, lo);
    uint32_t keep = 0;
    if constexpr (DROP) keep = keep_col16(dr, (uint64_t)bh * S + qrow0, k0, lane);
    // P in place of S, under the dP products: registers 8j..8j+7 are the 8 consecutive rows
    // 32 sub + 16j + 8h .., their statistics two 16-byte LDS reads each
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 ls =
          *reinterpret_cast<const f32x4*>(sl + 32 * sub + 16 * (g4 >> 1) + 8 * h + 4 * (g4 & 1));
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * g4 + e] = exp_acc(fmaf(s[4 * g4 + e], scale, -ls[e]));
    }
    // keys after a query, or rows past S, only where the chunk reaches the wave's first
    // keys or S (wave-uniform)
    if (qrow0 < k0 + 31 || qrow0 + 31 >= S) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int qrow = qrow0 + reg_row(u, h);
        s[u] = kj <= qrow && qrow < S ? s[u] : 0.f;
      }
    }
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 ds =
          *reinterpret_cast<const f32x4*>(sd + 32 * sub + 16 * (g4 >> 1) + 8 * h + 4 * (g4 & 1));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int u = 4 * g4 + e;
        const float p = s[u];
        float g = dp[u];
        if constexpr (DROP) {
          const float f = keep_factor(keep, u, dr.scale);
          g *= f;
          s[u] = p * f;  // the probability that multiplied V
        }
        dp[u] = p * fmaf(g, scale, -ds[e]);  // P (dP - delta) scale
      }
    }
    accumulate_t_px<D, TR>(dva, gc, s, lo);   // dV^T += dO^T P
    accumulate_t_px<D, TR>(dka, qc, dp, lo);  // dK^T += Q^T dS
  }
  __syncthreads();
  float* slot = reinterpret_cast<float*>(smem) + grp * kSlot;
  if constexpr (KS == 2) {
    if (sub == 1) put_acc(da, reinterpret_cast<AccLds*>(slot), lane);
    __syncthreads();
    if (sub == 1) return;
    add_acc(da, reinterpret_cast<const AccLds*>(slot), lane);
    __builtin_amdgcn_wave_barrier();
  }
  store_rows_t<D>(dk + base, k0, S, dka, 1.0f, slot, lane);
  store_rows_t<D>(dv + base, k0, S, dva, 1.0f, slot, lane);  // after the wave's dK reads
}

// One workgroup's dQ. OWN_DELTA: delta of its rows is computed here and written; otherwise read.
template <int D, bool DROP, int KS, bool OWN_DELTA>
__device__ __forceinline__ void dq_f32_workgroup(const F32BwdArgs& a, int bh, int blk,
                                                 F32BwdShared<D, KS>& sm) {
  // K and V tiles: planes and raw
  using Lds = BwdLds<D, KS>;
  constexpr int TR = Lds::TR, NT = 64 * kGroups * KS;
  char* smem = sm.tiles;
  bf16 *skp = reinterpret_cast<bf16*>(smem), *svp = skp + Lds::kPlane;
  float* raw = reinterpret_cast<float*>(svp + Lds::kPlane);
  constexpr int kSlot = Lds::slot_floats(D / 32);
  static_assert(kGroups * kSlot * 4 <= Lds::kBytes, "partials and staging fit");
  const float *q = a.q, *k = a.k, *v = a.v, *dout = a.dout, *lse = a.lse;
  float *dq = a.dq, *delta = a.delta;
  const int S = a.S;
  const float scale = a.scale;
  const DropParams& dr = a.dr;
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: scalar
  const int grp = wave % kGroups, sub = wave / kGroups;
  const size_t base = (size_t)bh * S * D;
  const int q0 = blk * kRows + 32 * grp;
  const int qi = q0 + l32;
  const int qc = min(qi, S - 1);
  const int last = min(S, (blk + 1) * kRows) - 1;
  const int n_tiles = last / TR + 1;

  X3 qb[D / 16], gb[D / 16];  // the lane's Q and dO rows (score-product B layout), split
  load_split_row<D>(qb, q + base + (size_t)qc * D, h);
  load_split_row<D>(gb, dout + base + (size_t)qc * D, h);
  const float my_lse = lse[(size_t)bh * S + qc];
  float my_delta;
  if constexpr (OWN_DELTA) {
    const float* g = dout + base + (size_t)qc * D + 8 * h;
    const float* o = a.out + base + (size_t)qc * D + 8 * h;
    float part = 0.f;
#pragma unroll
    for (int ds = 0; ds < D / 16; ++ds)
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(g + 16 * ds + e);
        const f32x4 y = *reinterpret_cast<const f32x4*>(o + 16 * ds + e);
        part += x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3];
      }
    my_delta = sum_halves(part);
    if (h == 0 && qi < S && sub == 0) delta[(size_t)bh * S + qi] = my_delta;
  } else {
    my_delta = delta[(size_t)bh * S + qc];
  }
  const float my_dscale = my_delta * scale;
  f32x16 acc[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db) acc[db] = zero16();

  const RawTile<D, TR, NT> tk{k + base, raw, S, wave, lane},
      tv{v + base, raw + TR * D, S, wave, lane};
  tk.issue(0);
  tv.issue(0);
  for (int t = 0; t < n_tiles; ++t) {
    wait_vm_lds<0>();  // this wave's pieces of the tile
    __syncthreads();   // every wave is done with the previous tile's planes
    store_x3<D, TR>(tk, skp);
    store_x3<D, TR>(tv, svp);
    __syncthreads();
    if (t + 1 < n_tiles) {
      tk.issue((t + 1) * TR);
      tv.issue((t + 1) * TR);
    }
    const int key0 = t * TR + 32 * sub;
    if (key0 > q0 + 31) continue;  // wave-uniform: the whole chunk is in the future
    // lane (l32, h), register u: query qi, key key0 + reg_row(u, h)
    f32x16 s = score_tile_p<D, TR>(skp, 32 * sub, qb, lane);   // K Q^T
    f32x16 dp = score_tile_p<D, TR>(svp, 32 * sub, gb, lane);  // V dO^T
    KeepWords16 keep = {};
    if constexpr (DROP) keep = keep_words16(dr, (uint64_t)bh * S + qi, key0, h);
    // only the chunk whose first key is the wave's first query holds keys after a query (or
    // past S): waves are 32-query aligned
    const bool diag = key0 == q0;
#pragma unroll
    for (int u = 0; u < 16; ++u) s[u] = exp_acc(fmaf(s[u], scale, -my_lse));  // P
    if (diag) {
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (key0 + reg_row(u, h) > qi) s[u] = 0.f;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const float p = s[u];
      float g = dp[u];
      if constexpr (DROP) g *= keep_factor(keep, u, dr);
      s[u] = p * fmaf(g, scale, -my_dscale);  // P (dP - delta) scale
    }
    accumulate_t_p<D, TR>(acc, skp, 32 * sub, s, lane);  // dQ^T += K^T dS^T
  }
  __syncthreads();
  float* slot = reinterpret_cast<float*>(smem) + grp * kSlot;
  if constexpr (KS == 2) {
    if (sub == 1) put_acc(acc, reinterpret_cast<AccLds*>(slot), lane);
    __syncthreads();
    if (sub == 1) return;
    add_acc(acc, reinterpret_cast<const AccLds*>(slot), lane);
    __builtin_amdgcn_wave_barrier();
  }
  store_rows_t<D>(dq + base, q0, S, acc, 1.0f, slot, lane);
}

// The backward is one launch: grid (BH, blocks, 2), dK/dV workgroups first (z = 0, the longer
// chains), then the dQ ones, which fill the CUs as those run out. As two launches, each
// with its own start, end and half-idle last round (B4 H12 S1024 / B1 H24 S1024 / B16 H12 S256,
// us): 158 -> 143, 140 -> 86, 68 -> 55; where the CUs are full anyway (B16 H12 S1024) 532 -> 527.
// OWN_DELTA: both kinds compute delta themselves, which saves the small grids a launch (4 x 64:
// 10.0 -> 8.3 us); past kOwnDeltaMaxS rows, where dK/dV would read O and dO once per key block
// more, a pass before does it (96 x 1024: 268 against 263.5 us).
constexpr int kOwnDeltaMaxS = 512;
template <int D, bool DROP, int KS, bool OWN_DELTA>
__global__ __launch_bounds__(64 * kGroups * KS, wgs_per_cu(KS)) void bwd_f32_kernel(
    const F32BwdArgs a) {
  __shared__ F32BwdShared<D, KS> sm;
  __shared__ float own_delta[OWN_DELTA ? kOwnDeltaMaxS : 1];
  if (blockIdx.z == 0)
    dkdv_f32_workgroup<D, DROP, KS, OWN_DELTA>(a, blockIdx.x, blockIdx.y, sm, own_delta);
  else
    dq_f32_workgroup<D, DROP, KS, OWN_DELTA>(a, blockIdx.x, gridDim.y - 1 - blockIdx.y, sm);
}

// A backward in place (dq = q or dout, or any gradient = out) runs as the delta pass, dK/dV and
// dQ, one after the other.
template <int D, bool DROP>
__global__ __launch_bounds__(64 * kGroups, wgs_per_cu(1)) void dkdv_f32_kernel(
    const F32BwdArgs a) {
  __shared__ F32BwdShared<D, 1> sm;
  dkdv_f32_workgroup<D, DROP, 1, false>(a, blockIdx.x, blockIdx.y, sm, nullptr);
}
template <int D, bool DROP>
__global__ __launch_bounds__(64 * kGroups, wgs_per_cu(1)) void dq_f32_kernel(const F32BwdArgs a) {
  __shared__ F32BwdShared<D, 1> sm;
  dq_f32_workgroup<D, DROP, 1, false>(a, blockIdx.x, gridDim.y - 1 - blockIdx.y, sm);
}

// Waves per row group. With one, a workgroup walks its chunks four waves wide, two workgroups
// to a CU; a grid of no more workgroups than that (all of them start at once) lasts as long as
// the longest one's chain, so each group then gets a second wave and the chain is half as long.
// Past one workgroup per CU the gain shrinks with the chain's length. Forward, one -> two (us):
// 128 x 256 (256 workgroups) 21.0 -> 18.4, 48 x 1024 (384) 64.6 -> 49.6, 64 x 1024 (512) 68.8 ->
// 64.7, 96 x 512 (384) 37.8 -> 32.7; 128 x 512 (512) 38.1 -> 39.0, 128 x 300 (384) 24.8 -> 27.3,
// 40 x 2048 (640) 141 -> 147, 192 x 1024 165 -> 186; up to three chunks (S <= 96) there is too
// little to share.
int fwd_waves_per_group(int BH, int S) {
  const long long wgs = (long long)BH * ((S + kRows - 1) / kRows), cus = device_cus();
  const long long most = S >= 768 ? 4 * cus : S >= 512 ? 3 * cus : 2 * cus;  // halves of a CU
  return S > 96 && 2 * wgs <= most ? 2 : 1;
}
// The backward's grid holds two workgroups per 128 rows, so its line is at half as many rows:
// 24 x 1024 (192 of each kind) 120 -> 86, 128 x 128 22.6 -> 19.6, 48 x 1024 (384) 143 -> 150,
// 96 x 512 81 -> 94. Short sequences: 4 x 64 8.4 -> 7.2, 192 x 64 15.5 -> 20.6.
int bwd_waves_per_group(int BH, int S) {
  const long long wgs = (long long)BH * ((S + kRows - 1) / kRows), cus = device_cus();
  return wgs <= (S > 96 ? cus : cus / 4) ? 2 : 1;
}

// f(whether to drop, waves per row group) as compile-time constants.
template <typename F>
void with_f32_shape(int waves_per_group, bool drop, F f) {
  const bool two = waves_per_group == 2;
  auto with_drop = [&](auto d) {
    if (two)
      f(d, std::integral_constant<int, 2>{});
    else
      f(d, std::integral_constant<int, 1>{});
  };
  if (drop)
    with_drop(std::true_type{});
  else
    with_drop(std::false_type{});
}

template <int D>
hipError_t fwd_f32_t(float* out, float* lse, const float* q, const float* k, const float* v,
                     int BH, int S, float scale, hipStream_t stream, const Dropout* drop) {
  const dim3 grid(BH, (S + kRows - 1) / kRows);
  const DropParams dr = drop_params(drop);
  with_f32_shape(fwd_waves_per_group(BH, S), drop != nullptr, [&](auto drop_c, auto ks) {
    auto launch = [&](auto once) {
      fwd_f32_kernel<D, drop_c(), ks(), once()>
          <<<grid, 64 * kGroups * ks(), 0, stream>>>(out, lse, q, k, v, S, scale, dr);
    };
    // At d_head 64 with one wave per group, up to two rounds of workgroups (two per CU), the last
    // of which run a wave per SIMD: a lone wave is faster if the conversions need not wait for
    // each other (once -> not: 192 x 400 54.7 -> 48.3 us, 256 x 384 47.1 -> 43.1, 128 x 777 90.8 ->
    // 85.8; 400 x 483 103 -> 107, 192 x 1024 158.4 -> 161.6). With dropout or at d_head 32 once is
    // faster everywhere.
    constexpr bool kEither = D == 64 && !drop_c() && ks() == 1;
    if constexpr (kEither)
      if ((long long)grid.x * grid.y <= 4LL * device_cus()) return launch(std::false_type{});
    launch(std::true_type{});
  });
  return hipGetLastError();
}

template <int D>
hipError_t bwd_f32_t(float* dq, float* dk, float* dv, float* delta, const float* dout,
                     const float* out, const float* lse, const float* q, const float* k,
                     const float* v, int BH, int S, float scale, hipStream_t stream,
                     const Dropout* drop) {
  const F32BwdArgs args{dq, dk, dv, delta, q, k, v, dout, out, lse, S, scale, drop_params(drop)};
  auto span = [&](const float* p) { return Span{p, (size_t)BH * S * D * sizeof(float)}; };
  const bool separate = in_place({span(dq), span(dk), span(dv)},
                                 {span(q), span(k), span(v), span(dout), span(out)});
  const bool own = S <= kOwnDeltaMaxS && !separate;
  hipError_t e = hipSuccess;
  if (!own) {
    const long long rows = (long long)BH * S, blocks = (rows * (D / 4) + 255) / 256;
    delta_f32_kernel<D><<<(unsigned)(blocks < 16384 ? blocks : 16384), 256, 0, stream>>>(
        delta, dout, out, rows);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  const dim3 blocks(BH, (S + kRows - 1) / kRows), grid(blocks.x, blocks.y, 2);
  with_f32_shape(bwd_waves_per_group(BH, S), drop != nullptr, [&](auto drop_c, auto ks) {
    constexpr int threads = 64 * kGroups * ks();
    if (separate) {
      dkdv_f32_kernel<D, drop_c()><<<blocks, 64 * kGroups, 0, stream>>>(args);
      if ((e = hipGetLastError()) != hipSuccess) return;
      dq_f32_kernel<D, drop_c()><<<blocks, 64 * kGroups, 0, stream>>>(args);
    } else if (own) {
      bwd_f32_kernel<D, drop_c(), ks(), true><<<grid, threads, 0, stream>>>(args);
    } else {
      bwd_f32_kernel<D, drop_c(), ks(), false><<<grid, threads, 0, stream>>>(args);
    }
    e = hipGetLastError();
  });
  return e;
}

}  // namespace

hipError_t launch_fwd_f32(float* out, float* lse, const float* q, const float* k,
                          const float* v, int BH, int S, int D, float scale,
                          hipStream_t stream, const Dropout* drop) {
  if (D == 64) return fwd_f32_t<64>(out, lse, q, k, v, BH, S, scale, stream, drop);
  if (D == 32) return fwd_f32_t<32>(out, lse, q, k, v, BH, S, scale, stream, drop);
  return hipErrorInvalidValue;
}

hipError_t launch_bwd_f32(float* dq, float* dk, float* dv, float* delta, const float* dout,
                          const float* out, const float* lse, const float* q, const float* k,
                          const float* v, int BH, int S, int D, float scale,
                          hipStream_t stream, const Dropout* drop) {
  if (D == 64)
    return bwd_f32_t<64>(dq, dk, dv, delta, dout, out, lse, q, k, v, BH, S, scale, stream,
                         drop);
  if (D == 32)
    return bwd_f32_t<32>(dq, dk, dv, delta, dout, out, lse, q, k, v, BH, S, scale, stream,
                         drop);
  return hipErrorInvalidValue;
}

}  // namespace dadgpt
