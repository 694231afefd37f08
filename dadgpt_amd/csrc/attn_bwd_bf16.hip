// Causal flash-attention backward for gfx950: bf16 operands, fp32 accumulation, P recomputed
// from the saved natural-log logsumexp. Covers what cuda/attention.cu:75-205 does in fp32
// (delta, dK/dV, dQ), restructured for MFMA:
//
//   dQ kernel      query-major; per 32-key chunk:  S^T = K Q^T, dP^T = V dO^T,
//                  dQ^T += K^T dS^T                                   (attention.cu:154-205)
//                  and, first, delta[r] = sum_d dO[r,d] * O[r,d] of its rows, written for
//                  the dK/dV kernel                                   (attention.cu:75-85)
//   dK/dV kernel   key-major; per 32-query block:  S = Q K^T, dP = dO V^T,
//                  P = exp(S*scale - lse), dS = P (dP - delta),
//                  dV^T += dO^T P, dK^T += Q^T dS                    (attention.cu:87-152)
//   delta kernel   delta as a pass of its own (the phase API; long rows on small grids)
//
// Small and medium grids run both in one launch (bwd_plan): dK/dV workgroups first, then dQ ones.
// Both MFMA kernels own their outputs outright (no atomics, bitwise repeatable). The score
// tiles use the same sigma32 row permutation as the forward so that P and dS feed the next
// MFMA as B operands from registers; the operands that must be read along the score dimension
// (Q^T and dO^T in the dK/dV kernel, K^T in the dQ kernel) are read across the rows of the
// row-major LDS tiles with ds_read_b64_tr_b16, so every tile is staged once, row-major.
// Masking runs only in the blocks that straddle the diagonal, behind a uniform branch around
// the instructions that zero P. The streamed tiles (Q and dO for dK/dV, K and V for dQ) are
// double-buffered in LDS through direct global->LDS loads, one tile ahead of the compute.
// On small grids (KS = 2, waves_per_group) a workgroup owns 64 rows instead of 128 and two waves
// share each 32-row group, taking one chunk of every tile each; their sums are merged at the end.
// STRIDED and DROP instantiations as in the forward: per-tensor strides, and dropout with
// the keep bits regenerated (dV from P keep/(1-p), dS = P (dP keep/(1-p) - delta)).
#include "common.hpp"
#include "dropout.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include "tiles.hpp"

namespace dadgpt {
namespace {

constexpr int kWaves = 4;
// Workgroups per CU the registers are sized for (4 waves each: 2 -> 256 VGPRs, 3 -> 168).
// dK/dV fits 168 with its LDS addresses derived at use (LaneLds); the dropout one keeps
// 256.
#ifndef DADGPT_DKDV_MINB
#define DADGPT_DKDV_MINB 2
#endif
#ifndef DADGPT_DKDV_MINB_NODROP
#define DADGPT_DKDV_MINB_NODROP 3
#endif
#ifndef DADGPT_DQ_MINB
#define DADGPT_DQ_MINB 3
#endif
constexpr int dkdv_wgs_per_cu(bool drop) {
  return drop ? DADGPT_DKDV_MINB : DADGPT_DKDV_MINB_NODROP;
}
constexpr int kDqMinBlocks = DADGPT_DQ_MINB;

// ---------------------------------------------------------------- delta
template <int D, bool STRIDED>
__global__ __launch_bounds__(256) void delta_bf16_kernel(float* __restrict__ delta,
                                                         const bf16* __restrict__ dout,
                                                         const bf16* __restrict__ out, int S,
                                                         long long rows, int row_blocks,
                                                         const AttnLayout L) {
  // 32 rows per workgroup, 8 lanes per row, 16 bytes each per step. Contiguous: rows of the
  // flat [BH*S, D] matrices (`rows` of them); strided: row_blocks workgroups per (b,h) slice.
  constexpr int LPR = 8;
  const int part = threadIdx.x % LPR;
  const bf16 *dor, *orow;
  long long drow;  // row of delta
  bool valid;
  if constexpr (STRIDED) {
    const int bh = blockIdx.x / row_blocks;
    const int row = (blockIdx.x - bh * row_blocks) * (256 / LPR) + threadIdx.x / LPR;
    const Slice<D, true> sl(L, bh, S);
    dor = sl.row(dout, kTDO, row);
    orow = sl.row(out, kTO, row);
    drow = (long long)bh * S + row;
    valid = row < S;
  } else {
    drow = (long long)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
    dor = dout + drow * D;
    orow = out + drow * D;
    valid = drow < rows;
  }
  float acc = 0.f;
  if (valid) {
#pragma unroll
    for (int c = part; c < D / 8; c += LPR) {
      const u32x4 a = ld_g128u(dor + c * 8);
      const u32x4 b = ld_g128u(orow + c * 8);
#pragma unroll
      for (int w = 0; w < 4; ++w)
        acc += bf16_lo(a[w]) * bf16_lo(b[w]) + bf16_hi(a[w]) * bf16_hi(b[w]);
    }
  }
  acc = lanes::group_sum<LPR>(acc);
  if (valid && part == 0) delta[drow] = acc;
}

// ---------------------------------------------------------------- dK / dV
constexpr int kKW = 32;  // keys per wave

// One 32-query block (tile rows 32*qb ..) against the wave's 32 keys. Register 8j+e of lane
// half hi holds tile query 32qb + 16j + 8hi + e. The two score products start from
// accumulators that already hold the per-query statistics, read from LDS straight into them:
//   s  = -lse/scale + Q K^T         so P = exp2(c s) with c = scale log2(e)
//   dp = -delta + dO V^T            so P dp = P (dP - delta) = dS
// which leaves two multiplies and an exp2 per score on the VALU. slc holds the tile's
// -lse/scale, sdl its -delta. `mask` zeroes P for keys after the query and for tile rows past
// S (rows_left = S - r0; those rows hold copies of row S-1). It is a runtime flag, not a
// template parameter, and guards only the few instructions that zero P: with two inlined copies
// of the block the compiler gave their MFMAs different accumulator registers and copied all 64
// accumulator values back after every block.
//
// With dropout (DROP; f = keep/(1-p) from bit 8j+e of `keep`): dV accumulates (P f)^T dO and
// dS = P (dP f - delta), so dp starts from zero and -delta is read separately.
// XA: operand addresses from `lo` (LaneLds, tiles.hpp), XORed once per phase, instead of
// computed per read: what brings dK/dV (all but the dropout instantiation) to 168 VGPRs,
// three workgroups per CU, without spilling in the loop. (The strided kernel of one launch with
// its own delta and one wave per group keeps two registers in scratch and reloads them as it
// issues a tile.)
template <int D, bool DROP, bool XA>
__device__ __forceinline__ void dkdv_block(bool mask, f32x16 (&dkacc)[D / 32],
                                           f32x16 (&dvacc)[D / 32], const bf16x8 (&kop)[D / 16],
                                           const bf16x8 (&vop)[D / 16], const bf16* sq,
                                           const bf16* sdo, const float* slc, const float* sdl,
                                           int qb, int key_minus_r0, int rows_left, int lane,
                                           float c, uint32_t keep, float dscale,
                                           const LaneLds& lo) {
  constexpr int DS = D / 16, DB = D / 32;
  const int l32 = lane & 31, hi = lane >> 5;
  const int qr = 32 * qb + sigma32(l32);
  // Phases: S = stats + Q K^T, dP = stats + dO V^T, softmax, dV += dO^T P, dK += Q^T dS,
  // ordered by the compiler's scheduler (fencing them apart measured 2-3% slower).
  auto stats = [&](const float* row, f32x16& acc) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int qt0 = 32 * qb + 16 * j + 8 * hi;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(row + qt0 + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[8 * j + 4 * h + e] = a[e];
      }
    }
  };
  f32x16 s, dp;
  uint32_t ra[DS] = {};
  if constexpr (XA) row_addr_xor<D>(ra, lo.ro);
  {
    bf16x8 qa[DS];
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
      qa[ds] = XA ? lds_row_at(sq + 32 * qb * D, ra[ds])
                  : lds_op(sq, rm_off<D>(qr, 2 * ds + hi));
    stats(slc, s);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) s = mfma32(qa[ds], kop[ds], s);
  }
  {
    bf16x8 da[DS];
#pragma unroll
    for (int ds = 0; ds < DS; ++ds)
      da[ds] = XA ? lds_row_at(sdo + 32 * qb * D, ra[ds])
                  : lds_op(sdo, rm_off<D>(qr, 2 * ds + hi));
    if constexpr (DROP)
      dp = f32x16{};
    else
      stats(sdl, dp);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) dp = mfma32(da[ds], vop[ds], dp);
  }
  bf16x8 pb[2], dsb[2];
  f32x16 nd;  // -delta of the block's queries (dropout only)
  if constexpr (DROP) stats(sdl, nd);
  float pr[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) pr[i] = fast_exp2(s[i] * c);
  if (mask) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int qt0 = 32 * qb + 16 * j + 8 * hi;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        pr[8 * j + e] = (key_minus_r0 > qt0 + e || qt0 + e >= rows_left) ? 0.f : pr[8 * j + e];
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    u32x4 wp, wd;
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2) {
      float p[2], d[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = 2 * e2 + h;
        const float pe = pr[8 * j + e];
        if constexpr (DROP) {
          const float f = keep_factor(keep, 8 * j + e, dscale);
          p[h] = pe * f;
          d[h] = pe * fmaf(dp[8 * j + e], f, nd[8 * j + e]);
        } else {
          p[h] = pe;
          d[h] = pe * dp[8 * j + e];
        }
      }
      wp[e2] = pack_bf16x2(p[0], p[1]);
      wd[e2] = pack_bf16x2(d[0], d[1]);
    }
    pb[j] = as_bf16x8(wp);
    dsb[j] = as_bf16x8(wd);
  }
  uint32_t ta[2][DB] = {};
  if constexpr (XA) tr_addr_xor<D>(ta, lo.tr);
  {
    bf16x8 t[DB][2];  // A = dO^T: lane d = 32db + l32 gets tile queries 32qb + 16j + 8hi + 0..7
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        t[db][j] = XA ? lds_tr_at(sdo + (32 * qb + 16 * j) * D, ta[0][db], ta[1][db])
                      : lds_tr_op<D>(sdo, 32 * qb + 16 * j, 32 * db, lane);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int db = 0; db < DB; ++db) dvacc[db] = mfma32(t[db][j], pb[j], dvacc[db]);
  }
  {
    bf16x8 t[DB][2];  // A = Q^T
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        t[db][j] = XA ? lds_tr_at(sq + (32 * qb + 16 * j) * D, ta[0][db], ta[1][db])
                      : lds_tr_op<D>(sq, 32 * qb + 16 * j, 32 * db, lane);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int db = 0; db < DB; ++db) dkacc[db] = mfma32(t[db][j], dsb[j], dkacc[db]);
  }
}

// What a backward kernel works on.
struct BwdArgs {
  bf16 *dq, *dk, *dv;
  float* delta;
  const bf16 *q, *k, *v, *dout, *out;
  const float* lse;
  int S;
  float scale, scale_log2;      // dQ: the scale, and times log2(e)
  float c, lse_mul;             // dK/dV: nonzero scale times log2(e), and -1/scale
  AttnLayout L;
  DropParams dr;
};

// LDS of a workgroup: two streamed tiles (Q and dO, or K and V), double-buffered (constant
// buffer indices in the unrolled loop; see the forward kernel).
template <int D>
struct BwdTiles {
  __attribute__((aligned(16))) bf16 a[2][kTileRows * D];
  __attribute__((aligned(16))) bf16 b[2][kTileRows * D];
};
// dK/dV: per wave and buffer the tile's lse and delta rows, converted in place to -lse/scale and
// -delta: each wave loads and converts its own copy, so the conversion needs no barrier.
struct BwdStats {
  __attribute__((aligned(16))) float row[kWaves][2][2][kTileRows];
};

// delta of rows row0 .. S-1 into LDS, for a dK/dV workgroup that runs beside the dQ ones
// instead of after them (the order of the sum differs from dQ's): 16 bytes of a row per lane,
// four groups of rows in flight.
template <int D, bool STRIDED>
__device__ __forceinline__ void delta_rows(float* delta, const Slice<D, STRIDED>& sl,
                                           const bf16* dout, const bf16* out, int row0, int S) {
  constexpr int LPR = D / 8, ROWS = 64 * kWaves / LPR, N = 4;
  const int part = threadIdx.x % LPR;
  for (int r0 = row0 + (int)threadIdx.x / LPR; r0 - (int)threadIdx.x / LPR < S; r0 += N * ROWS) {
    u32x4 g[N], o[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = min(r0 + i * ROWS, S - 1);
      g[i] = ld_g128u(sl.row(dout, kTDO, r) + part * 8);
      o[i] = ld_g128u(sl.row(out, kTO, r) + part * 8);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float acc = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        acc += bf16_lo(g[i][w]) * bf16_lo(o[i][w]) + bf16_hi(g[i][w]) * bf16_hi(o[i][w]);
      acc = lanes::group_sum<LPR>(acc);
      const int r = r0 + i * ROWS;
      if (part == 0 && r < S) delta[r - row0] = acc;
    }
  }
}

// One workgroup's dK and dV. OWN_DELTA: delta is computed here, into own_delta (one float for
// each row from the first tile on); otherwise it is read from a.delta.
template <int D, bool STRIDED, bool DROP, int KS, bool OWN_DELTA>
__device__ __forceinline__ void dkdv_workgroup(const BwdArgs& a, int bh, int kblk,
                                               BwdTiles<D>& tiles, BwdStats& stats,
                                               float* own_delta) {
  constexpr int kGroups = kWaves / KS, KB = kKW * kGroups;  // key groups, keys
  constexpr int DS = D / 16, DB = D / 32;
  auto& sq = tiles.a;
  auto& sdo = tiles.b;
  static_assert(kWaves * kKW <= 2 * kTileRows, "the epilogue stages every wave's rows in sq");
  const bf16 *q = a.q, *k = a.k, *v = a.v, *dout = a.dout;
  bf16 *dk = a.dk, *dv = a.dv;
  const int S = a.S;
  const DropParams& dr = a.dr;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int grp = wave % kGroups, sub = wave / kGroups;
  const Slice<D, STRIDED> sl(a.L, bh, S);
  const bf16* qg = sl.base(q, kTQ);
  const bf16* dog = sl.base(dout, kTDO);
  const int qp = sl.pitch(kTQ), dop = sl.pitch(kTDO);  // row pitches of the streamed tiles
  const float* lseg = a.lse + (size_t)bh * S;
  const float* delg = a.delta + (size_t)bh * S;

  const int kw0 = kblk * KB + grp * kKW;
  const int key = kw0 + l32;
  const int t_first = (kblk * KB) / kTileRows;
  const int t_end = (S - 1) / kTileRows + 1;

  // B operands (K^T, V^T along D): lane holds key row `key`, columns 16*ds + 8*hi + 0..7.
  bf16x8 kop[DS], vop[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    const bool in = key < S;
    kop[ds] = in ? ld_g128(sl.row(k, kTK, key) + 16 * ds + 8 * hi)
                 : as_bf16x8(u32x4{0, 0, 0, 0});
    vop[ds] = in ? ld_g128(sl.row(v, kTV, key) + 16 * ds + 8 * hi)
                 : as_bf16x8(u32x4{0, 0, 0, 0});
  }

  f32x16 dkacc[DB], dvacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dkacc[db] = f32x16{};
    dvacc[db] = f32x16{};
  }
  constexpr bool XA = !DROP;
  LaneLds lo{};
  if constexpr (XA) lo = lane_lds<D>(lane);

  // Direct loads per wave per tile: its share of Q and dO, and its own lse and delta rows.
  using Dma = DmaTile<D, kWaves>;
  uint32_t qoff[Dma::PER_WAVE], dooff[Dma::PER_WAVE];
  Dma::offsets(qoff, wave, lane, qp);
  Dma::offsets(dooff, wave, lane, dop);
  float(*st)[2][kTileRows] = stats.row[wave];
  auto issue = [&](int t, bf16* nq, bf16* ndo, int buf) {
    Dma::template load_any<true>(nq, qg, t * kTileRows, S, qoff, wave, lane, qp);
    Dma::template load_any<true>(ndo, dog, t * kTileRows, S, dooff, wave, lane, dop);
    dma_row64(st[buf][0], lseg, t * kTileRows, S, lane);
    if constexpr (!OWN_DELTA) dma_row64(st[buf][1], delg, t * kTileRows, S, lane);
  };
  // The first tile loads alongside the operands above: one wait covers all of them (the
  // compiler, which does not see the direct loads, then has nothing left to wait for).
  issue(t_first, sq[0], sdo[0], 0);
  if constexpr (OWN_DELTA)
    delta_rows<D, STRIDED>(own_delta, sl, dout, a.out, t_first * kTileRows, S);
  wait_vm_lds<0>();
  __builtin_amdgcn_s_barrier();

  // One query tile: prefetch tile t+1 (into the buffers of tile t-1, released by the last
  // barrier), convert this wave's statistics rows, compute tile t, wait for tile t+1 and
  // barrier.
  auto tile = [&](int t, const bf16* cq, const bf16* cdo, int cb, bf16* nq, bf16* ndo,
                  int nb) {
    const int r0 = t * kTileRows;
    if (t + 1 < t_end) issue(t + 1, nq, ndo, nb);
    if (kw0 < S && r0 + kTileRows - 1 >= kw0) {
      // -lse/scale and -delta (this wave's copy; its LDS accesses complete in order)
      st[cb][0][lane] *= a.lse_mul;
      st[cb][1][lane] = OWN_DELTA ? -own_delta[min(r0 + lane, S - 1) - t_first * kTileRows]
                                  : -st[cb][1][lane];
      const bool edge = r0 + kTileRows > S;
#pragma unroll
      for (int i = 0; i < 2 / KS; ++i) {
        const int qb = KS == 1 ? i : sub, qlo = r0 + 32 * qb;  // first query of the block
        if (qlo + 31 < kw0) continue;   // every key of the wave is after every query
        uint32_t keep = 0;
        if constexpr (DROP) keep = keep_col16(dr, (uint64_t)bh * S + qlo, kw0, lane);
        // some key after some query, or rows past S: mask
        dkdv_block<D, DROP, XA>(edge || qlo < kw0 + kKW - 1, dkacc, dvacc, kop, vop, cq, cdo,
                                st[cb][0], st[cb][1], qb, key - r0, S - r0, lane, a.c, keep,
                                dr.scale, lo);
      }
    }
    wait_vm_lds<0>();
    __builtin_amdgcn_s_barrier();
  };
  for (int t = t_first; t < t_end; t += 2) {
    tile(t, sq[0], sdo[0], 0, sq[1], sdo[1], 1);
    if (t + 1 < t_end) tile(t + 1, sq[1], sdo[1], 1, sq[0], sdo[0], 0);
  }

  // the tiles are free after the last barrier
  if constexpr (KS == 1) {
    // each wave stages its 32 rows in its quarter of sq (dK) and sdo (dV)
    if (kw0 < S) {
      store_rows_staged<D>(sl.row(dk, kTDK, kw0), sl.pitch(kTDK), S - kw0, dkacc, a.scale,
                           &sq[0][0] + wave * kKW * D, lane);
      store_rows_staged<D>(sl.row(dv, kTDV, kw0), sl.pitch(kTDV), S - kw0, dvacc, 1.0f,
                           &sdo[0][0] + wave * kKW * D, lane);
    }
  } else {
    // The group's two waves exchange partials: the first finishes dK, the second dV, each in
    // the group's slot of sq / sdo (partials in, rows staged out).
    static_assert(sizeof(sq) >= kGroups * DB * sizeof(AccLds), "a group's partials fit");
    AccLds* slot_k = reinterpret_cast<AccLds*>(&sq[0][0]) + grp * DB;
    AccLds* slot_v = reinterpret_cast<AccLds*>(&sdo[0][0]) + grp * DB;
    if (sub == 1)
      put_acc(dkacc, slot_k, lane);
    else
      put_acc(dvacc, slot_v, lane);
    __syncthreads();
    if (kw0 >= S) return;
    if (sub == 0) {
      add_acc(dkacc, slot_k, lane);
      store_rows_staged<D>(sl.row(dk, kTDK, kw0), sl.pitch(kTDK), S - kw0, dkacc, a.scale,
                           reinterpret_cast<bf16*>(slot_k), lane);
    } else {
      add_acc(dvacc, slot_v, lane);
      store_rows_staged<D>(sl.row(dv, kTDV, kw0), sl.pitch(kTDV), S - kw0, dvacc, 1.0f,
                           reinterpret_cast<bf16*>(slot_v), lane);
    }
  }
}

template <int D, bool STRIDED, bool DROP, int KS>
__global__ __launch_bounds__(64 * kWaves, dkdv_wgs_per_cu(DROP)) void dkdv_bf16_kernel(
    const BwdArgs a) {
  __shared__ BwdTiles<D> tiles;
  __shared__ BwdStats stats;
  // key block 0 sees the most query tiles: dispatched first
  dkdv_workgroup<D, STRIDED, DROP, KS, false>(a, blockIdx.x, blockIdx.y, tiles, stats, nullptr);
}

// ---------------------------------------------------------------- dQ
constexpr int kQW = 32;  // queries per wave

// One 32-key chunk (tile keys 32*kb ..) against the wave's 32 queries. Register 8j+e of lane
// half hi holds tile key 32kb + 16j + 8hi + e. FROM_DELTA: dP starts from `ndl`, -delta of the
// lane's query in every element, so that P dP is dS; otherwise -delta (ndl[0]) is added after.
// VALU and matrix pipe are both busy here: without the 16 subtractions dQ takes 284 us for 295 at
// [96, 4096, 64], 47.9 for 49.6 at [192, 1024, 64] (with a third tile buffer and loads two tiles
// ahead: 286 and 48.7; K^T read before the exponentials spills). The 16 registers held across the
// loop must not cost a wave per SIMD, though (see dq_bf16_kernel). With dropout (DROP), dS =
// P (dP * f - delta), f = keep/(1-p) from register 8j+e's uniform in `keep`: dP from zero, as
// those registers cost that kernel more too (96 x 1024: backward 88 -> 92.5).
template <int D, bool DROP, bool FROM_DELTA>
__device__ __forceinline__ void dq_chunk(bool diag, f32x16 (&dqacc)[D / 32],
                                         const bf16x8 (&qop)[D / 16],
                                         const bf16x8 (&doop)[D / 16], const bf16* sk,
                                         const bf16* sv, int kb, int qrow_minus_k0, float lse2,
                                         const f32x16& ndl, int lane, float scale_log2,
                                         const KeepWords16& keep, const DropParams& dr) {
  constexpr int DS = D / 16, DB = D / 32;
  const int l32 = lane & 31, hi = lane >> 5;
  f32x16 s = f32x16{}, dp = f32x16{};
  const int krow = 32 * kb + sigma32(l32);
  bf16x8 va[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) s = mfma32(lds_op(sk, rm_off<D>(krow, 2 * ds + hi)), qop[ds], s);
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) va[ds] = lds_op(sv, rm_off<D>(krow, 2 * ds + hi));
  __builtin_amdgcn_sched_barrier(0);
  // dP runs on the matrix pipe under the exponentials of S: one dP MFMA, then 16/DS of the
  // wave's exponentials, fenced so the compiler keeps the interleave (left to itself it
  // issued all exponentials first; this order took dQ ~2% faster)
  float pr[16];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    dp = mfma32(va[ds], doop[ds], FROM_DELTA && ds == 0 ? ndl : dp);
#pragma unroll
    for (int i = ds * (16 / DS); i < (ds + 1) * (16 / DS); ++i)
      pr[i] = fast_exp2(fmaf(s[i], scale_log2, -lse2));
    __builtin_amdgcn_sched_barrier(0);
  }
  if (diag) {  // runtime flag around the zeroing only (see dkdv_block)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      pr[i] = 32 * kb + 16 * (i / 8) + 8 * hi + i % 8 > qrow_minus_k0 ? 0.f : pr[i];
  }
  bf16x8 dsb[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    u32x4 w;
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2) {
      float d[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = 2 * e2 + h;
        const float p = pr[8 * j + e];
        if constexpr (DROP)
          d[h] = p * fmaf(dp[8 * j + e], keep_factor(keep, 8 * j + e, dr), ndl[0]);
        else
          d[h] = p * (FROM_DELTA ? dp[8 * j + e] : dp[8 * j + e] + ndl[0]);
      }
      w[e2] = pack_bf16x2(d[0], d[1]);
    }
    dsb[j] = as_bf16x8(w);
  }
#pragma unroll
  for (int db = 0; db < DB; ++db) {
#pragma unroll
    for (int j = 0; j < 2; ++j)  // A = K^T: lane d = 32db + l32 gets keys 32kb + 16j + 8hi ..
      dqacc[db] = mfma32(lds_tr_op<D>(sk, 32 * kb + 16 * j, 32 * db, lane), dsb[j], dqacc[db]);
  }
}

// dQ for one query block per wave; the kernel also computes delta = rowsum(dO * O) of its
// rows (from the dO operands it holds and one load of O) and writes it for the dK/dV kernel,
// so the backward needs no separate delta pass.
template <int D, bool STRIDED, bool DROP, int KS, bool WRITE_DELTA, bool FROM_DELTA>
__device__ __forceinline__ void dq_workgroup(const BwdArgs& a, int bh, int qblk,
                                             BwdTiles<D>& tiles) {
  constexpr int kGroups = kWaves / KS, QB = kQW * kGroups;  // query groups, queries
  constexpr int DS = D / 16, DB = D / 32;
  auto& sk = tiles.a;
  auto& sv = tiles.b;
  static_assert(kWaves * kQW <= 2 * kTileRows, "the epilogue stages every wave's rows in sk");
  const bf16 *q = a.q, *k = a.k, *v = a.v, *dout = a.dout, *out = a.out;
  bf16* dq = a.dq;
  float* delta = a.delta;
  const float* lse = a.lse;
  const int S = a.S;
  const float scale_log2 = a.scale_log2, scale = a.scale;
  const DropParams& dr = a.dr;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int grp = wave % kGroups, sub = wave / kGroups;
  const Slice<D, STRIDED> sl(a.L, bh, S);
  const bf16* kg = sl.base(k, kTK);
  const bf16* vg = sl.base(v, kTV);
  const int kp = sl.pitch(kTK), vp = sl.pitch(kTV);  // row pitches of the streamed tiles

  const int q0 = qblk * QB + grp * kQW;
  const int qrow = q0 + l32;
  const int wg_last = min(S, (qblk + 1) * QB) - 1;
  const int n_tiles = wg_last / kTileRows + 1;

  // lane holds row qrow, columns 16*ds + 8*hi + 0..7 of Q, dO and O (zeros past S)
  bf16x8 qop[DS], doop[DS], oop[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    const bool in = qrow < S;
    const u32x4 z{0, 0, 0, 0};
    qop[ds] = in ? ld_g128(sl.row(q, kTQ, qrow) + 16 * ds + 8 * hi) : as_bf16x8(z);
    doop[ds] = in ? ld_g128(sl.row(dout, kTDO, qrow) + 16 * ds + 8 * hi) : as_bf16x8(z);
    oop[ds] = in ? ld_g128(sl.row(out, kTO, qrow) + 16 * ds + 8 * hi) : as_bf16x8(z);
  }
  // (rows past S read row S-1: a finite value for rows that are never stored)
  float lse_q = lse[(size_t)bh * S + min(qrow, S - 1)];

  f32x16 dqacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dqacc[db] = f32x16{};

  // Keys past S read row S-1; every chunk holding such keys is a diagonal chunk (the key is after
  // every valid query), so they are masked. The first tile loads alongside the operands
  // above, under one wait (see the dK/dV kernel).
  using Dma = DmaTile<D, kWaves>;
  uint32_t koff[Dma::PER_WAVE], voff[Dma::PER_WAVE];
  Dma::offsets(koff, wave, lane, kp);
  Dma::offsets(voff, wave, lane, vp);
  Dma::load_any(sk[0], kg, 0, S, koff, wave, lane, kp);
  Dma::load_any(sv[0], vg, 0, S, voff, wave, lane, vp);
  wait_vm_lds<0>();
  __builtin_amdgcn_s_barrier();
  // Use the loaded values only from here on, so their loads share the wait above.
  asm volatile("" : "+v"(lse_q));
  const float lse2 = lse_q * kLog2e;
  // delta of this lane's row: its 32 columns, then the other lane half's
  float dpart = 0.f;
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    asm volatile("" : "+v"(oop[ds]));
    const u32x4 g = as_u32x4(doop[ds]), o = as_u32x4(oop[ds]);
#pragma unroll
    for (int w = 0; w < 4; ++w)
      dpart += bf16_lo(g[w]) * bf16_lo(o[w]) + bf16_hi(g[w]) * bf16_hi(o[w]);
  }
  const float dlt = sum_halves(dpart);
  f32x16 ndl;  // -delta (what dP starts from)
#pragma unroll
  for (int i = 0; i < 16; ++i) ndl[i] = -dlt;
  if (WRITE_DELTA && hi == 0 && qrow < S && sub == 0) delta[(size_t)bh * S + qrow] = dlt;

  auto tile = [&](int t, const bf16* ck, const bf16* cv, bf16* nk, bf16* nv) {
    const int k0 = t * kTileRows;
    if (t + 1 < n_tiles) {
      Dma::load_any(nk, kg, k0 + kTileRows, S, koff, wave, lane, kp);
      Dma::load_any(nv, vg, k0 + kTileRows, S, voff, wave, lane, vp);
    }
    if (q0 < S) {
#pragma unroll
      for (int i = 0; i < 2 / KS; ++i) {
        const int kb = KS == 1 ? i : sub, klo = k0 + 32 * kb;  // first key of the chunk
        if (klo > q0 + kQW - 1) continue;    // every key after every query of the wave
        KeepWords16 keep = {};
        if constexpr (DROP) keep = keep_words16(dr, (uint64_t)bh * S + qrow, klo, hi);
        // some key after some query: mask
        dq_chunk<D, DROP, FROM_DELTA>(klo + 31 > q0, dqacc, qop, doop, ck, cv, kb, qrow - k0,
                                      lse2, ndl, lane, scale_log2, keep, dr);
      }
    }
    wait_vm_lds<0>();
    __builtin_amdgcn_s_barrier();
  };
  for (int t = 0; t < n_tiles; t += 2) {
    tile(t, sk[0], sv[0], sk[1], sv[1]);
    if (t + 1 < n_tiles) tile(t + 1, sk[1], sv[1], sk[0], sv[0]);
  }

  if constexpr (KS == 2) {  // the group's second wave adds to the first
    static_assert(sizeof(sk) >= kGroups * DB * sizeof(AccLds), "a group's partials fit");
    AccLds* slot = reinterpret_cast<AccLds*>(&sk[0][0]) + grp * DB;
    if (sub == 1) put_acc(dqacc, slot, lane);
    __syncthreads();
    if (sub == 1) return;
    add_acc(dqacc, slot, lane);
  }
  if (q0 < S)
    store_rows_staged<D>(sl.row(dq, kTDQ, q0), sl.pitch(kTDQ), S - q0, dqacc, scale,
                         &sk[0][0] + (KS == 1 ? wave : grp * 2) * kQW * D, lane);
}

template <int D, bool STRIDED, bool DROP, int KS>
__global__ __launch_bounds__(64 * kWaves, kDqMinBlocks) void dq_bf16_kernel(const BwdArgs a) {
  __shared__ BwdTiles<D> tiles;
  // longest (latest) query blocks dispatch first
  // At d_head 32 with one wave per group, dP from zero keeps the kernel at 120 registers, four
  // waves per SIMD; from -delta it takes 138 and three: 320 x 384 backward 24.8 -> 26.8 us,
  // 640 x 300 35.1 -> 37.5. (In one launch the dK/dV workgroups set the registers anyway.)
  constexpr bool kFromDelta = !DROP && (D == 64 || KS == 2);
  dq_workgroup<D, STRIDED, DROP, KS, true, kFromDelta>(a, blockIdx.x,
                                                       gridDim.y - 1 - blockIdx.y, tiles);
}

// ---------------------------------------------------------------- both in one launch
// Grid (BH, blocks, 2): dK/dV workgroups first (z = 0, the longer chains), then the dQ ones.
// OWN_DELTA: the dK/dV workgroups compute delta of their rows themselves (up to kOwnDeltaMaxS of
// them) and the dQ workgroups write it; otherwise a pass before has.
constexpr int kOwnDeltaMaxS = 1024;
template <int D, bool STRIDED, bool DROP, int KS, bool OWN_DELTA>
__global__ __launch_bounds__(64 * kWaves, dkdv_wgs_per_cu(DROP)) void bwd_bf16_kernel(
    const BwdArgs a) {
  __shared__ BwdTiles<D> tiles;
  __shared__ BwdStats stats;
  __shared__ float own_delta[OWN_DELTA ? kOwnDeltaMaxS : 1];
  if (blockIdx.z == 0)
    dkdv_workgroup<D, STRIDED, DROP, KS, OWN_DELTA>(a, blockIdx.x, blockIdx.y, tiles, stats,
                                                    own_delta);
  else
    dq_workgroup<D, STRIDED, DROP, KS, OWN_DELTA, !DROP>(a, blockIdx.x,
                                                         gridDim.y - 1 - blockIdx.y, tiles);
}

// How a backward is launched: dQ, then dK/dV (kSeparate); both in one launch with delta
// computed where it is needed (kOneOwnDelta); or a delta pass, then both (kOneAfterDelta).
enum BwdLaunch { kSeparate, kOneOwnDelta, kOneAfterDelta };
struct BwdPlan {
  BwdLaunch how;
  int waves_per_group;
};

// One launch saves a kernel's start and end (~4 us) and lets the dQ workgroups fill the CUs that
// the dK/dV ones leave idle at the end of their chains; where the CUs are full anyway, delta
// summed twice and the two kinds' mixture cost more than that. Separate -> one launch, us (BH x S,
// D = 64): 128 x 128 11.5 -> 7.8, 192 x 256 20.0 -> 15.4, 24 x 1024 32.8 -> 24.5, 96 x 1024 67 ->
// 60, 128 x 1024 83 -> 80, 24 x 4096 211 -> 192. In 128-row workgroups of each kind per CU the
// line lies,
//  - up to two row blocks, at 5 (448 x 256 36.9 -> 33.2, 960 x 256 token-major 77.1 -> 80.9, 1536
//    x 256 114 -> 125; dropout 576 x 256 59.6 -> 59.4, 768 x 256 77.1 -> 81.2), for single blocks
//    without dropout at 13 (2500 x 128 token-major 82.2 -> 85.6); at D = 32, whose kernels hold
//    more workgroups, at 8 (640 x 256 26.6 -> 24.4, 960 x 256 token-major 62.5 -> 64.9), with
//    dropout none;
//  - then at 4.5, one more per head counted (160 x 900 82.5 -> 81.1, dropout 96 x 1024 86.9 ->
//    85.6, 128 x 600 56.6 -> 52.0; 192 x 1024 115 -> 122, dropout 256 x 400 58.7 -> 62.9); with the
//    delta pass, too (37 x 2886 163.7 -> 153.1, 48 x 2886 193.7 -> 188.4; 72 x 1500 86.5 -> 90.1);
//  - with dropout at D = 32 over 512 rows, where two waves per group gain more apart, at 1.5 (64 x
//    1024 44.7 -> 46.6, 48 x 1200 49.1 -> 53.3).
// Apart, too, where the heads fill seven eighths of the CUs or more in one round: each CU then has
// one workgroup of every block, and both kernels end together (256 x 384 31.1 -> 33.1, token-major
// 32.3 -> 35.9). The line must not tell the layouts apart: a strided call gives the contiguous
// one's bits. Up to 1,024 rows the dK/dV workgroups compute delta themselves (96 x 1024: 59
// against 61 us with the pass).
// Two waves per row group then pay only while the grid, twice as large now, still fits on the
// CUs, or for long chains up to twice that (one wave -> two): 64 x 256 10.8 -> 10.4, 24 x 1024
// 30.4 -> 24.5, 96 x 512 21.4 -> 24.4, 64 x 800 31.2 -> 33.2, 24 x 2048 61 -> 57; 128 x 128
// 7.7 -> 8.0.
bool bwd_in_one_launch(int BH, int S, int D, bool drop) {
  const long long cus = device_cus(), wgs = (long long)BH * ((S + 127) / 128);
  const bool full_round = 8LL * BH >= 7 * cus && BH <= cus;
  if (D == 64 && !drop && full_round && S >= 224 && S <= kOwnDeltaMaxS) return false;
  if (S <= 256) {
    if (D == 32) return drop || wgs <= (S <= 128 ? 13 : 8) * cus;
    return wgs <= (S <= 128 && !drop ? 13 : 5) * cus;
  }
  if (drop && D == 32 && S > 512) return 2 * (wgs + BH) <= 3 * cus;
  return 2 * (wgs + BH) <= 9 * cus;
}
BwdPlan bwd_plan(int BH, int S, int D, bool drop) {
  if (!bwd_in_one_launch(BH, S, D, drop)) return {kSeparate, waves_per_group(BH, S, D, drop)};
  const long long cus = device_cus(), rows64 = (long long)BH * ((S + 63) / 64);
  const bool two = S > 64 && (S <= 128    ? 2 * rows64 <= cus
                              : S < 1024 ? 2 * rows64 <= 3 * cus
                                         : rows64 <= 3 * cus);
  return {S <= kOwnDeltaMaxS ? kOneOwnDelta : kOneAfterDelta, two ? 2 : 1};
}

template <int D>
hipError_t launch_bwd_bf16_t(bf16* dq, bf16* dk, bf16* dv, float* delta, const bf16* dout,
                             const bf16* out, const float* lse, const bf16* q, const bf16* k,
                             const bf16* v, int BH, int S, float scale, const AttnLayout& L,
                             hipStream_t stream, int phases, const Dropout* drop) {
  hipError_t e = hipSuccess;
  const bool contiguous = is_contiguous(L, S, D);
  const DropParams dr = drop_params(drop);  // dropout: contiguous layout only (caller checks)
  auto span = [&](const bf16* p, int t) {  // tensor t's extent
    const HeadStrides& h = L.t[t];
    const size_t batches = BH / L.n_heads, heads = L.n_heads, rows = S;
    return Span{p, 2 * ((batches - 1) * h.batch + (heads - 1) * h.head + (rows - 1) * h.row + D)};
  };
  // The phase calls, and a backward in place (dk = k, dv = v, or any gradient = out), run dQ first,
  // then dK/dV.
  const bool separate =
      phases != kBwdAll || in_place({span(dq, kTDQ), span(dk, kTDK), span(dv, kTDV)},
                                    {span(q, kTQ), span(k, kTK), span(v, kTV), span(dout, kTDO),
                                     span(out, kTO)});
  const BwdPlan plan = separate ? BwdPlan{kSeparate, waves_per_group(BH, S, D, drop != nullptr)}
                                : bwd_plan(BH, S, D, drop != nullptr);
  if ((phases & kBwdDelta) || plan.how == kOneAfterDelta) {
    const long long rows = (long long)BH * S;
    const int row_blocks = (S + 31) / 32;
    if (contiguous)
      delta_bf16_kernel<D, false><<<(unsigned)((rows + 31) / 32), 256, 0, stream>>>(
          delta, dout, out, S, rows, row_blocks, L);
    else
      delta_bf16_kernel<D, true><<<(unsigned)BH * row_blocks, 256, 0, stream>>>(
          delta, dout, out, S, rows, row_blocks, L);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  // dQ: P = exp2(S * scale * log2(e) - lse * log2(e)) holds for either sign of the scale. dK/dV:
  // s = S - lse/scale needs a nonzero scale: a zero one (P = exp(-lse)) runs with 1e-30, whose
  // S*scale terms are then below fp32 resolution next to lse/scale.
  const float se = scale != 0.f ? scale : 1e-30f;
  const BwdArgs args{dq, dk, dv, delta, q,     k,     v,          dout,
                     out, lse, S, scale, scale * kLog2e, se * kLog2e, -1.0f / se, L, dr};
  const int ks = plan.waves_per_group;
  const unsigned blocks = (unsigned)((S + 32 * kWaves / ks - 1) / (32 * kWaves / ks));
  with_shape(ks, drop != nullptr, !contiguous, [&](auto strided, auto dropped, auto w) {
    if (plan.how == kOneOwnDelta)
      bwd_bf16_kernel<D, strided(), dropped(), w(), true>
          <<<dim3(BH, blocks, 2), 64 * kWaves, 0, stream>>>(args);
    else if (plan.how == kOneAfterDelta)
      bwd_bf16_kernel<D, strided(), dropped(), w(), false>
          <<<dim3(BH, blocks, 2), 64 * kWaves, 0, stream>>>(args);
    if (plan.how != kSeparate) {
      e = hipGetLastError();
      return;
    }
    const dim3 grid(BH, blocks);
    if (phases & kBwdDq) {
      dq_bf16_kernel<D, strided(), dropped(), w()><<<grid, 64 * kWaves, 0, stream>>>(args);
      if ((e = hipGetLastError()) != hipSuccess) return;
    }
    if (phases & kBwdDkdv) {
      dkdv_bf16_kernel<D, strided(), dropped(), w()><<<grid, 64 * kWaves, 0, stream>>>(args);
      e = hipGetLastError();
    }
  });
  return e;
}

}  // namespace

hipError_t launch_bwd_bf16(bf16* dq, bf16* dk, bf16* dv, float* delta, const bf16* dout,
                           const bf16* out, const float* lse, const bf16* q, const bf16* k,
                           const bf16* v, int BH, int S, int D, float scale,
                           const AttnLayout& layout, hipStream_t stream, int phases,
                           const Dropout* drop) {
  if (drop != nullptr && drop->p == 0.f) drop = nullptr;  // nothing to draw: the plain kernels
  if (D == 64)
    return launch_bwd_bf16_t<64>(dq, dk, dv, delta, dout, out, lse, q, k, v, BH, S, scale,
                                 layout, stream, phases, drop);
  if (D == 32)
    return launch_bwd_bf16_t<32>(dq, dk, dv, delta, dout, out, lse, q, k, v, BH, S, scale,
                                 layout, stream, phases, drop);
  return hipErrorInvalidValue;
}

}  // namespace dadgpt
