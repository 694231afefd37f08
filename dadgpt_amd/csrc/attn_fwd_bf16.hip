// Causal flash-attention forward for gfx950: bf16 Q/K/V/O, fp32 accumulation and softmax,
// fp32 natural-log logsumexp. Replaces the role of flash_fwd_kernel (cuda/attention.cu:17-73)
// at bf16; the fp32 path is attn_f32.hip.
//
// Work decomposition: one workgroup = WAVES waves x NQB*32 queries of one (b,h) slice; it
// walks the 64-key tiles up to its last query (causal tile skipping). Each wave owns NQB
// 32-query MFMA blocks and handles each key tile as two 32-key chunks; on small grids (KS = 2,
// waves_per_group) a workgroup owns half the queries, two waves share each query block, taking
// one chunk of every tile each, and their (m, l, O) are merged at the end. Per chunk and wave, on
// v_mfma_f32_32x32x16_bf16:
//   S^T[key][query] = K . Q^T   A = K rows from LDS (rows loaded through sigma32), B = Q held
//                               in registers for the whole kernel; one K operand read feeds
//                               every query block of the wave
//   online softmax in registers: each lane owns one query, so the row max is an in-lane max3
//                               chain plus one exchange with the other lane half
//   O^T[d][query] += V^T . P^T  A = V^T read across the rows of the row-major V tile with
//                               ds_read_b64_tr_b16, B = P straight from the score registers
//                               (bf16), no lane exchange
//
// VALU per score, the forward's other bound at d_head 64: the scale is folded into the
// exponent (one FMA: exp2(s*c - m)), the bf16 pack takes half a v_cvt_pk and the row sum one
// fp32 add (in fp32, before the bf16 rounding, so the saved logsumexp keeps fp32 accuracy).
// The running maximum m is not recomputed per chunk: it moves only when a chunk's P would
// reach 2^64 (see fwd_softmax_pv), so the row max leaves the per-chunk path. The causal mask
// costs no VALU either: a diagonal chunk's score MFMAs start from an accumulator of 0 / -inf
// read from a per-lane table in LDS, so masked scores arrive as -inf and exponentiate to
// exactly 0.
//
// The launch bound caps registers so that several waves share each SIMD, which interleaves
// one wave's softmax with another's MFMAs and covers LDS latency. K and V tiles are
// double-buffered in LDS and staged by direct global->LDS loads (no registers, no LDS-store
// instructions): tile t+1 is in flight while tile t is on the MFMA pipes; one barrier per
// tile. (Triple buffering measured slower: the third buffer's LDS cost more than the extra
// tile of lead gained.)
//
// Instantiations: STRIDED reads q, k, v and writes out at per-tensor (batch, head, row)
// strides (the token-major layout of the projections) instead of contiguous [BH, S, D]; DROP
// multiplies the probabilities that reach P V by keep/(1-p) (dropout.hpp), leaving the
// normaliser and logsumexp those of the undropped row.
#include "common.hpp"
#include "dropout.hpp"
#include "kernels.hpp"
#include "tiles.hpp"

namespace dadgpt {
namespace {

// Geometry: NQB 32-query blocks per wave, WAVES waves per workgroup, MINB workgroups per CU
// the register budget is sized for (512 / (MINB * WAVES / 4) per lane). The kernel takes 127
// registers and 36 KB of LDS, so up to 4 workgroups (4 waves per SIMD) are resident per CU
// when the grid has them (per-workgroup stamps at B16 H12 T1024 show 4). 4-wave workgroups of
// one query block measured fastest: 8- and 16-wave workgroups and two query blocks per wave
// were no faster, and 2-wave workgroups (twice as many, for small batches) were slower at
// both B16 and B8.
#ifndef DADGPT_FWD_NQB
#define DADGPT_FWD_NQB 1
#endif
#ifndef DADGPT_FWD_WAVES
#define DADGPT_FWD_WAVES 4
#endif
#ifndef DADGPT_FWD_MINB
#define DADGPT_FWD_MINB 3
#endif
constexpr int kNQB = DADGPT_FWD_NQB;
constexpr int kQW = 32 * kNQB;            // queries per wave
constexpr int kWaves = DADGPT_FWD_WAVES;  // waves per workgroup
constexpr int kMinBlocks = DADGPT_FWD_MINB;
// A chunk whose P reaches this in some row moves the running maximum (see fwd_softmax_pv):
// with P < 2^64, O and l stay far inside fp32 range over any sequence length.
constexpr float kMaxP = 0x1p64f;
// The diagonal-chunk mask table assumes one query block per wave: a wave's chunks are then
// either fully visible or its diagonal chunk (first key = first query).
static_assert(kNQB == 1, "one 32-query block per wave");

// Causal mask of a diagonal chunk (first key = first query of the wave) in score-accumulator
// layout: element r of lane (l32, hi) holds key 16*(r>>3) + 8*hi + (r&7) of query l32, -inf
// where the key comes after the query. Stored as table[j][lane] = elements 4j..4j+3.
__device__ __forceinline__ void write_mask_table(f32x4 (*table)[64], int lane) {
  const int l32 = lane & 31, hi = lane >> 5;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 m;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * j + e;
      m[e] = 16 * (r >> 3) + 8 * hi + (r & 7) > l32 ? neg_inf() : 0.0f;
    }
    table[j][lane] = m;
  }
}
__device__ __forceinline__ f32x16 read_mask_table(const f32x4 (*table)[64], int lane) {
  f32x16 m;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const f32x4 v = table[j][lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) m[4 * j + e] = v[e];
  }
  return m;
}

// K operands of one 32-key chunk (tile keys 32*kb ..): A operands of S^T = K Q^T, K rows read
// through sigma32 so that register r of lane half hi holds key 32kb + 16*(r>>3) + 8*hi + (r&7).
template <int D>
__device__ __forceinline__ void fwd_k_ops(bf16x8 (&ka)[D / 16], const bf16* lk, int kb,
                                          int lane) {
  const int l32 = lane & 31, hi = lane >> 5;
  const int krow = 32 * kb + sigma32(l32);
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds) ka[ds] = lds_op(lk, rm_off<D>(krow, 2 * ds + hi));
}

// s[i] = init + K[chunk] Q_i^T for the wave's NQB query blocks; each K operand feeds every
// block. init is 0, or the causal mask's 0 / -inf for a diagonal chunk.
template <int D, int NQB>
__device__ __forceinline__ void fwd_scores(f32x16 (&s)[NQB], const bf16x8 (&qop)[NQB][D / 16],
                                           const bf16x8 (&ka)[D / 16], const f32x16& init) {
#pragma unroll
  for (int i = 0; i < NQB; ++i) s[i] = init;
#pragma unroll
  for (int ds = 0; ds < D / 16; ++ds)
#pragma unroll
    for (int i = 0; i < NQB; ++i) s[i] = mfma32(ka[ds], qop[i][ds], s[i]);
}

// V^T operands of one chunk (A of O^T += V^T P^T), read across the rows of the V tile.
template <int D>
__device__ __forceinline__ void fwd_v_ops(bf16x8 (&va)[D / 32][2], const bf16* lv, int kb,
                                          int lane) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int j = 0; j < 2; ++j) va[db][j] = lds_tr_op<D>(lv, 32 * kb + 16 * j, 32 * db, lane);
}

// P = exp2(s*c - m) of one chunk as bf16 B operands; returns this lane's fp32 sum of them.
// With dropout (DROP), the operands are P * keep/(1-p) (register r kept iff its uniform in
// `keep` passes the threshold) and the sum stays that of P: the normaliser and logsumexp are
// those of the undropped row.
template <bool DROP>
__device__ __forceinline__ float fwd_exp(bf16x8 (&pb)[2], const f32x16& s, float m,
                                         float scale_log2, const KeepWords16& keep,
                                         const DropParams& dr) {
  const float mneg = -m;
  float ls = 0.f;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 8 * j + 2 * e;
      const float p0 = fast_exp2(fmaf(s[r], scale_log2, mneg));
      const float p1 = fast_exp2(fmaf(s[r + 1], scale_log2, mneg));
      if constexpr (DROP)
        w[e] = pack_bf16x2(p0 * keep_factor(keep, r, dr), p1 * keep_factor(keep, r + 1, dr));
      else
        w[e] = pack_bf16x2(p0, p1);
      // (the first pair starts the sum: 0 + x cannot be folded, since it maps -0 to +0)
      ls = r == 0 ? p0 + p1 : ls + (p0 + p1);
    }
    pb[j] = as_bf16x8(w);
  }
  return ls;
}

// What a row's exponentials are taken against: its running maximum, or 0 while every score it
// has seen is -inf (then each P is exp2(-inf) = 0, where -inf - (-inf) would make the row NaN for
// good; a second wave's first chunk may be such keys alone). A NaN maximum stays NaN: compared on
// the bits, as this file is built assuming no NaNs.
__device__ __forceinline__ float finite_max(float m) {
  return __float_as_uint(m) == __float_as_uint(neg_inf()) ? 0.f : m;
}

// Online softmax of one chunk's scores (masked ones already -inf) and
// O^T += V^T[:, chunk] P^T.
//
// The exponentials are taken against the running maximum m as it stands, without the
// chunk's own maximum: m only has to keep P finite and away from the fp32 limits, not equal
// the true maximum (O and l carry the same factor 2^-m, which the epilogue's division and
// lse = m + log2 l remove). A chunk whose P reaches 2^kMaxLog2P in some row (or is
// inf/NaN: m is -inf before a row's first chunk) takes the slow path: m moves to the
// chunk's maximum, O and l are rescaled, and the chunk's exponentials are redone. That is a
// wave's first chunk and, for ordinary scores, almost nothing else, so the row maximum is
// off the per-chunk path.
template <int D, int NQB, bool DROP>
__device__ __forceinline__ void fwd_softmax_pv(f32x16 (&s)[NQB], f32x16 (&oacc)[NQB][D / 32],
                                               float (&mrun)[NQB], float (&lrun)[NQB],
                                               const bf16x8 (&va)[D / 32][2], float scale_log2,
                                               const KeepWords16 (&keep)[NQB],
                                               const DropParams& dr) {
  constexpr int DB = D / 32;
  bf16x8 pb[NQB][2];
#pragma unroll
  for (int i = 0; i < NQB; ++i) {
    float ls = fwd_exp<DROP>(pb[i], s[i], mrun[i], scale_log2, keep[i], dr);
    // ls >= 2^64, +inf or NaN, compared on the bits: a row's first chunk with masked keys sums
    // to NaN (exp2 of -inf - (-inf)), and this file is built assuming no NaNs, under which a
    // floating-point compare may be folded to one that NaN fails. ls is +0, positive or NaN,
    // and the unsigned compare holds for every NaN (a negative one through its sign bit). Each
    // row then takes the slow path on its own first chunk, whatever its wave-mates hold (a NaN
    // query row included), and only the rows that need it move their maximum: the others keep
    // m (a correction of exp2(0) = 1 and the same exponentials), so no row's bits depend on
    // another row.
    const bool need = __float_as_uint(ls) >= __float_as_uint(kMaxP);
    if (__builtin_amdgcn_ballot_w64(need) != 0) {  // wave-uniform
      float mx = s[i][0];
#pragma unroll
      for (int r = 1; r < 15; r += 2) mx = fmaxf(fmaxf(mx, s[i][r]), s[i][r + 1]);
      // every row of a chunk the wave computes has an unmasked key: mx is -inf only if every
      // score of the row so far is
      mx = max_halves(fmaxf(mx, s[i][15])) * scale_log2;
      // the two lane halves of a row hold different keys of it, and P V sums both against one
      // maximum: the row moves it if either half needs to
      const float mnew = or_halves(need) ? fmaxf(mrun[i], mx) : mrun[i];
      const float mref = finite_max(mnew);
      const float corr = fast_exp2(mrun[i] - mref);  // 0 on a row's first chunk
      mrun[i] = mnew;
      lrun[i] *= corr;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[i][db] *= corr;
      ls = fwd_exp<DROP>(pb[i], s[i], mref, scale_log2, keep[i], dr);
    }
    lrun[i] += ls;
  }
  // ---- O^T += V^T[:, chunk] P^T; each V^T operand read once for every query block ----
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < NQB; ++i) oacc[i][db] = mfma32(va[db][j], pb[i][j], oacc[i][db]);
}

// FRESH: V's tile-edge correction computed at each issue (DmaTile::load_any).
template <int D, bool STRIDED, bool DROP, int KS, bool FRESH = false>
__global__ __launch_bounds__(64 * kWaves, kMinBlocks)
__attribute__((amdgpu_num_vgpr(512 / (kMinBlocks * kWaves / 4)))) void fwd_bf16_kernel(
    bf16* __restrict__ out, float* __restrict__ lse, const bf16* __restrict__ q,
    const bf16* __restrict__ k, const bf16* __restrict__ v, int S, float scale_log2,
    int negate_q, int snake, const AttnLayout L, const DropParams dr) {
  // scale_log2 = |scale| * log2(e); a negative scale is applied by negating Q (exact in bf16),
  // so the row max of the raw scores is the row max of the scaled ones.
  constexpr int kGroups = kWaves / KS, QB = kQW * kGroups;  // query groups, queries
  constexpr int DS = D / 16;  // 16-wide K-steps along D
  constexpr int DB = D / 32;  // 32-row blocks of O^T
  // K and V tiles, double-buffered: tile t is read while t+1 is in flight. With the tile loop
  // unrolled by two every access names its buffer by a constant index, so the compiler
  // addresses both from one register.
  __shared__ __attribute__((aligned(16))) bf16 sk[2][kTileRows * D];
  __shared__ __attribute__((aligned(16))) bf16 sv[2][kTileRows * D];
  __shared__ f32x4 smask[4][64];
  static_assert(kWaves * kQW <= 2 * kTileRows, "the epilogue stages every wave's rows in sk");
  static_assert(KS == 1 || sizeof(sk) >= kGroups * (D / 32) * sizeof(AccLds),
                "the second waves' partials fit sk");

  // Dispatch order: longest (latest) query blocks first, (b,h) fastest. With `snake` > 0 (a grid
  // that fits on the CUs in one round) every other group of `snake` workgroups in dispatch
  // order is reversed, so the workgroups a CU receives pair long query blocks with short ones.
  int bh = blockIdx.x, yrev = blockIdx.y;
  if (snake > 0) {
    const int i = blockIdx.y * gridDim.x + blockIdx.x, g = i / snake;
    if (g & 1) {
      const int n = min(snake, (int)(gridDim.x * gridDim.y) - g * snake);  // ids in the group
      const int j = g * snake + (n - 1 - (i - g * snake));
      bh = j % gridDim.x;
      yrev = j / gridDim.x;
    }
  }
  const int qblk = gridDim.y - 1 - yrev;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar
  const int l32 = lane & 31, hi = lane >> 5;
  const int grp = wave % kGroups, sub = wave / kGroups;
  const Slice<D, STRIDED> sl(L, bh, S);
  const bf16* qg = sl.base(q, kTQ);
  const bf16* kg = sl.base(k, kTK);
  const bf16* vg = sl.base(v, kTV);
  const int qp = sl.pitch(kTQ), kp = sl.pitch(kTK), vp = sl.pitch(kTV);  // row pitches

  const int q0 = qblk * QB + grp * kQW;
  const int wg_last = min(S, (qblk + 1) * QB) - 1;
  const int n_tiles = wg_last / kTileRows + 1;

  // B operands of S^T: lane holds query q0 + 32i + l32, columns 16*ds + 8*hi + 0..7.
  // (rows past S read row S-1: finite scores for rows that are never stored)
  bf16x8 qop[kNQB][DS];
#pragma unroll
  for (int i = 0; i < kNQB; ++i) {
    const int row = min(q0 + 32 * i + l32, S - 1);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) qop[i][ds] = ld_g128(qg + (size_t)row * qp + 16 * ds + 8 * hi);
  }

  f32x16 oacc[kNQB][DB];
  float mrun[kNQB], lrun[kNQB];  // running max (scaled log2 units); per-half row sums
#pragma unroll
  for (int i = 0; i < kNQB; ++i) {
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[i][db] = f32x16{};
    mrun[i] = neg_inf();
    lrun[i] = 0.f;
  }

  if (wave == 0) write_mask_table(smask, lane);  // published by the first barrier

  // The first tile loads alongside Q, under one wait; Q is touched only after it (the
  // compiler, which does not see the direct loads, then has nothing left to wait for).
  using Dma = DmaTile<D, kWaves>;
  uint32_t koff[Dma::PER_WAVE], voff[Dma::PER_WAVE];
  Dma::offsets(koff, wave, lane, kp);
  Dma::offsets(voff, wave, lane, vp);
  Dma::load_any(sk[0], kg, 0, S, koff, wave, lane, kp);
  Dma::load_any(sv[0], vg, 0, S, voff, wave, lane, vp);
  wait_vm_lds<0>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < kNQB; ++i)
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) {
      asm volatile("" : "+v"(qop[i][ds]));
      if (negate_q) qop[i][ds] = neg_bf16x8(qop[i][ds]);
    }

  // One key tile: prefetch tile t+1 into (nk, nv) (it held tile t-1, released by the last
  // barrier), compute tile t from (ck, cv), then wait for tile t+1 and barrier, which also
  // ends every wave's reads of tile t.
  auto tile = [&](int t, const bf16* ck, const bf16* cv, bf16* nk, bf16* nv) {
    const int k0 = t * kTileRows;
    const bool prefetch = t + 1 < n_tiles;
    if (prefetch) {
      Dma::load_any(nk, kg, k0 + kTileRows, S, koff, wave, lane, kp);
      Dma::template load_any<FRESH>(nv, vg, k0 + kTileRows, S, voff, wave, lane, vp);
    }
    if (q0 < S && k0 <= q0 + kQW - 1) {  // some key of the tile at or before a query
      // One 32-key chunk at a time (holding both chunks' scores at once measured no faster
      // and costs registers); the other waves on the SIMD cover the operand reads' latency.
#pragma unroll
      for (int i = 0; i < 2 / KS; ++i) {
        const int kb = KS == 1 ? i : sub, c0 = k0 + 32 * kb;
        if (c0 > q0 + kQW - 1) break;  // every key of the chunk after every query
        bf16x8 ka[DS], va[DB][2];
        f32x16 sc[kNQB];
        KeepWords16 keep[kNQB] = {};
        if constexpr (DROP) {
#pragma unroll
          for (int n = 0; n < kNQB; ++n)
            keep[n] = keep_words16(dr, (uint64_t)bh * S + q0 + 32 * n + l32, c0, hi);
        }
        fwd_k_ops<D>(ka, ck, kb, lane);
        // the chunk whose first key is the wave's first query is the one to mask
        if (c0 == q0)
          fwd_scores<D, kNQB>(sc, qop, ka, read_mask_table(smask, lane));
        else
          fwd_scores<D, kNQB>(sc, qop, ka, f32x16{});
        // V^T operands only now (K's are dead): their latency hides under the softmax
        __builtin_amdgcn_sched_barrier(0);
        fwd_v_ops<D>(va, cv, kb, lane);
        fwd_softmax_pv<D, kNQB, DROP>(sc, oacc, mrun, lrun, va, scale_log2, keep, dr);
      }
    }
    wait_vm_lds<0>();
    __builtin_amdgcn_s_barrier();
  };
  for (int t = 0; t < n_tiles; t += 2) {
    tile(t, sk[0], sv[0], sk[1], sv[1]);
    if (t + 1 < n_tiles) tile(t + 1, sk[1], sv[1], sk[0], sv[0]);
  }

  if constexpr (KS == 2) {
    // (m, l, O) of the group's second wave: rescaled to the larger maximum and added. A wave
    // that saw no chunk of the row, or only scores of -inf, has m = -inf and zeros, which get
    // weight 2^-inf = 0.
    AccLds* slot = reinterpret_cast<AccLds*>(&sk[0][0]) + grp * DB;
    float* ml = reinterpret_cast<float*>(&smask[0][0]) + grp * 128;
    if (sub == 1) {
      put_acc(oacc[0], slot, lane);
      ml[lane] = mrun[0];
      ml[64 + lane] = lrun[0];
    }
    __syncthreads();
    if (sub == 1) return;
    const float m1 = ml[lane], mn = fmaxf(mrun[0], m1);
    const float mref = finite_max(mn);
    const float a0 = fast_exp2(mrun[0] - mref), a1 = fast_exp2(m1 - mref);
    mrun[0] = mn;
    lrun[0] = lrun[0] * a0 + ml[64 + lane] * a1;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[0][db] *= a0;
    add_acc(oacc[0], slot, lane, a1);
  }

  // ---- epilogue: O = O^T / l, lse = ln2 * (m + log2 l) ----
#pragma unroll
  for (int i = 0; i < kNQB; ++i) {
    const int qrow = q0 + 32 * i + l32;
    const float l = sum_halves(lrun[i]);
    const float inv = 1.0f / l;
    // the tiles are free after the last barrier: each wave stages its rows in its quarter of sk
    if (q0 + 32 * i < S)
      store_rows_staged<D>(sl.row(out, kTO, q0 + 32 * i), sl.pitch(kTO), S - q0 - 32 * i,
                           oacc[i], inv,
                           &sk[0][0] + ((KS == 1 ? wave : grp * 2) * kNQB + i) * 32 * D, lane);
    if (qrow < S && hi == 0) lse[(size_t)bh * S + qrow] = (mrun[i] + __log2f(l)) * kLn2;
  }
}

template <int D>
hipError_t launch_fwd_bf16_t(bf16* out, float* lse, const bf16* q, const bf16* k, const bf16* v,
                             int BH, int S, float scale, const AttnLayout& L,
                             const Dropout* drop, hipStream_t stream) {
  const int cus = device_cus();
  // Masked scores are -inf and exponentiate as exp2(-inf * c - m), so c must be positive: a
  // zero scale (uniform attention) runs with c = 1e-30: every score below 1e22 in magnitude
  // then has |s*c - m| < 2^-25, an fp32 weight of exactly 1.
  const float c = fmaxf(fabsf(scale) * kLog2e, 1e-30f);
  const DropParams dr = drop_params(drop);
  auto launch = [&](auto strided, auto dropped, auto ks) {
    constexpr int QB = kQW * kWaves / ks();
    const dim3 grid(BH, (S + QB - 1) / QB);
    // Snake order only for grids of at most kMinBlocks workgroups per CU (all resident at once,
    // the dispatcher dealing each CU the same number): measured 2% faster at B8 H12 T1024 (768
    // workgroups, 3 per CU) and 6% slower at B16 (1,536).
    const int snake =
        cus > 0 && (long long)grid.x * grid.y <= (long long)cus * kMinBlocks ? cus : 0;
    auto run = [&](auto fresh) {
      fwd_bf16_kernel<D, strided(), dropped(), ks(), fresh()><<<grid, 64 * kWaves, 0, stream>>>(
          out, lse, q, k, v, S, c, scale < 0.f, snake, L, dr);
    };
    // With K's and V's edge corrections held, the two-wave strided kernel takes 129 registers,
    // three workgroups per CU; where the grid has more, V's is computed at each issue (125, four):
    // 96 x 600 token-major 13.2 -> 11.4 us, 120 x 467 12.3 -> 10.5, 64 x 900 16.2 -> 13.8, 48 x
    // 1200 17.2 -> 16.9, 60 x 777 11.5 -> 11.7; not on smaller grids (12 x 916 11.2 -> 11.8) or
    // longer rows, which last as long as one chain (36 x 1500 17.9 -> 19.1). (K's as well: 119
    // registers, 24 x 1024 12.5 -> 13.9.)
    if constexpr (D == 64 && strided() && ks() == 2)
      if (S <= 1200 && (long long)grid.x * grid.y > 3LL * cus) return run(std::true_type{});
    run(std::false_type{});
  };
  // dropout: contiguous layout only (checked by the caller)
  with_shape(waves_per_group(BH, S, D, drop != nullptr), drop != nullptr,
             !is_contiguous(L, S, D), launch);
  return hipGetLastError();
}

}  // namespace

int device_cus() {
  constexpr int kMaxDevices = 64;
  static int cus[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    cus[dev] = n;
  }
  return cus[dev];
}

hipError_t launch_fwd_bf16(bf16* out, float* lse, const bf16* q, const bf16* k, const bf16* v,
                           int BH, int S, int D, float scale, const AttnLayout& layout,
                           hipStream_t stream, const Dropout* drop) {
  if (drop != nullptr && drop->p == 0.f) drop = nullptr;  // the plain kernel's bits, undrawn
  if (D == 64)
    return launch_fwd_bf16_t<64>(out, lse, q, k, v, BH, S, scale, layout, drop, stream);
  if (D == 32)
    return launch_fwd_bf16_t<32>(out, lse, q, k, v, BH, S, scale, layout, drop, stream);
  return hipErrorInvalidValue;
}

}  // namespace dadgpt
