// Launch functions of the attention kernels (host side of each .hip file). Arguments are
// validated by capi.cpp before any of these is called; every function returns the
// hipGetLastError() status of its own launches.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>

namespace dadgpt {

typedef __bf16 bf16;

// Where the rows of one (b, h) slice of a bf16 attention tensor lie: row s of slice
// bh = b * n_heads + h starts at element b * batch + h * head + s * row, and its D elements
// are contiguous. A contiguous [BH, S, D] tensor is {S * D, 0, D} with n_heads = 1; the
// token-major [B * S, H * D] layout of the projections is {S * H * D, D, H * D}. The host
// keeps every stride a multiple of 8 elements (16 bytes) and row below 2^24.
struct HeadStrides {
  long long batch, head;
  int row;
};
enum AttnTensor { kTQ, kTK, kTV, kTO, kTDO, kTDQ, kTDK, kTDV, kAttnTensors };
struct AttnLayout {
  int n_heads;
  HeadStrides t[kAttnTensors];
};

inline AttnLayout contiguous_layout(int S, int D) {
  AttnLayout L{};
  L.n_heads = 1;
  for (auto& t : L.t) t = HeadStrides{(long long)S * D, 0, D};
  return L;
}

// Whether `L` places every tensor as contiguous [BH, S, D] (the kernels then use their
// compile-time contiguous addressing). Unit-stride heads count: b * H * S * D + h * S * D is
// the same element as bh * S * D.
inline bool is_contiguous(const AttnLayout& L, int S, int D) {
  const long long slice = (long long)S * D;
  for (const auto& t : L.t)
    if (t.row != D || t.head != slice || t.batch != slice * L.n_heads) {
      if (L.n_heads == 1 && t.row == D && t.batch == slice) continue;  // head unused
      return false;
    }
  return true;
}

// Whether two buffers share memory (their whole extents: interleaved rows count).
struct Span {
  const void* p;
  size_t bytes;
};
inline bool overlap(const Span& a, const Span& b) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a.p), y = reinterpret_cast<uintptr_t>(b.p);
  return x < y + b.bytes && y < x + a.bytes;
}
// Whether any of a backward's gradients shares memory with what it reads. Each workgroup reads
// its own rows of some inputs (dK/dV of K and V, dQ of Q, dO and O) before it writes theirs, so
// a gradient may take such an input's place, but only while the kernels run one after the other:
// in one launch the other kind's workgroups still read it.
inline bool in_place(std::initializer_list<Span> gradients, std::initializer_list<Span> inputs) {
  for (const Span& g : gradients)
    for (const Span& x : inputs)
      if (overlap(g, x)) return true;
  return false;
}

// Attention-probability dropout of a call: rate p in [0, 1) and the generator's seed (the
// mask definition is in dropout.hpp). The host checks p; dropout runs on the contiguous
// layout only.
struct Dropout {
  float p;
  uint64_t seed;
};

// Compute units of the current device (cached per device; 0 if unknown).
int device_cus();

// Waves per 32-row group in the bf16 kernels. A workgroup is four waves over 64-row tiles: with
// one wave per group it owns 128 rows (queries, or keys in dK/dV), each wave taking both
// 32-row chunks of a tile; with two it owns 64, two waves taking one chunk of each tile and
// merging at the end. Two make the chain of the longest workgroup half as long and its stream
// twice as expensive per row, so they pay where a grid is so small that it lasts as long as that
// chain, and cost 5-15% where the CUs are full anyway. Forward, one wave -> two, us (BH x S,
// D = 64): 48 x 1024 16.8 -> 14.3, 64 x 1024 18.2 -> 16.1, 72 x 1024 18.8 -> 19.1, 96 x 1024
// 21.5 -> 23.4; 36 x 2048 32.4 -> 29.0, 48 x 2048 35.7 -> 35.9; 12 x 4096 55 -> 39.6, 24 x 4096
// 64.4 -> 64.3; 96 x 512 11.7 -> 10.5, 100 x 520 11.6 -> 10.5, 128 x 512 11.8 -> 11.8, 192 x 512
// 16.1 -> 19.2: the line is at 2.4 128-row workgroups per CU, one more per head counted. Short
// sequences (S <= 256, at most two tiles' worth of chain to save) need one 64-row workgroup per
// CU: 128 x 128 5.5 -> 5.2, 192 x 128 5.6 -> 5.7, 192 x 256 7.6 -> 8.1; one tile (S <= 64) has
// nothing to share. At D = 32, where half the registers leave more workgroups resident, and with
// dropout, whose generator lengthens the chain, the line lies further out: D = 32 72 x 1024
// 14.4 -> 12.8, 96 x 1024 14.8 -> 14.8; dropout, forward and dQ + dK/dV 96 x 1024 32 / 99 ->
// 31 / 92, 128 x 1024 35.3 / 110 -> 37.5 / 115, 128 x 512 14.6 / 41.1 -> 14.6 / 42.7. (The backward
// follows this only where it runs as two launches, see bwd_plan.)
inline int waves_per_group(int BH, int S, int D, bool drop) {
  if (S <= 64) return 1;
  const long long cus = device_cus(), wgs = (long long)BH * ((S + 127) / 128 + 1);
  bool two;
  if (D == 32)
    two = wgs <= 3 * cus;
  else if (S <= 256)
    two = (long long)BH * ((S + 63) / 64) <= cus;
  else if (drop && S > 512)
    two = 2 * wgs <= 7 * cus;
  else
    two = 5 * wgs <= 12 * cus;
  return two ? 2 : 1;
}

// Causal flash forward, bf16 in/out, fp32 logsumexp (natural log) [BH, S]. q, k, v, out as
// `layout` places them (tensors kTQ, kTK, kTV, kTO), D in {32,64}. With `drop`, the
// probabilities multiplying V are dropped (the logsumexp is that of the undropped scores).
hipError_t launch_fwd_bf16(bf16* out, float* lse, const bf16* q, const bf16* k, const bf16* v,
                           int BH, int S, int D, float scale, const AttnLayout& layout,
                           hipStream_t stream, const Dropout* drop = nullptr);

// Causal flash backward, bf16 in/out. delta [BH,S] fp32 is written (scratch, as the
// reference's). dq/dk/dv are overwritten. `phases` selects the kernels launched, in order:
// bit 1 dQ (which also computes and writes delta), bit 2 dK/dV (reads delta); kBwdAll is the
// whole backward, which may run both in one launch. Bit 0 launches the standalone delta kernel
// (a separate pass, equal up to fp32 summation order; not part of kBwdAll).
constexpr int kBwdDelta = 1, kBwdDq = 2, kBwdDkdv = 4, kBwdAll = kBwdDq | kBwdDkdv;
hipError_t launch_bwd_bf16(bf16* dq, bf16* dk, bf16* dv, float* delta, const bf16* dout,
                           const bf16* out, const float* lse, const bf16* q, const bf16* k,
                           const bf16* v, int BH, int S, int D, float scale,
                           const AttnLayout& layout, hipStream_t stream, int phases = kBwdAll,
                           const Dropout* drop = nullptr);

// fp32 flash forward/backward (the reference's own precision), optionally with dropout.
hipError_t launch_fwd_f32(float* out, float* lse, const float* q, const float* k,
                          const float* v, int BH, int S, int D, float scale, hipStream_t stream,
                          const Dropout* drop = nullptr);
hipError_t launch_bwd_f32(float* dq, float* dk, float* dv, float* delta, const float* dout,
                          const float* out, const float* lse, const float* q, const float* k,
                          const float* v, int BH, int S, int D, float scale,
                          hipStream_t stream, const Dropout* drop = nullptr);

// Decode over ragged KV caches [n_seq,H,max_len,D]. A cache longer than one workgroup chunk
// (512 keys bf16, 256 fp32 at D=64) is split into chunks merged inside the kernel through the
// workspace: arrival counters at its start, fp32 partials packed against its end (its full
// size, workspace_bytes, places them). decode_workspace_bytes is 0 when no split is needed.
size_t decode_workspace_bytes(int n_seq, int H, int max_len, int D);
hipError_t launch_decode_bf16(bf16* out, const bf16* q, const bf16* k_cache,
                              const bf16* v_cache, const int* lens, int n_seq, int H,
                              int max_len, int D, float scale, void* workspace,
                              size_t workspace_bytes, hipStream_t stream);
hipError_t launch_decode_f32(float* out, const float* q, const float* k_cache,
                             const float* v_cache, const int* lens, int n_seq, int H,
                             int max_len, int D, float scale, void* workspace,
                             size_t workspace_bytes, hipStream_t stream);

// Row kernels of the materialized attention path (materialized.hip), fp32 [rows, cols]:
// the reference's softmax (out may be in), softmax backward (din += p (dout - rowsum(dout p))),
// causal fill of n_blocks S x S blocks (value above the diagonal) and scale; and the fused
// chains: attention_probs turns raw scores [BH, S, S] into probabilities in place (x scale,
// causal mask, softmax), attention_probs_backward writes d(scores) from d(probs) and probs
// (softmax backward, causal zero, x scale; ds may be dp), decode_probs turns decode scores
// [n_seq * H, max_len] into probabilities over each sequence's first lens[seq] keys.
hipError_t launch_softmax_rows(float* out, const float* in, long long rows, int cols,
                               hipStream_t stream);
hipError_t launch_softmax_backward_rows(float* din, const float* dout, const float* p,
                                        long long rows, int cols, hipStream_t stream);
hipError_t launch_causal_fill(float* m, int n_blocks, int S, float value, hipStream_t stream);
hipError_t launch_scale(float* x, long long n, float scale, hipStream_t stream);
hipError_t launch_attention_probs(float* p, int BH, int S, float scale, hipStream_t stream);
hipError_t launch_attention_probs_backward(float* ds, const float* dp, const float* p, int BH,
                                           int S, float scale, hipStream_t stream);
hipError_t launch_decode_probs(float* p, const int* lens, int n_seq, int H, int max_len,
                               float scale, hipStream_t stream);
// Attention-probability dropout of the materialized path, with the flash kernels' mask
// (dropout.hpp): out [BH, S, S] = p * keep / (1 - drop.p) (out may be p); and the backward row
// pass ds = causal_zero(softmax_backward(dpd * keep / (1 - drop.p), p)) * scale (ds may be dpd).
hipError_t launch_attention_dropout(float* out, const float* p, int BH, int S,
                                   const Dropout& drop, hipStream_t stream);
hipError_t launch_attention_probs_backward_dropout(float* ds, const float* dpd, const float* p,
                                                   int BH, int S, float scale,
                                                   const Dropout& drop, hipStream_t stream);
// The reference's head split [B*S, H*dh] -> [B*H, S, dh] and merge (its inverse), fp32
// (materialized.hip). out and in do not overlap; B*S < 2^31 rows.
hipError_t launch_split_heads(float* out, const float* in, int B, int S, int H, int dh,
                              hipStream_t stream);
hipError_t launch_merge_heads(float* out, const float* in, int B, int S, int H, int dh,
                              hipStream_t stream);

// Device scratch that stands in for the decode workspace in the allocation-free entry point:
// kDecodeScratchBytes per device, held until the process ends. decode_scratch returns the
// current device's address, looked up (and zero-filled by a kernel on `stream`) on the first
// call on that device.
constexpr size_t kDecodeScratchBytes = size_t(4) << 20;
hipError_t decode_scratch(void** ptr, hipStream_t stream);

}  // namespace dadgpt
