// Host-only half of the launchers of include/fa_fwd.h and include/fa_bwd.h: argument validation, kernel choice and
// workspace sizes.  Plain C++ without any HIP construct, so that a CPU build with sanitizers can exercise it
// (tests/test_cabi_host.py); fa_fwd_kernels.hip and fa_bwd_kernels.hip include it.  The checks restate those of
// torch_mlu's launchers (torch_mlu/csrc/aten/operators/cnnl/internal/FlashAttention_internal.cpp:73-127 forward,
// :288-366 backward) at the level of raw pointers and strides.
#ifndef FA_HOST_H_
#define FA_HOST_H_

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include "fa_bwd.h"
#include "fa_fwd.h"

namespace fa {
namespace host {

// ---- forward ------------------------------------------------------------------------------------------------
inline int padded_dim(int d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }
constexpr int64_t kMaxRowStrideBytes = 0xffffffffLL / 128;  // 128 rows x stride must fit an unsigned 32-bit offset
constexpr int32_t kMaxSeqlen = 1 << 29;                      // rows / keys per sequence

inline int validate(const fa_fwd_params* p) {
  if (!p) return FA_ERR_BAD_ARG;
  if (!p->q || !p->k || !p->v || !p->out || !p->lse) return FA_ERR_BAD_ARG;
  if ((p->cu_seqlens_q == nullptr) != (p->cu_seqlens_k == nullptr)) return FA_ERR_BAD_ARG;
  if (p->batch <= 0 || p->heads_q <= 0 || p->heads_k <= 0) return FA_ERR_BAD_ARG;
  if (p->seqlen_q < 0 || p->seqlen_k < 0 || p->head_dim <= 0) return FA_ERR_BAD_ARG;
  if (p->reserved != 0) return FA_ERR_BAD_ARG;
  if (p->dtype != FA_DTYPE_FP16 && p->dtype != FA_DTYPE_BF16) return FA_ERR_UNSUPPORTED;
  if (p->head_dim > 256 || (p->head_dim & 7)) return FA_ERR_UNSUPPORTED;
  if (p->heads_q % p->heads_k) return FA_ERR_UNSUPPORTED;
  // lengths and (sequence, head) counts that keep the kernels' 32-bit row / block arithmetic (row + Lk - Lq, grid
  // sizes) and the 64-bit products below from overflowing
  if (p->seqlen_q > kMaxSeqlen || p->seqlen_k > kMaxSeqlen) return FA_ERR_UNSUPPORTED;
  if ((int64_t)p->batch * p->heads_q > 0x7fffffffLL) return FA_ERR_UNSUPPORTED;
  if (p->kernel < FA_KERNEL_AUTO || p->kernel > FA_KERNEL_SPLITKV) return FA_ERR_BAD_ARG;
  if (p->num_splits < 0 || p->num_splits > FA_MAX_SPLITS) return FA_ERR_BAD_ARG;
  // 16-byte vector access on every row: base pointers and row strides must be multiples of 8 elements
  const uintptr_t al = (uintptr_t)p->q | (uintptr_t)p->k | (uintptr_t)p->v | (uintptr_t)p->out;
  if (al & 15) return FA_ERR_BAD_ARG;
  if ((uintptr_t)p->lse & 3) return FA_ERR_BAD_ARG;
  const int64_t st[] = {p->q_stride_s, p->q_stride_h, p->k_stride_s, p->k_stride_h, p->v_stride_s, p->v_stride_h,
                        p->o_stride_s, p->o_stride_h};
  for (int64_t s : st)
    if (s < 0 || (s & 7)) return FA_ERR_BAD_ARG;
  if (!p->cu_seqlens_q) {
    const int64_t sb[] = {p->q_stride_b, p->k_stride_b, p->v_stride_b, p->o_stride_b};
    for (int64_t s : sb)
      if (s < 0 || (s & 7)) return FA_ERR_BAD_ARG;
    if (p->lse_stride_b < 0) return FA_ERR_BAD_ARG;
  }
  if (p->lse_stride_h < 0 || p->lse_stride_s < 0) return FA_ERR_BAD_ARG;
  // the kernels form per-lane byte offsets inside a tile (up to 128 rows) as 32-bit row x 32-bit stride
  if (p->k_stride_s > kMaxRowStrideBytes / 2 || p->v_stride_s > kMaxRowStrideBytes / 2 ||
      p->q_stride_s > kMaxRowStrideBytes / 2)
    return FA_ERR_UNSUPPORTED;
  if (p->is_causal < FA_MASK_NONE || p->is_causal > FA_MASK_CAUSAL_TOP_LEFT) return FA_ERR_BAD_ARG;
  if (p->reserved2 != 0 || !(p->dropout_p >= 0.f && p->dropout_p < 1.f)) return FA_ERR_BAD_ARG;
  if (p->dropout_p > 0.f) {
    if (p->kernel == FA_KERNEL_SPLITKV && p->dropout_mask) return FA_ERR_UNSUPPORTED;  // only the tile kernel writes the debug mask
    if (p->dropout_mask && ((uintptr_t)p->dropout_mask & 3)) return FA_ERR_BAD_ARG;
    if (((uintptr_t)p->rng_seed_out | (uintptr_t)p->rng_offset_out) & 7) return FA_ERR_BAD_ARG;
    if (((uintptr_t)p->philox_seed_ptr | (uintptr_t)p->philox_offset_ptr) & 7) return FA_ERR_BAD_ARG;
    if (!p->philox_seed_ptr != !p->philox_offset_ptr) return FA_ERR_BAD_ARG;  // both or neither
  }
  if ((uintptr_t)p->seqused_k & 3) return FA_ERR_BAD_ARG;
  if (p->reserved3 != 0) return FA_ERR_BAD_ARG;
  if (p->block_table) {
    // paged K/V: dense mode, pages of whole 32-row blocks, a table wide enough.  Decode-shaped calls (what the
    // split-KV kernel takes) may use dropout; a prefill chunk (the tile kernel) may not.
    if ((uintptr_t)p->block_table & 3) return FA_ERR_BAD_ARG;
    if (p->page_size <= 0 || p->block_table_stride < 0) return FA_ERR_BAD_ARG;
    if (p->page_size % 32) return FA_ERR_UNSUPPORTED;
    if (p->block_table_stride < ((int64_t)p->seqlen_k + p->page_size - 1) / p->page_size) return FA_ERR_BAD_ARG;
    if (p->cu_seqlens_q || p->bias || (p->dropout_p > 0.f && p->dropout_mask) || p->is_causal == FA_MASK_CAUSAL_TOP_LEFT)
      return FA_ERR_UNSUPPORTED;
    if (p->seqlen_q < 1) return FA_ERR_UNSUPPORTED;
    const bool decode_shaped = (int64_t)p->seqlen_q * (p->heads_q / p->heads_k) <= 16;
    if (p->kernel == FA_KERNEL_SPLITKV && !decode_shaped) return FA_ERR_UNSUPPORTED;
    if ((p->kernel == FA_KERNEL_TILE || !decode_shaped) && p->dropout_p > 0.f) return FA_ERR_UNSUPPORTED;
    // the pools' pages are addressed as 64-bit page x stride; rows inside a page as 32-bit row x stride
    if (p->k_stride_b < 0 || p->v_stride_b < 0) return FA_ERR_BAD_ARG;
  }
  if (p->bias) {
    if (((uintptr_t)p->bias & 7) || p->bias_stride_b < 0 || p->bias_stride_h < 0 || p->bias_stride_q < 0 ||
        ((p->bias_stride_b | p->bias_stride_h | p->bias_stride_q) & 3))
      return FA_ERR_BAD_ARG;
    if (p->kernel == FA_KERNEL_SPLITKV) return FA_ERR_UNSUPPORTED;
  }
  if (p->kernel == FA_KERNEL_SPLITKV) {
    // the query rows x the heads of a GQA group are the 16 columns of its MFMA; packed mode: one row per sequence
    if (p->seqlen_q < 1 || (int64_t)p->seqlen_q * (p->heads_q / p->heads_k) > 16) return FA_ERR_UNSUPPORTED;
    if (p->is_causal == FA_MASK_CAUSAL_TOP_LEFT) return FA_ERR_UNSUPPORTED;  // the single query row would see key 0 only
  }
  return FA_OK;
}

// Split-KV kernel, ragged lengths (known on the device only; `rows`, the longest possible one, is what the host sees; a
// sequence's slices are cut from its own length; units = sequences x kv heads).  More slices even out the lengths over the
// CUs and cost a start, partials and a merge launch; a full batch has nothing to even out.  Measured with every sequence
// full, with lengths of 1/4 ... 1 and 1/16 ... 1 of the longest, and with one long sequence among short ones, 8 ... 1024
// units of 512 ... 32768 keys (us, whole op; head_dim 128 where not said):
//   - short caches stay whole: below 768 rows a slice saves less than it costs (160 units of 512 keys: one slice 11, four
//     17), from 144 units, more than half the CUs, below 2560 (160 of 1024 18 and 24, of 2048 30 and 37; lengths 1/4 ... 1 25
//     and 27), from 192 below 1536.  At head_dim 256, with twice the bytes a row, slices pay below 144 units (16 of 512: 12
//     against 19) and from 768 rows on (160 of 512: 26 and 32);
//   - two whole rounds of the CUs: two slices at most (512 units of 8192 keys: full 361 in two, 382 in three; lengths 1/4 ...
//     1: 262 and 265);
//   - otherwise up to three rounds of the 512 resident half-size workgroups while slices keep 512 rows, 640 from 192 units
//     on (1024 at head_dim 64: 448 of 2048 whole 31, in three 33), where it takes two rounds to be worth it, or one and a
//     half beyond 256 units (212 of 1728: whole 29, in three 36; 264 of 2048: 60 and 50); at least one round while slices
//     keep 128.
// What a full batch pays for that, against long slices or none: 128 units of 16384 keys 200 for 194 (lengths 1/4 ... 1: 122
// for 154), 224 of 8192 176 for 168 (125 for 146), 256 of 8192 199 for 192 (131 for 150).
inline bool two_rounds(int dp, int64_t units) { return dp == 128 && units >= 496 && units <= 512; }
inline int ragged_slices(int dp, int64_t units, int64_t rows) {
  const int64_t whole_below = units < 144 ? (dp == 256 ? 0 : 768) : (dp == 256 ? 768 : (units < 192 ? 2560 : 1536));
  if (rows < whole_below) return 1;
  if (two_rounds(dp, units)) return rows >= 2560 ? 2 : 1;
  auto most = [&](int64_t wgs, int64_t least) {  // slices that make `wgs` workgroups and keep `least` rows
    const int64_t fill = (wgs + units - 1) / units, cap = rows / least;
    return fill < cap ? fill : cap;
  };
  int64_t n;
  if (units < 192) {
    const int64_t one = most(512, 128), three = most(1536, 512);
    n = one > three ? one : three;
  } else {
    n = most(1536, dp == 64 ? 1024 : 640);
    if (units * n < (dp == 256 || units <= 256 || n < 3 ? 1024 : 768) || (dp == 64 && n < 3)) n = 1;
  }
  if (n > 8) n &= ~(int64_t)3;
  return (int)(n < 1 ? 1 : (n > FA_MAX_SPLITS ? FA_MAX_SPLITS : n));
}
// Two wavefronts a workgroup instead of four?  At head_dim 128 a workgroup of four has its CU to itself; of two, two share
// one, and one's start and merge are covered by the other's loads.  Four where a workgroup streams for long, is alone on its
// CU or in step with the others, and for few rows in something over one round (us: 512 units of 512 keys, full: four 27, two
// 25; 512 of 1024 43 and 46; 264 of 1024 35 and 32; 448 of 1024 39 and 41; 264 of 16384 in six slices 383 and 394, lengths
// 1/4 ... 1 235 and 250; 512 of 8192 in two slices 361 and 379).  At head_dim 64 two workgroups of four share a CU anyway
// (512 of 8192 in three slices, lengths 1/4 ... 1: four 138, two 146); at head_dim 256 there are no other than of two.
inline bool ragged_half(int dp, int64_t units, int64_t rows, int slices) {
  if (dp != 128) return false;
  if (two_rounds(dp, units)) return rows < 1024;
  if (slices > 1) return rows < (int64_t)2560 * slices;
  return units > 256 && !(units >= 320 && units <= 768 && rows >= 1024 && rows < 1536);
}

inline void plan(const fa_fwd_params* p, int* kernel, int* splits) {
  int kern = p->kernel;
  const int group = p->heads_q / p->heads_k;
  // a page table: decode-shaped calls go to the split-KV kernel, a prefill chunk to the tile kernel's paged variant
  if (p->block_table && kern == FA_KERNEL_AUTO)
    kern = ((int64_t)p->seqlen_q * group <= 16) ? FA_KERNEL_SPLITKV : FA_KERNEL_TILE;
  if (kern == FA_KERNEL_AUTO)
    kern = (p->seqlen_q >= 1 && (int64_t)p->seqlen_q * group <= 16 && p->seqlen_k >= 256 && !p->bias && p->is_causal != FA_MASK_CAUSAL_TOP_LEFT && !(p->dropout_p > 0.f && p->dropout_mask))
               ? FA_KERNEL_SPLITKV
               : FA_KERNEL_TILE;
  int ns = 1;
  if (kern == FA_KERNEL_SPLITKV) {
    ns = p->num_splits;
    if (ns == 0) {
      // A workgroup costs about 5 us to start and to merge, and a second launch merges the slices, so slices are long:
      // split only until every CU has one workgroup (256 CUs), give slices of 2048 rows and more
      // precedence over the last doubling while 128 workgroups remain, and never cut below 512 rows.  Measured on
      // B x 8 kv heads x {2k ... 128k} rows: within 8 % of the best power of two everywhere (the former rule, 2048
      // workgroups of at least 512 rows, was up to 1.7 x slower at batch 4-16).
      constexpr int64_t kCUs = 256;
      const int64_t units = (int64_t)p->batch * p->heads_k;
      ns = 1;
      if (p->seqused_k || p->cu_seqlens_q) {
        ns = ragged_slices(padded_dim(p->head_dim), units, p->seqlen_k);
      } else {
        while (ns * 2 <= FA_MAX_SPLITS && units * ns * 2 <= kCUs) ns *= 2;
        while (ns > 1 && p->seqlen_k / ns < 2048 && units * (ns / 2) >= kCUs / 2) ns /= 2;
        while (ns > 1 && p->seqlen_k / ns < 512) ns /= 2;
      }
    }
    const int nblk = (p->seqlen_k + 31) / 32;
    if (ns > nblk) ns = nblk > 0 ? nblk : 1;
  } else if (p->seqlen_q > 0) {
    // Tile kernel (dense or packed; an additive bias, either causal alignment and dropout — whose mask is a function
    // of the row and the key, not of the slice — are fine): with few query blocks against a long K/V (chunked prefill, speculative decoding, a
    // GQA group too wide for the split-KV kernel) the key range of each block is cut into slices so that the CUs
    // have two workgroups each; a slice keeps at least 32 tiles (2048 keys), or 16 where the chunk is much shorter
    // than the cache, so that a causal mask leaves every slice equally full.  Partials go through the workspace.
    const int64_t wgs = (int64_t)p->batch * p->heads_q * ((p->seqlen_q + 127) / 128);
    const int ntiles = (p->seqlen_k + 63) / 64;
    const int min_tiles = ((int64_t)p->seqlen_q * 4 <= p->seqlen_k) ? 16 : 32;
    ns = p->num_splits;
    if (ns == 0) {
      ns = 1;
      while (ns * 2 <= FA_MAX_SPLITS && wgs * ns * 2 <= 512 && ntiles / (ns * 2) >= min_tiles) ns *= 2;
    }
    if (ns > ntiles) ns = ntiles > 0 ? ntiles : 1;
    // keep the partials (fp32, one slot per query row and slice) within 1 GiB
    const int64_t rows = (int64_t)p->batch * p->heads_q * p->seqlen_q;  // <= 2^60
    while (ns > 1 && rows > (1LL << 30) / ((int64_t)ns * (p->head_dim * 4 + 8))) ns /= 2;
  }
  *kernel = kern;
  *splits = ns;
}

// partial slots: one per (sequence, query head, query row, slice) for both kernels (packed mode: seqlen_q rows per
// sequence, the longest one's)
inline size_t partial_slots(const fa_fwd_params* p, int kern, int ns) {
  (void)kern;
  return (size_t)p->batch * p->heads_q * ns * (size_t)p->seqlen_q;
}

inline size_t workspace_bytes(const fa_fwd_params* p, int kern, int ns) {
  if (ns <= 1) return 0;
  const size_t slots = partial_slots(p, kern, ns);
  return slots * (size_t)p->head_dim * 4 + slots * 8;
}

// ---- backward -----------------------------------------------------------------------------------------------

inline int bwd_validate(const fa_bwd_params* p) {
  if (!p) return FA_ERR_BAD_ARG;
  if (!p->q || !p->k || !p->v || !p->out || !p->dout || !p->lse || !p->dq || !p->dk || !p->dv) return FA_ERR_BAD_ARG;
  if ((p->cu_seqlens_q == nullptr) != (p->cu_seqlens_k == nullptr)) return FA_ERR_BAD_ARG;
  if (p->batch <= 0 || p->heads_q <= 0 || p->heads_k <= 0) return FA_ERR_BAD_ARG;
  if (p->seqlen_q < 0 || p->seqlen_k < 0 || p->head_dim <= 0) return FA_ERR_BAD_ARG;
  if (p->reserved != 0 || p->reserved2 != 0) return FA_ERR_BAD_ARG;
  if (!(p->dropout_p >= 0.f && p->dropout_p < 1.f)) return FA_ERR_BAD_ARG;
  if (p->dropout_p > 0.f && (!p->philox_seed || !p->philox_offset ||
                             (((uintptr_t)p->philox_seed | (uintptr_t)p->philox_offset) & 7)))
    return FA_ERR_BAD_ARG;
  if (p->cu_seqlens_q && p->total_q < 0) return FA_ERR_BAD_ARG;
  if (p->is_causal != FA_MASK_NONE && p->is_causal != FA_MASK_CAUSAL_BOTTOM_RIGHT && p->is_causal != FA_MASK_CAUSAL_TOP_LEFT)
    return FA_ERR_BAD_ARG;
  if (p->dbias && !p->bias) return FA_ERR_BAD_ARG;
  if (p->bias) {
    if (((uintptr_t)p->bias & 7) || p->bias_stride_b < 0 || p->bias_stride_h < 0 || p->bias_stride_q < 0 ||
        ((p->bias_stride_b | p->bias_stride_h | p->bias_stride_q) & 3))
      return FA_ERR_BAD_ARG;
  }
  if (p->dbias) {  // an output: aligned like the bias and not broadcast
    if (((uintptr_t)p->dbias & 7) || ((p->dbias_stride_b | p->dbias_stride_h | p->dbias_stride_q) & 3)) return FA_ERR_BAD_ARG;
    if (p->dbias_stride_q < p->seqlen_k || (p->seqlen_q > 1 && p->dbias_stride_q <= 0) ||
        (p->heads_q > 1 && p->dbias_stride_h <= 0) || (p->batch > 1 && p->dbias_stride_b <= 0))
      return FA_ERR_BAD_ARG;
  }
  if (p->dtype != FA_DTYPE_FP16 && p->dtype != FA_DTYPE_BF16) return FA_ERR_UNSUPPORTED;
  if (p->head_dim > 256 || (p->head_dim & 7)) return FA_ERR_UNSUPPORTED;
  if (p->heads_q % p->heads_k) return FA_ERR_UNSUPPORTED;
  if (p->seqlen_q > kMaxSeqlen || p->seqlen_k > kMaxSeqlen) return FA_ERR_UNSUPPORTED;
  if ((int64_t)p->batch * p->heads_q > 0x7fffffffLL) return FA_ERR_UNSUPPORTED;
  const uintptr_t al = (uintptr_t)p->q | (uintptr_t)p->k | (uintptr_t)p->v | (uintptr_t)p->out | (uintptr_t)p->dout |
                       (uintptr_t)p->dq | (uintptr_t)p->dk | (uintptr_t)p->dv;
  if (al & 15) return FA_ERR_BAD_ARG;
  if ((uintptr_t)p->lse & 3) return FA_ERR_BAD_ARG;
  const int64_t st[] = {p->q_stride_s,  p->q_stride_h,  p->k_stride_s,  p->k_stride_h,  p->v_stride_s,  p->v_stride_h,
                        p->o_stride_s,  p->o_stride_h,  p->do_stride_s, p->do_stride_h, p->dq_stride_s, p->dq_stride_h,
                        p->dk_stride_s, p->dk_stride_h, p->dv_stride_s, p->dv_stride_h};
  for (int64_t s : st)
    if (s < 0 || (s & 7)) return FA_ERR_BAD_ARG;
  if (!p->cu_seqlens_q) {
    const int64_t sb[] = {p->q_stride_b,  p->k_stride_b,  p->v_stride_b,  p->o_stride_b,
                          p->do_stride_b, p->dq_stride_b, p->dk_stride_b, p->dv_stride_b};
    for (int64_t s : sb)
      if (s < 0 || (s & 7)) return FA_ERR_BAD_ARG;
  }
  if (p->lse_stride_h < 0 || p->lse_stride_s < 0) return FA_ERR_BAD_ARG;
  // per-lane byte offsets inside a tile (up to 128 rows) are 32-bit row x 32-bit stride
  if (p->k_stride_s > kMaxRowStrideBytes / 2 || p->v_stride_s > kMaxRowStrideBytes / 2 ||
      p->q_stride_s > kMaxRowStrideBytes / 2 || p->do_stride_s > kMaxRowStrideBytes / 2)
    return FA_ERR_UNSUPPORTED;
  return FA_OK;
}

// two fp32 planes per (row, head): -delta and LSE log2(e)
inline size_t bwd_ws_plane(const fa_bwd_params* p) {
  const size_t rows = p->cu_seqlens_q ? (size_t)p->total_q : (size_t)p->batch * p->seqlen_q;
  return (rows * p->heads_q * 4 + 15) & ~(size_t)15;
}
// Slices of a key block's dK / dV.  A key block's workgroup walks the query tiles of all heads of its group one after
// the other, and one workgroup already keeps its CU's matrix cores as busy as two do, so a launch takes at least as long
// as its longest block alone: a group of 7 heads over 4096 rows is 448 steps of 1.7 us whatever the rest of the chip
// does.  Where that is more than the whole work spread over the 256 CUs, the blocks are cut into slices whose fp32
// partial sums a second kernel adds up.  A step costs 1.7 us of a CU for dK and 1.25 for dV (one workgroup each; at
// head_dim 64 one workgroup does both), a slice's partials, start and share of the merge about as much as 6 steps and
// the extra launch 10.  Whole backward, bf16, causal, unsliced -> sliced, us: 28 query / 4 kv heads, head_dim 128, 4096
// rows 882 -> 575, 700 rows 145 -> 60; 32 / 8, 2048 rows 272 -> 195, 4096 rows 642 -> 607; batch 4, 16 / 4, head_dim 64,
// 2048 rows 225 -> 165; 8 packed sequences of 187 ... 1500 rows, 16 / 4, 250 -> 232.  On the other side of the line:
// 16 / 16, 2048 rows 113 -> 133; 8 / 8, 4096 rows 209 -> 222; batch 2, 16 / 8, head_dim 256, 2000 rows 331 -> 423.
//
// The partial sums take at most four times the memory of the call's own tensors (q, out, dout, dq and k, v, dk, dv), which
// one kv head for many query heads comes near (8 / 1 heads, 4096 rows: 128 MiB beside 34; twice would cost it 6 %): slices
// get longer until they do, or the blocks stay whole.
//
// Pairs of (128-key block, 64-row query tile that sees some of its keys) in the first p key blocks: off = Lk - Lq, or 0 for
// the top-left mask.  Block i sees the tiles from max(0, 128 i - off) / 64 = max(0, 2 i + t) on.  (constexpr: the kernels
// call it too)
constexpr int64_t key_block_tiles_before(int64_t p, int64_t nq, int64_t off, bool causal) {
  if (!causal) return p * nq;
  const int64_t t = (-off) >> 6;
  const int64_t all = t > 0 ? 0 : -t / 2 + 1;         // blocks that see every tile
  const int64_t some = (nq - t + 1) >> 1;             // blocks that see any
  const int64_t a = p < all ? p : all, z0 = all > some ? all : some, z = p < z0 ? p : z0;
  return a * nq + (z - a) * (nq - t) - (z * (z - 1) - a * (a - 1));
}
// A block of n steps is cut into ceil(n / iters) slices; the first slot of block p, counted like that, is at or before
// floor(steps of the blocks before / iters) + p, which needs no sum over the blocks and leaves less than one slot unused each.
struct BwdSlices {
  int32_t count;  // most slices of a key block
  int32_t iters;  // most steps (query head of the group, 64-row query tile) of a slice
  int32_t slots;  // slots of 128 key rows: of each (sequence, kv head), packed: of each kv head, for all sequences
  size_t bytes;   // fp32 partial sums of dK, then of dV
  uint64_t per_row, per_seq;  // packed: slots that a row and a sequence add to the first slot of the next one, times 2^32
};
inline BwdSlices bwd_slices(const fa_bwd_params* p) {
  const BwdSlices whole = {1, 0x7fffffff, 0, 0, 0, 0};
  const int64_t group = p->heads_q / p->heads_k;
  const int64_t nk = ((int64_t)p->seqlen_k + 127) / 128, nq = ((int64_t)p->seqlen_q + 63) / 64;
  const int64_t units = (int64_t)p->batch * p->heads_k * nk, longest = group * nq;
  const bool causal = p->is_causal != FA_MASK_NONE;
  if (units == 0 || longest == 0) return whole;
  // steps of all blocks; packed lengths are known on the device only, and sum(n^2) lies between total^2 / batch (equal
  // lengths) and total x longest: the geometric mean of the two, with a margin for being an estimate
  double total = (double)units * (double)longest * (causal ? 0.5 : 1.0), margin = 1.0;
  if (p->cu_seqlens_q) {
    const double fill = (double)p->total_q / ((double)p->batch * p->seqlen_q);
    if (fill < 1.0) total *= fill * sqrt(fill);
    margin = 1.25;
  }
  const double spread = total / 256.0 * (p->head_dim <= 64 ? 1.2 : 1.75);
  if ((double)longest <= margin * (spread + 10.0)) return whole;
  // slices of 16 steps at least; about three per CU of each kind where dK and dV share a launch, else four (28 query / 4 kv
  // heads, 4096 rows, dropout: 1067 us with four, 1126 with three; head_dim 256, 16 / 2, 4096 rows, causal: 775 and 721)
  const bool alone = p->head_dim <= 64 || p->dropout_p > 0.f || p->bias;
  int64_t want = (int64_t)(total / (alone ? 1024.0 : 832.0));
  if (want < 16) want = 16;
  int64_t n = (longest + want - 1) / want;
  if (n > FA_MAX_SPLITS) n = FA_MAX_SPLITS;
  // steps and key blocks that share an array of slots: dense, those of a (sequence, kv head); packed, those of a kv head.
  // There a sequence of L rows gets room for as many as self-attention can have, at most L / 64 + 1 query tiles times (of a
  // causal mask half) the key blocks of the longest, and L / 128 + 1 blocks; one with more keys than that stays whole
  const int64_t rows_q = p->cu_seqlens_q ? p->total_q : (int64_t)p->batch * p->seqlen_q;
  const double wide = causal ? 0.5 * (double)nk + 1.0 : (double)nk;
  const int64_t off = p->is_causal == FA_MASK_CAUSAL_TOP_LEFT ? 0 : (int64_t)p->seqlen_k - p->seqlen_q;
  const double steps = (double)group * (double)key_block_tiles_before(nk, nq, off, causal);
  const int64_t arrays = p->cu_seqlens_q ? p->heads_k : (int64_t)p->batch * p->heads_k;
  const int64_t slot = (int64_t)128 * padded_dim(p->head_dim) * 4 * 2;
  int64_t rows_k = (int64_t)p->batch * p->seqlen_k;
  if (p->cu_seqlens_q && rows_k > rows_q) rows_k = rows_q;
  const double tensors = 8.0 * p->head_dim * ((double)rows_q * p->heads_q + (double)rows_k * p->heads_k);
  const double most = 4.0 * tensors < (double)(1LL << 30) ? 4.0 * tensors : (double)(1LL << 30);
  for (; n > 1; --n) {
    const int64_t iters = (longest + n - 1) / n;
    const double tile = (double)group * wide / (double)iters;  // packed: slots per query tile
    const double per_row = tile / 64 + 1.0 / 128, per_seq = tile + 1.0;
    const double slots = p->cu_seqlens_q ? ceil((double)p->total_q * per_row + (double)p->batch * per_seq)
                                         : floor(steps / (double)iters) + (double)nk;
    if (slots * (double)arrays * (double)slot > most || slots * (double)iters > (double)0x7fffffff) continue;
    BwdSlices r;
    r.count = (int32_t)n;
    r.iters = (int32_t)iters;
    r.slots = (int32_t)slots;
    r.bytes = (size_t)r.slots * (size_t)arrays * (size_t)slot;
    r.per_row = (uint64_t)ceil(per_row * 4294967296.0);
    r.per_seq = (uint64_t)ceil(per_seq * 4294967296.0);
    return r;
  }
  return whole;
}
inline size_t bwd_ws_bytes(const fa_bwd_params* p) { return 2 * bwd_ws_plane(p) + bwd_slices(p).bytes; }

}  // namespace host
}  // namespace fa

#endif  // FA_HOST_H_
