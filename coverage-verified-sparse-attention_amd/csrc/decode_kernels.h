// Paged decode attention over a per-KV-head page list, emitting the
// un-normalised softmax state (o, m, l) and/or the normalised output.
//
// Semantics follow the reference's sparse decode kernels
// (cvsa/kernels/sparse_decode.py:14-132, :136-234, :423-500): for each
// q-head, over the first n_sel listed pages of its KV head and the tokens
// t < min(bs, ctx - page*bs) of each page (:76-80), s = (q . K) * D^-0.5,
// m = max s, l = sum exp(s - m), o = sum exp(s - m) V (:101-124); the
// normalised output is o / max(l, 1e-6) (:127, :271).  Split-K partial
// states are combined with the log-sum-exp rule of _reduce_tiles_kernel
// (:237-276, :576-606).
//
// MI355X mapping.  The reference launches one program per q-head, so each
// K/V page tile is fetched G times.  Here a workgroup owns one KV head and a
// contiguous range of its page list; each of its four waves takes every
// fourth page, loads the page's 16 K rows and 16 V rows once (256 B per row,
// 16-byte lane loads) and applies them to all G query heads of the group as
// two small matrix-core tiles (S = K Q^T, O += P V; see MfmaEngine).  The
// four waves merge in LDS.  When a head's pages span several workgroups
// (splits), each stores its partial (o, m, l) and bumps the head's
// completion counter; the last one to arrive merges the partials and writes
// the outputs, so one launch does the whole decode.  The last workgroup
// resets the counter to zero for the next launch.
//
// Ordering of the split hand-off.  Partials are written and read through a
// raw buffer resource with the sc1 cache policy: on gfx950 such stores are
// written through the issuing XCD's L2 to the device coherence point and
// such loads miss in the reading XCD's L2, so no L2 writeback or invalidate
// (an agent-scope release / acquire fence) is needed.  A workgroup waits
// for its partial stores to complete (s_waitcnt vmcnt(0) and a barrier)
// before its relaxed agent-scope atomic increment of the head's counter; the
// last arriver issues its partial loads only after that atomic has
// returned.  This rests on the gfx950 cache policy described, not on the
// HIP memory model's release / acquire pairing.  Building with
// -DCVSA_FORMAL_HANDOFF=1 replaces it with that pairing (an agent-scope
// release fence in every thread before the counter, an acq_rel counter
// increment, an agent-scope acquire fence in the last arriver): the same
// bits, but the L2 writeback and invalidate those fences compile to cost
// the cfg3 listed decode 31.5 us against 19.3 us (one rejected head 67 vs
// 37 us, dense 135 vs 96 us; measured with an engine that took 19.3 us where
// this one takes 17.1), so the default build keeps the cache-policy protocol.
//
// Head modes: a listed head walks page_indices[b,h,:n_per_head]; an
// all-pages head walks pages 0..n_valid-1 (dense decode).  In verified mode
// accepted heads are listed and rejected heads walk every valid page: the
// draft pages plus the complement pages in one pass, which equals the LSE
// merge of the draft and complement partial softmaxes.  In approximate
// mode rejected heads walk their expanded selection instead
// (cvsa/backend.py:780-812: an expanded top-k at approx_recovery_pct of the
// pages, decoded and normalised on its own).
//
// Tiles: the kernels walk 16-token tiles.  A page (block) of block_size =
// 16 * 2^ts tokens is 2^ts consecutive tiles of its block, so tile sub of
// logical page lp is logical tile (lp << ts) | sub, stored at physical tile
// (block << ts) | sub, 16 * H_kv * D elements apart.  Head walks, splits and
// stream-K ranges count tiles; the effective-budget counters count pages.
#pragma once

#include "cvsa_common.h"
#include "score_body.h"
#include <hip/hip_fp16.h>

namespace cvsa {

// Split partials of head dimension D are rows of part_stride(D) floats:
// o[D], m, l and two pad words, so every row starts on a 16-byte boundary.
// A q-head's o is D / 4 float4 chunks.
__host__ __device__ constexpr int part_stride(int D) { return D + 4; }
constexpr int kMaxSplits = 256;            // partials per head (and workgroups per launch)
// Waves per workgroup, one per SIMD.  Eight waves (two per SIMD, the same
// tiles in flight per wave) measured slower: the listed decode 17.3 against
// 17.1 us at cfg3 and 44.4 against 43.2 us at B = 32 (ragged 8K contexts),
// dense at B = 4, 64K 186 against 178 us (172 since the chunks run on).
constexpr int kWavesPerWg = 4;
constexpr int kMinPagesPerWave = 2;        // pages per wave of a split, at least

struct DecodeArgs {
  const uint16_t *q;
  int64_t q_sb, q_sh;
  const uint16_t *k_cache;
  const uint16_t *v_cache;
  int64_t num_blocks;
  const int32_t *block_tables;
  int64_t bt_sb;
  const int32_t *ctx_lens;
  const int32_t *page_idx;  // NULL: every head walks all valid pages
  int64_t idx_stride;
  int max_sel;
  const int32_t *n_pages;
  const uint8_t *accept;  // non-NULL: verified mode
  int H_kv, W;
  int D;      // head dimension (the launch's engine is compiled for it)
  int ts;     // tiles per page = 1 << ts
  int tl;     // rows of a tile = 1 << tl: 4, or 3 for 8-token pages (picks the engine)
  // Query heads: the launch serves heads q_off .. q_off + G - 1 (G the
  // kernel's group, at most 16) of each KV head's group of q_group; a larger
  // group runs as one launch per 16 of its heads.
  int q_group, q_off;
  int heads;  // B * H_kv
  int pps, n_splits;  // listed partition: tiles per split, splits per head
  // Identity partition (every valid page of every head, in page order, as
  // a listed walk of the list 0, 1, 2, ...): tiles per split, splits per
  // head.  Verified launches whose heads are all rejected use it, and so
  // does the lazy check's speculative dense decode, so the two write the
  // same bits.
  int pps_all, n_splits_all;
  int sk_grid;        // stream-K partition: workgroups (<= kMaxSplits)
  float scale;
  float *o_unnorm, *m_out, *l_out;
  void *out;
  int out_dtype;
  float *part;               // split partials (see PartBuf)
  uint32_t part_bytes;
  unsigned *counters;        // per head, zero between launches
  unsigned long long *work;  // optional effective-budget counters
  // A lazy check's speculation (or NULL).  [0]: the prediction, 1 = the
  // check keeps its selection (speculative listed decode of the cached
  // selection), 2 = every head is rejected (speculative dense decode, the
  // identity partition), else none; the check's select-or-keep overwrites
  // it with its keep flag (0 / 1), and a verified launch whose heads are
  // all rejected sets it to 2.  [1]: which speculative decode ran and wrote
  // the outputs (0 none, 1 listed, 2 dense).
  int32_t *spec_state;
  // The speculative decode also writes the page scores of the pages it
  // walks into spec_scores [B * H_kv, W] (or NULL), as the page scoring
  // would (q_rep the group mean of q_group heads times inv_g).
  float *spec_scores;
  float inv_g;
  // Approximate recovery (kModeApprox): a rejected head walks the first
  // min(alt_budget, n_valid) pages of its expanded selection alt_idx[bh]
  // instead of every valid page.
  const int32_t *alt_idx;
  int64_t alt_stride;
  int alt_budget;
};

// A reuse step's token append folded into its listed decode
// (cvsa_sparse_decode_append): sequence b's new K/V rows go to token
// slot[b].x % 16 of logical page slot[b].x / 16 (16-token pages), into block
// slot[b].y when that page is allocated by this append, else the block its
// table entry names; the context length becomes slot[b].x + 1.  The
// workgroups that attend that page take the new token's rows from k_new /
// v_new, so no workgroup reads the cache slot being written.
constexpr int kMaxAppendSeqs = 256;
struct AppendArgs {
  const uint16_t *k_new, *v_new;  // [B, H_kv, D] rows, new_sb elements apart
  int64_t new_sb;
  int32_t *block_tables, *ctx_lens, *pages_allocated;  // updated by the append
  int max_pages;  // block-table width W
  // The slots in device memory (written before the launch, e.g. by a copy
  // that a captured graph replays), or NULL: the slots are slot[].  The host
  // checks slot[] before the launch; device slots are checked here: one out
  // of range (context length outside [0, 16 W), a new block outside
  // [-1, num_blocks), or a new block not at a page start) appends nothing,
  // leaves that sequence's outputs undefined and adds 1 to *slot_errors
  // (when given).
  const int2 *slot_dev;
  int32_t *slot_errors;
  int2 slot[kMaxAppendSeqs];  // (context length before the append, new block or -1)
};

// The new token of a walk's sequence: its logical page and row, its block
// when the append allocates it (else -1), and its K/V rows for this KV head.
struct NewToken {
  int page = -1, off = 0, new_blk = -1;
  const uint16_t *k = nullptr, *v = nullptr;
};

__device__ __forceinline__ void store_out(void *out, int dtype, int64_t i, float y) {
  if (dtype == CVSA_DTYPE_BF16) {
    reinterpret_cast<uint16_t *>(out)[i] = (uint16_t)f32_to_bf16_bits(y);
  } else if (dtype == CVSA_DTYPE_FP16) {
    reinterpret_cast<__half *>(out)[i] = __float2half_rn(y);
  } else {
    reinterpret_cast<float *>(out)[i] = y;
  }
}


template <int D>
__device__ __forceinline__ void write_outputs(const DecodeArgs &a, int64_t qrow, int d, float O,
                                              float M, float L) {
  if (a.o_unnorm != nullptr) {
    a.o_unnorm[qrow * D + d] = O;
    if (d == 0) {
      a.m_out[qrow] = M;
      a.l_out[qrow] = L;
    }
  }
  if (a.out != nullptr) store_out(a.out, a.out_dtype, qrow * D + d, O / fmaxf(L, 1e-6f));
}

// Effective-budget counters: pages attended by this head (n) and the valid
// pages of its sequence (nv).
__device__ __forceinline__ void add_work(const DecodeArgs &a, int n, int nv) {
  atomicAdd(&a.work[0], (unsigned long long)n);
  atomicAdd(&a.work[1], (unsigned long long)max(0, nv));
}

// n_valid_pages(ctx, 1 << sh) for pages of 1 << sh tokens (sh = tl + ts),
// the division a shift where ctx > 0.
__device__ __forceinline__ int valid_pages_sh(int ctx, int sh) {
  return ctx > 0 ? ((ctx - 1) >> sh) + 1 : n_valid_pages(ctx, 1 << sh);
}

// Logical tile of entry e of a head's listed walk: tile e & (2^ts - 1) of
// page idx_row[e >> ts].  ts is the engine's tile shift, a compile-time 0
// for 16-token pages; the result is valid iff it lies in [0, W << ts) (with
// ts > 0 a page outside [0, W) gives -1, so no shift can wrap into range).
__device__ __forceinline__ int listed_tile(const DecodeArgs &a, const int32_t *idx_row, int e,
                                           int ts) {
  const int lp = idx_row[e >> ts];
  if (ts == 0) return lp;
  return lp >= 0 && lp < a.W ? (lp << ts) | (e & ((1 << ts) - 1)) : -1;
}

// Physical tile of logical tile lt of sequence b: valid iff lt is valid and
// the result lies in [0, num_blocks << ts).  The block-table load is
// unconditional (index clamped).
__device__ __forceinline__ int tile_block(const DecodeArgs &a, int b, int lt, int ts) {
  const int phys = a.block_tables[b * a.bt_sb + min(max(lt, 0) >> ts, a.W - 1)];
  if (ts == 0) return phys;
  return lt >= 0 && phys >= 0 && phys < a.num_blocks ? (phys << ts) | (lt & ((1 << ts) - 1))
                                                     : -1;
}


// Tiles walked by head bh: those of its listed pages (page_indices[bh,
// :n_per_head]), or of every valid page (dense heads, rejected heads of a
// verified launch).
// MODE is a template parameter and verified mode loads accept[bh] and
// n_per_head[bh] unconditionally and picks with selects: an earlier form
// that branched on null pointers was miscompiled (a live scalar register was
// reused across the branch).
enum { kModeAll = 0, kModeListed = 1, kModeVerified = 2, kModeApprox = 3 };
// Page lists of a head's walk: every valid page, page_indices, alt_idx.
enum { kWalkAll = 0, kWalkListed = 1, kWalkAlt = 2 };

template <int MODE>
__device__ __forceinline__ int head_pages(const DecodeArgs &a, int bh, int &walk, int ts,
                                          int tl) {
  int n_all = 0, n_list = 0;
  if constexpr (MODE != kModeListed)
    n_all = max(0, min(valid_pages_sh(a.ctx_lens[bh / a.H_kv], tl + ts), a.W)) << ts;
  if constexpr (MODE != kModeAll) n_list = min(max(a.n_pages[bh], 0), a.max_sel) << ts;
  if constexpr (MODE == kModeAll) {
    walk = kWalkAll;
    return n_all;
  } else if constexpr (MODE == kModeListed) {
    walk = kWalkListed;
    return n_list;
  } else if constexpr (MODE == kModeVerified) {
    const bool acc = a.accept[bh] != 0;
    walk = acc ? kWalkListed : kWalkAll;
    return acc ? n_list : n_all;
  } else {
    const bool acc = a.accept[bh] != 0;
    const int n_alt = min(a.alt_budget << ts, n_all);
    walk = acc ? kWalkListed : kWalkAlt;
    return acc ? n_list : n_alt;
  }
}

// Pages booked in the effective-budget counters for head bh of an
// approximate-recovery launch in which some head was rejected
// (backend.py:812-850: the draft's n_per_head plus the expanded
// selection's min(exp_budget, n_valid) on every head).
__device__ __forceinline__ int approx_booked_pages(const DecodeArgs &a, int bh, int nv) {
  return min(max(a.n_pages[bh], 0), a.max_sel) + min(a.alt_budget, max(0, nv));
}

// Stream-K partition.  The heads' page walks are concatenated (head-major)
// into one list of T tiles and cut into n_wg equal ranges; workgroup w owns
// tiles [start(w), start(w + 1)), start(w) = floor(w * T / n_wg).  n_wg is the
// launch size, reduced so that a workgroup gets at least min_sk_tiles tiles.
// T < 2^31 and n_wg <= kMaxSplits, so every quantity is computed in
// 32 bits (64-bit division is a long instruction sequence on the GPU).
constexpr int kMaxHeads = 4096;  // B * H_kv of one launch
// Two-level merge of a stream-K head with more than kTwoLevelMin partials:
// groups of kMergeGroup consecutive contributors, each merged by its last
// arriver into the group's first partial row, then the groups by the last
// group merger.  Group counters follow the kMaxHeads head counters: word
// 2 w0 + (group > 0) for a group whose first contributor is workgroup w0 (a
// workgroup starts at most one head's first group and one head's later
// group, since a head with more than kTwoLevelMin partials covers every
// workgroup between its first and last entirely).
constexpr int kMergeGroup = 16;
constexpr int kTwoLevelMin = 48;
constexpr int kGroupCounters = 2 * 256;  // 2 x the largest stream-K grid
constexpr int kMinPagesPerWg = kMinPagesPerWave * kWavesPerWg;
// A stream-K workgroup takes at least this many tiles, so a short launch has
// fewer partials to hand off.  us a step with 8 / 16 / 32 (16-token pages,
// H_kv = 8, G = 4): scoring steps that recover half the heads, B = 1, 1K tokens
// 20.1 / 21.9 / 28.0, 4K 22.9 / 23.1 / 26.5, 8K 29.1 / 26.4 / 28.0, 16K 34.8 /
// 34.8 / 33.9, B = 4, 2K 26.5 / 24.4 / 27.7; dense 1K to 4K 12.0-12.4 /
// 12.0-12.3 / 14.4-14.7, from 8K on the same.  Approximate recovery walks
// lists of a like length per head and takes 8 (budget 5%, expanded 30%: 1K
// 24.3 / 25.7 / 31.6, 4K 24.4 / 26.4 / 32.7, 16K 31.8 / 33.8 / 36.3; 64-token
// pages 4K 26.4 / 30.9 / 34.6).
constexpr int kMinTilesPerSkWg = 2 * kMinPagesPerWg;
constexpr int min_sk_tiles(bool approx) { return approx ? kMinPagesPerWg : kMinTilesPerSkWg; }

struct Partition {
  int T, n, q, r;  // tiles, workgroups, T / n, T % n
  __device__ __forceinline__ Partition(int T_, int grid, int min_tiles) : T(T_) {
    n = max(1, min(grid, (T + min_tiles - 1) / min_tiles));
    q = T / n;
    r = T - q * n;
  }
  // floor(w * T / n) = w * q + floor(w * r / n), with w * r < n^2 < 2^31.
  __device__ __forceinline__ int start(int w) const { return w * q + (w * r) / n; }
  // The workgroup whose range holds page p (the largest w with start(w) <= p):
  // a float estimate of (p + 1) * n / T, off by at most one, then corrected.
  __device__ __forceinline__ int owner(int p) const {
    int w = min(n - 1, (int)((float)(p + 1) * (float)n / (float)T));
    if (start(w) > p) --w;
    else if (w + 1 < n && start(w + 1) <= p) ++w;
    return w;
  }
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// The split partials of one launch, accessed through a raw buffer resource
// with the agent-scope cache policy (sc1) at 16 (or 8) bytes per access:
// stores reach the device coherence point before the split's completion
// counter moves, and loads never return a line that another XCD's L2 still
// holds.  Offsets are in floats; accesses past the range read 0 / are
// dropped by the buffer bounds check.
struct PartBuf {
  static constexpr int kCpolAgent = 16;         // sc1
  static constexpr int kRsrcWord3 = 0x00020000;  // 32-bit data format, raw
  static constexpr uint32_t kNoRow = 0x3ffffffcu;  // past any launch's partials (< 2 GiB)
  __amdgpu_buffer_rsrc_t r;
  __device__ __forceinline__ PartBuf(float *base, uint32_t bytes)
      : r(__builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)bytes, kRsrcWord3)) {}
  __device__ __forceinline__ void store4(uint32_t off, f32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)(off * 4), 0,
                                           kCpolAgent);
  }
  __device__ __forceinline__ void store2(uint32_t off, f32x2 v) const {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)(off * 4), 0,
                                          kCpolAgent);
  }
  __device__ __forceinline__ f32x4 load4(uint32_t off) const {
    return __builtin_bit_cast(
        f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off * 4), 0, kCpolAgent));
  }
  __device__ __forceinline__ f32x2 load2(uint32_t off) const {
    return __builtin_bit_cast(
        f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)(off * 4), 0, kCpolAgent));
  }
};

// Outputs for q-row qrow, elements d0 .. d0+3 (one float4 chunk, d0 % 4 == 0):
// one 16-byte store of o_unnorm and one 8- or 16-byte store of out.  The
// outputs are the last stores of a launch, which cannot end before they
// complete, so they are written as few, wide stores.
template <int D>
__device__ __forceinline__ void write_outputs4(const DecodeArgs &a, int64_t qrow, int d0,
                                               f32x4 O, float M, float L) {
  const int64_t i = qrow * D + d0;
  if (a.o_unnorm != nullptr) {
    *reinterpret_cast<f32x4 *>(a.o_unnorm + i) = O;
    if (d0 == 0) {
      a.m_out[qrow] = M;
      a.l_out[qrow] = L;
    }
  }
  if (a.out == nullptr) return;
  if (a.out_dtype == CVSA_DTYPE_FP32) {
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = O[e] / fmaxf(L, 1e-6f);
    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(a.out) + i) = y;
    return;
  }
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float y = O[e] / fmaxf(L, 1e-6f);
    w[e] = a.out_dtype == CVSA_DTYPE_BF16 ? f32_to_bf16_bits(y)
                                          : (uint32_t)__half_as_ushort(__float2half_rn(y));
  }
  *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(a.out) + i) =
      make_uint2(w[0] | (w[1] << 16), w[2] | (w[3] << 16));
}

// LDS of the merge: (m, l) of every (split, g), rewritten in place as
// (weight, l); the head's totals; per-thread sums of the split lanes.
template <int G, int NT>
struct MergeLds {
  f32x2 ml[kMaxSplits * G];
  float M[G], L[G];
  f32x4 acc[NT];
};

// o chunks of one merging thread requested together: as many as read a
// 32-split head (cfg3's) in one memory round trip over the J threads that
// share a chunk, 4 to 16 of them (8 in the stream-K kernel, whose merge sits
// inside its segment loop, where 16 would spill).
constexpr int merge_batch(int J, int most) {
  return J >= 8 ? 4 : 32 / J < most ? 32 / J : most;
}

// Merge of a head's n_act split partials by the last of its workgroups
// (partial sp at row offset head_off + sp * row_step rows).  TO_PART: the
// merged (o, m, l) of the rows go to the partial row at part_off instead of
// the outputs (the first level of a two-level merge; no counters booked).
// Thread t owns float4 chunk c = t % NC of the head's G x D outputs and the
// splits j, j + J, ... (j = t / NC); their o chunks are loaded KB = merge_batch at a
// time, the first KB together with the (m, l) pairs.  When the
// outputs hold more chunks than the workgroup has threads (G x D > 4 NT) each
// thread takes chunks t, t + NT, ... in turn, every split of each.  The
// (m, l) pairs go to LDS first; one wave per q-head turns them into the
// weights exp(m_sp - M) and the totals (M, L).
template <int G, int D, int NT, int KMAX, bool TO_PART = false>
__device__ __forceinline__ void merge_partials(const DecodeArgs &a, const PartBuf &pb,
                                               uint32_t head_off, int n_act, int bh, int n,
                                               int nv, MergeLds<G, NT> &s, int row_step = 1,
                                               uint32_t part_off = 0) {
  constexpr int kChunksPerRow = D / 4;
  constexpr int kPartStride = part_stride(D);
  const uint32_t row_elems = (uint32_t)row_step * (uint32_t)(G * kPartStride);
  constexpr int NC = G * kChunksPerRow;
  constexpr int J = NT / NC > 0 ? NT / NC : 1;
  constexpr int NPASS = (NC + NT - 1) / NT;
  constexpr int NW = NT / kWave;
  constexpr int KB = merge_batch(J, KMAX);
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int j = NPASS == 1 ? t / NC : 0;
  const bool active = t < NC * J;

  for (int e = t; e < n_act * G; e += NT)
    s.ml[e] = pb.load2(head_off + (uint32_t)(e / G) * row_elems + (e % G) * kPartStride + D);
  const int per_lane = active ? (n_act - j + J - 1) / J : 0;  // splits of this thread
  auto load_batch = [&](int g, int d0, int b0, f32x4 (&v)[KB]) {
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      // Past the thread's splits: out of the buffer's range, not read.
      const uint32_t off = head_off + (uint32_t)(j + (b0 + k) * J) * row_elems +
                           g * kPartStride + d0;
      v[k] = pb.load4(b0 + k < per_lane ? off : PartBuf::kNoRow);
    }
  };
  f32x4 cur[KB];
  {
    const int c = NPASS == 1 ? t % NC : t;  // NPASS > 1: t < NT < NC
    load_batch(c / kChunksPerRow, 4 * (c % kChunksPerRow), 0, cur);
  }
  __syncthreads();
  for (int gg = wave; gg < G; gg += NW) {  // wave-uniform
    float mx = -INFINITY;
    for (int sp = lane; sp < n_act; sp += kWave) mx = fmaxf(mx, s.ml[sp * G + gg].x);
    mx = wave_max_from_groups<1>(mx);
    float ls = 0.f;
    for (int sp = lane; sp < n_act; sp += kWave) {
      const f32x2 v = s.ml[sp * G + gg];
      const float w = (mx == -INFINITY || v.x == -INFINITY) ? 0.f : fast_exp(v.x - mx);
      ls += w * v.y;
      s.ml[sp * G + gg].x = w;
    }
    ls = wave_sum_from_groups<1>(ls);
    if (lane == 0) {
      s.M[gg] = mx;
      s.L[gg] = ls;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int pass = 0; pass < NPASS; ++pass) {
    const int c = NPASS == 1 ? t % NC : min(t + pass * NT, NC - 1);
    const bool live = NPASS == 1 ? active : t + pass * NT < NC;
    const int g = c / kChunksPerRow;
    const int d0 = 4 * (c % kChunksPerRow);
    if (pass > 0) load_batch(g, d0, 0, cur);
    f32x4 O = {0.f, 0.f, 0.f, 0.f};
    // A thread's first KB splits were requested with the (m, l) pairs, so a
    // head of up to KB * J splits costs one memory round trip; more splits
    // are read KB at a time.
    for (int b0 = 0;;) {
#pragma unroll
      for (int k = 0; k < KB; ++k) {
        const int sp = min(j + (b0 + k) * J, n_act - 1);
        const float w = b0 + k < per_lane ? s.ml[sp * G + g].x : 0.f;
        O += w * cur[k];
      }
      b0 += KB;
      if (b0 >= per_lane) break;
      load_batch(g, d0, b0, cur);
    }
    if constexpr (J > 1) {
      s.acc[t] = O;
      __syncthreads();
      if (active && j == 0) {
#pragma unroll
        for (int jj = 1; jj < J; ++jj) O += s.acc[t + jj * NC];
      }
    }
    if (live && j == 0) {
      if constexpr (TO_PART) {
        pb.store4(part_off + g * kPartStride + d0, O);
        if (d0 == 0) pb.store2(part_off + g * kPartStride + D, f32x2{s.M[g], s.L[g]});
      } else {
        write_outputs4<D>(a, (int64_t)bh * a.q_group + a.q_off + g, d0, O, s.M[g], s.L[g]);
      }
    }
  }
  if (!TO_PART && t == 0 && a.work != nullptr) add_work(a, n, nv);
}

// ---------------------------------------------------------------- engines
// A page engine owns one wave's softmax state for the G query heads of a KV
// head and applies tiles to it.  The K rows (kr) and V rows (vr) of PD
// tiles (one from D = 128 on) are in registers at a time: each tile is staged
// to LDS as soon as it arrives and the loads of the tile PD further on are
// issued into the same registers at once, so a wave always has about PD tiles
// in flight; finish() leaves the wave's (o, m, l) in LDS.

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef short short8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

// RNE bf16 pair (v_cvt_pk_bf16_f32): the bits of f32_to_bf16_bits.
__device__ __forceinline__ uint32_t cvt_bf16x2(float lo, float hi) {
  const f32x2 x = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t));
}

// Logical tiles lie below kUnreadable.  kUnreadable + lt stands for tile lt of
// a block outside the pool, kNoTile for no tile at all: neither has a valid
// token (ctx - (kUnreadable << 4) < 0) and the loads of both are dropped.
constexpr int kUnreadable = 1 << 26;
constexpr int kNoTile = kUnreadable + (kUnreadable >> 1);
static_assert(((int64_t)kMaxPagesWide << 3) <= kNoTile - kUnreadable, "pages of 8 tiles at most");

// MFMA engine: the G query heads (padded to 16) of a KV head against a tile
// of 16 tokens are two small dense products for the matrix cores.
//   S = K Q^T: v_mfma_f32_16x16x32_bf16, four d-chunks of 32.  A operand =
//     K rows (lane l: token l%16, d 32kk + 8(l/16) .. +8), B operand = Q^T
//     (loaded once), result lane l: head l%16, tokens 4(l/16) .. +4.
//   O += P V: v_mfma_f32_16x16x16_bf16, one 16-column block of d at a time.
//     The S result layout is the A operand layout of P (head l%16, tokens
//     4(l/16) .. +4); P is split into a bf16 high part and a bf16 remainder
//     to keep ~16 mantissa bits, and the two products are added in that
//     order.  (Both as the eight A operands of one v_mfma_f32_16x16x32_bf16,
//     V taken twice, round the sum differently and save no time: 17.1 us
//     listed at 128K, 43.2 at B = 32, 172.1 dense at B = 4, 64K either way,
//     26.1 against 25.6 a scoring step at B = 1, 8K.)
//     The B operand wants 4 tokens of one d column per lane:
//     ds_read_b64_tr_b16 transposes it out of the row-major V tile.
//     Result lane l: heads 4(l/16) .. +4, d column 16 blk + l%16.
// Softmax state: m and the running l of head l%16 live in the four lanes of
// that head; a rescale of O rows goes through LDS (16 factors per wave).
//
// What bounds the walk is HBM reads of 256-byte rows 2 KiB apart.  K and V
// rows are both read whole (LPR lanes of 16 bytes per row, nontemporal) and
// K reaches the A operand layout through LDS: reading K in that layout
// directly (64 bytes of each of 16 rows per instruction, every line requested
// twice) streams 5% slower, and so do two tiles in flight per wave instead of
// one (a gather of the cfg3 selection, 64 MiB, without compute: 13.8 us with
// two tiles in flight, 12.8 with one, 12.15 with whole K rows as well; of
// B = 32, 128 pages per head, 256 MiB: 47.6, 46.5 and 43.6 us).  Tiles past
// the end of a walk are not read: their loads go out of the tile's buffer
// range and are dropped there (prefetches that read a wave's last tile again
// instead cost the cfg3 listed decode a quarter more requests).  With the
// engine of two tiles in flight the kernels took: listed 19.1 -> 17.1 us at
// cfg3, 47.2 -> 43.2 us at B = 32 (ragged 8K), 10.3 -> 8.9 us at B = 1, 8K;
// dense at B = 4, 64K, G = 8 185 -> 172 us.  Launches of fewer workgroups than
// CUs gain as well (136 / 192 / 248 heads, 8K, a workgroup each: 34.6 -> 31.1,
// 37.5 -> 35.3, 47.0 -> 43.5 us).
//
// PAGES: kPages16 (one 16-row tile per page), kPagesWide (2^ts of them) or
// kPages8.  An 8-token page is a tile of 8 rows: rows 8 .. 15 of the two LDS
// tiles are no token's (K: their scores are masked, V: zeros), nothing is read
// from memory for them, and twice as many tiles are in flight.  With 16-row
// loads folded onto the 8 rows and one tile in flight at D = 128 -> as here,
// H_kv = 8, G = 4: listed B = 1, 128K 25.0 -> 19.9 us, B = 32 (ragged 8K) 71.0 -> 49.5; dense
// B = 4, 64K 261.2 -> 186.2.
// KEYS_AGAIN: other workgroups of the launch read the same keys (a fused check
// whose scoring part scores the whole cache): K loads leave the lines in the
// caches.
enum { kPages16, kPagesWide, kPages8 };
template <int G, int D, int PAGES, bool KEYS_AGAIN = false>
struct MfmaEngine {
  static_assert(G <= 16, "GQA group larger than the MFMA tile");
  static_assert(D == 32 || D == 64 || D == 128 || D == 256, "head dimension");
  static constexpr int kD = D;
  static constexpr int kPages = PAGES;
  static constexpr bool kKeysOnce = !KEYS_AGAIN;
  // Tiles per page = 1 << tshift(a), rows per tile kRows = 1 << kRowsLog.
  static __device__ __forceinline__ int tshift(const DecodeArgs &a) {
    return PAGES == kPagesWide ? a.ts : 0;
  }
  static constexpr int kRowsLog = PAGES == kPages8 ? 3 : 4;
  static constexpr int kRows = 1 << kRowsLog;
  static constexpr int NK = D / 32;         // S = K Q^T MFMAs (32 dimensions each)
  static constexpr int NB = D / 16;         // O column blocks (16 dimensions each)
  static constexpr int LPR = D / 8;         // lanes per K or V row (16 bytes each)
  static constexpr int RPL = kWave / LPR;   // rows per wave load
  static constexpr int NL = kRows > RPL ? kRows / RPL : 1;  // K (or V) loads per tile
  static constexpr int kRow = D + 8;        // LDS row of a K or V tile, in bf16
  // Tiles in flight: 8 KiB of K and V or more.  Against the older engine (two
  // tiles in flight at every D below 256, K in the operand layout) at D = 64:
  // listed B = 1, 128K 15.3 -> 13.2 us, dense B = 4, 64K 99.2 -> 91.2, check
  // B = 4, 64K 157.5 -> 147.9.
  static constexpr int PD = kRows * D < 2048 ? 2048 / (kRows * D) : 1;
  static_assert(PD * kRows * D * 4 >= 8192, "8 KiB of K and V in flight per wave");
  // Waves per SIMD the listed decode's registers are held to: launches of more
  // than one workgroup per CU overlap one's hand-off with another's walk.
  // (8-token pages at D = 128 spill 27 registers at four.)
  static constexpr int kWalkWaves = D > 128 ? 2 : D == 128 && PAGES == kPages8 ? 3 : 4;
  struct Tiles {
    uint16_t k[kPageTokens * kRow], v[kPageTokens * kRow];
  };
  // One wave's LDS: the tiles of the walk, then the wave's o.
  struct Lds {
    union {
      Tiles t;
      float o[G * D];
    };
    float alpha[16];
  };
  static_assert(sizeof(float) * G * D <= sizeof(Tiles), "a wave's o fits its tiles");

  float4_t o[NB];
  bf16x8_t qb[NK];
  uint4 kr[PD][NL], vr[PD][NL];  // the tiles in flight
  float m_g, l_g;
  int lane;
  uint32_t voff, row_bytes, tile_bytes;
  float scale;

  __device__ __forceinline__ void init(const DecodeArgs &a, int b, int h, int lane_) {
    lane = lane_;
    scale = a.scale;
    row_bytes = (uint32_t)(a.H_kv * D * 2);
    tile_bytes = row_bytes << kRowsLog;
    const int c16 = lane & 15, grp = lane >> 4;
    voff = (lane / LPR) * row_bytes + (uint32_t)(h * D + 8 * (lane % LPR)) * 2;
    if (RPL > kRows && lane / LPR >= kRows) voff = kRegionSkip;  // no row of the tile
    // Rows past the group repeat head G-1: MFMA output rows are independent
    // and those rows are never written out.  No select on the loaded value,
    // so nothing waits for q before the first tile is consumed.
    const uint16_t *qrow =
        a.q + b * a.q_sb + (int64_t)(h * a.q_group + a.q_off + min(c16, G - 1)) * a.q_sh;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      qb[kk] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4 *>(qrow + 32 * kk + 8 * grp));
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) o[blk] = float4_t{0.f, 0.f, 0.f, 0.f};
    m_g = -INFINITY;
    l_g = 0.f;
  }

  // The rows of the tile at `base` (wave-uniform) into r.  No tile (live
  // false): nothing is read.  Load i reads rows RPL i + lane / LPR.  The
  // lanes of row `newrow` (-1: none) read nothing.
  template <bool APP, bool ONCE>
  __device__ __forceinline__ void fetch(const uint16_t *base, bool live, int newrow,
                                        uint4 (&r)[NL]) const {
    const uint32_t off = voff + (live ? 0u : kRegionSkip);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      uint32_t oi = off;
      if (APP && RPL * i + lane / LPR == newrow) oi = kRegionSkip;
      r[i] = region_load16<ONCE>(base, tile_bytes, oi, RPL * i * row_bytes);
    }
  }

  // Zeros for the V rows that no load of an 8-row tile covers, before a walk:
  // their weights are zero, and the rows stay as they are until finish().
  __device__ __forceinline__ void clear_v_tail(Lds &lds) const {
    uint16_t *dst = &lds.t.v[(lane / LPR) * kRow + 8 * (lane % LPR)];
#pragma unroll
    for (int i = NL; i < kPageTokens / RPL; ++i)
      *reinterpret_cast<uint4 *>(dst + RPL * i * kRow) = make_uint4(0u, 0u, 0u, 0u);
  }

  // A tile's K rows to the K tile, then back in the A operand layout (kop).  The row of a
  // token appended by this launch (newrow, -1: none) comes from k_new.
  template <bool APP>
  __device__ __forceinline__ void stage_k(Lds &lds, const uint4 (&r)[NL], int newrow,
                                          const uint16_t *k_new) const {
    uint16_t *dst = &lds.t.k[(lane / LPR) * kRow + 8 * (lane % LPR)];
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<uint4 *>(dst + RPL * i * kRow) = r[i];
    if (APP && newrow >= 0 && lane < LPR)
      *reinterpret_cast<uint4 *>(&lds.t.k[newrow * kRow + 8 * lane]) =
          *reinterpret_cast<const uint4 *>(k_new + 8 * lane);
  }
  __device__ __forceinline__ void k_operand(const Lds &lds, uint4 (&kop)[NK]) const {
    const int c16 = lane & 15, grp = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      kop[kk] = *reinterpret_cast<const uint4 *>(&lds.t.k[c16 * kRow + 32 * kk + 8 * grp]);
  }
  // A tile's V rows to the V tile (rows past the context are stored as zeros: the
  // reference never reads them).
  template <bool APP>
  __device__ __forceinline__ void stage_v(Lds &lds, uint4 (&r)[NL], int ntok, int newrow,
                                          const uint16_t *v_new) const {
    uint16_t *dst = &lds.t.v[(lane / LPR) * kRow + 8 * (lane % LPR)];
    if (ntok < kRows) {  // uniform: a sequence's last tile, or none
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (RPL * i + lane / LPR >= ntok) r[i] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<uint4 *>(dst + RPL * i * kRow) = r[i];
    if (APP && newrow >= 0 && lane < LPR)
      *reinterpret_cast<uint4 *>(&lds.t.v[newrow * kRow + 8 * lane]) =
          *reinterpret_cast<const uint4 *>(v_new + 8 * lane);
  }

  // Page score of the walk's KV head from the tile's keys, bit for bit the
  // page scoring's (score_group_wave): lane (c16, grp) holds dimensions
  // 32 kk + 8 grp .. +8 of token c16, the scorer's segment s = 4 kk + grp,
  // so the scorer's pairwise sum over s (bit 0, 1, 2, 3 of s in turn) is
  // the partner at lane ^ 16, at lane ^ 32, then the kk pairs; the maximum
  // over the ntok valid tokens follows.  qrep: the 16 segments of q_rep.
  __device__ __forceinline__ float page_score(const uint4 (&kop)[NK], int ntok,
                                              const uint4 *qrep) const {
    static_assert(NK == 4, "segment mapping of the 128-dimension rows");
    const int grp = lane >> 4;
    float x[NK];
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) x[kk] = dot8_bf16(kop[kk], qrep[4 * kk + grp], 0.f);
    float a, b;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      xchg16(x[kk], a, b);
      x[kk] = a + b;
    }
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      xchg32(x[kk], a, b);
      x[kk] = a + b;
    }
    const float sc = ((x[0] + x[1]) + (x[2] + x[3])) * scale;
    float m = (lane & 15) < ntok ? sc : -INFINITY;
    m = fmaxf(m, dpp_f<kDppQuadXor1>(m));
    m = fmaxf(m, dpp_f<kDppQuadXor2>(m));
    m = fmaxf(m, dpp_f<kDppRowHalfMirror>(m));
    m = fmaxf(m, dpp_f<kDppRowMirror>(m));
    return m + 0.f;
  }

  // Scores of the tile and the softmax state: returns P (head c16, tokens
  // t0 .. t0+3) as bf16 high parts and bf16 remainders.
  __device__ __forceinline__ short8_t softmax(const uint4 (&kop)[NK], int ntok, Lds &lds) {
    const int t0 = 4 * (lane >> 4);
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kop[kk]),
                                                    qb[kk], acc, 0, 0, 0);
    float sv[4];
    float pm = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sv[j] = t0 + j < ntok ? acc[j] * scale : -INFINITY;
      pm = fmaxf(pm, sv[j]);
    }
    float x, y;
    xchg16(pm, x, y);
    pm = fmaxf(x, y);
    xchg32(pm, x, y);
    pm = fmaxf(x, y);  // tile max of head c16, in all four of its lanes
    const float m_new = fmaxf(m_g, pm);
    if (__ballot(m_new > m_g) != 0) {  // some head of the wave rescales
      const float alpha = m_new > m_g ? (m_g == -INFINITY ? 0.f : fast_exp(m_g - m_new)) : 1.f;
      l_g *= alpha;
      m_g = m_new;
      if (lane < 16) lds.alpha[lane] = alpha;
      const float4 ar = *reinterpret_cast<const float4 *>(&lds.alpha[t0]);  // rows 4grp .. +4
#pragma unroll
      for (int blk = 0; blk < NB; ++blk) {
        o[blk][0] *= ar.x;
        o[blk][1] *= ar.y;
        o[blk][2] *= ar.z;
        o[blk][3] *= ar.w;
      }
    }
    float p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      p[j] = sv[j] == -INFINITY ? 0.f : fast_exp(sv[j] - m_g);
      l_g += p[j];
    }
    uint4 w;
    w.x = cvt_bf16x2(p[0], p[1]);
    w.y = cvt_bf16x2(p[2], p[3]);
    w.z = cvt_bf16x2(p[0] - bf16_lo(w.x), p[1] - bf16_hi(w.x));
    w.w = cvt_bf16x2(p[2] - bf16_lo(w.y), p[3] - bf16_hi(w.y));
    return __builtin_bit_cast(short8_t, w);
  }

  __device__ __forceinline__ void accumulate(short8_t p, Lds &lds) {
    const int c16 = lane & 15, t0 = 4 * (lane >> 4);
    const short4_t high = __builtin_shufflevector(p, p, 0, 1, 2, 3);
    const short4_t rest = __builtin_shufflevector(p, p, 4, 5, 6, 7);
    typedef __attribute__((address_space(3))) short4_t lds_short4;
    // Lane (c16, grp) names row t0 + c16/4, columns 4 (c16 % 4) .. +4 of a
    // block's 4 x 16 tokens x columns; the transposing read returns it the
    // four tokens t0 .. t0+3 of column c16.
    const uint16_t *src = &lds.t.v[(t0 + (c16 >> 2)) * kRow + 4 * (c16 & 3)];
    // The second product of a block depends on the first: one pass per part
    // over the blocks leaves no wait between them (scoring step at B = 1, 8K
    // 26.3 -> 25.6 us, dense B = 1, 8K 14.30 -> 14.09, 32K 28.2 -> 27.9).
    short4_t vb[NB];
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
      vb[blk] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4 *)(src + 16 * blk));
      o[blk] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(high, vb[blk], o[blk], 0, 0, 0);
    }
#pragma unroll
    for (int blk = 0; blk < NB; ++blk)
      o[blk] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(rest, vb[blk], o[blk], 0, 0, 0);
  }

  __device__ __forceinline__ void finish(Lds &lds, float *s_m, float *s_l) {
    const int c16 = lane & 15, grp = lane >> 4;
    float x, y;
    xchg16(l_g, x, y);
    l_g = x + y;
    xchg32(l_g, x, y);
    l_g = x + y;  // head c16's l over all 16 token rows
    if (lane < G) {
      s_m[lane] = m_g;
      s_l[lane] = l_g;
    }
#pragma unroll
    for (int blk = 0; blk < NB; ++blk)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int g = 4 * grp + j;
        if (g < G) lds.o[g * D + 16 * blk + c16] = o[blk][j];
      }
  }
};

// Tiles of a chunk of up to 64 of a wave's walk: lane j holds tile j's
// physical tile and logical tile (from kUnreadable on: nothing is read).
struct TileChunk {
  int phys = 0, lt = kNoTile;
};

// The rows of physical tile phys into r; logical tile lt from kUnreadable on:
// nothing is read.
template <class Engine, bool APP, bool ONCE>
__device__ __forceinline__ void fetch_tile(const Engine &eng, int phys, int lt, int newrow,
                                           const uint16_t *cache, uint4 (&r)[Engine::NL]) {
  const int64_t base = (int64_t)phys * (eng.tile_bytes / 2);
  eng.template fetch<APP, ONCE>(cache + base, lt < kUnreadable, newrow, r);
}

// Requests the first PD tiles of a walk (those of the first chunk, `cur`).
template <class Engine, bool APP = false>
__device__ __forceinline__ void start_walk(const DecodeArgs &a, Engine &eng, const TileChunk &cur,
                                           int new_tile = -1, int new_off = -1) {
#pragma unroll
  for (int u = 0; u < Engine::PD; ++u) {
    const int phys = __builtin_amdgcn_readlane(cur.phys, u);
    const int lt = __builtin_amdgcn_readlane(cur.lt, u);
    const int newrow = APP && lt == new_tile ? new_off : -1;
    // K before V, here and in the walk: the wait for a tile's K then leaves
    // its V in flight.
    __builtin_amdgcn_sched_barrier(0);
    fetch_tile<Engine, APP, Engine::kKeysOnce>(eng, phys, lt, newrow, a.k_cache, eng.kr[u]);
    __builtin_amdgcn_sched_barrier(0);
    fetch_tile<Engine, APP, true>(eng, phys, lt, newrow, a.v_cache, eng.vr[u]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One wave's walk over npw tiles.  `cur` is the first chunk's tiles, whose
// first PD tiles' loads are in flight (start_walk); chunk c's tiles come from
// lookup(c) while chunk c - 1 is walked, so the loads run on across chunks.
// score(lt, ntok, kop) sees each tile's keys first (SCORE).  APP: row new_off
// of logical tile new_tile is the appended token's (k_new / v_new).
template <class Engine, bool APP, bool SCORE, class Lookup, class Score>
__device__ __forceinline__ void walk_tiles(const DecodeArgs &a, Engine &eng, int npw, int ctx,
                                           TileChunk cur, Lookup lookup, Score score,
                                           typename Engine::Lds &lds, int new_tile = -1,
                                           int new_off = -1, const uint16_t *k_new = nullptr,
                                           const uint16_t *v_new = nullptr) {
  constexpr int tl = Engine::kRowsLog;
  constexpr int PD = Engine::PD;
  static_assert(kWave % PD == 0, "a chunk's tiles fill the slots evenly");
  eng.clear_v_tail(lds);
  TileChunk nxt;
  int lt[PD];
#pragma unroll
  for (int u = 0; u < PD; ++u) lt[u] = __builtin_amdgcn_readlane(cur.lt, u);
  for (int e = 0; e < npw; e += PD) {
    const int j = e & (kWave - 1);
    if (j == 0 && e + kWave < npw) nxt = lookup(e + kWave);
    if (j == kWave - PD) {  // the next tiles are the next chunk's first
      cur = nxt;
      nxt = TileChunk();
    }
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      if (PD > 1 && e + u >= npw) break;  // uniform
      // Lanes past the walk's end hold no tile.
      const int phys_n = __builtin_amdgcn_readlane(cur.phys, (j + u + PD) & (kWave - 1));
      const int lt_n = __builtin_amdgcn_readlane(cur.lt, (j + u + PD) & (kWave - 1));
      const int newrow = APP && lt[u] == new_tile ? new_off : -1;
      const int newrow_n = APP && lt_n == new_tile ? new_off : -1;
      const int ntok = min(1 << tl, max(0, ctx - (lt[u] << tl)));
      eng.template stage_k<APP>(lds, eng.kr[u], newrow, k_new);
      fetch_tile<Engine, APP, Engine::kKeysOnce>(eng, phys_n, lt_n, newrow_n, a.k_cache,
                                                 eng.kr[u]);
      uint4 kop[Engine::NK];
      eng.k_operand(lds, kop);
      if constexpr (SCORE) score(lt[u], ntok, kop);
      const short8_t p = eng.softmax(kop, ntok, lds);
      eng.template stage_v<APP>(lds, eng.vr[u], ntok, newrow, v_new);
      fetch_tile<Engine, APP, true>(eng, phys_n, lt_n, newrow_n, a.v_cache, eng.vr[u]);
      __builtin_amdgcn_sched_barrier(0);
      eng.accumulate(p, lds);
      lt[u] = lt_n;
    }
  }
}

// The split hand-off's three steps.  publish_partials: every thread's
// partial-row stores complete before the workgroup's counter moves;
// handoff_count: thread 0 bumps the counter and returns its old value;
// acquire_partials: the last arriver's partial loads come after it.
#ifndef CVSA_FORMAL_HANDOFF
#define CVSA_FORMAL_HANDOFF 0
#endif
__device__ __forceinline__ void publish_partials() {
#if CVSA_FORMAL_HANDOFF
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
#else
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
  __syncthreads();
}
__device__ __forceinline__ unsigned handoff_count(unsigned *ctr) {
#if CVSA_FORMAL_HANDOFF
  return __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
#else
  return __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
}
__device__ __forceinline__ void acquire_partials() {
#if CVSA_FORMAL_HANDOFF
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#endif
}

// LDS of a workgroup's page walk and epilogue: the waves' engines (their
// tiles, then their o), reused by the merge once the workgroup's partial is
// stored; the waves' (m, l); the last-arriver flag.
template <int G, class Engine, int NW>
struct WalkLds {
  union {
    typename Engine::Lds eng[NW];
    MergeLds<G, NW * kWave> merge;
  } __attribute__((aligned(16)));
  float m[NW][G];
  float l[NW][G];
  int last;
};

// End of one workgroup's walk over pages of head h (the waves' states are in
// lds, behind a barrier).  If the workgroup is the head's only
// contributor (n_act == 1) it writes the outputs.  Otherwise it stores its
// partial (o, m, l) in partial row my_row, bumps the head's counter, and the
// last of the n_act contributors merges rows first_row .. first_row+n_act-1.
// TWO (stream-K): a head with more than kTwoLevelMin contributors (rows
// consecutive, contributor i = my_row - first_row) merges in two levels:
// the last arriver of each group of kMergeGroup contributors merges the
// group into the group's first row (after loading every row of the group)
// and bumps the head's counter; the last of the groups merges the group
// rows and writes the outputs.  One workgroup merging ~140 partials takes
// ~9 dependent batches of loads; two levels take one batch each and one more
// store-wait-counter.
template <int G, class Engine, int NW, bool TWO = false>
__device__ __forceinline__ void segment_epilogue(const DecodeArgs &a, const PartBuf &pb, int h,
                                                 int n, int nv, int n_act, uint32_t my_row,
                                                 uint32_t first_row,
                                                 WalkLds<G, Engine, NW> &lds) {
  constexpr int D = Engine::kD;
  constexpr int NT = NW * kWave;
  // Chunks past one per thread (G D > 4 NT) are merged in several passes.
  constexpr int KMAX = TWO || G * D > 4 * NT ? 8 : 16;
  auto &s_m = lds.m;
  auto &s_l = lds.l;
  auto &s_last = lds.last;
  auto &s_merge = lds.merge;
  constexpr int kChunksPerRow = D / 4;
  constexpr int kPartStride = part_stride(D);
  // Workgroup state of float4 chunk c (q-head g = c / (D/4), elements d0 .. d0+3):
  // the waves' (o, m, l) rescaled to the workgroup maximum.
  auto wg_state4 = [&](int c, f32x4 &O, float &M, float &L) {
    const int g = c / kChunksPerRow, d0 = 4 * (c % kChunksPerRow);
    M = s_m[0][g];
#pragma unroll
    for (int wv = 1; wv < NW; ++wv) M = fmaxf(M, s_m[wv][g]);
    O = f32x4{0.f, 0.f, 0.f, 0.f};
    L = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) {
        const float mw = s_m[wv][g];
        if (mw != -INFINITY) {
          const float f = fast_exp(mw - M);
          O += f * *reinterpret_cast<const f32x4 *>(&lds.eng[wv].o[g * D + d0]);
          L += s_l[wv][g] * f;
        }
      }
    }
  };
  if (n_act <= 1) {
    for (int c = threadIdx.x; c < G * kChunksPerRow; c += NT) {
      f32x4 O;
      float M, L;
      wg_state4(c, O, M, L);
      write_outputs4<D>(a, (int64_t)h * a.q_group + a.q_off + c / kChunksPerRow,
                        4 * (c % kChunksPerRow), O, M, L);
    }
    if (threadIdx.x == 0 && a.work != nullptr) add_work(a, n, nv);
    return;
  }
  const uint32_t my_off = my_row * (uint32_t)(G * kPartStride);
  for (int c = threadIdx.x; c < G * kChunksPerRow; c += NT) {
    f32x4 O;
    float M, L;
    wg_state4(c, O, M, L);
    const int g = c / kChunksPerRow, d0 = 4 * (c % kChunksPerRow);
    pb.store4(my_off + g * kPartStride + d0, O);
    if (d0 == 0) pb.store2(my_off + g * kPartStride + D, f32x2{M, L});
  }
  publish_partials();
  constexpr uint32_t kRowElems = (uint32_t)(G * kPartStride);
  if (TWO && n_act > kTwoLevelMin) {  // uniform
    const int i = (int)(my_row - first_row);
    const int gi = i / kMergeGroup;
    const int g0 = gi * kMergeGroup;
    const int gsize = min(kMergeGroup, n_act - g0);
    const int ng = (n_act + kMergeGroup - 1) / kMergeGroup;
    const uint32_t w0 = first_row - (uint32_t)h + (uint32_t)g0;  // the group's first workgroup
    unsigned *gc = a.counters + kMaxHeads + 2 * w0 + (gi != 0 ? 1 : 0);
    if (threadIdx.x == 0) s_last = handoff_count(gc) == (unsigned)(gsize - 1);
    __syncthreads();
    if (!s_last) return;  // uniform
    acquire_partials();
    if (threadIdx.x == 0)
      __hip_atomic_store(gc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t grow = (first_row + (uint32_t)g0) * kRowElems;
    merge_partials<G, D, NT, KMAX, true>(a, pb, grow, gsize, h, 0, 0, s_merge, 1, grow);
    publish_partials();
    if (threadIdx.x == 0) s_last = handoff_count(&a.counters[h]) == (unsigned)(ng - 1);
    __syncthreads();
    if (s_last) {
      acquire_partials();
      if (threadIdx.x == 0)
        __hip_atomic_store(&a.counters[h], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      merge_partials<G, D, NT, KMAX>(a, pb, first_row * kRowElems, ng, h, n, nv, s_merge,
                                   kMergeGroup);
    }
    return;
  }
  if (threadIdx.x == 0) s_last = handoff_count(&a.counters[h]) == (unsigned)(n_act - 1);
  __syncthreads();
  if (s_last) {
    acquire_partials();
    // Last contributor of the head: merge its partials, write the outputs.
    if (threadIdx.x == 0)
      __hip_atomic_store(&a.counters[h], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    merge_partials<G, D, NT, KMAX>(a, pb, first_row * kRowElems, n_act, h, n, nv, s_merge);
  }
}

// The first page-list entries of split `split` of head bh (lane j of wave
// w: entry r0 + w + NW j) and their block-table entries, requested as early
// as possible: their position only needs r0 = split * pps.  Lanes past the
// head's pages are discarded by the walk.
template <int NW>
__device__ __forceinline__ int listed_first_entry(const DecodeArgs &a, int split, int bh,
                                                  int wave, int lane, int ts) {
  if (a.max_sel <= 0) return 0;
  return listed_tile(a, a.page_idx + (int64_t)bh * a.idx_stride,
                     min(split * a.pps + wave + NW * lane, (a.max_sel << ts) - 1), ts);
}

__device__ __forceinline__ int listed_first_block(const DecodeArgs &a, int bh, int lt, int ts) {
  if (a.max_sel <= 0) return 0;
  return tile_block(a, bh / a.H_kv, lt, ts);
}

template <int NW>
__device__ __forceinline__ void listed_first_pages(const DecodeArgs &a, int split, int bh,
                                                   int wave, int lane, int ts, int &lp,
                                                   int &phys) {
  lp = listed_first_entry<NW>(a, split, bh, wave, lane, ts);
  phys = listed_first_block(a, bh, lp, ts);
}

// The first tiles of split `split` of a head's identity walk (lane j of wave
// w: entry r0 + w + NW j, the tile of the same index) and their blocks.
template <int NW>
__device__ __forceinline__ void ident_first_pages(const DecodeArgs &a, int split, int bh,
                                                  int wave, int lane, int ts, int &lp,
                                                  int &phys) {
  lp = split * a.pps_all + wave + NW * lane;
  phys = tile_block(a, bh / a.H_kv, lp, ts);
}

// Tiles per split of a listed walk over n tiles: the launch's a.pps (sized
// on the host by its largest head, max_sel pages) for a head of max_sel
// pages, whose first entries were requested at split * a.pps before its
// count arrived; a shorter head (a per-head budget, a short context) sizes
// its splits by its own count over the launch's n_splits (a multiple of NW,
// at least kMinPagesPerWg pages), so its pages spread over every split
// instead of the first n / a.pps.  ceil(n / pps) <= n_splits either way.
template <int NW>
__device__ __forceinline__ int listed_pps(const DecodeArgs &a, int n, int ts) {
  if (n >= (a.max_sel << ts)) return a.pps;
  const int per = (n + a.n_splits - 1) / a.n_splits;
  return max((per + NW - 1) / NW * NW, kMinPagesPerWg << ts);
}

// Listed pages of a head (the sparse decode of reuse steps, and verified
// launches whose heads are all accepted): split s of head bh walks listed
// pages [s * pps, (s + 1) * pps) of bh (pps: listed_pps); splits past a
// head's pages only take part when the head is empty (split 0 writes its
// outputs).  Partial row of (split, head) = head * n_splits + split.
// With APP, the walk's sequence appends token nt in this launch: the
// context length is nt's page * 16 + row + 1 (16-token pages), and nt's page
// takes that row from nt's rows (its loads are dropped, stage_k and stage_v
// put the new row in place) and, when the append allocates the page, its
// block from nt.
// With SCORE and a.spec_scores, the walk also writes the page score of
// every page it walks (Engine::page_score; qrep: this wave's LDS copy of the
// 16 q_rep segments, 16-token pages).
template <int G, class Engine, int NW, bool APP = false, bool SCORE = false,
          bool IDENT = false>
__device__ __forceinline__ void listed_walk(const DecodeArgs &a, int split, int bh, int spec_lp,
                                            int spec_phys, WalkLds<G, Engine, NW> &L,
                                            const NewToken &nt = NewToken(),
                                            uint4 *qrep = nullptr) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = bh / a.H_kv;
  const int h = bh - b * a.H_kv;
  const int ctx = APP ? nt.page * kPageTokens + nt.off + 1
                      : __builtin_amdgcn_readfirstlane(a.ctx_lens[b]);
  const int n_spl = IDENT ? a.n_splits_all : a.n_splits;
  const int32_t *idx_row = a.page_idx + (int64_t)bh * a.idx_stride;
  const int ts = Engine::tshift(a);
  constexpr int tl = Engine::kRowsLog;
  // IDENT: entry e is tile e of the head's valid pages (n_valid as the
  // reference computes it, at most W).
  const int n = IDENT ? max(0, min(valid_pages_sh(ctx, tl + ts), a.W)) << ts
                      : min(max(__builtin_amdgcn_readfirstlane(a.n_pages[bh]), 0), a.max_sel)
                            << ts;
  const int pps = IDENT ? a.pps_all : listed_pps<NW>(a, n, ts);
  // The first entries (spec_lp, spec_phys) were requested at split * a.pps:
  // a head with splits of its own size requests them again.
  const bool refetch = !IDENT && pps != a.pps;  // uniform
  const int r0 = split * pps;
  const int r1 = min(n, r0 + pps);
  const int n_act = (n + pps - 1) / pps;  // splits holding pages of this head
  if (r0 >= r1 && !(split == 0 && n_act == 0)) return;  // uniform

  Engine eng;
  eng.init(a, b, h, lane);
  // Wave-private q_rep: lane < 16 computes segment `lane` (its loads go out
  // ahead of the first tile's) and stores it to LDS once the first tile is
  // requested; the LDS store and the later reads are the same wave's, in
  // order.
  const bool scoring = SCORE && a.spec_scores != nullptr;  // uniform
  uint4 qr_own = make_uint4(0u, 0u, 0u, 0u);
  if constexpr (SCORE) {
    if (scoring)
      qr_own = group_mean_q(a.q, a.q_sb, a.q_sh, b, h, a.q_group, min(lane, 15), a.inv_g);
  }
  const int npw = max(0, (r1 - r0 - wave + NW - 1) / NW);
  // Tile `lane` of the chunk that starts at the wave's tile c0: its entry's
  // logical tile, if valid, and that tile's physical one.
  auto chunk = [&](int c0, int lt, int phys) {
    TileChunk c;
    if (APP && lt == nt.page && nt.new_blk >= 0) phys = nt.new_blk;
    if (c0 + lane < npw && lt >= 0 && lt < (a.W << ts)) {
      const bool readable = phys >= 0 && phys < (a.num_blocks << ts);
      c.phys = readable ? phys : 0;
      c.lt = readable ? lt : kUnreadable + lt;
    }
    return c;
  };
  auto lookup = [&](int c0) {
    const int e = r0 + wave + NW * min(c0 + lane, max(npw - 1, 0));
    const int lt = IDENT ? e : listed_tile(a, idx_row, e, ts);
    return chunk(c0, lt, tile_block(a, b, lt, ts));
  };
  const TileChunk first = refetch && npw > 0 ? lookup(0) : chunk(0, spec_lp, spec_phys);
  start_walk<Engine, APP>(a, eng, first, nt.page, nt.off);
  if constexpr (SCORE) {
    if (scoring && lane < 16) qrep[lane] = qr_own;
  }
  walk_tiles<Engine, APP, SCORE>(
      a, eng, npw, ctx, first, lookup,
      [&](int lt, int ntok, const uint4 (&kop)[Engine::NK]) {
        if constexpr (SCORE) {
          if (scoring) {
            const float sc = eng.page_score(kop, ntok, qrep);
            // A page whose block is outside the pool scores -inf, as the page
            // scoring has it; the scoring workgroups leave it to this walk.
            if (lane == 0 && lt != kNoTile)
              a.spec_scores[(int64_t)bh * a.W + (lt & (kUnreadable - 1))] = sc;
          }
        }
      },
      L.eng[wave], nt.page, nt.off, nt.k, nt.v);
  eng.finish(L.eng[wave], L.m[wave], L.l[wave]);
  __syncthreads();
  const PartBuf pb(a.part, a.part_bytes);
  segment_epilogue<G, Engine, NW>(a, pb, bh, n >> ts, valid_pages_sh(ctx, tl + ts), n_act,
                                  (uint32_t)(bh * n_spl + split), (uint32_t)(bh * n_spl), L);
}

// The listed decode: a static grid of (split, head) workgroups.
template <int G, class Engine, int NW>
__global__ __launch_bounds__(NW * kWave, Engine::kWalkWaves) void listed_decode_kernel(
    const DecodeArgs a) {
  __shared__ WalkLds<G, Engine, NW> L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lp, phys;
  listed_first_pages<NW>(a, blockIdx.x, blockIdx.y, wave, lane, Engine::tshift(a), lp, phys);
  listed_walk<G, Engine, NW>(a, blockIdx.x, blockIdx.y, lp, phys, L);
}

// The listed decode of a reuse step with the step's token append folded in
// (16-token pages, D = 128): workgroup (split, bh) walks as
// listed_decode_kernel with its sequence's new token taken from k_new / v_new
// (NewToken), and split 0 of each head writes that head's new K/V rows to
// the cache slot, which no workgroup of the launch reads; split 0 of a
// sequence's first head also moves its context length, page-table entry
// and allocation count as cvsa_append_kv does.  Later launches see the
// appended cache.
// Three waves per SIMD (142 registers): at the listed decode's four (128) every
// instance spilled 1 or 2 of them to scratch, and no launch was faster for the
// fourth wave (8185 tokens, budget 25%, cold caches: B = 1 12.1 -> 11.8 us,
// B = 32 48.5 -> 47.6, B = 128 176.6 -> 173.9).
template <int G, class Engine, int NW>
__global__ __launch_bounds__(NW * kWave, 3) void listed_append_kernel(const DecodeArgs a,
                                                                      const AppendArgs app) {
  static_assert(Engine::kD == 128, "the fused append is built for D = 128");
  __shared__ WalkLds<G, Engine, NW> L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int split = blockIdx.x, bh = blockIdx.y;
  const int b = bh / a.H_kv;
  const int h = bh - b * a.H_kv;
  const int2 sl = app.slot_dev != nullptr ? app.slot_dev[b] : app.slot[b];  // uniform
  const bool ok = sl.x >= 0 && sl.x < app.max_pages * kPageTokens && sl.y >= -1 &&
                  sl.y < a.num_blocks && (sl.y < 0 || (sl.x & 15) == 0);
  NewToken nt;
  nt.page = ok ? sl.x >> 4 : -1;
  nt.off = ok ? sl.x & 15 : kPageTokens - 1;  // not ok: context length 0
  nt.new_blk = ok ? sl.y : -1;
  const int64_t row = (int64_t)b * app.new_sb + (int64_t)h * Engine::kD;
  nt.k = app.k_new + row;
  nt.v = app.v_new + row;
  int lp, phys;
  listed_first_pages<NW>(a, split, bh, wave, lane, 0, lp, phys);
  if (lp == nt.page && nt.new_blk >= 0) phys = nt.new_blk;
  // Split 0's wave 0 appends: lanes 0-15 copy the head's K row, lanes 16-31
  // its V row, 16 bytes each.  No workgroup of the launch reads the slot, the
  // context length or the new page's table entry, so the stores go out at
  // once, behind the walk's first lookups.
  const bool writer = ok && split == 0 && wave == 0;  // uniform
  if (writer) {
    const int blk =
        nt.new_blk >= 0 ? nt.new_blk : a.block_tables[(int64_t)b * a.bt_sb + nt.page];
    const uint4 x = *reinterpret_cast<const uint4 *>((lane >= 16 ? nt.v : nt.k) + 8 * (lane & 15));
    if (lane < 32 && blk >= 0 && blk < a.num_blocks) {
      const int64_t dst =
          (((int64_t)blk * kPageTokens + nt.off) * a.H_kv + h) * Engine::kD + 8 * (lane & 15);
      *reinterpret_cast<uint4 *>(const_cast<uint16_t *>(lane >= 16 ? a.v_cache : a.k_cache) +
                                 dst) = x;
    }
    if (h == 0 && lane == 0) {
      app.ctx_lens[b] = sl.x + 1;
      if (nt.new_blk >= 0) {
        app.block_tables[(int64_t)b * a.bt_sb + nt.page] = nt.new_blk;
        app.pages_allocated[b] += 1;
      }
    }
  }
  if (!ok && split == 0 && h == 0 && threadIdx.x == 0 && app.slot_errors != nullptr)
    atomicAdd(app.slot_errors, 1);  // a rejected device slot is reported, not dropped silently
  listed_walk<G, Engine, NW, true>(a, split, bh, lp, phys, L, nt);
}

// 16-token tiles per scoring wave of the fused launch below.
constexpr int kSpecScorePPW = 8;
// Pages per scoring wave of the fused launch at 16-token pages (one head per
// wave, score_head_wave).
constexpr int kSpecHeadPPW = 16;

// A lazy check's page scoring and the speculative listed decode of its
// cached selection in one launch.  Workgroups [0, n_splits * heads) are the
// listed decode's (split, head) workgroups, w -> (w % n_splits, w /
// n_splits), bit for bit listed_decode_kernel; they run only if
// spec_state[0] predicts that the check keeps its selection, and workgroup 0
// records in spec_state[1] whether they ran.  The other workgroups score
// pages (workgroup x of sequence b at index n_dec + b * score_gx + x): at
// 16-token pages one head and kSpecHeadPPW pages per wave (score_head_wave),
// else as score_pages_group_kernel<128, ...> (kSpecScorePPW tiles of 4 heads
// per wave).  With a selection map (s.skip_map) the decode part also writes
// the page scores of the pages it walks, from the keys it reads anyway, and
// the scoring part skips them when the decode runs: every page is scored
// once, with the same bits (the per-token arithmetic is the same).
// The parts share no memory otherwise: the decode reads the cached
// selection, which only the check's select-or-keep, launched after this
// kernel, rewrites.
// One launch lets the decode's dependent metadata loads and split hand-off
// overlap the scoring stream without a second stream and its events.
// Three waves per SIMD: the decode and scoring workgroups of a cfg3 launch all
// run at once.  Held to four (128 of the 137 registers it takes at G <= 8) a
// kept check takes 18.9 instead of 18.2 us at 8K, 60.2 instead of 59.8 at 128K,
// 116.7 instead of 114.4 at B = 8, 32K.  Reading the kept selection's keys once: kept check 64.0 -> 61.1 us
// at cfg3 (16 pages per scoring wave; 8 and 32 measured 61.2 and 62.0).
template <int G, class Engine, int NW>
__global__ __launch_bounds__(NW * kWave, Engine::kPages != kPages16 ? 2 : 3)
void score_spec_kernel(const DecodeArgs a, const ScoreArgs s, int score_gx) {
  __shared__ WalkLds<G, Engine, NW> L;
  __shared__ uint4 s_qrep[NW][16];  // decode part: q_rep per wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_dec = max(a.n_splits, a.n_splits_all) * a.heads;
  const int w = blockIdx.x;
  // The speculation that runs: 1 = listed decode of the cached selection
  // (predicted keep), 2 = dense decode, which needs the scoring from its
  // keys (16-token pages and a selection map), else 0.
  const int pred = __builtin_amdgcn_readfirstlane(a.spec_state[0]);
  const int go = pred == 1 ? 1
                 : pred == 2 && Engine::kPages == kPages16 && a.spec_scores != nullptr ? 2
                                                                                    : 0;
  if (w >= n_dec) {  // uniform
    const int sw = w - n_dec;
    const int gw = (sw % score_gx) * NW + wave, b = sw / score_gx;
    if constexpr (Engine::kPages == kPages16) {
      // With a skip map, the pages the speculative decode walks (when it
      // runs) are scored there: the selection's, or every valid page.
      const int ctx = __builtin_amdgcn_readfirstlane(s.context_lens[b]);
      score_head_wave<kSpecHeadPPW, 4>(s, a.H_kv, gw, b, s.skip_map != nullptr && go == 1,
                                       go == 2 ? n_valid_pages(ctx, kPageTokens) : 0);
    } else {
      score_group_wave<128, kSpecScorePPW>(s, a.H_kv, gw, b);
    }
    return;
  }
  if (w == 0 && threadIdx.x == 0) a.spec_state[1] = go;
  if (go == 1) {  // uniform
    if (w >= a.n_splits * a.heads) return;
    const int split = w % a.n_splits;
    const int bh = w / a.n_splits;
    int lp, phys;
    listed_first_pages<NW>(a, split, bh, wave, lane, Engine::tshift(a), lp, phys);
    listed_walk<G, Engine, NW, false, Engine::kPages == kPages16>(a, split, bh, lp, phys, L,
                                                                   NewToken(), s_qrep[wave]);
  } else if constexpr (Engine::kPages == kPages16) {
    if (go != 2 || w >= a.n_splits_all * a.heads) return;  // uniform
    const int split = w % a.n_splits_all;
    const int bh = w / a.n_splits_all;
    int lp, phys;
    ident_first_pages<NW>(a, split, bh, wave, lane, 0, lp, phys);
    listed_walk<G, Engine, NW, false, true, true>(a, split, bh, lp, phys, L, NewToken(),
                                                      s_qrep[wave]);
  }
}

// Every workgroup first computes the pages each head walks and their prefix
// (the same partition in every workgroup; the heads' counts and flags are
// requested together, and nothing is walked on a guess: a mixed launch, whose
// rejected heads walk other numbers of pages, would throw the guess away
// along with 8 MiB of requests), then walks the segments of its
// range: (head h, pages s0..s1 of h's walk).  A segment that is a whole head
// writes the outputs; otherwise it stores a partial (o, m, l) in row w + h of
// the partial buffer (unique: a later workgroup never starts at an earlier
// head, so (w, h) -> w + h is one-to-one, and head h's partials are the
// consecutive rows owner(first page) + h .. owner(last page) + h), bumps the
// head's counter, and the last contributor merges.  Heads that walk no pages
// are written by workgroup h mod n_wg.
template <int G, class Engine, int NW, int MODE>
__global__ __launch_bounds__(NW * kWave, Engine::kD > 128 ? 1 : 2) void streamk_decode_kernel(
    const DecodeArgs a) {
  constexpr int NT = NW * kWave;         // threads per workgroup

  __shared__ WalkLds<G, Engine, NW> L;
  __shared__ int s_wsum[NW];
  __shared__ int s_flags[NW];
  __shared__ int s_start[kMaxHeads + 1];  // exclusive prefix of pages per head
  __shared__ uint8_t s_listed[kMaxHeads];  // kWalk* of each head
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = blockIdx.x;
  const int heads = a.heads;
  constexpr int D = Engine::kD;
  const int ts = Engine::tshift(a);
  constexpr int tl = Engine::kRowsLog;

  // Tiles per head, scanned into their exclusive prefix in s_start, one head
  // per thread and pass of NT heads (loads issued without a branch, index
  // clamped); T their sum.
  int walk0 = kWalkAll, c0 = 0, T = 0;  // c0, walk0: head threadIdx.x
  auto scan_pass = [&](int hh, int c, int walk) {
    const int incl = (int)wave_incl_scan_u32((uint32_t)c);
    if (lane == kWave - 1) s_wsum[wave] = incl;
    lds_barrier();
    int excl = incl - c, total = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      if (i < wave) excl += s_wsum[i];
      total += s_wsum[i];
    }
    if (hh < heads) {
      s_start[hh] = T + excl;
      s_listed[hh] = (uint8_t)walk;
    }
    T += total;
  };

  // Verified launches whose heads are all accepted (a lazy check that keeps
  // its selection, or a scoring step whose gate passes everywhere) run the
  // listed decode's static partition: workgroup w takes split w % n_splits
  // of head w / n_splits, exactly as listed_decode_kernel, so the outputs
  // are bit for bit those of the listed decode.  Its first page-list
  // entries are requested together with the heads' counts and flags and
  // spec_state, their block-table entries once the launch is known to walk.  When the
  // check kept its selection (spec_state[0], written by the check's
  // select-or-keep) and a speculative listed decode of that selection
  // already wrote the outputs (spec_state[1]), there is nothing left: the
  // select-or-keep booked that decode's effective-budget counters.  Every
  // head accepted does not imply a kept selection: a rejected head is
  // reselected and accepted when the new selection passes its gate.
  if constexpr (MODE == kModeVerified || MODE == kModeApprox) {
    const int n_listed = a.n_splits * heads;
    const int split = w % max(a.n_splits, 1);
    const int bh = min(w / max(a.n_splits, 1), heads - 1);
    const int lp = listed_first_entry<NW>(a, split, bh, wave, lane, Engine::tshift(a));
    const bool has_spec = a.spec_state != nullptr;
    const int spec_keep = has_spec ? a.spec_state[0] : 0, spec_ran = has_spec ? a.spec_state[1] : 0;
    const bool acc0 = a.accept[min((int)threadIdx.x, heads - 1)] != 0;
    if (__builtin_amdgcn_readfirstlane(spec_keep == 1 && spec_ran == 1) != 0)
      return;  // uniform; every head was accepted (kept)
    c0 = head_pages<MODE>(a, min((int)threadIdx.x, heads - 1), walk0, ts, tl);
    // Whether some head is rejected, and some accepted: one barrier.
    enum { kSomeRejected = 1, kSomeAccepted = 2 };
    int f = acc0 ? kSomeAccepted : kSomeRejected;
    for (int i = threadIdx.x + NT; i < heads; i += NT)
      f |= a.accept[i] != 0 ? kSomeAccepted : kSomeRejected;
    f = (__ballot(f & kSomeRejected) != 0 ? kSomeRejected : 0) |
        (__ballot(f & kSomeAccepted) != 0 ? kSomeAccepted : 0);
    if (lane == 0) s_flags[wave] = f;
    lds_barrier();
    int flags = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) flags |= s_flags[i];
    flags = __builtin_amdgcn_readfirstlane(flags);
    if ((flags & kSomeRejected) == 0) {  // uniform
      if (w < n_listed)
        listed_walk<G, Engine, NW>(a, split, bh, lp,
                                   listed_first_block(a, bh, lp, Engine::tshift(a)), L);
      return;
    }
    // Every head rejected (exact recovery: each attends all its valid
    // pages): the identity partition, whose outputs a speculative dense
    // decode of the lazy check (spec_state[1] == 2) already wrote with the
    // same bits; then only its effective-budget counters are booked.  The
    // next check of the layer is told to speculate that way again.
    if (MODE == kModeVerified && (flags & kSomeAccepted) == 0) {  // uniform
      const bool dense_done = __builtin_amdgcn_readfirstlane(spec_ran) == 2;
      if (w == 0 && threadIdx.x == 0 && has_spec) a.spec_state[0] = 2;
      if (dense_done) {
        if (w == 0 && a.work != nullptr) {
          for (int i = threadIdx.x; i < heads; i += NT) {
            const int nv = valid_pages_sh(a.ctx_lens[i / a.H_kv], tl + ts);
            add_work(a, max(0, min(nv, a.W)), nv);
          }
        }
        return;
      }
      if (w >= a.n_splits_all * heads) return;
      const int isplit = w % a.n_splits_all;
      const int ibh = w / a.n_splits_all;
      int ilp, iphys;
      ident_first_pages<NW>(a, isplit, ibh, wave, lane, ts, ilp, iphys);
      listed_walk<G, Engine, NW, false, false, true>(a, isplit, ibh, ilp, iphys, L);
      return;
    }
  } else {
    c0 = head_pages<MODE>(a, min((int)threadIdx.x, heads - 1), walk0, ts, tl);
  }
  scan_pass(threadIdx.x, (int)threadIdx.x < heads ? c0 : 0, walk0);
  for (int base = NT; base < heads; base += NT) {  // uniform
    lds_barrier();  // s_wsum is rewritten
    const int hh = base + threadIdx.x;
    int walk = kWalkAll;
    const int c = head_pages<MODE>(a, min(hh, heads - 1), walk, ts, tl);
    scan_pass(hh, hh < heads ? c : 0, walk);
  }
  if (threadIdx.x == 0) s_start[heads] = T;
  lds_barrier();  // s_start and s_listed
  T = __builtin_amdgcn_readfirstlane(T);

  const Partition part(max(T, 1), a.sk_grid, min_sk_tiles(MODE == kModeApprox));
  const int n_wg = T > 0 ? part.n : a.sk_grid;
  if (w >= n_wg) return;  // uniform

  // Heads without pages: (o, m, l) = (0, -inf, 0), zero output.
  for (int hh = w; hh < heads; hh += n_wg) {
    if (s_start[hh + 1] != s_start[hh]) continue;  // uniform
    const int64_t row0 = (int64_t)hh * a.q_group + a.q_off;
    for (int i = threadIdx.x; i < G * D; i += NT)
      write_outputs<D>(a, row0 + i / D, i % D, 0.f, -INFINITY, 0.f);
    if (threadIdx.x == 0 && a.work != nullptr) {
      const int nv = valid_pages_sh(a.ctx_lens[hh / a.H_kv], tl + ts);
      add_work(a, MODE == kModeApprox ? approx_booked_pages(a, hh, nv) : 0, nv);
    }
  }
  if (T == 0) return;

  const int g0 = part.start(w);
  const int g1 = part.start(w + 1);
  // First head of the range: the last head that starts at or before g0 (it
  // holds tile g0, so it is not empty), a wave's worth of starts per read:
  // every `step`-th head, then the heads of one step.
  static_assert(kMaxHeads <= kWave * kWave, "two reads find the head");
  const int step = (heads + kWave - 1) / kWave;
  auto starts_at_or_before = [&](int h0, int each, int end) {
    const int h = h0 + lane * each;
    return __popcll(__ballot(h < end && s_start[min(h, heads)] <= g0));
  };
  int lo = (starts_at_or_before(0, step, heads) - 1) * step;
  if (step > 1) lo += starts_at_or_before(lo, 1, min(lo + step, heads)) - 1;
  const PartBuf pb(a.part, a.part_bytes);

  for (int h = lo; h < heads; ++h) {
    const int P = __builtin_amdgcn_readfirstlane(s_start[h]);
    if (P >= g1) break;  // uniform
    const int n = __builtin_amdgcn_readfirstlane(s_start[h + 1]) - P;
    if (n == 0) continue;
    const int s0 = max(g0, P) - P, s1 = min(g1, P + n) - P;
    const int b = h / a.H_kv;
    const int hk = h - b * a.H_kv;
    const int walk = s_listed[h];
    const bool listed = walk != kWalkAll;
    const int ctx = __builtin_amdgcn_readfirstlane(a.ctx_lens[b]);
    const int32_t *idx_row = MODE == kModeApprox && walk == kWalkAlt
                                 ? a.alt_idx + (int64_t)h * a.alt_stride
                                 : a.page_idx + (int64_t)h * a.idx_stride;
    const int npw = max(0, (s1 - s0 - wave + NW - 1) / NW);
    // Tiles e0 .. of the wave's part (tiles s0 + wave + NW e), one per lane.
    auto lookup = [&](int e0) {
      const int r = s0 + wave + NW * min(e0 + lane, max(npw - 1, 0));
      const int lt = listed ? listed_tile(a, idx_row, r, ts) : r;
      const int phys = tile_block(a, b, lt, ts);
      TileChunk c;
      if (e0 + lane < npw && lt >= 0 && lt < (a.W << ts) && phys >= 0 &&
          phys < (a.num_blocks << ts)) {
        c.phys = phys;
        c.lt = lt;
      }
      return c;
    };
    TileChunk first;
    if (npw > 0) first = lookup(0);
    Engine eng;
    eng.init(a, b, hk, lane);
    start_walk<Engine>(a, eng, first);
    walk_tiles<Engine, false, false>(
        a, eng, npw, ctx, first, lookup, [](int, int, const uint4 (&)[Engine::NK]) {},
        L.eng[wave]);
    eng.finish(L.eng[wave], L.m[wave], L.l[wave]);
    __syncthreads();

    const int first_wg = part.owner(P);
    const int nv = valid_pages_sh(ctx, tl + ts);
    const int booked = MODE == kModeApprox ? approx_booked_pages(a, h, nv) : n >> ts;
    segment_epilogue<G, Engine, NW, true>(a, pb, h, booked, nv,
                                          part.owner(P + n - 1) - first_wg + 1,
                                          (uint32_t)(w + h), (uint32_t)(first_wg + h), L);
    __syncthreads();  // LDS is reused by the next segment
  }
}

// Workgroups per launch, at most kMaxSplits (a head's partials are merged
// in one workgroup's LDS): one per CU of the 256-CU part.
constexpr int kTargetWorkgroups = 256;
static_assert(kTargetWorkgroups <= kMaxSplits, "one merge per head fits the merge LDS");

// Launches of a validated decode for GQA group size G, explicitly
// instantiated per G in the decode_g*.hip and decode_pages8_g*.hip files (one
// translation unit per four group sizes, so the objects compile in parallel).
enum { kLaunchListed = 0, kLaunchVerified = 1, kLaunchAll = 2, kLaunchApprox = 3 };

template <int G, int D, int PAGES>
void launch_decode_gdp(const DecodeArgs &a, int kind, dim3 grid, hipStream_t st) {
  const dim3 block(kWavesPerWg * kWave);
  using E = MfmaEngine<G, D, PAGES>;
  if (kind == kLaunchListed)
    hipLaunchKernelGGL((listed_decode_kernel<G, E, kWavesPerWg>), grid, block, 0, st, a);
  else if (kind == kLaunchVerified)
    hipLaunchKernelGGL((streamk_decode_kernel<G, E, kWavesPerWg, kModeVerified>), grid,
                       block, 0, st, a);
  else if (kind == kLaunchApprox)
    hipLaunchKernelGGL((streamk_decode_kernel<G, E, kWavesPerWg, kModeApprox>), grid,
                       block, 0, st, a);
  else
    hipLaunchKernelGGL((streamk_decode_kernel<G, E, kWavesPerWg, kModeAll>), grid, block, 0,
                       st, a);
}

template <int G, int PAGES>
void launch_decode_gp(const DecodeArgs &a, int kind, dim3 grid, hipStream_t st) {
  if (a.D == 32)
    launch_decode_gdp<G, 32, PAGES>(a, kind, grid, st);
  else if (a.D == 64)
    launch_decode_gdp<G, 64, PAGES>(a, kind, grid, st);
  else if (a.D == 256)
    launch_decode_gdp<G, 256, PAGES>(a, kind, grid, st);
  else
    launch_decode_gdp<G, 128, PAGES>(a, kind, grid, st);
}

// The reuse step's listed decode with the token append (D = 128, 16-token
// pages).
template <int G>
void launch_append_g(const DecodeArgs &a, const AppendArgs &app, dim3 grid, hipStream_t st) {
  hipLaunchKernelGGL((listed_append_kernel<G, MfmaEngine<G, 128, kPages16>, kWavesPerWg>), grid,
                     dim3(kWavesPerWg * kWave), 0, st, a, app);
}

// The lazy check's fused scoring + speculative decode (D = 128).
template <int G>
void launch_spec_g(const DecodeArgs &a, const ScoreArgs &s, int score_gx, dim3 grid,
                   hipStream_t st) {
  if (a.ts == 0)
    hipLaunchKernelGGL((score_spec_kernel<G, MfmaEngine<G, 128, kPages16>, kWavesPerWg>), grid,
                       dim3(kWavesPerWg * kWave), 0, st, a, s, score_gx);
  else
    // Pages of several tiles: the scoring part reads the selection's keys too.
    // us a kept check with K loads that stream -> as here (H_kv = 8, G = 4;
    // before the walk streamed whole K rows): 64-token pages, 128K tokens 62.0 ->
    // 60.0 (61.4), 512K 221 -> 206 (206), 8 ragged sequences of 32K 108.7 ->
    // 102.8 (102.7); 32-token pages, 512K 220 -> 207 (207).
    hipLaunchKernelGGL((score_spec_kernel<G, MfmaEngine<G, 128, kPagesWide, true>, kWavesPerWg>),
                       grid, dim3(kWavesPerWg * kWave), 0, st, a, s, score_gx);
}

#define CVSA_DECODE_LAUNCHERS(PREFIX, GG)                                                    \
  PREFIX template void launch_decode_gp<GG, kPages16>(const DecodeArgs &, int, dim3,          \
                                                      hipStream_t);                           \
  PREFIX template void launch_decode_gp<GG, kPagesWide>(const DecodeArgs &, int, dim3,        \
                                                        hipStream_t);                         \
  PREFIX template void launch_spec_g<GG>(const DecodeArgs &, const ScoreArgs &, int, dim3,   \
                                         hipStream_t);                                         \
  PREFIX template void launch_append_g<GG>(const DecodeArgs &, const AppendArgs &, dim3,      \
                                           hipStream_t);
#define CVSA_DECODE_EXTERN(GG) \
  CVSA_DECODE_LAUNCHERS(extern, GG) CVSA_PAGES8_LAUNCHERS(extern, GG)
#define CVSA_DECODE_INSTANTIATE(GG) CVSA_DECODE_LAUNCHERS(, GG)
// 8-token pages: decode_pages8_g*.hip.
#define CVSA_PAGES8_LAUNCHERS(PREFIX, GG)                                             \
  PREFIX template void launch_decode_gp<GG, kPages8>(const DecodeArgs &, int, dim3,   \
                                                     hipStream_t);
#define CVSA_PAGES8_INSTANTIATE(GG) CVSA_PAGES8_LAUNCHERS(, GG)

constexpr int kMaxGroup = 16;       // query heads of one launch: one MFMA tile
constexpr int kMaxGroupTotal = 128;  // query heads per KV head (launches of 16)

}  // namespace cvsa
