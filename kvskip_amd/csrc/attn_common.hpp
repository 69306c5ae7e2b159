// Shared device code of the split-K flash-decode kernels for gfx950 (attn_decode.hip: dense,
// block-list, per-block statistics, stats-only, fp16 P; attn_vskip.hip: single-pass V-skip,
// two-pass V-skip pass 2, read ceiling).
//
// Work decomposition. num_splits * Hkv * B workgroups of NWAVE wavefronts; a workgroup owns one
// contiguous range of "items" (64-token blocks, or entries of a block list) of one KV head
// and serves all G query heads of that head, so each K/V byte is read once. Workgroups are
// dispatched round-robin over the 8 XCDs; the launch index is remapped so that consecutive
// work items (the splits of one KV head) land on the same XCD.
// Inside the workgroup the wavefronts are independent streams: wavefront w takes items w,
// w+NWAVE, ... and keeps its own online-softmax state for the G heads, so the main loop has no
// workgroup barrier. A wavefront processes a whole 64-token block at a time, so the
// per-block statistics fall out of its own registers. The 4 states are merged once, in LDS,
// at the end. With num_splits > 1 each workgroup writes its partial state and a second,
// short kernel merges the splits (8 split classes x 32 dims per workgroup). A merge inside the
// same kernel (last-arriving workgroup) costs more than that launch on gfx950: with device-scope
// fences (an L2 write-back and invalidate per workgroup) 2x slower at 2 workgroups per CU; with
// the partials stored and read at agent scope (no write-back) and a self-resetting ticket, +3.8 us
// per op at config 2 (dense and masked alike, graph-replayed or eager): the pass's tail gains
// three dependent memory round trips (store completion, ticket, partials), more than the
// dispatch gap of the merge kernel.
//
// Pipeline per wavefront: K(j) and V(j) are in flight when block j starts; after QK(j) the K
// loads of block j+1 are issued, after PV(j) its V loads. Every load in the loop is unconditional
// (exact wait counts): the MFMA engine's last block requests one past the head's range (zeros, no
// memory access), the VALU engine peels its last block off.
//
// Two engines (chosen per launch, KVSKIP_AMD_QK=valu|mfma):
//   mfma  both products on v_mfma_f32_16x16x32_bf16, nothing through LDS between them. Scores come out
//         transposed: A = 16 tokens of K, B = the query heads as 16 columns, so a lane holds 16 scores
//         of ONE head (column c = lane % 16) of a 64-token block, its softmax is in-lane arithmetic plus
//         two lane swaps, and its weights already lie as the A operand of P V (row = lane % 16, tokens by
//         lane / 16). V is read with 8 (D 64: 4) dims of a row per lane; two rows' halves are paired by
//         v_perm into B operands whose column c is dim 8 c + j. Weights stay fp32: a weight is the exact
//         sum of three bf16 parts (hi, mid, lo: 8 + 8 + 8 bits), and since the group's G <= 8 heads leave
//         rows free, the 16 rows are the parts of the heads (4 heads x 3 parts in one product, or 8 heads
//         x 2 in two: hi / 2 and mid, hi / 2 and lo). The products are exact and
//         summed in fp32, as the VALU engine's.
//         What it replaced: P through LDS and G x 128 FMAs plus 128 conversions per lane and block
//         (D 128), which at G 7 took longer than the block's loads (figures at PFrag below).
//   valu  (below) dot products on v_dot2_f32_bf16, P V on fp32 FMAs.
// Lane layouts of the VALU engine (64 lanes, D = 64 or 128):
//   K   8 lanes per token row, 8 rows per load; lane (r8 = lane/8, sub = lane%8) holds rows
//       8*rg + r8 (rg = 0..7), dims [8 sub, 8 sub + 8) (+64 for D = 128), as packed bf16.
//       QK = v_dot2_f32_bf16 against the unscaled bf16 query (exact products, fp32 sums),
//       then a 3-step DPP sum over the 8 lanes of the row; the score is scaled after.
//   V   D/8 lanes per row, 8 dims per lane, 16-byte loads; lane accumulates its rows for
//       all G heads in fp32 (acc[G][8]); P reaches the V layout through a per-wavefront
//       LDS tile [64][G] written after the softmax.
// Softmax runs in log2 units (v_exp_f32); per head and block: block max mt, e = 2^(s - mt)
// (the block statistics), p = e * 2^(mt - m_run). K/V are read through buffer resources
// bounded to the head's rows, so rows past T read as zeros; their scores are masked to -inf.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace kvs {
namespace {

#ifndef KVS_NWAVE
#define KVS_NWAVE 4
#endif
constexpr int NWAVE = KVS_NWAVE;  // wavefronts per attention workgroup
constexpr int NT = NWAVE * WAVE;

template <int D>
struct Lay {
  static_assert(D == 64 || D == 128, "head dim");
  static constexpr int KC = D / 64;         // 16-byte K chunks per lane per row
  static constexpr int VLPR = D / 8;        // lanes per V row
  static constexpr int VRPI = WAVE / VLPR;  // V rows per load instruction
  static constexpr int VN = BLK / VRPI;     // V load instructions per block
};

template <int G>
constexpr int gpad() {
  return G <= 4 ? 4 : 8;
}

// Launch index -> work index, XCD-aware when n % 8 == 0: launch index i is dispatched to XCD
// i % 8, and w = (i % 8) * (n / 8) + i / 8 gives each XCD a contiguous run of work items (a
// launch whose first workgroups do other work only rotates which XCD holds which run).
__device__ __forceinline__ int xcd_remap(int i, int n) { return n % 8 == 0 ? (i % 8) * (n / 8) + i / 8 : i; }

// Work coordinates (split, KV head, sequence) of decode workgroup `bid`.
__device__ __forceinline__ void work_coords(int bid, int S, int Hkv, int B, int& split, int& h, int& b) {
  const int i = xcd_remap(bid, S * Hkv * B);
  split = i % S;
  const int r = i / S;
  h = r % Hkv;
  b = r / Hkv;
}
__device__ __forceinline__ void work_coords(int S, int Hkv, int B, int& split, int& h, int& b) {
  work_coords(blockIdx.x, S, Hkv, B, split, h, b);
}

// ---- Ragged batches (seq_lens): sequence b attends tokens [0, clamp(seq_lens[b], 1, T)).
__device__ __forceinline__ int seq_len(const AttnP& p, int b) {
  return p.seq_lens != nullptr ? min(max(p.seq_lens[b], 1), p.T) : p.T;
}

// Items of sequence b on KV head h: its blocks (dense) or its list entries (masked).
__device__ __forceinline__ int ragged_items(const AttnP& p, int b, int h, bool masked) {
  if (masked) return min(max(p.block_cnt[b * p.Hkv + h], 0), p.max_blocks);
  return (seq_len(p, b) + BLK - 1) / BLK;
}

// Chunk lengths of the ragged partitions. A length C0 set for S slots of a (S + B)-slot grid
// (S = num_splits) leaves the grid's last B slots to the sequences' (or lists') partial chunks, so
// where the whole grid is resident (at most RESIDENT_SLOTS workgroups: two per CU) most CUs hold
// full chunks and the rest partial ones. There, with long chunks (C0 >= 32 items), C is the smallest
// length whose chunks (sum of ceil(n / C) over the lanes' counts nv) still fit the slots, found by
// bisection between lo and C0 (C0 fits), and at least lo; with short chunks or a queued grid the
// shorter chunks' fixed costs win. Config 5's dense pass (per-head partition, one workgroup per CU):
// 121.0 -> 113.2 us per layer-step. Uniform.
constexpr int RESIDENT_SLOTS = 512;

// A ragged grid ((num_splits + B) * Hkv workgroups) longer than the resident slots: its queued
// workgroups start as others end.
__device__ __forceinline__ bool grid_queued(const AttnP& p) {
  return (p.num_splits + p.B) * p.Hkv > RESIDENT_SLOTS;
}

template <int NR>
__device__ __forceinline__ int fit_chunk_len(const AttnP& p, const int (&nv)[NR], int n_lists, int lo, int c0,
                                             int slots) {
  if (grid_queued(p) || c0 < 32) return c0;
  int hi = c0;
  lo = __builtin_amdgcn_readfirstlane(min(lo, c0));
  while (lo < hi) {  // the chunk count does not grow with C
    const int mid = (lo + hi) >> 1;
    int n = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (r * WAVE < n_lists) n += (nv[r] + mid - 1) / mid;
    n = __builtin_amdgcn_readfirstlane(wave_sum_int(n));
    if (n <= slots)
      hi = mid;
    else
      lo = mid + 1;
  }
  return lo;
}

// Ragged partition of KV head h (per head; list_partition 0): the items of its B sequences (blocks,
// or list entries when masked) in chunks of one length C, numbered sequence by sequence, at most
// S + B chunks per head (C0 = ceil(sum_b items_b / S); bisected as fit_chunk_len says, at least
// ceil(most / S) so that no sequence has more than S chunks). Lane j holds sequences j + 64 r in nv.
// Returns C, uniform.
constexpr int NRB = MAX_RAGGED_B / WAVE;

__device__ __forceinline__ int ragged_chunk_len(const AttnP& p, int h, bool masked, int (&nv)[NRB]) {
  const int lane = threadIdx.x % WAVE;
  int tot = 0, most = 0;
#pragma unroll
  for (int r = 0; r < NRB; ++r) {
    const int bb = r * WAVE + lane;
    nv[r] = bb < p.B ? ragged_items(p, bb, h, masked) : 0;
    tot += nv[r];
    most = max(most, nv[r]);
  }
  tot = wave_sum_int(tot);
  most = static_cast<int>(wave_max(static_cast<float>(most)));  // exact: counts <= 2^24
  const int S = p.num_splits;
  const int c0 = __builtin_amdgcn_readfirstlane(max(1, (tot + S - 1) / S));
  const int lo = max(max(1, (most + S - 1) / S), (tot + S + p.B - 1) / (S + p.B));
  return fit_chunk_len(p, nv, p.B, lo, c0, S + p.B);
}

// Chunk number `it` of KV head h's ragged partition, uniform over the wavefront: b (-1 past the
// head's last chunk), the chunk within b and b's item count. Returns C.
__device__ int ragged_lookup(const AttnP& p, int h, int it, bool masked, int& b, int& chunk, int& items) {
  const int lane = threadIdx.x % WAVE;
  int nv[NRB];
  const int C = ragged_chunk_len(p, h, masked, nv);
  b = -1;
  chunk = 0;
  items = 0;
  int base = 0;
#pragma unroll
  for (int r = 0; r < NRB; ++r) {
    if (r * WAVE >= p.B) break;
    const int ch = (nv[r] + C - 1) / C;
    const int incl = wave_incl_scan(ch);
    const int excl = base + incl - ch;
    const uint64_t hit = __ballot(ch > 0 && it >= excl && it < excl + ch);
    if (hit != 0) {
      const int l = __ffsll(static_cast<unsigned long long>(hit)) - 1;
      b = r * WAVE + l;
      chunk = it - __shfl(excl, l, WAVE);
      items = __shfl(nv[r], l, WAVE);
    }
    base += __shfl(incl, WAVE - 1, WAVE);
  }
  b = __builtin_amdgcn_readfirstlane(b);  // uniform: scalar registers for the addressing that follows
  chunk = __builtin_amdgcn_readfirstlane(chunk);
  items = __builtin_amdgcn_readfirstlane(items);
  return C;
}

// Chunks (split partials) of (b, KV head h) under the ragged partition.
__device__ __forceinline__ int ragged_chunks(const AttnP& p, int b, int h, bool masked) {
  int nv[NRB];
  const int C = ragged_chunk_len(p, h, masked, nv);
  return (ragged_items(p, b, h, masked) + C - 1) / C;
}

// Partition over all B * Hkv lists of a masked ragged pass (p.list_partition = 1): ceil(n / C)
// chunks of each list's n entries (their bounds: decode_body), numbered list by list (l = b Hkv +
// h), so a KV head whose lists hold more entries (a refreshing sequence) gets more workgroups
// instead of longer chunks. C0 = max(ceil(sum /
// (S Hkv)), ceil(most / S)) fits the grid's (S + B) Hkv slots (sum / C0 <= S Hkv, plus at most one
// partial chunk per list), bisected as fit_chunk_len says (per layer-step with carried updates,
// config 5 131.1 -> 125.0 us, B 8 179.1 -> 173.4; bisected for every grid, B 8 with stable queries
// +0.4 us and B 32 at 64k +3.5 us). Lane j holds lists j + 64 r in nv. Returns C, uniform.
constexpr int NRG = MAX_GLOBAL_LISTS / WAVE;

__device__ __forceinline__ int global_chunk_len(const AttnP& p, int (&nv)[NRG]) {
  const int lane = threadIdx.x % WAVE, nl = p.B * p.Hkv;
  int tot = 0, most = 0;
#pragma unroll
  for (int r = 0; r < NRG; ++r) {
    const int l = r * WAVE + lane;
    nv[r] = l < nl ? min(max(p.block_cnt[l], 0), p.max_blocks) : 0;
    tot += nv[r];
    most = max(most, nv[r]);
  }
  tot = wave_sum_int(tot);
  most = static_cast<int>(wave_max(static_cast<float>(most)));  // exact: counts <= 2^24
  const int S = p.num_splits, slots = (S + p.B) * p.Hkv;
  const int c_min = max(1, (most + S - 1) / S);
  const int c0 = __builtin_amdgcn_readfirstlane(max(c_min, (tot + S * p.Hkv - 1) / (S * p.Hkv)));
  return fit_chunk_len(p, nv, nl, max(c_min, (tot + slots - 1) / slots), c0, slots);
}

// Chunk number `it` of the partition over all lists: its list (b, h; b = -1 past the last chunk),
// the chunk within the list and the list's entry count. Returns C. Uniform results. A grid longer
// than the resident slots (queued workgroups start as others end) takes the lists' full chunks
// first and their partial last chunks after them, the longer half of those first, so that it ends
// on its shortest chunks (B 32 at 64k, stable queries: 592.4 -> 579.8 us per layer-step, and
// 580.2-582.0 -> 577.6-578.1 with the two classes of partial chunks); a resident grid takes them
// list by list.
__device__ int global_lookup(const AttnP& p, int it, int& b, int& h, int& chunk, int& items) {
  const int lane = threadIdx.x % WAVE, nl = p.B * p.Hkv;
  int nv[NRG];
  const int C = global_chunk_len(p, nv);
  const bool queued = grid_queued(p);
  int l_sel = -1;
  chunk = 0;
  items = 0;
  int base = 0;
  // round one: every chunk of a list (resident grid) or its full chunks (queued grid)
#pragma unroll
  for (int r = 0; r < NRG; ++r) {
    if (r * WAVE >= nl) break;
    const int ch = queued ? nv[r] / C : (nv[r] + C - 1) / C;
    const int incl = wave_incl_scan(ch);
    const int excl = base + incl - ch;
    const uint64_t hit = __ballot(ch > 0 && it >= excl && it < excl + ch);
    if (hit != 0) {
      const int j = __ffsll(static_cast<unsigned long long>(hit)) - 1;
      l_sel = r * WAVE + j;
      chunk = it - __shfl(excl, j, WAVE);
      items = __shfl(nv[r], j, WAVE);
    }
    base += __shfl(incl, WAVE - 1, WAVE);
  }
  // rounds two and three: the partial last chunks, the longer ones (at least C / 2) first
  for (int cls = 0; cls < 2 && queued && __builtin_amdgcn_readfirstlane(l_sel) < 0; ++cls) {
#pragma unroll
    for (int r = 0; r < NRG; ++r) {
      if (r * WAVE >= nl) break;
      const int rem = nv[r] % C;
      const int part = rem != 0 && (2 * rem >= C) == (cls == 0) ? 1 : 0;
      const int incl = wave_incl_scan(part);
      const uint64_t hit = __ballot(part != 0 && it == base + incl - 1);
      if (hit != 0) {
        const int j = __ffsll(static_cast<unsigned long long>(hit)) - 1;
        l_sel = r * WAVE + j;
        items = __shfl(nv[r], j, WAVE);
        chunk = items / C;
      }
      base += __shfl(incl, WAVE - 1, WAVE);
    }
  }
  l_sel = __builtin_amdgcn_readfirstlane(l_sel);
  b = l_sel >= 0 ? l_sel / p.Hkv : -1;
  h = l_sel >= 0 ? l_sel % p.Hkv : 0;
  chunk = __builtin_amdgcn_readfirstlane(chunk);
  items = __builtin_amdgcn_readfirstlane(items);
  return C;
}

// Blocks per wavefront from which on a pass with V streams "long" (K taken direct, see KStage; the
// rotation below short).
constexpr int LONG_BLOCKS = 24;

// Item of step k of a wavefront with nw > 0 items: k rotated by the workgroup's place among its sequence's (the
// KV head and the split alone: a sequence adds its blocks in the same order in every batch slot and wherever its
// rows lie, over pages too, and passes that cut alike add alike; decode_body adds a ragged batch's item counts).
// Without it every workgroup starts at the same offset of its own range, and where the ranges lie at multiples of
// the memory's channel interleave apart all of them read the same few channels at a time: B 1 at 64k in a buffer of
// 66048 tokens 61 -> 44.2 us per op, B 2 107 -> 81.4, single-pass V-skip at 64k 40.8 -> 24.4, B 64 at 2048 85.7 ->
// 79.3; other short ones within 2%.
// Long streams drift apart by themselves, and spread further they lose locality: they rotate by up to 4 of their
// items. B 8 at 64k 319.5 us (none: 325). Where a head is one split the ranges are a head stride apart and the gain
// depends on it (B 32 unless given, tokens of the buffer, us, rotated / not): 36864 697 / 722, 40960 816 / 858,
// 49152 965 / 1000, 65536 1268 / 1290, D 64 98304 940 / 1049; but 32784 617 / 607, 65568 1273 / 1262, 65792
// 1293 / 1277, 69632 1442 / 1429, B 64 at 32768 1300 / 1267; elsewhere within 0.5%. Rotated where the stride asks
// for it only, the sums' order would follow the buffer's shape, and pages would no longer give the contiguous
// cache's bits. By up to 3: D 64 98304 961, 65568 1281, 65792 1282, B 64 1269, else the same; by 8: 32784 651, 65568
// 1283, 49152 954, D 64 98304 919.
__device__ __forceinline__ int item_rotation(const AttnP& p, int h, int split, int nw) {
  const int span = nw < LONG_BLOCKS ? nw : 4;
  return nw > 0 ? __builtin_amdgcn_readfirstlane((h * p.num_splits + split) % span) : 0;
}
__device__ __forceinline__ int rotated(int k, int rot, int nw) {
  const int i = min(k, nw - 1) + rot;
  return i >= nw ? i - nw : i;
}

// Byte range of one (b, head) of a K or V view: rows 0..T-1 of D bf16 each, row stride st.
__device__ __forceinline__ uint32_t head_bytes(int T, int64_t st, int D) {
  return static_cast<uint32_t>((static_cast<int64_t>(T - 1) * st + D) * 2);
}

// ---- Paged cache: block blk of a sequence's KV head h is page pg of a pool (page stride psb
// elements, head stride sh, row stride st). The resource's base is placed 64 blk rows before the
// page, so the block's loads use the offsets of a view (token t0 = 64 blk); its range ends at the
// block's last token below Tb (rows past it read zero) and is empty for an empty block (blk or pg
// < 0). No offset below the page is ever formed.
__device__ __forceinline__ rsrc_t block_rsrc(const uint16_t* pool, int64_t psb, int64_t sh, int64_t st, int h,
                                             int blk, int pg, int Tb, int D) {
  if (blk < 0 || pg < 0) return make_rsrc(pool, 0u);
  return make_rsrc(pool + static_cast<int64_t>(pg) * psb + static_cast<int64_t>(h) * sh -
                       static_cast<int64_t>(blk) * BLK * st,
                   head_bytes(min(Tb, blk * BLK + BLK), st, D));
}

// The pages of a workgroup's items t < n (block blk_of(t)) of sequence b into LDS sPg (and the
// blocks into sBk, if given): -1 for blocks outside [0, nb) and page ids outside [0, num_pages).
// One pass of the workgroup's threads, then a barrier; the streaming loops read these without a
// vector-memory wait.
template <class BlockOf>
__device__ __forceinline__ void gather_pages(const AttnP& p, int b, int n, int nb, BlockOf blk_of, int* sPg,
                                             int* sBk) {
  const int* tbl = p.block_table + static_cast<int64_t>(b) * p.bt_stride;
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    int blk = blk_of(t);
    if (blk < 0 || blk >= nb) blk = -1;
    int pg = blk >= 0 ? tbl[blk] : -1;
    if (pg < 0 || pg >= p.num_pages) pg = -1;
    sPg[t] = pg;
    if (sBk != nullptr) sBk[t] = blk;
  }
  __syncthreads();
}

// K block at token t0: lane (r8, sub) gets rows t0 + 8 rg + r8, 16-byte chunks sub (+8).
// koff = r8 * k_st * 2 + 16 * sub (per lane, fixed).
template <int D>
__device__ __forceinline__ void load_k_block(u32x4 (&kr)[8][Lay<D>::KC], rsrc_t rk, uint32_t koff, int64_t k_st,
                                             int t0) {
  const uint32_t rowb = static_cast<uint32_t>(k_st * 2);
#pragma unroll
  for (int rg = 0; rg < 8; ++rg) {
    const uint32_t so = static_cast<uint32_t>(t0 + 8 * rg) * rowb;
#pragma unroll
    for (int c = 0; c < Lay<D>::KC; ++c) kr[rg][c] = bload16<BUF_NT>(rk, koff + 128 * c, so);
  }
}

// V block at token t0: lane (vrow, vsub) gets rows t0 + VRPI i + vrow, dims 8 vsub .. +8.
// voff = vrow * v_st * 2 + 16 * vsub.
template <int D>
__device__ __forceinline__ void load_v_block(u32x4 (&vr)[Lay<D>::VN], rsrc_t rv, uint32_t voff, int64_t v_st,
                                             int t0) {
  constexpr int VRPI = Lay<D>::VRPI;
  const uint32_t rowb = static_cast<uint32_t>(v_st * 2);
#pragma unroll
  for (int i = 0; i < Lay<D>::VN; ++i)
    vr[i] = bload16<BUF_NT>(rv, voff, static_cast<uint32_t>(t0 + VRPI * i) * rowb);
}

// Scores of one block in log2 units: s[rg][g] for row 8*rg + lane/8; rows t0 + r >= t_lim are
// masked to -inf (t_lim = T, or 0 for an invalid list entry).
template <int D, int G>
__device__ __forceinline__ void qk_block(float (&s)[8][G], const u32x4 (&kr)[8][Lay<D>::KC],
                                         const u32x4 (&qv)[G][Lay<D>::KC], float scale_log2, int t0, int t_lim,
                                         int lane) {
#pragma unroll
  for (int rg = 0; rg < 8; ++rg)
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float a = 0.f;
#pragma unroll
      for (int c = 0; c < Lay<D>::KC; ++c) a = dot8(qv[g][c], kr[rg][c], a);
      s[rg][g] = a;
    }
#pragma unroll
  for (int rg = 0; rg < 8; ++rg)
#pragma unroll
    for (int g = 0; g < G; ++g) s[rg][g] = sum8(s[rg][g]);
  const int r8 = lane >> 3;
#pragma unroll
  for (int rg = 0; rg < 8; ++rg) {
    const bool ok = t0 + 8 * rg + r8 < t_lim;
#pragma unroll
    for (int g = 0; g < G; ++g) s[rg][g] = ok ? s[rg][g] * scale_log2 : NEG_INF;
  }
}

// acc[g][e] += sum over the block's rows of P[row][g] * V[row][dims of this lane].
template <int D, int G>
__device__ __forceinline__ void pv_block(float (&acc)[G][8], const u32x4 (&vr)[Lay<D>::VN], const float* sPw,
                                         int lane) {
  constexpr int GP = gpad<G>();
  constexpr int VRPI = Lay<D>::VRPI;
  const int vrow = lane / Lay<D>::VLPR;
#pragma unroll
  for (int i = 0; i < Lay<D>::VN; ++i) {
    const float* pr = sPw + (VRPI * i + vrow) * GP;
    float pg[GP];
#pragma unroll
    for (int u = 0; u < GP; u += 4) {
      const float4 t = *reinterpret_cast<const float4*>(pr + u);
      pg[u] = t.x;
      pg[u + 1] = t.y;
      pg[u + 2] = t.z;
      pg[u + 3] = t.w;
    }
    float vf[8];
    vf[0] = bf_lo(vr[i].x);
    vf[1] = bf_hi(vr[i].x);
    vf[2] = bf_lo(vr[i].y);
    vf[3] = bf_hi(vr[i].y);
    vf[4] = bf_lo(vr[i].z);
    vf[5] = bf_hi(vr[i].z);
    vf[6] = bf_lo(vr[i].w);
    vf[7] = bf_hi(vr[i].w);
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][e] = fmaf(pg[g], vf[e], acc[g][e]);
  }
}

// Sum acc over the lanes that hold the same dims (the V row slots).
template <int D, int G>
__device__ __forceinline__ void reduce_acc_rows(float (&acc)[G][8]) {
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float a = acc[g][e];
      if constexpr (D == 64) a += dpp<DPP_ROR8>(a);
      a += xshfl(a, 16);
      a += xshfl(a, 32);
      acc[g][e] = a;
    }
}

// LDS of the workgroup epilogue. NP: parts of each accumulator (the MFMA engine's, PFrag::NP; 1 on the
// VALU engine; 0: no accumulators, K only).
template <int D, int G, int NP>
struct MergeLds {
  float acc[NP > 0 ? NWAVE * NP * G * D : 4];  // per-wavefront accumulators [wave][part][g][d]
  float ml[NWAVE * G * 2];                     // per-wavefront (m, l)
};

// Accumulators of (head g, dim d) of every wavefront from the epilogue's LDS: the parts' sum, or the
// first part where that is infinite (0 parts of a weight times an infinite V entry are NaN, and no part
// of it). All reads are issued before any is used (the empty asm keeps the compiler from placing the
// other parts' behind a branch on the first).
template <int D, int G, int NP>
__device__ __forceinline__ void merged_acc(float (&x)[NWAVE], const MergeLds<D, G, NP>& L, int g, int d) {
  float part[NP][NWAVE];
#pragma unroll
  for (int w = 0; w < NWAVE; ++w)
#pragma unroll
    for (int n = 0; n < NP; ++n) part[n][w] = L.acc[((w * NP + n) * G + g) * D + d];
#pragma unroll
  for (int w = 0; w < NWAVE; ++w) {
    if constexpr (NP == 1) {
      x[w] = part[0][w];
    } else {
      float sum = part[0][w] + (NP == 3 ? part[1][w] + part[NP - 1][w] : part[1][w]);
      asm("" : "+v"(sum));
      x[w] = __builtin_isinf(part[0][w]) ? part[0][w] : sum;
    }
  }
}

// Workgroup epilogue, after the wavefronts have put their states into L (m, l in log2 units, acc
// un-normalised): merge them, then write out/out_f32/lse (one split) or the split partials.
template <int D, int G, bool LOAD_V, int NP>
__device__ __forceinline__ void finish_merge(const AttnP& p, int b, int h, int split, const MergeLds<D, G, NP>& L,
                                             bool plain) {
  const int tid = threadIdx.x;
  __syncthreads();
  const int S = p.num_splits;
  const int64_t hq0 = static_cast<int64_t>(b) * p.Hq + static_cast<int64_t>(h) * G;
  if constexpr (LOAD_V) {
    for (int o = tid; o < G * D; o += NT) {
      const int g = o / D, d = o % D;
      float A = 0.f, Ls = 0.f, x[NWAVE];
      merged_acc(x, L, g, d);
      if (plain) {
#pragma unroll
        for (int w = 0; w < NWAVE; ++w) A += x[w];
        Ls = 1.f;
      } else {
        float M = NEG_INF;
#pragma unroll
        for (int w = 0; w < NWAVE; ++w) M = fmaxf(M, L.ml[(w * G + g) * 2]);
        const float mu = M == NEG_INF ? 0.f : M;
#pragma unroll
        for (int w = 0; w < NWAVE; ++w) {
          const float f = fexp2(L.ml[(w * G + g) * 2] - mu);
          Ls += L.ml[(w * G + g) * 2 + 1] * f;
          A += x[w] * f;
        }
      }
      const int64_t hq = hq0 + g;
      if (S == 1) {
        const float o_ = Ls > 0.f ? A / Ls : 0.f;
        p.out[hq * D + d] = f2bf(o_);
        if (p.out_f32) p.out_f32[hq * D + d] = o_;
      } else {
        p.part_acc[(hq * S + split) * D + d] = A;
      }
    }
  }
  if (!plain && tid < G) {
    const int g = tid;
    float M = NEG_INF, Ls = 0.f;
#pragma unroll
    for (int w = 0; w < NWAVE; ++w) M = fmaxf(M, L.ml[(w * G + g) * 2]);
    const float mu = M == NEG_INF ? 0.f : M;
#pragma unroll
    for (int w = 0; w < NWAVE; ++w) Ls += L.ml[(w * G + g) * 2 + 1] * fexp2(L.ml[(w * G + g) * 2] - mu);
    const int64_t hq = hq0 + g;
    if (S == 1) {
      if (p.lse) p.lse[hq] = Ls > 0.f ? (M + flog2(Ls)) * LN2 : NEG_INF;
    } else {
      p.part_ml[(hq * S + split) * 2] = M;
      p.part_ml[(hq * S + split) * 2 + 1] = Ls;
    }
  }
}

// The VALU engine's wavefront state into L (acc[g][8]: every lane's rows), then the merge.
template <int D, int G, bool LOAD_V>
__device__ __forceinline__ void finish(const AttnP& p, float (&m)[G], float (&l)[G], float (&acc)[G][8], int b,
                                       int h, int split, MergeLds<D, G, LOAD_V ? 1 : 0>& L, bool plain) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  constexpr int VLPR = Lay<D>::VLPR;
  if constexpr (LOAD_V) {
    reduce_acc_rows<D, G>(acc);
    if (lane < VLPR) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) L.acc[(wave * G + g) * D + 8 * lane + e] = acc[g][e];
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      L.ml[(wave * G + g) * 2] = m[g];
      L.ml[(wave * G + g) * 2 + 1] = l[g];
    }
  }
  finish_merge<D, G, LOAD_V>(p, b, h, split, L, plain);
}

template <int D, int G>
__device__ __forceinline__ void load_q(u32x4 (&qv)[G][Lay<D>::KC], const AttnP& p, int b, int h, int lane) {
  const int sub = lane & 7;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint16_t* qp = p.q + b * p.q_sb + (static_cast<int64_t>(h) * G + g) * p.q_sh + 8 * sub;
#pragma unroll
    for (int c = 0; c < Lay<D>::KC; ++c) qv[g][c] = ld16(qp + 64 * c);
  }
}

// One block's softmax step for head g: updates (m, l), returns alpha (rescale of acc) and the
// factor c with p = e * c; e = 2^(s - mt) and the block stats (mt, st) are left for the caller.
template <int G>
__device__ __forceinline__ void block_softmax(const float (&s)[8][G], int g, float& m, float& l, float (&e)[8],
                                              float& mt, float& st, float& alpha, float& c) {
  float x = s[0][g];
#pragma unroll
  for (int rg = 1; rg < 8; ++rg) x = fmaxf(x, s[rg][g]);
  mt = max_rows8(x);
  const float mtu = mt == NEG_INF ? 0.f : mt;
  float sum = 0.f;
#pragma unroll
  for (int rg = 0; rg < 8; ++rg) {
    e[rg] = fexp2(s[rg][g] - mtu);
    sum += e[rg];
  }
  st = sum_rows8(sum);
  const float m_new = fmaxf(m, mt);
  const float mu = m_new == NEG_INF ? 0.f : m_new;
  alpha = fexp2(m - mu);
  c = mt == NEG_INF ? 0.f : fexp2(mt - mu);
  l = l * alpha + st * c;
  m = m_new;
}


// ---------------------------------------------------------------- MFMA engine
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <int D>
struct MLay {
  static constexpr int KS = D / 32;   // 32-dim k-steps of v_mfma_f32_16x16x32_bf16
  static constexpr int VD = D / 16;   // output dims per column of a P V product
  static constexpr int VN = BLK * D / (WAVE * 8);  // 16-byte V loads per lane and block
};

// Token of score s[nt][i] on a lane with j4 = lane / 16: four consecutive tokens per lane (fp16 P is
// written and read in 8-byte pieces).
__device__ __forceinline__ int mf_tok(int nt, int i, int j4) { return 16 * nt + 4 * j4 + i; }

// K reaches the A operand's layout (16 rows x 64 bytes per k-step) in one of two ways.
//   staged  loaded in whole rows (an instruction covers 512 / D rows of 2 D bytes) and passed through LDS, a
//           16-token tile at a time. A tile is held as rows of D / 8 16-byte chunks, chunk c of row r at
//           c ^ r (D 64: c ^ (r / 2)): a write fills whole rows and a read takes 16 different chunk places,
//           so neither conflicts. Two tiles per wavefront.
//   direct  loaded in the operand's layout: every instruction takes half lines of 16 rows.
// Staged, a pass over K alone runs at 5.8 TB/s against 4.7 (B 8 at 32k 115.2 -> 94.0 us per op; D 64, 16 x 20k
// 84.1 -> 70.1) and a short pass with V ends sooner (B 1 at 32k, 4 blocks per wavefront, 25.3 -> 24.0; 7 heads
// 6 x 9k 25.7 -> 24.4; masked at 32k 15.1 -> 14.1). In a long pass with V, where both streams are in flight all
// the time, the two ways of reading K and V at once move more: B 8 at 32k (32 blocks per wavefront) 159.3
// staged, 155.0 direct; B 32 at 64k (256) 1249 and 1221; at 20 blocks per wavefront 101.7 and 102.6. So a
// wavefront of a pass with V takes K direct from LONG_BLOCKS items on.
template <int D>
struct KStage {
  static constexpr int TILE = 16 * 2 * D, TILES = 2, WAVE_BYTES = TILES * TILE, BYTES = NWAVE * WAVE_BYTES;
};
// Byte offset of this lane's row and chunk in a K load.
template <int D, bool STAGED>
__device__ __forceinline__ uint32_t mf_koff(int lane, int64_t k_st) {
  return STAGED ? static_cast<uint32_t>((lane / (D / 8)) * k_st * 2 + 16 * (lane % (D / 8)))
                : static_cast<uint32_t>((lane & 15) * k_st * 2 + 16 * (lane >> 4));
}
// Byte offsets in a tile of this lane's part of load 0 (load kk: ^ 64 kk, + 1024 kk) and of its chunk of
// k-step 0 (k-step kk: ^ 64 kk).
template <int D>
__device__ __forceinline__ uint32_t k_stage_w(int lane) {
  const int r = lane / (D / 8), c = lane % (D / 8);
  return static_cast<uint32_t>(r * 2 * D + 16 * (c ^ (D == 128 ? r : r >> 1)));
}
template <int D>
__device__ __forceinline__ uint32_t k_stage_r(int lane) {
  const int m = lane & 15, j4 = lane >> 4;
  return static_cast<uint32_t>(m * 2 * D + 16 * (j4 ^ (D == 128 ? m : m >> 1)));
}

// V loads are 16 bytes (8 dims) per lane. D 128: a 16-lane group loads one row, load 4 nt + i the rows
// mf_tok(nt, i, lane / 16), and column c holds dims 8 c .. + 7. D 64: a group loads two rows, load
// 2 nt + i the tokens mf_tok(nt, 2 i, lane / 16) (lanes c < 8) and mf_tok(nt, 2 i + 1, ..) (c >= 8);
// the lanes c and c ^ 8 then exchange halves (v_rows), so that column c holds four dims of both rows:
// 8 (c % 8) .. + 3, or + 4 .. + 7 for c >= 8. (8-byte loads of one row per group instead: B 16 at 20k,
// 106 -> 109 us per op.)
template <int D>
__device__ __forceinline__ uint32_t mf_voff(int lane, int64_t v_st) {
  const int j4 = lane >> 4, c = lane & 15;
  return D == 128 ? static_cast<uint32_t>(4 * j4 * v_st * 2 + 16 * c)
                  : static_cast<uint32_t>((4 * j4 + (c >> 3)) * v_st * 2 + 16 * (c & 7));
}
// First output dim of column c; its VD dims follow.
template <int D>
__device__ __forceinline__ int mf_vdim(int c) {
  return D == 128 ? 8 * c : 8 * (c & 7) + 4 * (c >> 3);
}

// Reductions over the four lanes that hold one head's other tokens (lane ^ 16, ^ 32).
__device__ __forceinline__ float swap_max(float v) {
  const uint32_t a = __float_as_uint(v);
  const u32x2 r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const uint32_t m = __float_as_uint(fmaxf(__uint_as_float(r.x), __uint_as_float(r.y)));
  const u32x2 t = __builtin_amdgcn_permlane16_swap(m, m, false, false);
  return fmaxf(__uint_as_float(t.x), __uint_as_float(t.y));
}
__device__ __forceinline__ float swap_sum(float v) {
  const uint32_t a = __float_as_uint(v);
  const u32x2 r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const uint32_t m = __float_as_uint(__uint_as_float(r.x) + __uint_as_float(r.y));
  const u32x2 t = __builtin_amdgcn_permlane16_swap(m, m, false, false);
  return __uint_as_float(t.x) + __uint_as_float(t.y);
}

// K of one 64-token block: kr[nt][kk] = this lane's row and chunk (mf_koff) of load kk of tile nt: staged, of
// rows (512 / D) kk ..; direct, of chunks 4 kk ...
template <int D, bool STAGED = true>
__device__ __forceinline__ void load_k_block_mf(u32x4 (&kr)[4][MLay<D>::KS], rsrc_t rk, uint32_t koffm,
                                                int64_t k_st, int t0) {
  const uint32_t rowb = static_cast<uint32_t>(k_st * 2);
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int kk = 0; kk < MLay<D>::KS; ++kk)
      kr[nt][kk] = STAGED ? bload16<BUF_NT>(rk, koffm, static_cast<uint32_t>(t0 + 16 * nt + (512 / D) * kk) * rowb)
                          : bload16<BUF_NT>(rk, koffm + 64 * kk, static_cast<uint32_t>(t0 + 16 * nt) * rowb);
}

// Sum over the rows of a block loaded staged (load_k_block_mf), for this lane's 8 dims 8 (lane % (D / 8)): pairs
// of rows by v_perm, added by v_dot2_f32_bf16 against ones (exact products, fp32 sums), then over the lanes that
// hold the chunk's other rows. About 210 instructions per block beside a stream that waits for memory.
// Measured (first step of a layer, us, pass + sums apart -> together): 32 x 40k, 32 / 8 heads, 776 + 491 -> 914;
// 16 ragged sequences to 64k, 28 / 4 heads, 134 + 102 -> 155.
template <int D>
__device__ __forceinline__ void block_key_sums(const u32x4 (&kr)[4][MLay<D>::KS], float (&sum)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = 0.f;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int kk = 0; kk < MLay<D>::KS; kk += 2)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t a = kr[nt][kk][d], c = kr[nt][kk + 1][d];
        sum[2 * d] = dot2(__builtin_amdgcn_perm(c, a, 0x05040100u), 0x3f803f80u, sum[2 * d]);
        sum[2 * d + 1] = dot2(__builtin_amdgcn_perm(c, a, 0x07060302u), 0x3f803f80u, sum[2 * d + 1]);
      }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if constexpr (D == 64) sum[e] += dpp<DPP_ROR8>(sum[e]);
    sum[e] = swap_sum(sum[e]);
  }
}

// V of one 64-token block. voffm = mf_voff.
template <int D>
__device__ __forceinline__ void load_v_block_mf(u32x4 (&vr)[MLay<D>::VN], rsrc_t rv, uint32_t voffm, int64_t v_st,
                                                int t0) {
  const uint32_t rowb = static_cast<uint32_t>(v_st * 2);
#pragma unroll
  for (int r = 0; r < MLay<D>::VN; ++r) {
    const int t = D == 128 ? mf_tok(r / 4, r % 4, 0) : mf_tok(r / 2, 2 * (r % 2), 0);
    vr[r] = bload16<BUF_NT>(rv, voffm, static_cast<uint32_t>(t0 + t) * rowb);
  }
}

// Dwords d (dims 2 d, 2 d + 1 of this lane's column) of tokens (nt, i) and (nt, i + 1), i even.
template <int D>
__device__ __forceinline__ void v_pair(const u32x4 (&vr)[MLay<D>::VN], int nt, int i, int d, bool up, uint32_t& a,
                                       uint32_t& c) {
  if constexpr (D == 128) {
    a = vr[4 * nt + i][d];
    c = vr[4 * nt + i + 1][d];
  } else {  // up: lanes c >= 8, which loaded the second token's row
    const u32x4 x = vr[2 * nt + i / 2];
    const uint32_t other = dppu<DPP_ROR8>(up ? x[d] : x[2 + d]);
    a = up ? other : x[d];
    c = up ? x[2 + d] : other;
  }
}

// B operand (Q^T): lane (j = lane / 16, c = lane % 16) holds head c % gpad's dims of chunk 4 kk + j
// (zero past G): every group of gpad columns repeats the group's heads.
template <int D, int G>
__device__ __forceinline__ void load_q_mf(u32x4 (&qb)[MLay<D>::KS], const AttnP& p, int b, int h, int lane) {
  const int c = (lane & 15) % gpad<G>(), j = lane >> 4;
  const uint16_t* qp = p.q + b * p.q_sb + (static_cast<int64_t>(h) * G + c) * p.q_sh + 8 * j;
#pragma unroll
  for (int kk = 0; kk < MLay<D>::KS; ++kk) qb[kk] = c < G ? ld16(qp + 32 * kk) : u32x4{0u, 0u, 0u, 0u};
}

// Scores of one block in log2 units: s[nt][i] = head (lane % 16) % gpad, token t0 + mf_tok(nt, i,
// lane / 16); tokens >= t_lim masked to -inf (only the block that t_lim cuts tests them). sK: this
// wavefront's KStage. A wavefront's LDS accesses complete in order, so a tile needs no wait between its
// writes, its reads and the next tile's writes; the fences keep the compiler's order.
template <int D, bool STAGED = true>
__device__ __forceinline__ void qk_block_mf(float (&s)[4][4], const u32x4 (&kr)[4][MLay<D>::KS],
                                            const u32x4 (&qb)[MLay<D>::KS], char* sK, float scale_log2, int t0,
                                            int t_lim, int lane) {
  constexpr int KS = MLay<D>::KS;
  const uint32_t w0 = k_stage_w<D>(lane), r0 = k_stage_r<D>(lane);
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    char* tile = sK + (nt % KStage<D>::TILES) * KStage<D>::TILE;
    if constexpr (STAGED) {
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        *reinterpret_cast<u32x4*>(tile + 1024 * kk + (w0 ^ (64u * kk))) = kr[nt][kk];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const u32x4 k = STAGED ? *reinterpret_cast<const u32x4*>(tile + (r0 ^ (64u * kk))) : kr[nt][kk];
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, k), __builtin_bit_cast(bf16x8_t, qb[kk]),
                                                  a, 0, 0, 0);
    }
    if constexpr (STAGED) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 4; ++i) s[nt][i] = a[i] * scale_log2;
  }
  if (t0 + BLK > t_lim) {  // uniform
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (t0 + mf_tok(nt, i, lane >> 4) >= t_lim) s[nt][i] = NEG_INF;
  }
}

// One block's maximum of a lane's head.
__device__ __forceinline__ float block_max_mf(const float (&s)[4][4]) {
  float x = s[0][0];
#pragma unroll
  for (int t = 1; t < 16; ++t) x = fmaxf(x, s[t / 4][t % 4]);
  return swap_max(x);
}

// e = 2^(s - mt) (mt the block's maximum; 0 where it is -inf) and their sum over the block.
__device__ __forceinline__ float block_exp_mf(float (&e)[4][4], const float (&s)[4][4], float mt) {
  const float mtu = mt == NEG_INF ? 0.f : mt;
  float r[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) e[nt][i] = fexp2(s[nt][i] - mtu);
    r[nt] = (e[nt][0] + e[nt][1]) + (e[nt][2] + e[nt][3]);
  }
  return swap_sum((r[0] + r[1]) + (r[2] + r[3]));
}

// Weights of one block as A operands of P V: k-step s covers tiles 2 s and 2 s + 1, element e of lane
// (c, j4) is the weight of s[2 s + e / 4][e % 4]. Row c is part c / gpad of head c % gpad, and the sum of
// a head's rows is its result; the parts are bf16 and sum to the fp32 weight (or to the product it was
// rounded from, where the compiler contracts).
//   4-head groups   one product, parts (hi, mid, lo, 0): the weight's top 8 significant bits, the next 8
//                   and the rest, each by truncation.
//   8-head groups   two products into the same accumulators, parts (hi / 2, mid) then (hi / 2, lo).
// An infinite V entry times a part that is 0 is NaN. Part 0 is hi alone, and merged_acc takes part 0 alone
// where it is infinite, so the infinity of an fp32 product comes out for every weight whose hi (8-head
// groups: hi / 2) is a bf16 other than 0: any |weight| >= 2^-125, whether or not the unit keeps bf16
// denormals (weights below 2^-126 only arise as products of a token's and its block's factors). The lo / 2
// in both parts that this replaced was 0 from about 2^-109 on.
// Measured against P through LDS and P V as fp32 FMAs (G x 128 per lane and block at D 128, and 128
// conversions; op, us, graph-replayed): B 1 at 32k 26.6 -> 25.9 dense, 16.3 -> 14.9 masked with statistics
// (35% listed); 7 heads, B 6 at 9k, 27.6 -> 24.7; 8 heads, B 4 at 16k, 48.6 -> 45.8; D 64 at 4k 8.7 -> 7.6;
// B 8 at 32k 156.6 -> 155.0. The loads bound all of these; what went is arithmetic that nothing covered.
template <int G>
struct PFrag {
  static constexpr int NX = gpad<G>() == 8 ? 2 : 1;  // products per k-step
  static constexpr int NP = gpad<G>() == 8 ? 2 : 3;  // parts (row groups) of a result
  u32x4 x[NX][2];
};

// Two values' high halves (bf16 by truncation), the first in the low half.
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}
constexpr uint32_t BF_HI = 0xffff0000u;

// The lane's column gives weight 0 where this is false (the unused fourth part of 4-head groups).
template <int G>
__device__ __forceinline__ bool part_used(int lane) {
  return gpad<G>() == 8 || (lane & 15) < 12;
}

template <int G>
__device__ __forceinline__ PFrag<G> make_frag(const float (&w)[4][4], int lane) {
  PFrag<G> f;
  const int part = (lane & 15) / gpad<G>();
  const uint32_t m1 = part >= 1 ? BF_HI : 0u, m2 = part >= 2 ? BF_HI : 0u;
  const float half = part == 0 ? 0.5f : 1.f;  // 8-head groups
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t v[2], lo[2];
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        const float a = w[2 * s + u / 2][2 * (u % 2) + o];
        const float r = a - __uint_as_float(__float_as_uint(a) & m1);  // part 0: the weight itself
        if constexpr (gpad<G>() == 8) {
          v[o] = __float_as_uint(half * r);
          lo[o] = __float_as_uint(half * r - __uint_as_float(v[o] & m1));
        } else {
          v[o] = __float_as_uint(r - __uint_as_float(__float_as_uint(r) & m2));
        }
      }
      f.x[0][s][u] = pack_hi(v[0], v[1]);
      if constexpr (gpad<G>() == 8) f.x[PFrag<G>::NX - 1][s][u] = pack_hi(lo[0], lo[1]);
    }
  return f;
}

// Accumulators of P V: a[j] on lane (c, j4) holds rows 4 j4 + i (part and head as PFrag's rows) of dim
// mf_vdim(c) + j.
template <int D, int G>
struct PVAcc {
  f32x4_t a[MLay<D>::VD];
};

template <int D, int G>
__device__ __forceinline__ void zero_acc(PVAcc<D, G>& acc) {
#pragma unroll
  for (int j = 0; j < MLay<D>::VD; ++j) acc.a[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// acc *= alpha of each row's head (alpha: this lane's head's; row r of a lane's accumulators is head
// r % gpad, found on lane r % gpad of every 16-lane row).
template <int D, int G>
__device__ __forceinline__ void rescale_acc(PVAcc<D, G>& acc, float alpha, int lane) {
  float al[4];
  al[0] = dpp<0x150>(alpha);  // row_newbcast
  al[1] = dpp<0x151>(alpha);
  al[2] = dpp<0x152>(alpha);
  al[3] = dpp<0x153>(alpha);
  if constexpr (gpad<G>() == 8) {
    const bool up = (lane & 16) != 0;  // rows 4 .. 7 of an 8-row part
    al[0] = up ? dpp<0x154>(alpha) : al[0];
    al[1] = up ? dpp<0x155>(alpha) : al[1];
    al[2] = up ? dpp<0x156>(alpha) : al[2];
    al[3] = up ? dpp<0x157>(alpha) : al[3];
  }
#pragma unroll
  for (int j = 0; j < MLay<D>::VD; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc.a[j][i] *= al[i];
}

// acc += P V of one block.
template <int D, int G>
__device__ __forceinline__ void pv_block_mf(PVAcc<D, G>& acc, const u32x4 (&vr)[MLay<D>::VN], const PFrag<G>& f,
                                            int lane) {
  const bool up = (lane & 8) != 0;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < MLay<D>::VD / 2; ++d) {
      u32x4 lo, hi;  // dims 2 d and 2 d + 1 of this lane's: tokens in pairs
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint32_t a, c;
        v_pair<D>(vr, 2 * s + u / 2, 2 * (u % 2), d, up, a, c);
        lo[u] = __builtin_amdgcn_perm(c, a, 0x05040100u);
        hi[u] = __builtin_amdgcn_perm(c, a, 0x07060302u);
      }
#pragma unroll
      for (int n = 0; n < PFrag<G>::NX; ++n) {
        const bf16x8_t w = __builtin_bit_cast(bf16x8_t, f.x[n][s]);
        acc.a[2 * d] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8_t, lo), acc.a[2 * d], 0, 0, 0);
        acc.a[2 * d + 1] =
            __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(bf16x8_t, hi), acc.a[2 * d + 1], 0, 0, 0);
      }
    }
}

// LDS of an MFMA pass: the wavefronts' K tiles, then (after a barrier) the epilogue's states.
template <int D, int G, bool LOAD_V>
union MfLds {
  char k[KStage<D>::BYTES];
  MergeLds<D, G, LOAD_V ? PFrag<G>::NP : 0> merge;
};

// The MFMA engine's wavefront state into the epilogue's LDS (m, l: this lane's head's), then the merge.
template <int D, int G, bool LOAD_V>
__device__ __forceinline__ void finish_mf(const AttnP& p, float m, float l, const PVAcc<D, G>& acc, int b, int h,
                                          int split, MfLds<D, G, LOAD_V>& lds, bool plain) {
  auto& L = lds.merge;
  __syncthreads();  // every wavefront has left its K tiles
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int j4 = lane >> 4, c16 = lane & 15;
  if constexpr (LOAD_V) {
    constexpr int VD = MLay<D>::VD, GP = gpad<G>(), NP = PFrag<G>::NP;
    const int part = 4 * j4 / GP;  // rows 4 j4 .. + 3
    if (part < NP) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int g = (4 * j4) % GP + i;
        if (g < G) {
          float* a = L.acc + ((wave * NP + part) * G + g) * D + mf_vdim<D>(c16);
#pragma unroll
          for (int j = 0; j < VD; j += 4)
            *reinterpret_cast<float4*>(a + j) =
                make_float4(acc.a[j][i], acc.a[j + 1][i], acc.a[j + 2][i], acc.a[j + 3][i]);
        }
      }
    }
  }
  if (lane < G) {
    L.ml[(wave * G + lane) * 2] = m;
    L.ml[(wave * G + lane) * 2 + 1] = l;
  }
  finish_merge<D, G, LOAD_V>(p, b, h, split, L, plain);
}

// Split merge: workgroup (b*Hq + hq, 32-dim slice), 256 threads = 8 split classes x 32 dims.
// Thread (cls, d) loads the partials of splits s = cls + 8 u, u < U (U = ceil(S / 8), a template
// parameter so every load is unconditional, clamped to S - 1, and in flight together), the
// classes agree on the max through LDS, then weight (2^(m_s - M), log-sum-exp mode; 1, plain
// mode for the two-pass pass 2) and add in LDS. WITH_V = false (stats-only): only lse.
// Body of one merge workgroup (query head hq, dims [32 slice, 32 slice + 32)) over its Sv <= 8 U
// partials. A workgroup wider than 256 threads (the fused merge + update launch) runs it with its
// first 256; the others only pass the barriers.
template <int D, int U, bool WITH_V>
__device__ __forceinline__ void merge_body(const AttnP& p, int plain, int64_t hq, int slice, int Sv) {
  constexpr int NC = 8;
  const int tid = threadIdx.x, cls = (tid / 32) % NC, dl = tid % 32;
  const bool act = tid < 256;
  const int d = slice * 32 + dl;
  const int S = p.num_splits;
  const float* ml = p.part_ml + hq * S * 2;
  __shared__ float rA[NC][32], rL[NC], rM[NC];
  float ms[U], ls[U], as[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int s = max(min(cls + NC * u, Sv - 1), 0);
    const float2 t = *reinterpret_cast<const float2*>(ml + 2 * s);
    ms[u] = t.x;
    ls[u] = t.y;
    if constexpr (WITH_V) as[u] = p.part_acc[(hq * S + s) * D + d];
  }
  float mloc = NEG_INF;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (cls + NC * u < Sv) mloc = fmaxf(mloc, ms[u]);
  if (act && dl == 0) rM[cls] = mloc;
  __syncthreads();
  float M = NEG_INF;
#pragma unroll
  for (int c = 0; c < NC; ++c) M = fmaxf(M, rM[c]);
  const float mu = M == NEG_INF ? 0.f : M;
  float A = 0.f, L = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (cls + NC * u < Sv && (plain || ls[u] > 0.f)) {  // an empty partial (l = 0) adds nothing
      const float w = plain ? 1.f : fexp2(ms[u] - mu);
      L += ls[u] * w;
      if constexpr (WITH_V) A += as[u] * w;
    }
  }
  if (act) rA[cls][dl] = A;
  if (act && dl == 0) rL[cls] = L;
  __syncthreads();
  if (tid < 32) {
    float a = 0.f, l = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      a += rA[c][tid];
      l += rL[c];
    }
    if (plain) l = 1.f;
    if constexpr (WITH_V) {
      const float o = l > 0.f ? a / l : 0.f;
      p.out[hq * D + d] = f2bf(o);
      if (p.out_f32) p.out_f32[hq * D + d] = o;
    }
    if (!plain && tid == 0 && slice == 0 && p.lse) p.lse[hq] = l > 0.f ? (M + flog2(l)) * LN2 : NEG_INF;
  }
}

// Partials of query head hq: S, or in a ragged batch its (sequence, KV head)'s chunk count (0:
// nothing attended, out 0 and lse -inf). Uniform over the workgroup.
__device__ __forceinline__ int merge_count(const AttnP& p, int64_t hq) {
  if (p.seq_lens == nullptr) return p.num_splits;
  const int b = static_cast<int>(hq / p.Hq), h = static_cast<int>(hq % p.Hq) / (p.Hq / p.Hkv);
  if (p.block_idx != nullptr && p.list_partition != 0) {
    int nv[NRG];
    const int C = global_chunk_len(p, nv);
    return (ragged_items(p, b, h, true) + C - 1) / C;
  }
  return ragged_chunks(p, b, h, p.block_idx != nullptr);
}

// merge_body with the fewest slots that hold Sv partials (U halved while 4 U still does): a ragged
// head with few chunks issues no loads for slots it does not have (at S = 128 most heads have a
// handful of chunks). Sv is uniform, so the choice is a uniform branch.
template <int D, int U, bool WITH_V>
__device__ void merge_fit(const AttnP& p, int plain, int64_t hq, int slice, int Sv) {
  if constexpr (U > 1) {
    if (Sv <= 8 * (U / 2)) {
      merge_fit<D, U / 2, WITH_V>(p, plain, hq, slice, Sv);
      return;
    }
  }
  merge_body<D, U, WITH_V>(p, plain, hq, slice, Sv);
}

// Workgroup (x, y) of the (B Hq, D / 32) grid takes item xcd_remap(x + y B Hq) in (query head, dim
// slice) order, so a KV head's merges run on the XCD that ran its splits (work_coords' mapping),
// whose L2 still holds the partials just written (config 2's op 26.87 -> 26.52 us).
template <int D, int U, bool WITH_V>
__global__ void __launch_bounds__(256) combine_kernel(const AttnP p, int plain) {
  const int nsl = gridDim.y;
  const int m = xcd_remap(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * nsl);
  const int64_t hq = m / nsl;
  merge_fit<D, U, WITH_V>(p, plain, hq, m % nsl, merge_count(p, hq));
}

// merge_body with U chosen at run time from the head's partial count.
template <int D>
__device__ void merge_body_rt(const AttnP& p, int64_t hq, int slice) {
  merge_fit<D, MAX_SPLITS / 8, true>(p, 0, hq, slice, merge_count(p, hq));
}

template <int D, bool WITH_V>
inline void launch_combine_u(const AttnP& p, dim3 grid, int plain, hipStream_t s) {
  const int u = (p.num_splits + 7) / 8;
  if (u <= 1) hipLaunchKernelGGL((combine_kernel<D, 1, WITH_V>), grid, dim3(256), 0, s, p, plain);
  else if (u <= 2) hipLaunchKernelGGL((combine_kernel<D, 2, WITH_V>), grid, dim3(256), 0, s, p, plain);
  else if (u <= 4) hipLaunchKernelGGL((combine_kernel<D, 4, WITH_V>), grid, dim3(256), 0, s, p, plain);
  else if (u <= 8) hipLaunchKernelGGL((combine_kernel<D, 8, WITH_V>), grid, dim3(256), 0, s, p, plain);
  else if (u <= 16) hipLaunchKernelGGL((combine_kernel<D, 16, WITH_V>), grid, dim3(256), 0, s, p, plain);
  else hipLaunchKernelGGL((combine_kernel<D, MAX_SPLITS / 8, WITH_V>), grid, dim3(256), 0, s, p, plain);
}

inline hipError_t launch_combine(const AttnP& p, int D, bool plain, hipStream_t s) {
  const bool with_v = p.out != nullptr;
  const dim3 grid(p.B * p.Hq, with_v ? D / 32 : 1);
  const int pl = plain ? 1 : 0;
  if (D == 128) {
    if (with_v) launch_combine_u<128, true>(p, grid, pl, s);
    else launch_combine_u<128, false>(p, grid, pl, s);
  } else {
    if (with_v) launch_combine_u<64, true>(p, grid, pl, s);
    else launch_combine_u<64, false>(p, grid, pl, s);
  }
  return hipGetLastError();
}

// Ragged: S + B chunk slots per KV head (a head has at most that many chunks).
inline dim3 attn_grid(const AttnP& p) {
  return dim3(p.seq_lens != nullptr ? (p.num_splits + p.B) * p.Hkv : p.num_splits * p.Hkv * p.B);
}

// Instantiated group sizes.
#define KVS_FOR_G(X, D) \
  X(D, 1)               \
  X(D, 2)               \
  X(D, 4)               \
  X(D, 7)               \
  X(D, 8)

}  // namespace
}  // namespace kvs
