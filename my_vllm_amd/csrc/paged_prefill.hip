// C-ABI entry points of the ragged causal prefill kernel and of the MIXED
// kernels (prefill tiles + decode items in one grid).
#include "mva_capi.h"
#include "paged_prefill.h"
#include "paged_prefill_pingpong.h"

#include <algorithm>
#include <cmath>
#include <exception>
#include <functional>
#include <vector>

namespace mva {

int fill_decode_params(DecodeParams& p, const void* q, int64_t q_token_stride, int64_t q_head_stride,
                       const void* k_cache, const void* v_cache, int64_t num_pages, int64_t page_stride,
                       int64_t token_stride, const int32_t* block_tables, int64_t block_table_stride,
                       const int32_t* seq_lens, const int32_t* items, int64_t num_items, int64_t num_waves,
                       const int32_t* wave_extra, const int32_t* merges, int64_t num_merges, int64_t num_part_slots, void* out,
                       int64_t out_token_stride,
                       int64_t out_head_stride, void* workspace, int64_t workspace_bytes,
                       int num_q_heads, int num_kv_heads, int head_dim, int page_size,
                       float softmax_scale);
int32_t* decode_arrival_counters(void* workspace);
int launch_decode_merge(const DecodeParams& p, const int32_t* merges, int64_t num_merges, int64_t num_part_slots,
                        int dtype, hipStream_t stream);

namespace {

// Decode wavefronts in a workgroup of paged_mixed_split_cus_kernel.
constexpr int kMixedDecodeWaves = kPrefillPPThreads / 64;

// Piece list and arrival counters, before the partials, in words.
constexpr int64_t kPrefillSplitMetaInts = kPrefillMaxItems * kPrefillPieceInts + kPrefillPieceSlots;
static_assert(kPrefillSplitMetaInts * 4 % kPrefillPartUnit == 0, "partials stay aligned");
// Word offset of the piece list of a plan of at most max_tiles tiles, and the
// bytes of such a plan with its split-K area.
int64_t prefill_piece_list(int64_t max_tiles) {
  const int64_t unit = kPrefillPartUnit / 4;
  return (kPrefillPlanHeaderInts + max_tiles * kPrefillPlanItemInts + unit - 1) / unit * unit;
}
int64_t prefill_plan_bytes(int64_t max_tiles) {
  return (kPrefillPlanHeaderInts + max_tiles * kPrefillPlanItemInts) * 4;
}
int64_t prefill_split_bytes(int64_t max_tiles) {
  return (prefill_piece_list(max_tiles) + kPrefillSplitMetaInts) * 4 + (int64_t)kPrefillPieceSlots * kPrefillPartBytes;
}

// Cuts the n planned tiles into split-K pieces where whole tiles would leave
// workgroups idle; returns the number of items of the piece list (whole tiles
// among them), or 0 when whole tiles are as good.  Tiles from number `start`
// on that have more than L key tiles (64 keys, 1.5 to 1.85 us) are cut into
// near-equal pieces of at most L; of 16 candidates the one with the lowest
// estimate, in key tiles, is taken:
//  * fixed (one item per workgroup; start 0, L = ceil(longest / k), k = 1 .. 8):
//    L and, for a split, 2.5 + 0.75 k (writing the partials and one workgroup
//    reading k of them: 4.7 and 5.3 us at k = 4 with all 256 workgroups busy);
//  * claimed items, longest first.  An item costs 2.5 besides its keys, a
//    split tile 3 and each of its pieces 2.75.  Long tiles cut (start 0, L =
//    longest / (1 + c / 2), c = 0 .. 7): the largest of the work per workgroup
//    and j + 1 times the length that more than j * per_head items have (whole
//    tiles: exactly, otherwise of 3/4 and 1/2 of L).  Or the tiles past one or two whole rounds cut (start = per_head or twice
//    that, where all tiles are sorted): the largest of the whole rounds and
//    the work per workgroup and half a piece.  Plus 5, and a gain under a tenth
//    is left.
// Measured, whole and claimed / cut and in turns: 32 / 8 heads, a prompt of 2048
// tokens (32 tiles of 1 to 32 for 32 workgroups a head) 59.6 / 52.8 us, 4
// chunks of 512 over up to 8k 172 / 124, 4 of 560 over 4k 233 / 187; 64 / 8
// heads, 4 of 280 over 7k 362 / 259; 16 / 8 heads, 6000 tokens 202 / 161.
// All 1024 threads call it; nt, first, best and len are LDS arrays of at least
// kPrefillMaxItems, 2 * kPrefillCutTiles + 2, 64 and kPrefillMaxItems ints.
// piece_list <= 0: no room for partials.  The first `sorted` tiles or fewer
// are longest first.
__device__ int plan_pieces(int32_t* __restrict__ plan, int n, bool fixed, int per_head, int num_kv_heads,
                           const int32_t* __restrict__ block_tables, int64_t bt_stride, int64_t num_pages,
                           int piece_list, int sorted, int* nt, int* first, int* best, int* len_of) {
  const int tid = threadIdx.x;
  const int slots = kPrefillPieceSlots / num_kv_heads;
  if (piece_list <= 0 || n == 0 || n > (fixed ? min(per_head, slots) : kPrefillCutTiles)) return 0;
  const int32_t* tiles = plan + kPrefillPlanHeaderInts;
  __syncthreads();
  if (tid < n) nt[tid] = tiles[tid * kPrefillPlanItemInts + 5];
  __syncthreads();
  // Wave c prices candidate c.
  const int lane = tid & 63, c = tid >> 6;
  auto wave_sum = [](int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
  };
  int longest = 0;
  for (int i = lane; i < n; i += 64) longest = max(longest, nt[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off));
  const int k = c + 1;
  // Claimed items: candidates 0 .. 7 cut long tiles, 8 .. 15 the tiles past
  // one (8 .. 11) or two (12 .. 15) rounds into 2, 4, 6 or 8.
  const bool late = !fixed && c >= 8;
  const int start = late ? per_head * (1 + ((c - 8) >> 2)) : 0;
  int len = fixed ? (longest + k - 1) / k : (2 * longest + 1 + c) / (2 + c);
  if (late) len = start < n ? (nt[start] + 2 * (c & 3) + 1) / (2 * (c & 3) + 2) : longest;
  len = max(len, 1);
  int items = 0, split = 0, work = 0, most = 0, half = 0, rounds = 0;
  for (int i = lane; i < n; i += 64) {
    const int cuts = i < start ? 1 : (nt[i] + len - 1) / len;
    items += cuts;
    split += cuts > 1 ? cuts : 0;
    work += 4 * nt[i] + 10 * cuts + (cuts > 1 ? 12 + 11 * cuts : 0);
    const int each = nt[i] / cuts;
    most += 4 * each >= 3 * len ? cuts : 0;
    half += 2 * each >= len ? cuts : 0;
    if ((c == 0 || i < start) && i % per_head == 0) rounds = max(rounds, (i / per_head + 1) * (4 * nt[i] + 10));
  }
  items = wave_sum(items), split = wave_sum(split), work = wave_sum(work), most = wave_sum(most), half = wave_sum(half);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) rounds = max(rounds, __shfl_xor(rounds, off));
  int price = 0x7fffffff;
  if (fixed) {
    if (k <= kPrefillMaxPieces && items <= min(per_head, slots)) price = k == 1 ? 4 * len : 4 * len + 10 + 3 * k;
  } else if (late) {
    if (n <= sorted && split > 0 && split <= slots) price = max(rounds, work / per_head + 2 * len) + 20;
  } else if (split <= slots && (c == 0 || split > 0)) {
    price = max(max(4 * len + 10, work / per_head),
                max(((most - 1) / per_head + 1) * (3 * len + 10), ((half - 1) / per_head + 1) * (2 * len + 10)));
    price += split > 0 ? 20 : 0;
    if (c == 0 && n <= sorted) price = max(price, rounds);
  }
  if (lane == 0) {
    best[3 * c] = price;
    best[3 * c + 1] = len;
    best[3 * c + 2] = start;
  }
  __syncthreads();
  int pick = 0;
  for (int i = 1; i < 16; ++i)
    if (best[3 * i] < best[3 * pick]) pick = i;
  if (pick == 0 || (!fixed && 10 * (best[3 * pick] / 9) > best[0])) return 0;
  const int cut = best[3 * pick + 1], from = best[3 * pick + 2];
  // First item and first slot of each tile (wave 0 scans 64 tiles at a time;
  // items in the low half, slots in the high half).
  int* const slot_of = first + kPrefillCutTiles + 1;
  if (tid < 64) {
    int carry = 0;
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int i = i0 + lane;
      const int cuts = i >= n ? 0 : i < from ? 1 : (nt[i] + cut - 1) / cut;
      const int v = cuts + (cuts > 1 ? cuts << 16 : 0);
      int incl = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
      }
      if (i < n) {
        first[i] = (carry + incl - v) & 0xffff;
        slot_of[i] = (carry + incl - v) >> 16;
      }
      carry += __shfl(incl, 63);
    }
    if (lane == 0) first[n] = carry & 0xffff;
  }
  __syncthreads();
  const int total = first[n];  // <= n + slots <= kPrefillMaxItems
  for (int i = tid; i < kPrefillPieceSlots; i += 1024) plan[piece_list + kPrefillMaxItems * kPrefillPieceInts + i] = 0;
  int lo = 0, cuts = 1, own = 0, a = 0, b = 0;
  if (tid < total) {
    int hi = n - 1;  // last tile whose first item is <= tid
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first[mid] <= tid) lo = mid;
      else hi = mid - 1;
    }
    cuts = first[lo + 1] - first[lo];
    own = tid - first[lo];
    a = own * nt[lo] / cuts, b = (own + 1) * nt[lo] / cuts;
    len_of[tid] = b - a;
  }
  __syncthreads();
  if (tid < total) {
    int at = tid;
    if (!fixed) {  // longest first, ties in tile order
      at = 0;
      for (int o = 0; o < total; ++o) at += len_of[o] > b - a || (len_of[o] == b - a && o < tid);
    }
    const int32_t* t = tiles + lo * kPrefillPlanItemInts;
    const int pages_per_tile = kPrefillKeys / kPageSize;
    const int npages = min(t[7] - a * pages_per_tile, (b - a) * pages_per_tile);
    const int32_t* bt = block_tables + (int64_t)t[0] * bt_stride + a * pages_per_tile;
    int32_t* d = plan + piece_list + (int64_t)at * kPrefillPieceInts;
    d[0] = t[0];
    d[1] = t[1];
    d[2] = t[2];
    d[3] = t[3];
    d[4] = t[4] - a * kPrefillKeys;
    d[5] = b - a;
    d[6] = min(max(t[6] - a, 0), b - a);
    d[7] = npages;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int v = bt[min(j, npages - 1)];
      d[8 + j] = (v >= 0 && v < num_pages) ? v : 0;
    }
    d[kPrefillPieceFirstPage] = a * pages_per_tile;
    d[kPrefillPieceCount] = cuts;
    d[kPrefillPieceFirst] = cuts > 1 ? slot_of[lo] : 0;
    d[kPrefillPieceOwn] = own;
  }
  return total;
}

// How a launch takes its items: claims; claims or turns, whole tiles or pieces
// (kPieces); one item a workgroup.
enum class PlanForm { kClaims, kTurns, kFixed };
// Rounds of items dealt out in turns at most.  One prompt, 32 / 8 heads,
// claimed / in turns: 3000 tokens (47 tiles for 32 workgroups a head) 114 / 95
// us, 4096 (64) 165 / 135, 6000 (94) 287 / 281; 8 sequences of 300-600 over up
// to 2k (59) 73 / 60; 64 / 8 heads, 2048 tokens (64) 90 / 72, 6000 (188) 533 /
// 519.  At 7 rounds of 16 sequences claims were 2% faster: workgroups of a
// faster XCD take more, and one sequence's pages are read together.
constexpr int kPrefillTurns = 6;

// The form of a plan of at most max_tiles tiles, on per_head workgroups a head.
PlanForm plan_form(int64_t max_tiles, int64_t per_head) {
  if (max_tiles <= per_head) return PlanForm::kFixed;
  return max_tiles <= kPrefillTurns * per_head ? PlanForm::kTurns : PlanForm::kClaims;
}

// Exact tile list of a prefill batch, built on the device from
// query_start_loc / seq_lens (one workgroup; see kPrefillPlanHeaderInts for
// the format).  Sequences are ordered longest context first (batches of up
// to kPrefillPlanSortMax sequences; larger batches keep batch order), and a
// sequence's tiles largest key count first, so the tiles that read one
// sequence's pages run together and long work starts early.  The last
// `tail` tiles (at most 1024) are then reordered by key count, largest
// first (ties keep their order): they are the work the persistent grid
// drains last, and without it a long tile of the last sequences could start
// after the workgroups of its head had run out of work.  A sequence with no
// queries, or with more queries than keys, gets no tile.  At most
// `capacity` tiles are written; word 0 receives their number and word 1
// the number left out.
__global__ __launch_bounds__(1024) void prefill_plan_kernel(const int32_t* __restrict__ qsl,
                                                            const int32_t* __restrict__ seq_lens,
                                                            const int32_t* __restrict__ block_tables,
                                                            int64_t bt_stride, int64_t num_pages, int num_seqs,
                                                            int tile_tokens, int num_kv_heads,
                                                            int32_t* __restrict__ plan, int capacity, int tail,
                                                            int grid, PlanForm form, int per_head, int piece_list) {
  // Sequences in plan order (rank -> sequence) and the first tile of each
  // rank; beyond kPrefillPlanSortMax sequences, all keep batch order and are
  // planned in passes of kPrefillPlanSortMax.
  __shared__ int kv_of[kPrefillPlanSortMax];
  __shared__ int order[kPrefillPlanSortMax];
  __shared__ int first_tile[kPrefillPlanSortMax + 1];
  __shared__ int scan[1024];
  __shared__ int carry;
  const int tid = threadIdx.x;
  const bool sorted = num_seqs <= kPrefillPlanSortMax;
  if (tid == 0) carry = 0;
  if (sorted) {
    for (int s = tid; s < num_seqs; s += 1024) kv_of[s] = seq_lens[s];
    __syncthreads();
    for (int s = tid; s < num_seqs; s += 1024) {
      const int mine = kv_of[s];
      int rank = 0;
      for (int o = 0; o < num_seqs; ++o) {
        const int v = kv_of[o];
        rank += (v > mine) || (v == mine && o < s);
      }
      order[rank] = s;
    }
  }
  __syncthreads();
  int32_t* out = plan + kPrefillPlanHeaderInts;
  for (int c = 0; c < num_seqs; c += kPrefillPlanSortMax) {
    const int span = min(kPrefillPlanSortMax, num_seqs - c);
    // Tiles per rank in this pass over the sequences, then their exclusive
    // prefix sum.
    for (int r0 = 0; r0 < span; r0 += 1024) {
      const int r = r0 + tid;
      int nt = 0;
      if (r < span) {
        const int s = sorted ? order[r] : c + r;
        const int q_len = qsl[s + 1] - qsl[s];
        const int kv = seq_lens[s];
        if (q_len > 0 && kv >= q_len) nt = (q_len + tile_tokens - 1) / tile_tokens;
      }
      scan[tid] = nt;
      __syncthreads();
      for (int off = 1; off < 1024; off <<= 1) {
        const int add = tid >= off ? scan[tid - off] : 0;
        __syncthreads();
        scan[tid] += add;
        __syncthreads();
      }
      if (r < span) first_tile[r] = carry + scan[tid] - nt;
      __syncthreads();
      if (tid == 0) carry += scan[1023];
      __syncthreads();
    }
    if (tid == 0) first_tile[span] = carry;
    __syncthreads();
    // One tile per thread: find its rank by binary search, write its record.
    const int lo_tile = first_tile[0], hi_tile = first_tile[span];
    for (int i = lo_tile + tid; i < hi_tile && i < capacity; i += 1024) {
      int lo = 0, hi = span - 1;  // last rank whose first tile is <= i
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first_tile[mid] <= i) lo = mid;
        else hi = mid - 1;
      }
      const int s = sorted ? order[lo] : c + lo;
      const int q0 = qsl[s];
      const int q_len = qsl[s + 1] - q0;
      const int kv = seq_lens[s];
      const int nt = (q_len + tile_tokens - 1) / tile_tokens;
      const int jt = i - first_tile[lo];
      const int t0 = (nt - 1 - jt) * tile_tokens;  // largest key count first
      const int bpos = kv - q_len;
      const int kv_end = bpos + min(t0 + tile_tokens, q_len);
      const int ntiles = (kv_end + kPrefillKeys - 1) / kPrefillKeys;
      const int full = min((bpos + t0 + 1) / kPrefillKeys, ntiles);
      const int npages = (kv_end + kPageSize - 1) / kPageSize;
      const int32_t* bt = block_tables + (int64_t)s * bt_stride;
      int pg[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int v = bt[min(k, npages - 1)];
        pg[k] = (v >= 0 && v < num_pages) ? v : 0;
      }
      int32_t* d = out + (int64_t)i * kPrefillPlanItemInts;
      *reinterpret_cast<int4*>(d) = int4{s, t0, q0, q_len};
      *reinterpret_cast<int4*>(d + 4) = int4{kv, ntiles, full, npages};
      *reinterpret_cast<int4*>(d + 8) = int4{pg[0], pg[1], pg[2], pg[3]};
      *reinterpret_cast<int4*>(d + 12) = int4{pg[4], pg[5], pg[6], pg[7]};
    }
    __syncthreads();
  }
  {
    // The tail: thread i holds tile base + i, ranks it among the tail by key
    // count (stable) and writes it to its rank.  Every thread has read its
    // record (the barrier waits for the loads) before any is written.
    const int n = min(carry, capacity);
    const int K = min(min(n, tail), 1024);
    if (K > 1) {
      const int base = n - K;
      int4 r0, r1, r2, r3;
      int key = -1;
      if (tid < K) {
        const int4* src = reinterpret_cast<const int4*>(out + (int64_t)(base + tid) * kPrefillPlanItemInts);
        r0 = src[0];
        r1 = src[1];
        r2 = src[2];
        r3 = src[3];
        key = r1.y;  // ntiles
      }
      scan[tid] = key;
      __syncthreads();
      if (tid < K) {
        int rank = 0;
        for (int o = 0; o < K; ++o) {
          const int v = scan[o];
          rank += (v > key) || (v == key && o < tid);
        }
        int4* dst = reinterpret_cast<int4*>(out + (int64_t)(base + rank) * kPrefillPlanItemInts);
        dst[0] = r0;
        dst[1] = r1;
        dst[2] = r2;
        dst[3] = r3;
      }
    }
  }
  const int n = min(carry, capacity);
  const int pieces = plan_pieces(plan, n, form == PlanForm::kFixed, per_head, num_kv_heads, block_tables, bt_stride,
                                 num_pages, piece_list, tail, scan, first_tile, order, kv_of);
  if (tid == 0) {
    plan[kPrefillPlanPiecesInt] = pieces;
    plan[kPrefillPlanPieceListInt] = piece_list;
    plan[kPrefillPlanArriveInt] = piece_list + kPrefillMaxItems * kPrefillPieceInts;
    plan[kPrefillPlanPartInt] = (int)((piece_list + kPrefillSplitMetaInts) / (kPrefillPartUnit / 4));
    // All tiles are longest first where the sorted tail holds them.
    plan[kPrefillPlanTurnInt] = form == PlanForm::kTurns && (pieces > 0 || n <= tail) ? per_head : 0;
    plan[0] = n;
    plan[kPrefillPlanDroppedInt] = max(carry - capacity, 0);
    plan[kPrefillPlanExitInt] = 0;
    plan[kPrefillPlanGridInt] = grid;
  }
  if (tid < kPrefillPlanMaxHeads) plan[kPrefillPlanLineInts * (1 + tid)] = 0;  // claim counters
}

// The last workgroup out zeroes the claim counters and the exit count, so
// the plan serves the next launch as it is.  Every claim and counter read
// of a workgroup has returned (its result decided the exit) before thread 0
// counts the workgroup out, and workgroups of any head claim from every
// head's counter, so only the grid's last exit may clear them.
// (The grid size comes from the plan header, which keeps the dispatch
// packet's registers out of the tile loop.)  Every thread of the workgroup
// calls it.
template <bool kPieces>
__device__ __attribute__((always_inline)) inline void leave_prefill_plan(int32_t* plan) {
  if (kPieces && sload(plan, kPrefillPlanTurnInt) > 0) return;  // nothing was claimed
  __syncthreads();
  if (threadIdx.x >= 64) return;
  int gone = 0;
  if (threadIdx.x == 0)
    gone = __hip_atomic_fetch_add(plan + kPrefillPlanExitInt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  gone = __builtin_amdgcn_readfirstlane(gone);
  if (gone != plan[kPrefillPlanGridInt] - 1) return;
  for (int hh = threadIdx.x; hh < kPrefillPlanMaxHeads; hh += 64)
    __hip_atomic_store(plan + kPrefillPlanLineInts * (1 + hh), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (threadIdx.x == 0) __hip_atomic_store(plan + kPrefillPlanExitInt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Persistent prefill: workgroup b serves KV head b % num_kv_heads (so head
// h stays on XCD h when the head count divides 8).  The workgroups of a head
// take tiles of the plan in order from that head's claim counter, one claim
// ahead (prefill_items_pingpong), so the grid never waits on dispatch and
// faster CUs simply run more tiles; once their head's queue is exhausted
// they take the remaining tiles of the other heads.
template <typename T, bool kPieces>
__global__ __launch_bounds__(kPrefillPPThreads) void paged_prefill_stream_kernel(PrefillParams p,
                                                                                 int32_t* __restrict__ plan) {
  __shared__ __attribute__((aligned(16))) uint8_t tiles[kPrefillPPLdsBytes];
  __shared__ int nextq[8];
  const int h = (int)(blockIdx.x % (uint32_t)p.num_kv_heads);
  const int rank = kPieces ? (int)(blockIdx.x / (uint32_t)p.num_kv_heads) : 0;
  if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) == 0)
    prefill_items_pingpong<T, 0, false, kPieces>(p, plan, h, rank, (lds_u8*)tiles, (lds_i32*)nextq);
  else
    prefill_items_pingpong<T, 1, false, kPieces>(p, plan, h, rank, (lds_u8*)tiles, (lds_i32*)nextq);
  leave_prefill_plan<kPieces>(plan);
}

// The fixed form, for a batch of at most one tile per workgroup of a head: no
// claims, and tiles may be cut into split-K pieces (plan_pieces).
template <typename T>
__global__ __launch_bounds__(kPrefillPPThreads) void paged_prefill_fixed_kernel(PrefillParams p,
                                                                                int32_t* __restrict__ plan) {
  __shared__ __attribute__((aligned(16))) uint8_t tiles[kPrefillPPLdsBytes];
  __shared__ int nextq[8];
  const int h = (int)(blockIdx.x % (uint32_t)p.num_kv_heads);
  const int rank = (int)(blockIdx.x / (uint32_t)p.num_kv_heads);
  if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) == 0)
    prefill_items_pingpong<T, 0, true, true>(p, plan, h, rank, (lds_u8*)tiles, (lds_i32*)nextq);
  else
    prefill_items_pingpong<T, 1, true, true>(p, plan, h, rank, (lds_u8*)tiles, (lds_i32*)nextq);
}

// A MIXED step on CUs of two kinds.  Workgroups of 512 threads, one per CU
// (128 KB of LDS): the first `n_prefill` (a whole number per KV head) run the
// prefill plan as the prefill-only kernels do, the rest run eight decode
// wavefronts each, as the piece-list decode kernel does.  With kFixed the
// plan has at most one item per prefill workgroup of a head.  Otherwise items
// are dealt out to the prefill workgroups in turns up to kPrefillTurns rounds,
// and a decode workgroup whose pieces are done ends; beyond that tiles are
// claimed, and it joins in.
//
// The two parts have different bounds (the matrix cores and HBM), so they are
// best run side by side; sharing every CU between decode wavefronts and a
// four-wave prefill core (paged_mixed_kernel) costs each part the other's
// registers, LDS and issue slots: it time-slices more than it overlaps, with
// prefill tiles half as large, none cut, at the end of a wave of work.  On
// CUs of their own each part runs its own kernel's schedule.  What bounds it:
// a CU of decode wavefronts has 64 KB in flight, 38 GB/s, so the CUs left to
// decode set its time until HBM does (5.8 TB/s), and the prefill CUs slow
// down beside it (power and L2).  Against paged_mixed_kernel, microseconds of
// a step: 300 tokens over 1936 and 20 decodes of 2250 (32 / 8 heads, fp16)
// 69 -> 47, 2 chunks over 4k and 64 decodes of 2700 211 -> 176, 4 chunks of a
// budget of 8192 and 256 decodes of 4391 974 -> 914, 1 decode of 12695 beside
// 109 prompt tokens (64 / 8 heads) 168 -> 20; small steps are left to that
// kernel (mva_mixed_prefill_share).  Split-K decode segments are
// merged by the merge kernel that follows: merging inside the launch cost 5
// to 17 us more (the merges run one after another on the last wavefronts).
template <typename T, bool kFixed>
__global__ __launch_bounds__(kPrefillPPThreads) void paged_mixed_split_cus_kernel(PrefillParams pp,
                                                                                  int32_t* __restrict__ plan,
                                                                                  DecodeParams dp,
                                                                                  uint32_t n_prefill) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kMixedDecodeWaves * kDecodeWaveLdsBytes];
  __shared__ int nextq[8];
  __shared__ int progress[kMixedDecodeWaves];
  if (blockIdx.x >= n_prefill) {
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wave = (int)(blockIdx.x - n_prefill) * kMixedDecodeWaves + w;
    if ((threadIdx.x & 63) == 0) progress[w] = 0x3fffffff;
    if (wave < dp.num_waves) decode_wave<T>(dp, wave, (lds_u8*)lds + w * kDecodeWaveLdsBytes, progress);
    if constexpr (kFixed) return;
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();  // the LDS of all eight is free
  }
  const int h = (int)(blockIdx.x % (uint32_t)pp.num_kv_heads);
  const int rank = (int)(blockIdx.x / (uint32_t)pp.num_kv_heads);
  if (__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) == 0)
    prefill_items_pingpong<T, 0, kFixed, true>(pp, plan, h, rank, (lds_u8*)lds, (lds_i32*)nextq);
  else
    prefill_items_pingpong<T, 1, kFixed, true>(pp, plan, h, rank, (lds_u8*)lds, (lds_i32*)nextq);
  if constexpr (!kFixed) leave_prefill_plan<true>(plan);
}

static_assert(kMixedDecodeWaves * kDecodeWaveLdsBytes >= kPrefillPPLdsBytes, "prefill tiles fit the decode buffers");

int device_cu_count() {
  static int counts[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (counts[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    counts[dev] = cus;
  }
  return counts[dev];
}

// Workgroup roles of the MIXED launch: the decode workgroups come first, in
// chunks of 8 blocks (blocks are dealt to the 8 XCDs round-robin), then the
// prefill workgroups.  The host sizes the decode part below the GPU's
// resident capacity, so every decode wavefront starts at once and prefill
// workgroups fill the remaining slots (and the slots decode frees): HBM-bound
// decode streaming overlaps MFMA-bound prefill on the same CUs.  Prefill
// blocks keep index % 8 == block % 8, so prefill workgroup i, which serves
// KV head i % num_kv_heads, runs on the XCD that serves that head in the
// prefill-only launch.
struct MixedRole {
  bool prefill;
  uint32_t index;  // prefill workgroup or decode workgroup number
};
__host__ __device__ inline uint32_t mixed_chunks(uint32_t n) { return (n + 7u) >> 3; }
__device__ inline MixedRole mixed_role(uint32_t block, uint32_t n_decode_wgs) {
  const uint32_t c = block >> 3, r = block & 7u;
  const uint32_t cd = mixed_chunks(n_decode_wgs);
  if (c < cd) return {false, c * 8u + r};
  return {true, (c - cd) * 8u + r};
}

// Prefill sequences a MIXED launch orders in LDS.
constexpr int kMixedPrefillSeqsMax = 1024;

// The prefill workgroups of a MIXED launch are a persistent pool of
// `per_head` workgroups per KV head.  Each builds the launch's query-tile
// order in LDS from query_start_loc / seq_lens of the leading p.num_seqs
// sequences -- sequences longest context first (ties by index), a
// sequence's 128-row tiles largest key count first, as the PREFILL planner
// orders them -- then takes tiles from its head's claim counter until none
// are left.  So every tile run is a real tile, and no query count is needed
// on the host.  A workgroup claims its next tile when its current one ends:
// with about two tiles per workgroup, claiming one ahead would reserve
// nearly every tile at the start and undo the balancing (measured 11%
// slower on the prefill half of a budget-8192 batch).  A sequence with no queries, or more
// queries than keys, has no tile.  The last workgroup of a head to leave
// clears that head's counters for the next launch.
template <typename T>
__device__ void mixed_prefill_pool(const PrefillParams& p, int32_t* sched, uint32_t index, uint32_t per_head,
                                   int* order, int* first_tile, int* claimed, lds_u8* k0, lds_u8* k1, lds_u8* v0,
                                   lds_u8* v1) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int S = p.num_seqs;
  const int BMT = p.tile_tokens;
  const int h = (int)(index % (uint32_t)p.num_kv_heads);
  int* const ctr = sched + kMixedPrefillCtrInt + h * kDecodeSchedLineInts;
  if (tid == 0) *claimed = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // Tile order.  The K/V tile buffers are free until the first tile: k0
  // holds the context lengths, k1 the tile counts by rank.
  int* const kv_of = (int*)k0;
  int* const tiles_of = (int*)k1;
  for (int s = tid; s < S; s += 256) kv_of[s] = p.seq_lens[s];
  __syncthreads();
  for (int s = tid; s < S; s += 256) {
    const int mine = kv_of[s];
    int rank = 0;
    for (int o = 0; o < S; ++o) {
      const int v = kv_of[o];
      rank += (v > mine) || (v == mine && o < s);
    }
    order[rank] = s;
  }
  __syncthreads();
  for (int r = tid; r < S; r += 256) {
    const int s = order[r];
    const int q_len = p.query_start_loc[s + 1] - p.query_start_loc[s];
    const int kv = kv_of[s];
    tiles_of[r] = (q_len > 0 && kv >= q_len) ? (q_len + BMT - 1) / BMT : 0;
  }
  __syncthreads();
  if (tid < 64) {
    // Exclusive prefix sum over ranks, 64 at a time, by wave 0.
    int carry = 0;
    for (int c = 0; c < S; c += 64) {
      const int v = c + lane < S ? tiles_of[c + lane] : 0;
      int incl = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off);
        if (lane >= off) incl += up;
      }
      if (c + lane < S) first_tile[c + lane] = carry + incl - v;
      carry += __shfl(incl, 63);
    }
    if (lane == 0) first_tile[S] = carry;
  }
  __syncthreads();
  const int total = __builtin_amdgcn_readfirstlane(first_tile[S]);

  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int idx = __builtin_amdgcn_readfirstlane(*claimed);
  while (idx < total) {
    // Rank of tile idx: the last rank whose first tile is <= idx.
    int lo = 0, hi = S - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (first_tile[mid] <= idx) lo = mid;
      else hi = mid - 1;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    PrefillWork wk;
    wk.s = __builtin_amdgcn_readfirstlane(order[lo]);
    wk.q0 = sload(p.query_start_loc, wk.s);
    wk.q_len = sload(p.query_start_loc, wk.s + 1) - wk.q0;
    wk.kv = sload(p.seq_lens, wk.s);
    const int nt = (wk.q_len + BMT - 1) / BMT;
    wk.t0 = (nt - 1 - (idx - __builtin_amdgcn_readfirstlane(first_tile[lo]))) * BMT;  // largest key count first
    const int base_pos = wk.kv - wk.q_len;
    const int kv_end = base_pos + min(wk.t0 + BMT, wk.q_len);  // keys [0, kv_end) are needed
    wk.ntiles = (kv_end + kPrefillKeys - 1) / kPrefillKeys;
    wk.full_tiles = min((base_pos + wk.t0 + 1) / kPrefillKeys, wk.ntiles);
    wk.npages = (kv_end + kPageSize - 1) / kPageSize;
    const int32_t* bt = p.block_tables + (int64_t)wk.s * p.bt_stride;
    auto page = [&](int i) {
      const int pg = sload(bt, min(i, wk.npages - 1));
      return (pg >= 0 && pg < p.num_pages) ? pg : 0;
    };
    wk.pg0 = page(w);
    wk.pg1 = page(kPrefillKeys / kPageSize + w);
    prefill_core<T>(p, wk, h, k0, k1, v0, v1);
    __syncthreads();  // every wave is done with this tile's LDS before `claimed` changes
    if (tid == 0) *claimed = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    idx = __builtin_amdgcn_readfirstlane(*claimed);
  }
  if (tid == 0) {
    // Every claim of this workgroup has returned (the last one ended the
    // loop), so all claims on the counter precede the clear.
    const int gone =
        __hip_atomic_fetch_add(ctr + kMixedPrefillExitOffset, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (gone == (int)per_head - 1) {
      __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(ctr + kMixedPrefillExitOffset, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Prefill workgroups run the prefill pool; decode workgroups run four
// decode wavefronts each, with private LDS buffers.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void paged_mixed_kernel(
    PrefillParams pp, DecodeParams dp, uint32_t n_prefill_wgs, uint32_t n_decode_wgs) {
  __shared__ __attribute__((aligned(16))) uint8_t k0[kPrefillTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t k1[kPrefillTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t v0[kPrefillTileBytes];
  __shared__ __attribute__((aligned(16))) uint8_t v1[kPrefillTileBytes];
  __shared__ int order[kMixedPrefillSeqsMax];
  __shared__ int first_tile[kMixedPrefillSeqsMax + 1];
  __shared__ int claimed;
  const MixedRole role = mixed_role(blockIdx.x, n_decode_wgs);
  if (role.prefill) {
    if (role.index >= n_prefill_wgs) return;
    mixed_prefill_pool<T>(pp, dp.sched, role.index, n_prefill_wgs / (uint32_t)pp.num_kv_heads, order, first_tile,
                          &claimed, (lds_u8*)k0, (lds_u8*)k1, (lds_u8*)v0, (lds_u8*)v1);
    return;
  }
  const int w = threadIdx.x >> 6;
  const int64_t wave = (int64_t)role.index * 4 + w;
  if (wave >= dp.num_waves) return;
  // Each decode wavefront gets one of the four prefill buffers.
  lds_u8* mine = (lds_u8*)(w == 0 ? k0 : w == 1 ? k1 : w == 2 ? v0 : v1);
  decode_wave<T, true>(dp, (int)wave, mine);
}

static_assert(kMixedPrefillSeqsMax * 4 <= kPrefillTileBytes, "context lengths fit one K/V tile buffer");
static_assert(kDecodeWaveLdsBytes <= kPrefillTileBytes, "a decode wave's buffers must fit one prefill buffer");

}  // namespace

int fill_prefill_params(PrefillParams& p, const void* q, int64_t q_token_stride, int64_t q_head_stride,
                        const void* k_cache, const void* v_cache, int64_t num_pages, int64_t page_stride,
                        int64_t token_stride, const int32_t* block_tables, int64_t block_table_stride,
                        const int32_t* seq_lens, const int32_t* query_start_loc, int64_t num_seqs,
                        void* out, int64_t out_token_stride, int64_t out_head_stride,
                        int num_q_heads, int num_kv_heads, int head_dim, int page_size, float softmax_scale) {
  if (head_dim != kHeadDim) return set_error("paged attention: head_dim must be 128");
  if (page_size != kPageSize) return set_error("paged attention: page_size must be 16");
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads)
    return set_error("paged attention: num_q_heads must be a positive multiple of num_kv_heads");
  const int group = num_q_heads / num_kv_heads;
  if (group > 16) return set_error("paged attention: at most 16 query heads per KV head");
  if (num_seqs < 0 || num_seqs > 0x7fffffffLL) return set_error("paged attention: invalid sequence count");
  if (num_pages <= 0) return set_error("paged attention: empty KV cache");
  const uint64_t align_bits = (uint64_t)(uintptr_t)q | (uint64_t)(uintptr_t)k_cache |
                              (uint64_t)(uintptr_t)v_cache | (uint64_t)(q_token_stride * 2) |
                              (uint64_t)(q_head_stride * 2) | (uint64_t)(page_stride * 2) |
                              (uint64_t)(token_stride * 2);
  if (align_bits % 16) return set_error("paged attention: q / cache buffers and strides must be 16-byte aligned");
  if (((uint64_t)(uintptr_t)out | (uint64_t)(out_token_stride * 2) | (uint64_t)(out_head_stride * 2)) % 8)
    return set_error("paged attention: output buffer and strides must be 8-byte aligned");
  p.q = q;
  p.q_tok_stride = q_token_stride;
  p.q_head_stride = q_head_stride;
  p.k_cache = k_cache;
  p.v_cache = v_cache;
  p.num_pages = num_pages;
  p.page_stride = page_stride;
  p.tok_stride = token_stride;
  p.block_tables = block_tables;
  p.bt_stride = block_table_stride;
  p.seq_lens = seq_lens;
  p.query_start_loc = query_start_loc;
  p.num_seqs = (int)num_seqs;
  p.out = out;
  p.out_tok_stride = out_token_stride;
  p.out_head_stride = out_head_stride;
  p.num_kv_heads = num_kv_heads;
  p.group = group;
  p.tile_tokens = kPrefillRows / group;
  p.scale_log2 = softmax_scale * 1.4426950408889634f;
  p.out16 = ((uint64_t)(uintptr_t)out | (uint64_t)(out_token_stride * 2) | (uint64_t)(out_head_stride * 2)) % 16 == 0;
  return 0;
}

}  // namespace mva

extern "C" int mva_prefill_tile_tokens(int num_q_heads, int num_kv_heads) {
  if (num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads) return -1;
  return mva::kPrefillRows / (num_q_heads / num_kv_heads);
}

extern "C" int64_t mva_prefill_workspace_bytes(int64_t max_tiles) {
  if (max_tiles < 0 || max_tiles > 0x7fffffffLL / mva::kPrefillPlanItemInts) return -1;
  // The split-K area at every size, though only plans of at most
  // kPrefillCutTiles tiles use it: a workspace sized for a program's largest
  // batch, or by its memory probe, then serves every smaller one in full.
  return mva::prefill_split_bytes(max_tiles);
}

namespace {

using namespace mva;

const char kBadTileCapacity[] = "paged attention: invalid tile capacity";

// Plans a batch for `per_head` prefill workgroups per KV head in a launch of
// `grid` workgroups that count themselves out of the plan.
int launch_prefill_plan(const PrefillParams& p, int64_t num_seqs, int64_t max_tiles, int32_t* plan,
                        int64_t workspace_bytes, int64_t per_head, int64_t grid, hipStream_t s) {
  const PlanForm form = plan_form(max_tiles, per_head);
  // All tiles of a plan dealt out in turns go largest first, otherwise the
  // last three per workgroup of a head.
  const int64_t last =
      form == PlanForm::kTurns ? max_tiles : 3 * (per_head < max_tiles ? per_head : max_tiles);
  const int tail = (int)(last < 1024 ? last : 1024);
  // Tiles may be cut where there is room for partials.
  const bool split = form != PlanForm::kClaims && max_tiles <= kPrefillCutTiles &&
                     workspace_bytes >= prefill_split_bytes(max_tiles);
  hipLaunchKernelGGL(prefill_plan_kernel, dim3(1), dim3(1024), 0, s, p.query_start_loc, p.seq_lens, p.block_tables,
                     p.bt_stride, p.num_pages, (int)num_seqs, p.tile_tokens, p.num_kv_heads, plan, (int)max_tiles, tail,
                     (int)grid, form, (int)per_head, split ? (int)prefill_piece_list(max_tiles) : 0);
  return check_launch("paged_prefill plan");
}

// The checks of a prefill plan's tile capacity, workspace and head count.
int check_prefill_plan(int64_t max_tiles, const void* workspace, int64_t workspace_bytes, int num_kv_heads) {
  if (mva_prefill_workspace_bytes(max_tiles) < 0) return set_error(kBadTileCapacity);
  // The plan itself must fit; without room for partials no tile is split.
  if (workspace == nullptr || workspace_bytes < prefill_plan_bytes(max_tiles))
    return set_error("paged attention: prefill workspace too small for max_tiles");
  if (((uintptr_t)workspace) % 16) return set_error("paged attention: prefill workspace must be 16-byte aligned");
  if (num_kv_heads > kPrefillPlanMaxHeads) return set_error("paged attention: at most 127 KV heads");
  return 0;
}

// Plans (plan_it) and/or streams (run_it) a prefill batch: the shared body
// of mva_paged_prefill, mva_paged_prefill_plan and mva_paged_prefill_run.
int prefill_launch(const void* q, int64_t q_token_stride, int64_t q_head_stride, const void* k_cache,
                   const void* v_cache, int64_t num_pages, int64_t page_stride, int64_t token_stride,
                   const int32_t* block_tables, int64_t block_table_stride, const int32_t* seq_lens,
                   const int32_t* query_start_loc, int64_t num_seqs, int64_t max_tiles, void* workspace,
                   int64_t workspace_bytes, void* out, int64_t out_token_stride, int64_t out_head_stride,
                   int num_q_heads, int num_kv_heads, int head_dim, int page_size, float softmax_scale, int dtype,
                   void* stream, bool plan_it, bool run_it) {
  PrefillParams p;
  int rc = fill_prefill_params(p, q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride,
                               token_stride, block_tables, block_table_stride, seq_lens, query_start_loc,
                               num_seqs, out, out_token_stride, out_head_stride, num_q_heads,
                               num_kv_heads, head_dim, page_size, softmax_scale);
  if (rc) return rc;
  if (dtype != kBF16 && dtype != kF16) return set_error("paged attention: dtype must be bf16 or fp16");
  if (mva_prefill_workspace_bytes(max_tiles) < 0) return set_error(kBadTileCapacity);
  if (num_seqs == 0 || max_tiles == 0) return 0;
  rc = check_prefill_plan(max_tiles, workspace, workspace_bytes, num_kv_heads);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  int32_t* plan = (int32_t*)workspace;
  p.tile_tokens = kPrefillPPRows / p.group;
  // Persistent grid: one workgroup per CU (96 KB of LDS and two waves per
  // SIMD each), a whole number per KV head, also where the tiles are fewer:
  // they may be planned as pieces.
  int64_t per_head = (int64_t)device_cu_count() / num_kv_heads;
  per_head = per_head < 1 ? 1 : per_head;
  const PlanForm form = plan_form(max_tiles, per_head);
  if (plan_it) {
    rc = launch_prefill_plan(p, num_seqs, max_tiles, plan, workspace_bytes, per_head, per_head * num_kv_heads, s);
    if (rc) return rc;
  }
  if (!run_it) return 0;
  const dim3 grid((uint32_t)(per_head * num_kv_heads));
  if (form == PlanForm::kFixed) {
    if (dtype == kBF16)
      hipLaunchKernelGGL(paged_prefill_fixed_kernel<__bf16>, grid, dim3(kPrefillPPThreads), 0, s, p, plan);
    else
      hipLaunchKernelGGL(paged_prefill_fixed_kernel<_Float16>, grid, dim3(kPrefillPPThreads), 0, s, p, plan);
    return check_launch("paged_prefill");
  }
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(kPrefillPPThreads), 0, s, p, plan); };
  const bool pieces = form == PlanForm::kTurns;
  if (dtype == kBF16) {
    if (pieces) launch(paged_prefill_stream_kernel<__bf16, true>);
    else launch(paged_prefill_stream_kernel<__bf16, false>);
  } else {
    if (pieces) launch(paged_prefill_stream_kernel<_Float16, true>);
    else launch(paged_prefill_stream_kernel<_Float16, false>);
  }
  return check_launch("paged_prefill");
}

// Stand-ins for the buffers a plan-only launch does not touch: they pass the
// alignment checks and are never dereferenced.
alignas(16) const uint8_t kPlanOnlyDummy[16] = {};

}  // namespace

extern "C" int mva_paged_prefill(const void* q, int64_t q_token_stride, int64_t q_head_stride,
                                 const void* k_cache, const void* v_cache, int64_t num_pages,
                                 int64_t page_stride, int64_t token_stride, const int32_t* block_tables,
                                 int64_t block_table_stride, const int32_t* seq_lens,
                                 const int32_t* query_start_loc, int64_t num_seqs, int64_t max_tiles,
                                 void* workspace, int64_t workspace_bytes, void* out, int64_t out_token_stride,
                                 int64_t out_head_stride, int num_q_heads, int num_kv_heads, int head_dim,
                                 int page_size, float softmax_scale, int dtype, void* stream) {
  return prefill_launch(q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride, token_stride,
                        block_tables, block_table_stride, seq_lens, query_start_loc, num_seqs, max_tiles, workspace,
                        workspace_bytes, out, out_token_stride, out_head_stride, num_q_heads, num_kv_heads, head_dim,
                        page_size, softmax_scale, dtype, stream, true, true);
}

extern "C" int mva_paged_prefill_plan(const int32_t* block_tables, int64_t block_table_stride, int64_t num_pages,
                                      const int32_t* seq_lens, const int32_t* query_start_loc, int64_t num_seqs,
                                      int64_t max_tiles, void* workspace, int64_t workspace_bytes,
                                      int num_q_heads, int num_kv_heads, void* stream) {
  const void* d = kPlanOnlyDummy;
  return prefill_launch(d, 0, 0, d, d, num_pages, 0, 0, block_tables, block_table_stride, seq_lens,
                        query_start_loc, num_seqs, max_tiles, workspace, workspace_bytes, (void*)d, 0, 0,
                        num_q_heads, num_kv_heads, mva::kHeadDim, mva::kPageSize, 1.0f, mva::kBF16, stream, true,
                        false);
}

extern "C" int mva_paged_prefill_run(const void* q, int64_t q_token_stride, int64_t q_head_stride,
                                     const void* k_cache, const void* v_cache, int64_t num_pages,
                                     int64_t page_stride, int64_t token_stride, const int32_t* block_tables,
                                     int64_t block_table_stride, const int32_t* seq_lens,
                                     const int32_t* query_start_loc, int64_t num_seqs, int64_t max_tiles,
                                     void* workspace, int64_t workspace_bytes, void* out,
                                     int64_t out_token_stride, int64_t out_head_stride, int num_q_heads,
                                     int num_kv_heads, int head_dim, int page_size, float softmax_scale, int dtype,
                                     void* stream) {
  return prefill_launch(q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride, token_stride,
                        block_tables, block_table_stride, seq_lens, query_start_loc, num_seqs, max_tiles, workspace,
                        workspace_bytes, out, out_token_stride, out_head_stride, num_q_heads, num_kv_heads, head_dim,
                        page_size, softmax_scale, dtype, stream, false, true);
}

extern "C" int mva_paged_mixed(const void* q, int64_t q_token_stride, int64_t q_head_stride,
                               const void* k_cache, const void* v_cache, int64_t num_pages,
                               int64_t page_stride, int64_t token_stride, const int32_t* block_tables,
                               int64_t block_table_stride, const int32_t* seq_lens,
                               const int32_t* query_start_loc, int64_t num_prefill_seqs, int64_t max_prefill_tiles,
                               const int32_t* decode_items, int64_t num_decode_items, int64_t num_decode_waves,
                               int64_t num_part_slots, void* out, int64_t out_token_stride, int64_t out_head_stride,
                               void* workspace, int64_t workspace_bytes, int num_q_heads,
                               int num_kv_heads, int head_dim, int page_size, float softmax_scale,
                               int dtype, void* stream) {
  using namespace mva;
  PrefillParams pp;
  int rc = fill_prefill_params(pp, q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride,
                               token_stride, block_tables, block_table_stride, seq_lens, query_start_loc,
                               num_prefill_seqs, out, out_token_stride, out_head_stride,
                               num_q_heads, num_kv_heads, head_dim, page_size, softmax_scale);
  if (rc) return rc;
  if (num_prefill_seqs > kMixedPrefillSeqsMax)
    return set_error("paged attention: a MIXED launch takes at most 1024 prefill sequences");
  if (max_prefill_tiles < 0 || max_prefill_tiles > 0x7fffffffLL)
    return set_error("paged attention: invalid prefill tile capacity");
  DecodeParams dp;
  rc = fill_decode_params(dp, q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride,
                          token_stride, block_tables, block_table_stride, seq_lens, decode_items,
                          num_decode_items, num_decode_waves, nullptr, nullptr, 0, num_part_slots, out,
                          out_token_stride, out_head_stride,
                          workspace, workspace_bytes, num_q_heads, num_kv_heads, head_dim, page_size,
                          softmax_scale);
  if (rc) return rc;
  // Split-K segments are merged inside the launch by their last piece.
  if (num_part_slots * num_kv_heads > kArrivalCounters)
    return set_error("paged attention: a MIXED launch takes at most 65536 split-K (partial slot, KV head) pairs");
  dp.arrive = decode_arrival_counters(workspace);
  // Prefill pool: two workgroups per CU (the CU's eight wave slots), a whole
  // number per KV head, never more than the tiles can use.
  int64_t per_head = 0;
  if (num_prefill_seqs > 0 && max_prefill_tiles > 0) {
    if (num_kv_heads > kMixedPrefillMaxHeads) return set_error("paged attention: a MIXED launch takes at most 64 KV heads");
    if (workspace == nullptr) return set_error("paged attention: MIXED launches need the decode workspace");
    per_head = 2 * (int64_t)device_cu_count() / num_kv_heads;
    per_head = per_head < 1 ? 1 : (per_head > max_prefill_tiles ? max_prefill_tiles : per_head);
  }
  const int64_t n_prefill_wgs = per_head * num_kv_heads;
  const int64_t n_decode_wgs = num_decode_items > 0 ? (num_decode_waves + 3) / 4 : 0;
  if (n_prefill_wgs + n_decode_wgs > 0x7fffff00LL) return set_error("paged attention: too many work items");
  if (n_prefill_wgs + n_decode_wgs == 0) return 0;
  const uint32_t np = (uint32_t)n_prefill_wgs, nd = (uint32_t)n_decode_wgs;
  const dim3 grid(8u * (mixed_chunks(np) + mixed_chunks(nd)));
  hipStream_t s = (hipStream_t)stream;
  if (dtype == kBF16)
    hipLaunchKernelGGL(paged_mixed_kernel<__bf16>, grid, dim3(256), 0, s, pp, dp, np, nd);
  else if (dtype == kF16)
    hipLaunchKernelGGL(paged_mixed_kernel<_Float16>, grid, dim3(256), 0, s, pp, dp, np, nd);
  else return set_error("paged attention: dtype must be bf16 or fp16");
  return check_launch("paged_mixed");
}

// Host estimates for MIXED steps (see mva_mixed_prefill_share): the time of
// mva_paged_mixed_run at a share of the CUs for its prefill part, and that of
// mva_paged_mixed, in microseconds fitted to sweeps of the share over 1170 drawn
// steps on one MI355X (11400 timings; one prefill sequence or more, even and
// skewed, less than 1 MB to 2.5 GB of decode K/V).  Of a timing over the
// estimate, the 5th and 95th percentiles: decode-bound 0.90 and 1.10,
// prefill-bound with an item a workgroup 0.92 and 1.09, in rounds 0.89 and
// 1.17; mva_paged_mixed 0.88 and 1.10 up to 30 us, 0.80 and 1.29 from there to
// 150, 0.90 and 1.11 beyond.  Tiles and pieces are counted as plan_pieces counts
// them, but its prices are its own: the two need not agree, and a share that is
// off costs time and nothing else.
namespace {

// Decode part: a CU of eight wavefronts streams 1 MB in 23.65 beside 0.0375 per
// MB of the launch, and all of them together no faster than 0.1746 (5.7 TB/s).
constexpr double kDecodeStartUs = 7.81, kDecodeUsPerMB = 0.0375, kDecodeUsPerMBCu = 23.65, kDecodeMinUsPerMB = 0.1746;
// Prefill part, one item a workgroup: whole tiles, or tiles cut into k.
constexpr double kWholeStartUs = 11.71, kWholeKeyUs = 1.334;
constexpr double kCutStartUs = 15.75, kCutPieceUs = 1.017, kCutKeyUs = 1.347;
// More tiles than workgroups: key tiles and items a workgroup, the tiles that
// must share one, and what a cut plan in turns has on top.
constexpr double kRoundsStartUs = 9.48, kRoundsKeyUs = 1.559, kRoundsItemUs = 4.56, kTogetherUs = 1.403;
constexpr double kItemKeys = 2.5, kTurnsCutUs = 16.0;
// The parts slow each other down: the longer one by kBeside of the shorter,
// times the root of their ratio.
constexpr double kBeside = 0.151;
// mva_paged_mixed: the longest tile, the longest decode piece and its merge
// (one pass of 32 chunks a query head after another), and the work of a CU
// with its decode wavefronts' pieces, in a root of squares.
constexpr double kOneStartUs = 4.05, kOneKeyUs = 1.287, kOnePageUs = 1.985, kOnePassUs = 0.912, kOneChunkUs = 0.031,
                 kOneWorkUs = 0.778, kOneTileUs = 3.42, kOneMBUs = 0.164, kOnePieceUs = 14.95;
constexpr double kMixedWavesPerCu = 6.0, kPiecesPerWave = 1.5;  // of its decode plan (plan_decode_claims)
constexpr int64_t kListTiles = 1024;  // batches of more tiles are taken as even

struct PrefillEstimate {
  int64_t tiles = 0, half_tiles = 0;  // query tiles of one KV head: 256 rows, 128 rows
  double work = 0, half_work = 0;     // 64-key tiles of all of them
  int longest = 0;
  int spare = 0;          // pieces that a cut keeps free (the lengths are not known)
  std::vector<int> keys;  // 64-key tiles of each 256-row tile, longest first (empty beyond kListTiles)
  // Pieces of all tiles when the longest is cut into k, once asked for.
  int64_t pieces[kPrefillMaxPieces + 1] = {};
  // Of the step at each share: a lower bound, and its time, 0 where not priced yet.
  std::vector<double> least_us, us;
};

// 64-key tiles that query tile t of a sequence of q queries and kv keys sees.
int key_tiles(int64_t kv, int64_t q, int64_t t, int64_t rows) {
  const int64_t end = kv - q + ((t + 1) * rows < q ? (t + 1) * rows : q);
  return (int)((end + kPrefillKeys - 1) / kPrefillKeys);
}

// Adds the query tiles of one sequence.
void add_tiles(PrefillEstimate& e, int64_t kv, int64_t q, int64_t rows) {
  auto sum = [&](int64_t height, int64_t& tiles, double& work) {
    const int64_t n = (q + height - 1) / height;
    tiles += n;
    if (n > kListTiles) {
      work += 0.5 * (double)n * ((double)key_tiles(kv, q, 0, height) + (double)key_tiles(kv, q, n - 1, height));
      return;
    }
    for (int64_t t = 0; t < n; ++t) work += key_tiles(kv, q, t, height);
  };
  if (q <= 0) return;
  sum(rows / 2, e.half_tiles, e.half_work);
  sum(rows, e.tiles, e.work);
  const int64_t n = (q + rows - 1) / rows;
  e.longest = std::max(e.longest, key_tiles(kv, q, n - 1, rows));
  if (e.tiles <= kListTiles)  // they are cleared where the batch has more
    for (int64_t t = 0; t < n; ++t) e.keys.push_back(key_tiles(kv, q, t, rows));
}

PrefillEstimate estimate_prefill(const int64_t* pages, const std::vector<int64_t>& queries, int tile_tokens) {
  PrefillEstimate e;
  for (size_t s = 0; s < queries.size(); ++s) add_tiles(e, pages[s] * kPageSize, queries[s], tile_tokens);
  if (e.tiles > kListTiles) e.keys.clear();
  std::sort(e.keys.begin(), e.keys.end(), std::greater<int>());
  return e;
}

// Query lengths are on the device.  Without a bound on them they are taken as
// evenly spread, no sequence having more queries than keys.
std::vector<int64_t> even_queries(const int64_t* pages, int64_t n, int64_t tokens) {
  double share = (double)tokens / (double)n, held = 0;
  int64_t longer = 0;
  for (int64_t s = 0; s < n; ++s) {
    const double kv = (double)pages[s] * kPageSize;
    if (kv < share) held += kv;
    else ++longer;
  }
  if (longer > 0) share = ((double)tokens - held) / (double)longer;
  std::vector<int64_t> q(n);
  for (int64_t s = 0; s < n; ++s) q[s] = std::min(pages[s] * kPageSize, (int64_t)(share + 0.999));
  return q;
}

// With a bound, all the work that `tokens` queries of at most max_query a
// sequence can be lies between two batches: the longest queries on the longest
// contexts, or on the shortest.
std::vector<int64_t> packed_queries(const int64_t* pages, int64_t n, int64_t tokens, int64_t max_query, bool longest) {
  std::vector<int64_t> order(n), q(n);
  for (int64_t s = 0; s < n; ++s) order[s] = s;
  std::sort(order.begin(), order.end(), [&](int64_t a, int64_t b) {
    return longest ? pages[a] > pages[b] : pages[a] < pages[b];
  });
  int64_t left = tokens;
  for (int64_t s = 0; s < n; ++s) left -= q[s] = pages[s] > 0 && left > 0 ? 1 : 0;
  for (int64_t s : order) {
    const int64_t more = std::max<int64_t>(std::min(left, std::min(max_query, pages[s] * kPageSize) - q[s]), 0);
    q[s] += more;
    left -= more;
  }
  return q;
}

// No prefill time on per_head workgroups per KV head is below this: the
// tiles' work in equal parts.
double least_prefill_us(const PrefillEstimate& e, int64_t per_head, int64_t max_tiles) {
  if (max_tiles > per_head)
    return kRoundsStartUs + (kRoundsKeyUs * e.work + kRoundsItemUs * (double)e.tiles) / (double)per_head;
  const double even = std::max(e.work / (double)per_head, (double)e.longest / kPrefillMaxPieces);
  return std::min(kWholeStartUs + kWholeKeyUs * e.longest, kCutStartUs + 2 * kCutPieceUs + kCutKeyUs * even);
}

// Time of the prefill part on per_head workgroups per KV head.
double prefill_part_us(PrefillEstimate& e, int64_t per_head, int64_t max_tiles, int num_kv_heads) {
  if (max_tiles > per_head) {
    const double even = (kRoundsKeyUs * e.work + kRoundsItemUs * (double)e.tiles) / (double)per_head;
    // j + 1 of the j * per_head + 1 longest tiles share a workgroup.
    double together = 0;
    for (int64_t j = 0; j * per_head < (int64_t)e.keys.size(); ++j)
      together = std::max(together, kTogetherUs * (double)(j + 1) * (e.keys[j * per_head] + kItemKeys));
    // Pieces in turns.
    if (plan_form(max_tiles, per_head) == PlanForm::kTurns && max_tiles <= kPrefillCutTiles)
      together = std::min(together, even + kTurnsCutUs);
    return kRoundsStartUs + std::max(even, together);
  }
  const int64_t limit = std::min<int64_t>(per_head, kPrefillPieceSlots / num_kv_heads);
  double best = kWholeStartUs + kWholeKeyUs * e.longest;
  for (int k = 2; k <= kPrefillMaxPieces; ++k) {
    const int len = e.longest > k ? (e.longest + k - 1) / k : 1;
    const double t = kCutStartUs + kCutPieceUs * k + kCutKeyUs * len;
    if (t >= best) continue;
    if (e.pieces[k] == 0)
      for (int keys : e.keys) e.pieces[k] += (keys + len - 1) / len;
    if (e.pieces[k] + e.spare <= limit) best = t;
  }
  return best;
}

// One MIXED step, and its time at a share of p workgroups per KV head.
struct MixedStep {
  double mb;  // decode K/V
  int64_t max_tiles;
  int num_kv_heads;
  int64_t num_cus;

  int64_t shares() const { return num_kv_heads < num_cus ? (num_cus - 1) / num_kv_heads : 1; }
  // With a prefill part of prefill_us; grows with it.
  double beside_us(int64_t p, double prefill_us) const {
    const int64_t left = num_cus - p * num_kv_heads;
    const double rate = kDecodeUsPerMB + kDecodeUsPerMBCu / (double)(left > 0 ? left : 1);
    const double decode_us = kDecodeStartUs + mb * std::max(rate, kDecodeMinUsPerMB);
    const double longer = std::max(decode_us, prefill_us), shorter = std::min(decode_us, prefill_us);
    return longer + kBeside * shorter * std::sqrt(shorter / longer);
  }
  // Prices e's lower bounds.
  void bound(PrefillEstimate& e) const {
    e.us.assign(shares() + 1, 0);
    e.least_us.assign(shares() + 1, 0);
    for (int64_t p = 1; p <= shares(); ++p) e.least_us[p] = beside_us(p, least_prefill_us(e, p, max_tiles));
  }
  double us(PrefillEstimate& e, int64_t p) const {
    if (e.us[p] == 0) e.us[p] = beside_us(p, prefill_part_us(e, p, max_tiles, num_kv_heads));
    return e.us[p];
  }
  // The lowest cost of any share, and the smallest share within kNear of it
  // (the decode part gains a little from more CUs where the estimate is level).
  // The share of the lowest bound is priced first, and most others fall to
  // theirs: at one KV head, 255 shares, pricing each cost 15 to 250 us a step.
  template <typename Cost, typename Least>
  double lowest(Cost cost, Least least, int64_t* share) const {
    constexpr double kNear = 1.01;
    int64_t first = 1;
    for (int64_t p = 2; p <= shares(); ++p)
      if (least(p) < least(first)) first = p;
    double best = cost(first);
    for (int64_t p = 1; p <= shares(); ++p)
      if (p != first && least(p) < best) best = std::min(best, cost(p));
    *share = 1;
    while (*share < shares() && (least(*share) > kNear * best || cost(*share) > kNear * best)) ++*share;
    return best;
  }
  double fastest(PrefillEstimate& e, int64_t* share) const {
    bound(e);
    return lowest([&](int64_t p) { return us(e, p); }, [&](int64_t p) { return e.least_us[p]; }, share);
  }
  // Little decode beside many short tiles: the 128-row tiles of
  // mva_paged_mixed, two to a CU, start sooner.  64 / 8 heads, 13 decodes of
  // 176 and 4 prompts of 426-604 tokens 38.9 against 41.1 us; longer tiles or
  // more decode run better on CUs of their own (32 / 8 heads, 4 chunks of 512
  // over up to 8k and 4 decodes 218 / 204 us, a 2048-token prompt and 10
  // decodes 66 / 60, 4 such prompts and 3 decodes 142 / 134).
  bool short_tiles(const PrefillEstimate& e, int64_t share, double step_us) const {
    return max_tiles > share && e.work < 8.0 * (double)e.tiles && mb * kDecodeMinUsPerMB < 0.1 * step_us;
  }
  // Time of mva_paged_mixed with its own decode plan.
  double one_launch_us(const PrefillEstimate& e, int64_t decode_seqs, int64_t decode_pages, int64_t max_decode_pages,
                       int group) const {
    const double per_cu = (double)num_kv_heads / (double)num_cus;
    const double waves = kMixedWavesPerCu * (double)num_cus;
    const double piece =
        std::min(std::max((double)decode_pages * num_kv_heads / (kPiecesPerWave * waves), 4.0), 128.0);
    const double chunks = std::ceil((double)max_decode_pages / piece);
    double decode = kOnePageUs * std::min(piece, (double)max_decode_pages);
    if (chunks > 1) decode += group * (kOnePassUs * std::ceil(chunks / 32.0) + kOneChunkUs * chunks);
    const double pieces =
        decode_seqs > 0 ? (double)decode_seqs * std::max(std::ceil((double)decode_pages / decode_seqs / piece), 1.0) : 0;
    const double prefill = kOneKeyUs * e.longest;
    const double work = per_cu * (kOneWorkUs * e.half_work + kOneTileUs * (double)e.half_tiles) + kOneMBUs * mb +
                        kOnePieceUs * pieces * num_kv_heads / waves;
    return kOneStartUs + std::sqrt(prefill * prefill + decode * decode + work * work);
  }
};

bool mixed_step(MixedStep& m, const int64_t* pages, int64_t n, int64_t tokens, int64_t decode_pages, int num_q_heads,
                int num_kv_heads, int64_t num_cus) {
  if (n < 0 || tokens < 0 || decode_pages < 0 || num_kv_heads <= 0 || num_q_heads <= 0 || num_q_heads % num_kv_heads ||
      num_q_heads / num_kv_heads > 16 || (n > 0 && pages == nullptr))
    return false;
  for (int64_t s = 0; s < n; ++s)
    if (pages[s] < 0 || pages[s] > 0x7fffffffLL) return false;
  m.mb = (double)decode_pages * kPageSize * num_kv_heads * kHeadDim * 2 * 2 * 1e-6;
  m.max_tiles = tokens / (kPrefillPPRows / (num_q_heads / num_kv_heads)) + n;
  m.num_kv_heads = num_kv_heads;
  m.num_cus = num_cus;
  return true;
}

}  // namespace

extern "C" int64_t mva_mixed_prefill_workgroups(const int64_t* prefill_pages, int64_t num_prefill_seqs,
                                                int64_t num_prefill_tokens, int64_t decode_pages, int num_q_heads,
                                                int num_kv_heads, int64_t num_cus) try {
  MixedStep m;
  if (!mixed_step(m, prefill_pages, num_prefill_seqs, num_prefill_tokens, decode_pages, num_q_heads, num_kv_heads,
                  num_cus))
    return -1;
  if (num_prefill_seqs == 0 || num_prefill_tokens == 0) return 0;
  PrefillEstimate e = estimate_prefill(prefill_pages, even_queries(prefill_pages, num_prefill_seqs, num_prefill_tokens),
                                       kPrefillPPRows / (num_q_heads / num_kv_heads));
  int64_t share;
  const double us = m.fastest(e, &share);
  return m.short_tiles(e, share, us) ? 0 : share * num_kv_heads;
} catch (const std::exception&) {  // out of memory
  return -1;
}

// The query lengths lie between two batches (packed_queries).  The share is the
// one that loses least, as a factor of the lowest time at any share: to a third
// over the worse of the two, to two thirds over evenly spread queries.
// Taken as evenly spread, a 2048-token prompt beside seven 8-token chunks over
// 8000 (32 / 8 heads, 64 decodes of 2000) got 208 CUs for its prefill and 300
// us, against 226 in mva_paged_mixed and 192 at the 168 CUs it gets now; the
// worse of the two alone gave the step of a 8192-token budget 96 CUs (939 us) in
// place of 88 (922).  And a step whose
// estimate is not below mva_paged_mixed's by kLaunchUs in either batch is left to
// that: steps of 15 to 25 us were 3 to 4 us slower on CUs of their own (the
// launch of the decode merges).  Over 1230 drawn steps 136 were slower than
// mva_paged_mixed by more than 3%, the worst by 84%; now 16, the worst by 14%,
// and the mean time is 3.4% lower; over 300 drawn after the fit 34 and 7.
extern "C" int64_t mva_mixed_prefill_share(const int64_t* prefill_pages, int64_t num_prefill_seqs,
                                           int64_t num_prefill_tokens, int64_t max_query_len, int64_t num_decode_seqs,
                                           int64_t decode_pages, int64_t max_decode_pages, int num_q_heads,
                                           int num_kv_heads, int64_t num_cus) try {
  constexpr double kLaunchUs = 1.0;
  MixedStep m;
  const int64_t n = num_prefill_seqs;
  if (!mixed_step(m, prefill_pages, n, num_prefill_tokens, decode_pages, num_q_heads, num_kv_heads, num_cus) ||
      max_query_len < 0 || num_decode_seqs < 0 || max_decode_pages < 0 || max_decode_pages > decode_pages)
    return -1;
  if (n == 0 || num_prefill_tokens == 0) return 0;
  const int group = num_q_heads / num_kv_heads;
  // A bound that the tokens do not fit under bounds nothing.
  if (max_query_len < (num_prefill_tokens + n - 1) / n) max_query_len = num_prefill_tokens;
  PrefillEstimate e[3];
  double best[3];
  const int bounds = n > 1 ? 2 : 1;
  int64_t share = 1;
  auto estimate = [&](int b, const std::vector<int64_t>& queries) {
    e[b] = estimate_prefill(prefill_pages, queries, kPrefillPPRows / group);
    e[b].spare = n > 1 ? (int)std::min<int64_t>(n, kPrefillPieceSlots) : 0;
    best[b] = m.fastest(e[b], &share);
  };
  for (int b = 0; b < bounds; ++b)
    estimate(b, packed_queries(prefill_pages, n, num_prefill_tokens, max_query_len, b == 0));
  if (bounds == 2) {
    estimate(2, even_queries(prefill_pages, n, num_prefill_tokens));
    auto lost = [&](auto us) { return 2 * us(2) / best[2] + std::max(us(0) / best[0], us(1) / best[1]); };
    m.lowest(
        [&](int64_t p) { return lost([&](int b) { return m.us(e[b], p); }); },
        [&](int64_t p) { return lost([&](int b) { return e[b].least_us[p]; }); }, &share);
  }
  for (int b = 0; b < bounds; ++b) {
    const double us = m.us(e[b], share);
    if (m.short_tiles(e[b], share, us) ||
        m.one_launch_us(e[b], num_decode_seqs, decode_pages, max_decode_pages, group) < us + kLaunchUs)
      return 0;
  }
  return share * num_kv_heads;
} catch (const std::exception&) {  // out of memory
  return -1;
}

extern "C" int mva_paged_mixed_run(const void* q, int64_t q_token_stride, int64_t q_head_stride,
                                   const void* k_cache, const void* v_cache, int64_t num_pages,
                                   int64_t page_stride, int64_t token_stride, const int32_t* block_tables,
                                   int64_t block_table_stride, const int32_t* seq_lens,
                                   const int32_t* query_start_loc, int64_t num_prefill_seqs, int64_t max_prefill_tiles,
                                   int64_t prefill_workgroups, void* prefill_workspace,
                                   int64_t prefill_workspace_bytes, int planned, const int32_t* decode_items,
                                   int64_t num_decode_items, int64_t num_decode_waves, const int32_t* wave_extra,
                                   const int32_t* merges, int64_t num_merges, int64_t num_part_slots, void* out,
                                   int64_t out_token_stride, int64_t out_head_stride, void* workspace,
                                   int64_t workspace_bytes, int num_q_heads, int num_kv_heads, int head_dim,
                                   int page_size, float softmax_scale, int dtype, void* stream) {
  PrefillParams pp;
  int rc = fill_prefill_params(pp, q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride,
                               token_stride, block_tables, block_table_stride, seq_lens, query_start_loc,
                               num_prefill_seqs, out, out_token_stride, out_head_stride, num_q_heads, num_kv_heads,
                               head_dim, page_size, softmax_scale);
  if (rc) return rc;
  if (dtype != kBF16 && dtype != kF16) return set_error("paged attention: dtype must be bf16 or fp16");
  if (num_decode_items > 0 && wave_extra == nullptr)
    return set_error("paged attention: a planned MIXED launch needs piece lists (wave_extra)");
  DecodeParams dp;
  rc = fill_decode_params(dp, q, q_token_stride, q_head_stride, k_cache, v_cache, num_pages, page_stride,
                          token_stride, block_tables, block_table_stride, seq_lens, decode_items, num_decode_items,
                          num_decode_waves, wave_extra, merges, num_merges, num_part_slots, out, out_token_stride,
                          out_head_stride, workspace, workspace_bytes, num_q_heads, num_kv_heads, head_dim, page_size,
                          softmax_scale);
  if (rc) return rc;
  const bool prefill = num_prefill_seqs > 0 && max_prefill_tiles > 0;
  hipStream_t s = (hipStream_t)stream;
  int64_t per_head = 0;
  if (prefill) {
    rc = check_prefill_plan(max_prefill_tiles, prefill_workspace, prefill_workspace_bytes, num_kv_heads);
    if (rc) return rc;
    if (prefill_workgroups <= 0 || prefill_workgroups % num_kv_heads)
      return set_error("paged attention: prefill_workgroups must be a positive multiple of num_kv_heads");
    per_head = prefill_workgroups / num_kv_heads;
  } else if (num_prefill_seqs > 0 && max_prefill_tiles < 0) {
    return set_error(kBadTileCapacity);
  }
  const int64_t n_decode_wgs =
      num_decode_items > 0 ? (num_decode_waves + kMixedDecodeWaves - 1) / kMixedDecodeWaves : 0;
  const int64_t grid = per_head * num_kv_heads + n_decode_wgs;
  // A launch has fewer than 2^32 threads.
  constexpr int64_t kMostWorkgroups = 0xffffffffLL / kPrefillPPThreads;
  if (prefill_workgroups > kMostWorkgroups || grid > kMostWorkgroups)
    return set_error("paged attention: too many work items");
  if (grid == 0) return 0;
  if (num_decode_items == 0) dp.num_waves = 0;
  // Without prefill sequences there is no plan: the fixed form ends after decode.
  const bool fixed = !prefill || max_prefill_tiles <= per_head;
  pp.tile_tokens = kPrefillPPRows / pp.group;
  int32_t* plan = (int32_t*)prefill_workspace;
  if (prefill && !planned) {
    rc = launch_prefill_plan(pp, num_prefill_seqs, max_prefill_tiles, plan, prefill_workspace_bytes, per_head, grid, s);
    if (rc) return rc;
  }
  const uint32_t np = (uint32_t)(per_head * num_kv_heads);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((uint32_t)grid), dim3(kPrefillPPThreads), 0, s, pp, plan, dp, np);
  };
  if (dtype == kBF16) {
    if (fixed) launch(paged_mixed_split_cus_kernel<__bf16, true>);
    else launch(paged_mixed_split_cus_kernel<__bf16, false>);
  } else {
    if (fixed) launch(paged_mixed_split_cus_kernel<_Float16, true>);
    else launch(paged_mixed_split_cus_kernel<_Float16, false>);
  }
  rc = check_launch("paged_mixed");
  if (rc) return rc;
  return launch_decode_merge(dp, merges, num_merges, num_part_slots, dtype, s);
}
