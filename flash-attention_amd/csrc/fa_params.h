// Kernel parameter blocks (passed by value to the kernels) and launcher entry points shared
// between the C-ABI front end and the kernel translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "fa_common.h"

namespace fa {

// Block-sparse activity, built on the device from the reference's converted block list
// (flash_blocksparse_attn_interface.py:8-40) by launch_build_sparse_maps(): the 16-row x 256-key block (rb, cb) is
// computed iff its bit is set.  Bit sets (bit j of 64-bit word w <-> block 64 w + j), so that a kernel holds what it
// needs in a register pair and re-reads memory only every 64 blocks.
struct SparseMaps {
  const uint64_t* rbits;  // [nrb][ncw]: 16-row block -> its active 256-key column blocks
  const uint64_t* qbits;  // [nqt][ncw]: forward query tile -> column blocks active for any of its row blocks
  const uint64_t* cbits;  // [ncb][nrw]: column block -> its active 16-row blocks
  int nrb;   // 16-row blocks  (= max_seqlen_q_rounded / 16)
  int ncb;   // 256-key blocks (= max_seqlen_k_rounded / 256)
  int nqt;   // forward query tiles
  int ncw;   // 64-bit words per row of rbits / qbits
  int nrw;   // 64-bit words per row of cbits
  // Row order (or null = 0, 1, 2, ...): a permutation of the 16-row blocks.  The forward and the dQ kernel give query tile t
  // the row blocks order[8 t .. 8 t + 7] (qbits is built for those), so that a caller who lists row blocks with similar key
  // blocks next to each other makes a workgroup stage few tiles that only one of its row blocks needs.  Not used under a
  // causal mask (the tile ranges there follow the rows' positions).
  const int32_t* order;
  int n_order;  // its entries, -1 for none (nrb without an order)
  // The key blocks, those with the most row blocks first (or null).  Where it is given the query tiles are in such an order, too (order and
  // qbits are), and workgroup ids enumerate ranks outermost, as under a causal mask: tiles differ in cost by a factor of two, and a launch that
  // ends on a dear one leaves a fifth of the compute units idle over its length.  us before / now, fp16, 16 queries x 256 keys blocks a
  // quarter full: 4 x 16 heads x 4096 forward 172 / 157, dQ 211 / 200, dK/dV 159 / 156; 8 x 12 x 1033 (bf16, 35 %) 38 / 28, 42 / 33,
  // 38 / 34; 256 x 256 blocks, 4 x 16 x 4096 121 / 110, 149 / 138, 194 / 176.  25 drawn shapes, step: 0.92 of the time, none above 1.012.
  const int32_t* corder;
};

// The two 16-row blocks of the 32-row slab `slab` (0 .. 3) of query tile qt: positions 8 qt + 2 slab and + 1 of the row
// order; -1 = none (past the last row block, or an entry that is not a row block).
FA_DEVICE void slab_row_blocks(const SparseMaps& sp, bool ordered, int qt, int slab, int* a, int* b) {
  const int pos = 8 * qt + 2 * slab;
  int ra = pos < sp.n_order ? pos : -1, rb = pos + 1 < sp.n_order ? pos + 1 : -1;
  if (ordered) {
    if (ra >= 0) ra = sp.order[pos];
    if (rb >= 0) rb = sp.order[pos + 1];
    if (ra >= sp.nrb) ra = -1;
    if (rb >= sp.nrb) rb = -1;
  }
  *a = __builtin_amdgcn_readfirstlane(ra);
  *b = __builtin_amdgcn_readfirstlane(rb);
}

// The lanes of a 32-row slab whose row block (of its two) is on: lane l owns row l % 32
FA_DEVICE uint64_t half_slab_lanes(bool a, bool b) {
  return (a ? 0x0000ffff0000ffffull : 0) | (b ? 0xffff0000ffff0000ull : 0);
}

// What is added to the scaled scores before the softmax (template parameter kBias of the kernels)
constexpr int kBiasNone = 0;    // nothing
constexpr int kBiasAlibi = 1;   // -slope[head] * |query - key| (alibi)
constexpr int kBiasTensor = 2;  // bias[b, h, query, key] (bias, strides in elements; batch and head stride may be 0)
constexpr int kPaddedRows = 3;  // nothing, and the rows are those of a padded batch (row_of; the forward kernel only)

struct FwdParams {
  const void* q;
  const void* k;
  const void* v;
  void* o;
  float* lse;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t q_rs, q_hs, k_rs, k_hs, v_rs, v_hs, o_rs, o_hs;  // strides in elements
  int B, H;
  int total_q, total_k;
  int max_sq, max_sk;  // caller's bounds on the sequence lengths; longer sequences are truncated to them
  int sq_r;  // rounded max_seqlen_q = innermost extent of lse
  int nq_tiles;
  int tile_group;    // causal launches: (batch, head) pairs of an XCD in flight together (map_tile); 0 = all; or kLongestFirst
  float scale;       // softmax_scale
  float scale_log2;  // softmax_scale * log2(e)
  float rp_keep;     // 1 / keep probability
  uint32_t keep_thr; // floor(keep * 65535)
  PhiloxKey pk;
  SparseMaps sp;
  // Key-split forward (few query tiles, many keys): split s of n_splits handles a contiguous share of the key tiles
  // and writes its normalised fp32 output and its lse to o_part [n_splits, total_q, H, d] / lse_part
  // [n_splits, B, H, sq_r]; fwd_combine_kernel merges them into o / lse.  n_splits <= 1: single pass.
  int n_splits;
  int split_keys;  // fa_decode_kernel: keys per split (a multiple of its waves' 32-key tiles); 0: shares of fa_fwd_kernel's tiles
  float* o_part;
  float* lse_part;
  const float* alibi;  // null, or one slope per head: the score of (query i, key j) gets -slope * |i - j| added
  const void* bias;    // null, or a tensor of the element type added to the scaled scores: [b, h, query, key]
  int64_t bias_bs, bias_hs, bias_rs;  // its batch, head (0: shared) and row strides in elements; keys are contiguous
  // Rotary position embedding of the queries inside the kernel (null: none): cos / sin tables [rot_rows, head_dim / 2] of
  // the element type; the row at position i of its sequence is turned by table row i when its Q fragment is loaded (the
  // keys come in rotated: their tiles go to LDS without passing through registers).  q_rot: null, or where the rotated
  // queries are left for the backward ([total_q, H, d], strides in elements).
  const void* rot_cos;
  const void* rot_sin;
  int rot_rows;
  void* q_rot;
  int64_t qr_rs, qr_hs;
  // Dropout keep words (fa_common.h), or null: the keep decisions of every score, left for the backward
  uint32_t* keep_words;
  int kw_q;   // query extent of the buffer (max_seqlen_q rounded up to 128)
  int kw_kb;  // 32-key blocks (max_seqlen_k rounded up to 128, / 32)
  // Padded batch (the forward's kPaddedRows variants; null: packed sequences), as launch_padding_rows() leaves them: entry b's tokens are the rows
  // b * max_sq + row_of[b * max_sq + i], i < row_info[4 b]; the rest of row_of's slice lists its padding rows
  const int32_t* row_of;
  const int32_t* row_info;
};

// What launch_padding_rows() leaves per batch entry in row_info: number of tokens, first token's position, 1 if they are consecutive
constexpr int kRowInfo = 4;

struct DumpParams {  // return_softmax path
  const void* q;
  const void* k;
  const float* lse;
  void* s;  // [B, H, sq_r, sk_r]
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t q_rs, q_hs, k_rs, k_hs;
  int B, H, D;
  int total_q, total_k;
  int max_sq, max_sk;
  int sq_r, sk_r;
  float scale;
  int causal, dropout, sparse;
  uint32_t keep_thr;
  PhiloxKey pk;
  SparseMaps sp;
  const float* alibi;
  const void* bias;  // as in FwdParams
  int64_t bias_bs, bias_hs, bias_rs;
};

struct BwdParams {
  const void* dout;
  const void* q;
  const void* k;
  const void* v;
  const void* out;
  const float* lse;
  float* dsoftmax;  // softmax_d [B, H, sq_r]
  void* dq;
  void* dk;
  void* dv;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t do_rs, do_hs, q_rs, q_hs, k_rs, k_hs, v_rs, v_hs, o_rs, o_hs;
  int64_t dq_rs, dq_hs, dk_rs, dk_hs, dv_rs, dv_hs;
  int B, H;
  int total_q, total_k;
  int max_sq, max_sk;
  int sq_r;        // innermost extent of dsoftmax
  int lse_stride;  // innermost extent of lse
  int nk_tiles;      // key tiles of the dK/dV kernel
  int merged_dkdv_blocks, merged_nq_tiles;  // fa_bwd_merged_kernel: its dK/dV workgroups come first; query tiles of the dQ part
  int nq_tiles;      // query tiles of the dQ kernel
  int tile_group;    // causal launches: (batch, head) pairs of an XCD in flight together (map_tile); 0 = all; or kLongestFirst
  float scale;
  float scale_log2;
  float p_keep;
  float rp_keep;
  uint32_t keep_thr;
  PhiloxKey pk;
  SparseMaps sp;
  // Key-split dQ (one query tile, many keys; see FwdParams): split s of n_splits walks its share of the key tiles and
  // writes its scaled fp32 partial dQ to dq_part [n_splits, total_q, H, d]; dq_combine_kernel sums them into dq.
  int n_splits;
  float* dq_part;
  const float* alibi;  // as in FwdParams
  const void* bias;    // as in FwdParams
  int64_t bias_bs, bias_hs, bias_rs;
  void* dbias;         // null, or where the dK/dV kernel leaves d(loss)/d(bias) = dS / keep: [b, h, query, key], written for the queries and
  int64_t dbias_bs, dbias_hs, dbias_rs;  // keys a sequence has (causal: up to the diagonal; block layout: listed blocks); the rest is left as it is
  // Rotary position embedding (as in FwdParams; null: none): q and k are the rotated tensors, and dq and dk are turned back
  // by the opposite angles in the kernels' epilogues, before they are rounded
  const void* rot_cos;
  const void* rot_sin;
  int rot_rows;
  // Dropout keep words (fa_common.h) as the forward left them, or null: read by both kernels in place of Philox
  const uint32_t* keep_words;
  int kw_q;   // query extent of the buffer (max_seqlen_q rounded up to 128)
  int kw_kb;  // 32-key blocks (max_seqlen_k rounded up to 128, / 32)
  // One-kernel backward (fa_bwd_fused_kernel.h): fp32 running sums of dQ [B * H, nqt_ring tiles, 2048] and their hand-over
  // counters [B * H, nqt_ring, 4]
  float* dq_acc;
  int* dq_flags;
  int nqt_ring;     // query tiles of max_seqlen_q
  int ring_stride;  // tiles between the starting points of consecutive key tiles (0: the kernel's default)
};

// Sequence extent of batch entry b, clamped so that a cu_seqlens array that disagrees with the declared
// totals or maxima can never index outside the tensors: returns false if the entry must be skipped.
FA_DEVICE bool seq_extent(const int32_t* cu, int b, int total, int max_len, int* begin, int* len) {
  const int s = cu[b], e = cu[b + 1];
  int n = e - s;
  if (s < 0 || n <= 0 || e > total) return false;
  *begin = s;
  *len = n < max_len ? n : max_len;
  return true;
}

// Ragged batches: workgroup ids enumerate the batch entries longest first.  A launch deals its workgroups out in id order;
// the entries with the longest walks should be under way first and - in a grid that is resident all at once - spread over
// the compute units instead of arriving together as some units' third workgroup.  Slot `slot` of the launch's batch
// dimension therefore goes to the entry with the slot-th largest length in cu (ties: lower index first, so a batch of
// equal lengths keeps its order).  Every wave finds the entry itself: lane i holds entry i's length, counts the entries
// that precede it (one readlane and compare per entry), and the lane whose count is `slot` is the answer.  Batches of
// more than 64 entries keep their order.  The search costs every workgroup's prologue a few instructions per batch entry,
// so the launchers ask for it (tile_group == kLongestFirst in a launch without a mask) only for grids that are resident all at once
// (longest_first_launch), where the spreading is what it buys.
// (info: the lengths stand in row_info instead, see FwdParams)
FA_DEVICE int longest_first(const int32_t* cu, int B, int slot, const int32_t* info = nullptr) {
  if (B > 64 || B < 2) return slot;
  const int lane = threadIdx.x & 63;
  const int i = lane < B ? lane : B - 1;
  const int len = info ? info[kRowInfo * i] : cu[i + 1] - cu[i];
  int before = 0;
  for (int j = 0; j < B; j++) {
    const int lj = __builtin_amdgcn_readlane(len, j);
    before += (lj > len || (lj == len && j < lane)) ? 1 : 0;
  }
  const uint64_t hit = __builtin_amdgcn_ballot_w64(lane < B && before == slot);
  return __builtin_amdgcn_readfirstlane(hit != 0 ? (int)__builtin_ctzll(hit) : slot);
}

// Workgroup id -> (batch*head, tile rank).  The hardware deals consecutive workgroup ids to the 8 XCDs in turn
// (id % 8), and each XCD has its own L2.
//   kTileMajor = false (tiles of equal cost): the tiles of one (batch, head) are consecutive in one XCD's share of the
//     ids, so they run on one XCD at about the same time and share its L2 copy of the streamed operand.
//   kTileMajor = true (causal: tile cost grows with the rank reversed): ids enumerate tile ranks outermost, so the
//     most expensive tiles of all (batch, head) pairs start first; batch*head is padded to a multiple of 8 so that a
//     given (batch, head) still always lands on the same XCD.
template <bool kTileMajor>
FA_DEVICE bool map_tile(int block, int tiles_per_bh, int BH, int* bh, int* rank, int group = 0) {
  if (kTileMajor) {
    const int bhp = (BH + 7) & ~7;
    const int P = bhp >> 3;  // (batch, head) pairs per XCD
    if (group > 0 && group < P) {
      // Long sequences: an XCD that streams the K and V of all its pairs at once reads them from memory again for every
      // query tile (they exceed its L2 many times over).  The pairs of an XCD are therefore taken `group` at a time -
      // ranks outermost inside a group, the groups one after the other - so that what is in flight shares a few pairs' keys.
      const int x = block & 7, j = block >> 3;
      const int g = j / (group * tiles_per_bh);
      const int r = j - g * group * tiles_per_bh;
      const int members = P - g * group < group ? P - g * group : group;
      *rank = r / members;
      *bh = x + 8 * (g * group + (r - *rank * members));
      return *bh < BH && *rank < tiles_per_bh;
    }
    // A grid small enough to be resident all at once (up to 4 workgroups on each of the 256 compute units) is dealt
    // out in one go, compute unit c getting ids c, c + 256, ...: then every odd group of 256 ids is walked backwards
    // (in steps of 8, so that id % 8 is kept), and a compute unit that got one of the dearest tiles of a group gets
    // one of the cheapest of the next.  Larger grids are scheduled as workgroups retire; plain dearest-first is best.
    const int grp = block >> 8;
    if ((grp & 1) && bhp * tiles_per_bh <= 1024) {
      const int left = bhp * tiles_per_bh - (grp << 8);
      const int size8 = (left < 256 ? left : 256) >> 3;
      const int pos = block & 255;
      block = (grp << 8) + ((size8 - 1 - (pos >> 3)) << 3) + (pos & 7);
    }
    *rank = block / bhp;
    *bh = block - *rank * bhp;
    return *bh < BH && *rank < tiles_per_bh;
  }
  // XCD x takes the (batch, head) pairs x, x + 8, x + 16, ... and all their tiles: the heads of one batch entry - which
  // share its sequence length - are spread over the XCDs, so a ragged batch loads the XCDs evenly
  // The tile ranks are rotated from one pair to the next: the hardware deals consecutive ids of an XCD to its compute
  // units in turn, so with a power-of-two tile count a compute unit would always get the same rank - and in a ragged
  // batch the last ranks are the ones that often lie beyond a sequence's end.
  const int j = block >> 3;
  const int q = j / tiles_per_bh;
  *bh = (block & 7) + 8 * q;
  *rank = (j - q * tiles_per_bh + q) % tiles_per_bh;
  return *bh < BH;
}
// Ragged batches (the kernels' kLive variants): workgroup ids enumerate the tiles that hold rows, the dearest first, and behind them the ones
// that hold none.  The other two orders deal out (pair, rank) slots as if every sequence were the longest: the slots past a shorter one's end
// exit at once, but the dispatcher gives the ids of an XCD to its shader engines strictly in turn, so where the live slots recur with a
// period of 2 or 4 half of the compute units hold every live workgroup and the rest stand idle until the ids have passed (4 x 16 heads x 600 ..
// 3001, d = 128, causal: 65 of 100 us); and the longest walks come where their pair comes.  us of the kernels in the other orders / here, same
// bits: forward 4 x 16 x 600 .. 3001 d = 128 causal 102 / 90, 4 x 12 x 1800 .. 6000 d = 64 causal 186 / 146 (backward 567 / 438), 12 x 12 x 214 ..
// 550 15.9 / 13.5, 64 x 8 x 36 .. 129 13.6 / 7.7; backward 7 x 12 x 1051 .. 2132 d = 128 causal 321 / 250, 57 x 8 x 55 .. 139 41.2 / 22.2.
//
// Lane i of a wave holds batch entry i (at most 64).  Every tile falls into one of 64 buckets, bucket 0 the dearest; a histogram in LDS and a
// prefix sum over it find the bucket that a workgroup id falls into, and a prefix sum over the entries the tile in it: some 0.4 us, whatever
// the batch (ranking the entries by readlanes took 1.5 us at 64 of them).
//   kByTile (causal): cost grows with the tile's distance from the cheap end (its level); bucket = level, a lane's weight its pairs on this XCD;
//   otherwise: bucket = length of the walk (cu_walk: the side that a tile walks over), weight = pairs x tiles, a pair's tiles one after the other.
// The pairs of an entry go to the XCDs in turn and stay there.  Where the heads are no multiple of 8, the entries (up to 16) take their turns
// longest first, so that neighbours in length share the rounding.
// A launch that is resident all at once (at most four workgroups on each of an XCD's 32 compute units, which get ids in turn) walks every other
// group of 32 backwards: the unit with the dearest of one group gets the cheapest of the next.
// info: null, or the lengths of a padded batch (FwdParams::row_info), whose `tiles` tiles a pair are all visited (rows to be zeroed).
// lds_wave: 256 bytes of the wave's own.
constexpr int kLongestFirst = -1;
struct TileId {
  int b, h, tile;
  int own_begin, own_len, walk_begin, walk_len;  // as seq_extent has them (walk: 0 keys or queries where it skips the entry)
};
FA_DEVICE int wave_prefix_sum(int x) {  // inclusive
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}
template <bool kByTile>
FA_DEVICE bool map_live(int block, const int32_t* cu_own, int total_own, int max_own, const int32_t* cu_walk, int total_walk, int max_walk, int rows,
                        int tiles, bool cheap_last, int B, int H, const int32_t* info, void* lds_wave, TileId* id) {
  const int lane = threadIdx.x & 63;
  const int i = lane < B ? lane : B - 1;
  int begin = 0, n, walk_begin = 0, walk;
  if (info) {
    n = walk = info[kRowInfo * i];
  } else {
    begin = cu_own[i];
    walk_begin = cu_walk[i];
    const int e = cu_own[i + 1], we = cu_walk[i + 1];
    n = e - begin;
    if (begin < 0 || n <= 0 || e > total_own) n = 0;
    n = n < max_own ? n : max_own;
    walk = we - walk_begin;
    if (walk_begin < 0 || walk <= 0 || we > total_walk) walk = 0;
    walk = walk < max_walk ? walk : max_walk;
  }
  const int x = block & 7;
  int j = block >> 3;
  const int t = (int)(((uint32_t)n + rows - 1) / (uint32_t)rows);
  int turn = i;
  if ((H & 7) != 0 && B <= 16) {
    const int key = walk << 4 | (15 - (i & 15));
    turn = 0;
    for (int e = 0; e < B; e++) turn += __builtin_amdgcn_readlane(key, e) > key ? 1 : 0;
  }
  // this XCD's pairs of entry i: heads h0, h0 + 8, ...
  const int h0 = (x - turn * H) & 7, cnt = lane < B ? (H + 7 - h0) >> 3 : 0;
  const int weight = kByTile ? cnt : cnt * t;
  const int bucket = kByTile ? 64 - t : 63 - (int)((float)walk * (63.5f / (float)max_walk));  // 0: the dearest
  volatile FA_LDS int* const hist = (volatile FA_LDS int*)lds_wave;
  hist[lane] = 0;
  if (t > 0) __hip_atomic_fetch_add((FA_LDS int*)lds_wave + bucket, weight, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  int size = hist[lane];
  if (kByTile) size = wave_prefix_sum(size);  // pairs that reach level 63 - lane
  const int end = wave_prefix_sum(size);
  const int live = __builtin_amdgcn_readlane(end, 63);
  if (j >= live) {
    if (!info) return false;
    j -= live;
    const int rest = (tiles - t) * cnt, rest_end = wave_prefix_sum(rest);
    const uint64_t hit = __builtin_amdgcn_ballot_w64(rest_end > j);
    if (hit == 0) return false;
    const int k = (int)__builtin_ctzll(hit);
    const uint32_t r = (uint32_t)(j - (__builtin_amdgcn_readlane(rest_end, k) - __builtin_amdgcn_readlane(rest, k)));
    const int tk = __builtin_amdgcn_readlane(t, k);
    const uint32_t per = (uint32_t)(tiles - tk), q = r / per;
    id->tile = tk + (int)(r - q * per);
    id->h = __builtin_amdgcn_readlane(h0, k) + 8 * (int)q;
    id->b = k;
  } else {
    if (live <= 4 * 32 && (j & 32)) {
      const int left = live - (j & ~31);
      j = (j & ~31) + (left < 32 ? left : 32) - 1 - (j & 31);
    }
    const int l = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(end > j));
    int r = j - (__builtin_amdgcn_readlane(end, l) - __builtin_amdgcn_readlane(size, l));
    const int mine = (kByTile ? bucket <= l : bucket == l) && t > 0 ? weight : 0;
    const int mine_end = wave_prefix_sum(mine);
    const int k = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(mine_end > r));
    r -= __builtin_amdgcn_readlane(mine_end, k) - __builtin_amdgcn_readlane(mine, k);
    const uint32_t tk = (uint32_t)__builtin_amdgcn_readlane(t, k);
    uint32_t q = (uint32_t)r;
    if (kByTile) {
      id->tile = cheap_last ? (int)tk - 64 + l : 63 - l;
    } else {
      q = (uint32_t)r / tk;
      id->tile = (int)((uint32_t)r - q * tk);
    }
    id->h = __builtin_amdgcn_readlane(h0, k) + 8 * (int)q;
    id->b = k;
  }
  id->own_begin = __builtin_amdgcn_readlane(begin, id->b);
  id->own_len = __builtin_amdgcn_readlane(n, id->b);
  id->walk_begin = __builtin_amdgcn_readlane(walk_begin, id->b);
  id->walk_len = __builtin_amdgcn_readlane(walk, id->b);
  return true;
}
// Who takes it: dense launches of at most 64 batch entries (lanes) and 64 tiles a pair (buckets) whose lengths differ, at most 0.95 of batch x
// longest being tokens; below that nothing is gained and the prologue costs up to 2 %.
// - Without a mask all of them (0.54 to 1.04 of the time over 100 drawn shapes, 0.92 in the middle), but dQ and dK/dV in one launch only
//   where it is not resident at once: 3 x 12 x 414 .. 910 35.3 / 38.8, 2 x 16 x 728 .. 1234 48.1 / 51.7; 8 x 12 x 256 .. 512 33.4 / 31.8.
// - Under a causal mask the other orders have their empty slots at one end.  The forward and dQ take it where at most nine tenths of the slots hold
//   rows (38 x 16 x 414 .. 628 46.1 / 48.8), eight tenths at d = 128 without groups (forward 4 x 8 x 1836 .. 2384 61.3 / 63.8, 8 x 8 x 932 .. 1195 35.4 / 37.1;
//   backward 8 x 5 x 773 .. 920 67.5 / 70.3), of more than 256-token sequences (64 x 8 x 42 .. 109 7.9 / 8.2, 64 x 16 x 172 .. 202 d = 128 42.4 / 44.7),
//   in more workgroups with rows than `least`, below which the longer prologue is all there is: forward d = 64 4 x 12 x 344 .. 400 (163 of them) 8.1 / 8.5,
//   d = 16 12 x 3 x 631 .. 1147 (268) 10.7 / 11.2, d = 32 6 x 5 x 750 .. 1056 (226) 10.6 / 11.3, 8 x 12 x 181 .. 464 (290) 7.5 / 7.9; backward d = 32 2 x 12 x
//   1362 .. 2671 (390) 69.5 / 73.5, d = 128 12 x 3 x 385 .. 593 (155) 48.3 / 49.4; and not half-size tiles of the d = 64 forward from 640 on, over a round
//   of what is resident at once, but for long walks (12 x 12 x 204 .. 928 18.9 / 20.6, 5 x 24 x 268 .. 1115 19.2 / 20.6, 3 x 24 x 578 .. 1864 28.8 / 31.2;
//   2 x 24 x 471 .. 3139 51.5 / 45.5).  Over 900 drawn shapes without groups a forward takes 0.95 (d = 16 to 64), 0.99 (128), at most 1.06, a backward 0.99, at
//   most 1.06.  dK/dV, whose empty slots come last, takes it where its pairs are taken in groups
//   (causal_tile_group; 3 x 16 x 2821 .. 5841 dQ alone 481, both 441; 14 x 16 x 471 .. 703, no groups, 82.0 / 86.1) of more than 640 tokens (backward
//   d = 128 48 x 12 x 183 .. 262 90.2 / 94.3, 48 x 12 x 226 .. 452 164.8 / 170.2, d = 64 64 x 24 x 147 .. 587 261 / 270; up to 8 % given up where one of the
//   sequences is long, 16 x 16 x 82 .. 631 89.3 / 82.0).  At d = 32 many
//   pairs in groups stay with them, whose K and V it would read again: 64 x 16 x 509 .. 926 100.9 / 122.5, 38 x 12 x 353 .. 1766 91.2 / 101.2;
//   and so does what live_order_rereads names.
//
// Under a causal mask the live order has all of an XCD's pairs in flight and reads their K and V (dK/dV: Q and dO) past its L2 for every level; the
// other one takes them in groups that fit.  The more pairs share the L2 and the more the batch holds beyond the 256 MB of the memory-side cache,
// the more that costs, and the fuller the slots, the less the empty ones did.  Lines through the times of 1238 grouped shapes (d = 16 .. 128, 2 to
// 64 entries, 270 .. 7986 tokens, shortest 0.2 .. 0.9 of the longest).  Over 900 others a step's kernels take 0.92 (d = 64), 0.91 (128), 0.98 (32) of the
// groups' time, at most 1.03, and over 500 a forward alone 0.93, 0.93 and 0.98, at most 1.06; the live order regardless 0.93, 0.92, 0.99, at most
// 1.24, and 0.95, 0.97, 1.01, at most 1.51.
// us in groups / live: forward d = 128 64 x 16 x 614 .. 1024 286 / 409, 32 x 16 x 1229 .. 2048 459 / 541, 28 x 12 x 938 .. 1537 183 / 196, 16 x 8 x 1229 .. 4096 (live) 366 / 271, d = 64
// 64 x 16 x 1229 .. 2048 509 / 640, 63 x 8 x 1970 .. 2463 383 / 444, 32 x 16 x 614 .. 2048 (live) 215 / 192, d = 32 20 x 12 x 2458 .. 4096 281 / 366; dQ d = 64
// 64 x 16 x 1229 .. 2048 699 / 822, d = 128 41 x 16 x 1650 .. 2261 1142 / 1443, 64 x 12 x 416 .. 520 (live) 185 / 159; dK/dV d = 64 36 x 16 x 1785 .. 3719 1299 / 1407.
enum LiveKernel { kLiveFwd, kLiveDq, kLiveDkdv, kLiveMerged };
inline bool live_order_rereads(LiveKernel kernel, int head_dim, int64_t live, int64_t slots, int B, int H, int total) {
  const bool fwd = kernel == kLiveFwd, dq = kernel == kLiveDq;
  const double mb = (double)total * H * head_dim * 4 / (1 << 20), pairs = (B * H + 7) / 8;
  if (!fwd && head_dim >= 64 && mb <= 256) return false;
  const double most = head_dim == 16 ? (fwd || dq ? 1.5 : 2.0) : head_dim == 32 ? (fwd || dq ? 1.86 : 2.32)
                      : fwd ? (head_dim == 64 ? 2.28 : 2.16) : dq || head_dim == 64 ? 2.3 : 2.48;
  return (double)live / slots + 0.08 * std::log2(pairs * pairs * mb) > most;
}
inline bool live_order_launch(LiveKernel kernel, int head_dim, bool causal, int B, int H, int total, int max_s, int n_splits, int tiles, int tile_group,
                              int grid) {
  if (n_splits > 1 || B > 64 || tiles > 64 || (int64_t)total * 20 > (int64_t)19 * B * max_s) return false;
  if (kernel == kLiveMerged) return !causal && grid > 1024;
  if (!causal) return true;
  if (kernel == kLiveDkdv && (tile_group <= 0 || max_s <= 640)) return false;
  if (head_dim <= 32 && tile_group > 0 && B * H >= 256) return false;
  const int64_t live = (int64_t)H * (total + (int64_t)64 * B) / 128, slots = (int64_t)B * H * ((max_s + 127) / 128);
  if (tile_group > 0 && live_order_rereads(kernel, head_dim, live, slots, B, H, total)) return false;
  const bool fwd = kernel == kLiveFwd, half_size = tiles > (max_s + 127) / 128;
  const int least = fwd ? (head_dim == 16 ? 300 : head_dim == 32 ? 330 : 200) : head_dim == 32 ? 450 : head_dim == 128 ? 200 : 150;
  if (tile_group <= 0 && fwd && head_dim == 64 && half_size && live >= 640 && max_s < 2000) return false;
  return max_s > 256 && live > least && 10 * live <= (tile_group <= 0 && head_dim == 128 ? 8 : 9) * slots;
}
inline bool live_order_rows(int B, int tiles) { return B <= 64 && tiles <= 64; }
// The forward over a padded batch, whose number of tokens is not known here (map_live's info).  Without a mask wherever there is more than one entry to
// order (one: 12.5 / 12.7 us at 12 heads x 860, 17.3 / 17.7 at 5 x 1865; over 300 others at most 1.01 of the slot order's time, 0.95 in the mean).  Under a
// causal mask from two workgroups a compute unit on (16 x 3 heads x 172 6.4 / 7.0 us, 14 x 12 x 300 9.8 / 10.2), and not where its pairs, all in
// flight, read their K and V past the L2 (live_order_rereads, here by the rows there may be): all rows tokens, d = 64 64 x 16 x 2048 728 / 1028 us,
// 32 x 24 x 2197 654 / 839, 16 x 16 x 4096 (live) 688 / 674, d = 32 36 x 16 x 3218 718 / 983, 33 x 8 x 4321 543 / 661, d = 16 44 x 8 x 5687 1129 / 1459,
// 40 x 16 x 533 42.9 / 45.8.  700 drawn shapes: 0.94 (d = 64), 0.98 (32, 16), at most 1.01; given up where many rows are padding (32 x 16 x 2048, 30 %
// to all tokens, 231 / 203).
inline bool live_order_padded(int head_dim, bool causal, int B, int H, int max_s, int tiles) {
  if (!live_order_rows(B, tiles)) return false;
  if (!causal) return B > 1;
  const double mb = (double)B * max_s * H * head_dim * 4 / (1 << 20), pairs = (B * H + 7) / 8;
  return (int64_t)B * H * ((max_s + 127) / 128) >= 512 && pairs * pairs * mb <= (head_dim <= 16 ? 16384 : head_dim == 32 ? 32768 : 440000);
}
inline int tile_grid(bool tile_major, int tiles_per_bh, int BH) {
  return ((BH + 7) & ~7) * tiles_per_bh;
}
// see longest_first: dense launches without a mask whose grid is resident all at once (at most 4 workgroups on each of the
// 256 compute units), 2 to 64 batch entries
inline bool longest_first_launch(bool causal, bool sparse, int grid, int B) {
  return !causal && !sparse && grid <= 1024 && B >= 2 && B <= 64;
}

// Launch shape: with 128-row tiles a short-sequence batch gives the compute units one or two workgroups each, and one
// workgroup's walk over its keys is the launch's critical path; the forward and the dQ kernel then run their half-size
// tile variants (64 query rows, wave pairs split the keys: twice the workgroups, half the serial work of each).  The rule is
// read off a sweep over batch size, sequence length, mask and dropout (bench.py --tile-sweep): with x = full-size
// workgroups per compute unit,
//   forward: half-size for x < 2 (more than one key tile pair to split: sequences beyond 128), and up to x < 3 with dropout
//            (whose Philox work makes the serial walk longer);
//   dQ:      half-size for 1 <= x < 2 under a causal mask or with dropout.
// Where lengths differ, many launched workgroups find no rows: the rules that follow this one (causal forward, head dim 128, dQ without
// dropout, the backward in one launch) count those that do, and this one stays for the others.
// launch_policy() & 3: 0 = by this rule, 1 = always the full-size tiles, 2 = the half-size tiles wherever they exist
// (fa_set_launch_policy; the parity tests run both shapes on the same inputs).
int launch_policy();
// About the workgroups of 128 query rows that find any: a sequence of n has n / 128 and half a tile more on average
inline int64_t live_row_tiles(int nheads, int total_q, int batch) { return (int64_t)nheads * (total_q + (int64_t)64 * batch) / 128; }
// Pairs go to the 8 XCDs in turn (map_tile): of `live` workgroups, eight times what the fullest XCD gets (12 pairs load like 16)
inline int64_t fullest_xcd(int64_t live, int BH) { return live * ((BH + 7) / 8 * 8) / BH; }
constexpr int kSmallLaunchFwd = 0, kSmallLaunchDq = 1;
inline bool small_launch(int kernel, int BH, int max_s, bool causal, bool dropout) {
  const int policy = launch_policy() & 3;
  if (policy != 0) return policy == 2;
  const int64_t wgs = (int64_t)BH * ((max_s + 127) / 128);  // x = wgs / 256 compute units
  if (kernel == kSmallLaunchFwd) return max_s > 128 && (wgs < 2 * 256 || (dropout && wgs < 3 * 256));
  return wgs >= 256 && wgs < 2 * 256 && (causal || dropout);
}

// The forward at head dim 16 to 64 under a causal mask without dropout, longest sequence beyond 256: by the workgroups that find query rows
// instead of the launched ones, half-size below 600 and, where the lengths differ (at most 0.85 of batch x longest are tokens: the last tiles of
// the longest sequences decide), below 1000.  us of full-size / half-size tiles, fp16 and bf16, d = 64 (d = 16 and 32 alike): 3 x 8 x 2700 ..
// 3479 (528 workgroups, 672 launched) 55.6 / 44.1, 6 x 12 x 260 .. 1631 (564, 936) 31.4 / 24.9, 3 x 12 x 1823 (540) 33.6 / 29.5, 16 x 8 x 480 .. 1200 (896,
// 1280) 34.9 / 26.8, 3 x 12 x 1400 .. 2829 (624) 49.7 / 40.8; equal lengths 4 x 12 x 1700 (672) 32.3 / 33.0, 4 x 12 x 2300 (864) 47.8 / 51.2; uneven beyond
// 3 x 16 x 2100 .. 3348 (1056) 69.5 / 69.8, 16 x 16 x 1262 (2112) 63.6 / 69.9.  At d = 64 shorter walks cross sooner (on the fullest XCD): 16 x 12 x 329
// (589) 11.7 / 12.9, 11 x 16 x 355 (576) 11.5 / 12.4, 8 x 16 x 527 (591) 14.1 / 15.3, 7 x 12 x 838 (619) 19.7 / 21.1; uneven 21 x 12 x 290 (602) 11.4 / 12.9.
inline bool small_launch_causal(int head_dim, int64_t live, int BH, int max_s, int64_t total_q, int batch) {
  if ((launch_policy() & 3) != 0 || max_s <= 256) return small_launch(kSmallLaunchFwd, BH, max_s, true, false);
  const bool uneven = total_q * 20 <= (int64_t)17 * batch * max_s;
  if (head_dim == 64 && max_s <= 1000 && !(uneven && max_s > 400)) {
    const int64_t x = fullest_xcd(live, BH);
    return live < 600 && x <= (uneven || max_s > 640 ? 580 : max_s > 400 ? 560 : max_s > 320 ? 540 : 520);
  }
  return live < 600 || (live < 1000 && uneven);
}

// The forward's half-size tiles at head dim 128 (64-key tiles, 64 KB of LDS: two workgroups a compute unit), for launches whose time is one
// workgroup's walk over the keys.  By the workgroups that find query rows (live_row_tiles), on the fullest XCD (x below), and the longest
// sequence: the longer the walk, the more of them may share the chip.  us of full-size / half-size tiles, fp16 and bf16.  Causal: 8 x 2300 53.9
// / 35.8, 16 x 3100 (x = 400) 72.7 / 58.0, 4 x 12 x 360 .. 1200 (312) 32.7 / 24.8, 4 x 16 x 1200 (640) 40.7 / 43.5; 8 x 12 x 386 (317) 15.7 / 17.0, 10 x 8 x 405
// (293) 15.5 / 15.9, 5 x 16 x 518 (363) 18.4 / 18.9; 8 x 16 x 281 (345) 12.8 / 15.7, 10 x 12 x 250 .. 337 (339) 14.9 / 17.4, 10 x 12 x 190 .. 287 (283) 12.0 /
// 13.5, 4 x 16 x 300 (182) 11.9 / 11.0, 6 x 16 x 182 (184) 9.1 / 9.3, 16 x 12 x 52 .. 130 (204) 8.7 / 9.3.  No mask: 8 x 1700 39.3 / 28.1, 8 x 2300
// (148) 50.1 / 45.1, 3 x 16 x 286 (131) 10.8 / 10.0, 6 x 8 x 323 (145) 12.4 / 13.9, 4 x 8 x 531 (148) 16.2 / 17.1, 4 x 12 x 500 (192) 16.3 / 17.2.
// With rotary, which every workgroup's prologue pays for, they cross sooner: causal 12 x 8 x 150 .. 197 (x = 177) 12.0 / 14.4, 6 x 16 x 276 (255) 15.4 / 16.4; no
// mask 9 x 8 x 98 .. 229 (128) 13.5 / 15.3, 3 x 8 x 640 .. 706 (138) 23.1 / 24.7.
// Where keys are fewer than queries the walk is over them: causal 12 x 2413 over 603 keys 20.3 / 26.0, 3 x 8 x 1736 over 868 27.9 / 31.1; no mask 2 x 16 x
// 352 over 88 7.5 / 8.0.
inline bool small_launch_d128(int64_t live, int BH, int max_sq, int max_sk, bool causal, bool rotary) {
  const int policy = launch_policy() & 3;
  if (policy != 0) return policy == 2;
  if (causal && 4 * (int64_t)max_sk < 3 * (int64_t)max_sq) return false;
  const int max_s = max_sk < max_sq ? max_sk : max_sq;
  const int64_t x = fullest_xcd(live, BH);
  if (rotary) {
    if (!causal) return max_s > 192 && x <= (max_s > 768 ? 140 : 120);
    if (max_s <= 256) return max_s > 128 && x <= (max_s > 192 ? 140 : 125);
    return live <= 384 && (max_s > 2500 || x <= (max_s > 1100 ? 430 : max_s > 768 ? 360 : max_s > 512 ? 310 : max_s > 384 ? 200 : 150));
  }
  if (!causal) return max_s > 192 && x <= (max_s > 640 ? 150 : 140);
  if (max_s <= 256) return max_s > 128 && x <= (max_s > 192 ? 192 : 125);
  return live <= 384 && (max_s > 1100 || x <= (max_s > 768 ? 430 : max_s > 512 ? 360 : max_s > 384 ? 310 : 270));
}

// The forward over a padded batch, whose number of tokens is not known here: at head dim 128 as if three quarters of the rows were tokens, of
// short rows all; us of full-size / half-size tiles over 30 % .. 100 % of the rows, causal, 6 x 16 x 400 16.1 / 14.4, 4 x 12 x 1079 31.4 / 23.5, all rows tokens
// 2 x 12 x 1217 33.8 / 24.0, 8 x 16 x 218 .. 272 13.5 / 15.6 (over 1000 drawn shapes 2 % over the better of both, none more than 5 % slower than
// full-size throughout); below by the launched workgroups.
inline bool small_launch_rows(int head_dim, int batch, int nheads, int max_s, bool causal) {
  if (head_dim <= 64) return small_launch(kSmallLaunchFwd, batch * nheads, max_s, causal, false);
  const int64_t rows = (int64_t)batch * max_s;
  return small_launch_d128(live_row_tiles(nheads, (int)(max_s > 384 ? rows * 3 / 4 : rows), batch), batch * nheads, max_s, max_s, causal, false);
}

// Short backward launches run dQ and dK/dV as one grid (fa_bwd_merged_kernel: half-size dQ tiles, each part fills what the other leaves
// idle, one launch less; dQ at two waves per SIMD instead of three): at head dim 64, dense, no score bias, no rotation, no key split, dropout
// off or read from the keep words.  By the workgroups of 128 query rows that find any (live_row_tiles, `live`), the longest sequence n and, where
// the lengths are about equal, the launched workgroups on the fullest XCD (L): two launches are the better plan where L fills one or two rounds
// of the chip's 256 compute units, the more so the longer the walk; one launch where it leaves the last round half empty.  us in two
// launches / merged.
// Causal: 2 x 8 x 65 % of 842 (live 76) 41.2 / 26.3, 12 x 1812 (175) 75.3 / 50.1, 3 x 12 x 78 % of 2283 (521) 106.8 / 79.2, 4 x 8 x 2383 (611) 136.5 / 124.0;
// 27 x 8 x 273 (L 648) 30.5 / 33.4, 15 x 8 x 585 (600) 45.1 / 46.6, 16 x 16 x 219 (512) 26.6 / 27.6, 12 x 16 x 386 (live 675) 39.2 / 42.0; with
// dropout 6 x 16 x 69 % of 1258 (701) 82.9 / 71.9, 16 x 8 x 602 (L 640) 48.1 / 51.1.
// No mask: 3 x 8 x 846 (live 113) 39.8 / 25.7, 3 x 16 x 641 (264) 46.5 / 35.4, 8 x 12 x 77 % of 731 (469) 53.8 / 48.8; 7 x 16 x 239 (L 224) 20.4 / 21.6, 5 x 16 x
// 277 (240) 23.2 / 24.1, 11 x 8 x 276 (264) 29.0 / 23.1; 8 x 16 x 392 (512) 36.7 / 38.5, 16 x 3616 (464) 195 / 219, 8 x 7464 (472) 410 / 454, 12 x
// 3768 (480) 213 / 235, 3 x 16 x 1203 (480) 77 / 84, 8 x 6181 (392) 298 / 307, 12 x 4191 (528) 295 / 277; with dropout 7 x 16 x 380 .. 711 (533) 64.6 /
// 59.8, 4 x 8 x 2013 (L 512) 142 / 150.
// Up to 128 tokens: causal 16 x 12 x 97 (194) 16.4 / 10.6, 33 x 12 x 115 (553) 22.7 / 21.3, 32 x 16 x 76 (528) 22.5 / 23.1; no mask 12 x 16 x 45 (163) 12.7 /
// 9.3, 16 x 12 x 70 (201) 15.7 / 16.4; with dropout 33 x 12 x 73 (423) 23.5 / 22.1, 17 x 16 x 123 (397) 22.8 / 19.4, 21 x 12 x 81 (278) 17.2 / 19.0.
// (policy 0x10, the two-kernel plan, runs the same tiles in two launches: same bits)
inline bool merged_backward_shape(int head_dim, int64_t live, int BH, int max_sq, int max_sk, bool causal, bool dropout, bool keep_words,
                                  bool sparse, bool bias, bool rotary, int n_splits) {
  if (head_dim != 64 || sparse || bias || rotary || n_splits > 1 || (dropout && !keep_words)) return false;
  if ((launch_policy() & 3) != 0 || max_sk > 2 * max_sq) return small_launch(kSmallLaunchDq, BH, max_sq, causal, dropout);
  const int64_t L = fullest_xcd((int64_t)BH * ((max_sq + 127) / 128), BH);
  if (max_sq <= 128) {
    if (causal) return live <= (max_sq <= 64 || dropout ? 500 : max_sq <= 96 ? 435 : 600) || (dropout && L <= 512);
    return live <= 190 || (dropout && (max_sq <= 64 || BH > 256) && L <= 512);
  }
  if (live > (causal ? (dropout ? 700 : 620) : (dropout ? 670 : 480))) return false;
  if ((128 * live - 64 * BH) * 10 <= (int64_t)9 * BH * max_sq) return true;  // lengths differ: at most 0.9 of batch x longest are tokens
  if (causal) {
    if (max_sq <= 192 || max_sq > 800) return true;
    if (max_sq <= 256) return dropout || L <= 448;
    return L <= (dropout ? 608 : max_sq <= 384 ? 544 : 576);
  }
  if (max_sq <= 400 && L > 192 && L <= 256) return L < 232 && (max_sq <= 192 || max_sq > 256);
  if (L <= 512) return max_sq <= 384 || L <= (max_sq > 900 && !dropout ? 392 : 448);
  return max_sq <= 384 || L <= (max_sq > 900 && !dropout ? 600 : 640);
}
inline bool merged_backward_launch(int head_dim, int64_t live, int BH, int max_sq, int max_sk, bool causal, bool dropout, bool keep_words,
                                   bool sparse, bool bias, bool rotary, int n_splits) {
  return (launch_policy() & 0x30) != 0x10 &&
         merged_backward_shape(head_dim, live, BH, max_sq, max_sk, causal, dropout, keep_words, sparse, bias, rotary, n_splits);
}

// The dQ kernel's half-size tiles in a launch of its own, dropout off (with dropout: small_launch; at head dim 64 with keep words only where
// merged_backward_shape takes them, half-size tiles in two launches are the slowest plan there: 33 x 12 x 73 22.1 merged, 23.5 full-size, 29.1):
// causal d = 32 2 x 16 x 73 % of 707 (145) 27.6 / 25.1 with the dK/dV kernel, 3 x 16 x 70 % of 1785 (494) 59.5 / 53.0, 12 x 16 x 336 (551) 23.7 / 23.3;
// d = 16 2 x 8 x 3964 (503) 96.9 / 89.0; up to 128 tokens small_launch, 17 x 16 x 115 15.8 / 15.1; d = 64 8 x 12 x 460 (393) 34.0 / 32.6, 12 x 8 x 609
// (504) 40.5 / 42.7, with rotary (on the fullest XCD) 6 x 8 x 1012 (403) 57.6 / 53.1, 3 x 8 x 2177 (420) 102.6 / 96.5, 16 x 3394 (432) 144.8 / 135.1, 18 x 16 x 126
// (427) 26.3 / 25.4; no mask d = 64 2 x 12 x 615 (118) 30.5 / 27.8, 4 x 16 x 335 (199) 24.8 / 25.0.  d = 128 (the dK/dV kernel fills more of the
// chip there) causal 1 x 8 x 974 (64) 73.4 / 64.2, 4 x 12 x 272 (104) 31.4 / 28.8, 2 x 12 x 1500 (293) 110.3 / 101.0, short sequences cross sooner: 6 x 16 x 183
// (169) 25.6 / 27.1, 6 x 16 x 509 (345) 51.5 / 54.7; no mask, on the fullest XCD, 2 x 8 x 928 (124) 67.6 / 60.5, 3 x 16 x 789 (256) 70.7 / 75.7, 7 x 12 x 135
// (136) 25.3 / 27.7, 9 x 8 x 80 .. 244 (127) 29.6 / 30.3; over a quarter as many keys as queries, causal 2 x 16 x 1109 67.5 / 74.4.
inline bool small_launch_dq(int head_dim, int64_t live, int BH, int max_sq, int max_sk, bool causal, bool dropout, bool keep_words, bool rotary,
                            int n_splits) {
  if (merged_backward_shape(head_dim, live, BH, max_sq, max_sk, causal, dropout, keep_words, false, false, rotary, n_splits)) return true;
  const bool ruled = (launch_policy() & 3) == 0 && max_sk <= 2 * max_sq, swept = ruled && !dropout;
  if (head_dim == 128 && (launch_policy() & 3) == 0) {
    if (!swept || max_sq <= 128 || 2 * max_sk < max_sq) return false;
    return causal ? live <= (max_sq > 450 ? 300 : 150) : fullest_xcd(live, BH) <= (max_sq > 640 ? 140 : 120);
  }
  if (ruled && head_dim == 64 && dropout && keep_words && !rotary) return false;
  if (!swept || (head_dim < 64 && max_sq <= 128)) return small_launch(kSmallLaunchDq, BH, max_sq, causal, dropout);
  if (head_dim == 64 && causal) {
    const int64_t x = fullest_xcd(live, BH);
    if (max_sq <= 128) return rotary && max_sq > 96 && x <= 470;
    return x <= (max_sq > 1800 ? 520 : max_sq > 1200 ? 460 : max_sq > 800 ? 430 : max_sq > 384 ? 410 : 400);
  }
  return max_sq > 128 && live <= (causal ? 520 : 130);
}

// Launchers (defined in fa_fwd.hip / fa_bwd.hip / fa_aux.hip).  Return hipError_t of the launch.
// p.alibi != null selects the ALiBi variants (not available together with sparse)
hipError_t launch_fwd(const FwdParams& p, int dtype, int head_dim, bool causal, bool dropout, bool sparse,
                      hipStream_t stream);
// A few query rows (at most kDecodeMaxQ) against many keys: fa_decode_kernel (fa_decode.hip)
hipError_t launch_decode(const FwdParams& p, int dtype, int head_dim, hipStream_t stream);
hipError_t launch_fwd_combine(const FwdParams& p, int dtype, int head_dim, hipStream_t stream);
hipError_t launch_dq_combine(const BwdParams& p, int dtype, int head_dim, hipStream_t stream);
// The whole backward in one kernel (fa_bwd_fused_kernel.h; head_dim 64, dense, no mask, no dropout, no bias): softmax_d pass, then
// the kernel.  ev_start / ev_stop: null, or events recorded around the main kernel.
hipError_t launch_bwd_fused(const BwdParams& p, int dtype, hipStream_t stream, hipEvent_t ev_start, hipEvent_t ev_stop);
// fa_rotary: rotate the first n_rotated of n_parts (row, part, head, head_dim) slices, copy the others
struct RotaryParams {
  const void* src;
  void* dst;
  const void* cos;          // [table_rows, head_dim / 2], tensor dtype
  const void* sin;
  const int32_t* positions; // [n_rows] or null: position = row % seqlen
  int64_t n_rows;
  int64_t src_row_stride, src_part_stride, src_head_stride;  // elements
  int64_t dst_row_stride, dst_part_stride, dst_head_stride;
  int n_parts, n_rotated, n_heads, head_dim, seqlen, table_rows, conjugate;
  int64_t row_offset;  // set by launch_rotary: index of this launch's first row in the caller's tensor (position = row % seqlen)
};
hipError_t launch_rotary(const RotaryParams& p, int dtype, hipStream_t stream);
// positions[i] = i - cu[b], b the sequence that packed row i lies in
hipError_t launch_token_positions(const int32_t* cu, int batch, int total, int32_t* positions, hipStream_t stream);
hipError_t launch_gather_rows(const void* src, void* dst, const int64_t* idx, int64_t n_idx, int64_t n_src,
                              int64_t row_bytes, int64_t src_stride, int64_t dst_stride, int vec, hipStream_t stream);
hipError_t launch_scatter_rows(const void* src, void* dst, const int64_t* idx, int64_t n_idx, int64_t n_dst,
                               int64_t row_bytes, int64_t src_stride, int64_t dst_stride, int vec, int32_t* inv,
                               hipStream_t stream);
// From a (batch, seqlen) mask of bytes (nonzero: a token): row_of, row_info (FwdParams) and, if lens is not null, the lengths
hipError_t launch_padding_rows(const unsigned char* mask, int64_t mask_stride, int batch, int seqlen, int32_t* row_of, int32_t* row_info,
                               int32_t* lens, hipStream_t stream);
struct BiasGradLens {  // the batch's lengths as the backward had them (seq_extent); cu_q null: every element of the slices holds a gradient
  const int32_t* cu_q;
  const int32_t* cu_k;
  int total_q, total_k, max_sq, max_sk, causal;
};
hipError_t launch_bias_grad_reduce(const void* in, void* out, int dtype, int nb, int nh, int rows, int cols, int64_t in_bs,
                                   int64_t in_hs, int64_t in_rs, int sum_batch, int sum_heads, int64_t out_bs, int64_t out_hs,
                                   int64_t out_rs, const BiasGradLens& lens, bool vec_store, hipStream_t stream);
// Its launch: a workgroup per kPadBiasRows rows of a slice, as far as a grid may hold them (fewer than 2^32 threads: above 2^22 workgroups
// each takes several groups of rows)
constexpr int kPadBiasRows = 4;
struct PadBiasGrid {
  int64_t row_groups, groups;  // of a (batch, head) slice, of all
  unsigned blocks;
};
inline PadBiasGrid pad_bias_grid(int nb, int nh, int64_t rows) {
  PadBiasGrid g;
  g.row_groups = (rows + kPadBiasRows - 1) / kPadBiasRows;
  g.groups = g.row_groups * ((int64_t)nb * nh);
  g.blocks = (unsigned)(g.groups < (int64_t)1 << 22 ? g.groups : (int64_t)1 << 22);
  return g;
}
hipError_t launch_pad_bias_rows(const void* src, void* dst, int nb, int nh, int64_t rows, int64_t cols, int64_t s_bs, int64_t s_hs, int64_t s_rs,
                                int64_t s_ks, hipStream_t stream);
hipError_t launch_dump_probs(const DumpParams& p, int dtype, hipStream_t stream);
// which: 0 = dQ kernel, 1 = dK/dV kernel
hipError_t launch_bwd(const BwdParams& p, int which, int dtype, int head_dim, bool causal, bool dropout, bool sparse,
                      hipStream_t stream);
// maps, maps_bytes: the scratch that holds all of them (cleared where they are built with atomics)
// order / inv: null, or the row order (SparseMaps::order) and nrb ints of scratch for its inverse
// sorted: null, or scratch for SparseMaps::order and corder, dearest first; *is_sorted: whether they were left there
hipError_t launch_build_sparse_maps(const int32_t* blockmask, uint64_t* rbits, uint64_t* qbits, uint64_t* cbits, int nrb,
                                    int ncb, int rows_per_qt, int nqt, int ncw, int nrw, const int32_t* order, int32_t* inv, int32_t* sorted,
                                    bool* is_sorted, void* maps, size_t maps_bytes, hipStream_t stream);
hipError_t launch_fill_f32(float* p, size_t n, float value, hipStream_t stream);
// Zero a strided [total, H, D] tensor of 16-bit elements.
hipError_t launch_zero_rows(void* base, int64_t row_stride, int64_t head_stride, int total, int H, int D,
                            hipStream_t stream);
// softmax_d = keep * rowsum(dO o O) (fmha_dgrad_kernel_1xN_loop.h:15-30).

// Tile shapes, needed by the front end for grid sizes and workspace layout.
constexpr int kFwdBM = 128;   // query rows per forward workgroup
constexpr int kBwdBN = 128;   // keys per dK/dV workgroup
constexpr int kDecodeMaxQ = 32;  // query rows of fa_decode_kernel
constexpr int kDecodeWaves(int head_dim) { return head_dim >= 64 ? 2 : 4; }  // its waves (64 KB of tiles a workgroup at d = 128)
constexpr int kFusedBM = 32;  // query rows per step of the one-kernel backward

}  // namespace fa
