// Forward attention kernel for gfx950.
//
// Computes what the reference's device_1xN_loop does (csrc/flash_attn/src/fmha_fprop_kernel_1xN.h:199-671):
// O = dropout(softmax(scale * Q K^T + mask)) V and lse = logsumexp(scale * Q K^T + mask), but organised
// query-tile-outer: one workgroup owns 128 query rows of one (batch, head), keeps the output accumulator
// and the running (max, sum) in registers, streams K/V tiles through LDS, and writes o and lse once.
// There is no fp32 o_tmp round trip through global memory.
//
// Everything is computed transposed so that one lane owns one query row:
//   S^T = K Q^T   (A = K tile from LDS, B = Q fragment held in registers), C layout: lane -> query
//                 column l%32, registers -> 16 keys.  Row max / row sum are in-lane plus ONE exchange with lane l^32.
//   O^T = V^T P^T (A = V^T read from the row-major V tile with ds_read_b64_tr_b16, B = P^T taken straight from the
//                 S^T accumulator registers, rounded to fp16/bf16).  The contraction runs over keys in the order the
//                 accumulator registers hold them; the V^T fragment is fetched in the same order.
#pragma once

#include <type_traits>

#include "fa_common.h"
#include "fa_params.h"
#include "fa_stage.h"

// Measurement variants (-DFA_ABLATE_FWD=<bits> through FA_EXTRA_HIPCC_FLAGS; results are wrong, never a product build):
// what one part of the main loop costs is read off the kernel's time without it.  1: no wait for the staged tile and no
// workgroup barrier; 2: a multiplication in place of every exponential; 4: no P V products; 8: no Q K^T products; 16: the K
// and V fragments not read from LDS (registers stand in); 32: no row sums of P and no test of them.
#ifndef FA_ABLATE_FWD
#define FA_ABLATE_FWD 0
#endif

namespace fa {

// KS (key split) = 1: the workgroup's four waves own 32 of its 128 query rows each and every wave sees all keys of a tile.
// KS = 2 (short sequences, where 128-row tiles are too few workgroups to fill the chip and one workgroup's walk over the
// keys is the launch's critical path): 64 query rows per workgroup; waves w and w + 2 share 32 rows and split the keys
// of every tile between them, each with its own running maximum, sum and output accumulator, merged in the epilogue.
template <typename T, int D, int BN, int KS = 1>
struct FwdCfg {
  static constexpr int BM = kFwdBM / KS;
  static constexpr int NW = 4;                 // waves per workgroup
  static constexpr int RW = NW / KS;           // 32-row slabs per workgroup
  static constexpr int KBW = BN / 32 / KS;     // 32-key blocks of a tile per wave
  static_assert(KS == 1 || (KS == 2 && BN == 64), "key split: two waves per 32 rows, one 32-key block each");
  static constexpr int DV = D < 32 ? 32 : D;   // rows of the V^T MFMA operand (for D = 16 the upper 16 are don't-care)
  static constexpr int OS = D + 8;             // epilogue staging row stride
  // K tile (read as row fragments) followed by V tile (read transposed), double buffered; see fa_stage.h
  typedef TilePairStager<D, BN, kSwzRow, kSwzTr> Stager;
  static constexpr int kBufBytes = Stager::kPairBytes;
  static constexpr int kSlack = D < 32 ? 64 : 0;                // the 32-wide transposed reads run past a 16-wide V row
  static constexpr int kTileBytes = 2 * kBufBytes + kSlack;
  static constexpr int kEpiBytes = BM * OS * 2;
  static constexpr int kMergeBytes = KS > 1 ? RW * (DV / 32 * 16 + 2) * 64 * 4 : 0;  // partial (O, max, sum) of RW waves
  static constexpr int kLdsBytes0 = kTileBytes > kEpiBytes ? kTileBytes : kEpiBytes;
  static constexpr int kLdsBytes = kLdsBytes0 > kMergeBytes ? kLdsBytes0 : kMergeBytes;
  static constexpr int CH = D / 8;
};

// The variants that come in the live order, too (kLive below, map_live)
template <int D, bool kSparse, int kBias>
struct FwdLive {
  static constexpr bool value = !kSparse && kBias != kBiasTensor && !(kBias == kPaddedRows && D == 128);
};

// kBias (fa_params.h): 1 = ALiBi, the score of (query i, key j) gets -slope[head] * |i - j| added after scaling; 2 = it gets
// bias[b, h, i, j] of a tensor added.  The scores are then moved to the softmax's own units (base-2 exponent) before the row
// maximum is taken, and the running maximum is kept in those units.
// Waves per SIMD that the variants are bounded to: what their registers allow without a spill in the main loop, or with the few
// that tests/test_kernel_resources.py pins where the wave is worth more (d = 128 over a block layout, 4 x 16 heads x 4096, a quarter of
// the blocks, bf16: two registers in scratch, 305 us; two waves per SIMD 351).  The dense d = 128 forward takes 168 registers, three
// waves, by itself and is scheduled better than when it is told to (4 x 16 x 600 .. 3001 causal bf16 86.6 us, bounded 89.4).
constexpr int fwd_waves(int d, bool dropout, bool sparse, int bias, int ks, bool words) {
  if (dropout && ks == 2 && bias == 0 && d == 16 && !words) return 6;
  if ((!dropout || ks == 2) && bias == 0 && d <= 64) return 4;
  if (!dropout && ((bias == 0 && sparse) || (d <= 64 && !(sparse && bias == kBiasAlibi)))) return 3;
  return 2;
}
// kRoomy (dense, d = 128, no dropout, no bias): launches of at most two workgroups per compute unit that do not run the half-size tiles
// (small_launch_d128), which a third wave per SIMD does not help, keep
// all K fragments of a tile in flight also where its scores are redone, at two waves per SIMD: us of that build / the other,
// bf16, 64 workgroups (8 heads x 1000) 24.8 / 27.0, causal 26.5 / 27.8; 192 (16 x 1500) 34.8 / 38.1; 384 (16 x 3000) 92.5 / 95.3, causal 68.6 / 72.3;
// 576 (64 x 1100) 61.5 / 54.5; 1536 (64 x 3000) 303 / 286.
// kWords (dropout, dense): the keep decisions are also left in p.keep_words for the backward (fa_common.h)
// kBias = kPaddedRows (dense, no dropout): q, k, v and o are a padded batch, (batch, max_sq) rows of which p.row_of and p.row_info name the
// tokens; these attend each other, counted in their own order, and the padding rows of o are written as zeros.  32 x 512 rows, 256 .. 512 of
// them tokens, 16 heads, d = 64: one launch of 43 us in place of gather 29, forward 40 and scatter 15, 42 with tokens anywhere in their row (the
// module call 52 us, 175 gathered).
// kLive: the workgroups' ids enumerate the tiles that hold rows (map_live).  A kernel of its own: with both orders' code in one, launches in the slot order
// paid for the other's, in registers, parked scalars and arguments loaded again in the main loop.  us, both in one / apart, equal lengths: backward
// without a mask, d = 64 16 x 1500 45.2 / 41.5, 2 x 8 x 2000 72.9 / 69.5, 8 x 12 x 512 37.5 / 35.2; causal 7 x 24 x 132 .. 268 19.4 / 18.8; forward d = 16
// causal 3 x 3 x 4049 30.4 / 28.9, d = 128 causal with keep words 2 x 12 x 3218 108.9 / 106.1.
template <typename T, int D, int BN, bool kRoomy, bool kCausal, bool kDropout, bool kSparse, int kBias, int KS, bool kWords, bool kLive>
FA_DEVICE void fa_fwd_body(const FwdParams& p) {
  constexpr bool kRows = kBias == kPaddedRows;
  constexpr bool kBiased = kBias != 0 && !kRows;
  constexpr bool kAlibi = kBias == kBiasAlibi, kTensorBias = kBias == kBiasTensor;
  static_assert(!kWords || (kDropout && !kSparse), "keep words: dense dropout variants only");
  static_assert(!kRows || (!kDropout && !kSparse), "padded batches: dense, no dropout");
  static_assert(!kRoomy || (D == 128 && !kDropout && !kSparse && !kBiased), "built where a launch may be short of workgroups");
  using Cfg = FwdCfg<T, D, BN, KS>;
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  constexpr int BM = Cfg::BM, DV = Cfg::DV, CH = Cfg::CH, kBufBytes = Cfg::kBufBytes, KBW = Cfg::KBW;
  static_assert(KS == 1 || !kSparse, "the block-sparse maps are built for 128-row query tiles");

  // kTensorBias: behind the tiles, per wave 32 rows x BN keys of bias, rows padded by 8 bytes (see load_bias below)
  constexpr int kBiasRowBytes = BN * 2 + 8, kBiasWaveBytes = 32 * kBiasRowBytes;
  // kKeyWords: behind everything else, for the staged and the next tile, the key words of its BN / 2 Philox counters (fa_common.h).  us of the
  // forward with them / with whole outputs drawn, p = 0.1: 64 x 16 heads x 1004 .. 1023, d = 64, 535 / 551; 4 x 12 x 4096 313 / 319; 8 x 16 x
  // 1000, d = 32, 60.6 / 63.0.  Not at d = 128 (8 x 12 x 2048: 316 / 301), nor in the half-size tiles (causal, d = 64, 3 x 12 x 1200 24.8 / 23.4, 2 x 16 x
  // 1600 30.4 / 28.5; d = 32, 16 x 2600 32.1 / 30.0), nor where they cost a wave per SIMD: over a block layout at d = 32, nor under a causal mask
  // where keep words are left (d = 64, 68 x 8 x 273 32.8 / 31.4, 50 x 12 x 1006 185.7 / 181.7, 17 x 16 x 103 11.0 / 10.5; between 0.96 and 1.05, 1.00 in the
  // middle; without the words 0.97 to 0.99).
  // (Round keys stepped by the scalar unit in place of kept ones, which are parked in vector lanes: 550.)
  constexpr bool kKeyWords = kDropout && !kSparse && kBias == 0 && KS == 1 && !(kCausal && kWords) && (D == 32 || D == 64);
  constexpr int kKeyWordBytes = BN / 2 * 16, kKeyWordOff = Cfg::kLdsBytes + (kTensorBias ? 4 * kBiasWaveBytes : 0);
  constexpr int kRowSlotBytes = 2 * 64 * 4;  // kRows: behind the tiles, per wave (see fetch_rows below)
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[Cfg::kLdsBytes + (kTensorBias ? 4 * kBiasWaveBytes : kRows ? 4 * kRowSlotBytes : 0) +
                                                                  (kKeyWords ? 2 * kKeyWordBytes : 0)];

  // Workgroup -> (batch, head, query tile), XCD-aware (see map_tile): the query tiles of one (batch, head) share
  // one XCD's L2 copy of K and V.
  int b, h, qt, split = 0;
  int q_begin, Lq, k_begin = 0, Lk = 0;
  const int n_splits = p.n_splits > 1 ? p.n_splits : 1;  // key splits per query tile (see FwdParams)
  if constexpr (kLive) {
    TileId id;
    if (!map_live<kCausal>(blockIdx.x, p.cu_q, p.total_q, p.max_sq, p.cu_k, p.total_k, p.max_sk, BM, p.nq_tiles, false, p.B, p.H,
                           kRows ? p.row_info : nullptr, lds_raw + kBufBytes + (threadIdx.x >> 6) * 256, &id)) return;
    b = id.b; h = id.h; qt = id.tile;
    // (opaque: known to be 0 the first step over the keys is peeled off the loop, for 20 to 50 registers: the half-size tiles went to scratch, causal
    // d = 64 2 x 12 x 500 .. 1000 17.1 us for 13.4)
    asm volatile("" : "+s"(split));
    q_begin = id.own_begin; Lq = id.own_len; k_begin = id.walk_begin; Lk = id.walk_len;
  } else {
    int bh, rank;
    if (kSparse && p.sp.corder != nullptr ? !map_tile<true>(blockIdx.x, p.nq_tiles * n_splits, p.B * p.H, &bh, &rank, p.tile_group)
                                          : !map_tile<kCausal>(blockIdx.x, p.nq_tiles * n_splits, p.B * p.H, &bh, &rank, p.tile_group))
      return;
    split = rank % n_splits;
    rank /= n_splits;
    qt = kCausal ? p.nq_tiles - 1 - rank : rank;  // under a causal mask the last query tiles cost most
    h = bh % p.H;
    // (dense, no mask: the batch entries are taken longest keys first, see longest_first)
    b = (!kCausal && !kSparse && p.tile_group == kLongestFirst) ? longest_first(p.cu_k, p.B, bh / p.H, kRows ? p.row_info : nullptr) : bh / p.H;
  }
  const int bh = b * p.H + h;  // (what the dropout counters and the keep words are indexed by)

  // kRows: this entry's slice of row_of; its tokens lie one after the other (from row q_begin on) or, `listed`, anywhere in it
  const int32_t* const row_of = kRows ? p.row_of + (int64_t)b * p.max_sq : nullptr;
  bool listed = false;
  if constexpr (kRows) {
    Lq = Lk = __builtin_amdgcn_readfirstlane(p.row_info[kRowInfo * b]);
    listed = __builtin_amdgcn_readfirstlane(p.row_info[kRowInfo * b + 2]) == 0;
    q_begin = k_begin = b * p.max_sq + (listed ? 0 : __builtin_amdgcn_readfirstlane(p.row_info[kRowInfo * b + 1]));
  } else if constexpr (!kLive) {
    if (!seq_extent(p.cu_q, b, p.total_q, p.max_sq, &q_begin, &Lq)) return;
    if (!seq_extent(p.cu_k, b, p.total_k, p.max_sk, &k_begin, &Lk)) Lk = 0;  // no keys: o = 0, lse = -inf
  }
  const int m0 = qt * BM;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31, hf = lane >> 5;
  const int rs = KS > 1 ? wave % Cfg::RW : wave;  // this wave's 32-row slab of the tile
  const int kh = KS > 1 ? wave / Cfg::RW : 0;     // ... and its share of every key tile's 32-key blocks
  const int mw = m0 + rs * 32;    // first query row of this wave
  int qrow = mw + c;              // this lane's query row (sequence-local)
  // Sparse: the wave's 32 rows are two 16-row blocks, consecutive ones or - with a row order (SparseMaps) - two the caller
  // put next to each other; rows of no block count as lying past the end
  int rb_a = -1, rb_b = -1;
  bool wave_live = mw < Lq;  // some row of the wave exists
  if (kSparse) {
    const bool ordered = !kCausal && p.sp.order != nullptr;
    slab_row_blocks(p.sp, ordered, qt, rs, &rb_a, &rb_b);
    const int rbl = c < 16 ? rb_a : rb_b;
    qrow = rbl >= 0 ? rbl * 16 + (c & 15) : 0x3fffffff;
    wave_live = (rb_a >= 0 && rb_a * 16 < Lq) || (rb_b >= 0 && rb_b * 16 < Lq);
    if (ordered) {
      if (!__syncthreads_or(wave_live)) return;  // no row of the workgroup exists
    } else if (m0 >= Lq) {
      return;
    }
  } else if (m0 >= Lq) {
    if constexpr (kRows) {  // padding rows only: zeros
      for (int i = tid; i < BM * CH; i += 256) {
        const int j = m0 + i / CH;
        if (j < p.max_sq)
          st_global16(reinterpret_cast<T*>(p.o) + ((int64_t)b * p.max_sq + row_of[j]) * p.o_rs + (int64_t)h * p.o_hs + (i % CH) * 8,
                      u32x4{0, 0, 0, 0});
      }
    }
    return;
  }

  // ---- Q fragment (B operand of S^T = K Q^T), held in registers for the whole kernel
  vec8 qreg[D / 16];
  {
    int qr = qrow < Lq ? qrow : Lq - 1;
    if constexpr (kRows) {
      if (listed) qr = row_of[qr];
    }
    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)(q_begin + qr) * p.q_rs + (int64_t)h * p.q_hs + hf * 8;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++) qreg[ks] = bitcast<vec8>(ld_global16(qp + ks * 16));
    // rows past the end work on a copy of the last row and are never stored (no select on the loaded data here: it
    // would make the wave wait for the load before it has issued its first tile)
  }

  int n_end = Lk;
  if (kCausal) n_end = n_end < m0 + BM ? n_end : m0 + BM;
  const int ntiles_all = (n_end + BN - 1) / BN;
  const int tile0 = (int)((int64_t)split * ntiles_all / n_splits);        // this workgroup's share of the key tiles
  const int ntiles = (int)((int64_t)(split + 1) * ntiles_all / n_splits);

  // ---- K/V staging: global -> LDS without passing through registers (waves 0,1 fetch K tiles, waves 2,3 V tiles)
  typename Cfg::Stager stager;
  stager.init(wave, lane, reinterpret_cast<const T*>(p.k) + (int64_t)k_begin * p.k_rs + (int64_t)h * p.k_hs, p.k_rs,
              reinterpret_cast<const T*>(p.v) + (int64_t)k_begin * p.v_rs + (int64_t)h * p.v_hs, p.v_rs);
  // kRows, listed: the rows of a tile are read off row_of, which a wave brings into two LDS slots of its own, a tile ahead of the tile's own
  // loads (keys past the end: the last key's row)
  int32_t* const row_slots = reinterpret_cast<int32_t*>(lds_raw + Cfg::kLdsBytes + wave * kRowSlotBytes);
  auto fetch_rows = [&](int it) {
    const int j = it * BN + lane;
    dma4(reinterpret_cast<const char*>(row_of), 4u * (uint32_t)(j < Lk ? j : Lk - 1), reinterpret_cast<unsigned char*>(row_slots + (it & 1) * 64));
  };
  auto stage = [&](int it, int buf) {
    if constexpr (kRows) {
      if (listed) {
        stager.template issue_listed<D == 128 && KS == 1 && !kRoomy>(lds_raw + buf * kBufBytes, row_slots + (it & 1) * 64);
        if (it + 1 < ntiles) {
          __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the list has been read (and the slot of it + 1 was before it)
          fetch_rows(it + 1);
        }
        return;
      }
    }
    if constexpr (kKeyWords) {  // the waves take turns, one tile each
      if ((it & 3) == wave && lane < BN / 2)
        *reinterpret_cast<u32x4*>(lds_raw + kKeyWordOff + buf * kKeyWordBytes + lane * 16) =
            philox_key_words(p.pk, (uint32_t)bh, (uint32_t)(it * (BN / 2) + lane));
    }
    stager.issue(lds_raw + buf * kBufBytes, it * BN, Lk);
  };
  const uint64_t query_words = kKeyWords ? philox_query_words(p.pk, (uint32_t)bh, (uint32_t)qrow >> 2) : 0;

  // Sparse: tile `it` is computed iff its 256-key block is active for any 16-row block of this query tile.  Everything about it is
  // wave-uniform and kept in scalar registers: the activity bits of 64 consecutive key blocks (16384 keys) for the query tile and for
  // the wave's two row blocks, and the lanes whose row block attends the tile in hand.  The search sits in front of the next tile's loads
  // in every wave, a chain of dependent scalar instructions and branches, so it runs once per key block: within one the next tile is the
  // next (d = 64, a quarter to a third of the 16 x 256 blocks, 1 x 8 heads x 4959 70.3 / 66.3 us, 2 x 16 x 5584 148 / 140; the dQ kernel, with no register to
  // spare, is 1 % slower for it and searches tile by tile).
  uint64_t tile_bits = 0, bits_a = 0, bits_b = 0;
  int bits_word = -1;
  const int qt_u = __builtin_amdgcn_readfirstlane(qt);
  uint64_t row_mask_next = ~uint64_t(0);  // lanes whose row block attends the tile the last search found
  // First tile >= it whose 256-key block is active (ntiles if none): the bits of the loaded word are searched with a
  // count-trailing-zeros, not tile by tile.
  auto find_active = [&](int it) -> int {
    constexpr int kTilesPerBlock = 256 / BN;
    while (it < ntiles) {
      const int cb = __builtin_amdgcn_readfirstlane((it * BN) >> 8);
      if ((cb >> 6) != bits_word) {
        bits_word = cb >> 6;
        tile_bits = uniform64(p.sp.qbits[(int64_t)qt_u * p.sp.ncw + bits_word]);
        bits_a = rb_a >= 0 ? uniform64(p.sp.rbits[(int64_t)rb_a * p.sp.ncw + bits_word]) : 0;
        bits_b = rb_b >= 0 ? uniform64(p.sp.rbits[(int64_t)rb_b * p.sp.ncw + bits_word]) : 0;
      }
      const uint64_t rest = tile_bits >> (cb & 63);  // bit 0: this tile's block
      if (rest & 1) {
        row_mask_next = half_slab_lanes((bits_a >> (cb & 63)) & 1, (bits_b >> (cb & 63)) & 1);
        return it;
      }
      // first tile of the next active block of this word, or of the next word
      it = (rest ? cb + (int)__builtin_ctzll(rest) : (cb | 63) + 1) * kTilesPerBlock;
    }
    return ntiles;
  };
  auto next_active = [&](int it) -> int {  // the tile after `it`, which is active
    return !kSparse || (it + 1) % (256 / BN) != 0 ? it + 1 : find_active(it + 1);
  };

  f32x16 o_acc[DV / 32];
#pragma unroll
  for (int i = 0; i < DV / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) o_acc[i][r] = 0.f;
  float m_i = -INFINITY;  // running row max of raw scores (before scaling)
  float l_i = 0.f;        // this lane's share of the running row sum (other share in lane^32)

  const float cs = p.scale_log2;
  const float cse = kBiased ? 1.f : cs;                       // units of the scores the softmax works on
  const float sl2 = kAlibi ? p.alibi[h] * kLog2e : 0.f;          // slope in base-2 exponent units
  // kTensorBias: the wave's 32 rows x BN keys of the bias come in as whole rows - BN / 8 lanes fetch the BN * 2 contiguous
  // bytes of one row, 16 bytes each, so that an instruction touches 8 (16) rows and not 32: read lane by lane in the MFMA
  // layout (every lane another row) the requests, one per row and instruction, took as long as the whole kernel without a
  // bias - and are turned into that layout through LDS (wave-private, rows padded by 8 bytes: 32 lanes reading 8 bytes at the
  // same column of 32 rows hit 32 distinct bank pairs).  Asked for one tile ahead; chunks that begin past the last key are
  // not read, rows past the end read the last row (like Q).
  constexpr int kBiasCPR = BN / 8, kBiasRPI = 64 / kBiasCPR, kBiasNLD = 32 / kBiasRPI;
  const T* const bias_bh =
      kTensorBias ? reinterpret_cast<const T*>(p.bias) + (int64_t)b * p.bias_bs + (int64_t)h * p.bias_hs : nullptr;
  unsigned char* const bias_lds = lds_raw + Cfg::kLdsBytes + wave * kBiasWaveBytes;
  u32x4 braw[kTensorBias ? kBiasNLD : 1];
  auto load_bias = [&](int tile) {
#pragma unroll
    for (int i = 0; i < kBiasNLD; i++) {
      const int lr = i * kBiasRPI + lane / kBiasCPR, k0 = tile * BN + (lane % kBiasCPR) * 8;
      int row = mw + lr;
      if (kSparse) {  // the slab's two row blocks (rows of no block read the last row: their results are never stored)
        const int rbl = lr < 16 ? rb_a : rb_b;
        row = rbl >= 0 ? rbl * 16 + (lr & 15) : Lq;
      }
      braw[i] = u32x4{0, 0, 0, 0};
      if (k0 < Lk) braw[i] = ld_global16(bias_bh + (uint32_t)(row < Lq ? row : Lq - 1) * (uint32_t)p.bias_rs + (uint32_t)k0);
    }
  };
  auto bias_to_lds = [&]() {
#pragma unroll
    for (int i = 0; i < kBiasNLD; i++)
      *reinterpret_cast<u32x4*>(bias_lds + (i * kBiasRPI + lane / kBiasCPR) * kBiasRowBytes + (lane % kBiasCPR) * 16) = braw[i];
  };
  int voff[DV / 32];  // element offsets of this lane's transposed V reads and K row fragments inside a tile
#pragma unroll
  for (int db = 0; db < DV / 32; db++) voff[db] = tr_off<D, kSwzTr>(0, db * 4, lane);
  int koff[D / 16];
#pragma unroll
  for (int ks = 0; ks < D / 16; ks++) koff[ks] = frag_off<D, kSwzRow>(c, ks * 2 + hf);
  int buf = 0;

  // Dropout keep words for the backward (fa_common.h): a tile's words are stored at the top of the next step, ahead of
  // the next prefetch - stored where they are made, their acknowledgements would still be outstanding when the step
  // ends and waits for its prefetched tile (one counter serves loads and stores).
  uint32_t kwout[KBW];
  int kw_pending = -1;  // first key block (of 32) of the words waiting in kwout
  auto flush_keep_words = [&]() {
    if (kWords && kw_pending >= 0) {
      if (hf == 0) {
#pragma unroll
        for (int kb = 0; kb < KBW; kb++)
          p.keep_words[((int64_t)bh * p.kw_kb + kw_pending + kb) * p.kw_q + mw + (keep_word_slot(c) & 31)] = kwout[kb];
      }
      kw_pending = -1;
    }
  };

  int it = kSparse ? find_active(tile0) : tile0;
  if (it < ntiles) {
    if constexpr (kRows) {
      if (listed) {
        fetch_rows(it);
        wait_vmem();
      }
    }
    stage(it, 0);
    if (kTensorBias) load_bias(it);
  }
  // Rotary embedding of the queries (what the reference's FlashMHA does to q before attention, flash_attention.py:109-113,
  // with elementwise ops): the fragments are turned where they sit, after the first tile has been asked for; the rotated
  // rows are left in q_rot for the backward, whose kernels stream Q through LDS and cannot do the same
  if (p.rot_cos != nullptr) {
    int t = qrow < Lq ? qrow : Lq - 1;
    t = t < p.rot_rows ? t : p.rot_rows - 1;
    const T* const ct = reinterpret_cast<const T*>(p.rot_cos) + (int64_t)t * (D / 2) + hf * 4;
    const T* const st = reinterpret_cast<const T*>(p.rot_sin) + (int64_t)t * (D / 2) + hf * 4;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++)
      qreg[ks] = rotate8<T>(qreg[ks], *reinterpret_cast<const typename E::vec4*>(ct + ks * 8),
                            *reinterpret_cast<const typename E::vec4*>(st + ks * 8), false);
  }
  // Aligned, so that what precedes it does not move it against the instruction cache's lines: with one or two waves on a SIMD the loop waits for its
  // own instructions, and the same code elsewhere took up to 8 % longer (us, d = 32 causal 3 x 3 heads x 4049 33.3 / 31.2, 2 x 8 x 2000 18.1 / 17.4, d = 128
  // 2 x 8 x 2000 47.3 / 45.8, with keep words 2 x 12 x 1189 43.5 / 41.7; 300 drawn launches 0.996 in the mean).
  asm volatile(".p2align 7");
  while (it < ntiles) {
    const int n0 = it * BN;
    // Opaque redefinition of the accumulators at the top of every iteration: without it the register allocator
    // ties the last MFMA's result to the registers the epilogue reads and copies all of O back on every trip.
#pragma unroll
    for (int i = 0; i < DV / 32; i++) asm volatile("" : "+v"(o_acc[i]));
    if constexpr ((FA_ABLATE_FWD & 1) == 0) {
      wait_vmem();                       // this wave's share of tile `it` is in LDS
      flush_keep_words();
      __syncthreads();                   // so is everyone else's, and nobody still reads the other buffer
    }
    const uint64_t row_mask = row_mask_next;  // (of this tile: the search below moves on)
    const int it_next = next_active(it);
    if (it_next < ntiles) stage(it_next, buf ^ 1);
    if (kTensorBias) {  // (the wave's own reads of the last tile's values are behind it: LDS operations of a wave stay in order)
      bias_to_lds();
      if (it_next < ntiles) load_bias(it_next);
    }
    const T* Ks = reinterpret_cast<const T*>(lds_raw + buf * kBufBytes);
    const T* Vs = Ks + BN * D;
    const u32x4* const key_words = reinterpret_cast<const u32x4*>(lds_raw + kKeyWordOff + buf * kKeyWordBytes);
    buf ^= 1;

    bool wave_work = wave_live;  // a wave whose 32 rows all lie past the sequence's end only helps with the staging
    if (kCausal && n0 + kh * 32 * KBW > mw + 31) wave_work = false;  // every key of the wave's share is above its diagonal
    if (KS > 1 && n0 + kh * 32 * KBW >= Lk) wave_work = false;       // ... or past the last key
    if (kSparse && row_mask == 0) wave_work = false;
    const bool row_on = !kSparse || lane_bit(row_mask);

    if (wave_work) {
      // this wave's 32-key blocks of the tile: kb0, kb0 + 1, ... (all of them without a key split)
      const int kb0 = kh * KBW;
      f32x16 s[KBW];
      // ---- S^T = K Q^T, dead scores set to -inf, bias added
      // (again: the rare second time for a tile.  The fragments are then read one at a time where four at once do not fit the registers
      // and went through scratch, whose loads wait for the next tile's prefetch: eight registers at d = 128, and the half-size kernel's
      // dropout variants.)
      auto scores = [&](auto again) {
        // kTensorBias: the lane's 4 x 4 consecutive bias values per 32-key block (registers 4 j .. 4 j + 3 <-> keys
        // 8 j + 4 hf ..) of its row
        typename E::vec4 bv[kTensorBias ? KBW : 1][4];
        if (kTensorBias) {
#pragma unroll
          for (int kb = 0; kb < KBW; kb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
              bv[kb][j] = *reinterpret_cast<const typename E::vec4*>(bias_lds + c * kBiasRowBytes + ((kb0 + kb) * 32 + 8 * j + 4 * hf) * 2);
        }
#pragma unroll
        for (int kb = 0; kb < KBW; kb++) {
#pragma unroll
          for (int r = 0; r < 16; r++) s[kb][r] = 0.f;
#pragma unroll
          for (int ks = 0; ks < D / 16; ks++) {
            vec8 a = (FA_ABLATE_FWD & 16) ? qreg[(ks + 1) % (D / 16)] : *reinterpret_cast<const vec8*>(Ks + (kb0 + kb) * 32 * D + koff[ks]);
            if constexpr ((FA_ABLATE_FWD & 8) == 0) s[kb] = E::mfma32(a, qreg[ks], s[kb]);
            else s[kb][ks] = (float)a[ks] * (float)qreg[ks][0];
            if constexpr (decltype(again)::value && ((D == 128 && !kRoomy) || (kDropout && KS == 2))) __builtin_amdgcn_sched_barrier(0);
          }
        }
        // mask: only tiles that straddle the key length or the diagonal.  (An inactive row block inside an active tile is
        // not masked score by score: its lanes' exponentials are taken against +inf below.)
        const bool need_mask = (n0 + BN > Lk) || (kCausal && (n0 + BN - 1 > mw));
        if (need_mask) {
          // kFewMasks: keys from `limit` on are dead, counted from the lane's register 0, behind an opaque copy and four registers at a time.
          // Left alone the compiler holds the 32 compare masks of a tile in scalar registers, also for the case that its scores are redone,
          // and what it moves to vector lanes for them it reads back in every step: in the d = 64 forward with dropout 16 of them and a
          // scalar load (64 x 16 heads x 1004 .. 1023, p = 0.1, step 1670 / 1656 us), in the causal one 5 (8 x 12 x 4096 bf16, step 900 / 894; 13 x 16 x
          // 1380 forward 88.5 / 85.8), in the padded one 4 (63 x 8 x 867 .. 1352 222 / 216).  Not where it costs
          // registers instead: ALiBi terms or a block layout under a causal mask two to eight in scratch, the half-size tiles (one block a wave).
          constexpr bool kFewMasks = KS == 1 && KBW == 2 && !kAlibi && !(kSparse && kCausal);
          int limit = (kCausal && qrow < Lk ? qrow + 1 : Lk) - (n0 + kb0 * 32 + hf * 4);
          if constexpr (kFewMasks) asm volatile("" : "+v"(limit));
#pragma unroll
          for (int kb = 0; kb < KBW; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
              const int key = n0 + (kb0 + kb) * 32 + (r >> 2) * 8 + hf * 4 + (r & 3);
              bool dead = key >= Lk;
              if (kCausal) dead = dead || key > qrow;
              if (kFewMasks) dead = kb * 32 + (r >> 2) * 8 + (r & 3) >= limit;
              if (dead) s[kb][r] = -INFINITY;
              if (kFewMasks && (r & 3) == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (kTensorBias) {  // s <- s * scale * log2(e) + bias * log2(e)
          // Dead scores must stay -inf whatever lies behind them: past the last key a row of the caller's tensor may hold
          // anything, so on a tile that needs a mask +inf and NaN are cut off (fminf returns the number)
#pragma unroll
          for (int kb = 0; kb < KBW; kb++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
              float bf = (float)bv[kb][r >> 2][r & 3];
              if (need_mask) bf = fminf(bf, 3.0e38f);
              s[kb][r] = __builtin_fmaf(bf, kLog2e, s[kb][r] * cs);
            }
        }
        if (kAlibi) {  // s <- s * scale * log2(e) - slope2 * |key - query|; dead scores stay -inf
#pragma unroll
          for (int kb = 0; kb < KBW; kb++) {
            const float dbase = (float)(n0 + (kb0 + kb) * 32 + hf * 4 - qrow);  // key - query of register 0
#pragma unroll
            for (int r = 0; r < 16; r++) {
              const float cr = (float)((r >> 2) * 8 + (r & 3));
              // under a causal mask every live score has key <= query: -|key - query| = key - query, linear in cr
              const float bias = kCausal ? __builtin_fmaf(cr, sl2, sl2 * dbase) : -sl2 * __builtin_fabsf(dbase + cr);
              s[kb][r] = __builtin_fmaf(s[kb][r], cs, bias);
            }
          }
        }
      };
      // ---- P = exp2(scores - reference point m_i), rounded to the tensor dtype (what the P V product consumes); lt = this
      // lane's share of the tile's row sums: of the rounded values (sum8_acc), so that numerator and denominator of o share that
      // rounding, or with dropout of P before the rounding and the mask, in fp32 as the reference has it
      // (fmha_fprop_kernel_1xN.h:454 vs :471).  Sums of the unrounded P, one addition per value, save bf16 1.5 to 2.5 % of the
      // kernel (8 x 12 heads x 2048 d = 64 112.2 us for 114.8, 16 x 12 x 2048 d = 128 388 for 394) and put o up to 15 % further from float64
      // (8 x 12 x 1024, normal inputs x 2.5: 1.75e-3 of its norm with the rounded values, 2.01e-3 without; x 1: 2.359e-3 / 2.364e-3).
      vec8 pb[KBW][2];
      float lt;
      auto probabilities = [&]() {
        float mc = ((m_i == -INFINITY) ? 0.f : m_i) * cse;
        if (kSparse && !row_on) mc = INFINITY;  // this lane's row block does not attend the tile: P = exp2(x - inf) = 0
        float lp[KBW];  // (dropout: two chains of additions where a tile has two 32-key blocks; else lp[0] is the only one)
#pragma unroll
        for (int kb = 0; kb < KBW; kb++) {
          lp[kb] = 0.f;
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const float pe_arg = kBiased ? s[kb][r] - mc : __builtin_fmaf(s[kb][r], cs, -mc);
            s[kb][r] = (FA_ABLATE_FWD & 2) ? pe_arg * 1e-3f : fast_exp2(pe_arg);
            if constexpr (kDropout && (FA_ABLATE_FWD & 32) == 0) lp[kb] += s[kb][r];
          }
        }
#pragma unroll
        for (int kb = 0; kb < KBW; kb++)
#pragma unroll
          for (int t = 0; t < 2; t++) {
            f32x8 pf;
#pragma unroll
            for (int i = 0; i < 8; i++) pf[i] = s[kb][8 * t + i];
            pb[kb][t] = cvt8<T>(pf);
            if constexpr (!kDropout && (FA_ABLATE_FWD & 32) == 0) lp[0] = sum8_acc(pb[kb][t], lp[0]);
            // pinned here: sunk below the test of the row sums, the conversions would keep all fp32 values live across it (the dense d = 128
            // variant has the registers for that)
            if constexpr (D <= 64 || kDropout || kSparse) asm volatile("" : "+v"(pb[kb][t]));
          }
        lt = lp[0];
#pragma unroll
        for (int kb = 1; kb < KBW; kb++) lt += lp[kb];
        if (kDropout) {
#pragma unroll
          for (int kb = 0; kb < KBW; kb++) {
            KeepFields keep;
            if constexpr (kKeyWords) keep = keep_fields_row_layout(p.pk, key_words + (kb0 + kb) * 16, query_words, qrow, hf);
            else keep = keep_fields_row_layout(p.pk, (uint32_t)bh, qrow, n0 + (kb0 + kb) * 32, hf);
            // Dropped probabilities become 0 after the rounding, two a time: the keep decisions of a word of fields are 1 or 0 in each
            // half (two packed saturating subtractions), a packed 16-bit integer product applies them, and shifted together they are the
            // row's keep word.  Counted with SQ_INSTS_VALU over 64 x 16 heads x 1004 .. 1023, d = 64, p = 0.1, fp16, the forward issues 25.3 other
            // vector instructions per MFMA with this and the exchange of keep_fields_row_layout, 31.3 with a compare, a select and a shift per
            // score and the drawn words transposed over the quad: forward and backward together 1800 -> 1733 us.
            uint32_t kept[8];
#pragma unroll
            for (int i = 0; i < 8; i++) kept[i] = keep_pair(keep.w[i], p.keep_thr);
#pragma unroll
            for (int t = 0; t < 2; t++) {
              u32x4 pw = bitcast<u32x4>(pb[kb][t]);
#pragma unroll
              for (int i = 0; i < 4; i++) pw[i] = mul_pair(pw[i], kept[4 * t + i]);
              pb[kb][t] = bitcast<vec8>(pw);
            }
            if (kWords) {  // (dead scores keep whatever bit they drew: their P is 0)
              kwout[kb] = keep_word_of_row(kept, hf);
              kw_pending = (n0 >> 5) + kb0;
            }
          }
        }
      };
      // ---- online softmax (fmha_fprop_kernel_1xN.h:408-454,560-611 restated for a register-resident row).
      // The reference point m_i of the exponentials only moves when it has to: P may exceed 1 by a factor of up to
      // 2^kRescaleLog2, which the fp32 accumulators and the fp16/bf16 rounding of P absorb (numerator and denominator carry
      // the same factor, so the result is unchanged).  Whether it has to move is read off the tile's row sums - if a lane's
      // share is at most 2^kRescaleLog2, so is every P behind it - so the common tile takes no row maximum at all.  A tile
      // that fails the test (the first of a row always does: no reference point yet) is redone the long way: scores again,
      // row maxima, rescaled accumulators, probabilities against the new reference point.
      scores(std::false_type{});
      bool redo = __any(m_i == -INFINITY && (!kSparse || row_on));
      if (!redo) {
        probabilities();
        if constexpr ((FA_ABLATE_FWD & 32) == 0) redo = __any(!(lt <= kRescaleLimit));  // also catches inf and NaN
        if (__builtin_expect(redo, 0)) scores(std::true_type{});
      }
      if (__builtin_expect(redo, 0)) {
        float mt = s[0][0];
#pragma unroll
        for (int kb = 0; kb < KBW; kb++)
#pragma unroll
          for (int r = 0; r < 16; r++) mt = fmaxf(mt, s[kb][r]);
        mt = half_max(mt);
        if (kSparse && !row_on) mt = -INFINITY;
        const float m_new = fmaxf(m_i, mt);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = fast_exp2(m_i * cse - m_use * cse);
        m_i = m_new;
        l_i *= alpha;
#pragma unroll
        for (int i = 0; i < DV / 32; i++) o_acc[i] = o_acc[i] * alpha;
        probabilities();
      }
      l_i += lt;

      // ---- O^T += V^T P^T
#pragma unroll
      for (int kb = 0; kb < KBW; kb++) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
          for (int db = 0; db < DV / 32; db++) {
            const T* vp = Vs + ((kb0 + kb) * 32 + 16 * t) * D + voff[db];
            u32x4 av;
            if constexpr ((FA_ABLATE_FWD & 16) == 0) {
              u32x2 lo = lds_read_tr16(vp);
              u32x2 hi = lds_read_tr16(vp + 8 * D);
              av = u32x4{lo[0], lo[1], hi[0], hi[1]};
            } else {
              av = bitcast<u32x4>(qreg[db]);
            }
            if constexpr ((FA_ABLATE_FWD & 4) == 0) o_acc[db] = E::mfma32(bitcast<vec8>(av), pb[kb][t], o_acc[db]);
            else asm volatile("" ::"v"(av), "v"(pb[kb][t]));
          }
        }
      }
    }
    it = it_next;
  }
  flush_keep_words();
  // (the fragments are still there; stored in front of the loop, whose first step waits for everything outstanding, the rotated rows cost
  // every workgroup a store's latency: us of the kernel there / here, causal bf16, 8 x 12 x 1024 d = 64 27.0 / 26.6, d = 128 47.8 / 46.2, 2 x 16 x 2000 d = 128
  // 56.8 / 55.8; 23.3, 39 and 53.5 without rotary; kept out of the variants that take no rotary tables: a padded batch at d = 128 has no
  // register to spare, 169 are two waves per SIMD and 168 three: 16 x 16 heads x 512 .. 1024 fp16 130 / 119)
  if (!kSparse && kBias == 0 && p.q_rot != nullptr && kh == 0 && split == 0 && qrow < Lq) {
    T* const qo = reinterpret_cast<T*>(p.q_rot) + (int64_t)(q_begin + qrow) * p.qr_rs + (int64_t)h * p.qr_hs + hf * 8;
#pragma unroll
    for (int ks = 0; ks < D / 16; ks++) st_global16(qo + ks * 16, bitcast<u32x4>(qreg[ks]));
  }

  // ---- key split: the waves kh > 0 hand their partial (O, maximum, sum) to the wave kh == 0 of their rows, in the
  // accumulator's own register order (word (rs * (16 DV/32 + 2) + j) * 64 + lane: consecutive lanes, no bank conflicts)
  if (KS > 1) {
    __syncthreads();  // every wave has left the tiles
    constexpr int NJ = DV / 32 * 16 + 2;
    float* const X = reinterpret_cast<float*>(lds_raw) + rs * NJ * 64 + lane;
    if (kh != 0) {
#pragma unroll
      for (int db = 0; db < DV / 32; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) X[(db * 16 + r) * 64] = o_acc[db][r];
      X[(NJ - 2) * 64] = m_i;
      X[(NJ - 1) * 64] = l_i;
    }
    __syncthreads();
    if (kh == 0) {
      const float m_b = X[(NJ - 2) * 64], l_b = X[(NJ - 1) * 64];
      const float m_new = fmaxf(m_i, m_b);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float wa = fast_exp2(m_i * cse - m_use * cse), wb = fast_exp2(m_b * cse - m_use * cse);  // exp2(-inf) = 0
      m_i = m_new;
      l_i = l_i * wa + l_b * wb;
#pragma unroll
      for (int db = 0; db < DV / 32; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) o_acc[db][r] = o_acc[db][r] * wa + X[(db * 16 + r) * 64] * wb;
    }
    __syncthreads();  // the staging area of the stores below overlaps the exchange area
    if (kh != 0) return;
  }
  // ---- epilogue: normalise, write lse, transpose O^T through LDS for coalesced 16-byte stores
  const float l_tot = half_sum(l_i);
  const bool empty = !(l_tot > 0.f);  // also catches NaN (fmha_fprop_kernel_1xN.h:575,606)
  float inv = empty ? 1.f : fast_rcp(l_tot);
  if (kDropout) inv *= p.rp_keep;
  const float lse_val = empty ? -INFINITY : (m_i * cse + fast_log2(l_tot)) * kLn2;
  if (p.n_splits > 1) {  // partial result of this key split, fp32, merged by fwd_combine_kernel
    if (qrow < Lq) {
      if (hf == 0) p.lse_part[(((int64_t)split * p.B + b) * p.H + h) * p.sq_r + qrow] = lse_val;
      float* op = p.o_part + (((int64_t)split * p.total_q + q_begin + qrow) * p.H + h) * D;
#pragma unroll
      for (int db = 0; db < DV / 32; db++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
          const int d0 = db * 32 + g4 * 8 + hf * 4;
          if (d0 < D) {
            f32x4 x;
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = o_acc[db][g4 * 4 + i] * inv;
            *reinterpret_cast<f32x4*>(op + d0) = x;
          }
        }
    }
    return;
  }
  if (hf == 0 && qrow < Lq) p.lse[((int64_t)b * p.H + h) * p.sq_r + qrow] = lse_val;
  if (KS == 1) __syncthreads();
  constexpr int OS = Cfg::OS;
  T* Os = reinterpret_cast<T*>(lds_raw) + rs * 32 * OS;
#pragma unroll
  for (int db = 0; db < DV / 32; db++)
#pragma unroll
    for (int g4 = 0; g4 < 4; g4++) {
      const int d0 = db * 32 + g4 * 8 + hf * 4;
      if (d0 < D) {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = o_acc[db][g4 * 4 + i] * inv;
        *reinterpret_cast<typename E::vec4*>(Os + c * OS + d0) = cvt4<T>(x);
      }
    }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes have landed
  __builtin_amdgcn_wave_barrier();
  T* obase = reinterpret_cast<T*>(p.o) + (int64_t)q_begin * p.o_rs + (int64_t)h * p.o_hs;
#pragma unroll
  for (int i = 0; i < (32 * CH + 63) / 64; i++) {
    const int ch = lane + i * 64;
    const int row = ch / CH, col = (ch % CH) * 8;
    if constexpr (kRows) {  // rows past the last token are the entry's padding: zeros
      if ((32 * CH % 64 == 0 || ch < 32 * CH) && mw + row < p.max_sq) {
        u32x4 val = *reinterpret_cast<const u32x4*>(Os + row * OS + col);
        if (mw + row >= Lq) val = u32x4{0, 0, 0, 0};
        st_global16(reinterpret_cast<T*>(p.o) + ((int64_t)b * p.max_sq + row_of[mw + row]) * p.o_rs + (int64_t)h * p.o_hs + col, val);
      }
      continue;
    }
    int orow = mw + row;  // (sparse: the wave's rows are those of its two row blocks)
    if (kSparse) orow = (row < 16 ? rb_a : rb_b) < 0 ? 0x3fffffff : (row < 16 ? rb_a : rb_b) * 16 + (row & 15);
    if ((32 * CH % 64 == 0 || ch < 32 * CH) && orow < Lq) {
      u32x4 val = *reinterpret_cast<const u32x4*>(Os + row * OS + col);
      st_global16(obase + (int64_t)orow * p.o_rs + col, val);
    }
  }
}

template <typename T, int D, int BN, bool kRoomy, bool kCausal, bool kDropout, bool kSparse, int kBias = 0, int KS = 1,
          bool kWords = false>
__global__ void __launch_bounds__(256, fwd_waves(D, kDropout, kSparse, kBias % kPaddedRows, KS, kWords)) fa_fwd_kernel(const FwdParams p) {
  fa_fwd_body<T, D, BN, kRoomy, kCausal, kDropout, kSparse, kBias, KS, kWords, false>(p);
}
template <typename T, int D, int BN, bool kRoomy, bool kCausal, bool kDropout, bool kSparse, int kBias, int KS, bool kWords>
__global__ void __launch_bounds__(256, fwd_waves(D, kDropout, kSparse, kBias % kPaddedRows, KS, kWords)) fa_fwd_live_kernel(const FwdParams p) {
  fa_fwd_body<T, D, BN, kRoomy, kCausal, kDropout, kSparse, kBias, KS, kWords, true>(p);
}

}  // namespace fa
