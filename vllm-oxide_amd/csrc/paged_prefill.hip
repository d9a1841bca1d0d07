// Prefill attention over the paged KV cache (and over contiguous K/V), causal
// with an optional left window and GQA, for gfx950.
//
// What it computes: the seqlen_q >= 1 call of flash_attn_varlen_paged_windowed
// (crates/vllm-oxide/src/attention/flash_attn.rs:52-67) with window_right = 0,
// and, over contiguous K/V, flash_attn_varlen(..., causal = true)
// (flash_attn.rs:15-37, called from the prefill branch of qwen3.rs).  Sequence
// b has Lq = cu_seqlens_q[b+1] - cu_seqlens_q[b] query tokens and
// Lk = cu_seqlens_k[b+1] - cu_seqlens_k[b] keys; the masks are aligned to the
// bottom right (FlashAttention 2): query i, head h sees keys
//     j <= hi = i + Lk - Lq,   j >= hi - window_left (window_left >= 0 only),
// of kv head h / G.  Keys already in the cache before this step (a prefix
// hit, or earlier chunks of a chunked prefill) are simply the first Lk - Lq
// keys, so the paged form needs no gather.  A query with no visible key gets
// zeros.  fp32 accumulation, output rounded to the input dtype once.
//
// Work split: one workgroup of 4 waves per (128 (token, head) rows of one kv
// head's group, kv head, sequence).  Row r of the workgroup is token r / G,
// head r % G of the group, so the G heads that share a kv head share every
// K/V tile.  Each wave owns 32 rows, the 32 columns of its MFMA tiles (lanes l
// and l + 32 share row l % 32).  K/V advance in 64-key tiles loaded straight
// into LDS by the whole workgroup, two LDS buffers (one barrier per tile).
// Per tile and wave, with 32 x 32 x 16 MFMAs (half the issue cost per flop of
// 16 x 16 x 32, so the other wave's softmax work hides behind the matrix pipe):
//   * S^T[key][row] = K . Q^T: A = 32 keys x 16 d from the K tile (XOR-swizzled
//     16-byte chunks), B = the rows' queries, held in registers for the whole
//     kernel.  Lane l gets keys 8(r/4) + 4(l/32) + r%4 of each 32-key block.
//   * online softmax per row in the log2 domain; a row's keys sit in lanes l
//     and l ^ 32, so the maximum takes one v_permlane32_swap and the sums stay
//     per lane until the end.
//   * O^T[d][row] += V^T . P^T: A = V^T from two transposing LDS reads of the
//     row-major V tile (keys 16s + 4(l/32) + 0..3 and + 8 of a 32-key block),
//     B = the lane's own probabilities in the same key order (registers
//     8s..8s+7 of the score block), so P never moves between lanes.  Every
//     accumulator of a lane belongs to its own row: rescaling is a per-lane
//     multiply.
// Workgroup order is XCD-aware: all row tiles of one (sequence, kv head) run
// on one XCD (workgroup i runs on XCD i % 8), so its K/V is fetched from HBM
// once into that XCD's L2 and re-read from there; within a unit the tiles
// with the most keys (last tokens) start first.  Where such units would load the XCDs
// unevenly, each one's tiles alternate over 2, 4 or 8 of them (spread).  In large
// batches of short prompts of about one length (kPair) a workgroup takes two row tiles
// of its unit, n - 1 - i and then i; behind long cached contexts (kSplit) a row tile's
// keys are cut into pieces where that pays.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "cdna4_tile.hpp"
#include "decode_common.hpp"
#include "oxide_common.hpp"

namespace {

constexpr int kPfWaves = 4;
constexpr int kPfThreads = 64 * kPfWaves;
constexpr int kPfRows = kPfWaves * 32;  // (token, head) rows per workgroup
constexpr int kPfKeys = 64;             // keys per K/V tile
constexpr int kPfXcds = 8;

struct PrefillParams {
  const void* q;    // [total_q, Hq, D]
  const void* k;    // paged [NB, BS, Hkv, D] or contiguous [total_k, Hkv, D]
  const void* v;
  void* out;        // [total_q, Hq, D]
  const uint32_t* cu_seqlens_q;
  const uint32_t* cu_seqlens_k;
  const int32_t* block_table;  // null: contiguous K/V, key j of b at row cu_seqlens_k[b] + j
  int64_t max_blocks;
  int64_t num_rows;            // rows of the K/V view (clamp for bad indices)
  int num_blocks;
  int max_seqlen_q;
  int max_seqlen_k;
  int num_heads;
  int num_kv_heads;
  int group;
  int tokens_per_wg;
  int tiles_per_unit;
  int units;                   // batch * num_kv_heads
  int spread;                  // XCDs that share a unit's row tiles (plain grid)
  int share_tiles;             // row tiles of a unit per XCD of its share
  int block_size;
  int window_left;
  float scale_log2;
  // Shared-prefix pass of a decode batch (kernel instances with kPrefix): the rows
  // are the decode batch's (sequence, query head) pairs -- q [dec_batch, Hq, D],
  // cu_seqlens_k the decode batch's -- and the keys are the leading block-table
  // entries that every row shares (at most shared_hint of them; the kernel finds
  // how many), cut into pre_splits splits of split_keys keys.  Each (split,
  // sequence, head) writes a normalised partial row and its log2-sum-exp at row
  // pre_row0 + split * dec_batch * Hq + b * Hq + h of part_o / part_lse.
  float* part_o;
  float* part_lse;
  int64_t pre_row0;
  int pre_splits;
  int split_keys;
  int shared_hint;
  int dec_batch;
  int* shared_out;  // the number of shared blocks found (written by workgroup 0)
  int pair;         // 1: the kPair instances
  // Balanced launch (kernel instances with kSplit): the most pieces it cuts, and the
  // batch size.  Partial rows go to part_o / part_lse, row piece * kPfRows + row.
  int max_pieces;
  int slots;       // workgroups that run at once
  int may_be_whole;  // whether it asks the real lengths if cutting pays
  int batch;
  int* piece_len;  // the piece length chosen (workgroup 0 writes it, the merge reads it)
};

__device__ __forceinline__ int clamp_len(int64_t n, int cap) {
  return static_cast<int>(n < 0 ? 0 : (n > cap ? cap : n));
}

// Balanced launch: the 64-key steps of every row tile of sequence b are cut into n_b
// equal pieces, one workgroup each.  Pieces are numbered sequence by sequence, inside
// one by kv head, then key range, then row tile: neighbouring workgroups, on one XCD,
// walk the same keys for different rows, so K/V comes from that XCD's L2.  (Ranges of
// equal length over the rows' steps laid end to end balance perfectly, but every
// workgroup then streams its own keys: 337 us for two chunks behind 16k-24k keys
// against 300-310 with the pieces.)  The piece length is the shortest for which all
// pieces run at once (slots workgroups), or in two rounds where rounding to whole
// pieces costs the single round more than an eighth; where the lengths are such that
// whole tiles take no longer (plain_us, split_us), no tile is cut and the merge ends at
// once.
// Lane b of every wave holds sequence b's entry (so at most 64 sequences).
constexpr int kPfSplitBatch = 64;
constexpr int kPfMinPiece = 8;
struct SeqPieces {
  int q;       // clamped query count
  int tiles;   // row tiles per kv head
  int steps;   // steps of a tile (of its last tile; earlier ones leave a few empty)
  int n;       // pieces of a tile
  int first;   // number of its first piece
  int total;   // all sequences' pieces (the same in every lane)
  bool whole;  // no tile is cut (the same in every lane)
};
__host__ __device__ __forceinline__ int steps_per_tile(int keys, int window_left, int tokens_per_wg) {
  const int all = (keys + kPfKeys - 1) / kPfKeys;
  if (window_left < 0 || window_left >= keys) return all;
  const int n = (window_left + tokens_per_wg + 2 * kPfKeys - 2) / kPfKeys;
  return n < all ? n : all;
}
// Inclusive sums over the lanes (lane 63 holds the total), on the VALU.
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15, rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31, rows 2 and 3
  return v;
}
__device__ __forceinline__ int wave_total(int v) { return __builtin_amdgcn_readlane(wave_scan(v), 63); }
// The largest of the lanes' non-negative values.
__device__ __forceinline__ int wave_max(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
  return __builtin_amdgcn_readlane(v, 63);
}

// Expected times, in us, of whole tiles in the plain order (work steps in all, the longest
// tile's longest) and of pieces of at most len steps, start-up aside.  A step (128 rows x
// 64 keys) takes about 1.06 us with one workgroup on a CU and 1.9 with two at D = 128,
// 0.75 and 1.1 at D = 64.  More tiles than slots end raggedly: 640 tiles of 128 steps 380
// us, of 98-125 335 whole and 417 cut.
__host__ __device__ __forceinline__ float plain_us(int tiles, int work, int longest, int slots, int d) {
  const float alone = d == 128 ? 1.06f : 0.75f, both = d == 128 ? 1.9f : 1.1f;
  if (2 * tiles <= slots) return alone * longest;
  const float once = alone * longest + (both - alone) * (static_cast<float>(work) / tiles);
  return tiles > slots ? fmaxf(once, 1.25f * both * work / slots) : once;
}
// Each piece writes and the merge reads fp32 rows; the merge is a launch, and pieces in
// two rounds start up twice (28 x 64 behind 1k-4k 112 us whole, 123 cut; 14 x 128 99 and
// 110; 15 of 20-118 behind 0.5k-4k 103 and 88).
__host__ __device__ __forceinline__ float split_us(int pieces, int tiles, int work, int len, int slots, int d) {
  const float alone = d == 128 ? 1.06f : 0.75f, both = d == 128 ? 1.9f : 1.1f;
  const float steps = 2 * pieces <= slots ? alone * len
                      : pieces <= slots   ? both * len
                                          : both * (tiles > slots ? 1.6f : 1.15f) * work / slots + 18.f;
  return steps + 1e-4f * d * pieces + 7.f;
}
constexpr int kPfWhole = INT32_MAX;  // the piece length stored where no tile is cut

// The shortest piece length, at least kPfMinPiece, at which the sequences (units row
// tiles of steps steps each, per lane; tiles and work in all) make at most `slots` pieces.
__device__ __forceinline__ int shortest_piece(int units, int steps, int slots, int tiles, int work) {
  // units * steps / len <= pieces <= units * (steps / len + 1) bound the bisection.
  int lo = max(kPfMinPiece, (work + slots - 1) / slots);
  int hi = max(lo, slots > tiles ? (work + slots - tiles - 1) / (slots - tiles) : wave_max(units > 0 ? steps : 0));
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (wave_total(units * ((steps + mid - 1) / mid)) <= slots)
      hi = mid;
    else
      lo = mid + 1;
  }
  return lo;
}
// kMerge: the piece length comes from the first pass.
template <bool kMerge, int D>
__device__ __forceinline__ SeqPieces seq_pieces(const PrefillParams& p) {
  const int lane = threadIdx.x & 63;
  SeqPieces s{};
  int k = 0;
  if (lane < p.batch) {
    s.q = clamp_len(static_cast<int64_t>(p.cu_seqlens_q[lane + 1]) - p.cu_seqlens_q[lane], p.max_seqlen_q);
    k = clamp_len(static_cast<int64_t>(p.cu_seqlens_k[lane + 1]) - p.cu_seqlens_k[lane], p.max_seqlen_k);
  }
  s.tiles = (s.q + p.tokens_per_wg - 1) / p.tokens_per_wg;
  s.steps = max(steps_per_tile(k, p.window_left, p.tokens_per_wg), 1);
  const int units = p.num_kv_heads * s.tiles;  // row tiles of the sequence
  int len;
  if (kMerge) {
    len = __builtin_amdgcn_readfirstlane(*p.piece_len);
  } else {
    const int tiles = wave_total(units), work = wave_total(units * s.steps);
    len = shortest_piece(units, s.steps, p.max_pieces, tiles, work);
    if (p.max_pieces > p.slots && tiles <= p.slots) {
      const int one = shortest_piece(units, s.steps, p.slots, tiles, work);
      if (8 * one <= 18 * len) len = one;
    }
    if (p.may_be_whole) {
      const int longest = wave_max(units > 0 ? s.steps : 0);
      const int pieces = wave_total(units * ((s.steps + len - 1) / len));
      if (pieces == tiles ||
          plain_us(tiles, work, longest, p.slots, D) <= split_us(pieces, tiles, work, len, p.slots, D))
        len = kPfWhole;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *p.piece_len = len;
  }
  s.whole = len == kPfWhole;
  s.n = s.whole ? 1 : (s.steps + len - 1) / len;
  const int mine = units * s.n;
  const int sum = wave_scan(mine);
  s.first = sum - mine;
  s.total = __builtin_amdgcn_readlane(sum, 63);
  return s;
}

// LDS tile layouts (64 keys, row = one key's head slice of 2*D bytes):
//   K: 16-byte chunk c of row r at chunk position c ^ kswz(r).  One MFMA
//      operand read (16 lanes = 16 consecutive rows, one chunk each) then
//      covers all 64 banks: rows are 256 B apart at D = 128 (kswz = r % 16);
//      at D = 64 rows r and r + 1 sit in opposite bank halves and
//      kswz = (r >> 1) % 8 separates the 8 pairs.
//   V: 32-byte granule g of row r at granule position g ^ vswz(r).  One
//      transposing read covers 4 consecutive rows x 2 adjacent granules per
//      half-wave; vswz = 2 (r % 4) at D = 128 (and r & 2 at D = 64, where
//      odd rows add half a bank sweep) maps those 8 pieces to distinct banks.
// Both are written by direct global -> LDS loads (global_load_lds_dwordx4):
// lane i of a wave instruction fills bytes [16 i, 16 i + 16) of a 1 KiB run,
// so each lane loads the source chunk that belongs at its LDS position.
template <int D>
__device__ __forceinline__ int kswz(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int vswz(int r) {
  return D == 128 ? 2 * (r & 3) : (r & 2);
}

// One direct global -> LDS load of 16 bytes per lane: lane i writes LDS bytes
// [lds + 16 i, lds + 16 i + 16).  Issued as inline assembly so the compiler
// does not treat the in-flight loads as possibly aliasing the other buffer's
// LDS reads (it otherwise waits for them before some transposing reads); the
// kernel waits for them itself (vmcnt(0) before the barrier that publishes
// the tile).  `lds`, the LDS byte address, must be wave-uniform; the s_nop is the wait
// state between a scalar write of m0 and a load to LDS.
__device__ __forceinline__ void load_lds16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src)
               : "memory", "m0");
}
// The same from a wave-uniform base address plus a 32-bit per-lane byte offset.
__device__ __forceinline__ void load_lds16(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
// LDS byte address of a shared object (what m0 of a direct load holds).
__device__ __forceinline__ uint32_t lds_addr(const char* p) {
  return __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p)));
}

// K/V addressing of a kernel instance.
enum PrefillAddressing {
  kContiguous = 0,  // key j of sequence b at row cu_seqlens_k[b] + j
  kPagedTiles = 1,  // paged, block_size a multiple of the 64-key tile: one block per tile
  kPagedRows = 2,   // paged, any block_size: a block lookup per row
};

template <class Tag, int D, int MODE, bool kPrefix, bool kPair = false, bool kSplit = false>
__global__ __launch_bounds__(kPfThreads, 2) void paged_prefill_attn(PrefillParams p) {
  constexpr int CH = D / 8;                  // 16-byte chunks per head row
  constexpr int KS = D / 16;                 // MFMA k-steps of Q.K (16 dims each)
  constexpr int NDB = D / 32;                // 32-wide d blocks of O (two 32-byte V granules)
  constexpr int ROWB = 2 * D;                // bytes per tile row
  constexpr int TBYTES = kPfKeys * ROWB;     // one K or V tile
  constexpr int BUF = 2 * TBYTES;            // K tile | V tile
  constexpr int RPI = 1024 / ROWB;           // tile rows per wave load instruction
  constexpr int WROWS = kPfKeys / kPfWaves;  // tile rows loaded by each wave
  constexpr int NLD = WROWS / RPI;           // load instructions per wave and tensor
  static_assert(WROWS % RPI == 0, "tile rows");
  // Two LDS buffers as separate objects: the loop is unrolled by two so each
  // access names its buffer statically, which lets the compiler see that the
  // loads in flight into one buffer do not alias reads of the other.
  __shared__ __align__(1024) char smem0[BUF];
  __shared__ __align__(1024) char smem1[BUF];

  // XCD-aware work item: unit (sequence, kv head) u sits on XCD u % 8 and its
  // tiles are consecutive workgroups there, heaviest first; where the units are no
  // multiple of 8, each unit's tiles alternate over `spread` XCDs, so that all 8 get
  // the same share.  Shared-prefix pass:
  // unit (key split, kv head), all of them over table row 0 (the shared entries).
  // Balanced launch: XCD x takes the x-th eighth of the pieces.
  const int i = blockIdx.x;
  const int j = i / kPfXcds;
  int u = 0, jj = 0;  // unit and place among its tiles; false where the grid has none
  auto plain_item = [&]() {
    const int share = (j / p.share_tiles) * kPfXcds + i % kPfXcds;
    u = share / p.spread;
    jj = (j % p.share_tiles) * p.spread + share % p.spread;
    return u < p.units && jj < p.tiles_per_unit;
  };
  if (!kSplit && !plain_item()) return;
  // kPair: a workgroup takes row tiles n - 1 - jj and then jj (half of the workgroups
  // end at once) where the prompts are of about one length; in ragged batches the pairs
  // would be uneven.
  bool pair = false;
  if constexpr (kPair) {
    const int64_t total = static_cast<int64_t>(p.cu_seqlens_q[p.batch]) - p.cu_seqlens_q[0];
    pair = 4 * total >= 3 * static_cast<int64_t>(p.batch) * p.max_seqlen_q;
    if (pair && jj >= (p.tiles_per_unit + 1) / 2) return;
  }
  for (int pass = 0; pass < (kPair ? 2 : 1); ++pass) {
  int tile, b, kh, split = 0;
  int piece = 0, s0 = 0, s1 = 0;  // kSplit: the piece and its steps of the tile
  bool whole = true;
  if constexpr (kSplit) {
    const SeqPieces seqs = seq_pieces<false, D>(p);
    if (seqs.whole) {  // as the plain grid
      if (!plain_item()) return;
      tile = p.tiles_per_unit - 1 - jj;
      b = u / p.num_kv_heads;
      kh = u % p.num_kv_heads;
      s1 = 1 << 24;
    } else {
      const int per_xcd = (seqs.total + kPfXcds - 1) / kPfXcds;
      piece = (i % kPfXcds) * per_xcd + j;
      if (j >= per_xcd || piece >= min(seqs.total, p.max_pieces)) return;
      // The last sequence whose first piece is not past this one (sequences without
      // queries share their successor's first, so it is the one that holds it).
      b = 63 - __builtin_clzll(__ballot(static_cast<int>(threadIdx.x & 63) < p.batch && seqs.first <= piece));
      const int in_seq = piece - __builtin_amdgcn_readlane(seqs.first, b);
      const int tiles = __builtin_amdgcn_readlane(seqs.tiles, b);
      const int steps = __builtin_amdgcn_readlane(seqs.steps, b);
      const int n = __builtin_amdgcn_readlane(seqs.n, b);
      kh = in_seq / (tiles * n);
      const int x = in_seq / tiles % n;
      tile = in_seq % tiles;
      s0 = static_cast<int>(static_cast<int64_t>(steps) * x / n);
      s1 = static_cast<int>(static_cast<int64_t>(steps) * (x + 1) / n);
      whole = n == 1;
    }
  } else {
    tile = pass == 0 ? p.tiles_per_unit - 1 - jj : jj;
    if (pass == 1) {
      if (!pair || tile >= p.tiles_per_unit - 1 - jj) break;  // (the middle tile of an odd count: done)
      __syncthreads();  // the previous tile's last LDS reads before this tile's first loads
    }
    b = kPrefix ? 0 : u / p.num_kv_heads;
    kh = u % p.num_kv_heads;
    split = kPrefix ? u / p.num_kv_heads : 0;
  }

  int Lq, Lk;
  if constexpr (kPrefix) {
    const int shared = find_shared_blocks<kPfThreads>(p.cu_seqlens_k, p.block_table, p.max_blocks, p.dec_batch,
                                                      p.block_size, p.max_seqlen_k, p.shared_hint);
    if (blockIdx.x == 0 && threadIdx.x == 0) *p.shared_out = shared;
    Lq = p.dec_batch;
    Lk = shared * p.block_size;  // the shared keys; no sequence attends past them here
    if (split * p.split_keys >= Lk) continue;
  } else {
    Lq = clamp_len(static_cast<int64_t>(p.cu_seqlens_q[b + 1]) - p.cu_seqlens_q[b], p.max_seqlen_q);
    Lk = clamp_len(static_cast<int64_t>(p.cu_seqlens_k[b + 1]) - p.cu_seqlens_k[b], p.max_seqlen_k);
  }
  const int t0 = tile * p.tokens_per_wg;
  if (t0 >= Lq) continue;
  const int t1 = min(Lq, t0 + p.tokens_per_wg);
  const int off = Lk - Lq;  // hi of token t is t + off
  const int G = p.group;
  const int W = p.window_left;

  // Key range of the workgroup: [klo, khi] (empty when khi < klo).  Shared-prefix
  // pass: the split's keys, every row seeing all of them but those before its window.
  // Balanced launch: steps s0 .. s1 - 1 of the tile's keys.
  int khi = kPrefix ? min(Lk, (split + 1) * p.split_keys) - 1 : min(Lk - 1, t1 - 1 + off);
  const int klo = kPrefix ? split * p.split_keys : (W >= 0 ? max(0, t0 + off - W) : 0);
  int kt0 = klo & ~(kPfKeys - 1);
  if constexpr (kSplit) {
    khi = min(khi, kt0 + s1 * kPfKeys - 1);
    kt0 += s0 * kPfKeys;
    if (khi < kt0) khi = -1;  // past the tile's last key
  }
  const int ntiles = khi >= klo && khi >= kt0 ? (khi - kt0) / kPfKeys + 1 : 0;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t q0 = kPrefix ? 0 : p.cu_seqlens_q[b];
  const int rows_used = p.tokens_per_wg * G;

  // This lane's row (column l % 32 of the MFMA tiles; lanes l and l + 32 share
  // it and hold alternate groups of four keys): token, head, key range.
  const int r32 = lane & 31;
  const int half = lane >> 5;
  const int rr = wave * 32 + r32;
  const int tq = t0 + rr / G;
  const bool valid = rr < rows_used && tq < t1;
  const int64_t qrow = valid ? (q0 + tq) * p.num_heads + kh * G + rr % G : 0;
  int hi_r = valid ? tq + off : -1;
  int lo_r = valid && W >= 0 ? tq + off - W : 0;
  if constexpr (kPrefix) {
    // Decode sequence tq attends keys [max(0, L - 1 - W), L) of which the shared
    // ones are [.., Lk); this split holds [klo, khi].
    const int L = valid ? clamp_len(static_cast<int64_t>(p.cu_seqlens_k[tq + 1]) - p.cu_seqlens_k[tq],
                                    p.max_seqlen_k)
                        : 0;
    hi_r = valid ? khi : -1;
    lo_r = valid && W >= 0 ? L - 1 - W : 0;
  }
  // The wave's own tiles [it0, it1): those in which some row of it sees a key (none
  // without rows).  The others it only loads for the rest.
  const int wt_first = __builtin_amdgcn_readlane(tq, 0);  // lanes 0 and 31 hold its first and last row
  int it0 = ntiles, it1 = ntiles;
  if (wave * 32 < rows_used && wt_first < t1) {
    const int wt_last = min(t1 - 1, __builtin_amdgcn_readlane(tq, 31));
    const int wave_hi = kPrefix ? khi : min(Lk - 1, wt_last + off);
    const int wave_lo = !kPrefix && W >= 0 ? wt_first + off - W : 0;
    it1 = wave_hi >= kt0 ? min(ntiles, (wave_hi - kt0) / kPfKeys + 1) : 0;
    it0 = wave_lo > kt0 ? min(it1, (wave_lo - kt0) / kPfKeys) : 0;
  }

  // Queries (B operand of S^T, 16 dims per k-step).  A negative scale is
  // applied as a sign flip of q (exact) and |scale|, so the running maxima can
  // be taken on raw scores.
  const uint32_t qflip = p.scale_log2 < 0.f ? 0x80008000u : 0u;
  const float c_log2 = fabsf(p.scale_log2);
  uint4 qb[KS];  // loaded after the first tile's loads are issued

  // Direct tile loads: wave w fills tile rows [16 w, 16 w + 16); lane -> (row
  // within the 1 KiB run, 16-byte position), source chunk chosen by the swizzle.
  const int lrow = lane / CH;         // row within the run
  const int lpos = lane % CH;         // 16-byte position within the row
  const int64_t row_stride = static_cast<int64_t>(p.num_kv_heads) * D;
  const uint16_t* kbase = static_cast<const uint16_t*>(p.k) + kh * D;
  const uint16_t* vbase = static_cast<const uint16_t*>(p.v) + kh * D;
  const int64_t kstart = p.cu_seqlens_k[b];
  // Block table read through the constant address space (scalar loads, one per page).
  typedef __attribute__((address_space(4))) const int32_t bt_t;
  bt_t* bt = (bt_t*)(p.block_table + (MODE == kContiguous ? 0 : b * p.max_blocks));
  // Per-lane constants: tile row of each load, its byte offset in the tile's
  // source rows, and the swizzled source chunks.
  const uint32_t strideb = static_cast<uint32_t>(row_stride * 2);
  int trow[NLD];
  uint32_t rowb[NLD], kchb[NLD], vchb[NLD];
  int blk_row[NLD], in_row[NLD];  // kPagedRows: the next tile's block ids, the rows inside them
#pragma unroll
  for (int x = 0; x < NLD; ++x) {
    trow[x] = wave * WROWS + x * RPI + lrow;
    kchb[x] = 16 * (lpos ^ kswz<D>(trow[x]));
    vchb[x] = 32 * ((lpos >> 1) ^ vswz<D>(trow[x])) + 16 * (lpos & 1);
    rowb[x] = static_cast<uint32_t>(trow[x]) * strideb;
    blk_row[x] = in_row[x] = 0;
  }
  // The tile being fetched (tiles are fetched in order): its first key, and for
  // kPagedTiles its page, the offset inside it, that page's block and the next one's.
  int f_kb = kt0;
  int f_in = 0, f_page = 0, f_blk = 0, f_next = 0;
  const int last_page = ntiles > 0 ? khi / p.block_size : 0;
  if (MODE == kPagedTiles && ntiles > 0) {
    f_page = kt0 / p.block_size;
    f_in = kt0 % p.block_size;
    f_blk = bt[f_page];
    f_next = bt[min(f_page + 1, last_page)];
  }
  // kPagedRows: block ids of the tile at f_kb, read a tile ahead of its loads.
  // One division per row and tile: taking the remainder again at each of the row's loads
  // cost 64 more VALU operations between a step's score MFMAs (pages of 16, 4 x 2048
  // 169 -> 180 us).
  auto fetch_rows = [&]() {
    if (MODE == kPagedRows) {
#pragma unroll
      for (int x = 0; x < NLD; ++x) {
        const uint32_t key = min(f_kb + trow[x], Lk - 1);
        const uint32_t entry = key / static_cast<uint32_t>(p.block_size);
        blk_row[x] = p.block_table[b * p.max_blocks + entry];
        in_row[x] = static_cast<int>(key - entry * p.block_size);
      }
    }
  };
  // Wave-uniform source of the tile at f_kb: base rows and the byte offset of its
  // last valid row (rows past it repeat it).
  const uint16_t* f_k = kbase;
  const uint16_t* f_v = vbase;
  uint32_t f_limb = 0;
  auto locate_tile = [&]() {
    if (MODE == kPagedRows) return;
    int64_t row0;
    int lim;
    if (MODE == kPagedTiles) {
      row0 = static_cast<int64_t>(min(max(f_blk, 0), p.num_blocks - 1)) * p.block_size + f_in;
      lim = Lk - 1 - f_kb;
    } else {
      row0 = min(kstart + f_kb, p.num_rows - 1);
      lim = static_cast<int>(min<int64_t>(Lk - 1 - f_kb, p.num_rows - 1 - row0));
    }
    f_limb = static_cast<uint32_t>(min(lim, kPfKeys - 1)) * strideb;
    f_k = kbase + row0 * row_stride;
    f_v = vbase + row0 * row_stride;
  };
  // Load x of the 2 NLD loads of the located tile (K, V alternating).
  auto issue_load = [&](int x2, uint32_t sbuf) {
    const int x = x2 >> 1;
    const uint32_t dst = sbuf + (wave * WROWS + x * RPI) * ROWB + (x2 & 1) * TBYTES;
    if (MODE == kPagedRows) {
      // General pages: a 64-bit source address per lane.
      const int blk = min(max(blk_row[x], 0), p.num_blocks - 1);
      const int64_t row = static_cast<int64_t>(blk) * p.block_size + in_row[x];
      if (x2 & 1)
        load_lds16(vbase + row * row_stride + vchb[x] / 2, dst);
      else
        load_lds16(kbase + row * row_stride + kchb[x] / 2, dst);
    } else {
      const uint32_t rb = min(rowb[x], f_limb);
      if (x2 & 1)
        load_lds16(f_v, rb + vchb[x], dst);
      else
        load_lds16(f_k, rb + kchb[x], dst);
    }
  };
  // After a tile's loads are issued: on to the next one.
  auto next_tile = [&]() {
    f_kb += kPfKeys;
    if (f_kb > khi) {  // no further tile
      f_limb = 0;
      return;
    }
    if (MODE == kPagedTiles) {
      f_in += kPfKeys;
      if (f_in >= p.block_size) {
        f_in = 0;
        ++f_page;
        f_blk = f_next;
        f_next = bt[min(f_page + 1, last_page)];
      }
    }
    fetch_rows();
    locate_tile();
  };

  float m_r = -INFINITY;  // running max of raw scores (x |scale| log2 e)
  // Row sum of the probabilities as rounded for the P.V product (packed
  // pairs summed by v_dot2c), over this lane's half of the keys.
  float lsum = 0.f;
  floatx16 acc[NDB];
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db][r] = 0.f;

  const uint32_t lds0 = lds_addr(smem0), lds1 = lds_addr(smem1);
  // One tile: scores, softmax, P.V.  The next tile's loads go out between the score
  // MFMAs, one per k-step: issued together behind the barrier, the eight loads of all
  // four waves queued at the address unit for ~540-660 of a step's ~2900 (one wave per
  // SIMD) to ~3800 cycles (two), with the wave stalled at each.  4 x 4096 566 -> 530 us,
  // two 250-512-token chunks behind 8k-24k cached keys 452 -> 383 us.  After the last
  // tile they re-read one row of it (no branch in the MFMA sequence).
  auto step = [&](int it, const char* cur, uint32_t nxt) {
    const int kb0 = kt0 + it * kPfKeys;
    // Tile it has landed in LDS (own loads, then everyone's); the next tile goes
    // into the other buffer, whose readers finished before this barrier.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    {
      const uint4* sk = reinterpret_cast<const uint4*>(cur);
      const char* sv = cur + TBYTES;

      // S^T of two 32-key blocks: lane l holds keys 8 (r / 4) + 4 half + r % 4
      // of block kb for its row.  Operands are read kAhead k-steps early (2, 3 and 4
      // measured within 1 % of 1).
      constexpr int kAhead = 1;
      static_assert(2 * NLD == KS, "one load per k-step");
      floatx16 sc[2];
      uint4 ka[kAhead + 1][2];
      auto read_k = [&](int ks) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
          ka[ks % (kAhead + 1)][kb] = sk[(kb * 32 + r32) * CH + ((2 * ks + half) ^ kswz<D>(r32))];
      };
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kb][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < kAhead; ++ks) read_k(ks);
      // The score MFMAs ahead of the other workgroup's waves: 16 x 1024 186.6 -> 181.7 us,
      // 4 x 4096 unchanged; P.V too measured 1-8 % slower.
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + kAhead < KS) read_k(ks + kAhead);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) sc[kb] = mfma32x32x16(Tag{}, ka[ks % (kAhead + 1)][kb], qb[ks], sc[kb]);
        issue_load(ks, nxt);
        __builtin_amdgcn_sched_barrier(0);
      }

      // Mask only where the tile crosses some row's key range.
      const bool lane_mask = !(kb0 >= lo_r && kb0 + kPfKeys - 1 <= hi_r);
      if (__ballot(lane_mask) != 0) {
        const int k0 = kb0 + 4 * half;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = k0 + kb * 32 + 8 * (r / 4) + r % 4;
            sc[kb][r] = (key > hi_r || key < lo_r) ? -INFINITY : sc[kb][r];
          }
      }
      __builtin_amdgcn_s_setprio(0);

      // Row maximum: four independent chains of three-way maxima.
      float mc[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const floatx16& v = sc[c / 2];
        const int r = 8 * (c % 2);
        mc[c] = fmaxf(fmaxf(v[r], v[r + 1]), v[r + 2]);
        mc[c] = fmaxf(fmaxf(mc[c], v[r + 3]), v[r + 4]);
        mc[c] = fmaxf(fmaxf(mc[c], v[r + 5]), v[r + 6]);
      }
      float mt = fmaxf(fmaxf(mc[0], mc[1]), sc[0][7]);
      mt = fmaxf(fmaxf(mt, mc[2]), sc[0][15]);
      mt = fmaxf(fmaxf(mt, mc[3]), sc[1][7]);
      mt = fmaxf(mt, sc[1][15]);
      {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
        const float a = __uint_as_float(sw[0]), b = __uint_as_float(sw[1]);
        mt = a > b ? a : b;
      }
      // Lazy rescaling: keep the old maximum while the tile's stays within
      // 2^8 of it (probabilities <= 256, exact in fp32 and bf16 range), so
      // most tiles skip the accumulator multiplies.
      const float ms = mt * c_log2;
      const bool grow = ms > m_r + 8.f;
      float alpha = 1.f;
      if (grow) {
        alpha = __builtin_amdgcn_exp2f(m_r - ms);
        m_r = ms;
      }
      if (__ballot(grow) != 0) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) acc[db] *= alpha;
        lsum *= alpha;
      }
      const float msafe = m_r == -INFINITY ? 0.f : m_r;

      // P^T: the 8 registers 8 s .. 8 s + 7 of block kb are the B operand of
      // k-step (kb, s), keys kb * 32 + 16 s + 4 half + {0..3} and + 8 + {0..3}.
      uint4 pb[2][2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][r], c_log2, -msafe));
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          pb[kb][s2].x = pack2_cvt(Tag{}, x[8 * s2 + 0], x[8 * s2 + 1]);
          pb[kb][s2].y = pack2_cvt(Tag{}, x[8 * s2 + 2], x[8 * s2 + 3]);
          pb[kb][s2].z = pack2_cvt(Tag{}, x[8 * s2 + 4], x[8 * s2 + 5]);
          pb[kb][s2].w = pack2_cvt(Tag{}, x[8 * s2 + 6], x[8 * s2 + 7]);
          lsum = sum2_acc(Tag{}, pb[kb][s2].x, lsum);
          lsum = sum2_acc(Tag{}, pb[kb][s2].y, lsum);
          lsum = sum2_acc(Tag{}, pb[kb][s2].z, lsum);
          lsum = sum2_acc(Tag{}, pb[kb][s2].w, lsum);
        }
      }

      // O^T += V^T . P^T: the A operand of d block db for k-step (kb, s) is two
      // transposing reads; lane i of 16-lane group g reads key row
      // kb * 32 + 16 s + 4 half + i / 4 (and + 8), 4 dims at
      // 32 db + 16 (g % 2) + 4 (i % 4), i.e. granule 2 db + g % 2.
      const int gsub = (lane >> 4) & 1;
      const int i16 = lane & 15;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const int rlo = kb * 32 + 16 * s2 + 4 * half + i16 / 4;
          const char* vlo = sv + rlo * ROWB + 8 * (i16 % 4);
          const char* vhi = vlo + 8 * ROWB;
          const int zlo = vswz<D>(rlo), zhi = vswz<D>(rlo + 8);
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            const int g = 2 * db + gsub;
            const uint2 a0 = lds_read_tr16(vlo + 32 * (g ^ zlo));
            const uint2 a1 = lds_read_tr16(vhi + 32 * (g ^ zhi));
            const uint4 va = make_uint4(a0.x, a0.y, a1.x, a1.y);
            acc[db] = mfma32x32x16(Tag{}, va, pb[kb][s2], acc[db]);
          }
        }
    }
    next_tile();
  };
  if (ntiles > 0) {
    fetch_rows();
    locate_tile();
#pragma unroll
    for (int x = 0; x < 2 * NLD; ++x) issue_load(x, lds0);
    next_tile();
  }
  // The queries load while the first tile is in flight: k-step ks takes dims
  // 16 ks + 8 half .. + 7.
  {
    const uint16_t* qp = static_cast<const uint16_t*>(p.q) + qrow * D;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 v = valid ? *reinterpret_cast<const uint4*>(qp + 16 * ks + 8 * half) : make_uint4(0, 0, 0, 0);
      v.x ^= qflip; v.y ^= qflip; v.z ^= qflip; v.w ^= qflip;
      qb[ks] = v;
    }
  }

  // A tile that no row of the wave sees is left out of its math: P is 0 there, but 0
  // times an infinite or NaN V is not.  The loops are split at the borders because a
  // branch around the math inside step would cost every wave copies of its accumulators
  // where it joins.  Against running every tile of the workgroup, one query head per kv
  // head: 16 x 1024 115 -> 109 us, with a window of 128 66 -> 63; 4 x 2048, and groups of
  // two and four with or without a window, within 1 %.
  auto load_only = [&](int from, int to) {
    for (int it = from; it < to; ++it) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
#pragma unroll
      for (int x = 0; x < 2 * NLD; ++x) issue_load(x, it % 2 == 0 ? lds1 : lds0);
      next_tile();
    }
  };
  load_only(0, it0);
  int it = it0;
  if (it0 % 2 == 1 && it0 < it1) step(it++, smem1, lds0);
  for (; it < it1; it += 2) {
    step(it, smem0, lds1);
    if (it + 1 < it1) step(it + 1, smem1, lds0);
  }
  load_only(it1, ntiles);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last step's loads, before the wave ends

  // out[row][d] for d = 32 db + 8 q + 4 half + e (register 4 q + e), normalised
  // by the row total (both halves of the keys).
  lsum = sum_over_halves(lsum);
  const bool partial = kPrefix || !whole;
  if (partial && valid) {
    // Normalised partial row and its log2-sum-exp (scores are in units of
    // |scale| log2 e, as the decode passes' partials).
    const float l = lsum;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int64_t prow = kSplit ? static_cast<int64_t>(piece) * kPfRows + rr
                                : p.pre_row0 + static_cast<int64_t>(split) * p.dec_batch * p.num_heads + qrow;
    float* po = p.part_o + prow * D + 4 * half;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(po + 32 * db + 8 * q) =
            make_float4(acc[db][4 * q + 0] * inv, acc[db][4 * q + 1] * inv, acc[db][4 * q + 2] * inv,
                        acc[db][4 * q + 3] * inv);
    // A row whose sum is NaN says so in kSplit, whose merge would take -inf for no keys.
    const bool sums = kSplit ? l != 0.f : l > 0.f;
    if (half == 0) p.part_lse[prow] = sums ? m_r + log2f(l) : -INFINITY;
  } else if (valid) {
    const float l = lsum;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint16_t* op = static_cast<uint16_t*>(p.out) + qrow * D + 4 * half;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint2 w;
        w.x = pack2_cvt(Tag{}, acc[db][4 * q + 0] * inv, acc[db][4 * q + 1] * inv);
        w.y = pack2_cvt(Tag{}, acc[db][4 * q + 2] * inv, acc[db][4 * q + 3] * inv);
        *reinterpret_cast<uint2*>(op + 32 * db + 8 * q) = w;
      }
  }
  }
}

// Joins the pieces of the row tiles that the balanced launch cut, weighted by their
// log-sum-exps: a workgroup of 256 threads per 16 rows of a (sequence, kv head, row
// tile), D / 4 threads per row.  Bound by its reads (512 B per piece and row at D =
// 128); four pieces' rows are in flight per thread.
constexpr int kPfMergeRows = 16;
template <class Tag, int D>
__global__ __launch_bounds__(256) void paged_prefill_merge(PrefillParams p) {
  constexpr int TPR = D / 4;             // threads per row
  constexpr int RPP = 256 / TPR;         // rows per pass
  constexpr int PARTS = kPfRows / kPfMergeRows;
  const SeqPieces seqs = seq_pieces<true, D>(p);
  if (seqs.whole) return;
  const int part = blockIdx.x % PARTS;
  const int x = blockIdx.x / PARTS;
  const int b = x / (p.num_kv_heads * p.tiles_per_unit);
  const int kh = x / p.tiles_per_unit % p.num_kv_heads;
  const int tile = x % p.tiles_per_unit;
  const int tiles = __builtin_amdgcn_readlane(seqs.tiles, b);
  const int n = __builtin_amdgcn_readlane(seqs.n, b);
  if (tile >= tiles || n == 1) return;
  const int first = __builtin_amdgcn_readlane(seqs.first, b) + kh * n * tiles + tile;
  const int Lq = __builtin_amdgcn_readlane(seqs.q, b);
  const int64_t q0 = p.cu_seqlens_q[b];
  const int G = p.group;
  const int c = threadIdx.x % TPR;
  const int r1 = (part + 1) * kPfMergeRows;
  for (int r = part * kPfMergeRows + threadIdx.x / TPR; r < r1; r += RPP) {
    const int tq = tile * p.tokens_per_wg + r / G;
    if (r >= p.tokens_per_wg * G || tq >= Lq) break;
    auto row = [&](int y) { return static_cast<int64_t>(first + min(y, n - 1) * tiles) * kPfRows + r; };
    float m = -INFINITY, l = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int y = 0; y < n; y += 4) {
      float e[4];
      float4 v[4];
#pragma unroll
      for (int z = 0; z < 4; ++z) e[z] = y + z < n ? p.part_lse[row(y + z)] : -INFINITY;
#pragma unroll
      for (int z = 0; z < 4; ++z) v[z] = *reinterpret_cast<const float4*>(p.part_o + row(y + z) * D + 4 * c);
      const float mn = fmaxf(fmaxf(m, fmaxf(e[0], e[1])), fmaxf(e[2], e[3]));
      // fmaxf passes NaN over: only pieces without keys may be left out.
      if (mn == -INFINITY && e[0] == mn && e[1] == mn && e[2] == mn && e[3] == mn) continue;
#pragma unroll
      for (int z = 1; z < 4; ++z)  // past the last piece: its row again, maybe infinite
        if (y + z >= n) v[z] = make_float4(0.f, 0.f, 0.f, 0.f);
      const float a = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= a;
      o.x *= a;
      o.y *= a;
      o.z *= a;
      o.w *= a;
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        const float f = __builtin_amdgcn_exp2f(e[z] - mn);
        l += f;
        o.x += f * v[z].x;
        o.y += f * v[z].y;
        o.z += f * v[z].z;
        o.w += f * v[z].w;
      }
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    uint2 out;
    out.x = pack2_cvt(Tag{}, o.x * inv, o.y * inv);
    out.y = pack2_cvt(Tag{}, o.z * inv, o.w * inv);
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.out) + ((q0 + tq) * p.num_heads + kh * G + r % G) * D + 4 * c) =
        out;
  }
}

int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The balanced launch's most pieces, 0 = the plain grid, and whether the kernel has to ask
// the real lengths if cutting pays.
// Long cached contexts only (causal rows of a whole prompt carry unequal keys).  Taken
// where cutting pays with every sequence as long as the longest: two chunks of 342-512
// tokens behind 16k-24k keys 390 -> 310 us, 512 behind 8k 147 -> 85, 64 behind 32k 513 ->
// 62, 16 x 16 behind 4k-8k 149 -> 93, 4 x 256 behind 8k at D = 64 104 -> 91; left alone:
// 1024 behind 2k (64 vs 67 split), 2048 behind 8k (297 vs 316).  Other batches may still
// gain by being ragged, which only the kernel sees (15 of 20-118 behind 1k-8k 186 -> 150
// us, 4 x 256 behind 1k-4k 71 -> 62, 7 of 30-252 behind 1k-8k at D = 64 148 -> 83); where
// it then cuts no tile, looking costs 3-6 us (20 x 128 behind 6k-8k 330 -> 336, 14 x 128
// behind 4k 120 -> 125, 4 x 256 behind 4k 74 -> 78.5), so that it is done from 200 us on
// with more tiles than slots, 100 with more than CUs and 60 with fewer.
struct BalancedPlan {
  int pieces = 0;
  bool ask = false;
};
BalancedPlan balanced_plan(int64_t batch, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t max_seqlen_q,
                    int64_t max_seqlen_k, int64_t window_left) {
  if (batch <= 0 || batch > kPfSplitBatch || max_seqlen_q <= 0 || num_kv_heads <= 0 || num_heads < num_kv_heads ||
      num_heads / num_kv_heads > kPfRows || max_seqlen_k < 2 * max_seqlen_q || max_seqlen_k > INT32_MAX / 2)
    return {};
  const int64_t cus = oxide::device_cu_count();
  const int64_t slots = 2 * cus;
  const int64_t tpw = kPfRows / (num_heads / num_kv_heads);
  const int64_t tiles = batch * num_kv_heads * ceil_div64(max_seqlen_q, tpw);
  if (tiles > 2 * slots) return {};
  const int64_t w = window_left < 0 || window_left >= max_seqlen_k ? -1 : window_left;
  const int64_t steps = steps_per_tile(static_cast<int>(max_seqlen_k), static_cast<int>(w), static_cast<int>(tpw));
  const int64_t pieces = std::min(2 * slots, tiles * ceil_div64(steps, kPfMinPiece));
  if (pieces <= tiles || tiles * steps > INT32_MAX / 2) return {};  // the kernel sums steps in 32 bits
  // With equal lengths: the piece length the kernel would choose.
  const int t = static_cast<int>(tiles), n = static_cast<int>(steps), d = static_cast<int>(head_dim);
  auto equal = [&](int64_t most) {
    return std::max<int64_t>(kPfMinPiece, ceil_div64(n, std::max<int64_t>(most / tiles, 1)));
  };
  int64_t len = equal(pieces);
  if (pieces > slots && tiles <= slots && 8 * equal(slots) <= 18 * len) len = equal(slots);
  const int cut = static_cast<int>(tiles * ceil_div64(n, len)), w0 = static_cast<int>(tiles * steps);
  const float plain = plain_us(t, w0, n, static_cast<int>(slots), d);
  const bool pays = cut > t && split_us(cut, t, w0, static_cast<int>(len), static_cast<int>(slots), d) < plain;
  // Ragged: a sixth less work than equal lengths have.
  const bool may = batch > 1 && plain >= (tiles <= cus ? 60.f : tiles <= slots ? 100.f : 200.f) &&
                   (tiles > slots || 1.9 * 1.15 * 0.85 * tiles * steps / slots + 768.0 / d <
                                         steps * (tiles > cus ? 1.9 : 1.03));
  if (!pays && !may) return {};
  return {static_cast<int>(pieces), !pays};
}
size_t balanced_rows_bytes(int pieces, int64_t head_dim) {
  return static_cast<size_t>(pieces) * kPfRows * static_cast<size_t>(head_dim) * sizeof(float);
}
// Partial rows, their log-sum-exps, the piece length.
size_t balanced_bytes(int pieces, int64_t head_dim) {
  return balanced_rows_bytes(pieces, head_dim) + (static_cast<size_t>(pieces) * kPfRows + 1) * sizeof(float);
}

template <class Tag, int D>
void launch_mode(const PrefillParams& p, dim3 grid, hipStream_t s) {
  if (p.pair) {
    if (p.block_table == nullptr)
      hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kContiguous, false, true>), grid, dim3(kPfThreads), 0, s, p);
    else if (p.block_size % kPfKeys == 0)
      hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedTiles, false, true>), grid, dim3(kPfThreads), 0, s, p);
    else
      hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedRows, false, true>), grid, dim3(kPfThreads), 0, s, p);
    return;
  }
  if (p.block_table == nullptr)
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kContiguous, false>), grid, dim3(kPfThreads), 0, s, p);
  else if (p.block_size % kPfKeys == 0)
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedTiles, false>), grid, dim3(kPfThreads), 0, s, p);
  else
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedRows, false>), grid, dim3(kPfThreads), 0, s, p);
}

template <class Tag, int D>
void launch_balanced(const PrefillParams& p, unsigned plain, hipStream_t s) {
  // Workgroups for the most pieces and, where no tile is cut, for the plain grid.
  const dim3 grid(std::max(plain, static_cast<unsigned>(ceil_div64(p.max_pieces, kPfXcds) * kPfXcds)));
  if (p.block_table == nullptr)
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kContiguous, false, false, true>), grid, dim3(kPfThreads), 0, s, p);
  else if (p.block_size % kPfKeys == 0)
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedTiles, false, false, true>), grid, dim3(kPfThreads), 0, s, p);
  else
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedRows, false, false, true>), grid, dim3(kPfThreads), 0, s, p);
  oxide::check_launch();
  hipLaunchKernelGGL((paged_prefill_merge<Tag, D>), dim3(static_cast<unsigned>(
                     kPfRows / kPfMergeRows * p.units * p.tiles_per_unit)), dim3(256), 0, s, p);
}

template <class Tag, int D>
void launch_prefix_mode(const PrefillParams& p, dim3 grid, hipStream_t s) {
  if (p.block_size % kPfKeys == 0)
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedTiles, true>), grid, dim3(kPfThreads), 0, s, p);
  else
    hipLaunchKernelGGL((paged_prefill_attn<Tag, D, kPagedRows, true>), grid, dim3(kPfThreads), 0, s, p);
}

template <class Tag>
bool launch_prefill(const PrefillParams& p, int head_dim, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(ceil_div64(int64_t{p.units} * p.spread, kPfXcds) * kPfXcds * p.share_tiles));
  if (p.max_pieces > 0) {
    head_dim == 128 ? launch_balanced<Tag, 128>(p, grid.x, s) : launch_balanced<Tag, 64>(p, grid.x, s);
    return true;
  }
  if (head_dim == 128) {
    launch_mode<Tag, 128>(p, grid, s);
    return true;
  }
  if (head_dim == 64) {
    launch_mode<Tag, 64>(p, grid, s);
    return true;
  }
  return false;
}

void prefill_impl(void* out, const void* q, const void* k, const void* v, const uint32_t* cu_seqlens_q,
                  const uint32_t* cu_seqlens_k, const int32_t* block_table, int64_t max_blocks_per_seq,
                  int64_t num_blocks, int64_t num_rows, int64_t batch, int64_t num_heads,
                  int64_t num_kv_heads, int64_t head_dim, int64_t page_block_size,
                  int64_t max_seqlen_q, int64_t max_seqlen_k, int32_t window_left,
                  float softmax_scale, void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  if (dtype != OXIDE_DTYPE_BF16 && dtype != OXIDE_DTYPE_F16) {
    oxide::set_error(OXIDE_ERR_UNSUPPORTED_DTYPE);
    return;
  }
  if (batch < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 ||
      max_seqlen_q < 0 || max_seqlen_k < 0 || batch > 65535 || num_heads > 65535 ||
      max_seqlen_q > INT32_MAX / 2 || max_seqlen_k > INT32_MAX / 2) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  if (batch == 0 || max_seqlen_q == 0) return;
  if (!out || !q || !cu_seqlens_q || !cu_seqlens_k || !oxide::aligned16(out) || !oxide::aligned16(q)) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  if (max_seqlen_k > 0) {
    if (!k || !v || !oxide::aligned16(k) || !oxide::aligned16(v)) {
      oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
      return;
    }
    if (block_table != nullptr) {
      if (page_block_size <= 0 || num_blocks <= 0 || num_blocks > INT32_MAX || max_blocks_per_seq < 0 ||
          page_block_size > INT32_MAX || max_blocks_per_seq * page_block_size < max_seqlen_k) {
        oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
        return;
      }
    } else if (num_rows <= 0) {
      oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
      return;
    }
  }
  const int64_t group = num_heads / num_kv_heads;
  if ((head_dim != 64 && head_dim != 128) || group > kPfRows) {
    oxide::set_error(OXIDE_ERR_UNSUPPORTED_SHAPE);
    return;
  }
  PrefillParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.cu_seqlens_q = cu_seqlens_q;
  p.cu_seqlens_k = cu_seqlens_k;
  p.block_table = block_table;
  p.max_blocks = max_blocks_per_seq;
  p.num_rows = block_table ? num_blocks * page_block_size : num_rows;
  p.num_blocks = static_cast<int>(block_table ? num_blocks : 0);
  p.max_seqlen_q = static_cast<int>(max_seqlen_q);
  p.max_seqlen_k = static_cast<int>(max_seqlen_k);
  p.num_heads = static_cast<int>(num_heads);
  p.num_kv_heads = static_cast<int>(num_kv_heads);
  p.group = static_cast<int>(group);
  p.tokens_per_wg = static_cast<int>(kPfRows / group);
  const int64_t tiles = ceil_div64(max_seqlen_q, p.tokens_per_wg);
  const int64_t units = batch * num_kv_heads;
  if (units > INT32_MAX / 2 || ceil_div64(units, kPfXcds) * kPfXcds * tiles > INT32_MAX) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  p.tiles_per_unit = static_cast<int>(tiles);
  p.units = static_cast<int>(units);
  // Where whole units would load the 8 XCDs more than a fifth unevenly, a unit's tiles go
  // to the fewest XCDs that make the shares a multiple of 8; otherwise its K/V stays in
  // one L2.  One prompt of 4096 tokens on 28 heads / 4 kv heads 249 -> 131 us, on 8 heads
  // / 1 kv head 204 -> 70, 3 of 2000 (12 units) 133 -> 115; 7 units of 3000 lose by it
  // (148 -> 153).
  p.spread = 1;
  if (p.units < 1024 && 5 * ceil_div64(p.units, kPfXcds) * kPfXcds > 6 * int64_t{p.units})
    while (p.units * p.spread % kPfXcds != 0) p.spread *= 2;
  p.share_tiles = static_cast<int>(ceil_div64(tiles, p.spread));
  // Prompts with no cached prefix, of at most 2048 tokens and about one length (the
  // kernel looks), with work for four rounds of the chip's slots: a workgroup takes a
  // unit's row tiles n - 1 - i and then i (a separate kernel instance), the same keys per
  // workgroup and half the workgroup starts.  Single -> paired: 32 x 512 (G = 2) 69.0 ->
  // 62.7 us, 16 x 1024 188 -> 184, 8 x 2048 303 -> 296; smaller or ragged batches lose
  // (1 x 300 11.6 -> 17.0, 128 x 128 51 -> 62, 8 of 200-1000 81 -> 89), and so do 4 x
  // 4096 and prompts behind a cached prefix, whose tiles already carry equal keys.
  p.pair = (tiles >= 8 && p.spread == 1 && max_seqlen_k <= max_seqlen_q && max_seqlen_q <= 2048 &&
            tiles * units >= 8 * static_cast<int64_t>(oxide::device_cu_count()))
               ? 1
               : 0;
  p.block_size = static_cast<int>(block_table ? page_block_size : 1);
  p.window_left = window_left < 0 ? -1 : window_left;
  p.scale_log2 = softmax_scale * 1.4426950408889634f;
  p.batch = static_cast<int>(batch);
  if (workspace != nullptr && oxide::aligned16(workspace)) {
    const auto [pieces, ask] =
        balanced_plan(batch, num_heads, num_kv_heads, head_dim, max_seqlen_q, max_seqlen_k, window_left);
    if (pieces > 0 && workspace_bytes >= balanced_bytes(pieces, head_dim)) {
      p.max_pieces = pieces;
      p.may_be_whole = ask;
      p.slots = 2 * oxide::device_cu_count();
      p.part_o = static_cast<float*>(workspace);
      p.part_lse = reinterpret_cast<float*>(static_cast<char*>(workspace) + balanced_rows_bytes(pieces, head_dim));
      p.piece_len = reinterpret_cast<int*>(p.part_lse + static_cast<int64_t>(pieces) * kPfRows);
    }
  }
  hipStream_t s = oxide::as_stream(stream);
  const bool ok = dtype == OXIDE_DTYPE_BF16 ? launch_prefill<Bf16Tag>(p, static_cast<int>(head_dim), s)
                                            : launch_prefill<F16Tag>(p, static_cast<int>(head_dim), s);
  if (!ok) {
    oxide::set_error(OXIDE_ERR_UNSUPPORTED_SHAPE);
    return;
  }
  oxide::check_launch();
}

}  // namespace

extern "C" void paged_prefill_attention(void* out, const void* q, const void* k_cache,
                                        const void* v_cache, const uint32_t* cu_seqlens_q,
                                        const uint32_t* cu_seqlens_k, const int32_t* block_table,
                                        int64_t max_blocks_per_seq, int64_t num_blocks, int64_t batch,
                                        int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                        int64_t page_block_size, int64_t max_seqlen_q,
                                        int64_t max_seqlen_k, int32_t window_left,
                                        float softmax_scale, int dtype, void* stream) {
  if (block_table == nullptr && max_seqlen_k > 0) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  prefill_impl(out, q, k_cache, v_cache, cu_seqlens_q, cu_seqlens_k, block_table, max_blocks_per_seq,
               num_blocks, 0, batch, num_heads, num_kv_heads, head_dim, page_block_size, max_seqlen_q,
               max_seqlen_k, window_left, softmax_scale, nullptr, 0, dtype, stream);
}

extern "C" size_t prefill_attention_workspace_size(int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                                         int64_t head_dim, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                                         int32_t window_left) {
  if (head_dim != 64 && head_dim != 128) return 0;
  const int pieces =
      balanced_plan(batch, num_heads, num_kv_heads, head_dim, max_seqlen_q, max_seqlen_k, window_left).pieces;
  return pieces > 0 ? balanced_bytes(pieces, head_dim) : 0;
}

extern "C" void paged_prefill_attention_workspace(
    void* out, const void* q, const void* k_cache, const void* v_cache, const uint32_t* cu_seqlens_q,
    const uint32_t* cu_seqlens_k, const int32_t* block_table, int64_t max_blocks_per_seq, int64_t num_blocks,
    int64_t batch, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim, int64_t page_block_size,
    int64_t max_seqlen_q, int64_t max_seqlen_k, int32_t window_left, float softmax_scale, void* workspace,
    size_t workspace_bytes, int dtype, void* stream) {
  if (block_table == nullptr && max_seqlen_k > 0) {
    oxide::set_error(OXIDE_ERR_INVALID_ARGUMENT);
    return;
  }
  prefill_impl(out, q, k_cache, v_cache, cu_seqlens_q, cu_seqlens_k, block_table, max_blocks_per_seq,
               num_blocks, 0, batch, num_heads, num_kv_heads, head_dim, page_block_size, max_seqlen_q,
               max_seqlen_k, window_left, softmax_scale, workspace, workspace_bytes, dtype, stream);
}

extern "C" void varlen_prefill_attention(void* out, const void* q, const void* k, const void* v,
                                         const uint32_t* cu_seqlens_q, const uint32_t* cu_seqlens_k,
                                         int64_t total_k, int64_t batch, int64_t num_heads,
                                         int64_t num_kv_heads, int64_t head_dim, int64_t max_seqlen_q,
                                         int64_t max_seqlen_k, int32_t window_left, float softmax_scale,
                                         int dtype, void* stream) {
  prefill_impl(out, q, k, v, cu_seqlens_q, cu_seqlens_k, nullptr, 0, 0, total_k, batch, num_heads,
               num_kv_heads, head_dim, 1, max_seqlen_q, max_seqlen_k, window_left, softmax_scale,
               nullptr, 0, dtype, stream);
}

extern "C" void varlen_prefill_attention_workspace(
    void* out, const void* q, const void* k, const void* v, const uint32_t* cu_seqlens_q,
    const uint32_t* cu_seqlens_k, int64_t total_k, int64_t batch, int64_t num_heads, int64_t num_kv_heads,
    int64_t head_dim, int64_t max_seqlen_q, int64_t max_seqlen_k, int32_t window_left, float softmax_scale,
    void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  prefill_impl(out, q, k, v, cu_seqlens_q, cu_seqlens_k, nullptr, 0, 0, total_k, batch, num_heads,
               num_kv_heads, head_dim, 1, max_seqlen_q, max_seqlen_k, window_left, softmax_scale,
               workspace, workspace_bytes, dtype, stream);
}

namespace oxide {

// Shared-prefix pass of a cascaded decode call (declared in decode_common.hpp).
bool launch_decode_prefix(const DecodePrefixArgs& a, hipStream_t s) {
  PrefillParams p{};
  p.q = a.q;
  p.k = a.k;
  p.v = a.v;
  p.cu_seqlens_k = a.cu_seqlens_k;
  p.block_table = a.block_table;
  p.max_blocks = a.max_blocks;
  p.num_blocks = a.num_blocks;
  p.num_rows = static_cast<int64_t>(a.num_blocks) * a.block_size;
  p.max_seqlen_k = a.max_seqlen_k;
  p.num_heads = a.num_heads;
  p.num_kv_heads = a.num_kv_heads;
  p.group = a.num_heads / a.num_kv_heads;
  p.tokens_per_wg = kPfRows / p.group;
  p.tiles_per_unit = static_cast<int>(ceil_div64(a.batch, p.tokens_per_wg));
  p.units = a.num_kv_heads * a.pre_splits;
  p.spread = 1;
  p.share_tiles = p.tiles_per_unit;
  p.block_size = a.block_size;
  p.window_left = a.window_left < 0 ? -1 : a.window_left;
  p.scale_log2 = a.scale_log2;
  p.part_o = a.part_o;
  p.part_lse = a.part_lse;
  p.pre_row0 = a.pre_row0;
  p.pre_splits = a.pre_splits;
  p.split_keys = a.split_keys;
  p.shared_hint = a.shared_hint;
  p.dec_batch = a.batch;
  p.shared_out = a.shared_out;
  const dim3 grid(static_cast<unsigned>(ceil_div64(p.units, kPfXcds) * kPfXcds * p.tiles_per_unit));
  if (a.head_dim == 128) {
    a.bf16 ? launch_prefix_mode<Bf16Tag, 128>(p, grid, s) : launch_prefix_mode<F16Tag, 128>(p, grid, s);
    return true;
  }
  if (a.head_dim == 64) {
    a.bf16 ? launch_prefix_mode<Bf16Tag, 64>(p, grid, s) : launch_prefix_mode<F16Tag, 64>(p, grid, s);
    return true;
  }
  return false;
}

}  // namespace oxide
