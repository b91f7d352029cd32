// Internal launch interface of the paged-attention kernels (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mvllm {

// Largest number of physical pages one decode split may span and still have its page
// ids staged in LDS (4 KiB). The planner keeps splits at or below 1024 tokens, which is
// at most 1025 pages even at a page size of 1; a caller that understates
// max_context_len gets longer splits, which then read the table from global memory.
constexpr int kMaxSplitPages = 1040;
constexpr int kMaxSplitTokens = 1024;

// The stream schedule scans the context lengths of up to this many sequences in LDS.
constexpr int kMaxStreamSeqs = 4096;

// Query positions per prefill work item (4 waves x 32 MFMA columns) and keys per tile.
constexpr int kPrefillQueryTile = 128;
// Most stream-prefill workgroups (the merge lists an item's pieces in LDS).
constexpr int kMaxPrefillWgs = 2048;
// Stream prefill: the shares used of `wgs` workgroups, each of at least `min_tiles`
// 64-key tiles while that leaves a quarter of the workgroups busy. A share also pays
// for loading its items' queries and for writing and merging (m, l, O) pieces of 128
// query rows: a 512-token chunk behind a 1-2K prefix spread over every CU is cut into
// shares of two or three tiles, most of their time then going to that overhead
// (measured, 31 decode rows + one chunk, whole call: shares of >= 4 tiles 70-80 us
// against 76-81 us with one tile; 4K-16K prefixes 2-7% faster).
constexpr int kPrefillShareTiles = 4;
__host__ __device__ inline int64_t prefill_stream_shares(int64_t total_units, int64_t wgs,
                                                         int min_tiles) {
  const int64_t per = min_tiles > 1 ? min_tiles : 1;
  int64_t shares = (total_units + per - 1) / per;
  const int64_t floor = total_units < wgs / 4 ? total_units : wgs / 4;
  if (shares < floor) shares = floor;
  return shares < 1 ? 1 : (shares < wgs ? shares : wgs);
}
// XCDs (each with its own L2) that workgroups are dispatched to round robin on MI355X.
constexpr int kXcds = 8;
constexpr int kPrefillKeyTile = 64;

// The pair prefill kernel's items (64 or 128 query positions of two heads of a GQA group) and
// its schedule: items in a list without the grid's holes, those longer than a piece length
// (a percentage of the mean key tiles per workgroup) cut, where the plan says so, into key ranges
// ("pieces") run by workgroups of their own, whose (m, l, O) partials a second kernel
// merges. The schedule is formed on the device from the sequences' sizes.
// Times in units of 10 ns: a key tile of the longest item when items run whole, of the mean per
// CU when they are cut, and what cutting costs beside, for the host's choice and, where the
// launch is ready for both, the device's.
struct PairCosts {
  int whole, cut, fixed, weigh;
};
__host__ __device__ constexpr PairCosts pair_costs(int tile, bool fp8) {
  return tile == 64 ? (fp8 ? PairCosts{155, 185, 1300, 900} : PairCosts{93, 125, 1300, 900})
                    : (fp8 ? PairCosts{190, 230, 1800, 1800} : PairCosts{95, 190, 1800, 1800});
}
// Floats of one piece's partial: two heads x qt rows x (128 of O + (m, l)).
__host__ __device__ constexpr int pair_slot_floats(int qt) { return 2 * qt * 130; }
// The grid plan cuts at most this many 128-query items over at most this many columns.
constexpr int kSplitMaxItems = 64;
constexpr int kSplitMaxCols = 64;
constexpr int kSplitMaxRanks = 4096;
constexpr int kSplitDefaultPieces = 8;
constexpr int kSplitDefaultPct = 150;
// Host bounds of the split over `cols` columns and `cus` workgroups with pieces of at least
// pct% of the mean work per workgroup: the extra pieces of one column number fewer than
// 100 cus / (pct cols); the partial slots of one column (every piece of a cut item
// holds one) at most twice that.
__host__ __device__ inline int split_extra_ranks(int cus, int cols, int pct) {
  return (100 * cus + pct * cols - 1) / (pct * cols);
}
__host__ __device__ inline int split_slots(int cus, int cols, int pct) {
  return 2 * split_extra_ranks(cus, cols, pct);
}

// Query heads per prefill work item: two heads of a GQA group share every K/V tile
// staged in LDS when the group size is even.
__host__ __device__ inline int prefill_item_heads(int group) { return group % 2 == 0 ? 2 : 1; }

// Key tiles the prefill workgroup of query tile q walks for a sequence of `context`
// keys and `len` query tokens: keys [0, context - len + min((q + 1) * 128, len)).
__host__ __device__ inline int prefill_item_tiles(int context, int len, int q) {
  const int last = (q + 1) * kPrefillQueryTile < len ? (q + 1) * kPrefillQueryTile : len;
  return (context - len + last + kPrefillKeyTile - 1) / kPrefillKeyTile;
}

// Stream decode: the fewest keys of a share while there are several, the tokens one step of
// a wave covers (4 per row group of D / (16 / element bytes) lanes): 16 for 16-bit pools
// at D = 128, 8 for fp32, 32 for fp8. With few keys the launch is a chain of memory round trips
// per step, and a share of several steps leaves CUs idle meanwhile. (Shares of 64 keys
// whatever the type before: four fp32 sequences of 37-1000 keys 22.0 us a call, 15.7 with 16;
// one bf16 sequence of 1500 keys 14.8 -> 11.7, of 200 13.1 -> 9.9, of 8192 17.4 -> 16.9;
// batches of more than 64 keys per CU do not change.)
__host__ __device__ inline int decode_min_share_keys(int elem_bytes, int head_dim) {
  const int keys = 256 * (16 / elem_bytes) / head_dim;
  return keys < 8 ? 8 : keys;
}
// MFMA prefill: log2 units a row's scores may pass its running max by before O is rescaled
// (exponentials stay <= 2^8).
constexpr float kRescaleSlack = 8.0f;
// Pair prefill: the tiles whose probabilities are taken against the tile's own maxima, so that
// each query's largest one is 1 and not rounded to 16 bits: all of an item (or piece) of at
// most kExactTiles, every kExactEvery'th of a longer one, half as often where the items fill the
// chip or are of 128 positions, none of a longer one of 128 over fp8. Each costs a rescale of O, 64 multiplies of a tile's ~400 vector cycles per wave:
// 7% of a chip-filling launch (8 x 512 tokens after up to 1536 keys 57.3 -> 61.7 us, 2048 after
// 14336 526 -> 563), hidden in a small one (100 tokens after 300 keys 13.3 -> 14.2, 512 after
// 4000 42.6 -> 44.5). Errors against 64 bits without, with all, and as chosen, float16: 100
// tokens after 300 keys 2.88e-4, 2.62e-4 and 2.62e-4; three of 300 after 700 2.91e-4,
// 2.61e-4 and 2.79e-4; 512 after 4000 2.90e-4, 2.60e-4 and 2.83e-4 (cut
// in one- to nine-tile pieces, as the launch before the pair kernel had them, 2.62e-4,
// 2.84e-4 and 2.88e-4).
constexpr int kExactTiles = 12;
constexpr int kExactEvery = 4;

constexpr int kMaxDecodeWaves = 8;        // of a stream decode workgroup
constexpr int kMaxDecodeShares = 65535;  // DecodeShares' 32-bit products

// The stream decode's shares: share w owns keys [begin(w), begin(w + 1)) of the `total` laid
// end to end, begin(w) = floor(w total / count). Never empty: count <= max(1, ceil(total /
// min_keys)) <= max(1, total). Formed as w floor(total / count) + floor(w (total mod count) /
// count), in 32 bits: a 64-bit division is ~150 dependent instructions, and each launch made
// three. (count <= kMaxDecodeShares.)
struct DecodeShares {
  uint32_t total, count_u, whole, rest;
  int count;
  __host__ __device__ DecodeShares(int total_keys, int wgs, int min_keys)
      : total(static_cast<uint32_t>(total_keys)) {
    const uint32_t cap = (total + static_cast<uint32_t>(min_keys) - 1) / static_cast<uint32_t>(min_keys);
    count_u = cap < 1 ? 1 : (cap < static_cast<uint32_t>(wgs) ? cap : static_cast<uint32_t>(wgs));
    count = static_cast<int>(count_u);
    whole = total / count_u;
    rest = total - whole * count_u;
  }
  __host__ __device__ int begin(int w) const {
    const uint32_t u = static_cast<uint32_t>(w);
    return static_cast<int>(u * whole + u * rest / count_u);
  }
  // The share holding key x (0 <= x < total): an estimate within one, corrected.
  __host__ __device__ int owner(int x) const {
    int w = static_cast<int>((static_cast<float>(x) + 0.5f) * static_cast<float>(count_u) /
                             static_cast<float>(total));
    w = w < 0 ? 0 : (w >= count ? count - 1 : w);
    while (w > 0 && begin(w) > x) --w;
    while (w + 1 < count && begin(w + 1) <= x) ++w;
    return w;
  }
};

// Equal shares of `total` work units over `wgs` workgroups: workgroup w owns
// [floor(w * total / wgs), floor((w + 1) * total / wgs)).
__host__ __device__ inline int64_t share_begin(int64_t w, int64_t total, int64_t wgs) {
  return w * total / wgs;
}
// The workgroup owning unit x: the largest w whose share starts at or before x.
__host__ __device__ inline int64_t share_owner(int64_t x, int64_t total, int64_t wgs) {
  return ((x + 1) * wgs - 1) / total;
}

// Query heads per decode wave for a GQA group of `group` heads.
__host__ __device__ inline int decode_group_chunk(int group) {
  return group % 4 == 0 ? 4 : (group % 2 == 0 ? 2 : 1);
}

struct PagedParams {
  const void* q;
  const void* k_pool;
  const void* v_pool;
  const float* k_scales;  // [num_blocks, H_k], fp8 pools only
  const float* v_scales;
  void* out;
  const int32_t* block_tables;
  const int32_t* cu_seqlens_q;
  const int32_t* context_lens;
  const int32_t* seq_lens;
  int num_seqs;
  int num_tokens;
  int hq;
  int hk;
  int max_blocks;
  int block_shift;
  int block_mask;
  int table_shift;        // slot of a table entry's first row = entry << table_shift (a
                          // paged pool: block_shift, entries are page ids; 0: entries
                          // are slot ids themselves)
  int64_t kv_row_bytes;   // pool bytes between consecutive slots (a paged pool: H_k D elements)
  int64_t kv_head_bytes;  // pool bytes between kv heads of one slot (a paged pool: D elements)
  int dense_keys;     // stream decode of a dense cache: keys of every sequence (0: paged);
  int dense_slots;    // position i of sequence s at slot s * dense_slots + i, row s of q
  int stream_wgs;     // decode: > 0 selects the stream schedule with this many workgroups
  int split_tokens;   // grid decode: nominal keys per split
  int max_splits;     // grid decode: grid extent along the split axis
  int by_row;         // grid decode: 1 = one unit per query row (serves prefill rows too)
  float scale;
  float* part_o;      // split partials, D fp32 each
  float* part_ml;     // split partials' (running max in log2 units, sum)
  int stream_min_keys;  // stream decode: fewest keys of a share while there are several
  int* seq_prefix;    // stream decode: [num_seqs + 1] decode keys before each sequence
  int pf_wgs;         // prefill: > 0 selects the stream schedule with this many workgroups
  int* pf_prefix;     // stream prefill: [num_seqs + 1] work units before each sequence
  float* pf_o;        // stream prefill partials: [2 * pf_wgs][heads][128][D] fp32, each
                      // piece normalised by its own sum
  float* pf_ml;       // their (max in log2 units, sum) per row: [2 * pf_wgs][heads][128][2]
  int pf_share_tiles;       // stream prefill: fewest key tiles per share; pair prefill:
                            // fewest key tiles per piece
  int pf_register_staging;  // 1: the register-staged prefill kernel even where the
                            // direct-to-LDS one serves (a plan option, for measurement)
  int pf_tile;        // pair prefill: query positions of an item, 64 or 128
  int pf_pieces;      // pair prefill: 0 the (column, sequence, query tile) grid; else a 1-D grid
                      // of pf_ranks x columns by the schedule, items in at most this
                      // many pieces
  int pf_by_seq;      // schedule of whole items: 1 a sequence's after another's
  int pf_ranks;       // schedule: grid extent in ranks (items + extra pieces bound)
  int pf_slots;       // cut: partial slots per column
  int pf_cus;         // cut: the workgroups the pieces are sized for
  int pf_piece_pct;   // cut: piece length, percent of the mean tiles per workgroup
  int pf_weigh;       // cut: 1 leaves all items whole where their sizes make that faster
  float* pf_part;     // cut: [pf_slots][columns] partials of pair_slot_floats
  int4* pf_rec;       // [pf_ranks][2], each position's piece: for the merge, and from the
                      // schedule kernel (more than 64 sequences)
};

// Splits of one row: as many as its visible context needs at `split_tokens` keys
// each, never more than the grid provides. Shared by the decode kernel, the merge
// kernel and the host planner so that all three agree.
__host__ __device__ inline int decode_num_splits(int visible, int split_tokens, int max_splits) {
  int n = (visible + split_tokens - 1) / split_tokens;
  n = n < max_splits ? n : max_splits;
  return n < 1 ? 1 : n;
}

// Balanced split length: visible / n rounded up to a multiple of 16 keys.
__host__ __device__ inline int decode_split_len(int visible, int nsplit) {
  const int per = (visible + nsplit - 1) / nsplit;
  return (per + 15) & ~15;
}

hipError_t launch_paged_decode(const PagedParams& p, int q_dtype, int kv_dtype, int head_dim,
                               hipStream_t stream);

// The decode step's new token, taken by the stream decode from the projection's output
// rather than from the pool: every sequence s of a decode-only batch has its token at
// position context_lens[s] - 1; its q head vectors are QK-normed and rotated in the
// launch (as the QK-norm + RoPE kernel does, the same bits), its k row likewise, and k
// and v go to the pool slot the block table maps that position to (a page id outside
// [0, num_blocks) writes nothing) and into the attention straight from registers.
struct FreshParams {
  const void* q;          // raw q of row i at q + i q_stride (H_q D contiguous elements)
  const void* k;          // raw k and v of row i at k / v + i kv_stride (H_k D elements)
  const void* v;
  int64_t q_stride;       // elements between consecutive rows
  int64_t kv_stride;
  const void* q_weight;   // QK-norm weights, [D]
  const void* k_weight;
  const float* cos_t;     // [max_positions][D]
  const float* sin_t;
  int64_t max_positions;  // a position at or past it gives NaN rows, as the unfused kernel
  int64_t num_blocks;
  float eps;
};

// Stream decode with the new token formed in the launch (16-bit q and pool, head dim
// 128, p.stream_wgs > 0), then the merge, as launch_paged_decode.
hipError_t launch_paged_decode_fresh(const PagedParams& p, const FreshParams& f, int dtype,
                                     int head_dim, hipStream_t stream);

hipError_t launch_paged_prefill(const PagedParams& p, int q_dtype, int kv_dtype, int head_dim,
                                int max_query_len, hipStream_t stream);

// Whether launch_paged_prefill has a kernel for this shape; if not, prefill rows are
// served by the decode kernel in by-row mode.
bool paged_prefill_supported(int q_dtype, int kv_dtype, int head_dim, int hq, int hk,
                             int block_size);

}  // namespace mvllm
