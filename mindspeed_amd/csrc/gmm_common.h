// Declarations shared by the grouped-matmul translation units.
#pragma once

#include "common.h"

namespace ms {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxGroups = 4096;

struct GroupEntry {
    int row_begin, row_end;  // output rows of the group
    int red_begin, red_end;  // reduction range of the group
    int tile_begin;          // tiles of the entries before this one (entry of an XCD's own list: its first slot there)
    int num_row_tiles;
    int tile_rows;           // rows per full tile
    int tail_rows;           // rows of the group's last row tile if it is a smaller one (64 / 128), else 0
    int num_tiles;           // num_row_tiles * column tiles
    int share;               // entry of an XCD's own list: tiles of it that every XCD handles (whole: all of them)
    int split;               // 0, or 1 + the part number of a small tail tile whose reduction is split: such a
                             // tile writes fp32 partial sums to the split workspace (c_off then points there);
                             // kEvened: the last two row tiles share their rows (even_out)
    int whole;               // entry of an XCD's own list: 1 = that XCD takes all tiles of the group, 0 = its eighth
    int64_t b_off;           // element offset of the group's weight block
    int64_t c_off;           // element offset of the group's output block
};

// One small tail tile row whose reduction was split into `parts` ranges: the partial sums of part s and local row r
// are row (pair0 + s) * kSplitRows + r of the split workspace ([.., cols] fp32).
struct SplitTail {
    int row_begin, rows;
    int pair0, parts;
};
constexpr int kSplitRows = 128;          // rows reserved per (tail, part) pair: the largest small tile
constexpr int kMaxSplit = 4;             // most parts a reduction is split into
constexpr int kSplitCus = 256;           // a launch's split parts never number more than this (one round of MI355X's CUs)
constexpr int kSplitMinRed = 2048;       // shortest reduction range worth a part of its own
constexpr int kMaxListGroups = 256;      // most groups that may be dealt out whole to single XCDs (ranked by counting,
                                         // dealt out by one thread)

struct TileTable {
    int slots_per_xcd;       // an eighth of all tiles, rounded up; shares by cost and per-XCD lists: slots of the longest one
    int num_entries;
    int num_split_tails;     // tail tile rows whose reduction was split (entries of the SplitTail array in use)
    int lists_off;           // 0, or the byte offset from the table to eight lists of entries, one per XCD (whole groups
                             // dealt out to single XCDs); `entries` is then unused
    int list_stride;         // entries reserved per list
    int part_from, part_count, part_shift;   // tiles of the last round that run in parts (LastRound)
    int in_order;            // split on rows: of the first so many tile numbers every XCD takes consecutive ones (take_together) ..
    int by_cost;             // 0: an eighth each (consecutive_tile); 1: by share_begin
    int share_begin[9];      // first tile number of every XCD's share
    int begins[16];          // tile_begin of the first 16 entries (INT_MAX past the last): one load finds the entry
    int list_count[8];       // entries in use in every XCD's list
    GroupEntry entries[1];
};

struct GmmArgs {
    const void *a;
    const void *b;
    void *c;
    const TileTable *table;
    int64_t a_stride_row, a_stride_red;
    int64_t b_stride_red, b_stride_col;
    int64_t c_stride_row;
    int cols;          // n (fused SwiGLU form: the number of activation columns, ffn = n / 2)
    int num_col_tiles;
    int a_vec_ok, b_vec_ok, c_vec_ok;
    // fused SwiGLU form only (OUT_SWIGLU): second output and the per-row factor
    void *act;                 // [rows, cols] activation output, same dtype
    int64_t act_stride_row;
    const void *probs;         // optional per-row probability
    int probs_dtype;
    // fused SwiGLU backward form only (OUT_SWIGLU_GRAD): c is d_fc1 [rows, 2*cols]
    const void *fc1;           // [rows, 2*cols] saved output of the first matmul (gate | up)
    int64_t fc1_stride_row;
    float *partials;           // [rows, partials_per_row] row sums of dact * silu(gate) * up per 64 columns, or NULL
    int partials_per_row;
    // split tail tiles only (OUT_SAME): fp32 partial sums, rows of `cols` floats
    float *split_ws;
    // tiles found from the group list itself (tile_from_list), without a table; NULL: from the table
    const int64_t *group_list;
    const int64_t *b_offsets;   // element offsets of separately allocated weights, or NULL
    int64_t b_stride_group, c_stride_group;
    int group_list_type, group_type, num_groups;
    int m, k;
    int tile_rows;              // rows per full tile, a power of two: 256 for 16-bit operands; 32, 64 or 128 in fp32
    int small_tails;            // a group's last row tile may be a smaller one
    int even_tails;             // ... or the last two share their rows (EVEN_..)
    int tails_last_below;       // launches of fewer tiles take their small tiles last
    int part_cus;               // compute units if the last round may be divided (LastRound), else 0
};

struct TileCoord {
    GroupEntry e;
    int row_tile, col_tile;
    int tile_rows;           // rows of this tile (the entry's tile_rows, or its tail_rows for the last row tile)
    bool valid;
};

// Tile order inside a group of R row tiles x C column panels: the r-th tile the kernels take.  Column panels in sets of
// 8, row tiles in sets of 4, row-tile-fastest inside such a 4 x 8 block.  The 32 compute units of an XCD then work on
// one block at a time and fetch 4 + 8 operand panels for 32 tiles; with many row tiles (the weight gradient: hidden /
// 256 of them) plain row-tile-fastest order would have them on 16 x 2 tiles and fetch 18.  Up to 4 row tiles per group
// the two orders are the same.  A single row tile left over after the blocks of 4 (a group of 5 or 9 row tiles:
// typically the small tail tile of a ragged group) joins the last block instead of forming one of its own, so it runs
// beside the tiles whose column panels it shares (measured: 0.2 to 0.4 % per layer step).
__host__ __device__ __forceinline__ void tile_order(int r, int R, int C, int &row_tile, int &col_tile) {
    constexpr int BR = 4, BC = 8;      // measured against 8 x 4, 8 x 8, 2 x 16 and 4 x 16: the fastest for all three products
    const int cg = r / (BC * R);
    const int rem = r - cg * BC * R;
    const int wc = C - BC * cg < BC ? C - BC * cg : BC;    // column panels in this set
    int nb = (R + BR - 1) / BR;
    if (R > BR && R % BR == 1) nb -= 1;                     // a single left-over row tile joins the block before it
    int rb = rem / (BR * wc);
    rb = rb > nb - 1 ? nb - 1 : rb;
    const int rem2 = rem - rb * BR * wc;
    const int hr = rb == nb - 1 ? R - BR * rb : BR;        // row tiles in this block
    const int lc = rem2 / hr;
    col_tile = BC * cg + lc;
    row_tile = BR * rb + (rem2 - lc * hr);
}

// Last of n >= 1 entries whose tile_begin is at most `at` (the first entry's always is): bisected down to 64 candidates,
// which one load of the wavefront then compares at once (a bisection to the end is six dependent loads for 64 groups).
__device__ __forceinline__ int find_entry(const GroupEntry *entries, int n, int at) {
    int lo = 0, hi = n;
    while (hi - lo > 64) {
        const int mid = (lo + hi) >> 1;
        if (entries[mid].tile_begin <= at) lo = mid; else hi = mid;
    }
    const int i = lo + static_cast<int>(threadIdx.x & 63);
    const int begin = entries[i < hi ? i : hi - 1].tile_begin;
    return lo + __popcll(__ballot(i < hi && begin <= at)) - 1;
}

// The full tiles that a launch of few rounds leaves for its last, partly filled round (tiles from .. from + count - 1) run as
// two or four tiles of fewer rows each (1 << shift), as long as these and the launch's small tiles fit one round: such a
// launch's time goes by its rounds, and a round lasts as long as its longest tile.  16 groups of 768 rows, bf16, us per launch
// with whole tiles, halves only and halves or quarters (the present rule): K 1536, 1.12 rounds of tiles 80 / 70 / 66, 1.5
// rounds 81 / 76 / 76, 2.06 rounds 117 / 105 / 101, 0.38 rounds 37 / 31 / 31; K 3072, 1.12 rounds 144 / 124 / 115, 1.5 rounds
// 148 / 142 / 142, 2.25 rounds 218 / 208 / 206.  From six rounds on (kTailsLastRounds) it is not done: at the board's power
// limit the compute units that sit out leave the others a higher clock.
struct LastRound {
    int from, count, shift;
};
__device__ __forceinline__ LastRound divide_last_round(int full, int small, int cus) {
    const int left = full % cus;
    const int shift = left == 0 ? 0 : (4 * left + small <= cus ? 2 : (2 * left + small <= cus ? 1 : 0));
    return LastRound{full - left, shift != 0 ? left : 0, shift};
}
// Tile number of workgroup b, and which part of that tile it takes.  The parts of a tile follow each other on one XCD
// (their weight panel is fetched once), but for the last, incomplete eight tiles.
__device__ __forceinline__ int tile_of_workgroup(int b, const LastRound &lr, int &part) {
    const int s = b - lr.from;
    part = 0;
    if (s < 0) return b;
    const int extra = (lr.count << lr.shift) - lr.count;
    if (s >= lr.count + extra) return b - extra;
    const int whole = lr.count & ~7, in_whole = whole << lr.shift;
    if (s < in_whole) {
        part = (s >> 3) & ((1 << lr.shift) - 1);
        return lr.from + ((s >> (3 + lr.shift)) << 3) + (s & 7);
    }
    const int rest = lr.count & 7;
    part = (s - in_whole) / rest;
    return lr.from + whole + (s - in_whole) - part * rest;
}
// Turns a full tile into its part; a part without rows is no tile.
__device__ __forceinline__ void take_part(TileCoord &tc, int part, int shift) {
    tc.tile_rows >>= shift;
    tc.e.row_begin += part * tc.tile_rows;
    tc.valid = tc.e.row_begin + tc.row_tile * tc.e.tile_rows < tc.e.row_end;
}

// Tile number b, and the same with every XCD's of the n numbers (b = x, x + 8, ... of XCD x) consecutive.
__device__ __forceinline__ int share_of_eight(int b, int n) {
    const int x = b & 7, odd = n & 7;
    return x * (n >> 3) + (x < odd ? x : odd) + (b >> 3);
}

// Split on rows: whether every XCD takes consecutive tiles of the whole launch, entries laid end to end, or an eighth of every
// entry's.  Consecutive ones are blocks of 4 x 8 tiles out of one or two groups, 12 operand panels for the 32 compute units;
// eighths of small groups are pieces of many (three row tiles by 12 columns: five panels for four and a half tiles).  16 groups
// of 710 to 790 rows, bf16, us per launch with eighths and with consecutive tiles: K 2048, 3072 columns 147 / 143 (weights along
// K 141 / 136); K 1536, 2048 columns 84 / 75 (81 / 72).  8 groups of 2048 rows, K 2048, 28 column tiles 379 / 361; 64 groups of
// 0 to 6600 rows, K 1408 to 2816 360 to 655 / 352 to 640.
// Not where an eighth of a group is about a block by itself: the XCDs then share the group's panels, while eight XCDs in as many
// groups come back to panels that the last-level cache (256 MB) may no longer hold (8 x 12 of them, 512 K bytes each, are under
// way).  So from 6 row tiles on there is a limit on the reduction, and on the largest of few groups (row tiles times K) or the tiles
// in the average one of many.  Rows per group, eighths / consecutive, us per launch:
//   8 groups of 1600 (7 row tiles): K 3072, 2048 columns 148 / 140; 4096 columns: K 2560 232 / 225, 2816 254 / 250, 3072 278 / 282,
//   3584 318 / 319; 8 of 2100 (9): K 2048 240 / 234.5, 2816 319 / 324, 7168 (2048 rows) 1440 / 1483
//   16 groups of 2000 (8 or 9): 2048 columns: K 1536 190 / 183, 3072 346 / 344; 4096 columns: K 1536 365 / 357, 2048 467 / 465, 2560
//   564 / 575, 3072 660 / 666; of 2816 (11 or 12): 2048 columns: K 1536 257 / 248, 3072 461 / 455; 4096 columns: K 1536 483 / 488, 2048
//   616 / 624, 2560 750 / 764; of 4000 (16): 2048 columns: K 1536 347 / 365, 3072 650 / 667; 4096 columns: K 1024 497 / 505, 1536 670 /
//   696, 2560 1025 / 1055; of 100 to 2900 (6): K 1536, 2048 columns 127 / 122
//   64 and 128 groups of 65536 rows together: K 1408 to 3072, 2048 and 2816 columns 2 to 5 % less time, K 4096 level
// Up to 5 row tiles (one block) there is none: 16 of 750, K 5120, 2048 columns 251 / 237; 8 of 1200, K 4096 to 14336 275 to 917 / 267 to
// 900; 8 of 1024, K 28672 1416 / 1397 (small tiles that come last read their panels again in either order, and two XCDs read the
// panels at the border of their shares).
constexpr int kOneBlockRowTiles = 5, kTwoBlockRowTiles = 9, kTogetherRed = 3072, kTogetherGroups = 16;
constexpr int kLargestRowTilesRed = 7 * kTogetherRed, kAverageTiles = 112;
__host__ __device__ __forceinline__ int together_row_tiles(int k) {       // .. of the largest group
    if (k > kTogetherRed) return kOneBlockRowTiles;
    return kTwoBlockRowTiles * k <= kLargestRowTilesRed ? kTwoBlockRowTiles : (8 * k <= kLargestRowTilesRed ? 8 : 7);
}
// none_larger: no group has more than together_row_tiles; tiles: of all groups
__host__ __device__ __forceinline__ bool take_together(bool none_larger, int tiles, int k, int num_groups) {
    return none_larger || (k <= kTogetherRed && num_groups >= kTogetherGroups && tiles <= kAverageTiles * num_groups);
}

// ... and not where an XCD would have the tiles of a large group and another those of many small ones: full tiles are bound by the
// matrix cores, small ones by the weights that every one of them streams, and eighths put both on every XCD.  60 groups of 1 to
// 3100 rows (half of the row tiles small), K 792 / 1584, 18 column tiles: 168 / 174 and 312 / 334 us.  So small tiles are at
// most a quarter, or no group has twice the average (128 rows each: 298 / 282, 250 each: 399 / 342 and 210 / 185).
__host__ __device__ __forceinline__ bool few_small_tiles(int small, int row_tiles) { return 4 * small <= row_tiles; }
__host__ __device__ __forceinline__ bool much_above_average(int group_row_tiles, int row_tiles, int num_groups) {
    return static_cast<int64_t>(group_row_tiles) * num_groups > 2 * static_cast<int64_t>(row_tiles);
}

// In which launches the two ways to find a tile ask that at all.  From the group list shares are equal in number: with small
// tiles between the full ones (half of their cost) only up to a tenth of them are close enough to equal shares; with the small
// ones last any number, but there must be a full tile to place.  From a table they are equal in cost, or with the small tiles
// last in number, which takes a round of full tiles (the launches with a table that have fewer are decoding ones).
__host__ __device__ __forceinline__ bool list_places(bool tails_last, int full_tiles, int small, int row_tiles) {
    return tails_last ? full_tiles != 0 : row_tiles != 0 && 10 * small <= row_tiles;
}
__host__ __device__ __forceinline__ bool table_places(bool tails_last, int full_tiles, int cus) { return !tails_last || full_tiles >= cus; }

// Tile number t of the first n, dealt over the XCDs one by one, as one of consecutive ones of its XCD: those in front of the last
// round's parts, and the tiles that run in parts.
__device__ __forceinline__ int consecutive_tile(int t, int n, const LastRound &lr) {
    const int whole = lr.count != 0 ? lr.from : n;
    return t < whole ? share_of_eight(t, whole) : whole + share_of_eight(t - whole, n - whole);
}

// Rows of the small tile that a remainder of `rem` rows of a group goes to, 0 for a full one.
__host__ __device__ __forceinline__ int small_tile_rows(int rem) { return rem <= 64 ? 64 : (rem <= 128 ? 128 : 0); }

// A group of more than one row tile whose last one would be a small one may instead share the rows of its last two between
// them (`even`: EVEN_TWO only in groups of two, EVEN_ALL), 160 and up to 160 or 192 and up to 192: two tiles of five or six of the eight row blocks (gmm16_tile).
// What bounds a small tile is its own pass over the weight panel: it takes 0.45 to 0.65 of a full tile's time for a quarter
// or half of its products, and leaves the step of the tiles beside it.
constexpr int kEvened = -1;
enum { EVEN_NONE = 0, EVEN_TWO = 1, EVEN_ALL = 2 };
__host__ __device__ __forceinline__ bool shares_last_two(int rem, int row_tiles, int even) {
    return small_tile_rows(rem) != 0 && (even == EVEN_ALL ? row_tiles > 1 : even == EVEN_TWO && row_tiles == 2);
}
__host__ __device__ __forceinline__ int small_tail_of(int rem, int row_tiles, int even) {
    return shares_last_two(rem, row_tiles, even) ? 0 : small_tile_rows(rem);
}
// The rows of such a tile, as those of an entry in which it begins where its number says.
__device__ __forceinline__ void even_out(TileCoord &tc) {
    const int T = tc.e.tile_rows, n = tc.e.num_row_tiles;
    tc.e.split = 0;
    if (tc.row_tile < n - 2) return;
    const int rem = tc.e.row_end - tc.e.row_begin - (n - 1) * T;
    const int rows = rem <= 64 ? 160 : 192;
    const int from = tc.e.row_begin + (n - 2) * T + (tc.row_tile == n - 1 ? rows : 0);
    tc.e.row_end = from + rows < tc.e.row_end ? from + rows : tc.e.row_end;
    tc.e.row_begin = from - tc.row_tile * T;
}

// Tile number j of an entry: of the entry's tiles every XCD (workgroup number modulo 8) takes consecutive ones of the
// blocked order, the odd ones dealt in turn; in_order: the j-th one.
__device__ __forceinline__ void deal_tile(TileCoord &tc, int j, int num_col_tiles, bool in_order = false) {
    tile_order(in_order ? j : share_of_eight(j, tc.e.num_tiles), tc.e.num_row_tiles, num_col_tiles, tc.row_tile, tc.col_tile);
    tc.tile_rows = (tc.e.tail_rows != 0 && tc.row_tile == tc.e.num_row_tiles - 1) ? tc.e.tail_rows : tc.e.tile_rows;
    if (tc.e.split == kEvened) even_out(tc);
    tc.valid = true;
}

// Map this workgroup to its tile.  Workgroup b runs on XCD b % 8 (round-robin dispatch).  Normally it takes a tile of
// the entry that holds tile number b, entries laid end to end: of the entry's tiles every XCD then gets an eighth, the
// odd ones going to the XCDs in turn from entry to entry, so the XCDs' totals differ by one tile whatever the
// groups' sizes are (an eighth rounded up for every group left XCDs without work: a group of 12 tiles occupied six of
// them).  Inside the entry an XCD's tiles are consecutive in the blocked order above, so concurrently running
// workgroups of an XCD share operand panels in that XCD's L2.  With many groups the schedule may instead deal whole
// groups out to single XCDs (every XCD then has a list of its own): a group's operands are fetched into one L2 instead
// of eight.  Split on rows (ROWS), an XCD's tiles may instead be consecutive ones of the whole launch (take_together).
// LISTS: the kernel may meet per-XCD lists (the fast kernels of the split on rows); the others are compiled without that
// path, which costs the weight-gradient kernel 0.3 us per tile at its start when it is merely present.
template <bool LISTS, bool ROWS>
__device__ __forceinline__ TileCoord locate_tile(const TileTable *table, int b) {
    TileCoord tc;
    tc.valid = false;
    if ((b >> 3) >= table->slots_per_xcd) return tc;
    if (LISTS && table->num_entries == 0) {     // per-XCD lists (the common table is empty then); no further header
                                                // field is read on the way to the common case
        const int xcd = b & 7;
        const int slot = b >> 3;
        const GroupEntry *list = reinterpret_cast<const GroupEntry *>(reinterpret_cast<const char *>(table) + table->lists_off) +
                                 static_cast<int64_t>(xcd) * table->list_stride;
        const int count = table->list_count[xcd];
        if (count == 0) return tc;
        tc.e = list[find_entry(list, count, slot)];
        const int r = slot - tc.e.tile_begin + (tc.e.whole != 0 ? 0 : xcd * tc.e.share);
        if (r >= tc.e.num_tiles || (tc.e.whole == 0 && slot - tc.e.tile_begin >= tc.e.share)) return tc;
        tile_order(r, tc.e.num_row_tiles, tc.e.num_tiles / tc.e.num_row_tiles, tc.row_tile, tc.col_tile);
        tc.tile_rows = (tc.e.tail_rows != 0 && tc.row_tile == tc.e.num_row_tiles - 1) ? tc.e.tail_rows : tc.e.tile_rows;
        if (tc.e.split == kEvened) even_out(tc);
        tc.valid = true;
        return tc;
    }
    const LastRound lr{table->part_from, table->part_count, table->part_shift};
    int part;
    int t = tile_of_workgroup(b, lr, part);
    bool in_order = false;
    if constexpr (ROWS) {
        const int n = table->in_order;
        if (table->by_cost != 0) {
            const int x = b & 7, slot = b >> 3;
            const int from = table->share_begin[x], own = table->share_begin[x + 1] - from;
            in_order = slot < own;
            t = in_order ? from + slot : n + ((slot - own) << 3) + x;
        } else {
            in_order = t < n;
            if (in_order) t = consecutive_tile(t, n, lr);
        }
    }
    // Up to 16 entries (8 experts with their tail tiles) their begins lie in the table's header and are fetched at once.
    int lo = 0;
    if (table->num_entries <= 16) {
#pragma unroll
        for (int i = 1; i < 16; ++i) lo += table->begins[i] <= t ? 1 : 0;
    } else {
        lo = find_entry(table->entries, table->num_entries, t);
    }
    tc.e = table->entries[lo];
    const int j = t - tc.e.tile_begin;
    if (j >= tc.e.num_tiles) return tc;
    deal_tile(tc, j, tc.e.num_tiles / tc.e.num_row_tiles, in_order);
    if (t >= lr.from && t < lr.from + lr.count) take_part(tc, part, lr.shift);
    return tc;
}

// A tile of the launch, found by every wavefront for itself out of a group list of at most 64 groups: the entries and tile numbers
// of a table without per-XCD lists and split tails (gmm_schedule_kernel).  Lane g holds group g, the running quantities are
// prefix sums over the lanes, and the entry that holds this workgroup's tile comes out of one ballot.  One load instead of the
// table's two dependent ones, and no launch in front of the matmul.  Which tile number a workgroup takes may differ from a
// table's: consecutive tiles are shared out by number here, by cost there, and asked for in other launches (list_places,
// table_places).
constexpr int kMaxDirectGroups = 64;
template <bool SPLIT_RED>
__device__ __forceinline__ TileCoord tile_from_list(const GmmArgs &p, int b) {
    TileCoord tc;
    tc.valid = false;
    const int lane = threadIdx.x & 63;
    const int C = p.num_col_tiles;
    const unsigned m = static_cast<unsigned>(p.m);
    const bool mine = lane < p.num_groups;
    const int64_t v = p.group_list[mine ? lane : p.num_groups - 1];
    // Group ends as the schedule kernel derives them: never before the previous end, never past m.
    const unsigned c = !mine || v < 0 ? 0u : (v > p.m ? m : static_cast<unsigned>(v));
    const bool counts = p.group_list_type != 0;
    const unsigned end = wave_scan(c, [&](unsigned x, unsigned y) {
        const unsigned sum = x + y < m ? x + y : m;           // (both at most m < 2^31)
        return counts ? sum : (x > y ? x : y);
    });
    const unsigned prev = lane_below(end);
    const int len = mine ? static_cast<int>(end - prev) : 0;
    const int T = p.tile_rows, shift = 31 - __builtin_clz(T);
    LastRound lr{0, 0, 0};
    int t = b, part = 0;                           // tile number, and the part of it
    bool in_order = false;
    GroupEntry &e = tc.e;
    e = GroupEntry{};
    e.tile_rows = T;
    if constexpr (SPLIT_RED) {
        // every group has the tiles of one output block; groups of above-average length come first
        const int row_tiles = (p.k + T - 1) >> shift;
        e.num_tiles = row_tiles * C;
        const int q = b / e.num_tiles;
        if (q >= p.num_groups) return tc;
        const unsigned long long all = __ballot(mine);
        const unsigned long long first = __ballot(mine && len >= p.m / p.num_groups);
        const int nfirst = __popcll(first);
        const unsigned long long set = q < nfirst ? first : all & ~first;
        const int nth = q < nfirst ? q : q - nfirst;
        const bool in_set = (set >> lane) & 1;
        const unsigned long long hit = __ballot(in_set && __popcll(set & ((1ull << lane) - 1ull)) == nth);
        const int g = __builtin_ctzll(hit);
        e.row_end = p.k;
        e.red_begin = __builtin_amdgcn_readlane(static_cast<int>(prev), g);
        e.red_end = __builtin_amdgcn_readlane(static_cast<int>(end), g);
        e.c_off = g * p.c_stride_group;
        e.num_row_tiles = row_tiles;
        e.tail_rows = p.small_tails ? small_tile_rows(p.k - (row_tiles - 1) * T) : 0;
        e.tile_begin = q * e.num_tiles;
    } else {
        const int row_tiles = (len + T - 1) >> shift;
        const int rem = len - (row_tiles - 1) * T;
        const int tail = p.small_tails && len > 0 ? small_tail_of(rem, row_tiles, p.even_tails) : 0;
        const unsigned packed = static_cast<unsigned>(row_tiles) | (tail != 0 ? 1u << 25 : 0u);   // (fewer than 2^25 row tiles, at most 64 tails)
        const unsigned incl = wave_scan(packed, [](unsigned x, unsigned y) { return x + y; });
        const unsigned sums = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
        const unsigned before = incl - packed;
        const int all_rt = sums & ((1u << 25) - 1), all_tails = sums >> 25;
        const int rt_before = before & ((1u << 25) - 1), tails_before = before >> 25;
        const int total = all_rt * C;
        const bool tails_last = total < p.tails_last_below;
        const int total_first = tails_last ? (all_rt - all_tails) * C : total;
        if (tails_last && p.part_cus != 0) lr = divide_last_round(total_first, total - total_first, p.part_cus);
        t = tile_of_workgroup(b, lr, part);
        if (p.small_tails && list_places(tails_last, total_first, all_tails, all_rt) &&
            take_together(__ballot(row_tiles > together_row_tiles(p.k)) == 0, total, p.k, p.num_groups) &&
            (few_small_tiles(all_tails, all_rt) || __ballot(much_above_average(row_tiles, all_rt, p.num_groups)) == 0)) {
            in_order = t < total_first;
            if (in_order) t = consecutive_tile(t, total_first, lr);
        }
        e.red_end = p.k;
        if (t >= total) {                          // rows past the last offset: zero-fill (empty reduction range)
            const int last_end = __builtin_amdgcn_readlane(static_cast<int>(end), 63);
            const int rows = p.m - last_end;
            e.num_row_tiles = (rows + T - 1) >> shift;
            e.num_tiles = e.num_row_tiles * C;
            if (t - total >= e.num_tiles) return tc;
            e.row_begin = last_end;
            e.row_end = p.m;
            e.red_end = 0;
            e.tail_rows = p.small_tails ? small_tile_rows(rows - (e.num_row_tiles - 1) * T) : 0;
            e.tile_begin = total;
        } else {
            const bool apart = tails_last && tail != 0;              // this lane's small tile is an entry of its own
            const int full_tiles = row_tiles - (apart ? 1 : 0);
            const bool first = t < total_first;
            const int begin = first ? (tails_last ? rt_before - tails_before : rt_before) * C : total_first + tails_before * C;
            const int count = first ? full_tiles * C : (apart ? C : 0);
            const int g = __builtin_ctzll(__ballot(t >= begin && t < begin + count));
            const int g_prev = __builtin_amdgcn_readlane(static_cast<int>(prev), g);
            const int g_end = __builtin_amdgcn_readlane(static_cast<int>(end), g);
            const int g_tail = __builtin_amdgcn_readlane(tail, g);
            const int g_full = __builtin_amdgcn_readlane(full_tiles, g);
            const bool full_only = first && tails_last && g_tail != 0;
            e.row_begin = first ? g_prev : g_prev + g_full * T;
            e.row_end = full_only ? g_prev + g_full * T : g_end;
            e.num_row_tiles = first ? g_full : 1;
            e.tail_rows = full_only ? 0 : g_tail;
            if (__builtin_amdgcn_readlane(p.small_tails && shares_last_two(rem, row_tiles, p.even_tails) ? 1 : 0, g)) e.split = kEvened;
            e.num_tiles = e.num_row_tiles * C;
            e.tile_begin = __builtin_amdgcn_readlane(begin, g);
            e.b_off = p.b_offsets != nullptr ? p.b_offsets[g] : g * p.b_stride_group;
        }
    }
    deal_tile(tc, t - e.tile_begin, C, in_order);
    if (t >= lr.from && t < lr.from + lr.count) take_part(tc, part, lr.shift);
    return tc;
}

// This workgroup's tile, from the group list or from the table (which then has no per-XCD lists): the kernels that are not
// compiled for one of the two.
template <bool SPLIT_RED>
__device__ __forceinline__ TileCoord locate(const GmmArgs &p) {
    if (p.group_list != nullptr) return tile_from_list<SPLIT_RED>(p, blockIdx.x);
    return locate_tile<false, !SPLIT_RED>(p.table, blockIdx.x);
}
// ... nor for one kind of split
__device__ __forceinline__ TileCoord locate_any(const GmmArgs &p) { return p.group_type == 2 ? locate<true>(p) : locate<false>(p); }

constexpr int BM = 256, BN = 256, BK = 64;
constexpr int kTileBytes = BM * BK * 2;                 // 32 KB per operand per stage
constexpr int kLdsBytes16 = 4 * kTileBytes;             // A,B x 2 stages = 128 KB

enum OutMode { OUT_SAME = 0, OUT_F32 = 1, ACC_F32 = 2, OUT_SWIGLU = 3, OUT_SWIGLU_GRAD = 4 };

template <int DT>
__device__ __forceinline__ f32x16 mfma16(v16 a, v16 b, f32x16 c) {
    if constexpr (DT == MS_BF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
}

// acc += a^T-style 16 x 16 x 32 product, accumulating in place in the accumulation registers.  Inline assembly because of
// that pin: through the builtin the register allocator moves four-register accumulators between the two register files
// inside the K loop (up to 500 copies per step of 128 products, and spills).  The compiler therefore does not know that
// this is a matrix instruction: a caller must leave two instructions between an ordinary vector write of an operand and
// this (operands that come from LDS reads are covered by the wait the compiler inserts), and wait out the last results
// with s_nop before ordinary instructions read them (ready and settle of the K loops).
template <int DT>
__device__ __forceinline__ void mfma16x16(v16 a, v16 b, f32x4 &acc) {
    if constexpr (DT == MS_BF16) asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    else asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// The same pointer in scalar registers, whatever the compiler knows about its uniformity.
__device__ __forceinline__ const char *uniform(const char *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
    const uint64_t hi = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32)));
    return reinterpret_cast<const char *>(lo | hi << 32);
}

// LDS swizzle: 16-byte chunk position of (row, chunk) inside the row's 128 bytes.
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }


// Fast 16-bit kernels (gmm_fast.hip, gmm_pair.hip).  Returns MS_OK after launching, or -1 if
// this problem does not meet the fast kernels' alignment conditions.
// lists: the table may come as per-XCD lists (only asked of the weight-gradient product, whose common kernel is compiled
// without that lookup; the kernels of the split on rows always have it).
int launch_gmm16_fast(hipStream_t stream, const GmmArgs &args, int dtype, int out_mode, bool a_red, bool b_red,
                      unsigned grid, bool lists = false);
int launch_gmm16_fast_fp16(hipStream_t stream, const GmmArgs &args, int out_mode, bool a_red, bool b_red, unsigned grid, bool lists);
// dX (both operands contiguous along the reduction dim) and dW (neither) of one matmul in one launch (gmm_pair.hip); out_mode:
// dW's.  dw_first: its workgroups come first.  direct: tiles from the group list, else from the two tables.
int launch_gmm16_pair(hipStream_t stream, const GmmArgs &dx, unsigned dx_grid, const GmmArgs &dw, unsigned dw_grid, int dtype,
                      int out_mode, bool dw_first, bool direct);

}  // namespace ms
