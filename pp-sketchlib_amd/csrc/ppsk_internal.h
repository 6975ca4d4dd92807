// Internal declarations shared by the HIP kernels and the C-ABI layer.
//
// Device layout of a sketch set ("stripes"), for one k-mer length index kk:
//   S[kk][nb][w][hl][BLK]  (uint32)
//     nb : block of BLK = 128 samples (sample n -> nb = n / 128, lane n % 128)
//     w  : 64-bin word, 0 .. s64-1
//     hl : 32-bit plane, hl = h * BBITS + l, h = 0 low / 1 high dword of the
//          uint64 layer word, l = bit layer 0 .. BBITS-1
// so every (kk, nb, w) is one contiguous 28 x 128 dword slab (14 KiB) and a
// run of consecutive samples for one plane is contiguous.  Padding samples
// (n >= n_samples inside the last block) are zero and are masked on output.
#pragma once

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

namespace ppsk {

constexpr int BLK = 128;       // samples per stripe block
constexpr int BBITS = 14;      // bit layers per bin value (reference def_bbits)
constexpr int HL = 2 * BBITS;  // 32-bit planes per 64-bin word
constexpr int WAVES = 8;       // waves per workgroup
constexpr int MAXK = 32;       // most k-mer lengths per query
// zero words appended to every stripe buffer: the tile kernel stages whole
// groups of up to 8 words and may read one group past the last word
constexpr int STRIPE_PAD_WORDS = 8;

enum OutKind : int32_t { OUT_CORE_ACC = 0, OUT_JACCARD = 1, OUT_COUNTS = 2, OUT_ONE_MINUS_J = 3 };
enum RandomMode : int32_t { RANDOM_NONE = 0, RANDOM_EQUAL_BASE = 1, RANDOM_MC = 2 };

// Progress and cancellation of a call.  cancel: host-mapped flag written by
// ppsk_cancel, read by the kernels between work items with system-scope
// loads; progress: device counter of finished work items, mirrored (by every
// update, in split passes by one in 64) with a plain system-scope store into the
// host-mapped word progress_host (stores of different workgroups may land out of
// order: the host keeps the largest value it has read).
struct Control {
  const uint32_t* cancel;
  unsigned long long* progress;
  unsigned long long* progress_host;
  uint32_t* stop;  // device word: 1 once an item of the call has seen `cancel` set
};

// Tile: rows [bi * rows, +rows) x cols [ct * cols, +cols) of the variant's
// tile shape (variant_tile_rows / variant_tile_cols).
struct Tile {
  int32_t bi;
  int32_t ct;
};

struct DistParams {
  const uint32_t* row_stripes;  // set giving the tile rows (r1 of the Jaccard)
  const uint32_t* col_stripes;  // set giving the tile columns
  int64_t n_rows, n_cols;       // real sample counts
  int32_t nb_rows, nb_cols;     // stripe blocks in each set
  int32_t n_k, s64;
  int32_t self_mode;            // rows and cols are the same set, upper triangle
  int32_t full_square;          // self set, every i != j (kNN); i == j -> +inf
  const Tile* tiles;
  int64_t n_tiles;
  int64_t item_base;            // first (tile * n_k + kk) item of this launch
  uint16_t* counts;             // scratch [n_tiles][n_k][tile rows][tile cols]
  uint32_t* tile_done;          // [n_tiles] completion counters, left at zero
  // epilogue
  int32_t out_kind;
  void* out;                    // dense output (see OutKind)
  int64_t out_row_offset;       // subtracted from the dense row index
  int64_t out_stride_rows;      // for full_square: row stride of the [rows][n] block
  int64_t square_row0;          // for full_square: first global row in out
  float kvals[MAXK];            // k as float (reference kmer2mat)
  double tolerance;             // regression validity threshold
  int32_t random_mode;
  int32_t n_clusters;
  int32_t mc_ref_is_col;        // MC table index order: [col][row] instead of [row][col]
  const double* jv_rows;        // [n_rows][n_k] equal-base j(len) per sample
  const double* jv_cols;
  const float* mc_table;        // [n_k][C][C]
  const uint16_t* cl_rows;      // [n_rows] cluster ids
  const uint16_t* cl_cols;
  unsigned long long* fail_count;
  unsigned long long* fail_first;  // smallest failing dense row
  uint32_t* fail_rows;             // optional [n_rows] failures per tile row sample
  int32_t row_prefetch;            // pull each stage's row panel into L2 a stage ahead
  Control ctl;                     // progress and cancellation (all null: neither)
};

// Persistent batch kernel (dist_batch): work queues and items.
constexpr int BATCH_QUEUES = 8;  // one per XCD of the MI355X

struct BatchItem {  // one tile of one job: every k-mer length, then the epilogue
  int32_t job;
  int32_t bi;
  int32_t ct;
  int32_t pad;  // tile shape (variant) of the item for the mixed-shape kernel
};

struct BatchArgs {
  const DistParams* jobs;   // [n_jobs] per-job parameters (device memory)
  const BatchItem* items;   // queue q holds items [queue_begin[q], queue_begin[q + 1])
  int64_t queue_begin[BATCH_QUEUES + 1];
  uint32_t* queue_next;     // [BATCH_QUEUES] next item of each queue (zeroed before launch)
  uint16_t* scratch;        // [grid][max_k][tile rows][tile cols] per-workgroup counts
  int32_t max_k;
  Control ctl;              // progress and cancellation of the launch (null: neither)
};

// Split passes (dist_items): an item is one tile, one k-mer length and one run
// of words; tiles are 64, 32 or 16 rows x 256 columns.
struct ItemTile {
  int32_t row0;  // first row, a multiple of `rows`
  int32_t ct;    // columns [ct * 256, +256)
  int32_t rows;  // 64, 32 or 16
  int32_t group;  // row group of a coded pass
};
constexpr int ITEM_SLOTS = 512;        // workgroups resident at once: 2 per CU
constexpr int ITEM_COUNTS = 64 * 256;  // counts of one item (u16), whatever its height

// The (tile, k-mer length) pairs of a launch, k-mer length first, those of the
// 64-row tiles before those of the shorter ones: the first `whole` are one
// item each, every other is cut into `runs` items.  An item's counts go to
// block L (whole) or whole + (L - whole) * runs + run, L its pair's number.
struct ItemArgs {
  const ItemTile* tiles;  // [n_tiles], 64-row tiles first
  int32_t n_tiles;
  int32_t n_tall;  // 64-row tiles
  int32_t whole;
  int32_t runs;
  int32_t run_units;  // words (coded pass: halves) per run; the last may hold fewer
  int32_t n_items;    // whole + (n_tiles * n_k - whole) * runs
  int32_t unwatched;  // workgroups that do not look for a cancellation: the first ones
  int32_t out_rows;   // tile rows per output workgroup (divides 16)
};

// Coded passes (code_kernel, dist_coded): the rows of a group and the columns
// they meet, as ranks among the values the group's rows hold at each bin.
constexpr int CODE_ROWS = 768;    // most rows of a group: ranks 0 .. 768
constexpr int CODE_PLANES = 10;   // planes of the largest rank
constexpr int CODE_STAGE = 36;    // planes of one LDS stage (1 KiB each)
constexpr int CODE_BLOCK = 256;   // samples per block of coded planes

struct CodeGroup {
  uint32_t* cols;    // [n_k][ncb][2 s64][CODE_PLANES][256]; block 0 holds sample 256 cb0
  uint32_t* rows;    // the same with nrb, rb0; == cols when the rows are among the columns
  uint32_t* widths;  // [n_k][2 s64] planes used, and 16 more entries that may be read
  int32_t row0, n_rows;
  int32_t cb0, ncb;
  int32_t rb0, nrb;
};

// Rows past a pass's last multiple of 64 that take a 64-row tile instead of one of
// 32 and / or one of 16: more than 48, and from 64 (64-row tile, k-mer length)
// pairs on more than 32.  Every tile streams its columns, so 32 + 16 rows take
// longer than 64 once the pass fills the CUs: 97 queries x 6,000 references 1,073
// and 859 us, x 200,000 29.0 and 24.6 ms (coded), 40 x 20,000 1,579 and 1,377
// us; below that the shorter tiles' items end earlier: 33 x 1,000 143 and 149 us,
// 100 samples 107 and 124.
__host__ __device__ inline int64_t tall_from(int64_t pairs) { return pairs >= 64 ? 33 : 49; }

// Rows of a band in tiles, pairs as above: as many 64-row ones as fit (one more
// for tall_from rows left), the rest in one of 32 and / or one of 16.
struct BandTiles {
  int64_t tall;
  int shorts, first;  // shorter tiles (0 .. 2) and the height of the first
};
__host__ __device__ inline BandTiles band_tiles(int64_t rows, int64_t pairs) {
  const int64_t tall = (rows + 64 - tall_from(pairs)) / 64, left = rows - tall * 64;
  if (left <= 0) return {tall, 0, 0};
  return {tall, left > 32 ? 2 : 1, left > 16 ? 32 : 16};
}

// Split batches (dist_batch_items): the same items over the tiles of many jobs.
struct BatchTile {
  int32_t job, row0, ct, rows;
  int32_t block0, runs;  // counts of k-mer length k, run y: block0 + k * runs + y
};

struct BatchRun {  // one item; tile < 0: none
  int32_t tile, kk;
  int32_t word0, words;
  int32_t block;
};

struct BatchItemArgs {
  const DistParams* jobs;
  const BatchTile* tiles;  // [n_tiles]
  const BatchRun* items;   // [n_items], workgroup b takes item b
  uint16_t* counts;        // blocks of ITEM_COUNTS
  int32_t n_tiles, n_items;
  int32_t out_rows;  // tile rows per output workgroup (divides 16)
  Control ctl;
};

// Launchers (dist_kernels.hip).  All work goes on `stream`.
hipError_t launch_batch_items(const BatchItemArgs& a, hipStream_t stream);
// Coding of groups [first_group, + n_groups) of the device table `groups`,
// matching and output of their tiles (tile.group indexes the whole table);
// p.counts as for launch_items, a.run_units in halves.
hipError_t launch_coded(const DistParams& p, const ItemArgs& a, const CodeGroup* groups,
                        int first_group, int n_groups, hipStream_t stream);
// Matching and output of a split pass; p.counts holds n_items blocks of
// ITEM_COUNTS counts.
hipError_t launch_items(const DistParams& p, const ItemArgs& a, hipStream_t stream);
hipError_t launch_stripe(const uint64_t* raw, int64_t count, int64_t first,
                         int32_t n_k, int32_t s64, int32_t nb, uint32_t* stripes,
                         hipStream_t stream);

// Tile kernel configurations ("variants"): rows per wave RQ (row operands in
// SGPRs), columns per lane RR, row-operand pipeline PB (0 = left to the
// compiler, 2 = explicit double-buffered scalar loads of 2 planes); the 8
// waves of a workgroup form a grid of row groups x column groups.
//   1: RQ16 RR1 PB0, waves 8 x 1 (128 x 64)   3: RQ16 RR2 PB0, 8 x 1 (128 x 128)
//   2: RQ8  RR4 PB2, waves 8 x 1 (64 x 256)   4: RQ8  RR2 PB2, 4 x 2 (32 x 256)
//   5: RQ8  RR1 PB2, waves 2 x 4 (16 x 256)
// A pipelined (PB = 2) configuration is only correct if the compiler keeps
// the in-flight SGPR tuples in place; the build rejects any that spill.
constexpr int DEFAULT_VARIANT = 2;
constexpr int N_VARIANTS = 5;
bool variant_valid(int variant);
int variant_tile_rows(int variant);
int variant_tile_cols(int variant);
hipError_t launch_dists(const DistParams& p, int variant, int64_t n_items,
                        hipStream_t stream);

// Persistent launch with a tile shape per item (BatchItem.pad = 2, 4 or 5):
// the `variant` of batch_grid / launch_batch that selects it.  Its scratch
// holds [grid][max_k][64][256] counts whatever the shapes.
constexpr int BATCH_MIXED = 6;

// Persistent batch launch: `grid` workgroups (batch_grid: every workgroup
// resident at once).  batch_reset zeroes the queue counters and sets the
// per-job fail counters ([n_jobs][2]: count, first row) to (0, max) with a
// kernel, so that both launches can be captured in a graph.
hipError_t batch_grid(int variant, int* grid);
hipError_t launch_batch(const BatchArgs& a, int variant, int grid, hipStream_t stream);
// Split pass of a query band (dist_items over rows x every column): tiles of
// column blocks [0, n_ct), `step` of them per launch, a launch's 64-row tiles
// before its shorter ones; clears the band's fit failures.  No tiles written
// when step is 0.
hipError_t launch_band_setup(ItemTile* tiles, int64_t rows, const BandTiles& b, int64_t n_ct, int64_t step,
                             unsigned long long* fail, uint32_t* fail_rows, hipStream_t stream);
// Start of a call: fit failures {0, none}, a progress count of 0 and no stop.
hipError_t launch_call_reset(unsigned long long* fail, const Control& ctl, hipStream_t stream);
hipError_t launch_batch_reset(uint32_t* queue_next, unsigned long long* fail, int n_jobs,
                              hipStream_t stream, unsigned long long* progress = nullptr);
// Zeroes n tile completion counters and sets fail ([2]: count, first row; may
// be null) to (0, max), with a kernel.
// launch_dists for 64 x 256 tiles (variant 2) of a self pass (upper
// triangle): diagonal tiles skip the column blocks that hold no output pair.
hipError_t launch_dists_diagonal(const DistParams& p, int64_t n_items, hipStream_t stream);
// Writes the table of the distance epilogue's logarithm into the current
// device's copy (once per device, before its first distance kernel).
hipError_t upload_log_table();
hipError_t launch_tile_reset(uint32_t* tile_done, int64_t n, unsigned long long* fail,
                             hipStream_t stream);

}  // namespace ppsk
