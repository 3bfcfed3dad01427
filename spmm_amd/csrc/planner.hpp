// planner.hpp -- host-side planning of one SpMM: the wavefront task list of
// the row kernel and the row windows routed to the MFMA tile kernel.
//
// Replaces reference workload_manager (src/our_spmm.cu:353-477), which packs
// warps of 32 lanes into 8-warp thread blocks by row length and gives a long
// row at most N/64 blocks.  Here every task is one 64-lane wavefront over one
// column chunk of C; chunks are mapped to XCDs so each XCD's L2 holds only
// its slice of B; tasks run longest first; long rows are shared by the four
// wavefronts of a workgroup (LDS sum) or, longer still, split across
// workgroups with an ordered two-kernel sum.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

#include "../../include/tca_spmm.h"

namespace tca {

constexpr int kXcds = 8;  // XCDs of the MI355X: the hardware deals workgroup b to XCD b % 8
constexpr int64_t kMallBytes = int64_t(256) << 20;  // MI355X Infinity Cache (MALL), shared by the XCDs

// Task kinds of the row kernel (int4 {x, y, z, w}).  Multi tasks hold at most
// multi_group_rows() rows, walked `slots` at a time, except zero tasks
// (z == 0), which hold up to kZeroRows empty rows whose C rows the wavefront
// only clears.
enum TaskKind : int32_t {
    kTaskRow = 0,    // x = row, y = nnz begin, z = nnz end: all slots split one row
    kTaskMulti = 1,  // x = offset into perm, y = rows in group, z = longest row; z == 0: empty rows
    kTaskSeg = 2,    // x = long-row id, y = nnz begin, z = nnz end, w = 2 | (segment slot << 2)
    kTaskWide = 3,   // x = row, y = nnz begin, z = nnz end of this quarter; all 4 waves of a workgroup
};

constexpr int32_t kZeroRows = 64;
// Short rows per multi task: passes of `slots` rows (one row per slot and
// pass), at most kMultiPasses of them and 64 rows.  A pass waits for three
// loads in a row or more, so several only pay where the tasks are enough for
// the chip all the same: at least kMultiTasks of them, or so many others
// (row, wide and segment tasks) beside few short rows that these end long
// before.  us per product at one / four passes on the MI355X: a 300 x 200
// layer of 2 %, fp32 N = 47 3.1 / 5.4, bf16 4.2 / 9.8; 12,000 x 1000 of 2 %,
// fp32 N = 17 6.8 / 10.4, fp16 N = 48 8.8 / 12.6; R-MAT of 10,000 nodes and
// 110,000 nonzeros, fp32 N = 18 8.2 / 11.0; of 200,000 and 3.4M, N = 20 48.4 /
// 52.1; 60,000 rows of 5, N = 32 8.6 / 9.3; of 1.5M and 17M, N = 20 346 / 339; of
// 2.4M and 64M, N = 47 2101 / 2084; 2^20 rows, 20M nonzeros in 15,000 of them,
// fp16 N = 64 (23,000 other tasks, 1600 of short rows) 171.0 / 169.2; 100,000
// rows of the kind, N = 48 (4200 and 270) 17.6 / 24.2.  With four slots and two a
// pass has less to do and enough is a quarter and a sixteenth: R-MAT of 63,000
// nodes and 490,000 nonzeros, bf16 N = 25 (two) 23.2 / 20.8; 12,000 x 300 of 2 %,
// fp32 N = 47 (four) 4.9 / 6.4.  Rows beside panels keep four: the sampled
// product's kernel of their tasks wants full batches of 64 nonzeros (131,000
// nodes, fp32 N = 128 18.5 / 15.0).
constexpr int32_t kMultiPasses = 4;
constexpr int64_t kMultiTasks = 16384;
inline int32_t multi_group_rows(int32_t slots, int64_t n_short, int64_t n_other, bool beside_panels) {
    const int64_t tasks = n_short / slots;  // of one pass
    const bool hidden = n_other >= kMultiTasks && n_other >= 8 * tasks;
    const int64_t enough = slots < 8 ? kMultiTasks * slots * slots / 64 : kMultiTasks;
    const int64_t passes = hidden || beside_panels ? kMultiPasses : std::clamp<int64_t>(tasks / enough, 1, kMultiPasses);
    return static_cast<int32_t>(std::min<int64_t>(64, slots * passes));
}

// Widths whose widest dividing vector is one or two elements take whole
// 16-byte vectors instead, the last one ending at the row's end
// (RowPlan::ragged); narrower rows keep vectors that divide them.  us per
// product on the MI355X, dividing against whole vectors, a 3001 x 2049 layer
// of 8 % / an R-MAT graph of 200,000 nodes and 7M nonzeros: fp32 N = 17
// 9.7 -> 8.1 / 130 -> 84, N = 26 7.8 -> 8.1 / 110 -> 95, N = 47 graph of
// 400,000 nodes 356 -> 303; 16-bit N = 17 10.0 -> 10.9 / 127 -> 129, N = 30
// - / 96.5 -> 97.2, N = 39 13.0 -> 9.9 / 167 -> 136, N = 70 14.0 -> 9.5 /
// 183 -> 144, bf16 N = 333 72 -> 39 / -.
constexpr int32_t kRaggedMinN32 = 16;
constexpr int32_t kRaggedMinN16 = 33;

// Where every row is short and B is small, a wavefront of the dividing vectors
// of 16-bit types (N <= 64 of them) reads its row in a few steps, with nothing
// to add across slots, and they stay.  us per product on the MI355X, dividing
// against whole vectors, uniform layers: 300 x 200 of 2 % (4 a row), N = 33 2.8 /
// 3.8, N = 70 2.8 / 3.5; 5000 x 500 of 2 % (10), N = 47 4.1 / 5.1, N = 81 (two
// wavefronts' widths) 5.5 / 5.7; 12,000 x 1000 of 2 % (20), N = 34 6.9 / 9.1, N = 47
// 7.7 / 10.7, N = 70 8.0 / 9.6; of 4 % (40), N = 47 11.3 / 12.7, N = 70 11.9 / 11.6;
// 3000 x 2000 of 4 % (80), N = 34 6.4 / 6.0, N = 47 7.7 / 7.8; with rows of up to
// some 300 among 20, N = 47 14.2 / 9.4, of up to 60 among 4, 7.7 / 4.1.  60,000
// sampled rows of 5 of 240,000, N = 47 18.6 / 15.2.  fp32 gains from whole vectors
// there too (12,000 x 300 of 2 %, N = 47 7.2 / 4.9), but for the smallest (300 x
// 200 of 2 % 2.8 / 3.1).
constexpr int32_t kShortRowCols = 2048;
constexpr int64_t kShortRowNnz = 48;   // nonzeros a row on average,
constexpr int64_t kShortRowMore = 12;  // and at most twice as many and these
// Whether the longest row decides the vectors (K, the average and N fit).
bool short_rows_matter(int32_t M, int32_t K, int64_t nnz, int32_t N, int32_t es);

// Ragged rows gathered often enough are copied to an aligned pitch first
// (padded_pitch): to whole 128-byte lines where that adds at most an eighth,
// else to whole vectors (16-bit types of odd N; the others' vectors start at
// dwords and gained nothing).  Copied when the time saved, by gathered bytes,
// passes the copy's; by half as much again for plans made on the device, which
// may run once.  us per product in place -> copied (copy included) on the
// MI355X: 3001 x 2049 layer of 8 %, bf16 N = 47 11.2 -> 9.8, N = 333 36 -> 27,
// N = 1023 76 -> 47, fp32 N = 333 32 -> 36; R-MAT of 300,000 nodes and 10M
// nonzeros, fp16 N = 47 179 -> 140, N = 127 439 -> 294, N = 255 757 -> 613, fp32
// N = 62 235 -> 251, N = 127 771 -> 544; of 100,000 and 3.4M, fp16 N = 127 88 ->
// 97, fp32 N = 127 182 -> 155, N = 255 351 -> 309; of 30,000 and 1M, fp32 N = 255
// 63 -> 91; Zipf rows, 300,000 columns, 3M, fp16 N = 47 84 -> 79, N = 127 139 ->
// 253.
constexpr int64_t kPadFarBytes = int64_t(24) << 20;  // a B past this comes from behind the L2s:
constexpr double kPadFarGain = 4e-8;     // us saved per gathered byte (measured 1e-8 to 6.5e-8),
constexpr int64_t kPadFarRow = 640;      // of rows of at most so many bytes (a wider one too saves one line),
constexpr double kPadNearGain = 3e-8;    // and within them, 16-bit types (2.5e-8 to 6e-8; fp32 none)
constexpr double kPadFixedUs = 3.0;      // the copy's launch,
constexpr double kPadBytesPerUs = 4e6;   // and its rate, each byte read and written

// Column chunks of ragged rows read in place end inside lines, and with the
// 128-byte chunks of a wide B a row then costs up to twice its lines: they
// take one chunk (two of a small B whose rows fill a wavefront, for the
// parallelism) unless every row of B is gathered so often that the XCDs'
// slices of B pay.  us per product with the chunks of aligned rows / with one
// on the MI355X (before, with vectors that divide N, in brackets): Zipf rows of
// 100,000 columns, 1M nonzeros, fp32 N = 63 80 / 30 (34), N = 127 153 / 54 (116),
// fp16 N = 126 92 / 37 (38); 300,000 columns, 3M, fp32 N = 255 991 / 375 (723);
// R-MAT of 300,000 nodes and 3.5M, fp32 N = 62 158 / 113 (133), N = 127 404 / 326
// (384); of 10,000 and 110,000, N = 255 19.4, 23.5 with one and 17.2 with two (21);
// an 8000 x 8000 layer of 5 % (B's rows 400 times), fp32 N = 333 230 / 259, N =
// 1023 689 / 1063, bf16 N = 333 200 / 200.
constexpr int64_t kRaggedChunkReuse = 128;
constexpr int64_t kRaggedTwoChunkBytes = int64_t(16) << 20;

struct Int4 {
    int32_t x, y, z, w;
};

struct RowPlan {
    // lane geometry
    int32_t elems_per_lane = 1;  // B columns per lane per load (16-byte vectors when possible)
    bool ragged = false;         // elems_per_lane does not divide N: a row's last vector ends at its end
    int32_t log_lanes = 6;       // log2(G): lanes per slot, G >= chunk_lanes
    int32_t chunk_lanes = 64;    // lanes holding data in one column chunk
    int32_t col_chunks = 1;      // column chunks (grid.x = task groups * col_chunks)
    int32_t row_len = 0;         // rows up to this length: one wavefront
    int32_t wide_len = 0;        // rows up to this length: one workgroup (4 wavefronts)
    int32_t seg_len = 0;         // longer rows: segments of at most this length
    int32_t multi_max = 0;       // rows with length <= multi_max go to multi tasks
    std::vector<Int4> tasks;     // wide groups first (4-aligned), then seg, row, multi
    std::vector<int32_t> perm;   // row ids of multi tasks
    std::vector<Int4> longrows;  // {row, first segment slot, segments, 0}
    std::vector<int32_t> order;  // [wavefront slot]: task it runs, -1 idle; empty = task order
    int32_t n_multi = 0, n_seg = 0, n_rowtasks = 0, n_wide = 0;
};

// Row windows of 128 rows routed to an MFMA tile kernel.  For window i:
// windows[i] = {first row, steps, first global step, first nonzero}; step s
// of the window has B rows ucols[(first global step + s) * 32 + 0..31]
// (-1 = padding past the column union) and nonzeros
// entries[eoff[g] .. eoff[g + 1]) with g its global step; an entry packs the
// row within the window (7 bits), the column within the step (5 bits, bit 7)
// and the nonzero index minus the window's first nonzero (bit 12 up).
// Routing.  A window is eligible for the MFMA tile kernel when its condensed
// tile density nnz / (rows * padded |U|) is at least kMfmaMinDensity and no
// step holds more nonzeros than the kernel's entry slots.  The eligible
// windows then go to the tile kernel as a set when a cost model predicts it
// beats the row kernel on them:
//   tile kernel  ~ fixed_us + rounds * (max steps / 4 + fill_iters) * iter_us
//                  (rounds = ceil(workgroups / 256): one workgroup per CU;
//                   4 steps per iteration plus the pipeline fill),
//   row kernel   ~ eligible nnz * N * value size / kRowGatherBytesPerUs
//                  (B-row gathers through L2).
// Constants measured on MI355X (fp16, 4096-row lognormal and Bernoulli
// matrices, N = 256 / 512); the row kernel sustains ~20 TB/s of gathered B
// rows; density below ~0.04 never paid.
constexpr double kMfmaMinDensity = 0.04;
constexpr double kRowGatherBytesPerUs = 20.0e6;

struct MfmaShape {
    int32_t win_rows;          // rows per window
    int32_t tile_cols;         // C columns per workgroup
    int32_t max_step_entries;  // nonzeros a step may hold (entry slots of the kernel)
    double fixed_us, iter_us;  // cost model: launch + prologue, one 4-step iteration
    int32_t fill_iters;        // pipeline fill, in iterations
};
// Paired kernel: 128 x 64 tiles, up to 512 nonzeros per step, a 4-step
// iteration ~0.95 us.  Dense-tile kernels: 128 x 64 tiles, no per-step entry
// limit (a step is a dense 128 x 32 tile), a 4-step iteration ~0.5 us.
constexpr MfmaShape kMfmaPairShape = {128, 64, 512, 3.0, 0.95, 3};
constexpr MfmaShape kMfmaDenseShape = {128, 64, 128 * 32, 3.0, 0.5, 3};
inline const MfmaShape& mfma_shape(uint32_t flags) {
    if (flags & (TCA_PLAN_MFMA_DENSE | TCA_PLAN_MFMA_COMPACT)) return kMfmaDenseShape;
    return kMfmaPairShape;
}

struct MfmaPlan {
    int32_t win_rows = 128;
    std::vector<Int4> windows;
    std::vector<int32_t> ucols;
    std::vector<int32_t> eoff;
    std::vector<uint32_t> entries;
    std::vector<uint8_t> row_mfma;  // per row: covered by an MFMA window
    int64_t nnz = 0;                // nonzeros in MFMA windows
    int64_t cond_cols = 0;          // padded condensed columns, summed over windows
    int32_t rows = 0;
};

// Windows routed by the rule above (min_density replaces kMfmaMinDensity; with
// force every qualifying window, with disable none).  Only for fp16 / bf16 and
// N % 8 == 0; a window qualifies only while its nonzeros fit the entry
// encoding (< 2^20) and no step holds more than shape.max_step_entries.
void plan_mfma(const int32_t* rowptr, const int32_t* colidx, int32_t M, int32_t N, int32_t dtype, bool force,
               bool disable, double min_density, const MfmaShape& shape, MfmaPlan* p);

// Column chunks per XCD pay only when B overflows the L2s: 0 (automatic
// chunking) when B is larger than 8 MiB, else 1.  TCA_SLICES (tuning only)
// forces the number of chunks.
int32_t default_slices(int32_t K, int32_t N, int32_t dtype);

// Lane geometry for width N and value size `es` bytes: the widest vector
// (<= 16 bytes) whose element count divides N, and the column chunks: up to
// 8 chunks of at least 128 bytes (one L2 line of B per chunk row), at most
// 64 lanes each.  `slices` > 0 forces the number of chunks (tuning).
// short_rows: ragged widths keep the vectors that divide them.
void plan_geometry(int32_t N, int32_t es, int32_t slices, bool short_rows, RowPlan* p);

// Ragged rows (RowPlan::ragged) of B that a plan copies to an aligned pitch
// before each product: elements per row of the copy, 0 = read B in place
// (always with TCA_PLAN_NO_SCRATCH, and past the MALL).
int32_t padded_pitch(int32_t K, int64_t nnz, int32_t N, int32_t es, uint32_t flags, bool on_device, const RowPlan& p);

// Lane geometry and task-length thresholds (row_len, wide_len, seg_len,
// multi_max) of the row kernel for a matrix of nnz nonzeros.
// longest: the longest row's nonzeros, read where short_rows_matter.
void plan_row_params(int32_t M, int32_t K, int64_t nnz, int32_t N, int32_t es, uint32_t flags, int32_t slices,
                     int32_t longest, RowPlan* p);

// Row panels with B rows staged in LDS (the panel kernel).  Rows are taken
// longest first (ties by row id) in panels of R = waves * 4 * rpg rows; the
// sorted union of a panel's columns is cut into tiles of at most P columns
// in which no row holds more than kPanelMaxRun nonzeros, and a
// workgroup stages one tile's B rows (all N columns of a column chunk) into
// LDS while its consumer wavefronts multiply the previous tile: every row of
// the panel reads the staged rows of its nonzeros instead of gathering them
// from L2.  Since the CSR columns of a row are sorted and a tile is a range
// of the sorted union, a row's nonzeros in one tile are a contiguous CSR run.
//   slot s of panel p (s = (wave * rpg + i) * 4 + group): rows[p * R + s]
//     (-1 = empty slot); lane group `group` of consumer wave `wave` owns it as
//     its i-th row;
//   tile t (global index): cols[t * P + j] = the B row staged at position j
//     for j < width[t] (padding repeats a valid column; never read);
//   cnt[t * waves * 16 * 4 + (wave * 16 + i) * 4 + group] (bytes): nonzeros
//     of slot s's row in tile t (16 dwords per wave and tile: entries
//     i < rpg), and byte i % 4 of dword kPanelMaxDword + i / 4 the longest
//     of entry i's four counts (the steps the wave takes for entry i);
//   pos[k] for a CSR nonzero k of a panel row: 1 + its position in its tile
//     (the kernel's position 0 is a zero row);
//   units[u] = {panel, first tile, tiles, segment base or -1}: one
//     workgroup; a panel whose nonzeros exceed the unit size is split into
//     panel_units[panel] units by tiles, each writing partial rows that are
//     summed in a fixed order: unit k of a panel whose first segment is f has
//     segment base f + k, and slot s writes segment base + s * panel_units;
//   ustart[u * R + s] = CSR index of slot s's first nonzero in unit u;
//   longrows: {row, first segment, segments, 0} for split panels' rows.
// A panel is taken when its reuse nnz / |union| is at least min_reuse (or
// always with force).  Eligible: N % (16 * E) == 0 for the lane geometry of
// panel_geometry.
struct PanelPlan {
    int32_t waves = 0, rpg = 0, R = 0, P = 0;  // consumer waves, rows per lane group, rows per panel, tile columns
    int32_t elems = 0, chunks = 0;             // B elements per lane, column chunks of C
    int32_t n_panels = 0;
    std::vector<int32_t> rows;
    std::vector<int32_t> cols;
    std::vector<uint8_t> width;  // [tile]: columns of the tile (1..P)
    std::vector<uint8_t> cnt;
    std::vector<uint8_t> pos;  // indexed by CSR nonzero (0 outside panels)
    std::vector<Int4> units;
    std::vector<int32_t> order;  // [workgroup]: unit it runs, -1 = idle (see order_units)
    std::vector<int32_t> panel_units;
    std::vector<int32_t> ustart;
    std::vector<Int4> longrows;
    int64_t n_segments = 0;    // partial rows of split panels
    std::vector<uint8_t> row_panel;  // per row: in a panel
    int64_t nnz = 0;           // nonzeros in panels
    int64_t staged = 0;        // union columns summed over panels
    int32_t n_rows = 0;        // rows in panels
    std::vector<uint8_t> win;  // [panel]: 1 = the kernel takes its run data through per-row windows (panel_window)
    int32_t n_tiles() const { return P ? static_cast<int32_t>(cols.size() / P) : 0; }
};
constexpr int kPanelWaves = 12;   // consumer wavefronts per workgroup (plus four producers: 1024 threads)
constexpr int kPanelRpg = 4;      // rows per 16-lane group
constexpr int kPanelMaxDword = kPanelRpg;  // first dword of the entries' longest counts
constexpr int kPanelCntRows = (kPanelMaxDword + (kPanelRpg + 3) / 4 + 3) / 4 * 4;  // count dwords per wave and tile
static_assert(kPanelRpg <= kPanelMaxDword && kPanelMaxDword + (kPanelRpg + 3) / 4 <= kPanelCntRows, "cnt layout");
constexpr int kPanelMaxRun = 16;  // nonzeros of one row in one tile (one 16-lane batch)
// nnz / |union| a panel needs to be kept.  Measured on MI355X (per SpMM,
// config 2 / config 3): 1.2 1.77 / 3.50 ms, 1.05 - / 3.50, 1.02 1.73 / 3.39,
// 1.0 1.75 / 3.39: staged once per panel, even rows that share few columns
// cost less than the row kernel's gathers; rows that share none stay there.
constexpr double kPanelMinReuse = 1.02;
constexpr int64_t kPanelMinNnz = int64_t(1) << 21;  // fewer nonzeros in panels: none (unless forced)
// Whether the panel kernel takes a panel's run data through windows (a
// window of 16 nonzeros per row serves several tiles): when the panel's
// reuse nnz / |union| is below kPanelWindowReuse its rows hold few nonzeros
// per tile, and the kernel waits on memory more than on issue.  Measured on
// MI355X (panel phase; one box, alternating runs): every panel direct /
// every panel windowed: config 3 (reuse 1.67) 2.82 / 2.34 ms, config 2
// (5.74) 1.53 / 1.57 ms; per panel, config 2 / config 3 whole SpMM:
// threshold 3 1.527-1.534 / 2.672-2.679 ms (config 3's nine hub panels
// direct), 6 1.520-1.544 / 2.620-2.632, every panel windowed 1.575-1.591 /
// 2.626-2.631, none 1.546-1.555 / -.  TCA_PANEL_WINDOW=0 / 1 forces it for
// every panel (tests); TCA_PANEL_WINDOW_REUSE overrides the threshold
// (tuning).
constexpr double kPanelWindowReuse = 6.0;
bool panel_window(int64_t nnz, int64_t staged);
// Launch order of the units (PanelPlan::order).
void order_units(int32_t K, PanelPlan* p);
// The same from each unit's first and last staged column (the GPU planner
// builds those and runs this order on the host).
void order_unit_spans(int32_t K, int32_t chunks, const std::vector<Int4>& units, const std::vector<int64_t>& lo,
                      const std::vector<int64_t>& hi, std::vector<int32_t>* order);
// Routing parameters of the panels (shared by the host and the GPU planner):
// false when the plan takes no panels (TCA_PLAN_NO_PANELS, or by default B
// rows under 256 bytes); else force / min_reuse / min_nnz / unit_nnz for
// plan_panels (TCA_PANEL_MIN_REUSE, TCA_PANEL_MIN_NNZ, TCA_PANEL_UNIT: tuning
// overrides).
struct PanelRoute {
    bool force = false;
    double min_reuse = 0.0;
    int64_t min_nnz = 0, unit_nnz = 0;
};
bool panel_route(int32_t K, int32_t N, int32_t dtype, uint32_t flags, PanelRoute* r);
// Nonzeros per unit for panels holding `tot` nonzeros (unit_nnz > 0: forced).
int64_t panel_unit_nnz(int64_t unit_nnz, int64_t tot);
// Launch order of the row kernel's tasks (RowPlan::order): segments of long
// rows by column range, one range per XCD.  row_order_on: whether a plan
// gets one (one column chunk, at least 32 segments; TCA_ROW_ORDER=0 turns it
// off); the GPU planner builds the same order.
constexpr int32_t kRowOrderSlots = 4;  // wavefronts per row-kernel workgroup (kRowWaves)
bool row_order_on(const RowPlan& p);
void order_row_tasks(const int32_t* colidx, RowPlan* p);
// Lane geometry: 16 lanes cover one column chunk of a B row, E elements each
// (E = 8, 4 or 2 with E * elem_size in 8..32 bytes); 0 when N does not fit.
int32_t panel_elems(int32_t N, int32_t es);
// Default routing also needs B rows of at least 256 bytes (N * elem_size).
bool panel_default_ok(int32_t N, int32_t es);
// Tile width P for a chunk of `chunk_bytes` bytes: two LDS buffers of at most
// 76 KiB, positions fit one byte (P <= 255).
int32_t panel_tile_cols(int32_t chunk_bytes);
// plan_panels with the routing of a plan: none with TCA_PLAN_NO_PANELS, every
// eligible row with TCA_PLAN_FORCE_PANELS, else (B rows of >= 256 bytes)
// panels of reuse >= kPanelMinReuse (every panel when B is larger than the
// MALL) when they hold at least kPanelMinNnz nonzeros in all.
void plan_panels_routed(const int32_t* rowptr, const int32_t* colidx, int32_t M, int32_t K, int32_t N,
                        int32_t dtype, uint32_t flags, const std::vector<uint8_t>& skip, PanelPlan* p);
// Builds the panel plan over the rows with skip[r] == 0 (skip may be empty).
// unit_nnz: nonzeros per workgroup unit (0 = automatic).
// Unless forced, panels are kept only when they hold at least min_nnz nonzeros in all.
void plan_panels(const int32_t* rowptr, const int32_t* colidx, int32_t M, int32_t K, int32_t N, int32_t es,
                 const std::vector<uint8_t>& skip, bool force, double min_reuse, int64_t min_nnz, int64_t unit_nnz,
                 PanelPlan* p);

// Builds the row-kernel task list for rows with skip[r] == 0 (skip may be
// empty).  Rows are assigned longest first.  The categories, in task order:
// wide rows (row_len < length <= wide_len, 4 tasks each), long rows
// (length > wide_len, segments of at most seg_len, summed in a fixed order),
// row tasks (max(multi_max, 0) < length <= row_len), groups of `slots` short
// rows (0 < length <= multi_max), then groups of up to kZeroRows empty rows.
// Per-window statistics the MFMA routing decides on: nonzeros, size of the
// column union, most nonzeros in one 32-column condensed step.
struct WinStat {
    int64_t nz;
    int32_t ucount;
    int32_t maxper;
};
// Which windows (of shape.win_rows rows) go to the tile kernel: eligibility
// (nonzeros per step fit the kernel, density >= min_density unless forced)
// and the cost model against the row kernel.  Shared by the host planner
// (plan_mfma) and the planner on the GPU (statistics computed there).
void route_windows(const std::vector<WinStat>& st, int32_t M, int64_t nnz_total, int32_t N, bool force,
                   double min_density, const MfmaShape& shape, std::vector<uint8_t>* take);

void plan_rows(const int32_t* rowptr, int32_t M, int32_t K, int32_t N, int32_t es, uint32_t flags,
               const std::vector<uint8_t>& skip, bool panels, int32_t slices, RowPlan* p);

// Sorted column union of every window of `win` rows and each nonzero's
// position in it (the indexing exported by tca_condense_windows).
void condense(const int32_t* rowptr, const int32_t* colidx, int32_t M, int32_t win, std::vector<int64_t>* uoff,
              std::vector<int32_t>* ucols, std::vector<int32_t>* cpos);

}  // namespace tca
