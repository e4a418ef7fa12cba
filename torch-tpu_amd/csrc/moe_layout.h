// Host-side layout of the caller-provided workspaces (shared by the launchers).
#pragma once
#include <cmath>
#include <stddef.h>
#include <stdint.h>

namespace moe {

constexpr int kChunk = 256;   // slots ranked by one workgroup in the permutation kernels
// Slots up to which the permutation is one launch that counts every id itself (permute_direct_kernel).  Three launches / one, in
// us, 20480 / 24576 / 32768 / 65536 / 131072 slots: 8 picks of 128 experts 12.0 / 12.3 / 12.6 / 14.1 / 16.8 and 9.4 / 10.5 / 12.7 / 23.0 / 49.6; at
// 32768 slots 8 picks of 256 / 1024 experts 14.2 / 26.2 and 12.8 / 15.3, 2 of 8 10.4 and 14.4.  In a layer, where the first of the three
// rides in the routing launch: 128 experts of 2048 x 768 at 20480 / 24576 / 32768 / 131072 slots 260.8 / 282.0 / 342.9 / 940 and 259.7 / 281.1 /
// 344.8 / 961, 256 of 1024 x 256 at 32768 144.8 and 149.1, 8 of 256 x 128 at 20480 55.0 and 50.1.  So one launch is the better form up to
// 24576 slots at least and the worse one from 32768 on in most layers; the line stays below both.
constexpr int kDirectSlots = 64 * kChunk;

// What the grouped GEMMs multiply: FP8 activations x FP8 weights with scales (the path proper), bf16 x bf16
// (un-quantised experts), or bf16 activations x FP8 weights de-quantised to bf16 in registers (the reference's arithmetic)
enum { kNumericsFp8 = 0, kNumericsBf16 = 1, kNumericsW8A16 = 2 };

static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Rows of an activation-scale tensor are padded to whole 64-byte pieces: the grouped GEMMs fetch
// the scales of 16 reduction steps of a row with one aligned 64-byte read.
static inline int scale_pitch(int n_groups) { return (n_groups + 15) & ~15; }

// Rows of one expert that a grouped-GEMM workgroup owns.  A pure function of the problem
// shape so that the permutation (which builds the tile list) and the GEMM launchers agree
// without passing it around.  A token's K experts are distinct, so no expert ever holds
// more than T rows: small T gets small tiles.
static inline int choose_tile_m(int T, int K, int E) {
  if (T <= 16) return 16;
  if (T <= 32) return 32;
  if (T <= 64) return 64;
  // Balanced routing puts T*K/E rows on an expert, give or take a few standard deviations.  A
  // second, nearly empty tile costs as much weight traffic as a full one, so prefer the tile
  // that holds a typical expert whole.
  // Measured (step in ms with 64 / 128 / 192 rows forced; the 64-row kernel streams its weights into LDS with the
  // non-temporal hint when an expert's rows fit one tile, which the large tiles' register loads do not profit from):
  // DeepSeek-V3 shape, T=512 (16 rows per expert on average) 1.827 / 1.999 / -, T=768 1.877 / 2.033, T=1024 1.925 / 2.062,
  // T=1280 (40 rows) 2.000 / 2.114, T=1536 (48 rows) 2.120 / 2.149, T=2048 (64 rows) 2.412 / 2.227 / 2.252,
  // T=3072 2.993 / 2.404 / 2.410, T=4096 (128 rows) 3.627 / 2.924 / 2.651; Mixtral shape, T=96 (24 rows) 0.252 / 0.290 / 0.298,
  // T=192 (48 rows) 0.297 / 0.312 / 0.319, T=256 (64 rows) 0.338 / 0.319 / 0.325; Qwen3 shape under a skewed load, T=512
  // (32 rows) 0.130 / 0.140, T=768 (48 rows) 0.148 / 0.144, T=1024 0.172 / 0.156.
  // The rule those crossovers follow: under balanced routing an expert's row count is binomial (T*K draws, 1/E each);
  // take the smallest tile that holds mean + 2.4 standard deviations - an expert's rows with about 99 % probability.
  // That puts the 64 | 128 boundary at 47 rows per expert on average and the 128 | 192 boundary at 103.
  const double mean = (double)T * K / E;
  const double reach = mean + 2.4 * std::sqrt(mean * (1.0 - 1.0 / E));
  if (reach <= 64.0) return 64;
  return reach <= 128.0 ? 128 : 192;
}

// Row tile of the dense layers (one "expert" owns every row; M > 128 rows, `items_per_row_tile` strips of the output,
// `steps` 128-steps of the reduction).  Nothing is read from HBM more than once here and the matrix fits the caches,
// so what counts is how the work items fill the 256 compute units and what one item costs: a model instead of a
// table - rounds of work items x (steps x (cost of a step, which grows with the tile's m-tiles) + the item's fixed
// start and end).  Shader cycles measured with the operands coming from L2: a step costs about 300 + 150 per m-tile,
// start and end of an item about 20 000; the 96-row kernel runs two workgroups per unit (512 items per round), one
// hiding the other's start and end, which pays while the reduction is short (kHalfTileMaxSteps).
// Example: 4096 x 7168 -> 1536 (6 strips of 256 columns): 192 rows = 132 items, half the units idle, 56 steps x 2100
// cycles; 128 rows = 192 items x 56 x 1500, a third less.
constexpr int kHalfTileMaxSteps = 20;
static inline int choose_dense_tile_m(long rows, int items_per_row_tile, int steps) {
  int best = 192;
  double best_cost = 0.0;
  const int tiles[4] = {192, 128, 96, 64};
  for (int i = 0; i < 4; i++) {
    const int tm = tiles[i];
    if (tm == 96 && steps > kHalfTileMaxSteps) continue;
    const long items = (rows + tm - 1) / tm * (long)items_per_row_tile;
    const long per_round = tm == 96 ? 512 : 256;
    const long rounds = (items + per_round - 1) / per_round;
    const double item = (double)steps * (300.0 + 150.0 * (tm / 16)) + (tm == 96 ? 10000.0 : 20000.0);
    const double cost = (double)rounds * item * (tm == 96 ? 2.0 : 1.0);      // two resident workgroups share a unit
    if (i == 0 || cost < best_cost * 0.97) { best = tm; best_cost = cost; }     // near-ties go to the taller tile
  }
  return best;
}

// How a dense product on the grouped kernels is cut along its reduction.  A long reduction over few output strips leaves
// half of the compute units without work and the others with a chain of steps that each wait for the weight stream
// (18432 -> 7168 at 300 rows: 140 items of 64 rows x 144 steps, 115 us for 132 MB).  Slices of whole 16-step pieces on the
// tall tiles, fp32, added in order by a second kernel, when the same kind of model says it pays: rounds of items x
// (steps x step + start and end), in shader cycles, plus, for slices, 10 000 for the second launch and their bytes (written
// and read once) at 2000 a cycle.  A step of a 64-row tile counts what it takes with the weights coming from HBM, not L2
// (1500 wide, 1000 in narrow strips).  Up to 32 rows a product is one stream of weights and stays whole.
// Measured, whole op, before -> after: 16384 -> 1024 at 520 / 700 / 1500 / 4000 rows 70 / 72 / 83 / 126 -> 34 / 36 / 53 / 105 us;
// gated MLP 7168 / 18432 at 129 / 300 / 400 rows 165 / 209 / 245 -> 130 / 174 / 219 us (the second product 115 -> 57 + 6 us at 300
// rows, 2.3 TB/s of weights), 4096 / 14336 at 129 / 300 / 600 rows 99 / 107 / 167 -> 71 / 85 / 146 us.
//
// Strips of 128 columns (paired wavefronts, more than 128 rows and 256 columns) are twice the work items, each with a step of
// about 1100 cycles under 128 rows.  Whole, they take a layer of which they are more than half a round and no more than one: the wide
// 64-row tiles that it gets otherwise are one round of 1500-cycle steps.  (Not where that tile is worked on in strips of 64:
// those against these, 4096 -> 6144 at 257 / 320 / 321 rows 24.6 / 25.3 / 30.2 and 25.6 / 26.2 / 26.3 us, wide from 321 rows on, 2048 ->
// 6144 at 257 / 320 rows 15.2 / 15.8 and 16.7 / 16.9, 7168 -> 1536 at 1281 / 1344 / 1345 rows 40.8 / 41.1 / 49.4 and 42.1 / 42.0 / 42.2.)  Sliced,
// they compete by the model, which lets a layer of few strips have them.  Measured, whole op, before ->
// after in us: 7168 -> 1536 at 400 / 560 / 1500 / 2000 rows 28.6 / 35.3 / 50.6 / 53.6 -> 24.9 / 26.0 / 41.6 / 44.2, 7168 -> 7168 at
// 300 / 400 rows 46.3 / 48.0 -> 38.1 / 39.5, 4096 -> 4096 at 560 / 800 rows 30.3 / 31.5 -> 27.2 / 28.9, 16384 -> 1024 at 140 / 400
// rows 28.5 / 31.1 -> 23.8 / 27.0, 7168 -> 2112 at 200 / 1100 rows 27.8 / 48.7 -> 22.9 / 40.8; as the second product of a gated MLP
// 7168 / 2048 at 257 / 400 / 512 rows (the whole MLP) 64.0 / 65.3 / 65.9 -> 62.5 / 63.6 / 63.9.  Outside the line: fewer items
// 4096 -> 4096 at 300 rows (96) 24.8 -> 25.4, 2048 -> 7168 at 200 rows (112) 15.6 -> 16.4; more 7168 -> 1536 at 2800 rows (264: two
// rounds) 59.5 -> 78.4; short reductions 512 -> 4096 at 800 rows 10.7 -> 11.6.
//
// 192 rows of 128 columns take wide layers of 129 to 192 rows: one row tile instead of two of 128 rows that each load the
// weights.  Wide / these strips in us, the weights in the caches and (in brackets) rotated through 500 MB: 4096 -> 22528 at 129 / 192
// rows 34.2 (34.8) / 32.3 (36.8) and 28.2 (33.7) / 31.4 (36.1), 4096 -> 28672 40.0 (36.7) / 35.6 (39.2) and 29.0 (35.3) / 33.5 (38.4), 4096 ->
// 32768 (256 strips, the whole round) 44.5 (38.4) / 38.5 (40.9) and 31.3 (36.3) / 35.3 (40.5).  Outside the line they lose where the
// weights come from memory: fewer strips 4096 -> 18432 at 129 / 192 rows (31.9) / (34.0) and (32.1) / (34.7), longer reductions 5120 ->
// 24576 (42.9) / (45.7) and (44.3) / (46.6), 7168 -> 24576 (53.3) / (58.0) and (54.7) / (59.0), 12288 -> 28672 94.0 / 100.5 and 97.3 / 102.8; and several row
// tiles are no gain: 4096 -> 4096 at 1025 / 1200 rows 34.1 / 35.0 and 33.7 / 35.7, 14336 -> 4096 90.9 / 94.4 and 89.0 / 97.6, 7168 -> 1536 at
// 2800 / 3300 rows 55.7 / 57.6 and 55.5 / 59.1, 7168 -> 7168 at 576 / 768 rows 49.1 / 51.0 and 49.4 / 52.8.  Shorter reductions lose with
// the weights in memory as well, 3968 -> 28672 (39.7) / (40.6) and (40.2) / (41.6), 3072 -> 28672 (30.4) / (32.3) and (31.1) / (32.9), until 2048, which
// the line leaves out: 2048 -> 28672 23.7 (23.2) / 22.4 (24.4) and 19.8 (22.2) / 22.0 (24.5).
// Row tiles of 64 rows over at most this many strips of 256 columns are worked on in strips of 64 (launch_gemm).
constexpr int kNarrowMaxWideItems = 128;
struct DenseSplit {
  int tile_m, slices, k_steps, cols;                     // cols: output columns of a strip, 256 or 128
};
static inline DenseSplit dense_split(long rows, int K, int N) {
  const int steps = K / 128, strips = (N + 255) / 256;
  DenseSplit best = {choose_dense_tile_m(rows, strips, steps), 1, steps, 256};
  const auto rounds = [](long items) { return (double)((items + 255) / 256); };
  double best_cost;
  const long row_tiles = (rows + best.tile_m - 1) / best.tile_m;
  const bool narrow = best.tile_m == 64 && row_tiles * strips <= kNarrowMaxWideItems;
  {
    const double step = best.tile_m > 64 ? 300.0 + 150.0 * (best.tile_m / 16) : narrow ? 1000.0 : 1500.0;
    best_cost = 0.87 * rounds(row_tiles * strips) * (steps * step + 20000.0);      // a clear win or none
  }
  if (rows <= 32 || best.tile_m == 96) return best;
  for (int tm = rows <= 64 ? 64 : 128; tm <= 192; tm += 64) {
    const long items = (rows + tm - 1) / tm * (long)strips;
    for (int len = 16; len < steps; len += 16) {
      const int slices = (steps + len - 1) / len;
      const double cost = rounds(items * slices) * (len * (300.0 + 150.0 * (tm / 16)) + 20000.0) + 10000.0 +
                          8.0 * slices * (double)rows * N / 2000.0;
      if (cost < best_cost) { best = {tm, slices, len, 256}; best_cost = cost; }
    }
  }
  if (rows <= 128 || N <= 256) return best;
  const int pair_strips = (N + 127) / 128;
  const long pair128 = (rows + 127) / 128 * (long)pair_strips;
  if (best.slices == 1 && !narrow) {
    if (steps >= 16 && pair128 > 128 && pair128 <= 256) best = {128, 1, steps, 128};
    else if (rows <= 192 && steps >= 32 && steps < 40 && pair_strips >= 176 && pair_strips <= 256) best = {192, 1, steps, 128};
  }
  // Slices of narrow strips have to be 6 % better by the model.  Where it sees less, wide / narrow measure in us: 14336 -> 4096 at
  // 228 / 256 rows 33.7 / 34.7 and 35.1 / 35.3, 16384 -> 1024 at 700 / 850 / 1280 rows 34.6 / 37.5 / 48.7 and 35.1 / 37.2 / 49.3.  (7168 -> 1536
  // at 593 to 640 rows falls on the wrong side of it: 35.6 whole, 25.8 in slices of narrow strips.)
  best_cost *= 0.94;
  for (int len = 16; len < steps; len += 16) {
    const int slices = (steps + len - 1) / len;
    const double cost = rounds(pair128 * slices) * (len * 1100.0 + 20000.0) + 10000.0 + 8.0 * slices * (double)rows * N / 2000.0;
    if (cost < best_cost) { best = {128, slices, len, 128}; best_cost = cost; }
  }
  return best;
}
// No product of more rows is sliced: with q rounds of whole items of a tall tile the slices cost at least q (steps x step +
// 40 000) cycles and the whole product at most 0.87 / 0.97 (q + 1)(steps x step + 20 000) - the tile that is chosen is at
// most 1 / 0.97 dearer than any other, and not the 64-row one from four rounds on - which is less from q = 9 on.  (Narrow strips
// are the dearer slices there: two or more wide strips of N > 256 columns make at least 2 s - 1 narrow ones of 1100 cycles.  At least
// 512: up to there the per-wavefront kernels have slices of their own.)
static inline long dense_split_max_rows(int K, int N) {
  return K / 128 > 16 ? 512 + 192 * (9 * 256 / ((N + 255) / 256) + 1l) : 512;
}
static inline size_t dense_split_bytes(long rows, int K, int N) {
  const DenseSplit s = dense_split(rows, K, N);
  return s.slices > 1 ? (size_t)s.slices * rows * N * 4 : 0;
}

struct PermuteWs {
  int32_t *chunk_counts;   // [n_chunks, E]
  int32_t *tile_prefix;    // [E + 1] first tile of each expert; [E] = number of tiles
  int32_t *tile_expert;    // [max_tiles]
  int32_t *tile_desc;      // [max_tiles][8]: expert, its first tile, its tiles, its first row, its rows, 0, 0, 0
  int32_t *expert_count;   // [E] slots per expert (between the two halves of the scan kernel)
  int32_t *arrivals;       // [1] workgroups of the scan kernel that have finished their first half
  int n_chunks;
  int max_tiles;
};

static inline int permute_max_tiles(int T, int K, int E) {
  const int tm = choose_tile_m(T, K, E);
  long tk = (long)T * K;
  long a = tk / tm + E;           // sum_e ceil(n_e / tm) <= TK/tm + (#non-empty experts)
  long b = tk;                    // and never more than one tile per row
  long m = a < b ? a : b;
  return (int)(m < 1 ? 1 : m);
}

static inline size_t permute_ws_bytes(int T, int K, int E) {
  long tk = (long)T * K;
  size_t n_chunks = (size_t)((tk + kChunk - 1) / kChunk);
  if (n_chunks == 0) n_chunks = 1;
  size_t ints = n_chunks * (size_t)E + 2 * (size_t)(E + 1) + 9 * (size_t)permute_max_tiles(T, K, E) + 8;
  return align_up(ints * 4, 256);
}

static inline PermuteWs permute_ws_layout(void *ws, int T, int K, int E) {
  PermuteWs p;
  long tk = (long)T * K;
  p.n_chunks = (int)((tk + kChunk - 1) / kChunk);
  if (p.n_chunks == 0) p.n_chunks = 1;
  p.max_tiles = permute_max_tiles(T, K, E);
  p.chunk_counts = (int32_t *)ws;
  p.expert_count = p.chunk_counts + (size_t)p.n_chunks * E;
  p.arrivals = p.expert_count + E;
  p.tile_prefix = p.arrivals + 1;
  p.tile_expert = p.tile_prefix + (E + 1);
  // 32-byte aligned: one descriptor is fetched with a single scalar load
  p.tile_desc = (int32_t *)(((uintptr_t)(p.tile_expert + p.max_tiles) + 31) & ~(uintptr_t)31);
  return p;
}

}  // namespace moe
