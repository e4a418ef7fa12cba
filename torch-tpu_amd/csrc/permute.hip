// Token permutation: a stable counting sort of the flattened [T*K] expert ids.
//
// No host round trip: the grouped GEMMs that follow read the expert offsets and the tile list from device memory.
// Up to kChunk slots are done by one workgroup, up to kDirectSlots by one launch of a workgroup per chunk that counts all
// ids for itself (permute_direct_kernel); larger problems by three small kernels:
//   count    one wavefront per chunk of kChunk consecutive slots: per-chunk histogram in LDS.
//   scan     one wavefront per expert: running sum over the chunks (turns the histogram into
//            the chunk's starting rank inside its expert); the workgroup that finishes last adds
//            an exclusive scan over the experts -> expert_offsets, and the list of row tiles the
//            GEMMs walk.
//   scatter  one workgroup per chunk, one wavefront per 64 slots: ranks its slots in slot order
//            with a ballot "match-any" loop, so equal experts keep their original order (stable),
//            and writes sorted_slot / slot_to_row.
#include "moe_common.h"
#include "moe_layout.h"
#include "permute_small.h"
#include "act_quant.h"
#include "../../include/moe_hip.h"

namespace moe {

// rank of each lane among the lanes holding the same expert id, in lane order; also the
// size of that set and whether the lane is the last of it.
// One ballot per bit of the id: a lane's set is where all bits agree with its own.  (A loop over the distinct ids, each
// fetched from its first lane, is up to 64 dependent rounds where the bits of 256 experts are 8.  All three launches above
// kDirectSlots, loop -> ballots: 16384 x 8 slots of 128 experts 23.7 -> 16.8 us, 4096 x 8 of 256 / 1024 20.6 / 33.0 -> 14.1 / 26.2, 16384 x 2
// of 8 11.5 -> 10.5; every slot on the first 8 of 128 17.0 -> 15.9.)
__device__ __forceinline__ void match_rank(int v, bool valid, int lane, int n_bits, int &rank, int &cnt, bool &is_last) {
  uint64_t m = __ballot(valid);
  for (int b = 0; b < n_bits; b++) {
    const bool one = (v >> b) & 1;
    const uint64_t ones = __ballot(one);
    m &= one ? ones : ~ones;
  }
  if (!valid) m = 0;
  rank = __popcll(m & ((1ull << lane) - 1));
  cnt = __popcll(m);
  is_last = valid && lane == 63 - __clzll((long long)m);
}
__device__ __forceinline__ int id_bits(int E) { return 32 - __clz(E - 1 | 1); }

// The per-slot output row of a slot without an expert is zero: its one thread clears it (such slots are rare - a rank of
// an expert-parallel group sees them for the experts it does not hold).  rows null: nothing to clear.
__device__ __forceinline__ void zero_slot_row(uint16_t *__restrict__ rows, int row_len, int slot) {
  if (rows == nullptr) return;
  v4i *row = (v4i *)(rows + (size_t)slot * row_len);
  for (int i = 0; i < row_len / 8; i++) row[i] = (v4i){0, 0, 0, 0};
}

__global__ __launch_bounds__(64) void permute_count_kernel(const int32_t *__restrict__ ids, int TK, int E,
                                                           int32_t *__restrict__ chunk_counts,
                                                           int32_t *__restrict__ arrivals) {
  __shared__ int hist[MOE_MAX_EXPERTS];
  const int lane = threadIdx.x, c = blockIdx.x;
  if (c == 0 && lane == 0) *arrivals = 0;               // the scan kernel counts its workgroups here
  for (int e = lane; e < E; e += 64) hist[e] = 0;
  __syncthreads();
  const int lo = c * kChunk;
  for (int s = lo + lane; s < min(lo + kChunk, TK); s += 64) {
    int v = ids[s];
    if (v >= 0 && v < E) atomicAdd(&hist[v], 1);
  }
  __syncthreads();
  for (int e = lane; e < E; e += 64) chunk_counts[(size_t)c * E + e] = hist[e];
}

// exclusive scan of one value per thread over a 1024-thread workgroup
__device__ __forceinline__ int block_exclusive_scan(int x, int *lds_wave_sums, int &total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = x;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int y = __shfl_up(inc, off, 64);
    if (lane >= off) inc += y;
  }
  if (lane == 63) lds_wave_sums[wave] = inc;
  __syncthreads();
  int base = 0, tot = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
    int s = lds_wave_sums[w];
    if (w < wave) base += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return base + inc - x;
}

// What the GEMMs read, from the experts' totals (thread t of 256 holds those of experts 4 t .. 4 t + 3): the exclusive scan
// over the experts -> expert_offsets, and the list of row tiles.
struct ListSmem {
  int wave_sums[16];
  int t_first[MOE_MAX_EXPERTS + 1], t_count[MOE_MAX_EXPERTS], t_off[MOE_MAX_EXPERTS];
};
__device__ __forceinline__ void write_lists(ListSmem &sm, const int (&count)[4], int E, int tile_m, int max_tiles,
                                            int32_t *__restrict__ expert_offsets, int32_t *__restrict__ tile_prefix,
                                            int32_t *__restrict__ tile_expert, int32_t *__restrict__ tile_desc) {
  int tiles[4], rows_mine = 0, tiles_mine = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    tiles[j] = (count[j] + tile_m - 1) / tile_m;
    rows_mine += count[j];
    tiles_mine += tiles[j];
  }
  int total, total_tiles;
  int off = block_exclusive_scan(rows_mine, sm.wave_sums, total);
  int first_tile = block_exclusive_scan(tiles_mine, sm.wave_sums, total_tiles);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = 4 * threadIdx.x + j;
    if (e < E) {
      expert_offsets[e] = off;
      tile_prefix[e] = first_tile;
    }
    if (e < MOE_MAX_EXPERTS) {
      sm.t_first[e] = e < E ? first_tile : total_tiles;
      sm.t_count[e] = count[j];
      sm.t_off[e] = off;
    }
    off += count[j];
    first_tile += tiles[j];
  }
  if (threadIdx.x == 0) {
    expert_offsets[E] = total;
    tile_prefix[E] = total_tiles;
    sm.t_first[MOE_MAX_EXPERTS] = total_tiles;
  }
  __syncthreads();
  // The tile list, one thread per tile: under a skewed load one expert holds hundreds of row tiles, and a loop over
  // them in that expert's thread would be the longest chain of the kernel.  A tile finds its expert by bisection of
  // the first-tile table (experts without a tile share their successor's entry and are never the answer).
  const int n_tiles = min(total_tiles, max_tiles);
  for (int j = threadIdx.x; j < n_tiles; j += 256) {
    int lo = 0, hi = E;                                 // sm.t_first[lo] <= j < sm.t_first[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (sm.t_first[mid] <= j) lo = mid; else hi = mid;
    }
    const int c = sm.t_count[lo];
    tile_expert[j] = lo;
    v4i *d = (v4i *)(tile_desc + (size_t)j * 8);
    d[0] = (v4i){lo, sm.t_first[lo], (c + tile_m - 1) / tile_m, sm.t_off[lo]};
    d[1] = (v4i){c, 0, 0, 0};
  }
}

// Scan.  First half, one wavefront per expert: a running sum over the chunks turns each chunk's histogram entry into
// the rank of the chunk's first slot inside the expert (64 lanes x 8 chunks at a time: every load of a round is
// independent of the others), and leaves the expert's total.  Second half, by the workgroup that arrives last (a
// counter the count kernel cleared): exclusive scan over the experts -> expert_offsets, and the list of row tiles the
// GEMMs walk.  Workgroups of four wavefronts with a few registers each find room on a compute unit whatever else runs
// there.
constexpr int kScanWaves = 4;
__global__ __launch_bounds__(64 * kScanWaves) void permute_scan_kernel(int32_t *__restrict__ chunk_counts, int n_chunks,
                                                                       int E, int tile_m, int max_tiles,
                                                                       int32_t *__restrict__ expert_offsets,
                                                                       int32_t *__restrict__ tile_prefix,
                                                                       int32_t *__restrict__ tile_expert,
                                                                       int32_t *__restrict__ tile_desc,
                                                                       int32_t *__restrict__ expert_count,
                                                                       int32_t *__restrict__ arrivals, int n_scan,
                                                                       const QuantJob ride) {
  // The scan is a few dozen workgroups and a chain of latencies; workgroups past its own quantise the activations
  // (pure streaming, needed only by the GEMM after the permutation) in the shadow of it.
  if ((int)blockIdx.x >= n_scan) {
    act_quant_thread(ride.x, ride.n_groups, ride.groups_per_row, ride.pitch, ride.q, ride.s,
                     (size_t)(blockIdx.x - n_scan) * (64 * kScanWaves) + threadIdx.x);
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int e_mine = blockIdx.x * kScanWaves + wave;
  if (e_mine < E) {
    constexpr int B = 8;
    int running = 0;
    for (int c0 = 0; c0 < n_chunks; c0 += 64 * B) {
      const int c = c0 + lane * B;
      int x[B];
#pragma unroll
      for (int i = 0; i < B; i++) x[i] = c + i < n_chunks ? chunk_counts[(size_t)(c + i) * E + e_mine] : 0;
      int sum = 0;
#pragma unroll
      for (int i = 0; i < B; i++) sum += x[i];
      int inc = sum;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(inc, off, 64);
        if (lane >= off) inc += y;
      }
      int rank = running + inc - sum;
#pragma unroll
      for (int i = 0; i < B; i++) {
        if (c + i < n_chunks) chunk_counts[(size_t)(c + i) * E + e_mine] = rank;
        rank += x[i];
      }
      running += __shfl(inc, 63, 64);
    }
    if (lane == 0) expert_count[e_mine] = running;
  }
  __shared__ int is_last;
  // This workgroup's totals are visible device-wide before its arrival is counted.  One fence per workgroup, by the
  // thread that counts, after the barrier that orders the other wavefronts' stores before it: on this chip a
  // device-scope fence writes back and invalidates the whole L2 of its XCD, so they are worth counting.
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    is_last = atomicAdd(arrivals, 1) == n_scan - 1;
  }
  __syncthreads();
  if (!is_last) return;
  __threadfence();

  // thread t owns experts 4 t .. 4 t + 3 (MOE_MAX_EXPERTS = 4 x 256 threads)
  static_assert(MOE_MAX_EXPERTS <= 4 * 64 * kScanWaves, "four experts per thread");
  __shared__ ListSmem lists;
  int count[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = 4 * threadIdx.x + j;
    count[j] = e < E ? __hip_atomic_load(expert_count + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
  }
  write_lists(lists, count, E, tile_m, max_tiles, expert_offsets, tile_prefix, tile_expert, tile_desc);
}

// One workgroup per chunk, one wavefront per 64 consecutive slots of it: every wavefront ranks its
// slots among themselves, leaves its per-expert counts in LDS, and adds the counts of the
// wavefronts before it - all slots of the chunk are placed in one round.
__global__ __launch_bounds__(kChunk) void permute_scatter_kernel(const int32_t *__restrict__ ids, int TK, int E,
                                                                 const int32_t *__restrict__ chunk_counts,
                                                                 const int32_t *__restrict__ expert_offsets,
                                                                 int32_t *__restrict__ sorted_slot,
                                                                 int32_t *__restrict__ slot_to_row,
                                                                 uint16_t *__restrict__ zero_rows, int row_len) {
  constexpr int NWV = kChunk / 64;
  __shared__ int base[MOE_MAX_EXPERTS];
  __shared__ int wcount[NWV][MOE_MAX_EXPERTS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = blockIdx.x;
  for (int e = tid; e < E; e += kChunk) {
    base[e] = expert_offsets[e] + chunk_counts[(size_t)c * E + e];
#pragma unroll
    for (int w = 0; w < NWV; w++) wcount[w][e] = 0;
  }
  const int s = c * kChunk + tid;
  const int v = s < TK ? ids[s] : -1;
  const bool valid = s < TK && v >= 0 && v < E;
  int rank, cnt;
  bool is_last;
  match_rank(v, valid, lane, id_bits(E), rank, cnt, is_last);
  __syncthreads();
  if (valid && is_last) wcount[wave][v] = cnt;
  __syncthreads();
  int row = -1;
  if (valid) {
    row = base[v] + rank;
    for (int w = 0; w < wave; w++) row += wcount[w][v];
  }
  if (valid && row < TK) sorted_slot[row] = s;
  if (s < TK) slot_to_row[s] = row;
  if (s < TK && row < 0) zero_slot_row(zero_rows, row_len, s);
}

// The whole permutation in one launch, up to kDirectSlots: a workgroup per chunk reads every id - the 64 KB come from L2 -
// and counts those before its chunk apart from the rest, so that it knows the offsets of its own slots without waiting for
// anybody; one more workgroup leaves the offsets and the tile list, and those after it quantise the activations.  Three (with
// counts from the routing launch two) short dependent launches of 3 to 9 us each, a few dozen workgroups, become one.  Whole
// calls, before -> after in us: Qwen3 shape at 300 / 1500 tokens 148.5 -> 137.4 / 198.8 -> 189.3, its un-quantised experts at 2048
// tokens (64 chunks) 329 -> 320, the per-slot op at 470 tokens 149.6 -> 137.4, 81 experts of 1152 x 384 at 1143 tokens 65.9 ->
// 55.1, Mixtral shape at 256 tokens 326 -> 318, 8 experts of 256 x 512 at 516 tokens 46.2 -> 38.8.
// Reading everything grows with the square of the chunks: above kDirectSlots the three kernels take over.
//
// COPIES: lanes that add to one counter wait for one another, and a wavefront whose 64 slots all ask for one expert takes
// about ten times as long to count as one whose slots differ.  The experts of a token are distinct, so K picks put at most
// 64 / K slots of a wavefront on one expert.  For one pick, and for two among few experts, a load that collapsed made the
// launch as slow as the three that it replaces from about 30 and 56 chunks on, and slower above.  From 25 and 49 on the counts are
// kept in several copies, neighbouring lanes adding to different ones (at an odd pitch: the copies of a counter sit in different
// banks), which are added up afterwards.  Three launches / one copy / copies in us, every slot on the first K experts: 16384 x 1
// slots, 8 experts 10.5 / 18.0 / 9.1, 256 experts 12.5 / 18.4 / 9.7, 512 experts 14.7 / 18.5 / 12.4; 8192 x 2, 8 experts 10.6 / 11.4 / 9.1.
// Evenly spread: 16384 x 1, 8 experts 11.3 / 8.6 / 9.1, 256 experts 19.3 / 8.5 / 9.6; 8192 x 2, 8 experts 11.3 / 8.6 / 9.1.  Outside
// the line one copy is no slower than three launches however the load lies: collapsed, 4352 x 1 slots (17 chunks) 10.4 / 8.2, 6144 x 2 of
// 8 experts (48 chunks) 10.5 / 9.6, 8192 x 2 of 128 experts 12.0 / 11.6, 5461 x 3 of 8 experts 11.4 / 9.9, 2048 x 8 of 128 experts
// 12.7 / 8.2, 16384 x 1 of 1024 21.6 / 18.7.
constexpr int kCountTable = MOE_MAX_EXPERTS + 16;        // eight copies of up to 129 counts, four of 257, two of 513
static int direct_copies(int K, int E, int n_chunks) {
  if (!(K == 1 ? E <= 512 && n_chunks > 24 : K == 2 && E <= 64 && n_chunks > 48)) return 1;
  return E <= 128 ? 8 : E <= 256 ? 4 : 2;
}

template <int COPIES>
__global__ __launch_bounds__(kChunk) void permute_direct_kernel(
    const int32_t *__restrict__ ids, int TK, int E, int n_chunks, int tile_m, int max_tiles,
    int32_t *__restrict__ sorted_slot, int32_t *__restrict__ expert_offsets, int32_t *__restrict__ slot_to_row,
    int32_t *__restrict__ tile_prefix, int32_t *__restrict__ tile_expert, int32_t *__restrict__ tile_desc,
    uint16_t *__restrict__ zero_rows, int row_len, const QuantJob ride) {
  if ((int)blockIdx.x > n_chunks) {
    act_quant_thread(ride.x, ride.n_groups, ride.groups_per_row, ride.pitch, ride.q, ride.s,
                     (size_t)(blockIdx.x - n_chunks - 1) * kChunk + threadIdx.x);
    return;
  }
  constexpr int NWV = kChunk / 64;
  struct Place {
    int wave_sums[16];
    int wcount[NWV][MOE_MAX_EXPERTS];
  };
  constexpr int kTable = COPIES > 1 ? kCountTable : MOE_MAX_EXPERTS;
  __shared__ int before[kTable], rest[kTable];
  __shared__ union { Place place; ListSmem lists; } sm;
  // the workgroup of the lists goes first: its chain is the longer one
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = blockIdx.x == 0 ? n_chunks : (int)blockIdx.x - 1;
  for (int e = tid; e < E; e += kChunk) {
    before[e] = 0;
    rest[e] = 0;
    if (c < n_chunks) {
#pragma unroll
      for (int w = 0; w < NWV; w++) sm.place.wcount[w][e] = 0;
    }
  }
  const int pitch = E | 1;
  int *const my_before = before + (lane & (COPIES - 1)) * pitch, *const my_rest = rest + (lane & (COPIES - 1)) * pitch;
  if constexpr (COPIES > 1) {
    for (int i = E + tid; i < COPIES * pitch; i += kChunk) {
      before[i] = 0;
      rest[i] = 0;
    }
  }
  __syncthreads();
  constexpr int B = 16;                                  // chunks asked for at a time
  int v = -1;
  for (int i0 = 0; i0 < n_chunks; i0 += B) {
    int id[B];
#pragma unroll
    for (int i = 0; i < B; i++) {
      const int s = (i0 + i) * kChunk + tid;
      id[i] = s < TK ? ids[s] : -1;
    }
#pragma unroll
    for (int i = 0; i < B; i++) {
      if (i0 + i == c) v = id[i];
      if (id[i] >= 0 && id[i] < E) {
        if constexpr (COPIES > 1) atomicAdd((i0 + i < c ? my_before : my_rest) + id[i], 1);
        else atomicAdd(i0 + i < c ? &before[id[i]] : &rest[id[i]], 1);
      }
    }
  }
  __syncthreads();
  if constexpr (COPIES > 1) {
    for (int e = tid; e < E; e += kChunk) {
      int b = before[e], r = rest[e];
#pragma unroll
      for (int i = 1; i < COPIES; i++) {
        b += before[i * pitch + e];
        r += rest[i * pitch + e];
      }
      before[e] = b;
      rest[e] = r;
    }
    __syncthreads();
  }
  static_assert(MOE_MAX_EXPERTS <= 4 * kChunk, "four experts per thread");
  int first[4], count[4], mine = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int e = 4 * tid + j;
    first[j] = e < E ? before[e] : 0;
    count[j] = e < E ? first[j] + rest[e] : 0;
    mine += count[j];
  }
  if (c == n_chunks) {
    write_lists(sm.lists, count, E, tile_m, max_tiles, expert_offsets, tile_prefix, tile_expert, tile_desc);
    return;
  }
  const int s = c * kChunk + tid;
  const bool valid = v >= 0 && v < E;
  int rank, cnt, total;
  bool is_last;
  match_rank(v, valid, lane, id_bits(E), rank, cnt, is_last);
  if (is_last) sm.place.wcount[wave][v] = cnt;
  int off = block_exclusive_scan(mine, sm.place.wave_sums, total);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (4 * tid + j < E) before[4 * tid + j] = off + first[j];       // where the expert's slots of this chunk begin
    off += count[j];
  }
  __syncthreads();
  int row = -1;
  if (valid) {
    row = before[v] + rank;
    for (int w = 0; w < wave; w++) row += sm.place.wcount[w][v];
    sorted_slot[row] = s;
  }
  if (s < TK) {
    slot_to_row[s] = row;
    if (row < 0) zero_slot_row(zero_rows, row_len, s);
  }
}

__global__ __launch_bounds__(kChunk) void permute_small_kernel(const int32_t *__restrict__ ids, int TK, int E, int tile_m,
                                                              int max_tiles, int32_t *__restrict__ sorted_slot,
                                                              int32_t *__restrict__ expert_offsets,
                                                              int32_t *__restrict__ slot_to_row,
                                                              int32_t *__restrict__ tile_prefix,
                                                              int32_t *__restrict__ tile_expert,
                                                              int32_t *__restrict__ tile_desc,
                                                              uint16_t *__restrict__ zero_rows, int row_len) {
  __shared__ PermuteSmallSmem sm;
  const int s = threadIdx.x;
  const int v = (s < TK) ? ids[s] : -1;
  permute_small_block(sm, v, TK, E, tile_m, max_tiles, sorted_slot, expert_offsets, slot_to_row, tile_prefix, tile_expert,
                      tile_desc);
  if (s < TK && (v < 0 || v >= E)) zero_slot_row(zero_rows, row_len, s);
}

// The same with the activation quantisation in the launch: workgroup 0 permutes, the workgroups after it quantise x
// (eight lanes per 128-column group).  At this size either is one short dependent chain; side by side they cost one launch.
__global__ __launch_bounds__(kChunk) void permute_small_quant_kernel(
    const int32_t *__restrict__ ids, int TK, int E, int tile_m, int max_tiles, int32_t *__restrict__ sorted_slot,
    int32_t *__restrict__ expert_offsets, int32_t *__restrict__ slot_to_row, int32_t *__restrict__ tile_prefix,
    int32_t *__restrict__ tile_expert, int32_t *__restrict__ tile_desc, uint16_t *__restrict__ zero_rows, int row_len,
    const uint16_t *__restrict__ x, size_t n_groups, int groups_per_row, int pitch, uint8_t *__restrict__ xq,
    float *__restrict__ xs) {
  if (blockIdx.x > 0) {
    act_quant_thread(x, n_groups, groups_per_row, pitch, xq, xs, (size_t)(blockIdx.x - 1) * kChunk + threadIdx.x);
    return;
  }
  __shared__ PermuteSmallSmem sm;
  const int s = threadIdx.x;
  const int v = (s < TK) ? ids[s] : -1;
  permute_small_block(sm, v, TK, E, tile_m, max_tiles, sorted_slot, expert_offsets, slot_to_row, tile_prefix, tile_expert,
                      tile_desc);
  if (s < TK && (v < 0 || v >= E)) zero_slot_row(zero_rows, row_len, s);
}

// Permutation of at most kChunk slots and quantisation of x [T, H] bf16 -> xq e4m3fn [T, H], xs fp32 (pitch
// scale_pitch(H / 128)) in one launch.  The caller has checked T * K <= kChunk, H % 128 == 0 and the pointers.
int permute_quant_small_launch(hipStream_t st, const int32_t *ids, int T, int K, int E, int tile_m, int32_t *sorted_slot,
                               int32_t *expert_offsets, int32_t *slot_to_row, const PermuteWs &ws, uint16_t *zero_rows,
                               int row_len, const uint16_t *x, int H, uint8_t *xq, float *xs) {
  const size_t groups = (size_t)T * (H / kBlock);
  const unsigned quant_blocks = (unsigned)((quant_threads(groups) + kChunk - 1) / kChunk);
  permute_small_quant_kernel<<<1 + quant_blocks, kChunk, 0, st>>>(ids, T * K, E, tile_m, ws.max_tiles, sorted_slot,
                                                                  expert_offsets, slot_to_row, ws.tile_prefix,
                                                                  ws.tile_expert, ws.tile_desc, zero_rows, row_len, x,
                                                                  groups, H / kBlock, scale_pitch(H / kBlock), xq, xs);
  return (int)hipGetLastError();
}

// zero_rows (may be null): a [T*K, row_len] bf16 tensor in slot order whose rows of slots WITHOUT an expert (id outside
// [0, E)) are cleared here - the per-slot output form: nothing else ever writes those rows
// counted: the routing launch has filled ws.chunk_counts and ws.arrivals is zero (more than kDirectSlots slots only)
// ride (may be null; more than kChunk slots only): activations quantised by extra workgroups of the launch (of the scan, if there are three)
int permute_launch(hipStream_t st, const int32_t *ids, int T, int K, int E, int tile_m, int32_t *sorted_slot,
                   int32_t *expert_offsets, int32_t *slot_to_row, const PermuteWs &ws, uint16_t *zero_rows, int row_len,
                   bool counted, const QuantJob *ride) {
  const int TK = T * K;
  if (TK <= kChunk) {
    permute_small_kernel<<<1, kChunk, 0, st>>>(ids, TK, E, tile_m, ws.max_tiles, sorted_slot, expert_offsets, slot_to_row,
                                           ws.tile_prefix, ws.tile_expert, ws.tile_desc, zero_rows, row_len);
    return (int)hipGetLastError();
  }
  const QuantJob job = ride ? *ride : QuantJob{};
  if (!counted && TK <= kDirectSlots) {
    const int copies = direct_copies(K, E, ws.n_chunks);
    const auto kernel = copies == 8 ? permute_direct_kernel<8> : copies == 4 ? permute_direct_kernel<4>
                        : copies == 2 ? permute_direct_kernel<2> : permute_direct_kernel<1>;
    kernel<<<ws.n_chunks + 1 + job.blocks(), kChunk, 0, st>>>(
        ids, TK, E, ws.n_chunks, tile_m, ws.max_tiles, sorted_slot, expert_offsets, slot_to_row, ws.tile_prefix, ws.tile_expert,
        ws.tile_desc, zero_rows, row_len, job);
    return (int)hipGetLastError();
  }
  if (!counted) permute_count_kernel<<<ws.n_chunks, 64, 0, st>>>(ids, TK, E, ws.chunk_counts, ws.arrivals);
  static_assert(64 * kScanWaves == 256 && kChunk == 256, "a quantising workgroup has 256 threads");
  const int n_scan = (E + kScanWaves - 1) / kScanWaves;
  permute_scan_kernel<<<n_scan + job.blocks(), 64 * kScanWaves, 0, st>>>(
      ws.chunk_counts, ws.n_chunks, E, tile_m, ws.max_tiles, expert_offsets, ws.tile_prefix, ws.tile_expert, ws.tile_desc,
      ws.expert_count, ws.arrivals, n_scan, job);
  permute_scatter_kernel<<<ws.n_chunks, kChunk, 0, st>>>(ids, TK, E, ws.chunk_counts, expert_offsets, sorted_slot,
                                                     slot_to_row, zero_rows, row_len);
  return (int)hipGetLastError();
}

}  // namespace moe

extern "C" size_t moe_permute_workspace_bytes(int T, int K, int E) {
  if (T < 0 || K < 1 || E < 1) return 0;
  return moe::permute_ws_bytes(T, K, E);
}

extern "C" int moe_tile_rows(int T, int K, int E) { return moe::choose_tile_m(T, K, E); }

extern "C" int moe_permute(void *stream, const int32_t *ids, int T, int K, int E, int32_t *sorted_slot,
                           int32_t *expert_offsets, int32_t *slot_to_row, void *workspace, size_t workspace_bytes) {
  using namespace moe;
  if (!expert_offsets || !workspace) return MOE_E_NULL;
  if (T != 0 && (!ids || !sorted_slot || !slot_to_row)) return MOE_E_NULL;   // an empty batch still gets its (all zero) offsets
  if (T < 0 || K < 1 || K > MOE_MAX_TOPK || E < 1 || E > MOE_MAX_EXPERTS) return MOE_E_SHAPE;
  if ((long)T * K > (1l << 30)) return MOE_E_SHAPE;
  if (workspace_bytes < permute_ws_bytes(T, K, E)) return MOE_E_WORKSPACE;
  if ((uintptr_t)workspace % 4) return MOE_E_ALIGN;
  PermuteWs ws = permute_ws_layout(workspace, T, K, E);
  return permute_launch((hipStream_t)stream, ids, T, K, E, choose_tile_m(T, K, E), sorted_slot, expert_offsets,
                        slot_to_row, ws, nullptr, 0, false, nullptr);
}
