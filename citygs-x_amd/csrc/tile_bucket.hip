// Binning by tile without a global sort.  The list the rasterizer needs is "instances ordered by (tile, depth
// bits), ties in emission order" (cuda_rasterizer/rasterizer_impl.cu:74-144, :675-697: duplicateWithKeys, a stable
// radix sort on the (tile << 32 | depth) key, identifyTileRanges).  The tile part of that key takes few values
// and every tile's list is short, so the same list comes out of
//   1. a counting sort by tile: per-workgroup tile histograms in LDS, a prefix over workgroups and tiles (which
//      is also the table of tile ranges), and a scatter of every instance into its tile's segment, in any order;
//   2. one workgroup per tile sorting its segment in registers by (depth bits, emission index): the emission index
//      is unique, so the order does not depend on how the scatter happened to fill the segment, and it is the
//      order a stable sort on the depth bits would leave.
// No pass over all instances per digit, no look-back chain.  Lists of up to 4096 records are sorted in registers
// by a bitonic network (below); longer ones by a radix sort on the depth bits that stays inside the CU
// (tile_radix.hip).  The ranges kernel sorts the tiles into those classes.
#include <atomic>

#include "gs_common.h"
#include "gs_kernels.h"
#include "tile_lists.h"

namespace gs {
namespace {

constexpr int BK_THREADS = 1024;        // counting and scatter kernels
constexpr int BK_MAX_BLOCKS = 256;
// Gaussians per workgroup, at least.  The counting and scatter kernels of a small view take as long as one workgroup does:
// 50 k Gaussians, 640x480, 9.7 + 16.8 us with 4096, 6.1 + 12.1 with 1024, 5.4 + 11.4 with 512 (256: the same).
constexpr int BK_MIN_PER_BLOCK = 512;
constexpr int BK_BATCH = 4;             // Gaussians a thread loads ahead

__host__ __device__ inline int bucket_per_block(int P) {
  // a multiple of four, so that a thread's four consecutive Gaussians start at a 16-byte boundary of every
  // per-Gaussian array of words
  const int per = ((P + BK_MAX_BLOCKS - 1) / BK_MAX_BLOCKS + 3) & ~3;
  return per < BK_MIN_PER_BLOCK ? BK_MIN_PER_BLOCK : per;
}
__host__ __device__ inline int bucket_blocks(int P) {
  const int per = bucket_per_block(P);
  return (P + per - 1) / per;
}

// Which chunk of Gaussians a workgroup takes: a tile's records lie in chunk order, so with chunk = workgroup index
// the records that share a 64-byte line would come from eight different L2s, each of which writes its part of
// the line back on its own.  Dealt out by xcd_contiguous_index, neighbours in memory meet in one L2.
__device__ __forceinline__ int chunk_of_workgroup(int b, int n) { return (int)xcd_contiguous_index(b, n); }

// 1a. Per Gaussian the number of tiles it touches (rasterizer_impl.cu:264-288), per workgroup the number of
// instances of every tile.  The workgroup's Gaussians are a contiguous chunk; the scatter walks the same chunk.
__global__ void __launch_bounds__(BK_THREADS)
bucket_count_kernel(int P, int per_block, uint32_t gx, uint32_t gy, const int* __restrict__ radii,
                    const float2* __restrict__ means2D, const uint8_t* __restrict__ compute_locally,
                    uint32_t* __restrict__ tiles_touched, uint32_t* __restrict__ table,
                    uint32_t* __restrict__ block_sums, int* __restrict__ zero_per_gaussian) {
  extern __shared__ uint32_t s_hist[];
  __shared__ uint32_t s_sum[BK_THREADS / GS_WAVE];
  __shared__ uint32_t s_heads[BK_THREADS];
  uint32_t my_sum = 0;  // tiles touched by this thread's Gaussians
  const uint32_t T = gx * gy;
  uint8_t* s_local = reinterpret_cast<uint8_t*>(s_hist + T);  // the tile mask, read once per visited tile
  int masked = 0;
  for (uint32_t t = threadIdx.x; t < T; t += BK_THREADS) {
    s_hist[t] = 0u;
    const uint8_t c = compute_locally[t];
    s_local[t] = c;
    masked |= c == 0 ? 1 : 0;
  }
  // (also the barrier behind the loop) without a tile mask the rectangles are walked with the work spread evenly
  const bool all_local = __syncthreads_or(masked) == 0;
  lds_word* heads = (lds_word*)s_heads + (threadIdx.x / GS_WAVE) * GS_WAVE;
  const int chunk = chunk_of_workgroup(blockIdx.x, gridDim.x);
  const int first = chunk * per_block;
  const int last = first + per_block < P ? first + per_block : P;
  // four Gaussians per round: their loads go out together, then each is walked (the loop bounds are the same
  // for every thread of the workgroup, because the walk is a wave-wide operation)
  struct None { uint32_t unused; } none = {0u};
  for (int base = first; base < last; base += BK_BATCH * BK_THREADS) {
    int r[BK_BATCH];
    float2 p[BK_BATCH];
#pragma unroll
    for (int q = 0; q < BK_BATCH; q++) {
      const int i = base + (int)threadIdx.x + q * BK_THREADS;
      r[q] = i < last ? radii[i] : 0;
      p[q] = i < last ? means2D[i] : make_float2(0.0f, 0.0f);
    }
#pragma unroll
    for (int q = 0; q < BK_BATCH; q++) {
      const int i = base + (int)threadIdx.x + q * BK_THREADS;
      const bool live = i < last && r[q] > 0;
      const Rect rc = live ? get_rect(p[q].x, p[q].y, r[q], gx, gy) : Rect{0u, 0u, 0u, 0u};
      const uint32_t cnt =
          all_local ? walk_wave_rects_flat(live, rc, gx, none, heads,
                                           [&](const None&, uint32_t tile, uint32_t) { atomicAdd(&s_hist[tile], 1u); })
                    : walk_wave_rects(
                          live, rc, gx, none, [&](uint32_t tile) { return s_local[tile] != 0; },
                          [&](const None&, uint32_t tile, uint32_t) { atomicAdd(&s_hist[tile], 1u); });
      if (i < last) {
        tiles_touched[i] = cnt;
        my_sum += cnt;
        // an array of one word per Gaussian that the caller wants cleared on the way (saves a launch)
        if (zero_per_gaussian != nullptr) zero_per_gaussian[i] = 0;
      }
    }
  }
#pragma unroll
  for (int d = GS_WAVE / 2; d >= 1; d >>= 1) my_sum += __shfl_xor(my_sum, d, GS_WAVE);
  if ((threadIdx.x & (GS_WAVE - 1)) == 0) s_sum[threadIdx.x / GS_WAVE] = my_sum;
  __syncthreads();
  uint32_t* row = table + (size_t)chunk * T;
  for (uint32_t t = threadIdx.x; t < T; t += BK_THREADS) row[t] = s_hist[t];
  // the workgroup's share of the prefix sum over the Gaussians (the scatter kernel finishes it)
  if (threadIdx.x == 0) {
    uint32_t all = 0;
    for (int w = 0; w < BK_THREADS / GS_WAVE; w++) all += s_sum[w];
    block_sums[chunk] = all;
  }
}

// 1b. Per tile: the workgroups' counts become exclusive prefixes in place, their sum goes to totals.  A workgroup
// takes 32 tiles (one 128-byte row segment) by 8 runs of consecutive workgroup rows; a thread holds its run in
// registers, the runs' sums meet in LDS.
constexpr int COL_TILES = 32, COL_RUNS = 8, COL_RUN_MAX = BK_MAX_BLOCKS / COL_RUNS;
__global__ void __launch_bounds__(COL_TILES * COL_RUNS)
bucket_columns_kernel(int nblocks, uint32_t T, uint32_t* __restrict__ table, uint32_t* __restrict__ totals) {
  __shared__ uint32_t s_sum[COL_RUNS][COL_TILES];
  const int tx = threadIdx.x % COL_TILES, run = threadIdx.x / COL_TILES;
  const uint32_t t = blockIdx.x * COL_TILES + tx;
  const int len = (nblocks + COL_RUNS - 1) / COL_RUNS;  // <= COL_RUN_MAX
  const int b0 = run * len;
  uint32_t c[COL_RUN_MAX];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < COL_RUN_MAX; k++) {
    const int b = b0 + k;
    c[k] = (k < len && b < nblocks && t < T) ? table[(size_t)b * T + t] : 0u;
    sum += c[k];
  }
  s_sum[run][tx] = sum;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int r = 0; r < COL_RUNS; r++) {
    const uint32_t v = s_sum[r][tx];
    if (r < run) before += v;
    all += v;
  }
  if (t >= T) return;
#pragma unroll
  for (int k = 0; k < COL_RUN_MAX; k++) {
    const int b = b0 + k;
    if (k < len && b < nblocks) table[(size_t)b * T + t] = before;
    before += c[k];
  }
  if (run == 0) totals[t] = all;
}

__device__ __forceinline__ uint32_t wave_inclusive_scan_u32(uint32_t v, int lane) {
#pragma unroll
  for (int d = 1; d < GS_WAVE; d <<= 1) {
    const uint32_t o = __shfl_up(v, d, GS_WAVE);
    if (lane >= d) v += o;
  }
  return v;
}

// 1c. One workgroup: exclusive prefix of the tile totals = the tile ranges (rasterizer_impl.cu:122-144 leaves
// (0, 0) for a tile without instances).  Tiles whose lists are too long for the register sort are entered in two
// lists for the radix sort's kernels: lists of more than small_limit and at most mid_limit records ascending from
// tile_lists[0], longer ones descending from tile_lists[T - 1]; tile_lists[T] = (number of the longer ones << 16
// | number of the others) (T is at most 30000).  The lists beyond block_limit records, which are split before they
// are sorted, are entered a second time in a list of their own: their number in tile_lists[T + 1], the tiles ascending from
// tile_lists[T + 3] (tile_lists[T + 2]: see split_list).  The longest list, tile_lists[T] and then the number of instances are
// stored where the host can read them (host_words[1], [2] and [0]; the host polls word 0, so it is written last).
// The other workgroups of the launch, if there are any, clear the caller's arrays: one workgroup leaves the chip idle for 6 us,
// in which a fill of its own for each of two images of together 24 MB would take 11 (`cleared`).
__global__ void __launch_bounds__(1024)
bucket_ranges_kernel(uint32_t T, uint32_t small_limit, uint32_t mid_limit, uint32_t block_limit,
                     const uint32_t* __restrict__ totals,
                     uint32_t* __restrict__ ranges, uint32_t* __restrict__ tile_lists,
                     uint32_t* __restrict__ block_sums, int nblocks, uint32_t* __restrict__ host_words,
                     uint32_t cap_instances, uint32_t cap_longest, uint32_t* __restrict__ fits_word,
                     uint32_t* __restrict__ clear_word, ClearedArrays cleared) {
  if (blockIdx.x != 0) {
    // (whole 16-byte words, dealt out; the first of these workgroups has what is left of an array)
    const uint32_t first = (blockIdx.x - 1u) * 1024u + threadIdx.x, all = (gridDim.x - 1u) * 1024u;
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint64_t words = cleared.floats[k] / 4;
      float4* const to = reinterpret_cast<float4*>(cleared.data[k]);
      for (uint64_t i = first; i < words; i += all) to[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (first < cleared.floats[k] % 4) cleared.data[k][4 * words + first] = 0.f;
    }
    return;
  }
  constexpr int ITEMS = 4;  // consecutive tiles per thread: the usual grids (up to 4096 tiles) take one round
  __shared__ uint32_t s_wave[16], s_wave_class[16], s_wave_split[16], s_max[16];
  __shared__ double s_exact[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  {
    // the counting workgroups' sums of tiles touched (at most BK_MAX_BLOCKS <= 1024 of them) become exclusive
    // prefixes in place
    const uint32_t b = (int)threadIdx.x < nblocks ? block_sums[threadIdx.x] : 0u;
    const uint32_t inc = wave_inclusive_scan_u32(b, lane);
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t base = 0;
#pragma unroll
    for (int w = 0; w < 16; w++)
      if (w < wave) base += s_wave[w];
    if ((int)threadIdx.x < nblocks) block_sums[threadIdx.x] = base + inc - b;
    __syncthreads();
  }
  uint32_t carry = 0, carry_class = 0, carry_split = 0, longest = 0;
  double exact = 0.0;  // the number of instances without the 32-bit wrap-around of the prefix sums
  for (uint32_t start = 0; start < T; start += 1024 * ITEMS) {
    const uint32_t t0 = start + threadIdx.x * ITEMS;
    uint32_t v[ITEMS], c[ITEMS], sum = 0, sum_class = 0, sum_split = 0;
#pragma unroll
    for (int q = 0; q < ITEMS; q++) v[q] = t0 + q < T ? totals[t0 + q] : 0u;
#pragma unroll
    for (int q = 0; q < ITEMS; q++) {
      c[q] = v[q] > mid_limit ? 0x10000u : (v[q] > small_limit ? 1u : 0u);
      sum_split += v[q] > block_limit ? 1u : 0u;
      longest = v[q] > longest ? v[q] : longest;
      exact += (double)v[q];
      sum += v[q];
      sum_class += c[q];
    }
    const uint32_t inc = wave_inclusive_scan_u32(sum, lane);
    // (a wave without a long list, the usual case, has nothing to scan)
    const uint32_t inc_class = __ballot(sum_class != 0u) != 0ull ? wave_inclusive_scan_u32(sum_class, lane) : 0u;
    const uint32_t inc_split = __ballot(sum_split != 0u) != 0ull ? wave_inclusive_scan_u32(sum_split, lane) : 0u;
    if (lane == 63) {
      s_wave[wave] = inc;
      s_wave_class[wave] = inc_class;
      s_wave_split[wave] = inc_split;
    }
    __syncthreads();
    uint32_t base = 0, all = 0, base_class = 0, all_class = 0, base_split = 0, all_split = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) {
      const uint32_t s = s_wave[w], sc = s_wave_class[w], ss = s_wave_split[w];
      if (w < wave) {
        base += s;
        base_class += sc;
        base_split += ss;
      }
      all += s;
      all_class += sc;
      all_split += ss;
    }
    __syncthreads();
    uint32_t begin = carry + base + inc - sum, begin_class = carry_class + base_class + inc_class - sum_class;
    uint32_t begin_split = carry_split + base_split + inc_split - sum_split;
#pragma unroll
    for (int q = 0; q < ITEMS; q++) {
      if (t0 + q < T) {
        ranges[2 * (t0 + q)] = v[q] ? begin : 0u;
        ranges[2 * (t0 + q) + 1] = v[q] ? begin + v[q] : 0u;
        if (c[q] == 1u) tile_lists[begin_class & 0xFFFFu] = t0 + q;
        if (c[q] == 0x10000u) tile_lists[T - 1u - (begin_class >> 16)] = t0 + q;
        if (v[q] > block_limit) tile_lists[T + 3u + begin_split] = t0 + q;
      }
      begin += v[q];
      begin_class += c[q];
      begin_split += v[q] > block_limit ? 1u : 0u;
    }
    carry += all;
    carry_class += all_class;
    carry_split += all_split;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const uint32_t o = __shfl_xor(longest, d, GS_WAVE);
    longest = o > longest ? o : longest;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) exact += __shfl_xor(exact, d, GS_WAVE);
  if (lane == 0) {
    s_max[wave] = longest;
    s_exact[wave] = exact;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = 0;
    double all = 0.0;
    for (int w = 0; w < 16; w++) {
      m = s_max[w] > m ? s_max[w] : m;
      all += s_exact[w];
    }
    tile_lists[T] = carry_class;
    tile_lists[T + 1u] = carry_split;
    tile_lists[T + 2u] = 0u;
    if (clear_word != nullptr) clear_word[0] = clear_word[1] = 0u;  // (two words the caller wants cleared: saves a launch)
    // more instances than 32-bit positions can address: the host must not go on with the wrapped count
    const uint32_t reported = all > (double)GS_MAX_INSTANCES ? GS_TOO_MANY_INSTANCES : carry;
    // Kernels launched ahead of the host's decision (buffers sized from the caller's expectation) look at this
    // word and do nothing unless the view fits what they were launched for.
    *fits_word = (reported <= cap_instances && m <= cap_longest) ? 1u : 0u;
    __hip_atomic_store(host_words + 1, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(host_words + 2, carry_class, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(host_words, reported, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// 1d. Every instance goes to its tile's segment: segment start (ranges) + instances of earlier workgroups
// (table) + a place among this workgroup's own, handed out by an LDS counter.  The record is one 16-byte store
// (Gaussian, emission index, depth bits, 0) (rasterizer_impl.cu:74-117 writes the same instances in emission
// order); the per-tile sorts read the depth bits and look the other two up once a record's place is known, inside
// the tile's own segment.  The kernel also finishes the prefix sum
// over the Gaussians' tile counts (rasterizer_impl.cu:648) for its own chunk, which is where the emission
// indices come from: a thread owns four consecutive Gaussians, the workgroup scans the threads' sums, and the
// inclusive sums go to point_offsets on the way (the backward pass reads them).
// fits_word (optional): the kernel was launched before the host knew the instance count; it does nothing unless
// bucket_ranges_kernel found that the view fits the buffers it was launched with.
__global__ void __launch_bounds__(BK_THREADS)
bucket_scatter_kernel(int P, int per_block, uint32_t gx, uint32_t gy, const float2* __restrict__ means2D,
                      const float* __restrict__ depths, const uint32_t* __restrict__ tiles_touched,
                      const uint32_t* __restrict__ block_prefix, uint32_t* __restrict__ point_offsets,
                      const int* __restrict__ radii, const uint8_t* __restrict__ compute_locally,
                      const uint32_t* __restrict__ table, const uint32_t* __restrict__ ranges,
                      TileRecord* __restrict__ records, const uint32_t* __restrict__ fits_word,
                      int vector_loads) {
  extern __shared__ uint32_t s_next[];
  __shared__ uint32_t s_wave[BK_THREADS / GS_WAVE];
  __shared__ uint32_t s_heads[BK_THREADS];
  if (fits_word != nullptr && *fits_word == 0u) return;
  const uint32_t T = gx * gy;
  uint8_t* s_local = reinterpret_cast<uint8_t*>(s_next + T);
  const int chunk = chunk_of_workgroup(blockIdx.x, gridDim.x);
  const uint32_t* row = table + (size_t)chunk * T;
  int masked = 0;
  for (uint32_t t = threadIdx.x; t < T; t += BK_THREADS) {
    s_next[t] = ranges[2 * t] + row[t];
    const uint8_t c = compute_locally[t];
    s_local[t] = c;
    masked |= c == 0 ? 1 : 0;
  }
  const bool all_local = __syncthreads_or(masked) == 0;  // (as in the counting kernel; also the barrier)
  const int lane = threadIdx.x & (GS_WAVE - 1), wave = threadIdx.x / GS_WAVE;
  lds_word* heads = (lds_word*)s_heads + wave * GS_WAVE;
  const int first = chunk * per_block;
  const int last = first + per_block < P ? first + per_block : P;
  struct Owner { uint32_t first, depth_bits, id; };
  uint32_t carry = block_prefix[chunk];  // instances of the Gaussians before this round
  for (int base = first; base < last; base += BK_BATCH * BK_THREADS) {
    const int i0 = base + (int)threadIdx.x * BK_BATCH;
    int r[BK_BATCH];
    float2 p[BK_BATCH];
    uint32_t tt[BK_BATCH], dbits[BK_BATCH], sum = 0;
    static_assert(BK_BATCH == 4, "a thread's Gaussians are loaded as four-word vectors");
    const bool whole = vector_loads != 0 && i0 + BK_BATCH <= last;
    if (whole) {
      // (i0 is a multiple of four and the host found every array 16-byte aligned: 16-byte loads)
      const int4 rv = *reinterpret_cast<const int4*>(radii + i0);
      const uint4 tv = *reinterpret_cast<const uint4*>(tiles_touched + i0);
      const uint4 dv = *reinterpret_cast<const uint4*>(depths + i0);
      const float4 m01 = *reinterpret_cast<const float4*>(means2D + i0);
      const float4 m23 = *reinterpret_cast<const float4*>(means2D + i0 + 2);
      r[0] = rv.x; r[1] = rv.y; r[2] = rv.z; r[3] = rv.w;
      tt[0] = tv.x; tt[1] = tv.y; tt[2] = tv.z; tt[3] = tv.w;
      dbits[0] = dv.x; dbits[1] = dv.y; dbits[2] = dv.z; dbits[3] = dv.w;
      p[0] = make_float2(m01.x, m01.y); p[1] = make_float2(m01.z, m01.w);
      p[2] = make_float2(m23.x, m23.y); p[3] = make_float2(m23.z, m23.w);
    } else {
#pragma unroll
      for (int q = 0; q < BK_BATCH; q++) {
        const int i = i0 + q;
        r[q] = i < last ? radii[i] : 0;
        p[q] = i < last ? means2D[i] : make_float2(0.0f, 0.0f);
        dbits[q] = i < last ? __float_as_uint(depths[i]) : 0u;
        tt[q] = i < last ? tiles_touched[i] : 0u;
      }
    }
#pragma unroll
    for (int q = 0; q < BK_BATCH; q++) sum += tt[q];
    const uint32_t inc = wave_inclusive_scan_u32(sum, lane);
    if (lane == GS_WAVE - 1) s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < BK_THREADS / GS_WAVE; w++) {
      const uint32_t v = s_wave[w];
      if (w < wave) before += v;
      all += v;
    }
    __syncthreads();
    uint32_t run = carry + before + inc - sum;  // emission index of this thread's first instance
    carry += all;
#pragma unroll
    for (int q = 0; q < BK_BATCH; q++) {
      const int i = i0 + q;
      const bool live = i < last && r[q] > 0;
      const Rect rc = live ? get_rect(p[q].x, p[q].y, r[q], gx, gy) : Rect{0u, 0u, 0u, 0u};
      const Owner mine = {run, dbits[q], (uint32_t)i};
      run += tt[q];
      tt[q] = run;  // from here on: the inclusive sum
      const auto emit = [&](const Owner& o, uint32_t tile, uint32_t rank) {
        const uint32_t e = o.first + rank;
        const uint32_t pos = atomicAdd(&s_next[tile], 1u);
        records[pos] = make_uint4(o.id, e, o.depth_bits, 0u);
      };
      if (all_local) walk_wave_rects_flat(live, rc, gx, mine, heads, emit);
      else walk_wave_rects(live, rc, gx, mine, [&](uint32_t tile) { return s_local[tile] != 0; }, emit);
    }
    if (whole) {
      *reinterpret_cast<uint4*>(point_offsets + i0) = make_uint4(tt[0], tt[1], tt[2], tt[3]);
    } else {
#pragma unroll
      for (int q = 0; q < BK_BATCH; q++)
        if (i0 + q < last) point_offsets[i0 + q] = tt[q];
    }
  }
}

// 1d'. The same scatter for a view in which a workgroup walks its chunk of Gaussians in one round (at most
// BK_BATCH * BK_THREADS of them) and its instances fit the LDS: the records are staged in LDS, ordered by tile (the
// counting kernels' table gives the workgroup's own count per tile: the next workgroup's prefix minus its own), and
// written out tile by tile, so that the records a workgroup adds to one tile's segment leave as one run, all
// workgroups at about the same time.  Every 16-byte record written on its own costs the memory a 64-byte write;
// runs that meet in the L2 cost their bytes.  A workgroup with more than `cap` instances stores directly, as the
// kernel above does.
// A thread owns ITEMS consecutive Gaussians, as few as the chunk allows: it walks them one after the other.
// Dynamic LDS: 9 bytes per tile and 12 bytes per staged record.
template <int ITEMS>
__global__ void __launch_bounds__(BK_THREADS)
bucket_scatter_staged_kernel(int P, int per_block, int nblocks, uint32_t gx, uint32_t gy,
                             const float2* __restrict__ means2D, const float* __restrict__ depths,
                             const uint32_t* __restrict__ tiles_touched, const uint32_t* __restrict__ block_prefix,
                             uint32_t* __restrict__ point_offsets, const int* __restrict__ radii,
                             const uint8_t* __restrict__ compute_locally, const uint32_t* __restrict__ table,
                             const uint32_t* __restrict__ totals, const uint32_t* __restrict__ ranges,
                             TileRecord* __restrict__ records, const uint32_t* __restrict__ fits_word,
                             int vector_loads, uint32_t cap) {
  extern __shared__ uint32_t s_mem[];
  __shared__ uint32_t s_wave[BK_THREADS / GS_WAVE], s_wave_tiles[BK_THREADS / GS_WAVE];
  __shared__ uint32_t s_heads[BK_THREADS];
  if (fits_word != nullptr && *fits_word == 0u) return;
  const uint32_t T = gx * gy;
  uint32_t* s_next = s_mem;         // [T] where the workgroup's first record of a tile goes in memory
  uint32_t* s_cursor = s_mem + T;   // [T] next free place of a tile: in the staging arrays, or in memory
  uint32_t* stage_g = s_cursor + T; // [cap] x 3: Gaussian, emission index, depth bits
  uint32_t* stage_e = stage_g + cap;
  uint32_t* stage_z = stage_e + cap;
  uint8_t* s_local = reinterpret_cast<uint8_t*>(stage_z + cap);
  const int lane = threadIdx.x & (GS_WAVE - 1), wave = threadIdx.x / GS_WAVE;
  const int chunk = chunk_of_workgroup(blockIdx.x, gridDim.x);
  const uint32_t* row = table + (size_t)chunk * T;
  const uint32_t* next_row = chunk + 1 < nblocks ? table + (size_t)(chunk + 1) * T : totals;
  const int first = chunk * per_block;
  const int last = first + per_block < P ? first + per_block : P;
  // (the workgroup's Gaussians are asked for first: their latency passes behind the set-up of the tiles)
  const int i0 = first + (int)threadIdx.x * ITEMS;
  int r[ITEMS];
  float2 p[ITEMS];
  uint32_t tt[ITEMS], dbits[ITEMS], sum = 0;
  // (four are loaded as four-word vectors)
  const bool whole = ITEMS == 4 && vector_loads != 0 && i0 + ITEMS <= last;
  if constexpr (ITEMS == 4) {
    if (whole) {
      const int4 rv = *reinterpret_cast<const int4*>(radii + i0);
      const uint4 tv = *reinterpret_cast<const uint4*>(tiles_touched + i0);
      const uint4 dv = *reinterpret_cast<const uint4*>(depths + i0);
      const float4 m01 = *reinterpret_cast<const float4*>(means2D + i0);
      const float4 m23 = *reinterpret_cast<const float4*>(means2D + i0 + 2);
      r[0] = rv.x; r[1] = rv.y; r[2] = rv.z; r[3] = rv.w;
      tt[0] = tv.x; tt[1] = tv.y; tt[2] = tv.z; tt[3] = tv.w;
      dbits[0] = dv.x; dbits[1] = dv.y; dbits[2] = dv.z; dbits[3] = dv.w;
      p[0] = make_float2(m01.x, m01.y); p[1] = make_float2(m01.z, m01.w);
      p[2] = make_float2(m23.x, m23.y); p[3] = make_float2(m23.z, m23.w);
    }
  }
  if (!whole) {
#pragma unroll
    for (int q = 0; q < ITEMS; q++) {
      const int i = i0 + q;
      r[q] = i < last ? radii[i] : 0;
      p[q] = i < last ? means2D[i] : make_float2(0.0f, 0.0f);
      dbits[q] = i < last ? __float_as_uint(depths[i]) : 0u;
      tt[q] = i < last ? tiles_touched[i] : 0u;
    }
  }
  int masked = 0;
  constexpr int TILES_AHEAD = 4;  // tiles a thread has in flight: a usual grid is set up with one memory latency
  for (uint32_t t0 = threadIdx.x; t0 < T; t0 += TILES_AHEAD * BK_THREADS) {
    uint32_t before[TILES_AHEAD], upto[TILES_AHEAD], begin[TILES_AHEAD];
    uint8_t c[TILES_AHEAD];
#pragma unroll
    for (int u = 0; u < TILES_AHEAD; u++) {
      const uint32_t t = t0 + (uint32_t)u * BK_THREADS;
      before[u] = t < T ? row[t] : 0u;
      upto[u] = t < T ? next_row[t] : 0u;
      begin[u] = t < T ? ranges[2 * t] : 0u;
      c[u] = t < T ? compute_locally[t] : (uint8_t)1;
    }
#pragma unroll
    for (int u = 0; u < TILES_AHEAD; u++) {
      const uint32_t t = t0 + (uint32_t)u * BK_THREADS;
      if (t < T) {
        s_next[t] = begin[u] + before[u];
        s_cursor[t] = upto[u] - before[u];  // the workgroup's own instances of the tile
        s_local[t] = c[u];
        masked |= c[u] == 0 ? 1 : 0;
      }
    }
  }
  const bool all_local = __syncthreads_or(masked) == 0;
  // exclusive prefix of the counts over the tiles, in place: a thread owns `per` consecutive tiles
  const uint32_t per = (T + BK_THREADS - 1) / BK_THREADS, t_first = threadIdx.x * per;
  uint32_t own = 0;
  for (uint32_t k = 0; k < per; k++)
    if (t_first + k < T) own += s_cursor[t_first + k];
  const uint32_t own_inc = wave_inclusive_scan_u32(own, lane);
  // (the prefix sum over the Gaussians' tile counts shares the barrier)
#pragma unroll
  for (int q = 0; q < ITEMS; q++) sum += tt[q];
  const uint32_t inc = wave_inclusive_scan_u32(sum, lane);
  if (lane == GS_WAVE - 1) {
    s_wave_tiles[wave] = own_inc;
    s_wave[wave] = inc;
  }
  __syncthreads();
  uint32_t tiles_before = 0, total = 0, before = 0;
#pragma unroll
  for (int w = 0; w < BK_THREADS / GS_WAVE; w++) {
    const uint32_t v = s_wave_tiles[w];
    if (w < wave) {
      tiles_before += v;
      before += s_wave[w];
    }
    total += v;
  }
  const bool staged = total <= cap;  // (the same for the whole workgroup)
  {
    uint32_t run = tiles_before + own_inc - own;
    for (uint32_t k = 0; k < per; k++)
      if (t_first + k < T) {
        const uint32_t v = s_cursor[t_first + k];
        s_cursor[t_first + k] = staged ? run : s_next[t_first + k];
        run += v;
      }
  }
  __syncthreads();
  lds_word* heads = (lds_word*)s_heads + wave * GS_WAVE;
  struct Owner { uint32_t first, depth_bits, id; };
  {
    uint32_t run = block_prefix[chunk] + before + inc - sum;  // emission index of this thread's first instance
#pragma unroll
    for (int q = 0; q < ITEMS; q++) {
      const int i = i0 + q;
      const bool live = i < last && r[q] > 0;
      const Rect rc = live ? get_rect(p[q].x, p[q].y, r[q], gx, gy) : Rect{0u, 0u, 0u, 0u};
      const Owner mine = {run, dbits[q], (uint32_t)i};
      run += tt[q];
      tt[q] = run;  // from here on: the inclusive sum
      const auto emit = [&](const Owner& o, uint32_t tile, uint32_t rank) {
        const uint32_t e = o.first + rank;
        const uint32_t pos = atomicAdd(&s_cursor[tile], 1u);
        if (staged) {
          stage_g[pos] = o.id;
          stage_e[pos] = e;
          stage_z[pos] = o.depth_bits;
        } else {
          records[pos] = make_uint4(o.id, e, o.depth_bits, 0u);
        }
      };
      if (all_local) walk_wave_rects_flat(live, rc, gx, mine, heads, emit);
      else walk_wave_rects(live, rc, gx, mine, [&](uint32_t tile) { return s_local[tile] != 0; }, emit);
    }
    if (whole) {
      *reinterpret_cast<uint4*>(point_offsets + i0) = make_uint4(tt[0], tt[ITEMS > 1 ? 1 : 0], tt[ITEMS > 2 ? 2 : 0],
                                                                 tt[ITEMS > 3 ? 3 : 0]);
    } else {
#pragma unroll
      for (int q = 0; q < ITEMS; q++)
        if (i0 + q < last) point_offsets[i0 + q] = tt[q];
    }
  }
  if (!staged) return;
  __syncthreads();
  // every tile's run: staged at [cursor of the tile before, cursor of the tile), to memory from s_next on
  for (uint32_t t = threadIdx.x; t < T; t += BK_THREADS) {
    const uint32_t lo = t > 0u ? s_cursor[t - 1u] : 0u, hi = s_cursor[t];
    TileRecord* dst = records + s_next[t];
    for (uint32_t k = lo; k < hi; k++) dst[k - lo] = make_uint4(stage_g[k], stage_e[k], stage_z[k], 0u);
  }
}

// 2. Per-tile sort, register variant: one workgroup of W waves per tile (4 for lists of up to 256 records, 8 up
// to 4096).  A wave holds 64 E keys, key i = r * 64 + lane in register r of its lane, and the waves hold
// consecutive runs of 64 E, so a list of up to 64 E W records is sorted with E = 1 .. 8.  In the bitonic network
// a step pairs i with i ^ j:
//   j < 64        the partner sits in another lane, same register: one cross-lane read, keep the smaller or larger;
//   64 <= j < 64E the partner sits in another register of the same lane: no data moves at all;
//   j >= 64 E     the partner sits in another wave: one exchange through LDS (3 such steps in a whole sort with
//                 4 waves, 6 with 8).
// A tile takes as long as the instruction stream of one of its waves, and the kernel as long as its longest tiles:
// a long list is spread over more waves rather than more registers per lane (eight waves with four records per
// lane for 2048 records, not four with eight).  Lists of 2049 to 4096 records take eight, so that a view without longer
// ones needs no further launch and the others have these lists under way beside the shorter: with a radix sort in a
// launch of its own for them (tile_radix.hip, which is left with what a caller's options put between the limits) the two
// kernels took 25.0 + 27.8 us for 20 M Gaussians from 600 m, 22.8 + 25.8 for 4 M from the air, 21.2 + 30.6 and 28.5 + 30.5 in
// two views at street level and, with hardly such a list, 22.6 + 4.7 for 1 M; this one takes 43.2, 45.3, 56.8 and 56.8, and
// 24.1.
//
// The key is one 32-bit word: (depth bits - smallest depth bits of the list) >> shift in the high bits, the
// record's place in the unsorted segment in the low log2(64 E W) bits; shift is what it takes to fit the list's
// range of depth bits (0 when it fits as it is).  A step then costs two vector instructions per key (a cross-lane
// move and a median with 0 or all ones, or a minimum and a maximum that each read across lanes).  With all runs of a
// stage sorted upwards nothing depends on a run's direction any more but the complements at the start of the stage, and
// with the steps inside a wave unrolled the chains of a lane's registers overlap; with a compare, a scalar mask and a
// select per step, and the directions in masks, the kernel took 27.9 us at 1 M Gaussians, 1152 x 864 and 29.0 us at 4 M,
// now 22.0 and 22.8; 13.2 and 11.4 us at 300 k, 1237 x 822.  Keys whose depths agree in the bits kept end up next
// to each other in the order of their places; the last step (emit_list_entry) puts every such run into its true
// order, by all depth bits and then the emission index, exactly as it does for runs of equal depth bits.  Depths
// inside a tile are spread over the view's range, so with the 21 to 24 bits kept runs are as rare as before.

// A pair's smaller key where `keep` is 0, its larger one where it is all ones: the median of the three.  (The idle slots
// are for a cross-lane instruction that reads the result next: the compiler does not look into these statements for what
// such an instruction has to wait for.)
__device__ __forceinline__ uint32_t keep_pair(uint32_t a, uint32_t b, uint32_t keep) {
  uint32_t r;
  asm("v_med3_u32 %0, %1, %2, %3\n\ts_nop 1" : "=v"(r) : "v"(a), "v"(b), "v"(keep));
  return r;
}

// One step of the network with the partner in lane ^ J: the lanes whose bit J is clear keep the smaller key, the others
// the larger (upper: all ones there).  A variable-distance __shfl_xor is a ds_bpermute, whose latency every one of the
// sort's dependent steps would wait for.  All 64 lanes must be active.
//   J = 1, 2: a DPP move inside the quad and a median;
//   J = 4, 8: a minimum and a maximum whose DPP operands come from the other side, each for the quads of a row that take
//     its result (a DPP operand written by the preceding vector instruction needs two idle issue slots);
//   J = 16, 32: v_permlane16_swap / v_permlane32_swap exchange the odd rows (the upper half) of their first operand with
//     the even rows (the lower half) of the second: from two copies of x they leave the lower element of every pair in
//     all lanes of the first result and the upper element in the second.
template <int J>
__device__ __forceinline__ uint32_t lane_step(uint32_t x, uint32_t upper) {
  static_assert(J == 1 || J == 2 || J == 4 || J == 8 || J == 16 || J == 32, "a distance inside the wave");
  uint32_t r;
  if constexpr (J == 1) {
    asm("s_nop 1\n\t"
        "v_mov_b32_dpp %0, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_med3_u32 %0, %1, %0, %2"
        : "=&v"(r)
        : "v"(x), "v"(upper));
  } else if constexpr (J == 2) {
    asm("s_nop 1\n\t"
        "v_mov_b32_dpp %0, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_med3_u32 %0, %1, %0, %2"
        : "=&v"(r)
        : "v"(x), "v"(upper));
  } else if constexpr (J == 4) {
    asm("s_nop 1\n\t"
        "v_min_u32_dpp %0, %1, %1 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_max_u32_dpp %0, %1, %1 row_shr:4 row_mask:0xf bank_mask:0xa"
        : "=&v"(r)
        : "v"(x));
  } else if constexpr (J == 8) {
    asm("s_nop 1\n\t"
        "v_min_u32_dpp %0, %1, %1 row_shl:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_max_u32_dpp %0, %1, %1 row_shr:8 row_mask:0xf bank_mask:0xc"
        : "=&v"(r)
        : "v"(x));
  } else if constexpr (J == 16) {
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    r = keep_pair(p[0], p[1], upper);
  } else {
    const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    r = keep_pair(p[0], p[1], upper);
  }
  return r;
}

// The steps at distances J, J / 2 .. 1 of every register: the registers' chains of steps are independent of each other.
template <int J, int E>
__device__ __forceinline__ void lane_steps(uint32_t (&v)[E], const uint32_t (&upper)[6]) {
#pragma unroll
  for (int r = 0; r < E; r++) v[r] = lane_step<J>(v[r], upper[__builtin_ctz(J)]);
  if constexpr (J > 1) lane_steps<J / 2>(v, upper);
}

// Element i = (row << 6 | lane) is sorted upwards in the stage of runs of k where (i & k) == 0, which is a property of the
// lane below k = 64 and of the register (and wave) from there on.  Every step sorts upwards: the keys of the runs that a
// stage sorts downwards are complemented before it.  flipped: all ones where a key is held complemented.
template <int E>
__device__ __forceinline__ void turn_runs(uint32_t (&v)[E], uint32_t (&flipped)[E], uint32_t row0, uint32_t lane, uint32_t k) {
#pragma unroll
  for (int r = 0; r < E; r++) {
    const uint32_t flip = ((((row0 + (uint32_t)r) << 6) | lane) & k) != 0u ? ~0u : 0u;
    v[r] ^= flipped[r] ^ flip;
    flipped[r] = flip;
  }
}

// The stages of runs of K .. 32: all their pairs lie in one register.
template <int K, int E>
__device__ __forceinline__ void lane_stages(uint32_t (&v)[E], uint32_t (&flipped)[E], uint32_t row0, uint32_t lane,
                                            const uint32_t (&upper)[6]) {
  turn_runs(v, flipped, row0, lane, K);
  lane_steps<K / 2>(v, upper);
  if constexpr (K < 32) lane_stages<2 * K>(v, flipped, row0, lane, upper);
}

template <int E, int W>
__device__ __forceinline__ void register_sort(uint32_t (&v)[E], uint32_t wave, uint32_t lane, uint32_t* s_x) {
  constexpr uint32_t M = 64u * E * W;
  const uint32_t row0 = wave * E;
  uint32_t upper[6];
#pragma unroll
  for (int b = 0; b < 6; b++) upper[b] = (lane >> b & 1u) != 0u ? ~0u : 0u;
  uint32_t flipped[E];
#pragma unroll
  for (int r = 0; r < E; r++) flipped[r] = 0u;
  lane_stages<2>(v, flipped, row0, lane, upper);
  for (uint32_t k = 64; k <= M; k <<= 1) {
    turn_runs(v, flipped, row0, lane, k);
    for (uint32_t j = k >> 1; j >= 64; j >>= 1) {
      if (j < 64u * E) {
        const uint32_t jr = j >> 6;
#pragma unroll
        for (int b = 1; b < E; b <<= 1) {
          if (jr != (uint32_t)b) continue;
#pragma unroll
          for (int r = 0; r < E; r++) {
            if (r & b) continue;
            const uint32_t x = v[r], y = v[r | b];
            v[r] = x < y ? x : y;
            v[r | b] = x < y ? y : x;
          }
        }
      } else {
        // partner wave = wave ^ jw: everybody posts, everybody reads the partner's post
        const uint32_t jw = j / (64u * E);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; r++) s_x[((wave * E + r) << 6) | lane] = v[r];
        __syncthreads();
        const uint32_t keep = (wave & jw) == 0 ? 0u : ~0u;
#pragma unroll
        for (int r = 0; r < E; r++) v[r] = keep_pair(v[r], s_x[(((wave ^ jw) * E + r) << 6) | lane], keep);
      }
    }
    lane_steps<32>(v, upper);
  }
}

// Sorts the tile's one-word keys and hands every entry to emit_list_entry, which puts runs of keys with the same
// depth field into their order by all depth bits and then emission index.  s_x: at least 64 E W 8-byte words.
template <int E, int W>
__device__ __forceinline__ void register_sort_tile(uint32_t t, uint32_t start, uint32_t n,
                                                   const TileRecord* __restrict__ records,
                                                   uint64_t* __restrict__ keys, uint32_t* __restrict__ emission,
                                                   uint32_t* __restrict__ point_list, uint64_t* s_x) {
  constexpr uint32_t M = 64u * E * W;
  constexpr int PLACE_BITS = M == 256 ? 8 : M == 512 ? 9 : M == 1024 ? 10 : M == 2048 ? 11 : 12;
  static_assert(M == 1u << PLACE_BITS, "a list of 256 to 4096 places");
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t* s_words = reinterpret_cast<uint32_t*>(s_x);
  uint32_t v[E];
  uint32_t lo = 0xFFFFFFFFu, hi = 0u;
#pragma unroll
  for (int r = 0; r < E; r++) {
    const uint32_t i = ((wave * E + r) << 6) | lane;
    v[r] = i < n ? records[start + i].z : 0u;
    if (i < n) {
      lo = v[r] < lo ? v[r] : lo;
      hi = v[r] > hi ? v[r] : hi;
    }
  }
  // smallest and largest depth bits of the list: over the wave by a scan (its last lane holds the result), over
  // the waves through LDS
  lo = ~(uint32_t)__builtin_amdgcn_readlane((int)wave_scan_max(~lo), GS_WAVE - 1);
  hi = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan_max(hi), GS_WAVE - 1);
  if (lane == 0) {
    s_words[wave] = lo;
    s_words[W + wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; w++) {
    const uint32_t a = s_words[w], b = s_words[W + w];
    lo = a < lo ? a : lo;
    hi = b > hi ? b : hi;
  }
  const uint32_t range = hi - lo;  // (n >= 1, so lo <= hi)
  const int range_bits = range != 0u ? 32 - __builtin_clz(range) : 0;
  const uint32_t shift = range_bits + PLACE_BITS > 32 ? (uint32_t)(range_bits + PLACE_BITS - 32) : 0u;
#pragma unroll
  for (int r = 0; r < E; r++) {
    const uint32_t i = ((wave * E + r) << 6) | lane;
    v[r] = i < n ? ((((v[r] - lo) >> shift) << PLACE_BITS) | i) : 0xFFFFFFFFu;
  }
  // (a real key is below the padding's: a key of all ones would be the list's last place, which is padding
  // unless the list fills all M places, and then there is none)
  register_sort<E, W>(v, wave, lane, s_words);  // (starts its first exchange behind a barrier: lo and hi are read)
  uint32_t gaussian[E];
  uint64_t entry[E];
#pragma unroll
  for (int r = 0; r < E; r++) {
    const uint32_t i = ((wave * E + r) << 6) | lane;
    gaussian[r] = 0u;
    entry[r] = 0ull;
    if (i < n) {
      const TileRecord rec = records[start + (v[r] & (M - 1u))];
      gaussian[r] = rec.x;
      entry[r] = ((uint64_t)rec.z << 32) | (uint64_t)rec.y;
    }
  }
  __syncthreads();  // (the sort's last exchange between waves has been read by everybody)
#pragma unroll
  for (int r = 0; r < E; r++) {
    const uint32_t i = ((wave * E + r) << 6) | lane;
    if (i < n) s_x[i] = entry[r];
  }
  __syncthreads();
  const uint64_t* sorted = s_x;
#pragma unroll
  for (int r = 0; r < E; r++) {
    uint32_t i = ((wave * E + r) << 6) | lane;
    asm volatile("" : "+v"(i));  // (the lists' addresses are computed one entry at a time: of all eight at once they spill)
    if (i < n)
      emit_list_entry(t, start, n, i, gaussian[r], [&](uint32_t q) { return sorted[q]; }, keys, emission, point_list,
                      lo, shift);
  }
}

// The order in which the blend kernels take the tiles: by falling length of the lists, in steps of half a power of two.  A
// tile's workgroup works for as long as its list is, and workgroups start in the order of their numbers: taken row by
// row, a street-level view (10 M Gaussians, 1920x1080, lists up to 28 000 entries along the horizon, half way down
// the image) ends with a few long tiles on an idle chip (backward blend 904 -> 716 us, forward 610 -> 564; views from
// the air, whose lists differ less, take the same time either way).  The place inside a class is whatever the LDS counter
// hands out (about ascending): no result depends on it.
// order_word: 1 + the number of tiles that the forward blend splits, which are the first of the order (the rule: see
// GS_LONG_TILE; longest_split is what it depends on).  The two per-tile sums that the four workgroups of such a tile add up
// are cleared here.  s_count: CLASSES + 2 words.
__device__ __forceinline__ void order_tiles(uint32_t T, const uint32_t* __restrict__ ranges, uint32_t* __restrict__ order,
                                            uint32_t* __restrict__ order_word, uint32_t longest_split,
                                            int* __restrict__ n_consider, int* __restrict__ n_contrib, uint32_t* s_count) {
  constexpr int CLASSES = 64;
  auto class_of_length = [](uint32_t n) {  // 0 = the longest lists
    if (n == 0) return CLASSES - 1;
    const int msb = 31 - __clz((int)n);
    return CLASSES - 2 - (2 * msb + (msb > 0 ? (int)((n >> (msb - 1)) & 1u) : 0));
  };
  auto length = [&](uint32_t t) { return ranges[2 * t + 1] - ranges[2 * t]; };
  if (threadIdx.x < CLASSES + 2) s_count[threadIdx.x] = 0u;
  __syncthreads();
  uint32_t entries = 0u, longest = 0u;
  for (uint32_t t = threadIdx.x; t < T; t += blockDim.x) {
    const uint32_t n = length(t);
    entries += n;
    longest = max(longest, n);
    atomicAdd(&s_count[class_of_length(n)], 1u);
  }
#pragma unroll
  for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
    entries += __shfl_xor(entries, d, GS_WAVE);
    longest = max(longest, __shfl_xor(longest, d, GS_WAVE));
  }
  if ((threadIdx.x & (GS_WAVE - 1)) == 0) {
    atomicAdd(&s_count[CLASSES], entries);
    atomicMax(&s_count[CLASSES + 1], longest);
  }
  __syncthreads();
  if (threadIdx.x < CLASSES) {  // (one wave)
    const uint32_t c = s_count[threadIdx.x];
    s_count[threadIdx.x] = wave_inclusive_scan_u32(c, (int)threadIdx.x) - c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t split = 0u;
    if ((uint64_t)s_count[CLASSES + 1] * (GS_BLEND_SLOTS / 2) >= s_count[CLASSES]) {
#pragma unroll
      for (uint32_t from : {GS_LONG_TILE, GS_LONG_TILE / 3 * 4, GS_LONG_TILE * 2}) {
        split = s_count[class_of_length(from) + 1];
        if (split <= GS_LONG_TILES || from >= longest_split) break;
      }
    }
    *order_word = 1u + split;
  }
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < T; t += blockDim.x) {
    order[atomicAdd(&s_count[class_of_length(length(t))], 1u)] = t;
    n_consider[t] = 0;
    n_contrib[t] = 0;
  }
}

// A list of more than `blk` records is split for the radix sort, by depth, into groups that it takes like short lists.  A
// sample of the list gives the groups' bounds, in 256ths of the sample's range of depths, so that a group holds some four
// fifths of blk; what lies outside that range goes to the first and the last group, equal depth bits into one group (the
// sorts' last step sees runs of them whole), and a group beyond blk (many instances within 1/256 of the range) goes block by
// block through memory.  Every wave counts the groups in its part of the list and then moves the part to `parted`.  The
// groups' first places are left in list_words, from `start` on (an array that the blend kernel fills later), their number
// beside the tile in `entry`, the largest of all lists in *most.
// Here, beside the register sort, and not in the radix sort's own workgroups, each of which holds a CU for as long as its
// list is: 20 M Gaussians from 600 m, two views whose longest lists have 69 000 and 43 000 entries, 43 + 491 and 43 + 349 us
// (this kernel and the radix sort) -> 140 + 265 and 133 + 250.  Bound by the memory's traffic, 48 bytes a record.  With 256
// bins, counted and filled by LDS atomics, 177 us of this kernel instead of 137; the moved records through the caches 152,
// four of them in flight a lane instead of eight 165; three workgroups a list, each counting all of it, 198.  Without the
// move, every group's workgroup looking for its entries in the whole list: 43 + 380 us.
// s_words: SPLIT_WORDS words.
constexpr uint32_t SPLIT_BINS = 256, SPLIT_GROUPS = GS_WAVE;  // (a lane for every group)
constexpr uint32_t SPLIT_WAVES = 8;
constexpr uint32_t SPLIT_WORDS = SPLIT_BINS + SPLIT_BINS / 4 + SPLIT_WAVES * SPLIT_GROUPS + 2 * SPLIT_WAVES;
__device__ __forceinline__ void split_list(uint32_t t, uint32_t start, uint32_t n, uint32_t blk,
                                           const TileRecord* __restrict__ records, TileRecord* __restrict__ parted,
                                           uint32_t* __restrict__ list_words, uint32_t* __restrict__ entry,
                                           uint32_t* __restrict__ most, uint32_t* s_words) {
  constexpr uint32_t WAVES = SPLIT_WAVES, THREADS = WAVES * GS_WAVE, SAMPLED = 8, QUARTERS = SPLIT_BINS / GS_WAVE;
  constexpr uint32_t COUNTED = 16, MOVED = 8;  // loads a lane keeps in flight
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  uint32_t* const s_bins = s_words;
  uint8_t* const s_group = reinterpret_cast<uint8_t*>(s_words + SPLIT_BINS);  // a bin's group
  uint32_t* const s_count = s_words + SPLIT_BINS + SPLIT_BINS / 4;            // [WAVES][SPLIT_GROUPS]
  uint32_t* const s_scan = s_count + WAVES * SPLIT_GROUPS;
  const TileRecord* const list = records + start;
  const uint32_t step = n / (SAMPLED * THREADS) + 1u, in_all = (n + step - 1u) / step;
  const uint32_t samples = min(SAMPLED * THREADS, in_all);
  uint32_t z[SAMPLED], lo = 0xFFFFFFFFu, hi = 0u;
#pragma unroll
  for (uint32_t u = 0; u < SAMPLED; u++) z[u] = list[min(u * THREADS + tid, samples - 1u) * step].z;
#pragma unroll
  for (uint32_t u = 0; u < SAMPLED; u++) {
    lo = min(lo, z[u]);
    hi = max(hi, z[u]);
  }
  lo = ~(uint32_t)__builtin_amdgcn_readlane((int)wave_scan_max(~lo), GS_WAVE - 1);
  hi = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan_max(hi), GS_WAVE - 1);
  if (lane == 0u) {
    s_scan[wave] = lo;
    s_scan[WAVES + wave] = hi;
  }
  if (tid < SPLIT_BINS) s_bins[tid] = 0u;
  __syncthreads();
#pragma unroll
  for (uint32_t w = 0; w < WAVES; w++) {
    lo = min(lo, s_scan[w]);
    hi = max(hi, s_scan[WAVES + w]);
  }
  const uint32_t range = hi - lo;
  const int bits = range != 0u ? 32 - __builtin_clz(range) : 0, shift = bits > 8 ? bits - 8 : 0;
  auto bin_of = [&](uint32_t depth) { return (min(max(depth, lo), hi) - lo) >> shift; };
#pragma unroll
  for (uint32_t u = 0; u < SAMPLED; u++)
    if (u * THREADS + tid < samples) atomicAdd(&s_bins[bin_of(z[u])], 1u);
  __syncthreads();
  if (wave == 0u) {
    // ends[k] of lane l: the samples in the bins up to 64 k + l
    uint32_t ends[QUARTERS], carry = 0u;
#pragma unroll
    for (uint32_t k = 0; k < QUARTERS; k++) {
      ends[k] = carry + wave_inclusive_scan_u32(s_bins[k * GS_WAVE + lane], (int)lane);
      carry = (uint32_t)__builtin_amdgcn_readlane((int)ends[k], GS_WAVE - 1);
    }
#pragma unroll
    for (uint32_t k = 0; k < QUARTERS; k++) s_bins[k * GS_WAVE + lane] = ends[k];
    auto bins_up_to = [&](uint32_t place) {
      uint32_t c = 0u;
#pragma unroll
      for (uint32_t k = 0; k < QUARTERS; k++) c += (uint32_t)__popcll(gs_ballot(ends[k] <= place));
      return c;
    };
    const uint32_t share = (uint32_t)((uint64_t)samples * blk / 5u * 4u / n), least = samples / (SPLIT_GROUPS - 16u) + 1u;
    const uint32_t wanted = max(share, least);
    uint32_t groups = 0u, first = 0u, bin = 0u;
    while (bin < SPLIT_BINS) {
      const uint32_t before = bins_up_to(first), whole = bins_up_to(first + wanted);
      const uint32_t end =
          groups + 1u == min(SPLIT_GROUPS, n) ? SPLIT_BINS : min(whole > before ? whole : before + 1u, SPLIT_BINS);
#pragma unroll
      for (uint32_t k = 0; k < QUARTERS; k++) {
        const uint32_t b = k * GS_WAVE + lane;
        if (b >= bin && b < end) s_group[b] = (uint8_t)groups;
      }
      first = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_bins[end - 1u]);
      bin = end;
      groups++;
    }
    if (lane == 0u) s_scan[0] = groups;
  }
  __syncthreads();
  const uint32_t groups = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_scan[0]);
  const int group_bits = 32 - __builtin_clz(groups | 1u);  // (so that no group has all of them set: that is nobody's)
  const uint32_t nobody = (1u << group_bits) - 1u;  // (a lane without a record; at least `groups`)
  // The lanes whose g equals the lane's own `a`, and those with its `b`: from one ballot for every bit of g.  A ballot's result
  // is hidden from the compiler before the lanes select on it.  Where it saw both (a ballot of g == k, selected by the lane
  // with that k) it put the lane's own number into the ballot, as if it were one lane's comparison: the counts came out wrong
  // and the records that are placed by them out of the list.
  auto lanes_with = [&](uint32_t g, uint32_t a, uint32_t b, uint64_t& with_a, uint64_t& with_b) {
    with_a = with_b = ~0ull;
    for (int k = 0; k < group_bits; k++) {
      uint64_t set = gs_ballot((g >> k & 1u) != 0u);
      asm("" : "+s"(set));
      with_a &= (a >> k & 1u) != 0u ? set : ~set;
      with_b &= (b >> k & 1u) != 0u ? set : ~set;
    }
  };
  const uint32_t part = (n + THREADS - 1u) / THREADS * GS_WAVE;  // a wave's records
  const uint32_t from = min(wave * part, n), to = min(from + part, n);
  uint32_t found = 0u;  // lane g: the wave's records of group g (lanes from `groups` on: anything)
  for (uint32_t i0 = from; i0 < to; i0 += GS_WAVE * COUNTED) {
    uint32_t d[COUNTED];
#pragma unroll
    for (uint32_t u = 0; u < COUNTED; u++) d[u] = list[min(i0 + u * GS_WAVE + lane, to - 1u)].z;
#pragma unroll
    for (uint32_t u = 0; u < COUNTED; u++) {
      const uint32_t g = i0 + u * GS_WAVE + lane < to ? (uint32_t)s_group[bin_of(d[u])] : nobody;
      uint64_t mine, unused;
      lanes_with(g, lane, lane, mine, unused);
      found += (uint32_t)__popcll(mine);
    }
  }
  s_count[wave * SPLIT_GROUPS + lane] = found;
  __syncthreads();
  uint32_t total = 0u, place = 0u;  // lane g: all records of group g, and those of the waves before this one
#pragma unroll
  for (uint32_t w = 0; w < WAVES; w++) {
    const uint32_t c = s_count[w * SPLIT_GROUPS + lane];
    place += w < wave ? c : 0u;
    total += c;
  }
  if (lane >= groups) total = 0u;
  const uint32_t group_first = wave_inclusive_scan_u32(total, (int)lane) - total;
  place += group_first;  // where the wave's next record of group g goes
  for (uint32_t i0 = from; i0 < to; i0 += GS_WAVE * MOVED) {
    TileRecord r[MOVED];
#pragma unroll
    for (uint32_t u = 0; u < MOVED; u++) r[u] = list[min(i0 + u * GS_WAVE + lane, to - 1u)];
#pragma unroll
    for (uint32_t u = 0; u < MOVED; u++) {
      const uint32_t g = i0 + u * GS_WAVE + lane < to ? (uint32_t)s_group[bin_of(r[u].z)] : nobody;
      uint64_t same, mine;
      lanes_with(g, g, lane, same, mine);
      const uint32_t next = (uint32_t)__shfl((int)place, (int)(g & 63u), GS_WAVE);
      const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, next));
      if (g != nobody)
        store_streaming(reinterpret_cast<float4*>(parted + start + at),
                        make_float4(__uint_as_float(r[u].x), __uint_as_float(r[u].y), __uint_as_float(r[u].z), 0.f));
      place += (uint32_t)__popcll(mine);
    }
  }
  if (wave == 0u) {
    if (lane < groups) list_words[start + lane] = group_first;
    if (lane == 0u) {
      *entry = t | groups << 16;
      atomicMax(most, groups);
    }
  }
  __syncthreads();  // (the words are the next sort's)
}

// Workgroup 0 orders the tiles for the blend kernels, workgroup t + 1 sorts tile t; before that, the first workgroups split
// the lists that are too long for one workgroup of the radix sort (split_lists: the number of them, see split_list, the tiles;
// the kernel with MAX_E = 8 only).
// Dynamic LDS: 8 bytes per record of the longest list the kernel takes, rounded up to a power of two (at least
// 256 records).  Lists of more than max_n records are left to the radix sort's kernels.
// MAX_E: the most keys a lane has.  Views without lists beyond 2048 have a kernel without the way for eight: in the other one
// (64 registers to 40) the shorter lists take longer too.  1 M Gaussians, 1920x1080, lists up to 839: 27.2 us with it, 25.1
// without; 160 k, 1709x858, 13.5 and 12.3; 300 k, 1237x822, 12.4 and 11.7.
#define GS_SORT_CASE(EE, WW) register_sort_tile<EE, WW>(t, start, n, records, keys, emission, point_list, s_exchange)
template <int MAX_E>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(MAX_E == 8 ? 8 : 2)))
tile_sort_registers_kernel(const uint32_t* __restrict__ ranges, const TileRecord* __restrict__ records,
                           uint64_t* __restrict__ keys, uint32_t* __restrict__ emission,
                           uint32_t* __restrict__ point_list, uint32_t max_n,
                           const uint32_t* __restrict__ fits_word, uint32_t* __restrict__ order,
                           uint32_t* __restrict__ order_word, uint32_t longest_split, int* __restrict__ n_consider,
                           int* __restrict__ n_contrib, uint32_t* __restrict__ split_lists, uint32_t block_limit,
                           TileRecord* __restrict__ parted, uint32_t* __restrict__ list_words) {
  extern __shared__ uint64_t s_exchange[];
  if (fits_word != nullptr && *fits_word == 0u) return;  // launched ahead of the host's decision: see the scatter
  if (blockIdx.x == 0) {
    order_tiles(gridDim.x - 1, ranges, order, order_word, longest_split, n_consider, n_contrib,
                reinterpret_cast<uint32_t*>(s_exchange));
    return;
  }
  const uint32_t t = blockIdx.x - 1;
  if constexpr (MAX_E == 8) {
    if (t < split_lists[0]) {
      const uint32_t long_tile = split_lists[2u + t], first = ranges[2 * long_tile];
      split_list(long_tile, first, ranges[2 * long_tile + 1] - first, block_limit, records, parted, list_words,
                 split_lists + 2u + t, split_lists + 1, reinterpret_cast<uint32_t*>(s_exchange));
    }
  }
  const uint32_t start = ranges[2 * t];
  const uint32_t n = ranges[2 * t + 1] - start;
  if (n == 0 || n > 512u * MAX_E || n > max_n) return;
  if (n <= 256) {
    if (threadIdx.x >= 256) return;  // (half the workgroup is enough; a wave that has left is not waited for)
    GS_SORT_CASE(1, 4);
  } else if (n <= 512) GS_SORT_CASE(1, 8);
  else if (n <= 1024) GS_SORT_CASE(2, 8);
  else if (MAX_E == 4 || n <= 2048) GS_SORT_CASE(4, 8);
  else if constexpr (MAX_E == 8) GS_SORT_CASE(8, 8);
}
#undef GS_SORT_CASE

}  // namespace

// Tiles the LDS histograms of the counting kernels can hold.
int bucket_max_tiles() { return 30000; }

// workgroup-by-tile counts, then the tile totals, then the tile lists of the radix sort's kernels (2 T + 3 words), then
// the workgroups' sums of tiles touched and the word that says whether the view fits the buffers of kernels
// launched ahead of the host
size_t bucket_table_bytes(int T) {
  return (((size_t)BK_MAX_BLOCKS + 3) * (size_t)T + 3 + BK_MAX_BLOCKS + 1) * sizeof(uint32_t);
}
static uint32_t* bucket_block_sums(void* table, uint32_t T) {
  return (uint32_t*)table + ((size_t)BK_MAX_BLOCKS + 3) * (size_t)T + 3;
}
const uint32_t* bucket_fits_word(const void* table, int T) {
  return (const uint32_t*)table + ((size_t)BK_MAX_BLOCKS + 3) * (size_t)T + 3 + BK_MAX_BLOCKS;
}

// The longest list that the radix sort's smaller kernel takes (what one of its workgroups holds); longer ones go to the
// larger kernel.
static uint32_t radix_mid_limit(uint32_t small_limit, uint32_t block_limit) {
  uint32_t limit = (uint32_t)tile_radix_mid_records();
  if (block_limit != 0 && block_limit < limit) limit = block_limit;
  return limit < small_limit ? small_limit : limit;
}

int launch_bucket_count(int P, int W, int H, const int* radii, const float* means2D, const uint8_t* compute_locally,
                        uint32_t* tiles_touched, void* table, uint32_t* ranges, uint32_t small_limit,
                        uint32_t block_limit, uint32_t* host_words, int* zero_per_gaussian, uint32_t cap_instances,
                        uint32_t cap_longest, uint32_t* clear_word, const ClearedArrays& cleared, hipStream_t stream) {
  if (P <= 0) return 0;
  if (small_limit == 0 || small_limit > (uint32_t)TILE_SORT_SMALL) small_limit = TILE_SORT_SMALL;
  const uint32_t mid_limit = radix_mid_limit(small_limit, block_limit);
  // ... and the lists the larger kernel holds; longer ones are split first
  uint32_t split_limit = (uint32_t)tile_radix_block_records();
  if (block_limit != 0 && block_limit < split_limit) split_limit = block_limit;
  if (split_limit < mid_limit) split_limit = mid_limit;
  const uint32_t gx = (W + GS_TILE_X - 1) / GS_TILE_X, gy = (H + GS_TILE_Y - 1) / GS_TILE_Y;
  const uint32_t T = gx * gy;
  const size_t lds = (size_t)T * (sizeof(uint32_t) + 1);
  // more than 64 KB of dynamic LDS has to be asked for, once per kernel and device (two threads that both find
  // the bit clear both ask, which is harmless)
  static std::atomic<uint64_t> raised{0};
  int dev = 0;
  GS_HIP_TRY(hipGetDevice(&dev));
  const uint64_t dev_bit = 1ull << (dev & 63);
  if (lds > 64 * 1024 && (dev >= 64 || !(raised.load(std::memory_order_acquire) & dev_bit))) {
    GS_HIP_TRY(hipFuncSetAttribute((const void*)bucket_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   bucket_max_tiles() * (int)(sizeof(uint32_t) + 1)));
    GS_HIP_TRY(hipFuncSetAttribute((const void*)bucket_scatter_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   bucket_max_tiles() * (int)(sizeof(uint32_t) + 1)));
    raised.fetch_or(dev_bit, std::memory_order_release);
  }
  const int nb = bucket_blocks(P), per = bucket_per_block(P);
  uint32_t* tab = (uint32_t*)table;
  uint32_t* totals = tab + (size_t)BK_MAX_BLOCKS * T;
  hipLaunchKernelGGL(bucket_count_kernel, dim3(nb), dim3(BK_THREADS), lds, stream, P, per, gx, gy, radii,
                     (const float2*)means2D, compute_locally, tiles_touched, tab, bucket_block_sums(table, T),
                     zero_per_gaussian);
  hipLaunchKernelGGL(bucket_columns_kernel, dim3((T + COL_TILES - 1) / COL_TILES), dim3(COL_TILES * COL_RUNS), 0, stream, nb, T,
                     tab, totals);
  // (as many workgroups as have a 16-byte word for every thread, at most what the chip holds beside the first)
  const uint64_t groups = (cleared.floats[0] + cleared.floats[1] + 4095u) / 4096u;
  const uint32_t clearing = (uint32_t)(groups < 511u ? groups : 511u);
  hipLaunchKernelGGL(bucket_ranges_kernel, dim3(1 + clearing), dim3(1024), 0, stream, T, small_limit, mid_limit, split_limit,
                     totals, ranges, totals + T,
                     bucket_block_sums(table, T), nb, host_words, cap_instances, cap_longest,
                     const_cast<uint32_t*>(bucket_fits_word(table, (int)T)), clear_word, cleared);
  return 0;
}

int launch_bucket_scatter(int P, int W, int H, const float* means2D, const float* depths,
                          const uint32_t* tiles_touched, uint32_t* point_offsets, const int* radii,
                          const uint8_t* compute_locally, void* table, const uint32_t* ranges, void* records,
                          bool ahead_of_host, hipStream_t stream) {
  if (P <= 0) return 0;
  const uint32_t gx = (W + GS_TILE_X - 1) / GS_TILE_X, gy = (H + GS_TILE_Y - 1) / GS_TILE_Y;
  const size_t lds = (size_t)gx * gy * (sizeof(uint32_t) + 1);
  const int vector_loads = (((uintptr_t)means2D | (uintptr_t)depths | (uintptr_t)tiles_touched |
                             (uintptr_t)point_offsets | (uintptr_t)radii) & 15u) == 0u ? 1 : 0;
  // One round per workgroup and room in the LDS for its records: they are staged and leave tile by tile.
  const size_t tiles_bytes = (size_t)gx * gy * (2 * sizeof(uint32_t) + 1);
  const size_t lds_room = 150 * 1024;
  if (bucket_per_block(P) <= BK_BATCH * BK_THREADS && tiles_bytes + 12 * 4096 <= lds_room) {
    const uint32_t cap = (uint32_t)((lds_room - tiles_bytes) / 12) & ~63u;
    const uint32_t T = gx * gy;
    const uint32_t* tab = (const uint32_t*)table;
    static std::atomic<uint64_t> raised{0};
    int dev = 0;
    GS_HIP_TRY(hipGetDevice(&dev));
    const uint64_t dev_bit = 1ull << (dev & 63);
    if (dev >= 64 || !(raised.load(std::memory_order_acquire) & dev_bit)) {
      for (const void* k : {(const void*)bucket_scatter_staged_kernel<1>, (const void*)bucket_scatter_staged_kernel<2>,
                            (const void*)bucket_scatter_staged_kernel<BK_BATCH>})
        GS_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_room));
      raised.fetch_or(dev_bit, std::memory_order_release);
    }
    const int per = bucket_per_block(P);
    const auto kernel = per <= BK_THREADS ? bucket_scatter_staged_kernel<1>
                        : per <= 2 * BK_THREADS ? bucket_scatter_staged_kernel<2> : bucket_scatter_staged_kernel<BK_BATCH>;
    hipLaunchKernelGGL(kernel, dim3(bucket_blocks(P)), dim3(BK_THREADS),
                       tiles_bytes + (size_t)cap * 12, stream, P, per, bucket_blocks(P), gx, gy,
                       (const float2*)means2D, depths, tiles_touched, bucket_block_sums(table, T), point_offsets, radii,
                       compute_locally, tab, tab + (size_t)BK_MAX_BLOCKS * T, ranges, (TileRecord*)records,
                       ahead_of_host ? bucket_fits_word(table, (int)T) : nullptr, vector_loads, cap);
    return 0;
  }
  hipLaunchKernelGGL(bucket_scatter_kernel, dim3(bucket_blocks(P)), dim3(BK_THREADS), lds, stream, P,
                     bucket_per_block(P), gx, gy, (const float2*)means2D, depths, tiles_touched,
                     bucket_block_sums(table, gx * gy), point_offsets, radii, compute_locally, (const uint32_t*)table,
                     ranges, (TileRecord*)records,
                     ahead_of_host ? bucket_fits_word(table, (int)(gx * gy)) : nullptr, vector_loads);
  return 0;
}

// Sorts every tile's segment of `records`.  `longest` is the longest list the launch has to be ready for and
// `radix_tiles` what the ranges kernel reported (number of lists for the radix sort's larger kernel << 16 | number
// for its smaller one; a caller that does not know passes 0xFFFFFFFF): the kernels that have nothing to do are
// not launched.  small_limit (at most TILE_SORT_SMALL) and block_limit as given to launch_bucket_count; `scratch`
// holds 24 bytes for each of the `capacity` instances the binning arrays are laid out for.  tile_order (T words) and
// the word that says it is there: see order_tiles (neither is written where there is no list at all).
int launch_tile_sort(int T, uint32_t longest, uint32_t radix_tiles, uint32_t small_limit, uint32_t block_limit,
                     const uint32_t* ranges, void* table, const void* records, void* scratch, uint32_t* list_words,
                     int64_t capacity, uint64_t* keys, uint32_t* emission, uint32_t* point_list, uint32_t* tile_order,
                     uint32_t* tile_order_word, uint32_t longest_split, int* n_consider, int* n_contrib,
                     bool ahead_of_host, hipStream_t stream) {
  if (T <= 0 || longest == 0) return 0;
  const uint32_t* fits = ahead_of_host ? bucket_fits_word(table, T) : nullptr;
  if (small_limit == 0 || small_limit > (uint32_t)TILE_SORT_SMALL) small_limit = TILE_SORT_SMALL;
  const uint32_t whole = longest < small_limit ? longest : small_limit;  // the longest list sorted in registers
  const uint32_t block = (uint32_t)tile_radix_block_records();
  if (block_limit == 0 || block_limit > block) block_limit = block;
  const bool split = longest > block_limit;  // (there may be lists that the radix sort wants split)
  uint32_t m = split ? 512 : 256;
  static_assert(SPLIT_WORDS * sizeof(uint32_t) <= 512 * sizeof(uint64_t), "the split's words fit");
  while (m < whole) m <<= 1;
  uint32_t* const tile_lists = (uint32_t*)table + ((size_t)BK_MAX_BLOCKS + 1) * (size_t)T;
  hipLaunchKernelGGL(whole > 2048 || split ? tile_sort_registers_kernel<8> : tile_sort_registers_kernel<4>, dim3(T + 1),
                     dim3(512), (size_t)m * sizeof(uint64_t), stream, ranges, (const TileRecord*)records, keys, emission,
                     point_list, small_limit, fits, tile_order, tile_order_word, longest_split, n_consider, n_contrib,
                     tile_lists + T + 1, block_limit, (TileRecord*)scratch, list_words);
  if (longest > small_limit) {
    // (a launch with nothing to do takes 4.6 us of the device: a view whose longest list is bounded does without)
    const bool lng = (radix_tiles >> 16) != 0u && longest > radix_mid_limit(small_limit, block_limit);
    // scratch: `capacity` 16-byte records for the lists that are split first, then as many 8-byte words
    uint64_t* pong = (uint64_t*)((char*)scratch + (size_t)capacity * 16);
    // (the smaller kernel has lists only where the caller's options leave some between the two limits)
    const bool mid = (radix_tiles & 0xFFFFu) != 0u && radix_mid_limit(small_limit, block_limit) > small_limit;
    if (launch_tile_radix_sort(T, mid, lng, ranges, tile_lists,
                               tile_lists + T, block_limit, records, scratch, list_words, keys, pong, keys, emission, point_list,
                               fits, stream))
      return 1;
  }
  return 0;
}

}  // namespace gs
