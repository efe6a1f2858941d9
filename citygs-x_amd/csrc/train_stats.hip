// Densification statistics of one rendered view, the body of GaussianModel.training_statis
// (scene/gaussian_model.py:1181-1205, called per view at train_internal.py:376-392), without its chain of
// boolean-mask gathers and scatters.  With A anchors of k offsets each, V visible anchors, S selected neural
// Gaussians among the V*k candidates:
//   opacity_accum[a] += sum_j max(opacity[rank(a)*k + j], 0);  anchor_demon[a] += 1      for visible a
//   slot (a, j) is hit when a is visible, offset_selection_mask[i] is set at i = rank(a)*k + j, and
//   update_filter[r] is set at r = rank2(i);  then
//   offset_gradient_accum[a*k+j] += |grad[r, 0:2]|;  offset_denom[a*k+j] += 1
// where rank / rank2 count the set entries of anchor_visible_mask / offset_selection_mask before a / i:
// exactly what "x[mask] = y" enumerates.  For n_offsets <= 256, the case that matters, the masks' set entries are
// counted per chunk, the counts become prefixes, and one kernel ranks the entries of its chunks itself and does all
// four updates; beyond that two exclusive scans write every rank and a thread per slot does the updates.
#include "gs_common.h"
#include "gs_kernels.h"

namespace gs {

namespace {

// IDX: 32-bit indices whenever every count fits (64-bit division per thread is what this kernel would
// otherwise spend most of its time on)
template <typename IDX>
__global__ void __launch_bounds__(GS_BLOCK_1D)
train_stats_kernel(IDX slots, int k, IDX Vk, IDX M, const uint8_t* __restrict__ visible,
                   const uint32_t* __restrict__ rank_visible, const uint8_t* __restrict__ selected,
                   const uint32_t* __restrict__ rank_selected, const uint8_t* __restrict__ update_filter,
                   const float* __restrict__ grad, int grad_stride, const float* __restrict__ opacity,
                   float* __restrict__ opacity_accum, float* __restrict__ anchor_demon,
                   float* __restrict__ grad_accum, float* __restrict__ denom) {
  const IDX s = (IDX)blockIdx.x * GS_BLOCK_1D + threadIdx.x;
  if (s >= slots) return;
  const IDX a = s / (IDX)k;
  const int j = (int)(s - a * (IDX)k);
  if (!visible[a]) return;
  const IDX first = (IDX)rank_visible[a] * (IDX)k;  // the anchor's first candidate
  if (j == 0) {
    float sum = 0.f;
    for (int q = 0; q < k; q++) {
      if (first + q < Vk) {
        const float o = opacity[first + q];
        sum += o < 0.f ? 0.f : o;
      }
    }
    opacity_accum[a] += sum;
    anchor_demon[a] += 1.0f;
  }
  const IDX i = first + (IDX)j;
  if (i >= Vk || !selected[i]) return;
  const IDX r = rank_selected[i];
  if (r >= M || !update_filter[r]) return;
  const float gx = grad[(size_t)r * grad_stride], gy = grad[(size_t)r * grad_stride + 1];
  grad_accum[s] += sqrtf(gx * gx + gy * gy);
  denom[s] += 1.0f;
}

// ---- n_offsets <= STATS_MAX_OFFSETS

constexpr uint32_t STATS_ROWS = 256;          // anchors per workgroup at the most, one thread each for the visibility mask
constexpr uint32_t STATS_SLOTS = 4096;        // ... and slots, which LDS has to hold
constexpr uint32_t STATS_SEL_CHUNK = 1024;    // candidates per prefix of the selection mask
constexpr uint32_t STATS_ITEMS = 5;           // candidates per thread and round
constexpr uint32_t STATS_ROUND = GS_BLOCK_1D * STATS_ITEMS;
constexpr int STATS_MAX_OFFSETS = 256;
constexpr uint32_t STATS_COUNT_THREADS = 1024;
constexpr uint32_t STATS_SPAN = STATS_COUNT_THREADS * 16;  // mask entries per counting workgroup, 16 a thread
// Spans, of either mask, beyond which their totals are turned into prefixes by a launch of their own (4 us and its gap):
// up to here a thread adds up two of them at the most.
constexpr uint32_t STATS_SPANS = 512;
static_assert(STATS_ROWS == GS_BLOCK_1D && STATS_MAX_OFFSETS <= STATS_ROUND, "a round holds whole anchors");
static_assert(STATS_SPAN % STATS_ROWS == 0 && STATS_SPAN % STATS_SEL_CHUNK == 0, "whole chunks");

__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t x) {
  return (uint32_t)__popc((x | ((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu)) & 0x80808080u);
}

// Set entries of mask[at, at + 16), bounded by n.
__device__ __forceinline__ uint32_t count16(const uint8_t* __restrict__ mask, uint32_t at, uint32_t n) {
  if (at + 16 <= n && ((uintptr_t)mask & 15) == 0) {
    const uint4 v = *reinterpret_cast<const uint4*>(mask + at);
    return nonzero_bytes(v.x) + nonzero_bytes(v.y) + nonzero_bytes(v.z) + nonzero_bytes(v.w);
  }
  uint32_t c = 0;
  for (uint32_t e = at; e < n && e < at + 16; e++) c += mask[e] != 0;
  return c;
}

// The set entries of a span of one of the masks (the first vis_spans workgroups: visibility): the total of the span, and
// before every `rows` anchors or STATS_SEL_CHUNK candidates of it those that the span has before them.
__global__ void __launch_bounds__(STATS_COUNT_THREADS)
train_stats_count_kernel(uint32_t A, uint32_t Vk, uint32_t vis_spans, uint32_t rows, const uint8_t* __restrict__ visible,
                         const uint8_t* __restrict__ selected, uint32_t* __restrict__ vis_prefix,
                         uint32_t* __restrict__ sel_prefix, uint32_t* __restrict__ vis_totals,
                         uint32_t* __restrict__ sel_totals) {
  __shared__ uint32_t s_wave[STATS_COUNT_THREADS / GS_WAVE];
  const bool first_mask = blockIdx.x < vis_spans;
  const uint32_t span = first_mask ? blockIdx.x : blockIdx.x - vis_spans, n = first_mask ? A : Vk;
  const uint32_t at = span * STATS_SPAN + 16 * threadIdx.x;
  const uint32_t c = count16(first_mask ? visible : selected, at, n);
  uint32_t total;
  const uint32_t before = block_exclusive_scan<STATS_COUNT_THREADS>(c, s_wave, total);
  const uint32_t chunk = first_mask ? rows : STATS_SEL_CHUNK;
  if (at % chunk == 0 && at < n) (first_mask ? vis_prefix : sel_prefix)[at / chunk] = before;
  if (threadIdx.x == 0) (first_mask ? vis_totals : sel_totals)[span] = total;
}

// The totals of the spans as prefixes, where a wave would have to add up too many of them.
__global__ void __launch_bounds__(1024)
train_stats_spine_kernel(uint32_t vis_spans, uint32_t sel_spans, uint32_t* vis_totals, uint32_t* sel_totals) {
  __shared__ uint32_t s_wave[1024 / GS_WAVE];
  if (blockIdx.x == 0) exclusive_prefix_in_place(vis_spans, vis_totals, s_wave);
  else exclusive_prefix_in_place(sel_spans, sel_totals, s_wave);
}

// A thread's share of the set entries in the spans before this one.
__device__ __forceinline__ uint32_t before_span(const uint32_t* __restrict__ totals, uint32_t span, bool prefixes) {
  if (prefixes) return threadIdx.x == 0 ? totals[span] : 0u;
  uint32_t sum = 0;
  for (uint32_t s = threadIdx.x; s < span; s += GS_BLOCK_1D) sum += totals[s];
  return sum;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int d = 1; d < GS_WAVE; d <<= 1) v += __shfl_xor(v, d, GS_WAVE);
  return v;
}

// A workgroup owns `rows` consecutive anchors (a power of two that divides STATS_SPAN).  Its visible ones are listed in
// LDS; their candidates are one run of the candidate arrays, taken STATS_ITEMS per thread and round (whole anchors a
// round), so that mask bytes, opacities and gradients are read in order and every step of the chain mask -> rank ->
// filter has all of a thread's loads in flight at once.  What a candidate adds to its slot waits in LDS; the slots'
// accumulators follow in their own order, four a thread.
// Bound by memory, most of it the two slot accumulators, 80 MB of which a view touches three quarters of the sectors at
// 1 M anchors of 10 offsets (40 % visible, 60 % of those selected).  Where a lane loaded and stored the accumulators of its
// own candidates, sectors went back in part: reading and writing such a pattern alone takes 39.5 us, with whole sectors
// 30.0.  With the ranks written out by two scans and one slot per thread, each waiting for six loads one after the other,
// the call took 139 us.  Six sets of inputs in turn, slot by slot -> sectors, the next round's masks asked for ahead:
// 59 -> 56 us (the spans' totals turned into prefixes by a launch of its own: 62), 2 M anchors 108 -> 100.5, 5 offsets
// 40 -> 39.  Five candidates are what eight waves a SIMD have registers for: with six and five waves 53 us where five took
// 48 and four 50.  Not kept: a wave for every 64 anchors, without barriers (50 us for this kernel where it took 44); the
// accumulators asked for with the masks, before it is known which slots gain (59 -> 63); gradients and opacities past the
// caches (60); the workgroups of one XCD on neighbouring anchors (60).
__global__ void __launch_bounds__(GS_BLOCK_1D) __attribute__((amdgpu_waves_per_eu(8)))
train_stats_chunk_kernel(uint32_t A, uint32_t k, uint32_t k_magic, uint32_t rows_log2, uint32_t Vk, uint32_t M,
                         bool prefixes, bool whole, const uint8_t* __restrict__ visible, const uint32_t* __restrict__ vis_prefix,
                         const uint32_t* __restrict__ vis_totals, const uint8_t* __restrict__ selected,
                         const uint32_t* __restrict__ sel_prefix, const uint32_t* __restrict__ sel_totals,
                         const uint8_t* __restrict__ update_filter, const float* __restrict__ grad, int grad_stride,
                         const float* __restrict__ opacity, float* __restrict__ opacity_accum,
                         float* __restrict__ anchor_demon, float* __restrict__ grad_accum, float* __restrict__ denom) {
  constexpr int WAVES = GS_BLOCK_1D / GS_WAVE;
  constexpr uint32_t NONE = 0xFFFFFFFFu;
  extern __shared__ float s_add[];  // of every candidate of the workgroup: what its slot gains, -1 where it gains nothing
  __shared__ float s_op[STATS_ROUND];
  __shared__ uint32_t s_row[STATS_ROWS];    // the visible anchors
  __shared__ uint32_t s_first[STATS_ROWS];  // an anchor's first candidate among the workgroup's, NONE where it is not visible
  __shared__ uint32_t s_count[WAVES], s_before[WAVES], s_head[WAVES];
  __shared__ uint32_t s_sel[STATS_ITEMS][WAVES];
  const uint32_t tid = threadIdx.x, lane = tid & (GS_WAVE - 1), wave = tid / GS_WAVE;
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t row0 = blockIdx.x << rows_log2;
  const uint32_t vis_before = wave_sum(before_span(vis_totals, row0 / STATS_SPAN, prefixes));
  uint32_t vis0 = vis_prefix[blockIdx.x];
  const bool set = (tid >> rows_log2) == 0u && row0 + tid < A && visible[row0 + tid] != 0;
  const uint64_t vm = gs_ballot(set);
  if (lane == 0) {
    s_count[wave] = (uint32_t)__popcll(vm);
    s_before[wave] = vis_before;
  }
  __syncthreads();
  uint32_t place = (uint32_t)__popcll(vm & below), rows = 0;
#pragma unroll
  for (uint32_t w = 0; w < WAVES; w++) {
    vis0 += s_before[w];
    if (w < wave) place += s_count[w];
    rows += s_count[w];
  }
  const uint64_t first64 = (uint64_t)vis0 * k;
  const uint32_t first = first64 < Vk ? (uint32_t)first64 : Vk;
  const uint32_t candidates = min(rows * k, Vk - first);
  // a round's masks and opacities are asked for one round ahead
  const uint32_t rows_per_round = STATS_ROUND / k, round = rows_per_round * k;  // (at least 5 anchors)
  uint8_t sel_next[STATS_ITEMS];
  float op_next[STATS_ITEMS];
  auto ask = [&](uint32_t at) {
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
      const uint32_t c = q * GS_BLOCK_1D + tid;
      const bool have = c < round && at + c < candidates;
      sel_next[q] = have ? selected[first + at + c] : (uint8_t)0;
      op_next[q] = have ? opacity[first + at + c] : 0.f;
    }
  };
  ask(0);
  // the rank of the chunk's first candidate: what is set in the spans before, in the chunks of its span before, and
  // before it in its chunk
  const uint32_t sel_chunk = first / STATS_SEL_CHUNK;
  uint32_t rank0 = first < Vk ? sel_prefix[sel_chunk] : 0u;  // (no candidates left: never used)
  uint32_t head = 0;
#pragma unroll
  for (uint32_t q = 0; q < STATS_SEL_CHUNK / GS_BLOCK_1D; q++) {
    const uint32_t e = sel_chunk * STATS_SEL_CHUNK + q * GS_BLOCK_1D + tid;
    head += (uint32_t)__popcll(gs_ballot(e < first && selected[e] != 0));
  }
  if (first < Vk) head += wave_sum(before_span(sel_totals, first / STATS_SPAN, prefixes));
  if (lane == 0) s_head[wave] = head;
  if (set) s_row[place] = row0 + tid;
  s_first[tid] = set ? place * k : NONE;
  __syncthreads();
#pragma unroll
  for (uint32_t w = 0; w < WAVES; w++) rank0 += s_head[w];

  for (uint32_t r0 = 0; r0 < rows; r0 += rows_per_round) {
    const uint32_t nr = min(rows_per_round, rows - r0), n = nr * k;
    bool sel[STATS_ITEMS];
    float op[STATS_ITEMS];
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
      sel[q] = sel_next[q] != 0;
      op[q] = op_next[q];
    }
    if (r0 + rows_per_round < rows) ask((r0 + rows_per_round) * k);
    uint32_t rank[STATS_ITEMS];
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
      const uint64_t m = gs_ballot(sel[q]);
      rank[q] = (uint32_t)__popcll(m & below);
      if (lane == 0) s_sel[q][wave] = (uint32_t)__popcll(m);
      s_op[q * GS_BLOCK_1D + tid] = op[q] < 0.f ? 0.f : op[q];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
#pragma unroll
      for (uint32_t w = 0; w < WAVES; w++) {
        if (w == wave) rank[q] += rank0;
        rank0 += s_sel[q][w];
      }
    }
    bool hit[STATS_ITEMS];
    float gx[STATS_ITEMS], gy[STATS_ITEMS];
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
      hit[q] = sel[q] && rank[q] < M;
      gx[q] = gy[q] = 0.f;
      if (hit[q]) {
        hit[q] = update_filter[rank[q]] != 0;
        gx[q] = grad[(size_t)rank[q] * grad_stride];
        gy[q] = grad[(size_t)rank[q] * grad_stride + 1];
      }
    }
#pragma unroll
    for (uint32_t q = 0; q < STATS_ITEMS; q++) {
      const uint32_t c = q * GS_BLOCK_1D + tid;
      if (c < n) s_add[r0 * k + c] = hit[q] ? sqrtf(gx[q] * gx[q] + gy[q] * gy[q]) : -1.0f;
    }
    if (tid < nr) {
      float sum = 0.f;
      for (uint32_t j = 0; j < k; j++) sum += s_op[tid * k + j];
      const uint32_t a = s_row[r0 + tid];
      opacity_accum[a] += sum;
      anchor_demon[a] += 1.0f;
    }
    __syncthreads();  // (the next round's lists, the slots' gains)
  }

  // Sixteen slots, a sector of memory of either accumulator, are loaded and stored as a whole where one of them gains.
  const uint32_t slots = min(1u << rows_log2, A - row0) * k;
  float* const ga = grad_accum + (size_t)row0 * k;
  float* const de = denom + (size_t)row0 * k;
  for (uint32_t s0 = 4 * (tid & ~3u); s0 < slots; s0 += 4 * GS_BLOCK_1D) {
    const uint32_t s = s0 + 4 * (tid & 3u);
    float add[4];
    bool any = false;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
      add[i] = -1.0f;
      if (s + i < slots) {
        const uint32_t a = k == 1 ? s + i : __umulhi(s + i, k_magic), f = s_first[a];
        if (f != NONE) add[i] = s_add[f + (s + i - a * k)];
      }
      any |= !(add[i] < 0.f);
    }
    // (a quad takes part as a whole)
    const uint64_t gains = gs_ballot(any);
    if (((gains >> (lane & ~3u)) & 0xFull) == 0ull) continue;
    if (whole && s + 4 <= slots) {
      float4 g = *(const float4*)(ga + s), d = *(const float4*)(de + s);
      g.x = add[0] < 0.f ? g.x : g.x + add[0];
      g.y = add[1] < 0.f ? g.y : g.y + add[1];
      g.z = add[2] < 0.f ? g.z : g.z + add[2];
      g.w = add[3] < 0.f ? g.w : g.w + add[3];
      d.x = add[0] < 0.f ? d.x : d.x + 1.0f;
      d.y = add[1] < 0.f ? d.y : d.y + 1.0f;
      d.z = add[2] < 0.f ? d.z : d.z + 1.0f;
      d.w = add[3] < 0.f ? d.w : d.w + 1.0f;
      *(float4*)(ga + s) = g;
      *(float4*)(de + s) = d;
    } else {
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) {
        if (!(add[i] < 0.f)) {
          ga[s + i] += add[i];
          de[s + i] += 1.0f;
        }
      }
    }
  }
}

}  // namespace

size_t train_stats_temp_bytes(long long A, long long Vk) {
  return align_up((size_t)(A > 0 ? A : 1) * 4, 256) + align_up((size_t)(Vk > 0 ? Vk : 1) * 4, 256) +
         align_up(scan_temp_bytes(A > Vk ? A : Vk), 256);
}

// gaussians.max_radii2D[visibility_filter] = max(gaussians.max_radii2D[visibility_filter], radii[visibility_filter])
// (densification.py:71-73, add_densification_stats' companion in the Gaussian-splatting training loop).
namespace {
__global__ void __launch_bounds__(GS_BLOCK_1D)
max_radii_kernel(long long n, const int* __restrict__ radii, const uint8_t* __restrict__ visible,
                 float* __restrict__ max_radii) {
  const long long i = (long long)blockIdx.x * GS_BLOCK_1D + threadIdx.x;
  if (i < n && visible[i]) max_radii[i] = fmaxf(max_radii[i], (float)radii[i]);
}
}  // namespace

int launch_max_radii(long long n, const int* radii, const uint8_t* visible, float* max_radii, hipStream_t stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(max_radii_kernel, dim3((unsigned)((n + GS_BLOCK_1D - 1) / GS_BLOCK_1D)), dim3(GS_BLOCK_1D), 0,
                     stream, n, radii, visible, max_radii);
  return 0;
}

int launch_train_stats(long long A, int k, long long Vk, long long M, const uint8_t* visible,
                       const uint8_t* selected, const uint8_t* update_filter, const float* grad, int grad_stride,
                       const float* opacity, float* opacity_accum, float* anchor_demon, float* grad_accum,
                       float* denom, void* temp, hipStream_t stream) {
  if (A <= 0 || k <= 0) return 0;
  const long long slots = A * k;
  if (k <= STATS_MAX_OFFSETS && slots < 0x7FFFFFFFll && Vk < 0x7FFFFFFFll && M < 0x7FFFFFFFll) {
    uint32_t rows_log2 = 8;  // (16 anchors of STATS_MAX_OFFSETS at the least: whole sectors of slots whatever k)
    while ((uint32_t)k << rows_log2 > STATS_SLOTS) rows_log2--;
    static_assert(STATS_ROWS == 1u << 8 && STATS_SLOTS == STATS_MAX_OFFSETS << 4, "between 16 and 256 anchors");
    const uint32_t vis_chunks = (uint32_t)((A + (1ll << rows_log2) - 1) >> rows_log2);
    const uint32_t vis_spans = (uint32_t)((A + STATS_SPAN - 1) / STATS_SPAN);
    const uint32_t sel_spans = (uint32_t)((Vk + STATS_SPAN - 1) / STATS_SPAN);
    // (a prefix per chunk and a total per span: less than the ranks, an entry each, that the space is sized for, a total
    // beside fewer prefixes than there are entries at least)
    uint32_t* vis_prefix = (uint32_t*)temp;
    uint32_t* vis_totals = vis_prefix + vis_chunks;
    uint32_t* sel_prefix = (uint32_t*)((char*)temp + align_up((size_t)A * 4, 256));
    uint32_t* sel_totals = sel_prefix + (Vk + STATS_SEL_CHUNK - 1) / STATS_SEL_CHUNK;
    const bool prefixes = vis_spans > STATS_SPANS || sel_spans > STATS_SPANS;
    hipLaunchKernelGGL(train_stats_count_kernel, dim3(vis_spans + sel_spans), dim3(STATS_COUNT_THREADS), 0, stream,
                       (uint32_t)A, (uint32_t)Vk, vis_spans, 1u << rows_log2, visible, selected, vis_prefix, sel_prefix,
                       vis_totals, sel_totals);
    if (prefixes)
      hipLaunchKernelGGL(train_stats_spine_kernel, dim3(2), dim3(1024), 0, stream, vis_spans, sel_spans, vis_totals,
                         sel_totals);
    hipLaunchKernelGGL(train_stats_chunk_kernel, dim3(vis_chunks), dim3(GS_BLOCK_1D),
                       sizeof(float) * (size_t)k << rows_log2, stream, (uint32_t)A, (uint32_t)k,
                       (uint32_t)(((1ull << 32) + k - 1) / k), rows_log2, (uint32_t)Vk, (uint32_t)M, prefixes,
                       ((uintptr_t)grad_accum & 15) == 0 && ((uintptr_t)denom & 15) == 0, visible, vis_prefix,
                       vis_totals, selected, sel_prefix, sel_totals, update_filter, grad, grad_stride, opacity,
                       opacity_accum, anchor_demon, grad_accum, denom);
    return 0;
  }
  char* base = (char*)temp;
  uint32_t* rank_visible = (uint32_t*)base;
  base += align_up((size_t)A * 4, 256);
  uint32_t* rank_selected = (uint32_t*)base;
  base += align_up((size_t)(Vk > 0 ? Vk : 1) * 4, 256);
  launch_exclusive_sum_u8(A, visible, rank_visible, base, stream);
  if (Vk > 0) launch_exclusive_sum_u8(Vk, selected, rank_selected, base, stream);
  const dim3 grid((unsigned)((slots + GS_BLOCK_1D - 1) / GS_BLOCK_1D));
  if (slots < 0x7FFFFFFFll - GS_BLOCK_1D && Vk < 0x7FFFFFFFll && M < 0x7FFFFFFFll)
    hipLaunchKernelGGL(train_stats_kernel<uint32_t>, grid, dim3(GS_BLOCK_1D), 0, stream, (uint32_t)slots, k,
                       (uint32_t)Vk, (uint32_t)M, visible, rank_visible, selected, rank_selected, update_filter, grad,
                       grad_stride, opacity, opacity_accum, anchor_demon, grad_accum, denom);
  else
    hipLaunchKernelGGL(train_stats_kernel<unsigned long long>, grid, dim3(GS_BLOCK_1D), 0, stream,
                       (unsigned long long)slots, k, (unsigned long long)Vk, (unsigned long long)M, visible,
                       rank_visible, selected, rank_selected, update_filter, grad, grad_stride, opacity, opacity_accum,
                       anchor_demon, grad_accum, denom);
  return 0;
}

}  // namespace gs
