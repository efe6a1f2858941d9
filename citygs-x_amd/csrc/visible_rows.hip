// Rows of the anchor model that a view shows: anchor[visible_mask] and its three companions of
// gaussian_renderer/__init__.py:794-798 (anchor, feature, offsets, scaling) in one pass over the mask, and the
// gradient of the four gathers as one pass over the full arrays.
//
// Bound by memory.  As nonzero() and four index_select()s the forward part was nine launches and 97 us at 500 k
// anchors of 10 offsets (35 % visible), and the backward part (a fill and an index_add per array, whose atomic adds
// fetch every line they touch) eight launches and 117 us; here 4 + 3 + 27 and 41 us (142 MB written).  A workgroup
// owns 256 consecutive rows, so that both sides of the forward copy run through memory in order, and the backward
// kernel writes every element of the full arrays once, the gradient's row or zero.
#include "gs_common.h"
#include "gs_kernels.h"

namespace gs {
namespace {

constexpr int VR_ROWS = 256;  // rows per workgroup of the copying kernels, one thread each for the mask
constexpr uint32_t VR_NONE = 0xFFFFFFFFu;

// Number of set entries per chunk of VR_ROWS, one wave per chunk.
__global__ void __launch_bounds__(GS_BLOCK_1D)
visible_count_kernel(uint32_t A, uint32_t chunks, const uint8_t* __restrict__ mask, uint32_t* __restrict__ counts) {
  const uint32_t chunk = blockIdx.x * (GS_BLOCK_1D / GS_WAVE) + threadIdx.x / GS_WAVE;
  if (chunk >= chunks) return;
  const uint32_t lane = threadIdx.x & (GS_WAVE - 1);
  uint32_t n = 0;
#pragma unroll
  for (uint32_t q = 0; q < VR_ROWS / GS_WAVE; q++) {
    const uint32_t row = chunk * VR_ROWS + q * GS_WAVE + lane;
    n += (uint32_t)__popcll(gs_ballot(row < A && mask[row] != 0));
  }
  if (lane == 0) counts[chunk] = n;
}

// One workgroup turns the counts into exclusive prefixes in place and hands the total to the host.
__global__ void __launch_bounds__(1024)
visible_spine_kernel(uint32_t chunks, uint32_t* __restrict__ counts, uint32_t* total_out) {
  __shared__ uint32_t s_wave[1024 / GS_WAVE];
  const uint32_t carry = exclusive_prefix_in_place(chunks, counts, s_wave);
  if (threadIdx.x == 0) {
    counts[chunks] = carry;
    // the host may be polling this word (host-visible memory)
    if (total_out != nullptr)
      __hip_atomic_store(total_out, carry, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// e / width for e below 2^32 / width: the chunk's word indices (at most 256 x 768) by a multiplication.
struct RowWidth {
  uint32_t width, magic;
};
__device__ __forceinline__ uint32_t row_of(uint32_t e, RowWidth w) { return __umulhi(e, w.magic); }

template <typename T>
__device__ __forceinline__ void copy_rows(const T* __restrict__ in, T* __restrict__ out, uint32_t row0, size_t out0,
                                          uint32_t rows, RowWidth w, const uint32_t* s_row) {
  const uint32_t n = rows * w.width;
  out += out0 * w.width;
  in += (size_t)row0 * w.width;
#pragma unroll 4
  for (uint32_t e = threadIdx.x; e < n; e += VR_ROWS) {
    const uint32_t r = row_of(e, w);
    out[e] = in[(s_row[r] - r) * w.width + e];  // row s_row[r], word e - r * width
  }
}

__global__ void __launch_bounds__(VR_ROWS)
visible_gather_kernel(uint32_t A, uint32_t N, const uint8_t* __restrict__ mask, const uint32_t* __restrict__ prefix,
                      RowWidth w3, RowWidth w6, RowWidth w8, RowWidth woff, const float* __restrict__ anchor,
                      const float4* __restrict__ feat, const float* __restrict__ offsets,
                      const float* __restrict__ scaling, float* __restrict__ anchor_out,
                      float4* __restrict__ feat_out, float* __restrict__ offsets_out,
                      float* __restrict__ scaling_out, uint32_t* __restrict__ rank, int64_t* __restrict__ index) {
  __shared__ uint32_t s_row[VR_ROWS];
  __shared__ uint32_t s_count[VR_ROWS / GS_WAVE];
  const uint32_t lane = threadIdx.x & (GS_WAVE - 1), wave = threadIdx.x / GS_WAVE;
  const uint32_t row0 = blockIdx.x * VR_ROWS, row = row0 + threadIdx.x;
  const bool set = row < A && mask[row] != 0;
  const uint64_t m = gs_ballot(set);
  if (lane == 0) s_count[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = (uint32_t)__popcll(m & ((1ull << lane) - 1ull)), rows = 0;
#pragma unroll
  for (uint32_t v = 0; v < VR_ROWS / GS_WAVE; v++) {
    if (v < wave) before += s_count[v];
    rows += s_count[v];
  }
  const uint32_t out0 = prefix[blockIdx.x];
  // (N is what the host was told; a mask that changed since then must not lead outside the N rows)
  rows = out0 >= N ? 0u : (rows < N - out0 ? rows : N - out0);
  const bool kept = set && before < rows;
  if (kept) {
    s_row[before] = threadIdx.x;
    if (index != nullptr) index[out0 + before] = (int64_t)row;
  }
  if (row < A) rank[row] = kept ? out0 + before : VR_NONE;
  __syncthreads();
  copy_rows(feat, feat_out, row0, out0, rows, w8, s_row);
  copy_rows(offsets, offsets_out, row0, out0, rows, woff, s_row);
  copy_rows(scaling, scaling_out, row0, out0, rows, w6, s_row);
  copy_rows(anchor, anchor_out, row0, out0, rows, w3, s_row);
}

// One full array of the chunk: row r holds the gradient's row s_rank[r], or zeros.  Four words per store (a chunk
// starts at a multiple of 256 rows, so 16-byte aligned whatever the width).
__device__ __forceinline__ void spread_rows(const float* __restrict__ g, float* __restrict__ d, uint32_t row0,
                                            uint32_t rows, RowWidth w, const uint32_t* s_rank) {
  const uint32_t n = rows * w.width;
  d += (size_t)row0 * w.width;
  const auto word = [&](uint32_t e) -> float {
    const uint32_t r = row_of(e, w), k = s_rank[r];
    return k == VR_NONE ? 0.f : g[(size_t)k * w.width + (e - r * w.width)];
  };
#pragma unroll 2
  for (uint32_t e = 4 * threadIdx.x; e + 4 <= n; e += 4 * VR_ROWS)
    *(float4*)(d + e) = make_float4(word(e), word(e + 1), word(e + 2), word(e + 3));
  const uint32_t tail = (n & ~3u) + threadIdx.x;
  if (tail < n) d[tail] = word(tail);
}

__global__ void __launch_bounds__(VR_ROWS)
visible_spread_kernel(uint32_t A, RowWidth w3, RowWidth w6, RowWidth woff, const uint32_t* __restrict__ rank,
                      const float* __restrict__ g_anchor, const float4* __restrict__ g_feat,
                      const float* __restrict__ g_offsets, const float* __restrict__ g_scaling,
                      float* __restrict__ d_anchor, float4* __restrict__ d_feat, float* __restrict__ d_offsets,
                      float* __restrict__ d_scaling) {
  __shared__ uint32_t s_rank[VR_ROWS];
  const uint32_t row0 = blockIdx.x * VR_ROWS;
  const uint32_t rows = A - row0 < VR_ROWS ? A - row0 : VR_ROWS;
  s_rank[threadIdx.x] = threadIdx.x < rows ? rank[row0 + threadIdx.x] : VR_NONE;
  __syncthreads();
  if (d_feat != nullptr) {
#pragma unroll 4
    for (uint32_t e = threadIdx.x; e < rows * 8; e += VR_ROWS) {
      const uint32_t k = s_rank[e >> 3];
      d_feat[(size_t)row0 * 8 + e] =
          k == VR_NONE ? make_float4(0.f, 0.f, 0.f, 0.f) : g_feat[(size_t)k * 8 + (e & 7)];
    }
  }
  if (d_offsets != nullptr) spread_rows(g_offsets, d_offsets, row0, rows, woff, s_rank);
  if (d_scaling != nullptr) spread_rows(g_scaling, d_scaling, row0, rows, w6, s_rank);
  if (d_anchor != nullptr) spread_rows(g_anchor, d_anchor, row0, rows, w3, s_rank);
}

RowWidth row_width(uint32_t width) {
  return RowWidth{width, (uint32_t)(((1ull << 32) + width - 1) / width)};
}

uint32_t chunks_of(int64_t A) { return (uint32_t)((A + VR_ROWS - 1) / VR_ROWS); }

}  // namespace

size_t visible_rows_workspace_words(int64_t A) { return (size_t)chunks_of(A > 0 ? A : 0) + 1; }

const uint32_t* visible_rows_total(const uint32_t* workspace, int64_t A) { return workspace + chunks_of(A); }

void launch_visible_count(int64_t A, const uint8_t* mask, uint32_t* workspace, uint32_t* total_out,
                          hipStream_t stream) {
  const uint32_t chunks = chunks_of(A), per_block = GS_BLOCK_1D / GS_WAVE;
  hipLaunchKernelGGL(visible_count_kernel, dim3((chunks + per_block - 1) / per_block), dim3(GS_BLOCK_1D), 0, stream,
                     (uint32_t)A, chunks, mask, workspace);
  hipLaunchKernelGGL(visible_spine_kernel, dim3(1), dim3(1024), 0, stream, chunks, workspace, total_out);
}

void launch_visible_gather(int64_t A, int k, int64_t N, const uint8_t* mask, const uint32_t* workspace,
                           const float* anchor, const float* feat, const float* offsets, const float* scaling,
                           float* anchor_out, float* feat_out, float* offsets_out, float* scaling_out,
                           uint32_t* rank, int64_t* index, hipStream_t stream) {
  hipLaunchKernelGGL(visible_gather_kernel, dim3(chunks_of(A)), dim3(VR_ROWS), 0, stream, (uint32_t)A, (uint32_t)N,
                     mask, workspace, row_width(3), row_width(6), row_width(8), row_width(3u * (uint32_t)k), anchor,
                     (const float4*)feat, offsets, scaling, anchor_out, (float4*)feat_out, offsets_out, scaling_out,
                     rank, index);
}

void launch_visible_spread(int64_t A, int k, const uint32_t* rank, const float* g_anchor, const float* g_feat,
                           const float* g_offsets, const float* g_scaling, float* d_anchor, float* d_feat,
                           float* d_offsets, float* d_scaling, hipStream_t stream) {
  hipLaunchKernelGGL(visible_spread_kernel, dim3(chunks_of(A)), dim3(VR_ROWS), 0, stream, (uint32_t)A, row_width(3),
                     row_width(6), row_width(3u * (uint32_t)k), rank, g_anchor, (const float4*)g_feat, g_offsets,
                     g_scaling, d_anchor, (float4*)d_feat, d_offsets, d_scaling);
}

}  // namespace gs
