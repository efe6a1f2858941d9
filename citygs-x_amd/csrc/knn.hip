// Mean squared distance to the three nearest neighbours of every point
// (simple-knn/simple_knn.cu:185-221, distCUDA2): global bounding box, a 30-bit
// key along a space-filling curve (27-bit for few points), stable sort by key,
// bounding boxes of runs of 1024 sorted points, then an exact search that visits only boxes closer
// than the current third-best distance.  The search is exhaustive within that
// bound, so the three distances equal a brute-force search whatever the order
// of the points and whatever the visiting order.  That leaves the curve free:
// the reference sorts by Morton code on a grid stretched to the bounding box
// (simple_knn.cu:54-76); here the key is the Hilbert index on a grid with
// cubic cells.  The Morton curve jumps (a run of consecutive points can lie in
// two far-apart places, and its bounding box then spans everything between
// them), the Hilbert curve does not, and runs along it are compact: a wave
// opens 38 instead of 68 sixteen-point runs per leaf on a 200 x 200 x 30 m
// slab of a million uniform points.
#include <float.h>

#include "gs_common.h"
#include "gs_kernels.h"

namespace gs {

namespace {

constexpr int KNN_BOX = 1024;  // simple-knn/simple_knn.cu:12
constexpr int KNN_GROUP = 64;  // boxes per group (one group test replaces this many box tests)
constexpr int KNN_LEAF = 64;   // points per leaf box inside a box (one leaf test replaces this many distances)
constexpr int KNN_TWIG = 16;   // points per twig box inside a leaf (the finest level)
constexpr int MM_BLOCKS = 512;
constexpr int MM_THREADS = 256;
constexpr int KEY_THREADS = 512;
constexpr int KEY_BLOCKS = 256;  // at most: a workgroup adds its digit counts to the sort's once
constexpr int AXIS_BITS = 10;    // of the curve
constexpr int KEY_BITS = 3 * AXIS_BITS;
// Few points take the curve's first nine levels, which the sort orders in three passes instead of four; points of one
// cell then keep their input order, which the boxes do not mind until a cell holds many.  32 k points of an SfM-like
// cloud: 106-112 -> 94-100 us a call, 5 k 100 -> 90; in 64 tight clusters of a scene a hundred times their size, the
// worst for coarse cells, 32 k: 113-161 -> 98-152 us (ten draws each, faster in all).  Above, such clusters lose: 65 k
// 152 -> 201 us in one draw, 200 k 214 -> 260, 1 M 1186 -> 2204.  (Six levels and two passes: 20 k 84 us in the first
// cloud, but 50 k 145 instead of 134 us in the second.)
constexpr int KEY_SHORT_BITS = 27;
constexpr int KEY_SHORT_MAX = 1 << 15;

// The search takes the leaves by falling size where there are more of them than waves that run at a time (32 a CU): one
// among sparse points takes ten times as long as the median, and if it starts with the last ones the chip idles
// until it ends.  1 M points of an SfM-like cloud: all waves had started after 123 us, half of them had ended after 94,
// nine in ten after 161 and the last after 251.
constexpr int ORDER_THREADS = 1024;
constexpr int ORDER_MIN_LEAVES = 8192;
constexpr int ORDER_BINS = 512;  // of a leaf's longest side: the exponent and one bit of the fraction
constexpr uint32_t NO_LEAF = 0xFFFFFFFFu;

// The leaves are ordered in `segments` parts, leaf l in part l % segments: none where they are too few to order.
int order_segments(int P) {
  const int leaves = (P + KNN_LEAF - 1) / KNN_LEAF;
  return leaves > ORDER_MIN_LEAVES ? (leaves + ORDER_THREADS - 1) / ORDER_THREADS : 0;
}

struct KnnLayout {
  size_t partial, codes_a, codes_b, idx_a, idx_b, sorted_pts, boxes, groups, leaves, twigs, order, sort_temp, total;
};

KnnLayout knn_layout(int P) {
  KnnLayout L;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off += align_up(bytes, 256);
    return o;
  };
  const size_t n = (size_t)(P > 0 ? P : 1);
  const size_t nb = (n + KNN_BOX - 1) / KNN_BOX;
  L.partial = take(sizeof(float) * 6 * MM_BLOCKS);
  L.codes_a = take(sizeof(uint32_t) * n);
  L.codes_b = take(sizeof(uint32_t) * n);
  L.idx_a = take(sizeof(uint32_t) * n);
  L.idx_b = take(sizeof(uint32_t) * n);
  L.sorted_pts = take(sizeof(float4) * n);
  L.boxes = take(sizeof(float) * 6 * nb);
  L.leaves = take(sizeof(float) * 6 * ((n + KNN_LEAF - 1) / KNN_LEAF));
  L.twigs = take(sizeof(float) * 6 * ((n + KNN_TWIG - 1) / KNN_TWIG));
  L.groups = take(sizeof(float) * 6 * ((nb + KNN_GROUP - 1) / KNN_GROUP));
  L.order = take(sizeof(uint32_t) * ORDER_THREADS * (size_t)order_segments(P));
  L.sort_temp = take(sort_temp_bytes((int64_t)n));
  L.total = off;
  return L;
}

// v[0..2] min, v[3..5] max over the workgroup; thread 0 leaves them in out (LDS or memory)
template <int THREADS>
__device__ __forceinline__ void reduce6(float* v, float (*s)[THREADS / GS_WAVE], float* out) {
#pragma unroll
  for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      v[k] = fminf(v[k], __shfl_xor(v[k], d, GS_WAVE));
      v[3 + k] = fmaxf(v[3 + k], __shfl_xor(v[3 + k], d, GS_WAVE));
    }
  }
  const int lane = threadIdx.x & (GS_WAVE - 1), wave = threadIdx.x / GS_WAVE;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 6; k++) s[k][wave] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      float mn = s[k][0], mx = s[3 + k][0];
      for (int w = 1; w < THREADS / GS_WAVE; w++) {
        mn = fminf(mn, s[k][w]);
        mx = fmaxf(mx, s[3 + k][w]);
      }
      out[k] = mn;
      out[3 + k] = mx;
    }
  }
}

// (The reference reduces from 0, simple-knn/simple_knn.cu:191, which makes its grid include the origin; the keys
// here are only a means of ordering, so the grid is the points' own bounding box.)  Clears the sort's words on the way.
__global__ void __launch_bounds__(MM_THREADS) minmax_partial_kernel(int P, const float* __restrict__ pts,
                                                                     float* __restrict__ partial, int64_t clear_words,
                                                                     uint32_t* __restrict__ clear) {
  for (int64_t i = (int64_t)blockIdx.x * MM_THREADS + threadIdx.x; i < clear_words; i += MM_BLOCKS * MM_THREADS)
    clear[i] = 0u;
  __shared__ float s[6][MM_THREADS / GS_WAVE];
  float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (int i = blockIdx.x * MM_THREADS + threadIdx.x; i < P; i += MM_BLOCKS * MM_THREADS) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float c = pts[3 * (size_t)i + k];
      v[k] = fminf(v[k], c);
      v[3 + k] = fmaxf(v[3 + k], c);
    }
  }
  reduce6<MM_THREADS>(v, s, partial + 6 * blockIdx.x);
}

__device__ __forceinline__ uint32_t spread10(uint32_t x) {  // every bit of a 10-bit number to every third place
  x = (x | (x << 16)) & 0x030000FF;
  x = (x | (x << 8)) & 0x0300F00F;
  x = (x | (x << 4)) & 0x030C30C3;
  x = (x | (x << 2)) & 0x09249249;
  return x;
}

// Index of grid cell (x, y, z), 10 bits each, along the three-dimensional Hilbert curve (Skilling's transform:
// undo the curve's rotations and reflections level by level, Gray-code, interleave).  Consecutive indices are
// neighbouring cells.
__device__ __forceinline__ uint32_t hilbert30(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t X[3] = {x, y, z};
#pragma unroll
  for (uint32_t Q = 1u << 9; Q > 1u; Q >>= 1) {
    const uint32_t low = Q - 1u;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      if (X[i] & Q) {
        X[0] ^= low;
      } else {
        const uint32_t t = (X[0] ^ X[i]) & low;
        X[0] ^= t;
        X[i] ^= t;
      }
    }
  }
  X[1] ^= X[0];
  X[2] ^= X[1];
  uint32_t t = 0u;
#pragma unroll
  for (uint32_t Q = 1u << 9; Q > 1u; Q >>= 1)
    if (X[2] & Q) t ^= Q - 1u;
  return (spread10(X[0] ^ t) << 2) | (spread10(X[1] ^ t) << 1) | spread10(X[2] ^ t);
}

// Every point's key, and the digit counts of the sort that follows.  17 us at 1 M points (20 with twice the workgroups);
// as kernels of their own the keys took 9, the rest of the bounding box 4 and the counts, which read the keys again, 15.
template <int BITS>
__global__ void __launch_bounds__(KEY_THREADS) curve_key_kernel(int P, const float* __restrict__ pts,
                                                                const float* __restrict__ partial,
                                                                uint32_t* __restrict__ codes, uint32_t* __restrict__ idx,
                                                                uint32_t* __restrict__ hist) {
  constexpr int RADIX = 1 << SORT_DIGIT_BITS, PASSES = (BITS + SORT_DIGIT_BITS - 1) / SORT_DIGIT_BITS;
  // where the last digit has few values, which would make a wave's counts queue for the same words, they have several
  // counts each
  constexpr int LAST_COPIES = RADIX >> (BITS - (PASSES - 1) * SORT_DIGIT_BITS);
  static_assert(KEY_THREADS == RADIX && MM_BLOCKS == KEY_THREADS, "a thread per digit value and per partial box");
  __shared__ uint32_t s_hist[PASSES][RADIX];
  __shared__ float s[6][KEY_THREADS / GS_WAVE];
  __shared__ float s_box[6];
#pragma unroll
  for (int p = 0; p < PASSES; p++) s_hist[p][threadIdx.x] = 0u;
  {
    float v[6];
#pragma unroll
    for (int c = 0; c < 6; c++) v[c] = partial[6 * threadIdx.x + c];
    reduce6<KEY_THREADS>(v, s, s_box);
  }
  __syncthreads();
  const float lo[3] = {s_box[0], s_box[1], s_box[2]};
  // cubic cells: the longest side of the bounding box takes the 1024 steps
  const float side = fmaxf(fmaxf(s_box[3] - lo[0], s_box[4] - lo[1]), s_box[5] - lo[2]);
  for (int64_t i = (int64_t)blockIdx.x * KEY_THREADS + threadIdx.x; i < P; i += (int64_t)gridDim.x * KEY_THREADS) {
    uint32_t c[3];
#pragma unroll
    for (int k = 0; k < 3; k++)
      c[k] = min(f2u_sat(((pts[3 * i + k] - lo[k]) / side) * (float)((1 << AXIS_BITS) - 1)),
                 (1u << AXIS_BITS) - 1u);
    const uint32_t key = hilbert30(c[0], c[1], c[2]) >> (3 * AXIS_BITS - BITS);
    codes[i] = key;
    idx[i] = (uint32_t)i;
#pragma unroll
    for (int p = 0; p < PASSES - 1; p++) atomicAdd(&s_hist[p][(key >> (SORT_DIGIT_BITS * p)) & (RADIX - 1)], 1u);
    atomicAdd(&s_hist[PASSES - 1][(key >> (SORT_DIGIT_BITS * (PASSES - 1))) * LAST_COPIES + threadIdx.x % LAST_COPIES],
              1u);
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PASSES - 1; p++) {
    const uint32_t n = s_hist[p][threadIdx.x];
    if (n != 0u) atomicAdd(&hist[p * RADIX + threadIdx.x], n);
  }
  if (threadIdx.x < RADIX / LAST_COPIES) {
    uint32_t n = 0u;
    for (int q = 0; q < LAST_COPIES; q++) n += s_hist[PASSES - 1][threadIdx.x * LAST_COPIES + q];
    if (n != 0u) atomicAdd(&hist[(PASSES - 1) * RADIX + threadIdx.x], n);
  }
}

// A value moved round its row of sixteen lanes: lane i reads lane (i + 16 - N) % 16 of the row.
template <int N>
__device__ __forceinline__ float row_ror(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}

__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, row_ror<8>(v));
  v = fmaxf(v, row_ror<4>(v));
  v = fmaxf(v, row_ror<2>(v));
  return fmaxf(v, row_ror<1>(v));
}

__device__ __forceinline__ float row_min(float v) {
  v = fminf(v, row_ror<8>(v));
  v = fminf(v, row_ror<4>(v));
  v = fminf(v, row_ror<2>(v));
  return fminf(v, row_ror<1>(v));
}

// The points in curve order, and the bounding boxes of every run of KNN_BOX of them (simple-knn/simple_knn.cu:78-117),
// of every run of KNN_LEAF (one wave each) and of every run of KNN_TWIG (a row of sixteen lanes each): a workgroup
// per box, a thread per point.  Leaves and twigs are additions to the reference's boxes, which prune work without
// changing which neighbours are found.  (A gather, a box and a leaf kernel before: 32 us at
// 1 M points; now 20.)
__global__ void __launch_bounds__(KNN_BOX) gather_boxes_kernel(int P, const float* __restrict__ pts,
                                                               const uint32_t* __restrict__ idx,
                                                               float4* __restrict__ sorted_pts,
                                                               float* __restrict__ boxes, float* __restrict__ leaves,
                                                               float* __restrict__ twigs) {
  static_assert(KNN_LEAF == GS_WAVE && KNN_TWIG == 16, "a leaf is a wave, a twig a row of 16 lanes");
  constexpr int LEAVES = KNN_BOX / KNN_LEAF;
  static_assert(LEAVES == 16, "a box is combined from its leaves by one row of lanes");
  __shared__ float s[6][LEAVES];
  const int i = blockIdx.x * KNN_BOX + threadIdx.x;
  const int lane = threadIdx.x & (GS_WAVE - 1), wave = threadIdx.x / GS_WAVE;
  float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
  if (i < P) {
    const size_t g = idx[i];
    const float4 p = make_float4(pts[3 * g], pts[3 * g + 1], pts[3 * g + 2], 0.f);
    sorted_pts[i] = p;
    // (a NaN coordinate leaves the box as it is: minima and maxima pass it over)
    v[0] = fminf(v[0], p.x); v[1] = fminf(v[1], p.y); v[2] = fminf(v[2], p.z);
    v[3] = fmaxf(v[3], p.x); v[4] = fmaxf(v[4], p.y); v[5] = fmaxf(v[5], p.z);
  }
#pragma unroll
  for (int c = 0; c < 3; c++) {
    v[c] = row_min(v[c]);
    v[3 + c] = row_max(v[3 + c]);
  }
  if ((lane & (KNN_TWIG - 1)) == 0 && i < P) {
#pragma unroll
    for (int c = 0; c < 6; c++) twigs[6 * (size_t)(i / KNN_TWIG) + c] = v[c];
  }
#pragma unroll
  for (int d = KNN_TWIG; d < GS_WAVE; d <<= 1) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      v[c] = fminf(v[c], __shfl_xor(v[c], d, GS_WAVE));
      v[3 + c] = fmaxf(v[3 + c], __shfl_xor(v[3 + c], d, GS_WAVE));
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int c = 0; c < 6; c++) {
      if (i < P) leaves[6 * (size_t)(i / KNN_LEAF) + c] = v[c];
      s[c][wave] = v[c];
    }
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const float mn = row_min(s[c][lane & (LEAVES - 1)]), mx = row_max(s[3 + c][lane & (LEAVES - 1)]);
      if (lane == 0) {
        boxes[6 * blockIdx.x + c] = mn;
        boxes[6 * blockIdx.x + 3 + c] = mx;
      }
    }
  }
}

// Bounding box of every run of KNN_GROUP consecutive boxes: lets the search discard that many boxes with
// one test.  (Not in the reference, which tests every box for every point; the result is the same set of
// three nearest neighbours, because a group's box bounds its members' boxes from below.)
// Also hands a sort that gave up waiting on to the host (fault_word), as launch_sort_fault_report does, and orders the
// leaves for the search (order != nullptr): workgroup s those of part s, a thread each, by a counting sort over bins of
// their longest sides, largest first, leaves of one bin in their old order; entry i * segments + s is the i-th of them,
// so that the parts' largest come first together and neighbours along the curve stay neighbours.
__global__ void __launch_bounds__(ORDER_THREADS)
box_group_kernel(int nboxes, const float* __restrict__ boxes, float* __restrict__ groups, int nleaves,
                 const float* __restrict__ leaves, uint32_t* __restrict__ order, const uint32_t* __restrict__ sort_error,
                 uint32_t* __restrict__ fault_word) {
  constexpr int WAVES = ORDER_THREADS / GS_WAVE;
  __shared__ uint32_t s_count[WAVES][ORDER_BINS];
  __shared__ uint32_t s_scan[ORDER_BINS / GS_WAVE];
  const int tid = threadIdx.x, lane = tid & (GS_WAVE - 1), wave = tid / GS_WAVE;
  if (blockIdx.x == 0 && tid == 0 && fault_word != nullptr && *sort_error != 0u)
    __hip_atomic_store(fault_word, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  const int group = blockIdx.x * WAVES + wave;
  if (group < (nboxes + KNN_GROUP - 1) / KNN_GROUP) {
    static_assert(KNN_GROUP == GS_WAVE, "a lane per box of the group");
    const int b = group * KNN_GROUP + lane;
    float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
    if (b < nboxes) {
#pragma unroll
      for (int c = 0; c < 6; c++) v[c] = boxes[6 * b + c];
    }
#pragma unroll
    for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
#pragma unroll
      for (int c = 0; c < 3; c++) {
        v[c] = fminf(v[c], __shfl_xor(v[c], d, GS_WAVE));
        v[3 + c] = fmaxf(v[3 + c], __shfl_xor(v[3 + c], d, GS_WAVE));
      }
    }
    if (lane == 0) {
#pragma unroll
      for (int c = 0; c < 6; c++) groups[6 * group + c] = v[c];
    }
  }
  if (order == nullptr) return;
  const int leaf = (int)blockIdx.x + (int)gridDim.x * tid;
  uint32_t bin = ORDER_BINS - 1;  // (a leaf that does not exist comes last, behind those of side 0)
  if (leaf < nleaves) {
    float side = 0.f;
#pragma unroll
    for (int c = 0; c < 3; c++) side = fmaxf(side, leaves[6 * (size_t)leaf + 3 + c] - leaves[6 * (size_t)leaf + c]);
    const uint32_t size = __builtin_bit_cast(uint32_t, side) >> 22;  // (never negative: below 512)
    bin = size < ORDER_BINS - 2 ? ORDER_BINS - 2 - size : 0u;
  }
  for (int e = tid; e < WAVES * ORDER_BINS; e += ORDER_THREADS) (&s_count[0][0])[e] = 0u;
  __syncthreads();
  // a wave's leaves of the same bin: how many, and this one's place among them
  uint32_t place = 0u;
  for (uint64_t rest = ~0ull; rest != 0ull;) {
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)bin, (int)__builtin_ctzll(rest));
    const uint64_t same = gs_ballot(bin == b);
    if (bin == b) place = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
    if (lane == 0) s_count[wave][b] = (uint32_t)__popcll(same);
    rest &= ~same;
  }
  __syncthreads();
  uint32_t total = 0u, inc = 0u;
  if (tid < ORDER_BINS) {
#pragma unroll
    for (int w = 0; w < WAVES; w++) total += s_count[w][tid];
    inc = total;
#pragma unroll
    for (int d = 1; d < GS_WAVE; d <<= 1) {
      const uint32_t o = __shfl_up(inc, d, GS_WAVE);
      if (lane >= d) inc += o;
    }
    if (lane == GS_WAVE - 1) s_scan[wave] = inc;
  }
  __syncthreads();
  if (tid < ORDER_BINS) {
    uint32_t run = inc - total;
    for (int w = 0; w < wave; w++) run += s_scan[w];
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
      const uint32_t n = s_count[w][tid];
      s_count[w][tid] = run;
      run += n;
    }
  }
  __syncthreads();
  order[(size_t)(s_count[wave][bin] + place) * gridDim.x + blockIdx.x] = leaf < nleaves ? (uint32_t)leaf : NO_LEAF;
}

// A node's bounding box: lo = minimum corner, hi = maximum corner.  An absent node is an inverted box, infinitely far
// from everything.
struct NodeBox {
  float lo[3], hi[3];
};

__device__ __forceinline__ NodeBox load_box(const float* __restrict__ bx, bool exists) {
  NodeBox n = {{FLT_MAX, FLT_MAX, FLT_MAX}, {-FLT_MAX, -FLT_MAX, -FLT_MAX}};
  if (exists) {
    const float2 a = *(const float2*)(bx), b = *(const float2*)(bx + 2), c = *(const float2*)(bx + 4);
    n.lo[0] = a.x; n.lo[1] = a.y; n.lo[2] = b.x;
    n.hi[0] = b.y; n.hi[1] = c.x; n.hi[2] = c.y;
  }
  return n;
}

// lane `from`'s box, in every lane (`from` is wave-uniform)
__device__ __forceinline__ NodeBox box_of_lane(const NodeBox& n, int from) {
  NodeBox r;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    r.lo[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, n.lo[k]), from));
    r.hi[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, n.hi[k]), from));
  }
  return r;
}

// Squared distance between two axis-aligned boxes (0 where they overlap), and between a point and a box
// (simple_knn.cu:119-129 for the latter): lower bounds of the distance between any point of the one and any point
// of the other, also as rounded here and in update3 (differences, squares and the two additions are monotone, and
// the additions associate the same way).
__device__ __forceinline__ float boxes_dist2(const float* q, const NodeBox& n) {
  float gap[3];
#pragma unroll
  for (int k = 0; k < 3; k++) gap[k] = fmaxf(0.f, fmaxf(n.lo[k] - q[3 + k], q[k] - n.hi[k]));
  return (gap[0] * gap[0] + gap[1] * gap[1]) + gap[2] * gap[2];
}

__device__ __forceinline__ float point_box_dist2(const float4& p, const NodeBox& n) {
  const float pc[3] = {p.x, p.y, p.z};
  float gap[3];
#pragma unroll
  for (int k = 0; k < 3; k++) gap[k] = fmaxf(0.f, fmaxf(n.lo[k] - pc[k], pc[k] - n.hi[k]));
  return (gap[0] * gap[0] + gap[1] * gap[1]) + gap[2] * gap[2];
}

// Keeps the three smallest of {knn[0..2], dist} in ascending order (simple_knn.cu:131-145 inserts by
// compare-and-swap; minimum and medians leave the same three values).  A distance that is infinite or larger than
// FLT_MAX changes nothing.
__device__ __forceinline__ void update3(const float dist, float* knn) {
  const float n0 = fminf(knn[0], dist);
  const float n1 = __builtin_amdgcn_fmed3f(knn[0], knn[1], dist);
  const float n2 = __builtin_amdgcn_fmed3f(knn[1], knn[2], dist);
  knn[0] = n0;
  knn[1] = n1;
  knn[2] = n2;
}

// The squared distance to the point that the lane N places back in the row holds.  The rotation is an operand modifier of
// the subtractions: no instructions of its own and no memory access.
template <int N>
__device__ __forceinline__ float row_dist2(const float4& p, const float4& c) {
  float dx, dy, dz;
  if constexpr (N == 0) {
    dx = c.x - p.x, dy = c.y - p.y, dz = c.z - p.z;
  } else {
    dx = row_ror<N>(c.x) - p.x, dy = row_ror<N>(c.y) - p.y, dz = row_ror<N>(c.z) - p.z;
  }
  return (dx * dx + dy * dy) + dz * dz;
}

// Every lane meets the points that the sixteen lanes of its row hold (from the FIRST-th one round; 1 leaves out the
// lane's own).
template <int FIRST, int LAST = KNN_TWIG>
__device__ __forceinline__ void meet_row(const float4& p, const float4& c, float* knn) {
  if constexpr (FIRST < LAST) {
    update3(row_dist2<FIRST>(p, c), knn);
    meet_row<FIRST + 1, LAST>(p, c, knn);
  }
}

// The same, four points at a time, for twigs that few lanes gain from: where none of the four is nearer than the third
// best of any lane there is nothing to keep (1 M points: 209 -> 191 us).
template <int FIRST = 0>
__device__ __forceinline__ void meet_row_of_few(const float4& p, const float4& c, float* knn) {
  if constexpr (FIRST < KNN_TWIG) {
    const float d0 = row_dist2<FIRST>(p, c), d1 = row_dist2<FIRST + 1>(p, c), d2 = row_dist2<FIRST + 2>(p, c),
                d3 = row_dist2<FIRST + 3>(p, c);
    if (gs_ballot(fminf(fminf(fminf(d0, d1), d2), d3) < knn[2]) != 0ull) {
      update3(d0, knn);
      update3(d1, knn);
      update3(d2, knn);
      update3(d3, knn);
    }
    meet_row_of_few<FIRST + 4>(p, c, knn);
  }
}

// simple-knn/simple_knn.cu:147-183.  The reference gives every point a thread that seeds a rejection radius from
// the point's neighbours in sorted order and then walks all boxes, skipping those farther away than that radius or
// than the third-best distance so far (simple_knn.cu:161-171).  Here a wave owns a leaf, 64 consecutive points
// along the curve, and each of its four rows of sixteen lanes a twig of it:
//   * every point first meets the points of its own twig and of the SEED twigs on either side of it along the curve,
//     which gives it a third-best distance to start from;
//   * 64 nodes of a level (groups of boxes, boxes, twigs) are tested in one step, a lane each: groups and boxes
//     against the leaf's bounding box and the largest third-best distance of the wave, the twigs of a box against
//     each row's own bounding box and largest third-best distance; a box or twig that passes is then tested by every
//     lane for its own point and its own third-best distance, the reference's test, and opened by the rows (a box:
//     by the wave) that have a lane which needs it (the first test alone would open everything between the two ends
//     of a leaf whose points lie in two places, where the curve leaves the occupied part of the grid and comes back
//     elsewhere);
//   * every row then walks its own list of twigs, its sixteen lanes holding the sixteen points, the next twig's
//     points on their way meanwhile.
// A lane then also sees points that its own test would have skipped; only true distances are ever inserted, and
// nothing nearer than a point's third-best distance is ever skipped, so the three distances are those of a
// brute-force search whatever the order.
// Bound by vector issue.  With the whole leaf as the unit that opens twigs (64 points against every point of the
// three leaves around it and of the twigs any of them needs, over LDS) the search took 335 us for 1 M points of an
// SfM-like cloud; with the row as the unit 298 us, 265 us with a workgroup per wave, whose place is taken as soon
// as that wave ends (a leaf among sparse points takes ten times as long as the median), and 209 us with the leaves in
// falling order of their size (4 M points, the whole call: 1150 -> 1060 us; 600 k: 282 -> 246).
constexpr int SEED = 2;

__global__ void __launch_bounds__(GS_WAVE) box_mean_dist_kernel(int P, const float4* __restrict__ sorted_pts,
                                                                    const uint32_t* __restrict__ idx,
                                                                    const float* __restrict__ boxes, int nboxes,
                                                                    const float* __restrict__ groups,
                                                                    const float* __restrict__ leaves,
                                                                    const float* __restrict__ twigs,
                                                                    const uint32_t* __restrict__ order,
                                                                    float* __restrict__ out) {
  constexpr int TWIGS_PER_BOX = KNN_BOX / KNN_TWIG, ROWS = KNN_LEAF / KNN_TWIG;
  static_assert(TWIGS_PER_BOX == GS_WAVE && KNN_GROUP == GS_WAVE, "a lane tests one node of a level");
  const int lane = threadIdx.x, row = lane / KNN_TWIG, in_row = lane % KNN_TWIG;
  const uint32_t taken = order != nullptr ? order[blockIdx.x] : blockIdx.x;
  if (taken == NO_LEAF) return;
  const int own = (int)taken;  // this wave's leaf
  const int k = own * KNN_LEAF + lane;
  const int ntwigs = (P + KNN_TWIG - 1) / KNN_TWIG;
  const float4 nowhere = make_float4(__builtin_inff(), __builtin_inff(), __builtin_inff(), 0.f);
  // the row's lanes fetch the points of twig t; a lane without a point (t < 0: no twig) holds one that is infinitely
  // far away, and so does one whose point has a NaN coordinate (a NaN distance is never inserted, as with the
  // reference's `knn[j] > dist`)
  auto points_of = [&](int t) {
    const int at = t * KNN_TWIG + in_row;
    return t >= 0 && at < P ? sorted_pts[at] : nowhere;
  };
  auto without_nan = [&](float4 c) {
    return c.x == c.x && c.y == c.y && c.z == c.z ? c : nowhere;
  };
  const float4 p = k < P ? sorted_pts[k] : nowhere;
  // a point with a non-finite coordinate has no finite distance to anything: its result never changes
  const bool searching = fabsf(p.x) < __builtin_inff() && fabsf(p.y) < __builtin_inff() &&
                         fabsf(p.z) < __builtin_inff();
  float best[3] = {FLT_MAX, FLT_MAX, FLT_MAX};

  // The row's own twig and those before and after it along the curve come first, unconditionally: they hold most of
  // the neighbours, and the third-best distance they leave is the bound for everything that follows (the reference
  // seeds its rejection radius from a point's neighbours in sorted order too, simple_knn.cu:153-160).
  {
    const int t = own * ROWS + row;
    float4 seed[2 * SEED];
#pragma unroll
    for (int s = 0; s < 2 * SEED; s++) {
      const int other = t + (s < SEED ? s - SEED : s - SEED + 1);
      seed[s] = points_of(other < ntwigs ? other : -1);
    }
    meet_row<1>(p, without_nan(p), best);
#pragma unroll 1
    for (int s = 0; s < 2 * SEED; s++) meet_row<0>(p, without_nan(seed[s]), best);
  }

  float q[6];  // the leaf's bounding box
#pragma unroll
  for (int c = 0; c < 6; c++) q[c] = leaves[6 * (size_t)own + c];
  NodeBox row_box[ROWS];  // the twigs'
#pragma unroll
  for (int r = 0; r < ROWS; r++) row_box[r] = load_box(twigs + 6 * (size_t)(own * ROWS + r), own * ROWS + r < ntwigs);
  // (a margin of a few units in the last place: the node test and the point distances round differently)
  constexpr float MARGIN = 1.0f + 0x1p-20f;
  float row_reach[ROWS], reach;  // wave-uniform
  auto update_reach = [&] {
    const float m = row_max(searching ? best[2] : 0.f) * MARGIN;
    reach = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      row_reach[r] = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, m), r * KNN_TWIG));
      reach = fmaxf(reach, row_reach[r]);
    }
  };
  update_reach();

  const int own_box = own / (KNN_BOX / KNN_LEAF);
  const uint64_t searching_m = gs_ballot(searching);
  // which lanes need a node, by the reference's test (simple_knn.cu:161-171) for their own points?
  auto needing = [&](const NodeBox& n) { return searching_m & gs_ballot(!(point_box_dist2(p, n) > best[2])); };
  auto open_box = [&](int b) {
    const int t = b * TWIGS_PER_BOX + lane;
    const NodeBox mine_t = load_box(twigs + 6 * (size_t)t, t < ntwigs);
    uint64_t near[ROWS], any = 0ull;
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      const float qr[6] = {row_box[r].lo[0], row_box[r].lo[1], row_box[r].lo[2],
                           row_box[r].hi[0], row_box[r].hi[1], row_box[r].hi[2]};
      near[r] = gs_ballot(!(boxes_dist2(qr, mine_t) > row_reach[r]));
      // (the twigs met at the start are not met again)
      const int met = own * ROWS + r - SEED - b * TWIGS_PER_BOX;
      const int met_lo = max(met, 0), met_hi = min(met + 2 * SEED + 1, TWIGS_PER_BOX);
      if (met_lo < met_hi) near[r] &= ~(((1ull << (met_hi - met_lo)) - 1ull) << met_lo);
      any |= near[r];
    }
    if (any == 0ull) return;
    const uint64_t row_near = row == 0 ? near[0] : row == 1 ? near[1] : row == 2 ? near[2] : near[3];
    // the row's list, one bit per twig of the box
    uint64_t todo = 0ull;
    while (any != 0ull) {
      const int c = (int)__builtin_ctzll(any);
      any &= any - 1ull;
      const uint64_t need = needing(box_of_lane(mine_t, c));
      const bool row_needs = ((uint32_t)(need >> (row * KNN_TWIG)) & 0xFFFFu) != 0u;
      todo |= row_needs ? 1ull << c : 0ull;
    }
    todo &= row_near;
    auto next = [&] {
      const int c = todo != 0ull ? b * TWIGS_PER_BOX + (int)__builtin_ctzll(todo) : -1;
      todo &= todo - 1ull;
      return points_of(c);
    };
    uint64_t left = gs_ballot(todo != 0ull);
    float4 ahead = nowhere;
    if (left != 0ull) ahead = next();
    while (left != 0ull) {
      const float4 c = without_nan(ahead);
      left = gs_ballot(todo != 0ull);
      if (left != 0ull) ahead = next();
      meet_row_of_few(p, c, best);
    }
    update_reach();
  };

  open_box(own_box);
  const int ngroups = (nboxes + KNN_GROUP - 1) / KNN_GROUP;
  for (int g0 = 0; g0 < ngroups; g0 += GS_WAVE) {
    const int g = g0 + lane;
    uint64_t gm = gs_ballot(!(boxes_dist2(q, load_box(groups + 6 * (size_t)g, g < ngroups)) > reach));
    while (gm != 0ull) {
      const int gi = g0 + (int)__builtin_ctzll(gm);
      gm &= gm - 1ull;
      const int b = gi * KNN_GROUP + lane;
      const NodeBox mine_b = load_box(boxes + 6 * (size_t)b, b < nboxes);
      uint64_t bm = gs_ballot(!(boxes_dist2(q, mine_b) > reach));
      if (gi == own_box / KNN_GROUP) bm &= ~(1ull << (own_box % KNN_GROUP));
      while (bm != 0ull) {
        const int c = (int)__builtin_ctzll(bm);
        bm &= bm - 1ull;
        if (needing(box_of_lane(mine_b, c)) != 0ull) open_box(gi * KNN_GROUP + c);
      }
    }
  }
  if (!searching) best[0] = best[1] = best[2] = FLT_MAX;  // (what NaN differences left there)
  if (k < P) out[idx[k]] = ((best[0] + best[1]) + best[2]) / 3.0f;
}

}  // namespace

size_t knn_temp_bytes(int P) { return knn_layout(P).total; }

int launch_knn_dist2(int P, const float* points, float* mean_dist2, void* temp, uint32_t* fault_word,
                     hipStream_t stream) {
  if (P <= 0) return 0;
  const KnnLayout L = knn_layout(P);
  char* base = (char*)temp;
  float* partial = (float*)(base + L.partial);
  uint32_t* codes_a = (uint32_t*)(base + L.codes_a);
  uint32_t* codes_b = (uint32_t*)(base + L.codes_b);
  uint32_t* idx_a = (uint32_t*)(base + L.idx_a);
  uint32_t* idx_b = (uint32_t*)(base + L.idx_b);
  float4* sorted_pts = (float4*)(base + L.sorted_pts);
  float* boxes = (float*)(base + L.boxes);
  float* groups = (float*)(base + L.groups);
  float* leaves = (float*)(base + L.leaves);
  float* twigs = (float*)(base + L.twigs);
  const int segments = order_segments(P);
  uint32_t* order = segments > 0 ? (uint32_t*)(base + L.order) : nullptr;
  void* sort_temp = base + L.sort_temp;
  const int nboxes = (P + KNN_BOX - 1) / KNN_BOX;
  const int key_bits = P <= KEY_SHORT_MAX ? KEY_SHORT_BITS : KEY_BITS;
  const auto key_kernel = P <= KEY_SHORT_MAX ? curve_key_kernel<KEY_SHORT_BITS> : curve_key_kernel<KEY_BITS>;

  // (the per-phase scopes only record events while stage timing is enabled)
  {
    StageScope _t("knn_minmax", stream);
    hipLaunchKernelGGL(minmax_partial_kernel, dim3(MM_BLOCKS), dim3(MM_THREADS), 0, stream, P, points, partial,
                       sort_clear_words(P, key_bits), (uint32_t*)sort_temp);
  }
  {
    StageScope _t("knn_keys", stream);
    const int key_blocks = (P + KEY_THREADS - 1) / KEY_THREADS;
    hipLaunchKernelGGL(key_kernel, dim3(key_blocks < KEY_BLOCKS ? key_blocks : KEY_BLOCKS), dim3(KEY_THREADS), 0,
                       stream, P, points, partial, codes_a, idx_a, (uint32_t*)sort_temp);
  }
  {
    StageScope _t("knn_sort", stream);
    if (launch_sort_pairs_u32(P, codes_a, codes_b, idx_a, idx_b, key_bits, sort_temp, stream, true)) return 1;
  }
  const uint32_t* idx_sorted = sort_result_in_b(key_bits) ? idx_b : idx_a;
  {
    StageScope _t("knn_boxes", stream);
    hipLaunchKernelGGL(gather_boxes_kernel, dim3(nboxes), dim3(KNN_BOX), 0, stream, P, points, idx_sorted, sorted_pts,
                       boxes, leaves, twigs);
    // (a wave per group of boxes, of which the parts to order have plenty: a group is 1024 leaves, a part has 16 waves)
    const int group_blocks = ((nboxes + KNN_GROUP - 1) / KNN_GROUP + ORDER_THREADS / GS_WAVE - 1) / (ORDER_THREADS / GS_WAVE);
    hipLaunchKernelGGL(box_group_kernel, dim3(segments > 0 ? segments : group_blocks), dim3(ORDER_THREADS), 0, stream,
                       nboxes, boxes, groups, (P + KNN_LEAF - 1) / KNN_LEAF, leaves, order, sort_error_word(sort_temp),
                       fault_word);
  }
  {
    StageScope _t("knn_box_mean_dist", stream);
    hipLaunchKernelGGL(box_mean_dist_kernel, dim3(segments > 0 ? segments * ORDER_THREADS : (P + KNN_LEAF - 1) / KNN_LEAF),
                       dim3(GS_WAVE), 0, stream, P, sorted_pts, idx_sorted, boxes, nboxes, groups, leaves, twigs, order,
                       mean_dist2);
  }
  return 0;
}

}  // namespace gs
