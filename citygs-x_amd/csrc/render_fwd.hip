// Per-tile front-to-back alpha blending (cuda_rasterizer/forward.cu:264-437)
// with the per-tile statistics of cuda_rasterizer/rasterizer_impl.cu:219-262
// folded into the same kernel.
//
// One 256-thread workgroup per 16x16 tile; each 64-lane wave owns an 8x8
// quadrant and each 16-lane row of a wave a 4x4 pixel block.  The tile's
// depth-sorted Gaussians are staged through LDS in batches of 256 (centre,
// conic, opacity, the limit of the marks, colour, the five geometry channels
// and the blocks touched).
// The thread that stages a Gaussian tests which of the tile's sixteen 4x4 blocks its alpha >= 1/255 ellipse (slightly
// inflated) can reach; the sixteen bits are also left for the backward pass.  Per batch a wave compacts, for each of
// its four rows, the slot numbers of those that reach the row's block into a byte list in LDS (a lane's
// place in the list is the number of hits in the lanes below it).  A pixel
// blends about a quarter of its block's list, so the lists are walked 32
// entries at a time in two steps: every lane marks, one bit per entry, the
// entries that can reach its own pixel (a fused quadratic form against a
// limit, eleven instructions an entry), then blends its marked entries in
// order, the k-th marked one in pass k, whichever entry that is for the other
// lanes; a chunk takes as many blend passes as its busiest pixel has marks.
// Pixels keep their own front-to-back order, which is all the blend needs.
// A row stops when its 16 pixels have saturated; a batch is not fetched once
// all have.
// Registers decide how many waves a SIMD holds here (80 allow six), and a
// kernel that spills to scratch memory starts its waves much more slowly, so
// index arithmetic is kept from being hoisted across the blend loop.
// What bounds it: the vector ALU (about 0.8 busy; additions, multiplications, fused multiply-adds, moves and bitwise
// operations of vector registers take two cycles a wave here, everything else four) and the LDS pipe (0.5).  So a blend
// works on -2 times the exponent (one constant less a pass), its tests are lane masks combined in scalar registers, and
// what a pass counts it counts under the mask: 57 vector instructions a pass where there were 71, and a block test per
// staged Gaussian where every wave made its own.  1 M Gaussians, 1152x864: 98 -> 94 us, 4 M from the air 279 -> 262, 20 M
// 660 -> 643, 300 k without geometry channels 59.5 -> 57.
//
// A tile's workgroup takes some 31 ns an entry whatever else the chip does: the chain of its waves' own instructions.  A
// view whose lists differ much in length ended on a few such chains (4 M Gaussians from the air, lists up to 9600: 293 us,
// in the last 150 of which less than a quarter of the chip had work; wave priorities change nothing).  Long tiles (which:
// GS_LONG_TILE) therefore go to four workgroups, one per quadrant, whose waves have 16 pixels instead of 64 and four lanes for each
// (blend_quadrant): 4.4 us per 256 entries instead of 8, for about 1.45 times the instructions of a tile.
// 4 M, 1152x864: 263 -> 196 us; 20 M from 600 m, lists up to 69 000, of which 0.4 is walked: 643 -> 408.
//
// The per-pixel arithmetic keeps a fixed operation order, so contributor
// counts and images match a CPU evaluation bit for bit; exp() is gs_expf.
// out_observe increments are counted per lane in LDS, a word per slot, and
// added once per (tile, Gaussian).
#include <type_traits>

#include "gs_common.h"
#include "gs_kernels.h"
#include "render_common.h"

namespace gs {

namespace {

constexpr int BATCH = GS_TILE_PIX;
// Tiles that four workgroups each may take, at most: the launch has three workgroups more for each of them, which do
// nothing where a view has fewer.
constexpr uint32_t LONG_TILES = 1024;
constexpr int CHUNK = 32;  // entries of a list marked, then blended, at a time: one bit each in a register

// The value itself, but opaque to the optimizer from here on: what is computed from it stays behind this point
// instead of being hoisted out of the batch loop, where every hoisted LDS address holds a register through the
// blend loop (the kernel has none to spare: one more costs a wave per SIMD, or scratch memory).
__device__ __forceinline__ int not_hoisted(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// The value that lane E of a quad (four neighbouring lanes) holds, in all four lanes.
template <int E>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), E * 0x55, 0xF, 0xF, true));
}
template <int E>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, E * 0x55, 0xF, 0xF, true);
}
// v of the lane whose number differs in bit 0 (in bit 1).
__device__ __forceinline__ uint32_t quad_xor1(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t quad_xor2(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);
}

// What a workgroup has in LDS (see the kernel).
template <bool RENDER_GEO>
struct BlendLds {
  float4 *geo0, *geo1, *col0, *col1;
  uint32_t *obs, *idx;
  uint16_t* hits;
  int *done, *bad;
};

// One quadrant of a long tile by a workgroup of its own: a wave has one 4x4 block, a quad of its lanes one pixel.  The
// four lanes of a pixel mark a quarter of a chunk each and blend the pixel's next four marked entries together: lane k has
// the exponent and alpha of entry k, all four the transmittance in front of every entry (a chain of four products), and
// lane k the sums of channels 2 k and 2 k + 1 (channel k where only the colour is rendered), in the order of the entries.
// Every number is formed by the operations the other way has, in its order: the same bits.
// Of packed records only.  Operands gathered from their arrays come five lines of memory to an entry, and four workgroups
// gather them four times: 10 M at street level whose records are not packed take 705 us unsplit, 810 split, and 860 with the
// gathers a batch ahead like the records here; the sparser of two such views 253, 258 and 258.
template <bool RENDER_GEO>
__device__ __forceinline__ void blend_quadrant(
    const BlendLds<RENDER_GEO> lds, uint32_t tile, uint32_t quadrant, uint32_t tile_x, uint32_t tile_y, uint2 range,
    const uint32_t* __restrict__ point_list, int W, int H, float fx, float fy, float cx, float cy, bool computed_here,
    const float* __restrict__ bg, float* __restrict__ final_T, uint32_t* __restrict__ n_contrib_px,
    uint32_t* __restrict__ n_contrib2loss_px, float* __restrict__ out_color, int* __restrict__ out_observe,
    float* __restrict__ out_all_map, float* __restrict__ out_plane_depth, int* __restrict__ n_render,
    int* __restrict__ n_consider, int* __restrict__ n_contrib_tile, uint32_t* __restrict__ block_hits,
    const float4* __restrict__ packed) {
  const int tid = threadIdx.x, lane = tid & (GS_WAVE - 1), wave = tid / GS_WAVE;
  const uint32_t k = (uint32_t)lane & 3u;
  const uint32_t x0 = tile_x * GS_TILE_X + 8u * (quadrant & 1u), y0 = tile_y * GS_TILE_Y + 8u * (quadrant >> 1);
  const uint32_t px = x0 + 4u * (uint32_t)(wave & 1) + ((uint32_t)lane >> 2 & 3u);
  const uint32_t py = y0 + 4u * (uint32_t)(wave >> 1) + ((uint32_t)lane >> 4);
  const bool inside = px < (uint32_t)W && py < (uint32_t)H;
  const int total = (int)(range.y - range.x);
  if (quadrant == 0u && tid == 0) n_render[tile] = total;
  if (!computed_here) {  // (as in the other way)
    const size_t HW = (size_t)H * W, pid = (size_t)W * py + px;
    if (inside && k == 0u) {
#pragma unroll
      for (int ch = 0; ch < GS_N_RGB; ch++) out_color[ch * HW + pid] = 0.f;
      if (RENDER_GEO) {
#pragma unroll
        for (int ch = 0; ch < GS_N_MAP; ch++) out_all_map[ch * HW + pid] = 0.f;
        out_plane_depth[pid] = 0.f;
      }
    }
    return;
  }
  const float pfx = (float)px, pfy = (float)py;
  uint64_t alive = gs_ballot(inside);  // pixels that still blend, four bits each
  constexpr int SUMS = RENDER_GEO ? 2 : 1;
  float T = 1.0f, C[SUMS];
  uint32_t last = 0, n2l = 0;  // of the entries this lane has blended
#pragma unroll
  for (int ch = 0; ch < SUMS; ch++) C[ch] = 0.f;
  const char* const my_channels =
      RENDER_GEO ? reinterpret_cast<const char*>(k < 2u ? lds.col0 : lds.col1) + 8u * (k & 1u)
                 : reinterpret_cast<const char*>(lds.col0) + 4u * k;
  uint8_t* const my_list = reinterpret_cast<uint8_t*>(lds.idx) + wave * BATCH;

  // The operands of a thread's slot are fetched a batch ahead, their Gaussian two.
  uint32_t g = tid < total ? point_list[range.x + (uint32_t)tid] : 0u;
  uint32_t g_next = tid + BATCH < total ? point_list[range.x + (uint32_t)(tid + BATCH)] : 0u;
  float4 r0, r1, r2;
  auto fetch = [&](uint32_t gaussian) {
    const float4* rec = packed + 4 * (size_t)gaussian;
    r0 = rec[0], r1 = rec[1], r2 = rec[2];
  };
  r0 = r1 = r2 = make_float4(0.f, 0.f, 0.f, 0.f);
  if (tid < total) fetch(g);
  for (int base = 0;; base += BATCH) {
    const int count = total - base < BATCH ? total - base : BATCH;
    bool finite = true;
    uint32_t hits = 0u;
    const int ts = not_hoisted(tid);
    if (ts < count) {
      auto stage = [&](const float2 xy, const float4 co, const float c0, const float c1, const float c2,
                       const float (&m)[GS_N_MAP]) {
        const float4 cp = block_test_params(co, xy, (float)(tile_x * GS_TILE_X), (float)(tile_y * GS_TILE_Y));
        lds.geo0[ts] = make_float4(xy.x, xy.y, co.x, co.y);
        lds.geo1[ts] = make_float4(0.25f * co.z, cp.w, co.z, -0.5f * co.w);
        float mag = fmaxf(fmaxf(fabsf(c0), fabsf(c1)), fabsf(c2));
        bool fin = c0 == c0 && c1 == c1 && c2 == c2;
        if (RENDER_GEO) {
#pragma unroll
          for (int ch = 0; ch < GS_N_MAP; ch++) {
            mag = fmaxf(mag, fabsf(m[ch]));
            fin = fin && m[ch] == m[ch];
          }
        }
        lds.col0[ts] = make_float4(c0, c1, c2, m[0]);
        if (RENDER_GEO) lds.col1[ts] = make_float4(m[1], m[2], m[3], m[4]);
        hits = ellipse_hits_quadrant(xy, co, cp.x, cp.y, cp.z, (float)x0, (float)y0);
        return fin && mag < __builtin_inff();
      };
      // (the last two words are on the line that the others came with)
      const float2 r3 = RENDER_GEO ? *reinterpret_cast<const float2*>(packed + 4 * (size_t)g + 3) : make_float2(0.f, 0.f);
      const float m[GS_N_MAP] = {r2.y, r2.z, r2.w, r3.x, r3.y};
      finite = stage(make_float2(r0.x, r0.y), make_float4(r0.z, r0.w, r1.x, r1.y), r1.z, r1.w, r2.x, m);
      if (block_hits != nullptr)
        reinterpret_cast<uint8_t*>(block_hits + range.x + (uint32_t)(base + ts))[quadrant] = (uint8_t)hits;
    }
    {
      const uint64_t bad_m = gs_ballot(!finite);
      if (lane == 0) lds.bad[wave] = bad_m != 0ull;
    }
    lds.obs[ts] = 0u;
    lds.hits[ts] = (uint16_t)hits;
    lds.idx[ts] = 0u;  // (a word of the four lists per thread; bytes behind a list's end are slot 0)
    __syncthreads();
    g = g_next;
    if (base + BATCH + tid < total) fetch(g);
    {
      const int tn = not_hoisted(tid) + base + 2 * BATCH;
      g_next = tn < total ? point_list[range.x + (uint32_t)tn] : 0u;
    }
    const bool select_blend = (lds.bad[0] | lds.bad[1] | lds.bad[2] | lds.bad[3]) != 0;

    if (alive != 0ull) {
      uint32_t len = 0u;
#pragma unroll
      for (int q = 0; q < BATCH / GS_WAVE; q++) {
        const int jj = q * GS_WAVE + (not_hoisted(tid) & (GS_WAVE - 1));
        const uint64_t b = gs_ballot(((uint32_t)lds.hits[jj] >> wave & 1u) != 0u);
        const uint32_t at = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, len));
        if (__builtin_amdgcn_inverse_ballot_w64(b)) my_list[at] = (uint8_t)jj;
        len += (uint32_t)__popcll(b);
      }
      len = (uint32_t)__builtin_amdgcn_readfirstlane((int)len);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      auto walk = [&](auto select_tag) {
        constexpr bool SELECT = decltype(select_tag)::value;
        const float pfy_m2 = -2.0f * pfy;
        for (uint32_t c0 = 0; c0 < len && alive != 0ull; c0 += CHUNK) {
          // lane k of a pixel marks entries 8 k .. 8 k + 7 of the chunk, the last one first
          uint32_t marks = 0u;
          const uint2 words = *reinterpret_cast<const uint2*>(my_list + c0 + 8u * k);
#pragma unroll
          for (int u = 7; u >= 0; u -= 2) {
            float form[2], limit[2];
#pragma unroll
            for (int v = 0; v < 2; v++) {
              const int e = u - v;
              const int j = (int)__builtin_amdgcn_ubfe(e >= 4 ? words.y : words.x, 8u * (e & 3), 8u);
              const float4 g0 = lds.geo0[j];
              const float2 g1 = *reinterpret_cast<const float2*>(&lds.geo1[j]);  // C / 4 and the mark limit
              const float dx = g0.x - pfx, dy2 = __builtin_fmaf(g0.y, 2.0f, pfy_m2);
              form[v] = __builtin_fmaf(g1.x * dy2, dy2, __builtin_fmaf(g0.z, dx, g0.w * dy2) * dx);
              limit[v] = g1.y;
            }
            shift_in_two(marks, form[0], limit[0], form[1], limit[1]);
          }
          marks <<= 8u * k;
          marks |= quad_xor1(marks);
          marks |= quad_xor2(marks);
          const uint32_t mine = len - c0;  // entries of the chunk that are in the list
          marks = mine >= (uint32_t)CHUNK ? marks : (marks & ((1u << mine) - 1u));
          marks = __builtin_amdgcn_inverse_ballot_w64(alive) ? marks : 0u;
          // the pixel's next four entries: lane k's is the k-th mark that is left
          auto take_four = [&](uint32_t& left) {
            const uint32_t m1 = left & (left - 1u), m2 = m1 & (m1 - 1u), m3 = m2 & (m2 - 1u);
            const uint32_t own = k == 0u ? left : (k == 1u ? m1 : (k == 2u ? m2 : m3));
            left = m3 & (m3 - 1u);
            return own;
          };
          uint32_t own_next = take_four(marks);
          uint32_t slot_next = my_list[c0 + (uint32_t)__builtin_ctz(own_next | 0x80000000u)];
          uint64_t marked = gs_ballot(own_next != 0u);
          while (marked != 0ull) {
            const uint32_t j = slot_next, at = j * 16u;
            const uint64_t has = marked;
            own_next = take_four(marks);
            slot_next = my_list[c0 + (uint32_t)__builtin_ctz(own_next | 0x80000000u)];
            const float4 g0 = lds.geo0[j];
            const float2 g1 = *(reinterpret_cast<const float2*>(&lds.geo1[j]) + 1);  // C and -opacity / 2
            float c[4][SUMS];
            auto channels = [&](auto e_tag) {
              constexpr int e = decltype(e_tag)::value;
              const float* p = reinterpret_cast<const float*>(my_channels + quad_lane<e>(at));
              if constexpr (RENDER_GEO) {
                const float2 two = *reinterpret_cast<const float2*>(p);
                c[e][0] = two.x, c[e][SUMS - 1] = two.y;
              } else {
                c[e][0] = *p;
              }
            };
            channels(std::integral_constant<int, 0>{});
            channels(std::integral_constant<int, 1>{});
            channels(std::integral_constant<int, 2>{});
            channels(std::integral_constant<int, 3>{});
            const float form = gauss_form(g0.z, g0.w, g1.x, g0.x - pfx, g0.y - pfy);
            float alpha = fminf(0.99f, g1.y * gs_neg2_exp_of_form(form));
            uint64_t counts = has & gs_ballot(!(form < 0.0f)) & gs_ballot(!(form > GS_FORM_MAX)) &
                              gs_ballot(!(alpha < 1.0f / 255.0f));
            // (an entry that does not count is blended with alpha 0, which changes nothing)
            alpha = __builtin_amdgcn_inverse_ballot_w64(counts) ? alpha : 0.f;
            const float oma = 1 - alpha;
            const float T1 = T * quad_lane<0>(oma), T2 = T1 * quad_lane<1>(oma), T3 = T2 * quad_lane<2>(oma);
            float T4 = T3 * quad_lane<3>(oma);
            const float before = k == 0u ? T : (k == 1u ? T1 : (k == 2u ? T2 : T3));
            const uint64_t stops = gs_ballot(T4 < 0.0001f);  // (a pixel that has stopped before keeps a T above)
            if (stops != 0ull) {
              // the first entry that takes a pixel's transmittance below the limit is not blended, nor what is behind it
              const bool over = before * oma < 0.0001f;
              counts &= ~gs_ballot(over);
              alpha = over ? 0.f : alpha;
              T4 = !(T4 < 0.0001f) ? T4 : !(T3 < 0.0001f) ? T3 : !(T2 < 0.0001f) ? T2 : !(T1 < 0.0001f) ? T1 : T;
              alive &= ~stops;
              marks = __builtin_amdgcn_inverse_ballot_w64(stops) ? 0u : marks;
              own_next = __builtin_amdgcn_inverse_ballot_w64(stops) ? 0u : own_next;
            }
            const float w[4] = {quad_lane<0>(alpha) * T, quad_lane<1>(alpha) * T1, quad_lane<2>(alpha) * T2,
                                quad_lane<3>(alpha) * T3};
            T = T4;
            if (__builtin_amdgcn_inverse_ballot_w64(counts)) {
              if (before > 0.5f) atomicAdd(&lds.obs[j], 1u);
              last = (uint32_t)(base + 1) + j;
              n2l++;
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma unroll
              for (int ch = 0; ch < SUMS; ch++) {
                const float sum = __builtin_fmaf(c[e][ch], w[e], C[ch]);
                C[ch] = (!SELECT || w[e] != 0.f) ? sum : C[ch];  // (a weight that counts is at least 1e-4 / 255)
              }
            }
            marked = gs_ballot(own_next != 0u);
          }
        }
      };
      if (select_blend) walk(std::true_type{});
      else walk(std::false_type{});
    }
    if (lane == 0) lds.done[wave] = alive == 0ull;
    __syncthreads();
    const int tf = not_hoisted(tid);
    if (tf < count) {
      const uint32_t seen = lds.obs[tf];
      if (seen != 0u) atomicAdd(&out_observe[point_list[range.x + (uint32_t)(base + tf)]], (int)seen);
    }
    if (base + BATCH >= total || (lds.done[0] && lds.done[1] && lds.done[2] && lds.done[3])) break;
  }

  const size_t HW = (size_t)H * W, pid = (size_t)W * (uint32_t)pfy + (uint32_t)pfx;
  // what the four lanes of a pixel have counted
  last = max(last, quad_xor1(last));
  last = max(last, quad_xor2(last));
  n2l += quad_xor1(n2l);
  n2l += quad_xor2(n2l);
  if (inside && k == 0u) {
    final_T[pid] = T;
    n_contrib_px[pid] = last;
    n_contrib2loss_px[pid] = n2l;
  }
  if constexpr (RENDER_GEO) {
    // (lanes 0 .. 3: red and green; blue and channel 0; channels 1 and 2; channels 3 and 4)
    const float m0 = quad_lane<1>(C[1]), m1 = quad_lane<2>(C[0]), m2 = quad_lane<2>(C[SUMS - 1]);
    const float m4 = quad_lane<3>(C[SUMS - 1]);
    if (inside) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const uint32_t ch = 2u * k + (uint32_t)h;
        if (ch < GS_N_RGB) out_color[ch * HW + pid] = C[h] + T * bg[ch];
        else out_all_map[(ch - GS_N_RGB) * HW + pid] = C[h];
      }
      if (k == 3u) {
        const float rayx = (pfx - cx) / fx, rayy = (pfy - cy) / fy;
        const float den_f = (m0 * rayx + m1 * rayy) + m2;
        out_plane_depth[pid] = (float)((double)m4 / -((double)den_f + 1.0e-8));
      }
    }
  } else {
    if (inside && k < GS_N_RGB) out_color[k * HW + pid] = C[0] + T * bg[k];
  }
  // per-tile integer sums of the two per-pixel counters; the tile's four workgroups add up
  int a = inside && k == 0u ? (int)last : 0, b = inside && k == 0u ? (int)n2l : 0;
#pragma unroll
  for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
    a += __shfl_xor(a, d, GS_WAVE);
    b += __shfl_xor(b, d, GS_WAVE);
  }
  if (lane == 0) {
    atomicAdd(&n_consider[tile], a);
    atomicAdd(&n_contrib_tile[tile], b);
  }
}

// MAX_DEPTH adds one output with no counterpart in the reference: per pixel, the view-space depth of the Gaussian
// that blends with the largest weight alpha * T (the front-most one among equals; 0 where nothing blends).  It
// leaves every other output as it is.
// LONG: the first tiles of the order are split as far as they are long; the operands are packed, the order is there.
template <bool RENDER_GEO, bool MAX_DEPTH, bool LONG>
__global__ void __launch_bounds__(GS_TILE_PIX) __attribute__((amdgpu_waves_per_eu(MAX_DEPTH ? 5 : 6)))
render_fwd_kernel(const uint2* __restrict__ ranges, const uint32_t* __restrict__ point_list, int W, int H, float fx,
                  float fy, float cx, float cy, const float2* __restrict__ means2D, const float* __restrict__ rgb,
                  const float* __restrict__ all_map, const float4* __restrict__ conic_opacity,
                  const uint8_t* __restrict__ compute_locally, const float* __restrict__ bg,
                  float* __restrict__ final_T, uint32_t* __restrict__ n_contrib_px,
                  uint32_t* __restrict__ n_contrib2loss_px, float* __restrict__ out_color,
                  int* __restrict__ out_observe, float* __restrict__ out_all_map,
                  float* __restrict__ out_plane_depth, int* __restrict__ n_render, int* __restrict__ n_consider,
                  int* __restrict__ n_contrib_tile, const float* __restrict__ depths,
                  float* __restrict__ out_max_weight_depth, const uint32_t* __restrict__ fits_word,
                  uint32_t* __restrict__ block_hits, const float4* __restrict__ packed,
                  const uint32_t* __restrict__ tile_order, const uint32_t* __restrict__ order_word, uint32_t long_cap,
                  uint32_t tiles, uint32_t tiles_x) {
  constexpr bool render_geo = RENDER_GEO;
  // launched ahead of the host's decision on how the per-tile lists are built: nothing to do if they were not
  uint32_t tile, long_tiles = 0u;
  if constexpr (LONG) {
    // (asked for together: one memory latency instead of three)
    uint32_t fits = 1u;
    if (fits_word != nullptr) fits = *fits_word;
    long_tiles = *order_word - 1u;
    tile = tile_order[blockIdx.x < tiles ? blockIdx.x : 0u];
    asm volatile("" : "+s"(fits), "+s"(long_tiles), "+s"(tile));
    if (fits == 0u) return;
  } else {
    if (fits_word != nullptr && *fits_word == 0u) return;
    tile = tile_order != nullptr ? tile_order[blockIdx.x] : blockIdx.x;
  }
  __shared__ float s_depth[MAX_DEPTH ? BATCH : 1];
  // a slot's geometry, (x, y, A, B) and (C / 4, mark limit, C, -opacity / 2), and its channels, (r, g, b, map0)
  // and (map1 .. map4), in four arrays of 16-byte elements: one address per slot serves them all, and lanes
  // that read different slots spread over all the banks
  __shared__ float4 s_geo0[BATCH];
  __shared__ float4 s_geo1[BATCH];
  __shared__ float4 s_col0[BATCH];
  __shared__ float4 s_col1[RENDER_GEO ? BATCH : 1];
  __shared__ uint32_t s_obs[BATCH];  // observation counts of the slots
  // the four rows' lists of every wave: the slots of the batch that can touch the row's block, one byte each, in
  // depth order; bytes behind a list's end are 0
  __shared__ __attribute__((aligned(16))) uint32_t s_idx[GS_TILE_PIX / GS_WAVE][4][BATCH / 4];
  // which of the tile's sixteen blocks a slot's Gaussian can touch: bits 4 w .. 4 w + 3 are the rows of wave w
  __shared__ uint16_t s_hits[BATCH];
  __shared__ int s_done[GS_TILE_PIX / GS_WAVE];
  __shared__ int s_bad[GS_TILE_PIX / GS_WAVE];
  __shared__ int s_red[2][GS_TILE_PIX / GS_WAVE];

  const int tid = threadIdx.x;
  // The first tiles of the order, as many as are long (rounded up to whole groups of eight), take four workgroups each:
  // the four of a tile on one XCD, whose L2 they share the records in.
  if constexpr (LONG) {
    const uint32_t split = min((long_tiles + 7u) & ~7u, long_cap);
    if (blockIdx.x < 4u * split) {
      const uint32_t quadrant = blockIdx.x / 8u & 3u;
      tile = tile_order[blockIdx.x / 32u * 8u + blockIdx.x % 8u];
      const uint32_t ty = tile / tiles_x;
      const BlendLds<RENDER_GEO> lds = {s_geo0, s_geo1, s_col0, s_col1, s_obs, &s_idx[0][0][0], s_hits, s_done, s_bad};
      blend_quadrant<RENDER_GEO>(lds, tile, quadrant, tile - ty * tiles_x, ty, ranges[tile], point_list, W, H, fx, fy, cx,
                                 cy, compute_locally[tile] != 0, bg, final_T, n_contrib_px, n_contrib2loss_px, out_color,
                                 out_observe, out_all_map, out_plane_depth, n_render, n_consider, n_contrib_tile,
                                 block_hits, packed);
      return;
    }
    if (blockIdx.x - 3u * split >= tiles) return;
    if (split != 0u) tile = tile_order[blockIdx.x - 3u * split];
  }
  const uint32_t tile_y = tile / tiles_x, tile_x = tile - tile_y * tiles_x;
  const RowThread rt = row_thread(tile_x, tile_y);
  const int lane = rt.lane, wave = rt.wave, row = rt.row;
  const uint2 range = ranges[tile];
  if (tid == 0) n_render[tile] = (int)(range.y - range.x);
  const uint32_t px = rt.px, py = rt.py;
  const bool inside = px < (uint32_t)W && py < (uint32_t)H;
  if (!compute_locally[tile]) {
    // A tile that is not computed here reads zero in every image, as in the reference, whose binding
    // allocates the images zero-filled (rasterize_points.cu:303-307) and whose kernel returns before writing.
    if (inside) {
      const size_t HW = (size_t)H * W, pid = (size_t)W * py + px;
#pragma unroll
      for (int ch = 0; ch < GS_N_RGB; ch++) out_color[ch * HW + pid] = 0.f;
      if (render_geo) {
#pragma unroll
        for (int ch = 0; ch < GS_N_MAP; ch++) out_all_map[ch * HW + pid] = 0.f;
        out_plane_depth[pid] = 0.f;
      }
      if (MAX_DEPTH) out_max_weight_depth[pid] = 0.f;
    }
    if (tid == 0) {
      n_consider[tile] = 0;
      n_contrib_tile[tile] = 0;
    }
    return;
  }
  const float pfx = (float)px, pfy = (float)py;
  // pixels that still blend, as a lane mask (wave-uniform, so it lives in scalar registers)
  uint64_t alive = gs_ballot(inside);
  const int row_shift = 16 * row;

  int todo = (int)(range.y - range.x);
  const int rounds = (todo + BATCH - 1) / BATCH;

  float T = 1.0f;
  uint32_t last = 0, n2l = 0;
  float C[GS_N_RGB] = {0.f, 0.f, 0.f};
  float Mp[GS_N_MAP] = {0.f, 0.f, 0.f, 0.f, 0.f};
  float best_w = 0.f, best_depth = 0.f;

  // (the Gaussian of a thread's slot is fetched one batch ahead: the operands' address is known when a batch starts)
  uint32_t g_next = tid < todo ? point_list[range.x + (uint32_t)tid] : 0u;
  for (int i = 0; i < rounds; i++, todo -= BATCH) {
    const uint64_t alive_mask = alive;
    if (lane == 0) s_done[wave] = alive_mask == 0ull;
    __syncthreads();
    if (s_done[0] && s_done[1] && s_done[2] && s_done[3]) break;

    const int count = todo < BATCH ? todo : BATCH;
    // A lane for which a Gaussian does not count blends it with weight 0, which is exact as long as the
    // Gaussian's colour and geometry channels are finite; a batch that holds a non-finite one is walked by
    // the variant of the loop that selects instead (below).
    bool finite = true;
    uint32_t hits = 0u;
    const int ts = not_hoisted(tid);
    const uint32_t g = g_next;
    if (ts + BATCH < todo) g_next = point_list[range.x + (uint32_t)(i + 1) * BATCH + ts];
    if (ts < count) {
      // A Gaussian's operands: one 64-byte record where the caller had them packed (a single line of memory,
      // every byte of it used), else gathered from the five arrays.  (Each route loads and then stages by itself:
      // with the loaded values merged across the two routes the compiler splits the gathers into single words.)
      auto stage = [&](const float2 xy, const float4 co, const float c0, const float c1, const float c2,
                       const float (&m)[GS_N_MAP], const float depth_g) {
        // (the marking step evaluates the quadratic form with fused operations, the blend the exponent with one
        // rounding per operation: the mark limit's margin covers both, and the blend tests the exponent itself
        // again)
        uint32_t ox = tile_x * GS_TILE_X, oy = tile_y * GS_TILE_Y;
        asm volatile("" : "+s"(ox), "+s"(oy));  // (as in not_hoisted)
        const float tile_x0 = (float)ox, tile_y0 = (float)oy;
        const float4 cp = block_test_params(co, xy, tile_x0, tile_y0);
        s_geo0[ts] = make_float4(xy.x, xy.y, co.x, co.y);
        s_geo1[ts] = make_float4(0.25f * co.z, cp.w, co.z, -0.5f * co.w);
        float mag = fmaxf(fmaxf(fabsf(c0), fabsf(c1)), fabsf(c2));
        bool fin = c0 == c0 && c1 == c1 && c2 == c2;
        if (render_geo) {
#pragma unroll
          for (int ch = 0; ch < GS_N_MAP; ch++) {
            mag = fmaxf(mag, fabsf(m[ch]));
            fin = fin && m[ch] == m[ch];
          }
        }
        s_col0[ts] = make_float4(c0, c1, c2, m[0]);
        if constexpr (RENDER_GEO) s_col1[ts] = make_float4(m[1], m[2], m[3], m[4]);
        if (MAX_DEPTH) s_depth[ts] = depth_g;
        hits = ellipse_hits_tile(xy, co, cp.x, cp.y, cp.z, tile_x0, tile_y0);
        return fin && mag < __builtin_inff();
      };
      if (LONG || packed != nullptr) {
        const float4* rec = packed + 4 * (size_t)g;
        const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
        float m[GS_N_MAP] = {r2.y, r2.z, r2.w, 0.f, 0.f};
        float depth_g = 0.f;
        if (render_geo || MAX_DEPTH) {
          const float4 r3 = rec[3];
          m[3] = r3.x, m[4] = r3.y, depth_g = r3.z;
        }
        finite = stage(make_float2(r0.x, r0.y), make_float4(r0.z, r0.w, r1.x, r1.y), r1.z, r1.w, r2.x, m, depth_g);
      } else {
        const float2 xy = means2D[g];
        const float4 co = conic_opacity[g];
        const float c0 = rgb[3 * (size_t)g], c1 = rgb[3 * (size_t)g + 1], c2 = rgb[3 * (size_t)g + 2];
        float m[GS_N_MAP] = {0.f, 0.f, 0.f, 0.f, 0.f};
        if (render_geo) {
#pragma unroll
          for (int ch = 0; ch < GS_N_MAP; ch++) m[ch] = all_map[5 * (size_t)g + ch];
        }
        finite = stage(xy, co, c0, c1, c2, m, MAX_DEPTH ? depths[g] : 0.f);
      }
    }
    {
      const uint64_t bad_m = gs_ballot(!finite);
      if (lane == 0) s_bad[wave] = bad_m != 0ull;
    }
    s_obs[ts] = 0u;
    s_hits[ts] = (uint16_t)hits;
    // (for the backward pass; a row that has saturated lists nothing, and nothing behind a row's last contributor is
    // looked at there)
    if (block_hits != nullptr && ts < count) block_hits[range.x + (uint32_t)i * BATCH + ts] = hits_to_bytes(hits);
    static_assert(sizeof(s_idx) == 16 * GS_TILE_PIX, "four words of the lists per thread");
    *reinterpret_cast<uint4*>(&s_idx[0][0][0] + 4 * ts) = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const bool select_blend = (s_bad[0] | s_bad[1] | s_bad[2] | s_bad[3]) != 0;

    if (alive_mask != 0ull) {
      // Per-row lists.  A wave looks at 64 slots at a time, lane = slot: the lanes whose Gaussian can touch row
      // r's 4x4 block append their slot numbers to the row's list, in lane order (a lane's place is the number of
      // set bits below its own).
      uint32_t len0 = 0u, len1 = 0u, len2 = 0u, len3 = 0u;  // the lists' lengths (wave-uniform)
      const int tb = not_hoisted(tid);
      const int lane_b = tb & (GS_WAVE - 1), wave_b = tb / GS_WAVE;
#pragma unroll
      for (int k = 0; k < BATCH / GS_WAVE; k++) {
        if (k * GS_WAVE >= count) break;  // (the last batch of a list is rarely full)
        const int jj = k * GS_WAVE + lane_b;
        const uint32_t rows = (uint32_t)s_hits[jj] >> (4 * wave_b);
        uint64_t hit_m[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const bool row_alive = ((alive_mask >> (16 * r)) & 0xFFFFull) != 0ull;
          hit_m[r] = row_alive ? gs_ballot(((rows >> r) & 1u) != 0u) : 0ull;
        }
        auto list_row = [&](auto row_tag, const uint32_t len) {
          constexpr int r = decltype(row_tag)::value;
          const uint64_t b = hit_m[r];
          const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
          if (__builtin_amdgcn_inverse_ballot_w64(b))
            reinterpret_cast<uint8_t*>(&s_idx[0][0][0])[(uint32_t)((wave_b * 4 + r) * BATCH) + len + below] = (uint8_t)jj;
          return len + (uint32_t)__popcll(b);
        };
        len0 = list_row(std::integral_constant<int, 0>{}, len0);
        len1 = list_row(std::integral_constant<int, 1>{}, len1);
        len2 = list_row(std::integral_constant<int, 2>{}, len2);
        len3 = list_row(std::integral_constant<int, 3>{}, len3);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

      // SELECT: a lane that does not blend keeps its sums by a select instead of adding a product with weight 0
      // (0 * NaN and 0 * inf are NaN): the reference only lets a non-finite colour reach the pixels that blend
      // it (cuda_rasterizer/forward.cu:381-407).  Same bits for finite inputs.
      len0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)len0);
      len1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)len1);
      len2 = (uint32_t)__builtin_amdgcn_readfirstlane((int)len2);
      len3 = (uint32_t)__builtin_amdgcn_readfirstlane((int)len3);
      const uint32_t row_len = row == 0 ? len0 : (row == 1 ? len1 : (row == 2 ? len2 : len3));
      auto walk = [&, len0, len1, len2, len3, row_len](auto select_tag) {
      constexpr bool SELECT = decltype(select_tag)::value;
      uint32_t my_len = row_len;
      uint32_t passes = max(max(len0, len1), max(len2, len3));  // wave-uniform
      // Of a 4x4 block's list a single pixel blends about a quarter, so the lists are walked a chunk of 32 entries
      // at a time, in two steps.  First every lane marks, one bit per entry, the entries whose exponent lies in
      // its window (the cheap part of a blend: centre, conic, two comparisons).  Then each lane blends its own
      // marked entries in order, the k-th marked one in pass k, whichever entry that is for its neighbours: a
      // chunk takes as many passes as its busiest pixel has marks.  A pixel's entries keep their order, which is
      // all the blend needs.
      const uint8_t* const my_list = reinterpret_cast<const uint8_t*>(&s_idx[wave][row][0]);
      for (uint32_t base = 0; base < passes; base += CHUNK) {
        uint32_t marks = 0u;
        // (the marking step works on 2 dy and C / 4, so that the conic's B serves it and the blend as it is)
        float pfy_m2 = pfy;
        asm volatile("" : "+v"(pfy_m2));  // (as in not_hoisted)
        pfy_m2 *= -2.0f;
        const uint32_t words = min((uint32_t)CHUNK / 4u, (passes - base + 3u) / 4u);
        // (last entry first: a mark is shifted in at bit 0, as the carry of marks + marks, so entry e of the chunk
        // ends at bit e)
        for (int q = (int)words - 1; q >= 0; q--) {
          const uint32_t word = s_idx[wave][row][(base >> 2) + (uint32_t)q];  // (zero, slot 0, behind the list's end)
#pragma unroll
          for (int u = 3; u >= 0; u -= 2) {
            float form[2], limit[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
              const int j = (int)__builtin_amdgcn_ubfe(word, 8u * (u - k), 8u);
              const float4 g0 = s_geo0[j];
              const float2 g1 = *reinterpret_cast<const float2*>(&s_geo1[j]);  // C / 4 and the mark limit
              const float dx = g0.x - pfx, dy2 = __builtin_fmaf(g0.y, 2.0f, pfy_m2);
              form[k] = __builtin_fmaf(g1.x * dy2, dy2, __builtin_fmaf(g0.z, dx, g0.w * dy2) * dx);
              limit[k] = g1.y;
            }
            // marked unless the form exceeds the limit (so a NaN marks, as the blend's own tests let it through)
            shift_in_two(marks, form[0], limit[0], form[1], limit[1]);
          }
        }
        {
          const uint32_t mine = my_len > base ? my_len - base : 0u;  // entries of the chunk that are in the list
          marks = mine >= (uint32_t)CHUNK ? marks : (marks & ((1u << mine) - 1u));
          marks = __builtin_amdgcn_inverse_ballot_w64(alive) ? marks : 0u;
        }
        // (the slot of a lane's next marked entry is fetched one pass ahead; a lane without one has some other slot of
        // its list or slot 0, whose data are this batch's)
        uint32_t slot_next = my_list[base + ((uint32_t)__builtin_ctz(marks | 0x80000000u))];
        // (tested at the bottom: the ballot cannot be copied, so a loop tested at the top is not rotated and pays
        // a register copy per accumulator and pass)
        uint64_t marked = gs_ballot(marks != 0u);
        if (marked != 0ull) do {
          const uint32_t j = slot_next;
          marks &= marks - 1u;
          slot_next = my_list[base + ((uint32_t)__builtin_ctz(marks | 0x80000000u))];
          const float4 g0 = s_geo0[j];
          const float2 g1 = *(reinterpret_cast<const float2*>(&s_geo1[j]) + 1);  // C and -opacity / 2
          float c[GS_N_RGB + GS_N_MAP] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          {
            const float4 c0 = s_col0[j];
            c[0] = c0.x, c[1] = c0.y, c[2] = c0.z, c[3] = c0.w;
            if constexpr (RENDER_GEO) {
              const float4 c1 = s_col1[j];
              c[4] = c1.x, c[5] = c1.y, c[6] = c1.z, c[7] = c1.w;
            }
          }
          float depth_j = 0.f;
          if (MAX_DEPTH) depth_j = s_depth[j];

          const float form = gauss_form(g0.z, g0.w, g1.x, g0.x - pfx, g0.y - pfy);
          const float alpha = fminf(0.99f, g1.y * gs_neg2_exp_of_form(form));
          // the lanes whose entry counts: they have one in this pass, the exponent lies in the window and alpha reaches
          // 1/255 (a NaN passes: the reference blends it too).  Lane masks of single comparisons, combined in scalar
          // registers.
          const uint64_t counts = marked & gs_ballot(!(form < 0.0f)) & gs_ballot(!(form > GS_FORM_MAX)) &
                                  gs_ballot(!(alpha < 1.0f / 255.0f));
          const float test_T = T * (1 - alpha);
          const uint64_t saturated = gs_ballot(test_T < 0.0001f);
          const uint64_t blends = counts & ~saturated, stops = counts & saturated;
          const bool blend = __builtin_amdgcn_inverse_ballot_w64(blends);
          // weight once, then one fused multiply-add per channel; w == 0 where the entry does not blend
          float w = blend ? alpha * T : 0.f;
          asm("" : "+v"(w));  // (formed here, so that T can be replaced in place)
          if (blend) {
            // observation count of the entry: one for a lane that blends it with T > 0.5
            if (T > 0.5f) atomicAdd(&s_obs[j], 1u);
            T = test_T;
            last = (uint32_t)(i * BATCH + 1) + j;
            n2l++;
          }
          alive &= ~stops;
          marks = __builtin_amdgcn_inverse_ballot_w64(stops) ? 0u : marks;
#pragma unroll
          for (int ch = 0; ch < GS_N_RGB; ch++) {
            const float sum = __builtin_fmaf(c[ch], w, C[ch]);
            C[ch] = (!SELECT || blend) ? sum : C[ch];
          }
          if (render_geo) {
#pragma unroll
            for (int ch = 0; ch < GS_N_MAP; ch++) {
              const float sum = __builtin_fmaf(c[GS_N_RGB + ch], w, Mp[ch]);
              Mp[ch] = (!SELECT || blend) ? sum : Mp[ch];
            }
          }
          if (MAX_DEPTH) {
            const bool better = w > best_w;  // w is 0 for a lane that does not blend
            best_depth = better ? depth_j : best_depth;
            best_w = better ? w : best_w;
          }
          marked = gs_ballot(marks != 0u);
        } while (marked != 0ull);
        // a row whose 16 pixels have all saturated drops the rest of its list
        if (((uint32_t)(alive >> row_shift) & 0xFFFFu) == 0u) my_len = 0u;
        uint32_t left = 0u;
        if (((uint32_t)alive & 0xFFFFu) != 0u) left = len0;
        if (((uint32_t)(alive >> 16) & 0xFFFFu) != 0u) left = max(left, len1);
        if (((uint32_t)(alive >> 32) & 0xFFFFu) != 0u) left = max(left, len2);
        if (((uint32_t)(alive >> 48) & 0xFFFFu) != 0u) left = max(left, len3);
        passes = left;
      }
      };
      if (select_blend) walk(std::true_type{});
      else walk(std::false_type{});
    }
    __syncthreads();
    const int tf = not_hoisted(tid);
    if (tf < count) {
      const uint32_t c = s_obs[tf];
      if (c != 0u) atomicAdd(&out_observe[point_list[range.x + (uint32_t)i * BATCH + tf]], (int)c);
    }
  }

  if (inside) {
    const size_t HW = (size_t)H * W, pid = (size_t)W * (uint32_t)pfy + (uint32_t)pfx;
    final_T[pid] = T;
    n_contrib_px[pid] = last;
    n_contrib2loss_px[pid] = n2l;
#pragma unroll
    for (int ch = 0; ch < GS_N_RGB; ch++) out_color[ch * HW + pid] = C[ch] + T * bg[ch];
    if (render_geo) {
#pragma unroll
      for (int ch = 0; ch < GS_N_MAP; ch++) out_all_map[ch * HW + pid] = Mp[ch];
      const float rayx = (pfx - cx) / fx, rayy = (pfy - cy) / fy;
      const float den_f = (Mp[0] * rayx + Mp[1] * rayy) + Mp[2];
      out_plane_depth[pid] = (float)((double)Mp[4] / -((double)den_f + 1.0e-8));
    }
    if (MAX_DEPTH) out_max_weight_depth[pid] = best_depth;
  }

  // per-tile integer sums of the two per-pixel counters
  int a = inside ? (int)last : 0, b = inside ? (int)n2l : 0;
#pragma unroll
  for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
    a += __shfl_xor(a, d, GS_WAVE);
    b += __shfl_xor(b, d, GS_WAVE);
  }
  __syncthreads();
  const int te = not_hoisted(tid);
  if ((te & (GS_WAVE - 1)) == 0) {
    s_red[0][te / GS_WAVE] = a;
    s_red[1][te / GS_WAVE] = b;
  }
  __syncthreads();
  if (tid == 0) {
    n_consider[tile] = s_red[0][0] + s_red[0][1] + s_red[0][2] + s_red[0][3];
    n_contrib_tile[tile] = s_red[1][0] + s_red[1][1] + s_red[1][2] + s_red[1][3];
  }
}

}  // namespace

template <bool GEO, bool MAXD, bool LONG>
static void launch_render_fwd_variant(const RenderFwdArgs& a, uint32_t long_cap, hipStream_t stream) {
  const uint32_t gx = (a.W + GS_TILE_X - 1) / GS_TILE_X, gy = (a.H + GS_TILE_Y - 1) / GS_TILE_Y;
  hipLaunchKernelGGL((render_fwd_kernel<GEO, MAXD, LONG>), dim3(gx * gy + 3 * long_cap), dim3(GS_TILE_PIX), 0, stream,
                     (const uint2*)a.ranges, a.point_list, a.W, a.H, a.fx, a.fy, a.cx, a.cy, (const float2*)a.means2D, a.rgb,
                     a.all_map, (const float4*)a.conic_opacity, a.compute_locally, a.bg, a.final_T, a.n_contrib_px,
                     a.n_contrib2loss_px, a.out_color, a.out_observe, a.out_all_map, a.out_plane_depth, a.n_render,
                     a.n_consider, a.n_contrib_tile, a.depths, a.out_max_weight_depth, a.fits_word, a.block_hits,
                     (const float4*)a.packed, a.tile_order, a.tile_order_word, long_cap, gx * gy, gx);
}

// A view that may have long tiles (as far as the bound on its longest list says) and whose operands are packed has a kernel
// that splits them.  The others' is without: in one kernel the second way costs the first registers and its start three
// loads.  1 M Gaussians, 1152x864: 94.8 us with it, 92.7 without, rendering alone 100.6 and 97.9; 300 k, colour only, 55.7 and
// 54.5.
template <bool GEO>
static void launch_render_fwd_geo(const RenderFwdArgs& a, hipStream_t stream) {
  const uint32_t tiles = (uint32_t)((a.W + GS_TILE_X - 1) / GS_TILE_X) * (uint32_t)((a.H + GS_TILE_Y - 1) / GS_TILE_Y);
  const uint32_t long_cap = (tiles < LONG_TILES ? tiles : LONG_TILES) & ~7u;
  if (a.out_max_weight_depth != nullptr)
    launch_render_fwd_variant<GEO, true, false>(a, 0u, stream);
  else if (a.packed != nullptr && a.tile_order != nullptr && a.tile_order_word != nullptr && a.longest >= GS_LONG_TILE &&
           long_cap != 0u)
    launch_render_fwd_variant<GEO, false, true>(a, long_cap, stream);
  else
    launch_render_fwd_variant<GEO, false, false>(a, 0u, stream);
}

int launch_render_fwd(const RenderFwdArgs& a, hipStream_t stream) {
  if (a.render_geo) launch_render_fwd_geo<true>(a, stream);
  else launch_render_fwd_geo<false>(a, stream);
  return 0;
}

}  // namespace gs
