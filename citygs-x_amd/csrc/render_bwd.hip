// Backward of the per-tile blend (cuda_rasterizer/backward.cu:324-567): each
// pixel replays its Gaussians back to front from the stored final
// transmittance and contributor count, and per-Gaussian gradients are summed
// over pixels.
//
// Workgroup = one 16x16 tile = four 64-lane waves; a wave owns an 8x8 quadrant
// and each of its 16-lane rows a 4x4 pixel block, a quad of lanes one of the
// block's columns.
//   * The tile's list is scanned back to front, 256 entries at a time, and the
//     entries that touch a block in front of its deepest contributor (the
//     forward kernel's own answer, a word per instance, when the caller hands
//     them on; otherwise the inflated alpha >= 1/255 ellipse is tested again)
//     are compacted into a ring; the others' records are zero.
//   * Out of a window of up to 256 waiting Gaussians every wave picks those
//     that touch its own quadrant, stages up to SLOTS of them in LDS, compacts
//     for each of its rows the slots that touch the row's block into a byte
//     list, and the four rows walk their own lists concurrently, four entries
//     per pass.  The window ends where a wave has no slot left.
//   * A pass has two halves.  In the first, lane = pixel: the recurrence over
//     the four entries, which leaves w = alpha T and q = G dL/dalpha per
//     (entry, pixel).  In the second, lane e of a quad works for entry e: the
//     4x4 blocks of w and q are transposed inside the quads, the sums over
//     pixels of q and its moments are plain additions over registers, those of
//     w times the eight upstream channels are matrix instructions (so is the
//     dot product of an entry's channels with a pixel's upstream gradients in
//     the first half), and two halving steps add up the quads of a row.
//   * The sixteen sums of an entry go into the wave's own accumulator in LDS,
//     row after row, with a plain read-add-write (no atomics: an LDS float
//     atomic costs about three cycles per active lane here).
//   * After the window the accumulators of the waves that have staged a
//     Gaussian are added in wave order and
//     every (tile, Gaussian) instance's sums are stored as one 64-byte record,
//     at the instance's index in emission order (the order key emission wrote
//     them: all instances of a Gaussian are consecutive there).  No global
//     atomics either.
//   * Instances that no pixel blends have records of zeros.  In views with many
//     instances per pixel, where those are nearly all, they are left out: a byte
//     per instance (`written`, cleared first) says which records there are.  The
//     zeros' stores were in the chain of the longest tiles, too (a load behind
//     them waits for them): 10 M Gaussians at street level, two views of 2.7 M and
//     6.2 M instances, 313 and 734 us -> 312 and 620.
// A second kernel then sums, for every Gaussian, its consecutive records and
// writes the five gradient tensors: a streaming pass.  Every sum is taken in a
// fixed order, so the gradients are the same bits from run to run.  (The
// reference issues 16 global float atomics per pixel and Gaussian,
// cuda_rasterizer/backward.cu:510-563.)
//
// What bounds it: the vector ALU (about 0.7 busy), which the matrix instructions
// share (a 4x4x1 one takes the time of four additions), and latency that four
// waves a SIMD do not hide (the head of a pass is a chain of LDS reads: list word
// and slot, operands).  A pass has some 300
// vector instructions of two or four cycles each and 16 matrix instructions, about
// 17 passes a wave at 1 M Gaussians, 1152x864; the steps between the walks a fifth
// of the whole.  With the staging shared by the four waves (batches of 128, 64 of
// them walked at a time) there were 13 barriers per 256 entries; a window has three
// and a scan of 256 positions one, so that it is four where Gaussians are small and
// a wave has slots for all of its own, and 13 to 16 where every Gaussian covers
// the tile and 256 entries take four or five windows.  Lists are four times
// shorter, passes 12 % more.  Before and after: 208 -> 197 us there, 491 -> 464 us
// for 4 M Gaussians from the air, 567 -> 549 us for 10 M at street level, 104 -> 96
// us for 300 k without geometry channels.  Four workgroups a CU with 64 slots, or
// five with 48: 464 and 522 us at 4 M with geometry channels, whose 118 registers
// do not fit five; without them 56 slots and five (96 us against 106).  The
// accumulators' reads a pass ahead of their use gain nothing.  The list words a pass
// ahead and the Gaussians' numbers in the ring (at 60 slots): 463 -> 450 us at 4 M,
// 467 -> 457 at street level, where the longest tiles' chains decide; at 1 M the same.
// The records' places asked for before the walk: 473.
// The matrix cores take what contracts an operand that all
// entries or all pixels share; the recurrence itself is a serial chain per
// pixel.
//
// The per-pixel arithmetic follows the CPU statement's operation for operation
// in everything that decides what counts (the exponent, alpha, the tests) and
// in the transmittance, with these exceptions after that: the order in which
// pixels are summed (fixed for thin Gaussians, see `aligned`); the factors that
// are constant per Gaussian (W/2, H/2, the opacity, the conic and -1/2 of the
// geometric gradients), which multiply the sums instead of every term; and the
// blend of everything behind a Gaussian, background included, which the
// reference keeps per channel and this kernel keeps as its dot product with the
// upstream gradients (one recurrence instead of eight: see `behind_dot`).
// Gradients therefore agree with a CPU evaluation to rounding (rel. L2 of the
// order of 1e-7 on the test scenes), not bit for bit.
#include <type_traits>

#include "gs_common.h"
#include "gs_kernels.h"
#include "render_common.h"

namespace gs {

namespace {

constexpr int WINDOW = GS_TILE_PIX;  // waiting Gaussians that are looked at together
constexpr int PENDING = 512;         // ring of list positions that wait: at most WINDOW - 1 + GS_TILE_PIX of them
constexpr int RUN = GS_WAVE;        // consecutive positions of a tile's list that stay together (see the order of the sums)
constexpr float THIN = 0.8f;        // squared correlation b * b / (a * c) from which a Gaussian counts as thin
constexpr int GROUP = 4;            // entries of a list handled per pass of the walk, one per lane of a quad
constexpr int WAVES = GS_TILE_PIX / GS_WAVE;
constexpr uint32_t NO_SLOT = 255u;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The value lane E of a quad (four neighbouring lanes) holds, in all four lanes.
template <int E>
__device__ __forceinline__ float quad_lane(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), E * 0x55, 0xF, 0xF, true));
}

// HITS: the forward blend left, per sorted instance, which 4x4 blocks of the tile the Gaussian can touch; without
// it the same test is made again here.
template <bool RENDER_GEO, bool HITS>
__global__ void __launch_bounds__(GS_TILE_PIX) __attribute__((amdgpu_waves_per_eu(RENDER_GEO ? 4 : 5)))
render_bwd_kernel(const uint2* __restrict__ ranges, const uint32_t* __restrict__ point_list, int W, int H, float fx,
                  float fy, const float* __restrict__ bg, const float2* __restrict__ means2D,
                  const float4* __restrict__ conic_opacity, const float* __restrict__ rgb,
                  const float* __restrict__ all_map, const float* __restrict__ all_map_pixels,
                  const float* __restrict__ final_Ts, const uint32_t* __restrict__ n_contrib_px,
                  const uint8_t* __restrict__ compute_locally, const float* __restrict__ dL_dpix,
                  const float* __restrict__ dL_dout_all_map, const float* __restrict__ dL_dout_plane_depth,
                  const uint32_t* __restrict__ emission_sorted, float4* __restrict__ instance_grads,
                  uint8_t* __restrict__ written, const uint32_t* __restrict__ block_hits,
                  const float4* __restrict__ packed_records,
                  const uint32_t* __restrict__ packed_valid, const uint32_t* __restrict__ tile_order,
                  const uint32_t* __restrict__ tile_order_valid, uint32_t tiles_x) {
  // (whether the forward call packed the records is its decision per view: a word beside them says)
  const float4* packed = (packed_records != nullptr && (packed_valid == nullptr || *packed_valid != 0u))
                             ? packed_records : nullptr;
  constexpr bool render_geo = RENDER_GEO;
  // Which Gaussian a position holds is fetched with the position's hit word and waits beside it: a window's staging then has
  // one trip to memory in its chain, not two.  It takes the LDS of four slots a wave.  (Without channels, five workgroups a
  // CU, it costs more than it saves: 300 k 101 us, 108 so.)
  constexpr bool GAUSSIANS_WAIT = RENDER_GEO;
  // The Gaussians a wave can stage at a time: as many as the LDS holds with four or five workgroups.
  constexpr int SLOTS = RENDER_GEO ? 60 : 56;
  constexpr int LIST_BYTES = SLOTS + RUN;  // a row's list: its entries, and what keeps the places of a run that began earlier
  static_assert(SLOTS <= GS_WAVE && SLOTS % GROUP == 0 && LIST_BYTES % GROUP == 0, "a lane per slot, whole words of lists");
  static_assert(LIST_BYTES <= 2 * GS_WAVE, "a wave clears its four lists in two rounds");
  // What a wave has staged.  (Slot SLOTS: what an entry behind the end of a list refers to, a Gaussian of opacity 0.)
  __shared__ float4 s_xyp[WAVES][SLOTS + 1];  // centre x, y; as bits: the position in the list; 1 thin, 2 exact
  __shared__ float4 s_co[WAVES][SLOTS + 1];   // the conic, and -1/2 of the opacity
  // colour, then the five geometry channels: eight floats per Gaussian, read as two 16-byte words
  __shared__ float4 s_chan[WAVES][SLOTS + 1][RENDER_GEO ? 2 : 1];
  // accumulators: word 4 slot + (part ^ (slot / 4 & 3)) holds sums 4 part .. 4 part + 3 of a slot, so that
  // neither the walk's accesses (a part of consecutive slots) nor the hand-over's pile up on a few banks
  __shared__ float4 s_acc[WAVES][4 * SLOTS];
  // the four rows' lists of every wave: the slots that can touch the row's block and are not
  // behind its deepest contributor, one byte each, in walking order; bytes behind a list's end are SLOTS
  __shared__ uint32_t s_idx[WAVES][4][LIST_BYTES / 4];
  // the Gaussians that wait to be staged: position in the list, blocks touched
  __shared__ int s_pend[PENDING];
  __shared__ uint16_t s_pend_hits[PENDING];
  __shared__ uint32_t s_pend_gaussian[GAUSSIANS_WAIT ? PENDING : 1];
  __shared__ int s_found[2][WAVES];
  // which slot each wave has given a Gaussian of the window (byte w of a word: wave w's, or NO_SLOT); a wave's own slots:
  // place in the window, rows touched << 8; how much of the window the wave has slots for
  __shared__ uint32_t s_place[WINDOW];
  __shared__ uint16_t s_own[WAVES][SLOTS];
  __shared__ int s_limit[WAVES];
  __shared__ int4 s_row_last[WAVES];  // the deepest contributor of every row

  const int tid = threadIdx.x;
  uint32_t tile = blockIdx.x;
  if (tile_order != nullptr) {
    const uint32_t ordered = tile_order[blockIdx.x];
    tile = *tile_order_valid != 0u ? ordered : tile;
  }
  const uint32_t tile_y = tile / tiles_x, tile_x = tile - tile_y * tiles_x;
  const RowThread rt = row_thread(tile_x, tile_y);
  const int lane = rt.lane, wave = rt.wave, row = rt.row;
  // (a quad of lanes holds one column of the row's 4x4 block: see the order of the sums below)
  const uint32_t px = (uint32_t)rt.qx0 + (uint32_t)(row & 1) * 4u + (uint32_t)(rt.l16 >> 2);
  const uint32_t py = (uint32_t)rt.qy0 + (uint32_t)(row >> 1) * 4u + (uint32_t)(rt.l16 & 3);
  const bool inside = px < (uint32_t)W && py < (uint32_t)H;
  const size_t pid = (size_t)W * py + px;
  const size_t HW = (size_t)H * W;
  const float pfx = (float)px, pfy = (float)py;
  const float rayx = (float)(((double)pfx - W * 0.5) / (double)fx);
  const float rayy = (float)(((double)pfy - H * 0.5) / (double)fy);
  const uint2 range = ranges[tile];
  const int total = (int)(range.y - range.x);
  // The record of an instance that no pixel blends, where there is to be one
  auto no_record = [&](int p) {
    float4* rec = instance_grads + 4 * (size_t)emission_sorted[range.x + (uint32_t)p];
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    rec[0] = z; rec[1] = z; rec[2] = z; rec[3] = z;
  };
  if (!compute_locally[tile]) {
    // normally an empty range; if the forward pass binned this tile under a wider mask its records are zeros
    if (written == nullptr)
      for (int p = tid; p < total; p += GS_TILE_PIX) no_record(p);
    return;
  }

  const float T_final = inside ? final_Ts[pid] : 0.f;
  float T = T_final;
  const int last_contributor = inside ? (int)n_contrib_px[pid] : 0;

  // deepest contributor of each row, of this wave and of the whole tile: nothing behind it is ever touched
  int row_last = last_contributor;
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) row_last = max(row_last, __shfl_xor(row_last, d, GS_WAVE));
  if ((lane & 15) == 0) reinterpret_cast<int*>(&s_row_last[wave])[row] = row_last;
  __syncthreads();
  int tile_last = 0;
#pragma unroll
  for (int w = 0; w < WAVES; w++) {
    const int4 r = s_row_last[w];
    tile_last = max(tile_last, max(max(r.x, r.y), max(r.z, r.w)));
  }
  tile_last = __builtin_amdgcn_readfirstlane(tile_last);
  // Every instance record of the tile is written at most once: the ones behind the deepest contributor
  // are zeros, the others are written at the end of their batch.
  if (written == nullptr)
    for (int p = tile_last + tid; p < total; p += GS_TILE_PIX) no_record(p);
  if (tile_last == 0) return;

  float gpix[GS_N_RGB] = {0.f, 0.f, 0.f}, gmap[GS_N_MAP] = {0.f, 0.f, 0.f, 0.f, 0.f};
  if (inside) {
#pragma unroll
    for (int ch = 0; ch < GS_N_RGB; ch++) gpix[ch] = dL_dpix[ch * HW + pid];
    if (render_geo) {
#pragma unroll
      for (int ch = 0; ch < GS_N_MAP; ch++) gmap[ch] = dL_dout_all_map[ch * HW + pid];
      const float nx = all_map_pixels[pid], ny = all_map_pixels[HW + pid], nz = all_map_pixels[2 * HW + pid];
      const float dist = all_map_pixels[4 * HW + pid];
      const float tmp = (float)((double)((nx * rayx + ny * rayy) + nz) + 1.0e-8);
      const float gd = dL_dout_plane_depth[pid];
      gmap[GS_N_MAP - 1] += (-gd / tmp);
      gmap[0] += gd * (dist / (tmp * tmp) * rayx);
      gmap[1] += gd * (dist / (tmp * tmp) * rayy);
      gmap[2] += gd * (dist / (tmp * tmp));
    }
  }
  float bg_dot = 0.f;
#pragma unroll
  for (int ch = 0; ch < GS_N_RGB; ch++) bg_dot += bg[ch] * gpix[ch];
  // dL/dalpha of a Gaussian needs sum_ch (c_ch - b_ch) g_ch, with b the blend of everything behind it and g the
  // upstream gradients of the eight channels.  The reference keeps b per channel (accum_rec,
  // cuda_rasterizer/backward.cu:463-472: b <- alpha c + (1 - alpha) b at every step); the sum is linear in b, so
  // here the pixel keeps the one number B = sum_ch b_ch g_ch instead, which obeys the same recurrence with
  // S = sum_ch c_ch g_ch in place of c: the term is S - B, and B <- alpha S + (1 - alpha) B.  Same value, eight
  // multiply-adds per step instead of forty operations; it is rounded differently (an error of the order of
  // eps |c| |g| per term where the per-channel form has eps |c - b| |g|), well inside the stated tolerance.  The
  // background is what lies behind the last Gaussian: B starts as its dot product, which is the reference's separate
  // term -T_final / (1 - alpha) sum_ch bg_ch g_ch (cuda_rasterizer/backward.cu:505-508).
  float behind_dot = bg_dot;

  // The pixels' upstream gradients as the matrix instructions that sum over pixels take them: register p of lane i of
  // a quad holds channel i (and 4 + i) of the quad's pixel p.
  float grad_t[RENDER_GEO ? 2 : 1][4];
  {
    const float chan[8] = {gpix[0], gpix[1], gpix[2], gmap[0], gmap[1], gmap[2], gmap[3], gmap[4]};
#pragma unroll
    for (int h = 0; h < (RENDER_GEO ? 2 : 1); h++) {
      float t[4] = {chan[4 * h], chan[4 * h + 1], chan[4 * h + 2], chan[4 * h + 3]}, unused[4] = {0.f, 0.f, 0.f, 0.f};
      quad_transpose2(t, unused);
#pragma unroll
      for (int p = 0; p < 4; p++) grad_t[h][p] = t[p];
    }
  }
  // Does a pixel of the wave have an upstream gradient that is not finite?  It belongs to the Gaussians the pixel
  // blended; the others' weight 0 would make a NaN of it in the sums.
  bool odd = false;
  {
    float top = 0.f;  // (0 x is 0 for every finite x)
#pragma unroll
    for (int ch = 0; ch < GS_N_RGB; ch++) top += 0.f * gpix[ch];
#pragma unroll
    for (int ch = 0; ch < GS_N_MAP; ch++) top += 0.f * gmap[ch];
    odd = gs_ballot(top != 0.f) != 0ull;
  }

  if (lane == 0) {
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    s_xyp[wave][SLOTS] = z;
    s_co[wave][SLOTS] = z;
#pragma unroll
    for (int h = 0; h < (RENDER_GEO ? 2 : 1); h++) s_chan[wave][SLOTS][h] = z;
  }
  const uint32_t quad_shift = 8u * (uint32_t)(lane & 3), quad = (uint32_t)(rt.l16 >> 2);
  const float block_y0 = (float)(py & ~3u);  // the first of the four pixels of a quad

  // Positions are 0-based indices into the tile's list; the walk goes down from the tile's deepest contributor.  Every wave
  // picks, out of a window of positions, the Gaussians that touch one of its rows in front of the row's deepest contributor,
  // a quarter of the list where Gaussians are small, stages those and walks them; the window ends where a wave has no slot
  // left.  A position that no wave has taken has a record of zeros.
  auto hits_at = [&](int pos) { return pos >= 0 ? block_hits[range.x + (uint32_t)pos] : 0u; };
  auto hits_by_test = [&](int pos) {
    if (pos < 0) return 0u;
    const uint32_t g = point_list[range.x + (uint32_t)pos];
    const float2 xy = means2D[g];
    const float4 co = conic_opacity[g];
    const float tile_x0 = (float)(tile_x * GS_TILE_X), tile_y0 = (float)(tile_y * GS_TILE_Y);
    const float4 cp = block_test_params(co, xy, tile_x0, tile_y0);
    return ellipse_hits_tile(xy, co, cp.x, cp.y, cp.z, tile_x0, tile_y0);
  };
  auto sync_wave = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  int unscanned = tile_last;  // positions below this one have not been looked at
  uint32_t head = 0u, tail = 0u, parity = 0u;
  // (fetched one step ahead, and taken apart where it is used: taken apart at once, every step waits for the next one's word,
  // 0.45 us of a chain that decides how long the kernel takes.  10 M Gaussians at street level, lists up to 22 k entries, two
  // pairs of views: 569 and 867 us a launch so, 551 and 829 now)
  uint32_t hits_next = HITS ? hits_at(unscanned - 1 - tid) : 0u;
  auto gaussian_at = [&](int pos) { return GAUSSIANS_WAIT && pos >= 0 ? point_list[range.x + (uint32_t)pos] : 0u; };
  uint32_t gaussian_next = gaussian_at(unscanned - 1 - tid);
  uint32_t carried[4] = {0u, 0u, 0u, 0u}, carried_run = 0xFFFFFFFFu;  // see `aligned` below
  for (;;) {
    while (tail - head < (uint32_t)WINDOW && unscanned > 0) {
      const int pos = unscanned - 1 - tid;
      uint32_t hits = HITS ? hits_from_bytes(hits_next) : hits_by_test(pos);
      unscanned = max(unscanned - GS_TILE_PIX, 0);
      if (HITS) hits_next = hits_at(unscanned - 1 - tid);
      const uint32_t gaussian = gaussian_next;
      gaussian_next = gaussian_at(unscanned - 1 - tid);
#pragma unroll
      for (int w = 0; w < WAVES; w++) {
        const int4 last = s_row_last[w];
        hits &= ~((pos >= last.x ? 1u << (4 * w) : 0u) | (pos >= last.y ? 2u << (4 * w) : 0u) |
                  (pos >= last.z ? 4u << (4 * w) : 0u) | (pos >= last.w ? 8u << (4 * w) : 0u));
      }
      const bool take = pos >= 0 && hits != 0u;
      const uint64_t take_m = gs_ballot(take);
      if (lane == 0) s_found[parity][wave] = (int)__popcll(take_m);
      if (written == nullptr && pos >= 0 && !take) no_record(pos);
      __syncthreads();
      uint32_t before = tail;
#pragma unroll
      for (int w = 0; w < WAVES; w++) {
        const uint32_t n = (uint32_t)s_found[parity][w];
        before += w < wave ? n : 0u;
        tail += n;
      }
      if (take) {
        const uint32_t at = (before + __builtin_amdgcn_mbcnt_hi((uint32_t)(take_m >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)take_m, 0u))) &
                            (PENDING - 1);
        s_pend[at] = pos;
        if (GAUSSIANS_WAIT) s_pend_gaussian[at] = gaussian;
        s_pend_hits[at] = (uint16_t)hits;
      }
      parity ^= 1u;  // (the counts are rewritten two barriers later)
    }
    const int waiting = (int)min((uint32_t)WINDOW, tail - head);
    if (waiting == 0) break;
    __syncthreads();
    // the wave's slots in the window
    uint32_t found = 0u;
    {
      int limit = waiting;
#pragma unroll
      for (int k = 0; k < WINDOW / GS_WAVE; k++) {
        const int at = k * GS_WAVE + lane;
        const uint32_t rows = at < waiting ? (uint32_t)s_pend_hits[(head + (uint32_t)at) & (PENDING - 1)] >> (4 * wave) & 15u : 0u;
        const uint64_t take_m = gs_ballot(rows != 0u);
        const uint32_t slot = __builtin_amdgcn_mbcnt_hi((uint32_t)(take_m >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)take_m, found));
        reinterpret_cast<uint8_t*>(s_place)[4 * at + wave] = (uint8_t)(rows != 0u ? slot : NO_SLOT);
        if (rows != 0u && slot < (uint32_t)SLOTS) s_own[wave][slot] = (uint16_t)((uint32_t)at | rows << 8);
        const uint64_t over_m = gs_ballot(rows != 0u && slot == (uint32_t)SLOTS);
        if (over_m != 0ull) limit = k * GS_WAVE + (int)__builtin_ctzll(over_m);
        found += (uint32_t)__popcll(take_m);
      }
      if (lane == 0) s_limit[wave] = limit;
      found = min(found, (uint32_t)SLOTS);
    }
    __syncthreads();
    int length = waiting;
#pragma unroll
    for (int w = 0; w < WAVES; w++) length = min(length, s_limit[w]);
    length = __builtin_amdgcn_readfirstlane(length);
    // lane = slot
    const uint32_t own = (uint32_t)lane < found ? (uint32_t)s_own[wave][lane] : (uint32_t)WINDOW;
    const bool have = (uint32_t)lane < found && (int)(own & 255u) < length;
    const int count = (int)__popcll(gs_ballot(have));
    if (count != 0) {
      const int pos = s_pend[(head + (own & 255u)) & (PENDING - 1)];
      const uint32_t nibble = have ? own >> 8 : 0u;
      bool is_thin = false;
      if (have) {
        const uint32_t g = GAUSSIANS_WAIT ? s_pend_gaussian[(head + (own & 255u)) & (PENDING - 1)] : point_list[range.x + (uint32_t)pos];
        // A Gaussian's operands: one 64-byte record where the forward call packed them (a single line of memory,
        // every byte of it used), else gathered from the four arrays.  (Each route loads and then stages by itself:
        // with the loaded values merged across the two routes the compiler splits the gathers into single words.)
        auto stage = [&](const float2 xy, const float4 co, const float c0, const float c1, const float c2,
                         const float (&m)[GS_N_MAP]) {
          s_co[wave][lane] = make_float4(co.x, co.y, co.z, -0.5f * co.w);
          is_thin = !(co.y * co.y < THIN * co.x * co.z);
          s_xyp[wave][lane] =
              make_float4(xy.x, xy.y, __int_as_float(pos),
                          __int_as_float(!is_thin ? 0 : ((0xE880u >> nibble) & 1u) != 0u ? 2 : 1));
          if (render_geo) s_chan[wave][lane][RENDER_GEO ? 1 : 0] = make_float4(m[1], m[2], m[3], m[4]);
          s_chan[wave][lane][0] = make_float4(c0, c1, c2, m[0]);
        };
        if (packed != nullptr) {
          const float4* rec = packed + 4 * (size_t)g;
          const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
          float m[GS_N_MAP] = {r2.y, r2.z, r2.w, 0.f, 0.f};
          if (render_geo) {
            const float4 r3 = rec[3];
            m[3] = r3.x, m[4] = r3.y;
          }
          stage(make_float2(r0.x, r0.y), make_float4(r0.z, r0.w, r1.x, r1.y), r1.z, r1.w, r2.x, m);
        } else {
          const float2 xy = means2D[g];
          const float4 co = conic_opacity[g];
          const float c0 = rgb[3 * (size_t)g], c1 = rgb[3 * (size_t)g + 1], c2 = rgb[3 * (size_t)g + 2];
          float m[GS_N_MAP] = {0.f, 0.f, 0.f, 0.f, 0.f};
          if (render_geo) {
#pragma unroll
            for (int ch = 0; ch < GS_N_MAP; ch++) m[ch] = all_map[5 * (size_t)g + ch];
          }
          stage(xy, co, c0, c1, c2, m);
        }
      }
      // (every wave has read the accumulators of the window before: the barriers above)
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (k * GS_WAVE + lane < 4 * SLOTS) s_acc[wave][k * GS_WAVE + lane] = make_float4(0.f, 0.f, 0.f, 0.f);

      // Per-row lists: the lanes whose Gaussian counts for row r append their slot
      // numbers to the row's list, in lane order (a lane's place is the number of set bits below its own).
      uint32_t passes;  // wave-uniform, like all that follows here: the longest of the four lists
      bool aligned;
      {
        uint32_t* const words = &s_idx[wave][0][0];
        words[lane] = (uint32_t)SLOTS * 0x01010101u;
        if (GS_WAVE + lane < LIST_BYTES) words[GS_WAVE + lane] = (uint32_t)SLOTS * 0x01010101u;
        uint64_t hit_m[4];
#pragma unroll
        for (int r = 0; r < 4; r++) hit_m[r] = gs_ballot(((nibble >> r) & 1u) != 0u);
        auto list_row = [&](int r, uint64_t b, uint32_t from) {
          const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, from));
          if (__builtin_amdgcn_inverse_ballot_w64(b)) reinterpret_cast<uint8_t*>(&s_idx[wave][r][0])[below] = (uint8_t)lane;
          return from + (uint32_t)__popcll(b);
        };
        // The gradient of a thin Gaussian's covariance is a small difference of its three conic sums: a change in how
        // they are rounded comes back multiplied by a c / (a c - b b), squared for scale and rotation.  Where a wave has
        // such a Gaussian its conic sums are taken in a fixed order (`thin`: the sixteen pixels of a row as a tree; and
        // `exact`, if three or four rows touch it: the rows by their places in the lists of a run of 64 positions, rows
        // at the same place merged first), whatever else is staged or skipped: its lists keep the places (`aligned`),
        // and the passes that hold it take the sums in that order.  Below THIN the factor is at most 25.
        // That is the order of a kernel that takes one entry per pass and reduces its sums over the row's lanes.  On 16
        // scenes of 60 to 4000 Gaussians, a quarter of them thin, the covariance gradients of the thin ones are a relative
        // 7.9e-6 from float64 in this order, 7.9e-6 in that kernel and 8.9e-6 with the order left to the lists (12 of the
        // 16 worse); the conic gradients themselves are 2.1e-6 off in all three.
        aligned = gs_ballot(is_thin && ((0xE880u >> nibble) & 1u) != 0u) != 0ull;
        const uint32_t run = (uint32_t)(tile_last - 1 - pos) / RUN;
        const uint32_t first_run = (uint32_t)__builtin_amdgcn_readlane((int)run, 0);
        const uint32_t last_run = (uint32_t)__builtin_amdgcn_readlane((int)run, count - 1);
        if (!aligned) {
          const uint32_t l0 = list_row(0, hit_m[0], 0u), l1 = list_row(1, hit_m[1], 0u);
          const uint32_t l2 = list_row(2, hit_m[2], 0u), l3 = list_row(3, hit_m[3], 0u);
          passes = max(max(l0, l1), max(l2, l3));
        } else {
          // (a run that began in an earlier window has `carried` entries per row there)
          const uint32_t least = min(min(carried[0], carried[1]), min(carried[2], carried[3]));
          uint64_t todo = gs_ballot(have);
          passes = 0u;
          while (todo != 0ull) {
            const uint32_t this_run = (uint32_t)__builtin_amdgcn_readlane((int)run, (int)__builtin_ctzll(todo));
            const uint64_t run_m = todo & gs_ballot(run == this_run);
            todo &= ~run_m;
            uint32_t end = passes;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const uint32_t from = passes + (this_run == carried_run ? carried[r] - least : 0u);
              end = max(end, list_row(r, hit_m[r] & run_m, from));
            }
            passes = end;
          }
        }
        passes = (uint32_t)__builtin_amdgcn_readfirstlane((int)passes);
        const uint64_t last_m = gs_ballot(have && run == last_run);
#pragma unroll
        for (int r = 0; r < 4; r++)
          carried[r] = (first_run == last_run && last_run == carried_run ? carried[r] : 0u) + (uint32_t)__popcll(hit_m[r] & last_m);
        carried_run = last_run;
      }
      sync_wave();
      uint32_t word_next = s_idx[wave][row][0];  // (read a pass ahead: the head of a pass is a chain of LDS reads)
      for (uint32_t n = 0; n < passes; n += GROUP) {
        // Four entries of every row's list.  Lane e of each of the row's quads fetches entry e.
        const uint32_t word = word_next;
        word_next = s_idx[wave][row][min(n / GROUP + 1u, (uint32_t)LIST_BYTES / 4u - 1u)];
        const uint32_t j_own = __builtin_amdgcn_ubfe(word, quad_shift, 8u);
        const float4 xyp = s_xyp[wave][j_own];
        const float4 co = s_co[wave][j_own];
        const bool thin = gs_ballot(__float_as_int(xyp.w) > 0) != 0ull;
        const bool exact = gs_ballot(__float_as_int(xyp.w) > 1) != 0ull;
        // S = sum_ch c_ch g_ch of every (entry, pixel): a contraction over the channels, of the entries' colours and the
        // pixels' upstream gradients.  Register e of lane p of a quad receives entry e at pixel p (one fused
        // multiply-add per channel, in channel order: the bits of the same chain of vector instructions).
        f32x4 S = {0.f, 0.f, 0.f, 0.f};
        {
          const float4 c4 = s_chan[wave][j_own][0];
          S = __builtin_amdgcn_mfma_f32_4x4x1f32(c4.x, gpix[0], S, 0, 0, 0);
          S = __builtin_amdgcn_mfma_f32_4x4x1f32(c4.y, gpix[1], S, 0, 0, 0);
          S = __builtin_amdgcn_mfma_f32_4x4x1f32(c4.z, gpix[2], S, 0, 0, 0);
          if (render_geo) {
            const float4 m4 = s_chan[wave][j_own][RENDER_GEO ? 1 : 0];
            S = __builtin_amdgcn_mfma_f32_4x4x1f32(c4.w, gmap[0], S, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f32_4x4x1f32(m4.x, gmap[1], S, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f32_4x4x1f32(m4.y, gmap[2], S, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f32_4x4x1f32(m4.z, gmap[3], S, 0, 0, 0);
            S = __builtin_amdgcn_mfma_f32_4x4x1f32(m4.w, gmap[4], S, 0, 0, 0);
          }
        }
        // The recurrence, entry after entry, lane = pixel.  Straight-line: every lane evaluates its row's Gaussian, and
        // a lane for which it does not count (behind the pixel's last contributor, outside the power window, alpha
        // below 1/255) takes part with alpha = 0, G = 0: T and what lies behind stay as they are, w and q are 0.
        // Same tests as the forward pass, on the same bits.
        float w[GROUP], q[GROUP];
        auto step = [&](auto e_tag) {
          constexpr int e = decltype(e_tag)::value;
          const float dx = quad_lane<e>(xyp.x) - pfx, dy = quad_lane<e>(xyp.y) - pfy;
          const float form = gauss_form(quad_lane<e>(co.x), quad_lane<e>(co.y), quad_lane<e>(co.z), dx, dy);
          const int pos_e = __float_as_int(quad_lane<e>(xyp.z));
          const float G_raw = gs_neg2_exp_of_form(form);  // -2 times the Gaussian's value
          const float alpha_raw = fminf(0.99f, quad_lane<e>(co.w) * G_raw);
          // (lane masks of single comparisons, combined in scalar registers)
          const uint64_t active_m = gs_ballot(pos_e < last_contributor) & gs_ballot(!(form < 0.0f)) &
                                    gs_ballot(!(form > GS_FORM_MAX)) & gs_ballot(!(alpha_raw < 1.0f / 255.0f));
          const bool active = __builtin_amdgcn_inverse_ballot_w64(active_m);
          const float alpha = active ? alpha_raw : 0.f;
          // The transmittance follows the CPU statement's operation sequence exactly (IEEE reciprocal):
          // upstream gradients of the geometry channels can be many orders of magnitude larger than the
          // result (plane depth divides by a blended normal that may be nearly perpendicular to the ray), so
          // T, which multiplies them, decides how far a gradient can drift.
          const float oma = 1.f - alpha;
          const float rcp1ma = gs_rcp_normal(oma);  // alpha <= 0.99: the bits of 1.f / (1.f - alpha)
          T = T * rcp1ma;
          w[e] = alpha * T;
          // (S may be NaN or infinite where the Gaussian does not count: a non-finite channel only reaches the pixels
          // that blended it in the forward pass, as in the reference, cuda_rasterizer/backward.cu:463-472)
          const float ahead = S[e] - behind_dot;
          const float behind_next = __builtin_fmaf(alpha, S[e], oma * behind_dot);
          behind_dot = active ? behind_next : behind_dot;
          const float g_dalpha = G_raw * (ahead * T);
          q[e] = active ? g_dalpha : 0.f;
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        // (q is -2 times what it stands for below, as G is: the thread that hands the record over takes the factor out)
        // The sums over pixels.  From here on lane e of a quad works for entry e, register p is the quad's pixel p (the
        // quad's four pixels are one column of the block: dx is the quad's, dy the register's).  The per-Gaussian factors
        // of the geometric gradients stay out of the sums: with
        // q = G dL/dalpha, u = conic (dx, dy), a pixel's terms are dL/dmean = -opacity q u,
        // dL/dconic = -opacity/2 q (dx dx, dx dy, dy dy) and dL/dopacity = q
        // (cuda_rasterizer/backward.cu:520-541); sum q u is formed from sum q (dx, dy) by the thread that hands the
        // record over, sum q |u| here.  (The factors W/2 and H/2 from pixel to normalised coordinates are applied once
        // per Gaussian by the reduction kernel.)
        quad_transpose2(w, q);
        f32x4 c_lo = {0.f, 0.f, 0.f, 0.f}, c_hi = {0.f, 0.f, 0.f, 0.f};  // sum_p w g: registers = channels
        if (__builtin_expect(!odd, 1)) {
#pragma unroll
          for (int p = 0; p < 4; p++) {
            c_lo = __builtin_amdgcn_mfma_f32_4x4x1f32(grad_t[0][p], w[p], c_lo, 0, 0, 0);
            if (render_geo) c_hi = __builtin_amdgcn_mfma_f32_4x4x1f32(grad_t[RENDER_GEO ? 1 : 0][p], w[p], c_hi, 0, 0, 0);
          }
        } else {
          // the same chains of multiply-adds, of the pixels that blended the entry (whose weights are not zero)
          auto channel = [&](auto ch_tag, const float (&g)[4], f32x4& c) {
            constexpr int ch = decltype(ch_tag)::value;
#pragma unroll
            for (int p = 0; p < 4; p++) {
              const float sum = __builtin_fmaf(quad_lane<ch>(g[p]), w[p], c[ch]);
              c[ch] = w[p] != 0.f ? sum : c[ch];
            }
          };
          auto channels = [&](const float (&g)[4], f32x4& c) {
            channel(std::integral_constant<int, 0>{}, g, c);
            channel(std::integral_constant<int, 1>{}, g, c);
            channel(std::integral_constant<int, 2>{}, g, c);
            channel(std::integral_constant<int, 3>{}, g, c);
          };
          channels(grad_t[0], c_lo);
          if (render_geo) channels(grad_t[RENDER_GEO ? 1 : 0], c_hi);
        }
        const float dx = xyp.x - pfx, a_dx = co.x * dx, b_dx = co.y * dx;
        float dy[4], q_dy[4], ax = 0.f, ay = 0.f;
#pragma unroll
        for (int p = 0; p < 4; p++) {
          dy[p] = xyp.y - (block_y0 + (float)p);
          q_dy[p] = q[p] * dy[p];
          const float ux = __builtin_fmaf(co.y, dy[p], a_dx), uy = __builtin_fmaf(co.z, dy[p], b_dx);
          ax = __builtin_fmaf(fabsf(q[p]), fabsf(ux), ax);
          ay = __builtin_fmaf(fabsf(q[p]), fabsf(uy), ay);
        }
        auto sum4 = [](const float (&t)[4]) { return (t[0] + t[2]) + (t[1] + t[3]); };
        const float q0 = sum4(q), qy = sum4(q_dy);
        float qx = q0 * dx, xx = qx * dx, xy = qy * dx;
        float yy = __builtin_fmaf(q_dy[3], dy[3], __builtin_fmaf(q_dy[2], dy[2], __builtin_fmaf(q_dy[1], dy[1], q_dy[0] * dy[0])));
        if (thin) {  // (every product rounded by itself, sums as a tree over y, then x)
          float t0[4], t1[4], t2[4], t3[4];
#pragma unroll
          for (int p = 0; p < 4; p++) {
            t0[p] = q[p] * dx;
            t1[p] = t0[p] * dx;
            t2[p] = t0[p] * dy[p];
            t3[p] = q_dy[p] * dy[p];
          }
          qx = sum4(t0); xx = sum4(t1); xy = sum4(t2); yy = sum4(t3);
        }
        float v[16] = {qx, qy, ax, ay, xx, xy, yy, q0, c_lo[0], c_lo[1], c_lo[2], c_lo[3],
                       c_hi[0], c_hi[1], c_hi[2], c_hi[3]};
        quads_reduce16<RENDER_GEO>(v);
        float sum[4] = {v[0], v[1], v[2], v[3]};
        asm("" : "+v"(sum[0]), "+v"(sum[1]), "+v"(sum[2]), "+v"(sum[3]));  // (four registers, not a part of sixteen)
        // Quad k of a row now holds components 4 k .. 4 k + 3 of its entry e.  They go into the wave's own accumulator with
        // a plain read-add-write (the LDS accesses of a wave complete in order), one row after the other, since two rows
        // may be at the same Gaussian.  An LDS float atomic takes about three cycles per active lane.
        float4* const acc = &s_acc[wave][4u * j_own + (quad ^ ((j_own >> 2) & 3u))];
        uint64_t write_m = gs_ballot(j_own < (uint32_t)SLOTS);
        if (exact) {
          const float own[4] = {sum[0], sum[1], sum[2], sum[3]};
#pragma unroll
          for (int d = 1; d < 4; d++) {
            // (entries behind the ends of two lists are the same too: their sums are zero and go nowhere)
            const bool same = (uint32_t)__shfl_xor((int)j_own, 16 * d, GS_WAVE) == j_own;
            float t[4];
#pragma unroll
            for (int k = 0; k < 4; k++) t[k] = __shfl_xor(own[k], 16 * d, GS_WAVE);
            if (same) {
#pragma unroll
              for (int k = 0; k < 4; k++) sum[k] += t[k];
            }
            write_m &= ~gs_ballot(same && (row ^ d) < row);
          }
        }
        // (exact: entry after entry; otherwise row after row)
        uint64_t turn_m = exact ? 0x1111111111111111ull : 0xFFFFull;
        const int turn_shift = exact ? 1 : 16;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (__builtin_amdgcn_inverse_ballot_w64(write_m & turn_m)) {
            float4 a = *acc;
            a.x += sum[0]; a.y += sum[1]; a.z += sum[2]; a.w += sum[3];
            *acc = a;
          }
          turn_m <<= turn_shift;
          sync_wave();
        }
      }
    }
    __syncthreads();
    // A thread stores a quarter of a record: the sums of four components of the waves that have the Gaussian, added in
    // wave order.
    const int part = tid & 3;
    for (int at = tid >> 2; at < length; at += GS_TILE_PIX / 4) {
      const uint32_t emission = emission_sorted[range.x + (uint32_t)s_pend[(head + (uint32_t)at) & (PENDING - 1)]];
      const uint32_t places = s_place[at];
      float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
      if (places != 0xFFFFFFFFu) {
        uint32_t staged = 0u;  // where the Gaussian is
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
          const uint32_t slot = places >> (8 * w) & 255u;
          if (slot != NO_SLOT) {
            const float4 o = s_acc[w][4u * slot + ((uint32_t)part ^ ((slot >> 2) & 3u))];
            c.x += o.x; c.y += o.y; c.z += o.z; c.w += o.w;
            staged = (uint32_t)(w * (SLOTS + 1)) + slot;
          }
        }
        // (the sums are those of -2 q)
        const float4 co = (&s_co[0][0])[staged];
        if (part == 0) {  // mean2D x, y and their sums of absolute values
          c = make_float4(-co.w * (co.x * c.x + co.y * c.y), -co.w * (co.y * c.x + co.z * c.y), c.z * fabsf(co.w),
                          c.w * fabsf(co.w));
        } else if (part == 1) {  // conic x, y, w; the fourth component is the opacity gradient itself
          const float h = -0.5f * co.w;
          c.x *= h; c.y *= h; c.z *= h;
          c.w *= -0.5f;
        }
      }
      instance_grads[4 * (size_t)emission + part] = c;
      if (written != nullptr && part == 0) written[emission] = 1;
    }
    head += (uint32_t)length;
  }
}

// The rows of N floats that the lanes of a wave hold leave through LDS, past the caches, as N runs of consecutive floats.
template <int N>
__device__ __forceinline__ void stream_rows(float* __restrict__ out, int rows, const float (&own)[N], float* lds, int lane) {
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  sync();  // (everyone has read what the buffer last held)
#pragma unroll
  for (int k = 0; k < N; k++) lds[N * lane + k] = own[k];
  sync();
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int e = j * GS_WAVE + lane;
    if (e < N * rows) store_streaming(out + e, lds[e]);
  }
}

// Where reduce_instances_kernel streams: from this many Gaussians on, whose results outgrow what the caches keep for
// the next kernel.  This kernel and the preprocess backward kernel at 1152 x 864, stored plainly and streamed: 0.6 M
// 68.3 and 71.2 us, 1 M 102.3 and 104.7, 1.5 M 145.6 and 143.3, 2 M 201.6 and 183.9, 3 M 293.7 and 268.6 (2.5 M without
// geometry channels 132.4 and 127.0).
constexpr int REDUCE_STREAM_GAUSSIANS = 1'500'000;

// Sums the instance records of every Gaussian (consecutive in emission order) into the gradient
// tensors.  Record layout: [mean2D.x, mean2D.y, |mean2D|.x, |mean2D|.y, conic.x, conic.y, conic.w,
// opacity, rgb(3), map(5)].  Every output element is written.
// Bound by memory (64 bytes per instance in, 68 or 48 per Gaussian out).  STREAM: the records are read and the results
// stored past the caches.  Where the results are more than the caches hold anyway, the preprocess backward kernel that
// follows otherwise runs beside the write-back of the lines they left dirty: 4 M Gaussians, 1152 x 864, 79.3 + 277 us ->
// 79.5 + 248 (this kernel + that one), 10 M, 1920 x 1080, 175 + 633 -> 175 + 595.  That wants whole lines per store, so
// the rows of 3 and 5 floats are turned in LDS (stored from the lanes that hold them, 80.5 and 180).
// SPARSE: only the records that `written` tells of are there.  Kernels of their own: as a test of the pointer it cost the
// views with every record 3 to 11 % here (3 M at 1920 x 1080 89.0 -> 94.5 us, 1 M 33.4 -> 34.3, 300 k 15.3 -> 17.0).
template <bool STREAM, bool SPARSE>
__global__ void __launch_bounds__(GS_BLOCK_1D)
reduce_instances_kernel(int P, const uint32_t* __restrict__ point_offsets, const float4* __restrict__ instance_grads,
                        const uint8_t* __restrict__ written, float ddelx_dx, float ddely_dy, int render_geo,
                        float2* __restrict__ dL_dmean2D, float* __restrict__ dL_dmean2D_abs,
                        float4* __restrict__ dL_dconic_opacity, float* __restrict__ dL_dcolors,
                        float* __restrict__ dL_dall_map) {
  const int i = blockIdx.x * GS_BLOCK_1D + threadIdx.x;
  const int lane = threadIdx.x & (GS_WAVE - 1);
  const bool live = i < P;
  const uint32_t b = (!live || i == 0) ? 0u : point_offsets[i - 1], e = live ? point_offsets[i] : 0u;
  const uint32_t n = e - b;
  float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), a1 = a0, a2 = a0, a3 = a0;
  auto add = [](float4& a, const float4& r) { a.x += r.x; a.y += r.y; a.z += r.z; a.w += r.w; };
  // A Gaussian with many instances (in a street-level view one can cover thousands of tiles) is summed by the
  // whole wave: lane l takes records l, l + 64, ..., then the 64 partial sums are added across the lanes in a fixed
  // order.  Everything else is summed by its own thread, record after record.
  constexpr uint32_t MANY = 32;
  constexpr uint32_t REC_CHUNK = GS_WAVE, REC_STRIDE4 = 5;
  __shared__ float4 s_rec[GS_BLOCK_1D / GS_WAVE][REC_CHUNK * REC_STRIDE4];
  uint64_t many = gs_ballot(n > MANY);
  const uint64_t many_in_wave = many;
  while (many != 0ull) {
    const int owner = (int)__builtin_ctzll(many);
    many &= many - 1ull;
    const uint32_t ob = __shfl(b, owner, GS_WAVE), on = __shfl(n, owner, GS_WAVE);
    float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f), p1 = p0, p2 = p0, p3 = p0;
    auto add_record = [&](uint32_t k) {
      const float4* rec = instance_grads + 4 * (size_t)(ob + k);
      add(p0, rec[0]); add(p1, rec[1]); add(p2, rec[2]); add(p3, rec[3]);
    };
    if constexpr (SPARSE) {
      // (two rounds' bytes are asked for together: for four there are no registers at seven waves a SIMD)
      for (uint32_t k = (uint32_t)lane; k < on; k += 2 * GS_WAVE) {
        bool have[2];
#pragma unroll
        for (uint32_t j = 0; j < 2; j++) have[j] = k + j * GS_WAVE < on && written[ob + k + j * GS_WAVE] != 0;
#pragma unroll
        for (uint32_t j = 0; j < 2; j++)
          if (have[j]) add_record(k + j * GS_WAVE);
      }
    } else {
      for (uint32_t k = (uint32_t)lane; k < on; k += GS_WAVE) add_record(k);
    }
#pragma unroll
    for (int d = GS_WAVE / 2; d >= 1; d >>= 1) {
      float4* parts[4] = {&p0, &p1, &p2, &p3};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        parts[q]->x += __shfl_xor(parts[q]->x, d, GS_WAVE);
        parts[q]->y += __shfl_xor(parts[q]->y, d, GS_WAVE);
        parts[q]->z += __shfl_xor(parts[q]->z, d, GS_WAVE);
        parts[q]->w += __shfl_xor(parts[q]->w, d, GS_WAVE);
      }
    }
    if (lane == owner) { a0 = p0; a1 = p1; a2 = p2; a3 = p3; }
  }
  if (many_in_wave != 0ull) {
    // (a wave that holds such a Gaussian reads the others' records directly: rare)
    if (live && n <= MANY) {
      for (uint32_t k = b; k < e; k++) {
        if (SPARSE && written[k] == 0) continue;
        const float4* rec = instance_grads + 4 * (size_t)k;
        add(a0, rec[0]); add(a1, rec[1]); add(a2, rec[2]); add(a3, rec[3]);
      }
    }
  } else {
    // The records of a wave's 64 Gaussians are one contiguous run.  It is fetched 64 records at a time with
    // whole-wave 16-byte loads (the four lanes of a record share its 64-byte line), parked in LDS (records
    // padded to five 16-byte words: neither access pattern has bank conflicts) and every lane then adds up its own
    // records from there, in order.  With every lane loading its own records directly, a line passed through
    // the first-level cache once per 16-byte part.
    float4* mine = s_rec[threadIdx.x / GS_WAVE];
    const uint32_t run_begin = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
    uint32_t run_end = e;
#pragma unroll
    for (int d = GS_WAVE / 2; d >= 1; d >>= 1) run_end = max(run_end, (uint32_t)__shfl_xor((int)run_end, d, GS_WAVE));
    run_end = (uint32_t)__builtin_amdgcn_readfirstlane((int)run_end);
    for (uint32_t c = run_begin; c < run_end; c += REC_CHUNK) {
      uint64_t have_m = ~0ull;
      if constexpr (SPARSE) {
        have_m = gs_ballot(c + (uint32_t)lane < run_end && written[c + (uint32_t)lane] != 0);
        if (have_m == 0ull) continue;
      }
      float4 v[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t idx = (uint32_t)(j * GS_WAVE + lane), r = c + (idx >> 2);
        const float4* part = instance_grads + 4 * (size_t)r + (idx & 3u);
        const bool there = r < run_end && (!SPARSE || (have_m >> (idx >> 2) & 1u));
        if constexpr (STREAM)
          v[j] = there ? load_streaming(part) : make_float4(0.f, 0.f, 0.f, 0.f);
        else
          v[j] = there ? *part : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const uint32_t idx = (uint32_t)(j * GS_WAVE + lane);
        mine[(idx >> 2) * REC_STRIDE4 + (idx & 3u)] = v[j];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const uint32_t lo = max(b, c), hi = min(e, c + REC_CHUNK);
      for (uint32_t k = lo; k < hi; k++) {
        if (SPARSE && !((have_m >> (k - c)) & 1u)) continue;
        const float4* rec = mine + (k - c) * REC_STRIDE4;
        add(a0, rec[0]); add(a1, rec[1]); add(a2, rec[2]); add(a3, rec[3]);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  if constexpr (STREAM) {
    const int first = i - lane, rows = P - first < GS_WAVE ? P - first : GS_WAVE;
    if (rows <= 0) return;
    if (live) {
      store_streaming(dL_dmean2D + i, make_float2(a0.x * ddelx_dx, a0.y * ddely_dy));
      store_streaming(dL_dconic_opacity + i, a1);
    }
    float* const lds = reinterpret_cast<float*>(s_rec[threadIdx.x / GS_WAVE]);
    const float abs_row[3] = {a0.z * ddelx_dx, a0.w * ddely_dy, 0.f}, colour_row[3] = {a2.x, a2.y, a2.z};
    stream_rows(dL_dmean2D_abs + 3 * (size_t)first, rows, abs_row, lds, lane);
    stream_rows(dL_dcolors + 3 * (size_t)first, rows, colour_row, lds, lane);
    if (dL_dall_map) {
      const float map_row[5] = {render_geo ? a2.w : 0.f, render_geo ? a3.x : 0.f, render_geo ? a3.y : 0.f,
                                render_geo ? a3.z : 0.f, render_geo ? a3.w : 0.f};
      stream_rows(dL_dall_map + 5 * (size_t)first, rows, map_row, lds, lane);
    }
    return;
  }
  if (!live) return;
  // records hold the mean2D sums per pixel unit: d(pixel offset)/d(normalised coordinate) = W/2, H/2
  dL_dmean2D[i] = make_float2(a0.x * ddelx_dx, a0.y * ddely_dy);
  dL_dmean2D_abs[3 * (size_t)i] = a0.z * ddelx_dx;
  dL_dmean2D_abs[3 * (size_t)i + 1] = a0.w * ddely_dy;
  dL_dmean2D_abs[3 * (size_t)i + 2] = 0.f;
  dL_dconic_opacity[i] = a1;
  dL_dcolors[3 * (size_t)i] = a2.x;
  dL_dcolors[3 * (size_t)i + 1] = a2.y;
  dL_dcolors[3 * (size_t)i + 2] = a2.z;
  if (dL_dall_map) {
    float* m = dL_dall_map + 5 * (size_t)i;
    m[0] = render_geo ? a2.w : 0.f;
    m[1] = render_geo ? a3.x : 0.f;
    m[2] = render_geo ? a3.y : 0.f;
    m[3] = render_geo ? a3.z : 0.f;
    m[4] = render_geo ? a3.w : 0.f;
  }
}

}  // namespace

// Instances per pixel from which on records of zeros are left out.  A pixel blends some twenty Gaussians, whatever its tile's
// list holds, so it is the lists' length per pixel that says how many instances have no record.  The bytes cost a launch that
// clears them (5 us) and the sums a round trip for every 64 instances of a wave.  119 training views (23 thousand to 10 M
// Gaussians, 320 x 240 to 1920 x 1080, 0.05 to 18 instances a Gaussian), us with the zeros left out less us with them: up to 1
// instance a pixel 2 to 21 lost; 1 to 1.5 18 lost to 3 gained; 1.5 to 2 8 lost to 38 gained; 2 to 2.5 7 lost to 42 gained (two of
// 14 above 10, street level); 2.5 to 4 8 to 126 gained in 26 views, 5 to 14 lost in four (of 614 to 1932), the others within
// 3; from 4 on 5 to 112 gained in 25, 8 lost in one (of 1337), the others within 2.  (Gaussians per pixel, those out of view
// included, are no measure: a view of a tenth of 10 M Gaussians, 10 of them a pixel, lost 21 of 1477, one of 200 thousand large
// ones, 0.2 a pixel, gains 44 of 698.)
constexpr int64_t SPARSE_INSTANCES = 2;

int launch_render_bwd(const RenderBwdArgs& a, hipStream_t stream) {
  const uint32_t gx = (a.W + GS_TILE_X - 1) / GS_TILE_X, gy = (a.H + GS_TILE_Y - 1) / GS_TILE_Y;
  uint8_t* const written = a.R >= SPARSE_INSTANCES * (int64_t)a.W * a.H ? a.written : nullptr;
  if (written != nullptr) launch_fill_u32(((int64_t)a.R + 3) / 4, 0u, reinterpret_cast<uint32_t*>(written), stream);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(gx * gy), dim3(GS_TILE_PIX), 0, stream, (const uint2*)a.ranges, a.point_list, a.W, a.H,
                       a.fx, a.fy, a.bg, (const float2*)a.means2D, (const float4*)a.conic_opacity, a.rgb, a.all_map,
                       a.all_map_pixels, a.final_T, a.n_contrib_px, a.compute_locally, a.dL_dpix, a.dL_dout_all_map,
                       a.dL_dout_plane_depth, a.emission_sorted, (float4*)a.instance_grads, written, a.block_hits,
                       (const float4*)a.packed, a.packed_valid, a.tile_order, a.tile_order_valid, gx);
  };
  if (a.render_geo) {
    if (a.block_hits) go(render_bwd_kernel<true, true>);
    else go(render_bwd_kernel<true, false>);
  } else {
    if (a.block_hits) go(render_bwd_kernel<false, true>);
    else go(render_bwd_kernel<false, false>);
  }
  auto reduce = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((a.P + GS_BLOCK_1D - 1) / GS_BLOCK_1D), dim3(GS_BLOCK_1D), 0, stream, a.P,
                       a.point_offsets, (const float4*)a.instance_grads, written, (float)(0.5 * a.W), (float)(0.5 * a.H),
                       a.render_geo, (float2*)a.dL_dmean2D, a.dL_dmean2D_abs, (float4*)a.dL_dconic_opacity,
                       a.dL_dcolors, a.dL_dall_map);
  };
  if (a.P >= REDUCE_STREAM_GAUSSIANS) {
    if (written != nullptr) reduce(reduce_instances_kernel<true, true>);
    else reduce(reduce_instances_kernel<true, false>);
  } else {
    if (written != nullptr) reduce(reduce_instances_kernel<false, true>);
    else reduce(reduce_instances_kernel<false, false>);
  }
  return 0;
}

}  // namespace gs
