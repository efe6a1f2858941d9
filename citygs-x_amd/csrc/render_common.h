// Pieces shared by the forward and backward tile kernels: the pixel layout of a
// workgroup, the conservative test that culls Gaussians per 4x4 pixel block, and
// the cross-lane steps of the backward kernel's sums over pixels.
#pragma once

#include "gs_common.h"

namespace gs {

// Which Gaussians can pass the blend tests of cuda_rasterizer/forward.cu:381-393 (power <= 0 and
// opacity * exp(power) >= 1/255) somewhere in a block of pixels.  With conic (A, B, C) and
// tau = ln(255 * opacity), alpha >= 1/255 needs q(d) = A dx^2 + 2 B dx dy + C dy^2 <= 2 tau.
// cull_params returns (1/A, 1/C, q_max, q_pixel) with q_max = q_pixel = 2 (tau + 0.01).  q_max is +infinity when the conic
// cannot be trusted (every block then counts as hit) and negative when the opacity alone rules every pixel out; q_pixel
// does not depend on the conic and is never above 174, beyond which gs_expf returns 0 anyway.  Culling with these only
// skips work, it never changes a result.
__device__ __forceinline__ float4 cull_params(float4 co) {
  const float inf = __builtin_inff();
  const float o = co.w;
  if (o < 0.0039f) return make_float4(0.f, 0.f, -1.0f, GS_FORM_MAX);
  float4 cp = make_float4(0.f, 0.f, inf, GS_FORM_MAX);
  if (o < 1.0e30f) {
    const float tau = __logf(255.0f * o) + 0.01f;
    if (tau == tau) {
      cp.w = fminf(2.0f * tau, GS_FORM_MAX);
      const float det = co.x * co.z - co.y * co.y;
      // (the hardware reciprocal: 1/A and 1/C only place the point of a block edge where q is evaluated, and q
      // there exceeds the edge's minimum by the square of the placement error)
      const float ia = __builtin_amdgcn_rcpf(co.x), ic = __builtin_amdgcn_rcpf(co.z);
      if (det > 0.0f && co.x > 0.0f && co.z > 0.0f && ia < inf && ic < inf) cp = make_float4(ia, ic, 2.0f * tau, cp.w);
    }
  }
  return cp;
}

// What the block tests of a tile's kernels need of a Gaussian centred at xy: (1/A, 1/C, limit on q for a block, limit on
// q for a single pixel of the tile; the forward blend marks the pixels an entry can reach with the latter).  Both limits
// are those of cull_params plus a margin for rounding: the block test, the pixel mark and the blend itself
// evaluate q by different operation sequences at different points, each within a few units in the last place of
// the LARGEST term, which for a long thin Gaussian far from its centre is much larger than q itself.  Every such
// term is at most S = |A| X^2 + 2 |B| X Y + |C| Y^2 with X, Y the largest offsets of a pixel of the tile from the
// centre; the margin is 2e-6 S (about 32 units in the last place of S), on top of the 0.02 from tau + 0.01.  The
// block limit is negative when the opacity alone rules every pixel out and +infinity when the conic cannot be
// trusted.  The same numbers in the forward and the backward kernel, so both build the same lists.
__device__ __forceinline__ float4 block_test_params(float4 co, float2 xy, float tile_x0, float tile_y0) {
  const float4 cp = cull_params(co);
  const float far_x = fmaxf(fabsf(xy.x - tile_x0), fabsf(xy.x - (tile_x0 + (float)(GS_TILE_X - 1))));
  const float far_y = fmaxf(fabsf(xy.y - tile_y0), fabsf(xy.y - (tile_y0 + (float)(GS_TILE_Y - 1))));
  const float spread = fabsf(co.x) * far_x * far_x + 2.0f * fabsf(co.y) * far_x * far_y + fabsf(co.z) * far_y * far_y;
  const float pixel_limit = __builtin_fmaf(2e-6f, spread, cp.w);
  const bool never = cp.z < 0.f, untrusted = cp.z == __builtin_inff();
  return make_float4(cp.x, cp.y, never ? -1.0f : (untrusted ? cp.z : pixel_limit), pixel_limit);
}

// bits <- 4 bits + 2 [a does not exceed limit_a] + [b does not exceed limit_b], NaNs not exceeding: each answer is shifted
// in at bit 0, as the carry of bits + bits.  A vector instruction that reads a lane mask needs two issue slots between it
// and the vector instruction that wrote the mask, and the compiler does not look into the statement to put them there: the
// other comparison, the other addition and one idle slot are in between.
__device__ __forceinline__ void shift_in_two(uint32_t& bits, float a, float limit_a, float b, float limit_b) {
  uint64_t mask;
  asm("v_cmp_ngt_f32 %1, %2, %3\n\t"
      "v_cmp_ngt_f32 vcc, %4, %5\n\t"
      "s_nop 0\n\t"
      "v_addc_co_u32 %0, %1, %0, %0, %1\n\t"
      "v_addc_co_u32 %0, vcc, %0, %0, vcc"
      : "+v"(bits), "=&s"(mask)
      : "v"(a), "v"(limit_a), "v"(b), "v"(limit_b)
      : "vcc");
}

// What the block tests of two neighbouring columns of 4x4 blocks have in common (x0: the left one's first pixel).
struct BlockColumns {
  float lox[2], t1[2], a1[2], b1[2];
};

__device__ __forceinline__ BlockColumns block_columns(float2 mu, float4 co, float inv_c, float x0) {
  const float two_b = 2.0f * co.y;
  BlockColumns b;
#pragma unroll
  for (int c = 0; c < 2; c++) {
    b.lox[c] = (x0 + (float)(4 * c)) - mu.x;
    const float dxc = __builtin_amdgcn_fmed3f(0.f, b.lox[c], b.lox[c] + 3.0f);  // offset of the block's nearest column
    b.t1[c] = -co.y * dxc * inv_c;                                              // where q is smallest along that column
    b.a1[c] = co.x * dxc * dxc;
    b.b1[c] = two_b * dxc;
  }
  return b;
}

// hits <- 4 hits + 2 [right block] + [left block] of the two columns' row of blocks whose first pixel is at y0.
__device__ __forceinline__ void test_block_pair(uint32_t& hits, const BlockColumns& b, float2 mu, float4 co, float inv_a,
                                                float limit, float y0) {
  const float loy = y0 - mu.y;
  const float hiy = loy + 3.0f;
  const float dyc = __builtin_amdgcn_fmed3f(0.f, loy, hiy);  // offset of the block's nearest row
  const float t2 = -co.y * dyc * inv_a;                      // where q is smallest along that row
  const float a2 = co.z * dyc * dyc;
  const float b2 = 2.0f * co.y * dyc;
  float nearest[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const float dy1 = __builtin_amdgcn_fmed3f(b.t1[c], loy, hiy);  // best point of the column x = dxc
    const float q1 = __builtin_fmaf(__builtin_fmaf(co.z, dy1, b.b1[c]), dy1, b.a1[c]);
    const float dx2 = __builtin_amdgcn_fmed3f(t2, b.lox[c], b.lox[c] + 3.0f);  // best point of the row y = dyc
    const float q2 = __builtin_fmaf(__builtin_fmaf(co.x, dx2, b2), dx2, a2);
    nearest[c] = fminf(q1, q2);
  }
  shift_in_two(hits, nearest[1], limit, nearest[0], limit);
}

// The sixteen 4x4 pixel blocks of the tile at (tile_x0, tile_y0): bit 4 k + r of the result is block r of quadrant k
// (quadrant k at offset 8 (k & 1), 8 (k >> 1), block r in it at 4 (r & 1), 4 (r >> 1)): can any point of the block have
// q <= limit?  q is convex, so over a block it is smallest either at the centre (inside the block: 0) or on one of the two
// block edges that face the centre; along an edge it is a parabola whose minimiser is clamped to the edge.  A block is
// treated as a continuous rectangle, which can only add hits.  What the four columns and the four rows of blocks have in
// common is computed once; the parabolas are evaluated in Horner form with fused multiply-adds.  inv_a, inv_c and limit:
// block_test_params.  NaNs count as hits.
__device__ __forceinline__ uint32_t ellipse_hits_tile(float2 mu, float4 co, float inv_a, float inv_c, float limit,
                                                      float tile_x0, float tile_y0) {
  uint32_t hits = 0u;  // (columns 2 h and 2 h + 1 of row d: bits 8 h + 2 d and the next)
#pragma unroll 1
  for (int h = 1; h >= 0; h--) {  // (loops: unrolled they take registers that the blend kernels do not have)
    const BlockColumns b = block_columns(mu, co, inv_c, tile_x0 + (float)(8 * h));
#pragma unroll 1
    for (int d = 3; d >= 0; d--) test_block_pair(hits, b, mu, co, inv_a, limit, tile_y0 + (float)(4 * d));
  }
  // row d of columns 2 h, 2 h + 1 are blocks 2 (d & 1), 2 (d & 1) + 1 of quadrant 2 (d >> 1) + h
  return (hits & 0xF00Fu) | ((hits & 0x00F0u) << 4) | ((hits & 0x0F00u) >> 4);
}

// The same tests for the four blocks of the quadrant at (x0, y0): bits 4 k .. 4 k + 3 of ellipse_hits_tile (the offsets of
// pixels are whole numbers, so they are the same whichever corner they are counted from).
__device__ __forceinline__ uint32_t ellipse_hits_quadrant(float2 mu, float4 co, float inv_a, float inv_c, float limit,
                                                          float x0, float y0) {
  uint32_t hits = 0u;
  const BlockColumns b = block_columns(mu, co, inv_c, x0);
#pragma unroll
  for (int d = 1; d >= 0; d--) test_block_pair(hits, b, mu, co, inv_a, limit, y0 + (float)(4 * d));
  return hits;
}

// How the forward blend hands a Gaussian's sixteen hits to the backward blend: a word with byte k for quadrant k, whose
// lower four bits are the quadrant's blocks (bytes, because the quadrants of a long tile are blended by workgroups of
// their own).
__device__ __forceinline__ uint32_t hits_to_bytes(uint32_t hits) {
  return (hits & 0xFu) | ((hits & 0xF0u) << 4) | ((hits & 0xF00u) << 8) | ((hits & 0xF000u) << 12);
}
__device__ __forceinline__ uint32_t hits_from_bytes(uint32_t bytes) {
  return (bytes & 0xFu) | ((bytes >> 4) & 0xF0u) | ((bytes >> 8) & 0xF00u) | ((bytes >> 12) & 0xF000u);
}

// ---- 4x4-pixel rows -------------------------------------------------------
// Inside a wave's 8x8 quadrant every 16-lane DPP row owns a 4x4 pixel block
// (row r at x offset 4*(r&1), y offset 4*(r>>1); lane l16 of the row is pixel
// (l16 & 3, l16 >> 2) of the block).  The blend loops let the four rows of a
// wave walk four different Gaussians at the same time, each row following its
// own list of Gaussians whose box meets its 4x4 block.
struct RowThread {
  int lane, wave, row, l16;
  uint32_t px, py;
  float qx0, qy0;  // top-left pixel of the wave's quadrant
};

__device__ __forceinline__ RowThread row_thread(uint32_t tile_x, uint32_t tile_y) {
  RowThread t;
  const int tid = threadIdx.x;
  t.lane = tid & (GS_WAVE - 1);
  t.wave = tid / GS_WAVE;
  t.row = t.lane >> 4;
  t.l16 = t.lane & 15;
  const uint32_t x0 = tile_x * GS_TILE_X + (uint32_t)(t.wave & 1) * 8u;
  const uint32_t y0 = tile_y * GS_TILE_Y + (uint32_t)(t.wave >> 1) * 8u;
  t.px = x0 + (uint32_t)(t.row & 1) * 4u + (uint32_t)(t.l16 & 3);
  t.py = y0 + (uint32_t)(t.row >> 1) * 4u + (uint32_t)(t.l16 >> 2);
  t.qx0 = (float)x0;
  t.qy0 = (float)y0;
  return t;
}

// ---- quads ----------------------------------------------------------------
// In the backward blend's second half a quad of lanes works for four entries and its registers for four pixels.

// Transposes the 4x4 blocks of a and b inside every quad: register e of lane p becomes register p of lane e.  A DPP
// operand written by the preceding VALU instruction needs two idle issue slots first, a matrix instruction one.
__device__ __forceinline__ void quad_transpose2(float (&a)[4], float (&b)[4]) {
  const uint64_t bit0 = 0xAAAAAAAAAAAAAAAAull, bit1 = 0xCCCCCCCCCCCCCCCCull;
  float c[4], d[4];
  asm volatile(
      "s_nop 1\n\t"
      "s_mov_b64 vcc, %16\n\t"
      "v_cndmask_b32_dpp %1, %8, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %10, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %12, %13, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %14, %15, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"
      "v_cndmask_b32_dpp %0, %9, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %2, %11, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %4, %13, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %15, %14, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      : "=&v"(c[0]), "=&v"(c[1]), "=&v"(c[2]), "=&v"(c[3]), "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "s"(bit0)
      : "vcc", "scc");
  asm volatile(
      "s_nop 1\n\t"
      "s_mov_b64 vcc, %16\n\t"
      "v_cndmask_b32_dpp %2, %8, %10, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %9, %11, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %12, %14, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %13, %15, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"
      "v_cndmask_b32_dpp %0, %10, %8, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %1, %11, %9, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %4, %14, %12, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %15, %13, vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
      "s_nop 1"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3])
      : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "s"(bit1)
      : "vcc", "scc");
}

// Sums sixteen values over the four quads of every 16-lane row and leaves values 4 q .. 4 q + 3 in quad q, in v[0..3]
// (v is overwritten).  Two halving steps, two instructions per value kept: the bank mask of a DPP addition selects the
// quads that take its result.  Results are written before the last operands are read, so no operand may share a result's
// register, whatever its value.  The matrix results among the inputs need up to seven idle slots first.  LAST = false:
// v[12..15] are not given, and quad 3 ends up with no meaningful sums.
template <bool LAST>
__device__ __forceinline__ void quads_reduce16(float (&v)[16]) {
  if (LAST)
    asm volatile(
        "s_nop 7\n\t"
        "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %6, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %7, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %4, %12, %12 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %5, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %6, %14, %14 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %7, %15, %15 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        : "+&v"(v[0]), "+&v"(v[1]), "+&v"(v[2]), "+&v"(v[3]), "+&v"(v[4]), "+&v"(v[5]), "+&v"(v[6]), "+&v"(v[7])
        : "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]), "v"(v[12]), "v"(v[13]), "v"(v[14]), "v"(v[15]));
  else
    asm volatile(
        "s_nop 7\n\t"
        "v_add_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %3, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %4, %4, %4 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %5, %5, %5 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %6, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %7, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        : "+&v"(v[0]), "+&v"(v[1]), "+&v"(v[2]), "+&v"(v[3]), "+&v"(v[4]), "+&v"(v[5]), "+&v"(v[6]), "+&v"(v[7])
        : "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]));
  asm volatile(
      "s_nop 1\n\t"
      "v_add_f32_dpp %0, %0, %0 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %1, %1, %1 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %2, %2, %2 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %3, %3, %3 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
      "v_add_f32_dpp %0, %4, %4 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %1, %5, %5 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %2, %6, %6 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
      "v_add_f32_dpp %3, %7, %7 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
      : "+&v"(v[0]), "+&v"(v[1]), "+&v"(v[2]), "+&v"(v[3])
      : "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
}

}  // namespace gs
