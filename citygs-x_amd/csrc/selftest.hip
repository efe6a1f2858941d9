// Device self-tests of what the blend kernels build on and no result of theirs shows on its own: the cross-lane steps
// in inline assembly, and the reciprocal, whose rounding rests on the hardware's approximation.
#include "gs_common.h"
#include "gs_kernels.h"
#include "render_common.h"

namespace gs {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// in: [64 lanes][16 values]; out_wave[16] = sums over the 64 lanes;
// out_rows[4][16] = sums over each 16-lane row.
__global__ void __launch_bounds__(GS_WAVE) reduce_selftest_kernel(const float* __restrict__ in,
                                                                  float* __restrict__ out_wave,
                                                                  float* __restrict__ out_rows) {
  const int lane = threadIdx.x, row = lane >> 4, quad = (lane & 15) >> 2, e = lane & 3;
  float v[16], s[4];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = in[lane * 16 + q];
  // over a quad's lanes: s[c] in lane e belongs to value 4 c + e
#pragma unroll
  for (int c = 0; c < 4; c += 2) {
    float a[4] = {v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]};
    float b[4] = {v[4 * c + 4], v[4 * c + 5], v[4 * c + 6], v[4 * c + 7]};
    quad_transpose2(a, b);
    s[c] = (a[0] + a[1]) + (a[2] + a[3]);
    s[c + 1] = (b[0] + b[1]) + (b[2] + b[3]);
  }
  // over the row's quads, the same four sums for every quad
  float w[16];
#pragma unroll
  for (int q = 0; q < 16; q++) w[q] = s[q & 3];
  quads_reduce16<true>(w);
  const float mine = quad == 0 ? w[0] : quad == 1 ? w[1] : quad == 2 ? w[2] : w[3];
  out_rows[row * 16 + 4 * quad + e] = mine;
  float t = mine + __shfl_xor(mine, 16, GS_WAVE);
  t += __shfl_xor(t, 32, GS_WAVE);
  if (row == 0) out_wave[4 * quad + e] = t;
}

// Every step on its own.  in: [64 lanes][16 values v]; out, [64 lanes][24]: 0-7 quad_transpose2 of v[0..3] and v[4..7];
// 8-11 quads_reduce16 of v; 12-15 the same without v[12..15]; 16-19 of v[0..7] twice (operands of equal value);
// 20-23 the 4x4 outer product of v[0] and v[1].
__global__ void __launch_bounds__(GS_WAVE) quad_selftest_kernel(const float* __restrict__ in, float* __restrict__ out) {
  const int lane = threadIdx.x;
  float v[16];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = in[lane * 16 + q];
  float* o = out + 24 * lane;
  auto put = [&](int at, const float* r) {
#pragma unroll
    for (int k = 0; k < 4; k++) o[at + k] = r[k];
  };
  float a[4] = {v[0], v[1], v[2], v[3]}, b[4] = {v[4], v[5], v[6], v[7]}, w[16];
  quad_transpose2(a, b);
  put(0, a);
  put(4, b);
#pragma unroll
  for (int q = 0; q < 16; q++) w[q] = v[q];
  quads_reduce16<true>(w);
  put(8, w);
#pragma unroll
  for (int q = 0; q < 16; q++) w[q] = v[q];
  quads_reduce16<false>(w);
  put(12, w);
#pragma unroll
  for (int q = 0; q < 16; q++) w[q] = v[q & 7];
  quads_reduce16<true>(w);
  put(16, w);
  f32x4 d = {0.f, 0.f, 0.f, 0.f};
  d = __builtin_amdgcn_mfma_f32_4x4x1f32(v[0], v[1], d, 0, 0, 0);
#pragma unroll
  for (int k = 0; k < 4; k++) o[20 + k] = d[k];
}

// gs_rcp_normal against the division on the floats whose bits are first, first + 1, ...: out[0] counts those it
// rounds differently, out[1] is the largest of them.
__global__ void __launch_bounds__(GS_BLOCK_1D) reciprocal_selftest_kernel(uint32_t first, uint32_t n,
                                                                          uint32_t* __restrict__ out) {
  for (uint32_t i = blockIdx.x * GS_BLOCK_1D + threadIdx.x; i < n; i += gridDim.x * GS_BLOCK_1D) {
    const float d = __uint_as_float(first + i);
    if (__float_as_uint(gs_rcp_normal(d)) != __float_as_uint(1.0f / d)) {
      atomicAdd(&out[0], 1u);
      atomicMax(&out[1], first + i);
    }
  }
}

}  // namespace

int launch_reduce_selftest(const float* in, float* out_wave, float* out_rows, hipStream_t stream) {
  hipLaunchKernelGGL(reduce_selftest_kernel, dim3(1), dim3(GS_WAVE), 0, stream, in, out_wave, out_rows);
  return 0;
}

int launch_reciprocal_selftest(uint32_t first, uint32_t n, uint32_t* out, hipStream_t stream) {
  hipLaunchKernelGGL(reciprocal_selftest_kernel, dim3(2048), dim3(GS_BLOCK_1D), 0, stream, first, n, out);
  return 0;
}

int launch_quad_selftest(const float* in, float* out, hipStream_t stream) {
  hipLaunchKernelGGL(quad_selftest_kernel, dim3(1), dim3(GS_WAVE), 0, stream, in, out);
  return 0;
}

}  // namespace gs
