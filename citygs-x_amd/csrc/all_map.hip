// Per-Gaussian geometry channels of the blend ("all_map": camera-space normal, 1, plane distance) and
// their backward pass: the torch lines of gaussian_renderer/__init__.py:1501-1518 (quaternion_to_matrix
// of pytorch3d 0.3.0 on the normalised rotation, the axis of the smallest scale as normal, flipped
// towards the camera, rotated into the camera frame, distance = |normal . p_cam|) as one streaming
// kernel each way instead of about ten elementwise launches.  One thread per Gaussian; 40 bytes in and
// 20 out forward, 60 in and 28 out backward.  Sums run left to right with one rounding per operation.
#include "all_map_common.h"
#include "gs_common.h"
#include "gs_kernels.h"

namespace gs {

namespace {

__global__ void __launch_bounds__(GS_BLOCK_1D)
all_map_fwd_kernel(int P, const float* __restrict__ means, const float* __restrict__ scales,
                   const float* __restrict__ rots, const float* __restrict__ Vg, const float* __restrict__ camg,
                   float* __restrict__ out) {
  // the workgroup's 256 rows of 5 floats leave through LDS as 1280 consecutive floats (20-byte rows written
  // lane by lane would touch every line five times)
  __shared__ float s_out[5 * GS_BLOCK_1D];
  const int raw = blockIdx.x * GS_BLOCK_1D + threadIdx.x;
  const int i = raw < P ? raw : P - 1;
  float V[16], cam[3];
#pragma unroll
  for (int k = 0; k < 16; k++) V[k] = Vg[k];
#pragma unroll
  for (int k = 0; k < 3; k++) cam[k] = camg[k];
  const float m[3] = {means[3 * (size_t)i], means[3 * (size_t)i + 1], means[3 * (size_t)i + 2]};
  const float s[3] = {scales[3 * (size_t)i], scales[3 * (size_t)i + 1], scales[3 * (size_t)i + 2]};
  AllMapGeom g;
  all_map_geom(m, s, reinterpret_cast<const float4*>(rots)[i], V, cam, g);
  all_map_channels(g, s_out + 5 * threadIdx.x);
  __syncthreads();
  const size_t first = 5 * (size_t)blockIdx.x * GS_BLOCK_1D, total = 5 * (size_t)P;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const size_t e = first + (size_t)k * GS_BLOCK_1D + threadIdx.x;
    if (e < total) out[e] = s_out[k * GS_BLOCK_1D + threadIdx.x];
  }
}

__global__ void __launch_bounds__(GS_BLOCK_1D)
all_map_bwd_kernel(int P, const float* __restrict__ means, const float* __restrict__ scales,
                   const float* __restrict__ rots, const float* __restrict__ Vg, const float* __restrict__ camg,
                   const float* __restrict__ gout, float* __restrict__ dmeans, float* __restrict__ drots) {
  const int idx = blockIdx.x * GS_BLOCK_1D + threadIdx.x;
  if (idx >= P) return;
  float V[16], cam[3];
#pragma unroll
  for (int k = 0; k < 16; k++) V[k] = Vg[k];
#pragma unroll
  for (int k = 0; k < 3; k++) cam[k] = camg[k];
  const float m[3] = {means[3 * (size_t)idx], means[3 * (size_t)idx + 1], means[3 * (size_t)idx + 2]};
  const float s[3] = {scales[3 * (size_t)idx], scales[3 * (size_t)idx + 1], scales[3 * (size_t)idx + 2]};
  AllMapGeom g;
  all_map_geom(m, s, reinterpret_cast<const float4*>(rots)[idx], V, cam, g);
  const float* go = gout + 5 * (size_t)idx;
  float dmean[3], dq[4];
  all_map_gradient(g, V, go[0], go[1], go[2], go[4], dmean, dq);
#pragma unroll
  for (int a = 0; a < 3; a++) dmeans[3 * (size_t)idx + a] = dmean[a];
  reinterpret_cast<float4*>(drots)[idx] = make_float4(dq[0], dq[1], dq[2], dq[3]);
}

}  // namespace

int launch_all_map_fwd(int P, const float* means, const float* scales, const float* rots, const float* V,
                       const float* campos, float* out, hipStream_t stream) {
  if (P <= 0) return 0;
  hipLaunchKernelGGL(all_map_fwd_kernel, dim3((P + GS_BLOCK_1D - 1) / GS_BLOCK_1D), dim3(GS_BLOCK_1D), 0, stream, P,
                     means, scales, rots, V, campos, out);
  return 0;
}

int launch_all_map_bwd(int P, const float* means, const float* scales, const float* rots, const float* V,
                       const float* campos, const float* grad_out, float* dmeans, float* drots,
                       hipStream_t stream) {
  if (P <= 0) return 0;
  hipLaunchKernelGGL(all_map_bwd_kernel, dim3((P + GS_BLOCK_1D - 1) / GS_BLOCK_1D), dim3(GS_BLOCK_1D), 0, stream, P,
                     means, scales, rots, V, campos, grad_out, dmeans, drots);
  return 0;
}

}  // namespace gs
