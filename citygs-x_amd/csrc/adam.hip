// Fused multi-tensor Adam step: the optimizer the reference trains every parameter group with,
// torch.optim.Adam(lr=0.0, eps=1e-15) with per-group learning rates (scene/gaussian_model.py:574;
// stepped at train_internal.py:404-417, after "param.grad /= bsz" at :407-410, which is folded in here as
// grad_scale).  Update rule of torch 2.0.0 (the version the reference pins), default betas, no weight
// decay, no amsgrad:
// (hyper-parameters arrive as doubles, like the Python floats of that optimizer: 1-b is formed in double
// and only then rounded to fp32)
//   m = m*b1 + (1-b1)*g;  v = v*b2 + (1-b2)*g*g;
//   p = p - (lr / (1-b1^t)) * m / (sqrt(v)/sqrt(1-b2^t) + eps)
// One launch covers up to ADAM_MAX_TENSORS tensors: a workgroup looks its (tensor, chunk) up in a small
// table passed by value, so the ~20 small MLP tensors cost no launches of their own.  28 bytes per
// element (p, g, m, v in; p, m, v out), 16-byte accesses wherever the four pointers allow.
//
// Bound by HBM.  A step over more than the last-level cache holds goes past the caches in both directions (loads alone or
// stores alone gain nothing), one 16-byte vector of each array per thread in workgroups of two waves: 59 M elements
// take 264 us, 6.26 TB/s, against 307 us and 5.38 TB/s with cached accesses, four vectors a thread and four waves; workgroups
// of one to sixteen waves with one to eight vectors lie between 264 and 296 us.
#include "gs_common.h"
#include "gs_kernels.h"

namespace gs {

namespace {

constexpr int ADAM_THREADS = 128;
constexpr int ADAM_VEC = 4;  // one 16-byte vector of each array per thread
constexpr int ADAM_CHUNK = ADAM_THREADS * ADAM_VEC;  // elements per workgroup
// From here on (320 MB in the four arrays) a step streams.  Below, the 256 MB cache keeps a part from one step to the next
// if nothing else runs between them: 17.7 M elements 72 us cached and 79 streamed in a loop of steps, 23.6 M 112 and 106.
// (With 640 MB written between the steps streaming is the faster at every size: 17.7 M 85 against 106 us, 1.2 M 11 against 13.)
constexpr long long ADAM_STREAM_ELEMENTS = 20'000'000;
// A launch's threads are counted in 32 bits (2^25 workgroups), and the tensors of one step may fill the memory with more:
// a launch takes at most this many workgroups (537 M elements, 2.4 ms), and a tensor that does not fit goes on in the next.
constexpr int ADAM_MAX_CHUNKS = 1 << 20;

struct AdamTable {
  float* p[ADAM_MAX_TENSORS];
  const float* g[ADAM_MAX_TENSORS];
  float* m[ADAM_MAX_TENSORS];
  float* v[ADAM_MAX_TENSORS];
  long long n[ADAM_MAX_TENSORS];
  float neg_step_size[ADAM_MAX_TENSORS];  // -(lr / (1 - b1^t)), per tensor (per-group lr and step)
  float bc2_sqrt[ADAM_MAX_TENSORS];       // sqrt(1 - b2^t)
  int first_chunk[ADAM_MAX_TENSORS + 1];  // prefix sum of chunk counts
  int count;
};

__device__ __forceinline__ void adam_update(float& p, float g, float& m, float& v, float b1, float omb1, float b2,
                                            float omb2, float eps, float neg_step, float bc2s) {
  m = m * b1 + omb1 * g;
  v = v * b2 + (omb2 * g) * g;
  const float denom = sqrtf(v) / bc2s + eps;
  p = p + (neg_step * m) / denom;
}

typedef float v4f __attribute__((ext_vector_type(4)));

// STREAM: past the caches
template <bool STREAM, typename T>
__device__ __forceinline__ T get(const T* p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(p);
  return *p;
}

template <bool STREAM, typename T>
__device__ __forceinline__ void put(T* p, T v) {
  if constexpr (STREAM) __builtin_nontemporal_store(v, p);
  else *p = v;
}

template <bool STREAM>
__global__ void __launch_bounds__(ADAM_THREADS)
adam_kernel(const AdamTable t, float b1, float omb1, float b2, float omb2, float eps, float grad_scale) {
  // which tensor does this workgroup belong to (the table is tiny and uniform: scalar loads)
  int k = 0;
  while (k + 1 < t.count && (int)blockIdx.x >= t.first_chunk[k + 1]) k++;
  const long long n = t.n[k];
  const long long base = (long long)((int)blockIdx.x - t.first_chunk[k]) * ADAM_CHUNK;
  float* __restrict__ p = t.p[k];
  const float* __restrict__ g = t.g[k];
  float* __restrict__ m = t.m[k];
  float* __restrict__ v = t.v[k];
  const float neg_step = t.neg_step_size[k], bc2s = t.bc2_sqrt[k];
  const bool aligned = ((((uintptr_t)p | (uintptr_t)g | (uintptr_t)m | (uintptr_t)v) & 15) == 0);
  if (aligned && base + ADAM_CHUNK <= n) {
    const long long e = base + (long long)threadIdx.x * ADAM_VEC;
    v4f P = get<STREAM>((const v4f*)(p + e));
    const v4f G = get<STREAM>((const v4f*)(g + e));
    v4f M = get<STREAM>((const v4f*)(m + e)), V = get<STREAM>((const v4f*)(v + e));
#pragma unroll
    for (int c = 0; c < ADAM_VEC; c++) {
      float pe = P[c], me = M[c], ve = V[c];
      adam_update(pe, G[c] * grad_scale, me, ve, b1, omb1, b2, omb2, eps, neg_step, bc2s);
      P[c] = pe;
      M[c] = me;
      V[c] = ve;
    }
    put<STREAM>((v4f*)(p + e), P);
    put<STREAM>((v4f*)(m + e), M);
    put<STREAM>((v4f*)(v + e), V);
  } else {
    float pe[ADAM_VEC], ge[ADAM_VEC], me[ADAM_VEC], ve[ADAM_VEC];
#pragma unroll
    for (int i = 0; i < ADAM_VEC; i++) {
      const long long e = base + (long long)i * ADAM_THREADS + threadIdx.x;
      if (e < n) {
        pe[i] = get<STREAM>(p + e);
        ge[i] = get<STREAM>(g + e);
        me[i] = get<STREAM>(m + e);
        ve[i] = get<STREAM>(v + e);
      }
    }
#pragma unroll
    for (int i = 0; i < ADAM_VEC; i++) {
      const long long e = base + (long long)i * ADAM_THREADS + threadIdx.x;
      if (e < n) {
        adam_update(pe[i], ge[i] * grad_scale, me[i], ve[i], b1, omb1, b2, omb2, eps, neg_step, bc2s);
        put<STREAM>(p + e, pe[i]);
        put<STREAM>(m + e, me[i]);
        put<STREAM>(v + e, ve[i]);
      }
    }
  }
}

// The next launch of a step over `count` tensors: slice i is the elements first[i] .. first[i] + n[i] - 1 of tensor
// index[i] and begins at workgroup first_chunk[i].  (tensor, element) is where the launch begins and is moved on; no slice
// is left when all tensors are done.
struct AdamSlices {
  int count, chunks;
  int index[ADAM_MAX_TENSORS], first_chunk[ADAM_MAX_TENSORS];
  long long first[ADAM_MAX_TENSORS], n[ADAM_MAX_TENSORS];
};

AdamSlices adam_next_launch(int count, const long long* sizes, int& tensor, long long& element) {
  AdamSlices s;
  s.count = s.chunks = 0;
  while (tensor < count && s.count < ADAM_MAX_TENSORS && s.chunks < ADAM_MAX_CHUNKS) {
    const long long left = sizes[tensor] - element, room = (long long)(ADAM_MAX_CHUNKS - s.chunks) * ADAM_CHUNK;
    const long long n = left < room ? left : room;
    if (n > 0) {
      s.index[s.count] = tensor;
      s.first_chunk[s.count] = s.chunks;
      s.first[s.count] = element;
      s.n[s.count++] = n;
      s.chunks += (int)((n + ADAM_CHUNK - 1) / ADAM_CHUNK);
      element += n;
    }
    if (n == left || left <= 0) {
      tensor++;
      element = 0;
    }
  }
  return s;
}

}  // namespace

long long adam_plan(int count, const long long* sizes, long long* out, long long capacity) {
  long long rows = 0;
  int tensor = 0;
  long long element = 0;
  for (int launch = 0;; launch++) {
    const AdamSlices s = adam_next_launch(count, sizes, tensor, element);
    if (s.count == 0) return rows;
    for (int i = 0; i < s.count; i++, rows++) {
      if (rows >= capacity) continue;
      const long long row[5] = {launch, s.index[i], s.first[i], s.n[i], (long long)s.chunks * ADAM_THREADS};
      for (int k = 0; k < 5; k++) out[5 * rows + k] = row[k];
    }
  }
}

int launch_adam(int count, float* const* params, const float* const* grads, float* const* exp_avg,
                float* const* exp_avg_sq, const long long* sizes, const double* lrs, const int* steps, double beta1,
                double beta2, double eps, float grad_scale, hipStream_t stream) {
  long long elements = 0;
  for (int i = 0; i < count; i++) elements += sizes[i] > 0 ? sizes[i] : 0;
  const auto kernel = elements > ADAM_STREAM_ELEMENTS ? adam_kernel<true> : adam_kernel<false>;
  int tensor = 0;
  long long element = 0;
  for (;;) {
    const AdamSlices s = adam_next_launch(count, sizes, tensor, element);
    if (s.count == 0) break;
    AdamTable t;
    for (int k = 0; k < s.count; k++) {
      const int i = s.index[k];
      t.p[k] = params[i] + s.first[k];
      t.g[k] = grads[i] + s.first[k];
      t.m[k] = exp_avg[i] + s.first[k];
      t.v[k] = exp_avg_sq[i] + s.first[k];
      t.n[k] = s.n[k];
      // bias corrections in double, like the Python floats of the reference optimizer
      const double bc1 = 1.0 - pow(beta1, (double)steps[i]);
      const double bc2 = 1.0 - pow(beta2, (double)steps[i]);
      t.neg_step_size[k] = (float)(-(lrs[i] / bc1));
      t.bc2_sqrt[k] = (float)sqrt(bc2);
      t.first_chunk[k] = s.first_chunk[k];
    }
    t.first_chunk[s.count] = s.chunks;
    t.count = s.count;
    hipLaunchKernelGGL(kernel, dim3(s.chunks), dim3(ADAM_THREADS), 0, stream, t, (float)beta1,
                       (float)(1.0 - beta1), (float)beta2, (float)(1.0 - beta2), (float)eps, grad_scale);
  }
  return 0;
}

}  // namespace gs
