// RMS norm whose gain is ONE number for all coordinates, in the two places a model uses it:
//   rows:   out[r] = g * x[rows[r]] / sqrt(mean(x^2) + eps)             (the norm before the output head)
//   add:    residual[t] += g * y[t] / sqrt(mean(y[t]^2) + eps)          (a norm on a sublayer's OUTPUT: the
//           sublayer's result is normalised and then added to the 32-bit residual stream), optionally with a copy
//           of the new residual row in the compute dtype, which is what the next matrix product reads.
// All arithmetic in 32-bit; the sum over a row is taken in an order that depends on the row's length alone.
#include "common.h"
#include "ginfer_amd.h"

#define SN_THREADS 256

template <typename T, typename G>
__global__ __launch_bounds__(SN_THREADS) void scalar_rmsnorm_rows_kernel(T* __restrict__ out, const float* __restrict__ x,
                                                                          const G* __restrict__ gain,
                                                                          const int32_t* __restrict__ rows, int hidden,
                                                                          float eps) {
  __shared__ float scratch[SN_THREADS / WAVE];
  const int64_t r = blockIdx.x;
  const int64_t t = rows ? (int64_t)rows[r] : r;
  const float* row = x + t * hidden;
  float ss = 0.f;
  for (int i = threadIdx.x; i < hidden; i += SN_THREADS) ss += row[i] * row[i];
  ss = block_sum<SN_THREADS / WAVE>(ss, scratch);
  const float rms = sqrtf(ss / (float)hidden + eps), g = Num<G>::ld(gain);
  for (int i = threadIdx.x; i < hidden; i += SN_THREADS) Num<T>::st(out + r * hidden + i, row[i] / rms * g);
}

// Y: the sublayer's output (compute dtype, or float partial sums); C: the dtype of the copy
template <typename Y, typename G, typename C>
__global__ __launch_bounds__(SN_THREADS) void add_scalar_rmsnorm_kernel(float* __restrict__ residual, const Y* __restrict__ y,
                                                                         const G* __restrict__ gain, C* __restrict__ copy,
                                                                         int hidden, float eps) {
  __shared__ float scratch[SN_THREADS / WAVE];
  const int64_t t = blockIdx.x;
  const Y* row = y + t * hidden;
  float ss = 0.f;
  for (int i = threadIdx.x; i < hidden; i += SN_THREADS) {
    const float v = Num<Y>::ld(row + i);
    ss += v * v;
  }
  ss = block_sum<SN_THREADS / WAVE>(ss, scratch);
  const float rms = sqrtf(ss / (float)hidden + eps), g = Num<G>::ld(gain);
  for (int i = threadIdx.x; i < hidden; i += SN_THREADS) {
    const float h = residual[t * hidden + i] + Num<Y>::ld(row + i) / rms * g;
    residual[t * hidden + i] = h;
    if (copy) Num<C>::st(copy + t * hidden + i, h);
  }
}

// The same where a row is at most SN_THREADS * 4 * PER elements, a multiple of 4 at 16-byte addresses: a thread asks for all of
// its row's operands (four elements an access) before it uses the first, and the row stays in registers between the sum of
// squares and the add.  y may come as `parts` float rows, `part_stride` elements apart (a product with K split over
// workgroups), which are added up in order.  What bounds it is one way to memory and the sum over the workgroup.  Measured
// on MI355X, a decode step of 16 rows, six layers of 1,536 with 8,960 columns between: 596 -> 525 us with this kernel and the
// down product (96 workgroups over the whole of K before) in five parts of K.
template <typename Y, typename G, typename C, int PER>
__global__ __launch_bounds__(SN_THREADS) void add_scalar_rmsnorm_vec_kernel(float* __restrict__ residual,
                                                                             const Y* __restrict__ y, int parts,
                                                                             int64_t part_stride, const G* __restrict__ gain,
                                                                             C* __restrict__ copy, int hidden, float eps) {
  __shared__ float scratch[SN_THREADS / WAVE];
  const int64_t t = blockIdx.x;
  float4 v[PER], h[PER];
  auto four = [&](const Y* from) {
    if (sizeof(Y) == 4) return *reinterpret_cast<const float4*>(from);
    const uint2 u = *reinterpret_cast<const uint2*>(from);
    return make_float4(bf16_to_f32((bf16_t)(u.x & 0xffffu)), bf16_to_f32((bf16_t)(u.x >> 16)), bf16_to_f32((bf16_t)(u.y & 0xffffu)),
                       bf16_to_f32((bf16_t)(u.y >> 16)));
  };
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = 4 * (threadIdx.x + p * SN_THREADS);
    v[p] = h[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < hidden) {
      h[p] = *reinterpret_cast<const float4*>(residual + t * hidden + i);
      v[p] = four(y + t * hidden + i);
      for (int q = 1; q < parts; ++q) {
        const float4 more = four(y + q * part_stride + t * hidden + i);
        v[p] = make_float4(v[p].x + more.x, v[p].y + more.y, v[p].z + more.z, v[p].w + more.w);
      }
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    ss = fmaf(v[p].x, v[p].x, ss);
    ss = fmaf(v[p].y, v[p].y, ss);
    ss = fmaf(v[p].z, v[p].z, ss);
    ss = fmaf(v[p].w, v[p].w, ss);
  }
  ss = block_sum<SN_THREADS / WAVE>(ss, scratch);
  const float rms = sqrtf(ss / (float)hidden + eps), g = Num<G>::ld(gain);
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int i = 4 * (threadIdx.x + p * SN_THREADS);
    if (i >= hidden) continue;
    const float e[4] = {h[p].x + v[p].x / rms * g, h[p].y + v[p].y / rms * g, h[p].z + v[p].z / rms * g, h[p].w + v[p].w / rms * g};
    *reinterpret_cast<float4*>(residual + t * hidden + i) = make_float4(e[0], e[1], e[2], e[3]);
    if (copy) {
      union { C e[4]; uint2 u2; uint4 u4; } pk;
#pragma unroll
      for (int x = 0; x < 4; ++x) Num<C>::st(pk.e + x, e[x]);
      if (sizeof(C) == 2) *reinterpret_cast<uint2*>(copy + t * hidden + i) = pk.u2;
      else *reinterpret_cast<uint4*>(copy + t * hidden + i) = pk.u4;
    }
  }
}

extern "C" int ga_scalar_rmsnorm_rows(void* out, const void* x, const void* gain, const void* rows, int num_rows,
                                      int hidden, float eps, int out_bf16, int gain_bf16, hipStream_t stream) {
  if (num_rows <= 0) return 0;
  if (hidden <= 0) return -1;
  dim3 grid(num_rows), block(SN_THREADS);
#define GO(T, G) hipLaunchKernelGGL((scalar_rmsnorm_rows_kernel<T, G>), grid, block, 0, stream, (T*)out, (const float*)x, \
                                    (const G*)gain, (const int32_t*)rows, hidden, eps)
  if (out_bf16) { if (gain_bf16) GO(bf16_t, bf16_t); else GO(bf16_t, float); }
  else { if (gain_bf16) GO(float, bf16_t); else GO(float, float); }
#undef GO
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_add_scalar_rmsnorm(void* residual, const void* y, const void* gain, void* copy, int tokens, int hidden,
                                     float eps, int y_bf16, int gain_bf16, int parts, int copy_bf16, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (hidden <= 0 || parts < 1 || (y_bf16 && (parts > 1 || (copy && !copy_bf16)))) return -1;
  dim3 grid(tokens), block(SN_THREADS);
  const bool vec = hidden % 4 == 0 && hidden <= SN_THREADS * 16 &&
                   ((uintptr_t)residual & 15) == 0 && ((uintptr_t)y & (y_bf16 ? 7 : 15)) == 0 &&
                   ((uintptr_t)copy & (copy_bf16 ? 7 : 15)) == 0;
  if (parts > 1 && !vec) return -2;                      // the caller adds such rows up itself
  const int64_t part_stride = (int64_t)tokens * hidden;
#define GV(Y, G, C, PER) hipLaunchKernelGGL((add_scalar_rmsnorm_vec_kernel<Y, G, C, PER>), grid, block, 0, stream, (float*)residual, \
                                            (const Y*)y, parts, part_stride, (const G*)gain, (C*)copy, hidden, eps)
#define GS(Y, G, C) hipLaunchKernelGGL((add_scalar_rmsnorm_kernel<Y, G, C>), grid, block, 0, stream, (float*)residual, \
                                       (const Y*)y, (const G*)gain, (C*)copy, hidden, eps)
#define GO(Y, G, C)                                                                                                       \
  do {                                                                                                                    \
    if (!vec) GS(Y, G, C);                                                                                                \
    else if (hidden <= SN_THREADS * 4) GV(Y, G, C, 1);                                                                    \
    else if (hidden <= SN_THREADS * 8) GV(Y, G, C, 2);                                                                    \
    else GV(Y, G, C, 4);                                                                                                  \
  } while (0)
  if (y_bf16) { if (gain_bf16) GO(bf16_t, bf16_t, bf16_t); else GO(bf16_t, float, bf16_t); }
  else if (copy_bf16) { if (gain_bf16) GO(float, bf16_t, bf16_t); else GO(float, float, bf16_t); }
  else { if (gain_bf16) GO(float, bf16_t, float); else GO(float, float, float); }
#undef GO
#undef GS
#undef GV
  return GA_CHECK_LAUNCH();
}
