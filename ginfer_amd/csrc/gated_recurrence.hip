// Linear attention whose forget gate also decides what is written (HGRN2), as a recurrence over per-request state:
//   q = silu(pq),  f = lower + (1 - lower) * sigmoid(pf + bias),  v = pv           (pq | pf | pv: one projection, 32-bit)
//   per head:  S_t = diag(f_t) S_(t-1) + (1 - f_t) v_t^T   (S is [dim, vdim]; f acts on the rows, which belong to q),
//              o_t = S_t^T q_t
// The state is 32-bit, [slot][head][dim][vdim]; a request whose q_start is 0 starts from zeros.  Gates, state and the
// output sum are 32-bit.  A workgroup owns one (entry, head, block of 8 or 16 value columns) and walks the entry's tokens in
// order (decay_walk.h): a token's result does not depend on how the request's tokens were cut into steps, nor on what else
// is in the batch.
// A second kernel norms each head's output over its value columns (RMS, with a weight per column).
#include "decay_rows.h"
#include "decay_walk.h"
#include "ginfer_amd.h"

#define GR_THREADS 256

// Measured on MI355X, the caches emptied before, us, before the walk of decay_walk.h -> now.  12 heads of 64 x 128: 2,048 tokens of
// one request 534 -> 181; five entries of 918 262 -> 183; 495 tokens beside 16 single ones 136 -> 64; 64 entries of 33 79 -> 65,
// of 9 34.1 -> 33.3, of one 24.5 -> 20.2.  28 heads of 128 x 128: 934 -> 511, 880 -> 564, 252 -> 191, 310 -> 244, 129 -> 121, 80 ->
// 70.  With k kept beside f in LDS, as the general walk has it, the reads of LDS made many entries slower than before (64 of 33
// tokens, 16 heads of 32 x 64, 35.2 -> 37.9, now 35.4; of 48 x 64 47 -> 61, now 46; 300 of 5, 16 x 32, 20.7 -> 28.6, now 19.8).
// What takes longer than before: 64 entries of 9 tokens of 32 x 64 and 48 x 64 (9 %), and 16 rows of state at 9 to 33 tokens of 64
// to 200 entries (17.8 against 16.7, 41 against 37).
template <int R, int COLS, int TILE>          // R rows of the state per thread: dim <= 16 * R
__global__ __launch_bounds__(dw_threads(COLS)) void hgrn2_scan_kernel(float* __restrict__ out, const float* __restrict__ proj,
                                                                       int64_t proj_stride, const float* __restrict__ f_bias,
                                                                       const float* __restrict__ lower, float* __restrict__ state,
                                                                       const int64_t* __restrict__ slots, const int32_t* __restrict__ cu,
                                                                       const int32_t* __restrict__ q_start, int heads, int dim, int vdim,
                                                                       int most) {
  const int e = blockIdx.x, h = blockIdx.y;
  const int first = cu[e], n = cu[e + 1] - first;
  if (n <= 0 || n > most) return;
  ForgetRows rows;
  rows.proj = proj + first * proj_stride + h * dim;
  rows.v = proj + first * proj_stride + 2 * heads * dim + h * vdim;
  rows.bias = f_bias + h * dim;
  rows.lower = lower + h * dim;
  rows.stride = proj_stride;
  rows.hd = heads * dim;
  decay_walk<R, COLS, TILE>(out + ((int64_t)first * heads + h) * vdim, rows, state + ((slots[e] * heads + h) * (int64_t)dim) * vdim,
                            q_start[e] == 0, n, heads, dim, vdim, (int)blockIdx.z * COLS);
}

// out[t, h, :] = x[t, h, :] / sqrt(mean(x[t, h, :]^2) + eps) * weight[:], one wavefront per (token, head)
template <typename T>
__global__ __launch_bounds__(GR_THREADS) void headwise_rmsnorm_kernel(T* __restrict__ out, const float* __restrict__ x,
                                                                       const float* __restrict__ weight, int64_t rows, int vdim,
                                                                       float eps) {
  const int64_t row = (int64_t)blockIdx.x * (GR_THREADS / WAVE) + threadIdx.x / WAVE;
  if (row >= rows) return;
  const int lane = threadIdx.x % WAVE;
  const float* p = x + row * vdim;
  float ss = 0.f;
  for (int i = lane; i < vdim; i += WAVE) ss += p[i] * p[i];
  ss = wave_sum(ss);
  const float rms = sqrtf(ss / (float)vdim + eps);
  for (int i = lane; i < vdim; i += WAVE) Num<T>::st(out + row * vdim + i, p[i] / rms * weight[i]);
}

extern "C" int ga_hgrn2_scan(void* out, const void* proj, int64_t proj_stride, const void* f_bias, const void* lower,
                             void* state, const void* slots, const void* cu, const void* q_start, int way, int most, int entries,
                             int heads, int dim, int vdim, hipStream_t stream) {
  if (entries <= 0) return 0;
  if (heads <= 0 || dim <= 0 || vdim <= 0 || dim > 16 * DW_SLICES || (way != 1 && way != 8 && way != 16)) return -1;
  if (heads > 65535 || (vdim + (way == 8 ? 7 : 15)) / (way == 8 ? 8 : 16) > 65535 || proj_stride >= (1ll << 27)) return -2;    // (a tile's offsets are 32-bit)
  const int rows = (dim + DW_SLICES - 1) / DW_SLICES;
#define GO(R, C, T) hipLaunchKernelGGL((hgrn2_scan_kernel<R, C, T>), dim3(entries, heads, (vdim + C - 1) / C), dim3(dw_threads(C)), 0, stream, \
                                       (float*)out, (const float*)proj, proj_stride, (const float*)f_bias, (const float*)lower,            \
                                       (float*)state, (const int64_t*)slots, (const int32_t*)cu, (const int32_t*)q_start, heads, dim, vdim, most)
  DW_WAY(way, rows, dw_many(entries, heads, vdim), GO);
#undef GO
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_headwise_rmsnorm(void* out, const void* x, const void* weight, int64_t rows, int vdim, float eps,
                                   int out_bf16, hipStream_t stream) {
  if (rows <= 0) return 0;
  if (vdim <= 0) return -1;
  const int per = GR_THREADS / WAVE;
  dim3 grid((unsigned)((rows + per - 1) / per)), block(GR_THREADS);
  if (out_bf16)
    hipLaunchKernelGGL(headwise_rmsnorm_kernel<bf16_t>, grid, block, 0, stream, (bf16_t*)out, (const float*)x,
                       (const float*)weight, rows, vdim, eps);
  else
    hipLaunchKernelGGL(headwise_rmsnorm_kernel<float>, grid, block, 0, stream, (float*)out, (const float*)x,
                       (const float*)weight, rows, vdim, eps);
  return GA_CHECK_LAUNCH();
}
