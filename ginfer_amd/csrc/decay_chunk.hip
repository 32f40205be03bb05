// The recurrences of decay_walk.h in chunks of 64 tokens on the matrix cores' 32-bit instruction, for prompt portions long enough that the
// walk's chain of tokens is what they wait for.  Per head, S in front of the chunk, P_t the product of the decays a up to token t (from
// the chunk's start), R_t the product of those behind it (to the chunk's end), all per key channel:
//   states   U = (K R)^T V and D = P_63, for every chunk and head at once
//   carry    S <- D S + U from chunk to chunk, an element of the state a thread; leaves each chunk the state in front of it
//   out      O = (Q P) S + M V, M_ts = sum_i q_ti k_si a_(s+1)i .. a_ti for s <= t, for every chunk and head at once
// Decays enter only as products of up to 64 of them (no logarithms, no quotients), so a decay of 0 or next to it is like any other.  A
// chunk's 64 tokens are four runs of 16, a wavefront each: within a run M is added up channel by channel along the running product; between runs it is a matrix
// product of q times what decayed since its run began and k times what decays to its run's end (times the runs between).
//
// Why chunks: a walk's token costs its chain of dependent instructions, 57 ns at 64 rows of state, however idle the chip is.  Here a
// prompt of 2,048 with 12 heads makes 384 workgroups twice and the chain is 32 links of one multiply-add.  us, walk -> chunks, 12 heads
// of 64 x 128, 2,048 tokens: a decay per channel 116 -> 43, retention with rotation 145 -> 45, HGRN2 152 -> 45 (decay_in_chunks in
// kernels/ops.py has other sizes); of the 43 states take 13, carry 8.5 and out 21.  What bounds them: the states' way to memory and back (four times
// 3 MB a chunk of 12 heads), and in states and out one workgroup's own chain of loads, meetings and products (6.5 and 13.5 us with two
// chunks in all); two workgroups of out to a compute unit, where its 130 operands of the last products are not held along from the
// start, were 33 -> 25 us, whole chunks without conditions 25 -> 21.  Against 64 bits, walk and chunks, 1e-7 of the result (2-norm), 300 tokens: out 1.2 and 1.3 with a
// decay per channel, 2.0 and 1.7 with a constant one, 0.8 and 0.9 HGRN2; states 0.8 and 0.9, 2.0 and 1.4, 1.1 both.
//
// v_mfma_f32_16x16x4_f32: D[m][n] += sum_k A[m][k] B[k][n]; lane l supplies A[l % 16][k] and B[k][l % 16] of one k and receives D[4 (l /
// 16) + i][l % 16].  Four instructions i = 0 .. 3 cover 16 values of k, lane l supplying k = 4 (l / 16) + i.  Of 32 columns of v, a lane
// has 2 (l % 16) and the one behind it, one for each of two products.
#include "decay_rows.h"
#include "ginfer_amd.h"

#define DK_CHUNK 64
#define DK_RUN 16
#define DK_THREADS 256
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 dk_mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// chunks of entry e: numbers dk_first(e) on (never overlapping, some numbers unused, all below tokens / DK_CHUNK + entries)
__device__ __forceinline__ int dk_first(const int32_t* __restrict__ cu, int e) { return cu[e] / DK_CHUNK + e; }
__host__ __device__ constexpr int dk_cols(int vdim) { return (vdim + 31) / 32 * 32; }

struct DecayChunkArgs {
  float* out;
  float *u, *d;                        // [chunk][head][DP][dk_cols(vdim)]: U, then the state in front of the chunk; [chunk][head][DP]
  const float *q, *k, *v;              // (HGRN2: q the projection, k unused)
  int64_t stride;
  const float *decay, *head_decay, *cos_t, *sin_t;
  int rot_dims;
  float q_scale, k_scale;
  const float *f_bias, *lower;
  float* state;
  const int64_t* slots;
  const int32_t *cu, *q_start;
  int entries, heads, dim, vdim, least;      // least: shorter entries are left alone
};

enum { DK_PLAIN = 0, DK_ROT = 1, DK_SILU = 2, DK_FORGET = 3 };
template <int KIND>
struct ChunkRows {
  typedef typename std::conditional<KIND == DK_FORGET, ForgetRows, DecayRows<KIND == DK_ROT>>::type Rows;
};
// a head's rows from token `first` of the step on, which is at position `pos`
__device__ __forceinline__ void dk_rows(ForgetRows& r, const DecayChunkArgs& x, int64_t first, int, int h) {
  r.proj = x.q + first * x.stride + h * x.dim;
  r.v = x.v + first * x.stride + h * x.vdim;
  r.bias = x.f_bias + h * x.dim;
  r.lower = x.lower + h * x.dim;
  r.stride = x.stride;
  r.hd = x.heads * x.dim;
}
template <bool ROT>
__device__ __forceinline__ void dk_rows(DecayRows<ROT>& r, const DecayChunkArgs& x, int64_t first, int pos, int h) {
  r.q = x.q + first * x.stride + h * x.dim;
  r.k = x.k + first * x.stride + h * x.dim;
  r.v = x.v + first * x.stride + h * x.vdim;
  r.decay = x.decay ? x.decay + first * x.heads * x.dim + h * x.dim : x.head_decay + h;
  r.decay_token = x.decay ? x.heads * x.dim : 0;
  r.decay_channel = x.decay ? 1 : 0;
  r.half = x.rot_dims / 2;
  r.cos_t = ROT ? x.cos_t + (int64_t)pos * r.half : nullptr;
  r.sin_t = ROT ? x.sin_t + (int64_t)pos * r.half : nullptr;
  r.stride = x.stride;
  r.q_scale = x.q_scale;
  r.k_scale = x.k_scale;
  r.acts = false;                      // (unused: the kind says it)
}

// The chunk with a number: its entry's, or none.
struct ChunkPlace {
  int first, pos, n;                   // its first token in the step, that token's position, its tokens
  __device__ __forceinline__ bool find(const DecayChunkArgs& x, int id) {
    int lo = 0, hi = x.entries - 1;    // the last entry whose first chunk is not behind this one
    while (lo < hi) {
      const int m = (lo + hi + 1) / 2;
      if (dk_first(x.cu, m) <= id) lo = m;
      else hi = m - 1;
    }
    const int from = (id - dk_first(x.cu, lo)) * DK_CHUNK, begin = x.cu[lo], tokens = x.cu[lo + 1] - begin;
    if (from < 0 || from >= tokens || tokens < x.least) return false;
    first = begin + from;
    pos = x.q_start[lo] + from;
    n = min(tokens - from, DK_CHUNK);
    return true;
  }
};

// A channel's q, k and decay for the 16 tokens of a run, as the recurrence reads them; tokens and channels that do not exist write nothing
// and do not decay.  FULL: all of them exist.
template <int KIND, bool FULL, class Rows>
__device__ __forceinline__ void dk_run(const Rows& rows, int run, int n, int c, int dim, float (&q)[DK_RUN], float (&k)[DK_RUN],
                                       float (&a)[DK_RUN]) {
  typename Rows::Raw raw[DK_RUN];
  const int start = FULL ? run * DK_RUN : min(run * DK_RUN, n - 1), last = n - 1 - start, cc = FULL ? c : min(c, dim - 1);
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t) rows.load(raw[t], start, FULL ? t : min(t, last), cc);
  const typename Rows::Fixed fixed = rows.fixed(cc);
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t) {
    rows.template finish<KIND == DK_SILU>(raw[t], fixed, cc, q[t], k[t], a[t]);
    const bool in = FULL || (run * DK_RUN + t < n && c < dim);
    q[t] = in ? q[t] : 0.f;
    k[t] = in ? k[t] : 0.f;
    a[t] = in ? a[t] : 1.f;
  }
}

// Products of a run's decays up to each token, and behind each token to the run's end, rounded once: a decay that is the same for all tokens
// would lose the same way in every step of a product rounded each time, and in every chunk again.  Returns the whole run's.
__device__ __forceinline__ double dk_products(const float (&a)[DK_RUN], float (&up_to)[DK_RUN], float (&behind)[DK_RUN]) {
  double f = 1., r = 1.;
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t) up_to[t] = (float)(f *= (double)a[t]);
#pragma unroll
  for (int t = DK_RUN - 1; t >= 0; --t) {
    behind[t] = (float)r;
    r *= (double)a[t];
  }
  return f;
}

// 32 columns of v from c0 on, as the products take them: v[4 b + x] of row 16 b + 4 lg + x; zeros for what does not exist
template <int KIND, bool FULL, class Rows>
__device__ __forceinline__ void dk_values(const Rows& rows, int n, int c0, int vdim, int l16, int lg, float2 (&v)[16]) {
  const int c = c0 + 2 * l16, a = FULL ? c : min(c, vdim - 1), b = FULL ? c + 1 : min(c + 1, vdim - 1);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int run = i / 4, t = 4 * lg + i % 4, start = FULL ? run * DK_RUN : min(run * DK_RUN, n - 1), at = FULL ? t : min(t, n - 1 - start);
    v[i] = make_float2(rows.load_v(start, at, a), rows.load_v(start, at, b));
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const bool in = FULL || i / 4 * DK_RUN + 4 * lg + i % 4 < n;
    v[i].x = in && (FULL || c < vdim) ? rows.template finish_v<KIND == DK_SILU>(v[i].x) : 0.f;
    v[i].y = in && (FULL || c + 1 < vdim) ? rows.template finish_v<KIND == DK_SILU>(v[i].y) : 0.f;
  }
}

// DP: key channels, rounded up to 64 or 128; FULL: a whole chunk, and no channel or column that does not exist
template <int DP, int KIND, bool FULL>
__device__ __forceinline__ void decay_chunk_states(const DecayChunkArgs& x, const ChunkPlace& at, float (*ks)[DP + 4], double (*tot)[DP]) {
  constexpr int NB = DP / 16;
  const int id = blockIdx.x, h = blockIdx.y;
  typename ChunkRows<KIND>::Rows rows;
  dk_rows(rows, x, at.first, at.pos, h);
  const int tid = threadIdx.x, lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE), l16 = lane & 15, lg = lane >> 4;
  const int VP = dk_cols(x.vdim);
  const int c0 = blockIdx.z * 128 + 32 * w;
  float2 v[16];
  if (c0 < VP) dk_values<KIND, FULL>(rows, at.n, c0, x.vdim, l16, lg, v);
  float k[DP / 64][DK_RUN];            // times what decays to the run's end
#pragma unroll
  for (int p = 0; p < DP / 64; ++p) {
    const int c = lane + 64 * p;
    float q[DK_RUN], a[DK_RUN], up_to[DK_RUN], behind[DK_RUN];
    dk_run<KIND, FULL>(rows, w, at.n, c, x.dim, q, k[p], a);
    tot[w][c] = dk_products(a, up_to, behind);
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) k[p][t] *= behind[t];
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < DP / 64; ++p) {
    const int c = lane + 64 * p;
    double r = 1.;
    for (int o = 3; o > w; --o) r *= tot[o][c];
    const float rest = (float)r;
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) ks[w * DK_RUN + t][c] = k[p][t] * rest;
    if (w == 0 && blockIdx.z == 0) x.d[((int64_t)id * x.heads + h) * DP + c] = (float)(r * tot[0][c]);
  }
  __syncthreads();
  if (c0 >= VP) return;
  f32x4 acc[NB][2];
#pragma unroll
  for (int m = 0; m < NB; ++m) acc[m][0] = acc[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float* row = &ks[i / 4 * 16 + 4 * lg + i % 4][l16];
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const float kv = row[16 * m];
      acc[m][0] = dk_mfma(kv, v[i].x, acc[m][0]);
      acc[m][1] = dk_mfma(kv, v[i].y, acc[m][1]);
    }
  }
  float* u = x.u + ((int64_t)id * x.heads + h) * DP * VP;
#pragma unroll
  for (int m = 0; m < NB; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<float2*>(u + (16 * m + 4 * lg + i) * VP + c0 + 2 * l16) = make_float2(acc[m][0][i], acc[m][1][i]);
}

template <int DP, int KIND>
__global__ __launch_bounds__(DK_THREADS) void decay_chunk_states_kernel(const DecayChunkArgs x) {
  __shared__ __attribute__((aligned(16))) float ks[DK_CHUNK][DP + 4];
  __shared__ double tot[4][DP];
  ChunkPlace at;
  if (!at.find(x, blockIdx.x)) return;
  if (at.n == DK_CHUNK && x.dim == DP && x.vdim % 32 == 0) decay_chunk_states<DP, KIND, true>(x, at, ks, tot);
  else decay_chunk_states<DP, KIND, false>(x, at, ks, tot);
}

#define DK_AHEAD 16
template <int DP>
__global__ __launch_bounds__(DK_THREADS) void decay_chunk_carry_kernel(const DecayChunkArgs x) {
  const int e = blockIdx.x, h = blockIdx.y, VP = dk_cols(x.vdim), idx = blockIdx.z * DK_THREADS + threadIdx.x;
  const int i = idx / VP, c = idx % VP, n = x.cu[e + 1] - x.cu[e];
  if (n <= 0 || n < x.least || i >= x.dim || c >= x.vdim) return;
  float* st = x.state + (((int64_t)x.slots[e] * x.heads + h) * x.dim + i) * x.vdim + c;
  float S = x.q_start[e] == 0 ? 0.f : *st;
  const int chunks = (n + DK_CHUNK - 1) / DK_CHUNK, first = dk_first(x.cu, e);
  const int64_t step_u = (int64_t)x.heads * DP * VP, step_d = (int64_t)x.heads * DP;
  float* u = x.u + first * step_u + (int64_t)h * DP * VP + idx;
  const float* d = x.d + first * step_d + h * DP + i;
  for (int k0 = 0; k0 < chunks; k0 += DK_AHEAD) {
    float us[DK_AHEAD], ds[DK_AHEAD];
#pragma unroll
    for (int k = 0; k < DK_AHEAD; ++k) {
      const int at = min(k0 + k, chunks - 1);
      us[k] = u[at * step_u];
      ds[k] = d[at * step_d];
    }
#pragma unroll
    for (int k = 0; k < DK_AHEAD; ++k)
      if (k0 + k < chunks) {
        u[(k0 + k) * step_u] = S;
        S = fmaf(ds[k], S, us[k]);
      }
  }
  *st = S;
}

template <int DP, int KIND, bool FULL>
__device__ __forceinline__ void decay_chunk_out(const DecayChunkArgs& x, const ChunkPlace& at, float* lds) {
  constexpr int PITCH = DP + 4, NB = DP / 16;
  float (*qs)[PITCH] = reinterpret_cast<float (*)[PITCH]>(lds);
  float (*ks)[PITCH] = qs + DK_CHUNK;
  float (*as)[PITCH] = ks + DK_CHUNK;                      // the decays, then M
  float (*tot)[DP] = reinterpret_cast<float (*)[DP]>(as + DK_CHUNK);
  const int id = blockIdx.x, h = blockIdx.y;
  typename ChunkRows<KIND>::Rows rows;
  dk_rows(rows, x, at.first, at.pos, h);
  const int tid = threadIdx.x, lane = tid % WAVE, w = __builtin_amdgcn_readfirstlane(tid / WAVE), l16 = lane & 15, lg = lane >> 4;
  const int VP = dk_cols(x.vdim);
  const float* before = x.u + ((int64_t)id * x.heads + h) * DP * VP;
  const int c0 = blockIdx.z * 128 + 32 * w;
  auto stage = [&](int p) {
    const int c = lane + 64 * p;
    float q[DK_RUN], k[DK_RUN], a[DK_RUN];
    dk_run<KIND, FULL>(rows, w, at.n, c, x.dim, q, k, a);
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) {
      const int r = w * DK_RUN + t;
      qs[r][c] = q[t];
      ks[r][c] = k[t];
      as[r][c] = a[t];
    }
  };
#pragma unroll
  for (int p = 0; p < DP / 64; ++p) stage(p);
  float2 v[16], s[DP / 4];
  if (c0 < VP) {
    dk_values<KIND, FULL>(rows, at.n, c0, x.vdim, l16, lg, v);
    const uint32_t from = 4 * lg * VP + c0 + 2 * l16;
#pragma unroll
    for (int i = 0; i < DP / 4; ++i) s[i] = *reinterpret_cast<const float2*>(before + (i / 4 * 16 + i % 4) * VP + from);
  }
  __syncthreads();
  // within the run: lane (s, lg) follows k_s along the run, channels 16 j + 4 lg .. + 3
  float m[DK_RUN];
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t) m[t] = 0.f;
#pragma unroll 1
  for (int j = 0; j < NB; ++j) {
    const f32x4 k4 = *reinterpret_cast<const f32x4*>(&ks[w * DK_RUN + l16][16 * j + 4 * lg]);
    f32x4 d = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) {
      const f32x4 a4 = *reinterpret_cast<const f32x4*>(&as[w * DK_RUN + t][16 * j + 4 * lg]);
      const f32x4 q4 = *reinterpret_cast<const f32x4*>(&qs[w * DK_RUN + t][16 * j + 4 * lg]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = t == l16 ? k4[i] : d[i] * a4[i];
        m[t] = fmaf(q4[i], d[i], m[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t) {
    m[t] = add_across_16(m[t]);
    m[t] = add_across_32(m[t]);
  }
  __syncthreads();
  // q times what decayed since the run began, k times what decays to its end
#pragma unroll
  for (int p = 0; p < DP / 64; ++p) {
    const int c = lane + 64 * p;
    float a[DK_RUN], up_to[DK_RUN], behind[DK_RUN];
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) a[t] = as[w * DK_RUN + t][c];
    tot[w][c] = (float)dk_products(a, up_to, behind);
#pragma unroll
    for (int t = 0; t < DK_RUN; ++t) {
      qs[w * DK_RUN + t][c] *= up_to[t];
      ks[w * DK_RUN + t][c] *= behind[t];
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < DK_RUN; ++t)
    if (t / 4 == lg) as[w * DK_RUN + t][w * DK_RUN + l16] = m[t];
  // between runs ri > rj: six blocks of 16 x 16 over four wavefronts
  for (int b = w; b < 6; b += 4) {
    const int ri = b == 0 ? 1 : b < 3 ? 2 : 3, rj = b == 0 ? 0 : b < 3 ? b - 1 : b - 3;
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int c = 16 * j + 4 * lg;
      const f32x4 q4 = *reinterpret_cast<const f32x4*>(&qs[ri * DK_RUN + l16][c]);
      f32x4 k4 = *reinterpret_cast<const f32x4*>(&ks[rj * DK_RUN + l16][c]);
      for (int o = rj + 1; o < ri; ++o) k4 *= *reinterpret_cast<const f32x4*>(&tot[o][c]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j % 2] = dk_mfma(q4[i], k4[i], acc[j % 2]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) as[ri * DK_RUN + 4 * lg + i][rj * DK_RUN + l16] = acc[0][i] + acc[1][i];
  }
  __syncthreads();
  if (c0 >= VP) return;
  const int c = c0 + 2 * l16;
  // a run's 16 rows at a time, their sums in four chains (even and odd blocks of the state, of the tokens): chains of 32 terms lose less than one of 128
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    f32x4 acc[4][2];
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[y][0] = acc[y][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      f32x4 q4 = *reinterpret_cast<const f32x4*>(&qs[r * DK_RUN + l16][16 * j + 4 * lg]);
#pragma unroll
      for (int o = 0; o < r; ++o) q4 *= *reinterpret_cast<const f32x4*>(&tot[o][16 * j + 4 * lg]);       // what decayed before the run
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[j % 2][0] = dk_mfma(q4[i], s[4 * j + i].x, acc[j % 2][0]);
        acc[j % 2][1] = dk_mfma(q4[i], s[4 * j + i].y, acc[j % 2][1]);
      }
    }
#pragma unroll
    for (int o = 0; o <= r; ++o) {
      const f32x4 m4 = *reinterpret_cast<const f32x4*>(&as[r * DK_RUN + l16][o * DK_RUN + 4 * lg]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 + o % 2][0] = dk_mfma(m4[i], v[4 * o + i].x, acc[2 + o % 2][0]);
        acc[2 + o % 2][1] = dk_mfma(m4[i], v[4 * o + i].y, acc[2 + o % 2][1]);
      }
    }
    const f32x4 first = (acc[0][0] + acc[1][0]) + (acc[2][0] + acc[3][0]), second = (acc[0][1] + acc[1][1]) + (acc[2][1] + acc[3][1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = r * DK_RUN + 4 * lg + i;
      float* o = x.out + ((int64_t)(at.first + t) * x.heads + h) * x.vdim + c;
      if (!FULL && (t >= at.n || c >= x.vdim)) continue;
      if (FULL || x.vdim % 2 == 0) {
        *reinterpret_cast<float2*>(o) = make_float2(first[i], second[i]);
      } else {
        o[0] = first[i];
        if (c + 1 < x.vdim) o[1] = second[i];
      }
    }
  }
}

template <int DP, int KIND>
__global__ __launch_bounds__(DK_THREADS, DP == 64 ? 2 : 1) void decay_chunk_out_kernel(const DecayChunkArgs x) {
  extern __shared__ __attribute__((aligned(16))) float dk_lds[];
  ChunkPlace at;
  if (!at.find(x, blockIdx.x)) return;
  if (at.n == DK_CHUNK && x.dim == DP && x.vdim % 32 == 0) decay_chunk_out<DP, KIND, true>(x, at, dk_lds);
  else decay_chunk_out<DP, KIND, false>(x, at, dk_lds);
}

static int64_t dk_ids(int tokens, int entries) { return (int64_t)(tokens / DK_CHUNK) + entries; }
static int dk_channels(int dim) { return dim <= 64 ? 64 : 128; }

extern "C" int64_t ga_decay_chunk_floats(int tokens, int entries, int heads, int dim, int vdim) {
  return dk_ids(tokens, entries) * heads * dk_channels(dim) * (dk_cols(vdim) + 1);
}

template <int DP, int KIND>
static int dk_launch(const DecayChunkArgs& x, int tokens, hipStream_t stream) {
  constexpr int lds = (3 * DK_CHUNK * (DP + 4) + 4 * DP) * (int)sizeof(float);
  const int64_t ids = dk_ids(tokens, x.entries);
  const auto out = decay_chunk_out_kernel<DP, KIND>;
  if (const int raised = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(out), hipFuncAttributeMaxDynamicSharedMemorySize, lds))
    return raised;
  const unsigned columns = (x.vdim + 127) / 128;
  hipLaunchKernelGGL((decay_chunk_states_kernel<DP, KIND>), dim3((unsigned)ids, x.heads, columns), dim3(DK_THREADS), 0, stream, x);
  hipLaunchKernelGGL(decay_chunk_carry_kernel<DP>, dim3(x.entries, x.heads, (x.dim * dk_cols(x.vdim) + DK_THREADS - 1) / DK_THREADS),
                     dim3(DK_THREADS), 0, stream, x);
  hipLaunchKernelGGL(out, dim3((unsigned)ids, x.heads, columns), dim3(DK_THREADS), lds, stream, x);
  return GA_CHECK_LAUNCH();
}
static int dk_check(const DecayChunkArgs& x, int tokens) {
  if (x.heads <= 0 || x.heads > 65535 || x.dim <= 0 || x.dim > 128 || x.vdim <= 0 || x.vdim > 65536) return -1;
  if (x.stride >= (1ll << 27) || dk_ids(tokens, x.entries) >= (1ll << 31)) return -2;       // (a run's offsets are 32-bit)
  if (((uintptr_t)x.u | (uintptr_t)x.out) & 7) return -5;
  return 0;
}

extern "C" int ga_decay_chunk(void* out, void* work, const void* q, const void* k, const void* v, int64_t stride, const void* decay,
                              const void* head_decay, const void* cos_t, const void* sin_t, int rot_dims, float q_scale, float k_scale,
                              void* state, const void* slots, const void* cu, const void* q_start, int tokens, int entries, int heads,
                              int dim, int vdim, int silu_inputs, int least, hipStream_t stream) {
  if (entries <= 0 || tokens <= 0) return 0;
  if ((decay == nullptr) == (head_decay == nullptr)) return -3;
  if (rot_dims < 0 || rot_dims % 2 || rot_dims > dim || (rot_dims > 0 && (!cos_t || !sin_t))) return -4;
  float* u = (float*)work;
  const DecayChunkArgs x = {(float*)out, u, u + dk_ids(tokens, entries) * heads * dk_channels(dim) * dk_cols(vdim), (const float*)q, (const float*)k,
                            (const float*)v, stride, (const float*)decay, (const float*)head_decay, (const float*)cos_t, (const float*)sin_t, rot_dims,
                            q_scale, k_scale, nullptr, nullptr, (float*)state, (const int64_t*)slots, (const int32_t*)cu,
                            (const int32_t*)q_start, entries, heads, dim, vdim, least};
  if (const int rc = dk_check(x, tokens)) return rc;
  if (silu_inputs && rot_dims > 0) return -6;
#define GO(KIND) (dim <= 64 ? dk_launch<64, KIND>(x, tokens, stream) : dk_launch<128, KIND>(x, tokens, stream))
  return silu_inputs ? GO(DK_SILU) : rot_dims > 0 ? GO(DK_ROT) : GO(DK_PLAIN);
#undef GO
}

extern "C" int ga_hgrn2_chunk(void* out, void* work, const void* proj, int64_t stride, const void* f_bias, const void* lower, void* state,
                              const void* slots, const void* cu, const void* q_start, int tokens, int entries, int heads, int dim,
                              int vdim, int least, hipStream_t stream) {
  if (entries <= 0 || tokens <= 0) return 0;
  float* u = (float*)work;
  const float* p = (const float*)proj;
  const DecayChunkArgs x = {(float*)out, u, u + dk_ids(tokens, entries) * heads * dk_channels(dim) * dk_cols(vdim), p, nullptr,
                            p + 2 * (int64_t)heads * dim, stride, nullptr, nullptr, nullptr, nullptr, 0, 1.f, 1.f, (const float*)f_bias, (const float*)lower,
                            (float*)state, (const int64_t*)slots, (const int32_t*)cu, (const int32_t*)q_start, entries, heads, dim, vdim, least};
  if (const int rc = dk_check(x, tokens)) return rc;
  return dim <= 64 ? dk_launch<64, DK_FORGET>(x, tokens, stream) : dk_launch<128, DK_FORGET>(x, tokens, stream);
}
