// What the recurrences with a decaying outer-product state read, element by element: decay_walk.h's and decay_chunk.hip's sources.
// load(Raw, start, token, channel) asks for an element of q, k and a, finish(Raw, Fixed, channel, q, k, a) makes them of it; load_v and
// finish_v the same for v.
#pragma once
#include "common.h"
#include <type_traits>

// q, k and v as the recurrence reads them: the projection's numbers or their silu, turned by position, scaled
template <bool ROT>
struct DecayRows {
  static constexpr bool K_OF_A = false;
  struct Fixed {};
  __device__ __forceinline__ Fixed fixed(int) const { return {}; }
  struct Plain { float q, k, a; };
  struct Turned { float q, k, a, q2, k2, c, s; };
  typedef typename std::conditional<ROT, Turned, Plain>::type Raw;
  const float *q, *k, *v;              // the entry's first token, the head's first channel or column
  const float* decay;                  // the same of [tokens, heads * dim]; or one number, and both steps are 0
  const float *cos_t, *sin_t;          // the first token's position
  int64_t stride;
  int decay_token, decay_channel, half;
  float q_scale, k_scale;
  bool acts;                           // whether finish and finish_v apply the silu: asked once a tile, not per element
  template <bool ACT>
  __device__ __forceinline__ float act(float z) const { return ACT ? z / (1.0f + expf(-z)) : z; }
  __device__ __forceinline__ void load(Raw& x, int start, int t, int i) const {
    const float *qp = q + start * stride, *kp = k + start * stride;
    const uint32_t row = (uint32_t)t * (uint32_t)stride;
    x.q = qp[row + i];
    x.k = kp[row + i];
    x.a = (decay + (int64_t)start * decay_token)[(uint32_t)(t * decay_token + i * decay_channel)];
    if constexpr (ROT) {               // (a channel that is not turned reads what channel 0 reads, and drops it)
      const int at = i < 2 * half ? i : 0, f = at < half ? at : at - half, other = at < half ? at + half : at - half;
      x.c = (cos_t + (int64_t)start * half)[(uint32_t)(t * half + f)];
      x.s = (sin_t + (int64_t)start * half)[(uint32_t)(t * half + f)];
      x.q2 = qp[row + other];
      x.k2 = kp[row + other];
    }
  }
  template <bool ACT>
  __device__ __forceinline__ void finish(const Raw& x, const Fixed&, int i, float& qv, float& kv, float& a) const {
    qv = act<ACT>(x.q);
    kv = act<ACT>(x.k);
    if constexpr (ROT) {
      if (i < 2 * half) {              // the pair (lo, hi) becomes (lo c - hi s, hi c + lo s)
        const float qo = act<ACT>(x.q2), ko = act<ACT>(x.k2);
        qv = i < half ? qv * x.c - qo * x.s : qv * x.c + qo * x.s;
        kv = i < half ? kv * x.c - ko * x.s : kv * x.c + ko * x.s;
      }
    }
    qv *= q_scale;
    kv *= k_scale;
    a = x.a;
  }
  __device__ __forceinline__ float load_v(int start, int t, int c) const {
    return (v + start * stride)[(uint32_t)t * (uint32_t)stride + c];
  }
  template <bool ACT>
  __device__ __forceinline__ float finish_v(float x) const { return act<ACT>(x); }
};

// q = silu(pq), f = lower + (1 - lower) * sigmoid(pf + bias), k = 1 - f (HGRN2)
__device__ __forceinline__ float gr_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

struct ForgetRows {
  struct Raw { float q, f; };
  struct Fixed { float bias, lower; };
  const float *proj, *v;               // the entry's first token, the head's first channel or column
  const float *bias, *lower;           // the head's
  int64_t stride;
  int hd;
  static constexpr bool acts = false, K_OF_A = true;
  __device__ __forceinline__ Fixed fixed(int i) const { return {bias[i], lower[i]}; }
  __device__ __forceinline__ void load(Raw& x, int start, int t, int i) const {
    const float* p = proj + start * stride;
    const uint32_t at = (uint32_t)t * (uint32_t)stride + i;
    x.q = p[at];
    x.f = p[at + hd];
  }
  template <bool>
  __device__ __forceinline__ void finish(const Raw& x, const Fixed& c, int i, float& q, float& k, float& f) const {
    q = x.q * gr_sigmoid(x.q);
    f = c.lower + (1.0f - c.lower) * gr_sigmoid(x.f + c.bias);
    k = 1.0f - f;
  }
  __device__ __forceinline__ float load_v(int start, int t, int c) const {
    return (v + start * stride)[(uint32_t)t * (uint32_t)stride + c];
  }
  template <bool>
  __device__ __forceinline__ float finish_v(float x) const { return x; }
};
