// Matrix products C[M, N] = A[M, K] . W[N, K]^T (+ bias[N]) with W stored [out, in] row-major, the
// layout of the checkpoint (ginfer/core/layer/linear.cc:9-20); 32-bit accumulation and the bias
// added in 32-bit before the one rounding (ginfer/core/op/kernels/cuda/gemm_kernel/
// gemm_kernel.cu:100-121, ginfer/core/op/kernels/cuda/gemv_kernel.cu:52-55).
//
// Three kernels make the true 32-bit product (no reduced-precision mode anywhere).  In all of them every element of
// C is ONE accumulator that takes its terms over ascending k as fused multiply-adds, so its bits do not depend on M,
// on the tile it falls in, on the rest of the batch, or on which of the three ran:
//   gemm_nt_few_rows_kernel  up to 64 rows (a decode step, a small portion): the matrix cores' 32-bit instruction, a
//                            wavefront per 16 columns and up to four blocks of 16 rows, operands straight from memory;
//   gemm_nt_matrix_kernel    more rows: the matrix cores again, over tiles of 32 x 32 to 64 x 96 through LDS;
//   gemm_nt_kernel           plain FMA, a tile of 64 x 64 per workgroup staged through LDS in steps of K: 33 to 64 rows
//                            times 65,536 columns and more (a head), where it is the fastest of the three.
// They are templated on storage, so that they also serve bfloat16 operands (the kernel tests' oracle and the
// fallback for shapes the bfloat16 kernels refuse).
//
// A step of K is asked for (in 16-byte loads, in the first and the third kernel where rows allow it, consecutive lanes on
// consecutive elements) while the step before is being multiplied.
#include "common.h"
#include "ginfer_amd.h"   // the entry points below are checked against their declarations

#define GEMM_THREADS 256
#ifndef GEMM_MATRIX_FROM_ROWS
#define GEMM_MATRIX_FROM_ROWS 64    // more rows than this: the kernel on the matrix cores (the same bits)
#endif

// four consecutive elements as floats; `wide`: one load (the address is a multiple of four elements)
template <typename T>
__device__ __forceinline__ void load4(float (&v)[4], const T* p, int valid, bool wide);
template <>
__device__ __forceinline__ void load4<float>(float (&v)[4], const float* p, int valid, bool wide) {
  if (wide && valid == 4) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i < valid ? p[i] : 0.f;
  }
}
template <>
__device__ __forceinline__ void load4<bf16_t>(float (&v)[4], const bf16_t* p, int valid, bool wide) {
  if (wide && valid == 4) {
    const uint2 x = *reinterpret_cast<const uint2*>(p);
    v[0] = bf16_to_f32((bf16_t)(x.x & 0xffffu)); v[1] = bf16_to_f32((bf16_t)(x.x >> 16));
    v[2] = bf16_to_f32((bf16_t)(x.y & 0xffffu)); v[3] = bf16_to_f32((bf16_t)(x.y >> 16));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = i < valid ? bf16_to_f32(p[i]) : 0.f;
  }
}

// four consecutive elements at any address that an element may have, in one load all the same: the device takes vector loads
// at such addresses, and a type that promises no more says so
typedef float any_float4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint16_t any_half4 __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ void load4_anywhere(float (&v)[4], const float* p) {
  const any_float4 x = *reinterpret_cast<const any_float4*>(p);
  v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
}
__device__ __forceinline__ void load4_anywhere(float (&v)[4], const bf16_t* p) {
  const any_half4 x = *reinterpret_cast<const any_half4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = bf16_to_f32(x[i]);
}

// TM x TN: the workgroup's tile of C; TK: elements of K per step; a thread owns RM x RN elements, the threads
// lie 16 x 16 over the tile (TM = 16 RM, TN = 16 RN).
template <typename TA, typename TW, typename TC, int TM, int TN, int TK>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_nt_kernel(TC* __restrict__ C, int64_t ldc,
                                                               const TA* __restrict__ A, int64_t lda,
                                                               const TW* __restrict__ W,
                                                               const TW* __restrict__ bias, int M, int N,
                                                               int K, int wide_a, int wide_w) {
  constexpr int RM = TM / 16, RN = TN / 16;
  constexpr int GA = TM * TK / 4 / GEMM_THREADS, GW = TN * TK / 4 / GEMM_THREADS;     // groups of four per thread
  static_assert(GA >= 1 && GW >= 1 && TM % 16 == 0 && TN % 16 == 0, "tile sizes");
  __shared__ float a_s[TK][TM + 4];
  __shared__ float w_s[TK][TN + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int tx = tid % 16, ty = tid / 16;  // the thread's block: rows ty*RM.., columns tx*RN..
  float acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = 0.f;

  float ra[GA][4], rw[GW][4];
  // group number gi of a step: row gi / (TK / 4) of the tile, elements 4 (gi % (TK / 4)) .. + 3 of the step
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < GA; ++i) {
      const int gi = tid + i * GEMM_THREADS, row = gi / (TK / 4), k = k0 + (gi % (TK / 4)) * 4;
      const int m = m0 + row;
      const int valid = (m < M && k < K) ? (K - k < 4 ? K - k : 4) : 0;
      if (valid) load4<TA>(ra[i], A + (int64_t)m * lda + k, valid, wide_a != 0);
      else ra[i][0] = ra[i][1] = ra[i][2] = ra[i][3] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < GW; ++i) {
      const int gi = tid + i * GEMM_THREADS, row = gi / (TK / 4), k = k0 + (gi % (TK / 4)) * 4;
      const int n = n0 + row;
      const int valid = (n < N && k < K) ? (K - k < 4 ? K - k : 4) : 0;
      if (valid) load4<TW>(rw[i], W + (int64_t)n * K + k, valid, wide_w != 0);
      else rw[i][0] = rw[i][1] = rw[i][2] = rw[i][3] = 0.f;
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
    for (int i = 0; i < GA; ++i) {
      const int gi = tid + i * GEMM_THREADS, row = gi / (TK / 4), kk = (gi % (TK / 4)) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) a_s[kk + j][row] = ra[i][j];
    }
#pragma unroll
    for (int i = 0; i < GW; ++i) {
      const int gi = tid + i * GEMM_THREADS, row = gi / (TK / 4), kk = (gi % (TK / 4)) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) w_s[kk + j][row] = rw[i][j];
    }
    __syncthreads();
    if (k0 + TK < K) fetch(k0 + TK);        // on its way while this step is multiplied
#pragma unroll 8
    for (int k = 0; k < TK; ++k) {
      float a[RM], w[RN];
#pragma unroll
      for (int i = 0; i < RM; ++i) a[i] = a_s[k][ty * RM + i];
#pragma unroll
      for (int j = 0; j < RN; ++j) w[j] = w_s[k][tx * RN + j];
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = __builtin_fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int m = m0 + ty * RM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      const int n = n0 + tx * RN + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (bias) v += Num<TW>::ld(bias + n);
      Num<TC>::st(C + (int64_t)m * ldc + n, v);
    }
  }
}

// The same product on the matrix cores, for many rows.  v_mfma_f32_16x16x4_f32 takes, from lane l, row l % 16 of A and of
// W at k = step + l / 16 and adds its four products into the accumulator in ascending k as fused multiply-adds: measured
// on the device, its results over a K of 512 equal the chain of fmaf over ascending k bit for bit, for every element of
// the tile.  So this kernel gives the bits of the kernel above.  Register r of lane l receives row 4 (l / 16) + r, column
// l % 16 of a block.
//
// A workgroup of four wavefronts, 2 x 2 over a tile of 32 BM x 32 BN; a wavefront owns BM x BN blocks of 16 x 16.  K must
// not be split (one accumulator per element), so a block of 16 x 16 is a chain of K / 4 instructions of 32 cycles however
// the chip is filled (30 us for a K of 8,960): small blocks, so that a few hundred rows make enough chains for all 1,024
// SIMDs, and a chain that never waits.  DEPTH steps of TK elements are on their way from memory in registers while a step
// is multiplied out of one of two buffers in LDS, one barrier a step; nothing in the loop is conditional (loads past the
// end repeat the last step's), so that the compiler waits for just the step it stages.  A row of LDS holds every 16
// elements of K with the four of a lane side by side (k = g, 4 + g, 8 + g, 12 + g): the operands of four instructions
// come in one 16-byte read and need no exchange between lanes (with the row swaps of gfx950 after the read the chain of
// a K of 8,960 took 91 us instead of 62), and with rows padded by four words neither side has bank conflicts.
// Workgroups that share rows of W are neighbours on one XCD, whose L2 then reads W once: columns of tiles go to the XCDs in
// turn, and the tiles of the columns that are left over to all eight alike (as whole columns they made a second round on the
// XCDs that got one more: 300 rows by 4,864, 51 columns of tiles, K 1,536, 84 us, now 54.5; 1,536 by 640 60 and 39.7; 2,048 by
// 32, one column, 21.5 and 14.5).  Rows that are not aligned take the same loads (4,096 rows by 5,000 of a K of 521, us: 264 in the
// tiles before, 330 element by element here, now 206; 256 by 1,536 of 1,537: 90, 49, 24).
// Measured on MI355X, us, before (32 x 32 x 2 blocks in tiles of 64 x 64 to 128 x 128, two barriers a step) -> now, for
// [rows] x 1,536 of a K of 8,960, x 2,048 of 1,536, and x 17,920 of 1,536: 65 rows 335 -> 59, 55 -> 12.4, 157 -> 56;
// 256 rows 232 -> 93, 45 -> 19.6, 224 -> 116; 512 rows 232 -> 136, 47.5 -> 36, 327 -> 229; 2,048 rows 634 -> 433,
// 136 -> 105, 905 -> 868 (130 of the 154 TFLOP/s that a large product reaches on this card).
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <typename TA, typename TW, typename TC, int BM, int BN, int TK, int DEPTH>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_nt_matrix_kernel(TC* __restrict__ C, int64_t ldc,
                                                                     const TA* __restrict__ A, int64_t lda,
                                                                     const TW* __restrict__ W,
                                                                     const TW* __restrict__ bias, int M, int N, int K,
                                                                     int m_tiles, int n_tiles) {
  constexpr int TM = 32 * BM, TN = 32 * BN, PAD = TK + 4;
  constexpr int GA = TM * TK / 4 / GEMM_THREADS, GW = TN * TK / 4 / GEMM_THREADS;
  static_assert(GA >= 1 && GW >= 1 && TK % 16 == 0 && DEPTH % 2 == 0, "tile sizes");
  __shared__ float a_s[2][TM][PAD];
  __shared__ float w_s[2][TN][PAD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, kq = lane >> 4;
  const int at = blockIdx.x >> 3, xcd = blockIdx.x & 7, whole = n_tiles / 8 * m_tiles;
  int mt = at % m_tiles, nt = at / m_tiles * 8 + xcd;
  if (at >= whole) {
    const int rest = n_tiles % 8 * m_tiles, run = (rest + 7) / 8, id = xcd * run + at - whole;
    if (at - whole >= run || id >= rest) return;
    mt = id % m_tiles;
    nt = n_tiles / 8 * 8 + id / m_tiles;
  }
  const int m0 = mt * TM, n0 = nt * TN;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
  f32x4 acc[BM][BN];
#pragma unroll
  for (int i = 0; i < BM; ++i)
#pragma unroll
    for (int j = 0; j < BN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ra[DEPTH][GA][4], rw[DEPTH][GW][4];
  // rows beyond the matrix are read as row 0's and dropped at the end: no branch in the loop
  const TA* pa[GA];
  const TW* pw[GW];
#pragma unroll
  for (int i = 0; i < GA; ++i) {
    const int gi = tid + i * GEMM_THREADS, m = m0 + gi / (TK / 4);
    pa[i] = A + (int64_t)(m < M ? m : 0) * lda + (gi % (TK / 4)) * 4;
  }
#pragma unroll
  for (int i = 0; i < GW; ++i) {
    const int gi = tid + i * GEMM_THREADS, n = n0 + gi / (TK / 4);
    pw[i] = W + (int64_t)(n < N ? n : 0) * K + (gi % (TK / 4)) * 4;
  }
  auto fetch = [&](float (&xa)[GA][4], float (&xw)[GW][4], int k0) {
#pragma unroll
    for (int i = 0; i < GA; ++i) load4_anywhere(xa[i], pa[i] + k0);
#pragma unroll
    for (int i = 0; i < GW; ++i) load4_anywhere(xw[i], pw[i] + k0);
  };
  auto fetch_carefully = [&](float (&xa)[GA][4], float (&xw)[GW][4], int k0) {
    const int k = k0 + (tid % (TK / 4)) * 4, valid = k < K ? (K - k < 4 ? K - k : 4) : 0;
#pragma unroll
    for (int i = 0; i < GA; ++i) load4<TA>(xa[i], pa[i] + k0, valid, false);
#pragma unroll
    for (int i = 0; i < GW; ++i) load4<TW>(xw[i], pw[i] + k0, valid, false);
  };
  auto stage = [&](int b, float (&xa)[GA][4], float (&xw)[GW][4]) {
#pragma unroll
    for (int i = 0; i < GA; ++i) {
      const int gi = tid + i * GEMM_THREADS;
      float* to = &a_s[b][gi / (TK / 4)][(gi % (TK / 4)) / 4 * 16 + gi % 4];
#pragma unroll
      for (int g = 0; g < 4; ++g) to[4 * g] = xa[i][g];
    }
#pragma unroll
    for (int i = 0; i < GW; ++i) {
      const int gi = tid + i * GEMM_THREADS;
      float* to = &w_s[b][gi / (TK / 4)][(gi % (TK / 4)) / 4 * 16 + gi % 4];
#pragma unroll
      for (int g = 0; g < 4; ++g) to[4 * g] = xw[i][g];
    }
  };
  auto read = [&](int b, int kk, float (&x)[BM][4], float (&y)[BN][4]) {
#pragma unroll
    for (int i = 0; i < BM; ++i) {
      const float4 v = *reinterpret_cast<const float4*>(&a_s[b][wm + i * 16 + i16][kk + 4 * kq]);
      x[i][0] = v.x; x[i][1] = v.y; x[i][2] = v.z; x[i][3] = v.w;
    }
#pragma unroll
    for (int j = 0; j < BN; ++j) {
      const float4 v = *reinterpret_cast<const float4*>(&w_s[b][wn + j * 16 + i16][kk + 4 * kq]);
      y[j][0] = v.x; y[j][1] = v.y; y[j][2] = v.z; y[j][3] = v.w;
    }
  };
  // all operands of a step are asked for before the first is multiplied
  auto multiply = [&](int b) {
    float x[TK / 16][BM][4], y[TK / 16][BN][4];
#pragma unroll
    for (int c = 0; c < TK / 16; ++c) read(b, c * 16, x[c], y[c]);
#pragma unroll
    for (int c = 0; c < TK / 16; ++c) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < BM; ++i)
#pragma unroll
          for (int j = 0; j < BN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[c][i][st], y[c][j][st], acc[i][j], 0, 0, 0);
    }
  };
  const int steps = K / TK, last = (steps - 1) * TK;
  if (steps > 0) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(ra[d], rw[d], d * TK < last ? d * TK : last);
    stage(0, ra[0], rw[0]);
    const int k1 = DEPTH * TK < last ? DEPTH * TK : last;
    fetch(ra[0], rw[0], k1);
    __syncthreads();
    int s0 = 0;
    for (; s0 + DEPTH <= steps; s0 += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        multiply(d & 1);
        stage((d & 1) ^ 1, ra[(d + 1) % DEPTH], rw[(d + 1) % DEPTH]);
        const int k = (s0 + d + 1 + DEPTH) * TK;
        fetch(ra[(d + 1) % DEPTH], rw[(d + 1) % DEPTH], k < last ? k : last);
        __syncthreads();
      }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (s0 + d < steps) {
        multiply(d & 1);
        stage((d & 1) ^ 1, ra[(d + 1) % DEPTH], rw[(d + 1) % DEPTH]);
        __syncthreads();
      }
    }
  }
  for (int k0 = steps * TK; k0 < K; k0 += TK) {
    fetch_carefully(ra[0], rw[0], k0);
    stage(0, ra[0], rw[0]);
    __syncthreads();
    multiply(0);
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < BN; ++j) {
    const int n = n0 + wn + j * 16 + i16;
    if (n >= N) continue;
    const float bv = bias ? Num<TW>::ld(bias + n) : 0.f;
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + i * 16 + 4 * kq + r;
        if (m >= M) continue;
        float v = acc[i][j][r];
        if (bias) v += bv;
        Num<TC>::st(C + (int64_t)m * ldc + n, v);
      }
  }
}

// Up to 16 rows (a decode step): one wavefront per 16 columns, no LDS.  v_mfma_f32_16x16x4_f32 takes, from lane l, row
// l % 16 of A and of W at k = step + l / 16, and adds its four products into the accumulator in ascending k as fused
// multiply-adds (the same measurement as above): the bits of the other two kernels again.  A lane loads four
// consecutive elements of its row (16 bytes; the four lanes of a row 64 consecutive bytes), which is the operand of
// four steps once the four lanes of the row have exchanged elements (a 4 x 4 transpose in two rounds of swaps between
// lanes 16 and 32 apart).  Of FEW_SETS sets of FEW_DEPTH such loads of A and of W one is multiplied while the others
// are under way.
// Register r of lane l receives row 4 (l / 16) + r, column l % 16.
#define FEW_DEPTH 8
#define FEW_SETS 2
#define FEW_DEPTH_BLOCKS 4     // ... with several blocks of rows (measured: 2, 4, 8)

// x[c] of the lane 16 s + i (s = 0..3) becomes what was x[s] of the lane 16 c + i: a 4 x 4 transpose between the
// registers and the wavefront's four rows of 16 lanes, by gfx950's row swaps (v_permlane16_swap exchanges the odd rows
// of its first operand with the even rows of its second, v_permlane32_swap the upper half of the first with the lower
// half of the second): the 2 x 2 blocks transposed in themselves, then the two off the diagonal exchanged
__device__ __forceinline__ void swap_rows_16(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap_rows_32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void transpose_over_lane_rows(float (&x)[4]) {
  swap_rows_16(x[0], x[1]);
  swap_rows_16(x[2], x[3]);
  swap_rows_32(x[0], x[2]);
  swap_rows_32(x[1], x[3]);
}

// four consecutive elements at an address that is a multiple of four elements, no questions asked
template <typename T>
__device__ __forceinline__ void load4_aligned(float (&v)[4], const T* p) {
  load4<T>(v, p, 4, true);
}

template <typename TA, typename TW, typename TC, int RB>
__global__ __launch_bounds__(64) void gemm_nt_few_rows_kernel(TC* __restrict__ C, int64_t ldc,
                                                              const TA* __restrict__ A, int64_t lda,
                                                              const TW* __restrict__ W,
                                                              const TW* __restrict__ bias, int M, int N, int K,
                                                              int wide_a, int wide_w) {
  // RB blocks of 16 rows: the wavefront's 16 columns of W are loaded once for all of them, and the blocks' chains of
  // matrix instructions run side by side
  const int lane = threadIdx.x, i = lane & 15, kq = lane >> 4;
  const int n = blockIdx.x * 16 + i;
  const bool w_ok = n < N;
  // a lane whose row does not exist reads row 0 and drops what it read: no branch in the loop
  const TA* pa[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) pa[rb] = A + (int64_t)(16 * rb + i < M ? 16 * rb + i : 0) * lda + 4 * kq;
  const TW* pw = W + (int64_t)(w_ok ? n : 0) * K + 4 * kq;
  f32x4 acc[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // FEW_SETS sets of DEPTH loads of A's blocks and of W: one is multiplied while the others are on their way (a
  // wavefront has the registers of its SIMD to itself: so few wavefronts run here that the bytes each keeps under way
  // are what decides)
  constexpr int DEPTH = RB == 1 ? FEW_DEPTH : FEW_DEPTH_BLOCKS;
  float a[FEW_SETS][DEPTH][RB][4], w[FEW_SETS][DEPTH][4];
  // whole chunks of 16 elements, with aligned rows, take the loop without branches; what is left of K (and everything,
  // with rows that are not aligned) takes the careful loads afterwards: ascending k all the same
  const int chunks = (wide_a && wide_w) ? K / 16 : 0;
  // (a lane without a row of its own multiplies row 0's numbers: they meet nobody else's, a row of A and a row of W
  // make one element of C, and that element is not stored)
  auto multiply = [&](float (&x)[RB][4], float (&y)[4]) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) transpose_over_lane_rows(x[rb]);
    transpose_over_lane_rows(y);
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) acc[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[rb][st], y[st], acc[rb], 0, 0, 0);
  };
  // the loads of the chunks first .. first + DEPTH - 1 (those of them that exist; `all`: they all do)
  auto fetch = [&](float (&x)[DEPTH][RB][4], float (&y)[DEPTH][4], int first, bool all) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (all || first + d < chunks) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) load4_aligned<TA>(x[d][rb], pa[rb] + (first + d) * 16);
        load4_aligned<TW>(y[d], pw + (first + d) * 16);
      }
  };
  auto multiply_set = [&](float (&x)[DEPTH][RB][4], float (&y)[DEPTH][4], int first, bool all) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (all || first + d < chunks) multiply(x[d], y[d]);
  };
#pragma unroll
  for (int st = 0; st < FEW_SETS - 1; ++st) fetch(a[st], w[st], st * DEPTH, false);
  int c0 = 0;
  // while every set of a round and the sets asked for in it lie inside K nothing in the loop is conditional: the
  // compiler then counts the loads and waits for just those of the set it multiplies
  for (; c0 + (2 * FEW_SETS - 1) * DEPTH <= chunks; c0 += FEW_SETS * DEPTH) {
#pragma unroll
    for (int st = 0; st < FEW_SETS; ++st) {
      fetch(a[(st + FEW_SETS - 1) % FEW_SETS], w[(st + FEW_SETS - 1) % FEW_SETS], c0 + (st + FEW_SETS - 1) * DEPTH, true);
      multiply_set(a[st], w[st], c0 + st * DEPTH, true);
    }
  }
  for (; c0 < chunks; c0 += FEW_SETS * DEPTH) {
#pragma unroll
    for (int st = 0; st < FEW_SETS; ++st) {
      fetch(a[(st + FEW_SETS - 1) % FEW_SETS], w[(st + FEW_SETS - 1) % FEW_SETS], c0 + (st + FEW_SETS - 1) * DEPTH, false);
      multiply_set(a[st], w[st], c0 + st * DEPTH, false);
    }
  }
  for (int k0 = chunks * 16; k0 < K; k0 += 16) {
    const int k = k0 + 4 * kq;
    const int valid = k < K ? (K - k < 4 ? K - k : 4) : 0;
    float x[RB][4], y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) x[rb][0] = x[rb][1] = x[rb][2] = x[rb][3] = 0.f;
    if (valid) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) load4<TA>(x[rb], pa[rb] + k0, valid, false);
      load4<TW>(y, pw + k0, valid, false);
    }
    multiply(x, y);
  }
  if (!w_ok) return;
  const float b = bias ? Num<TW>::ld(bias + n) : 0.f;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * rb + 4 * kq + r;
      if (m >= M) continue;
      float v = acc[rb][r];
      if (bias) v += b;
      Num<TC>::st(C + (int64_t)m * ldc + n, v);
    }
}

// in_bf16: A, W and bias are bfloat16 (else float); out_bf16: C is bfloat16 (else float).
extern "C" int ga_gemm_nt(void* C, int64_t ldc, const void* A, int64_t lda, const void* W,
                          const void* bias, int M, int N, int K, int in_bf16, int out_bf16,
                          hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0) return -1;
  // up to 64 rows: a wavefront per 16 columns, which it streams once for up to four blocks of 16 rows (with more than 32
  // rows and very many columns, a head over a large vocabulary, the plain kernel is faster: measured at 151,936 columns)
  const bool few = M <= GEMM_MATRIX_FROM_ROWS && !(M > 32 && N >= 65536);
  const int row_blocks = (M + 15) / 16;
  // many rows: the matrix cores, in tiles of 32 x 32, 64 x 64 or 64 x 96, whichever takes the least time by this sum.  A
  // chip of 256 compute units works off `rounds` tiles each; the first costs a tile's whole chain, further ones overlap
  // with it.  Measured in us at a K of 1,536 (alone / each further round): 13.2 / 8.5, 35.5 / 25.5, 47.5 / 39; the sums
  // are what the sizes above take at that K or up to 15 % more (512 rows by 2,048: 35.5 against 36; 65 by 17,920: 64 against 56).
  const bool matrix = M > GEMM_MATRIX_FROM_ROWS;
  const int tile_m[3] = {32, 64, 64}, tile_n[3] = {32, 64, 96};
  const float alone[3] = {13.2f, 35.5f, 47.5f}, further[3] = {8.5f, 25.5f, 39.f};
  int tiling = -1, m_tiles = 0, n_tiles = 0;
  int64_t groups = 0;
  float least = 0.f;
  for (int t = 0; matrix && t < 3; ++t) {
    const int64_t mt = (M + (int64_t)tile_m[t] - 1) / tile_m[t], nt = (N + (int64_t)tile_n[t] - 1) / tile_n[t];
    const int64_t blocks = (mt * (nt / 8) + (mt * (nt % 8) + 7) / 8) * 8;     // one dimension: see the kernel's mapping
    if (blocks > 0xffffffffll / GEMM_THREADS) continue;                       // more threads than a launch may have
    const float us = alone[t] + further[t] * (float)((mt * nt + 255) / 256 - 1);
    if (tiling < 0 || us < least) {
      least = us;
      tiling = t;
      groups = blocks;
      m_tiles = (int)mt;
      n_tiles = (int)nt;
    }
  }
  const int tm = 64, tn = few ? 16 : 64;
  dim3 grid((N + tn - 1) / tn, (M + tm - 1) / tm), block(GEMM_THREADS);
  if (matrix) {
    if ((M + 127) / 128 > 65535 || tiling < 0) return -2;
    grid = dim3((unsigned)groups);
  }
  if (grid.y > 65535) return -2;
  // 16-byte loads (8 bytes for bfloat16) need rows that start at multiples of four elements
  const size_t unit = in_bf16 ? 8 : 16;
  const int wide_a = (K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % unit == 0) ? 1 : 0;
  const int wide_w = (K % 4 == 0 && (uintptr_t)W % unit == 0) ? 1 : 0;
#define LAUNCH(TA, TW, TC)                                                                                   \
  do {                                                                                                       \
    if (few && row_blocks == 1)                                                                              \
      hipLaunchKernelGGL((gemm_nt_few_rows_kernel<TA, TW, TC, 1>), grid, dim3(64), 0, stream, (TC*)C, ldc,   \
                         (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, wide_a, wide_w);         \
    else if (few && row_blocks == 2)                                                                         \
      hipLaunchKernelGGL((gemm_nt_few_rows_kernel<TA, TW, TC, 2>), grid, dim3(64), 0, stream, (TC*)C, ldc,   \
                         (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, wide_a, wide_w);         \
    else if (few && row_blocks == 3)                                                                         \
      hipLaunchKernelGGL((gemm_nt_few_rows_kernel<TA, TW, TC, 3>), grid, dim3(64), 0, stream, (TC*)C, ldc,   \
                         (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, wide_a, wide_w);         \
    else if (few)                                                                                            \
      hipLaunchKernelGGL((gemm_nt_few_rows_kernel<TA, TW, TC, 4>), grid, dim3(64), 0, stream, (TC*)C, ldc,   \
                         (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, wide_a, wide_w);         \
    else if (matrix && tiling == 0)                                                                          \
      hipLaunchKernelGGL((gemm_nt_matrix_kernel<TA, TW, TC, 1, 1, 64, 2>), grid, block, 0, stream,           \
                         (TC*)C, ldc, (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, m_tiles,    \
                         n_tiles);                                                                           \
    else if (matrix && tiling == 1)                                                                          \
      hipLaunchKernelGGL((gemm_nt_matrix_kernel<TA, TW, TC, 2, 2, 32, 2>), grid, block, 0, stream,           \
                         (TC*)C, ldc, (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, m_tiles,    \
                         n_tiles);                                                                           \
    else if (matrix)                                                                                         \
      hipLaunchKernelGGL((gemm_nt_matrix_kernel<TA, TW, TC, 2, 3, 32, 2>), grid, block, 0, stream,           \
                         (TC*)C, ldc, (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, m_tiles,    \
                         n_tiles);                                                                           \
    else                                                                                                     \
      hipLaunchKernelGGL((gemm_nt_kernel<TA, TW, TC, 64, 64, 32>), grid, block, 0, stream, (TC*)C, ldc,      \
                         (const TA*)A, lda, (const TW*)W, (const TW*)bias, M, N, K, wide_a, wide_w);         \
  } while (0)
  if (in_bf16) {
    if (out_bf16) LAUNCH(bf16_t, bf16_t, bf16_t); else LAUNCH(bf16_t, bf16_t, float);
  } else {
    if (out_bf16) return -3;
    LAUNCH(float, float, float);
  }
#undef LAUNCH
  return GA_CHECK_LAUNCH();
}
