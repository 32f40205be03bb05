// Matrix products C[M, N] = A[M, K] . W[N, K]^T (+ bias[N]) with W stored [out, in] row-major, the
// layout of the checkpoint (ginfer/core/layer/linear.cc:9-20); 32-bit accumulation and the bias
// added in 32-bit before the one rounding (ginfer/core/op/kernels/cuda/gemm_kernel/
// gemm_kernel.cu:100-121, ginfer/core/op/kernels/cuda/gemv_kernel.cu:52-55).
//
// One kernel makes the true 32-bit product (no reduced-precision mode anywhere), on the matrix cores' 32-bit instruction over tiles of 32 x 32
// to 64 x 96 through LDS.  Every element of C is ONE accumulator that takes its terms over ascending k as fused multiply-adds, so its bits
// do not depend on M, on the tile it falls in or on the rest of the batch.  (Kernels of their own stood here for up to 64 rows, a
// wavefront per 16 columns with operands straight from memory, and for a head of 33 to 64 rows, on plain multiply-adds: each
// waited for memory after every few steps of its chain.  us of them -> of the tiles at 1, 16, 32 and 64 rows: 1,536 columns of 8,960 84, 90,
// 146, 247 -> 46, 47, 47, 47; 17,920 of 1,536 32, 35, 53, 98 -> 27, 28, 32, 45; 2,048 of 1,536 16.5, 17.9, 28.7, 44.2 -> 10.5, 11.2, 11.4, 11.3;
// 151,936 of 1,536 175, 245, 369, 488 -> 165, 189, 220, 265.)
// It is templated on storage, so that it also serves bfloat16 operands (the kernel tests' oracle and the
// fallback for shapes the bfloat16 kernels refuse).
#include "common.h"
#include <type_traits>
#include "ginfer_amd.h"   // the entry points below are checked against their declarations

#define GEMM_THREADS 256

// the first `valid` of four consecutive elements as floats, zeros behind them
template <typename T>
__device__ __forceinline__ void load4(float (&v)[4], const T* p, int valid) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = i < valid ? Num<T>::ld(p + i) : 0.f;
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

// v_mfma_f32_16x16x4_f32 takes, from lane l, row l % 16 of A and of
// W at k = step + l / 16 and adds its four products into the accumulator in ascending k as fused multiply-adds: measured
// on the device, its results over a K of 512 equal the chain of fmaf over ascending k bit for bit, for every element of
// the tile.  Register r of lane l receives row 4 (l / 16) + r, column
// l % 16 of a block.
//
// A workgroup of four wavefronts, 2 x 2 over a tile of 32 BM x 32 BN; a wavefront owns BM x BN blocks of 16 x 16.  K must
// not be split (one accumulator per element), so a block of 16 x 16 is a chain of K / 4 instructions of 32 cycles however
// the chip is filled (30 us for a K of 8,960): small blocks, so that few rows make enough chains for the 1,024
// SIMDs, and a chain that never waits.  Two steps of TK elements are on their way from memory in registers while a step
// is multiplied; the steps between lie in two buffers in LDS, one barrier a step; nothing in the loop is conditional (loads past the
// end repeat the last step's).  PIPED: a step's operands are in registers when it begins, and the next step's, the stores to LDS and the
// loads stand between its products (a K of 8,960 at up to 128 rows 59 -> 47 us, 256 rows 93 -> 85; what is left above the chain is the LDS pipe's, busy as
// long as the products are: twice the loads under way change nothing); with many tiles of 64 x 64 and more the workgroups of a compute unit
// cover each other's steps, and the registers that it costs are worth more (17,920 columns of 1,536 at 256 rows in tiles of 64 x 96 117 us, piped 123).  A row of LDS holds every 16
// elements of K with the four of a lane side by side (k = g, 4 + g, 8 + g, 12 + g): the operands of four instructions
// come in one 16-byte read and need no exchange between lanes (with the row swaps of gfx950 after the read the chain of
// a K of 8,960 took 91 us instead of 62), and with rows padded by four words neither side has bank conflicts.
// Workgroups that share rows of W are neighbours on one XCD, whose L2 then reads W once: columns of tiles go to the XCDs in
// turn, and the tiles of the columns that are left over to all eight alike (as whole columns they made a second round on the
// XCDs that got one more: 300 rows by 4,864, 51 columns of tiles, K 1,536, 84 us, now 54.5; 1,536 by 640 60 and 39.7; 2,048 by
// 32, one column, 21.5 and 14.5).  Rows that are not aligned take the same loads (4,096 rows by 5,000 of a K of 521, us: 264 in the
// tiles before, 330 element by element here, now 206; 256 by 1,536 of 1,537: 90, 49, 24).
// Measured on MI355X, us, before (32 x 32 x 2 blocks in tiles of 64 x 64 to 128 x 128, two barriers a step) -> now, for
// [rows] x 1,536 of a K of 8,960, x 2,048 of 1,536, and x 17,920 of 1,536: 64 rows 335 -> 47, 55 -> 11.3, 157 -> 45;
// 256 rows 232 -> 85, 45 -> 18.8, 224 -> 117; 512 rows 232 -> 134, 47.5 -> 31, 327 -> 229; 2,048 rows 634 -> 433,
// 136 -> 105, 905 -> 868 (130 of the 154 TFLOP/s that a large product reaches on this card).
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <typename TA, typename TW, typename TC, int BM, int BN, int TK, bool PIPED>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_nt_matrix_kernel(const TA* __restrict__ A, const TW* __restrict__ W, int64_t lda,
                                                                     int M, int N, int K, int m_tiles, int n_tiles,
                                                                     TC* __restrict__ C, int64_t ldc,
                                                                     const TW* __restrict__ bias) {
  constexpr int TM = 32 * BM, TN = 32 * BN, PAD = TK + 4;
  constexpr int GA = TM * TK / 4 / GEMM_THREADS, GW = TN * TK / 4 / GEMM_THREADS;
  static_assert(GA >= 1 && GW >= 1 && TK % 16 == 0, "tile sizes");
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
  float ra[2][GA][4], rw[2][GW][4];
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
    for (int i = 0; i < GA; ++i) load4<TA>(xa[i], pa[i] + k0, valid);
#pragma unroll
    for (int i = 0; i < GW; ++i) load4<TW>(xw[i], pw[i] + k0, valid);
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
  // A step: its operands lie in registers; between its products the next step's come out of LDS, the step behind that goes
  // into the buffer that this one's came from, and the loads of a later one are asked for, so that the chain of products waits for none of
  // it.  A wavefront all of whose rows or columns lie beyond the matrix only helps the others to their operands.
  constexpr int CHUNKS = TK / 16, GROUPS = CHUNKS * 4, READS = CHUNKS * (BM + BN), MOVES = GA + GW;
  struct Operands {
    float x[CHUNKS][BM][4], y[CHUNKS][BN][4];
  };
  auto read_one = [&](int b, int r, Operands& o) {
    const int c = r / (BM + BN), i = r % (BM + BN);
    const float4 v = i < BM ? *reinterpret_cast<const float4*>(&a_s[b][wm + (i < BM ? i : 0) * 16 + i16][c * 16 + 4 * kq])
                            : *reinterpret_cast<const float4*>(&w_s[b][wn + (i < BM ? 0 : i - BM) * 16 + i16][c * 16 + 4 * kq]);
    float (&to)[4] = i < BM ? o.x[c][i < BM ? i : 0] : o.y[c][i < BM ? 0 : i - BM];
    to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
  };
  auto stage_one = [&](int b, int i, float (&xa)[GA][4], float (&xw)[GW][4]) {
    const int gi = tid + (i < GA ? i : i - GA) * GEMM_THREADS, at16 = (gi % (TK / 4)) / 4 * 16 + gi % 4;
    float* to = i < GA ? &a_s[b][gi / (TK / 4)][at16] : &w_s[b][gi / (TK / 4)][at16];
    const float (&from)[4] = i < GA ? xa[i < GA ? i : 0] : xw[i < GA ? 0 : i - GA];
#pragma unroll
    for (int g = 0; g < 4; ++g) to[4 * g] = from[g];
  };
  auto fetch_one = [&](int i, float (&xa)[GA][4], float (&xw)[GW][4], int k0) {
    if (i < GA) load4_anywhere(xa[i < GA ? i : 0], pa[i < GA ? i : 0] + k0);
    else load4_anywhere(xw[i < GA ? 0 : i - GA], pw[i < GA ? 0 : i - GA] + k0);
  };
  auto step = [&](auto live, int b, const Operands& now, Operands& next, float (&xa)[GA][4], float (&xw)[GW][4], int k) {
#pragma unroll
    for (int p = 0; p < GROUPS; ++p) {
      const int c = p / 4, st = p % 4;
      if constexpr (decltype(live)::value) {
#pragma unroll
        for (int r = 0; r < READS; ++r)
          if (r * (GROUPS / 2) / READS == p) read_one(b ^ 1, r, next);
      }
#pragma unroll
      for (int i = 0; i < MOVES; ++i) {
        if (GROUPS / 4 + i * (GROUPS / 2) / MOVES == p) stage_one(b, i, xa, xw);
        if (GROUPS / 4 + i * (GROUPS / 2) / MOVES + 1 == p) fetch_one(i, xa, xw, k);
      }
      if constexpr (decltype(live)::value) {
#pragma unroll
        for (int i = 0; i < BM; ++i)
#pragma unroll
          for (int j = 0; j < BN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.x[c][i][st], now.y[c][j][st], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  };
  const int steps = K / TK, last = (steps - 1) * TK;
  const bool live = m0 + wm < M && n0 + wn < N;
  auto start = [&](int s) { return s * TK < last ? s * TK : last; };
  auto run = [&](auto on) {
    Operands o[2];
    fetch(ra[0], rw[0], 0);
    fetch(ra[1], rw[1], start(1));
    stage(0, ra[0], rw[0]);
    fetch(ra[0], rw[0], start(2));
    __syncthreads();
    if constexpr (decltype(on)::value) {
#pragma unroll
      for (int r = 0; r < READS; ++r) read_one(0, r, o[0]);
    }
    stage(1, ra[1], rw[1]);
    fetch(ra[1], rw[1], start(3));
    __syncthreads();
    // buffer 0 holds step 0 (in registers by now), buffer 1 step 1; ra[0] is step 2, ra[1] step 3
    int s = 0;
    for (; s + 2 <= steps; s += 2) {
      step(on, 0, o[0], o[1], ra[0], rw[0], start(s + 4));
      step(on, 1, o[1], o[0], ra[1], rw[1], start(s + 5));
    }
    if (s < steps) step(on, 0, o[0], o[1], ra[0], rw[0], last);
  };
  // a step, and what is left of K: all operands are asked for before the first is multiplied
  auto multiply = [&](int b) {
    Operands o;
#pragma unroll
    for (int r = 0; r < READS; ++r) read_one(b, r, o);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int i = 0; i < BM; ++i)
#pragma unroll
          for (int j = 0; j < BN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.x[c][i][st], o.y[c][j][st], acc[i][j], 0, 0, 0);
    }
  };
  auto plain = [&]() {
    fetch(ra[0], rw[0], 0);
    fetch(ra[1], rw[1], start(1));
    stage(0, ra[0], rw[0]);
    fetch(ra[0], rw[0], start(2));
    __syncthreads();
    int s = 0;
    for (; s + 2 <= steps; s += 2) {
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        multiply(d);
        stage(d ^ 1, ra[d ^ 1], rw[d ^ 1]);
        fetch(ra[d ^ 1], rw[d ^ 1], start(s + d + 3));
        __syncthreads();
      }
    }
    if (s < steps) {
      multiply(0);
      __syncthreads();
    }
  };
  if (steps > 0) {
    if constexpr (!PIPED) plain();
    else if (live) run(std::true_type());
    else run(std::false_type());
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

// in_bf16: A, W and bias are bfloat16 (else float); out_bf16: C is bfloat16 (else float).
extern "C" int ga_gemm_nt(void* C, int64_t ldc, const void* A, int64_t lda, const void* W,
                          const void* bias, int M, int N, int K, int in_bf16, int out_bf16,
                          hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0) return -1;
  // Tiles of 32 x 32, 64 x 64 (piped or not) or 64 x 96, whichever takes the least time by this sum.  A chip of 256 compute units works
  // off `rounds` tiles each; the first costs a tile's whole chain, further ones overlap with it.  Measured in us at a K of 1,536
  // (alone / each further round): 11.2 / 7.9, 30.5 / 26, 35.5 / 25.1, 47.5 / 39; the sums are what the sizes above take at that K or up to 15 %
  // more.
  const int tile_m[4] = {32, 64, 64, 64}, tile_n[4] = {32, 64, 64, 96};
  const float alone[4] = {11.2f, 30.5f, 35.5f, 47.5f}, further[4] = {7.9f, 26.f, 25.1f, 39.f};
  int tiling = -1, m_tiles = 0, n_tiles = 0;
  int64_t groups = 0;
  float least = 0.f;
  for (int t = 0; t < 4; ++t) {
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
  if ((M + 127) / 128 > 65535 || tiling < 0) return -2;
#define TILES(TA, TW, TC, ...)                                                                                                   \
  hipLaunchKernelGGL((gemm_nt_matrix_kernel<TA, TW, TC, __VA_ARGS__>), dim3((unsigned)groups), dim3(GEMM_THREADS), 0, stream,    \
                     (const TA*)A, (const TW*)W, lda, M, N, K, m_tiles, n_tiles, (TC*)C, ldc, (const TW*)bias)
#define LAUNCH(TA, TW, TC)                                    \
  do {                                                        \
    if (tiling == 0) TILES(TA, TW, TC, 1, 1, 64, true);       \
    else if (tiling == 1) TILES(TA, TW, TC, 2, 2, 32, true);  \
    else if (tiling == 2) TILES(TA, TW, TC, 2, 2, 32, false); \
    else TILES(TA, TW, TC, 2, 3, 32, false);                  \
  } while (0)
  if (in_bf16) {
    if (out_bf16) LAUNCH(bf16_t, bf16_t, bf16_t); else LAUNCH(bf16_t, bf16_t, float);
  } else {
    if (out_bf16) return -3;
    LAUNCH(float, float, float);
  }
#undef LAUNCH
#undef TILES
  return GA_CHECK_LAUNCH();
}
