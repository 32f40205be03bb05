// bfloat16 products A[M, K] . W[N, K]^T on the matrix cores over tiles through LDS, for the two products of a feed-forward
// whose results nobody wants as they are:
//   gated   W holds two stacked matrices of `cols` rows each (gate over up); out[M, cols] = the gate's activation times the up
//           product, rounded once (a library's product writes both to memory, rounded, and a second kernel reads them again);
//   parts   32-bit partial sums [parts][M][cols] of a K split over workgroups, for the norm that adds them up.
//
// A workgroup owns TN rows of W and TM rows of A; its wavefronts, WN x WM of them, own 32 NI x 32 MJ of the tile as blocks of
// v_mfma_f32_32x32x16_bf16 (one wavefront keeps that instruction busy; the 16x16x32 one is issued every 27 cycles from one
// wavefront where it takes 16).  K comes in slabs of 64 elements, which go from memory straight into one of NBUF buffers in
// LDS; operands come out of LDS half a slab ahead of their products.  In the middle of a slab its second half's operands are in
// registers: there all wait for the next slab and meet, once a slab, and from there on the slab's own buffer is filled with the
// slab NBUF on.  Loads and LDS reads are dealt between the products, so that no wavefront waits to issue them.  In the gated
// product a wavefront's first half of rows is the gate's and its second the up matrix's of the same columns, so that both
// sums of a result lie in one lane.  Workgroups that share rows of W are neighbours on one XCD, whose L2 then reads W once.
//
// What bounds it: many rows, the chip's power (products of random numbers run at 1,700 to 1,800 TFLOP/s, 2,400 of zeros) and the
// way of a slab from memory; few rows, the weights' way from memory.
#include "lds_load.h"
#include <type_traits>
#include "ginfer_amd.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// act.kind 0: SiLU(v) * u; 1: g * sigmoid(alpha g) * (u + shift), g = min(v, limit), u = clamp(u, -limit, limit); 2: the same
// with the sigmoid's limit, a step.  exp2 and the reciprocal are the hardware's: against 64 bits SiLU is off by at most 3 units of
// the 32-bit result's last place for v > -0.5, 6 down to -4, 18 down to -20 and 65 (4e-6 of it) down to -87, below which it is 0;
// with expf and a division, as the kernel for up to 16 rows has it, by at most 3.4 everywhere.  The one rounding that follows is
// 2^-9 of the result.  expf and the division cost 1 us of 27 at 64 rows and 41 of 464 at 2,048 (one tile's 128 results a thread
// are straight code that no one else has fetched yet), a correction of exp2's argument and one step on the reciprocal 21.
struct GateAct {
  int kind;
  float limit, alpha, shift;
};
__device__ __forceinline__ float gt_sigmoid(float z) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.4426950408889634f)); }
__device__ __forceinline__ float gt_act(float v, float u, const GateAct act) {
  if (act.kind == 0) return (v * gt_sigmoid(v)) * u;
  v = fminf(v, act.limit);
  u = fminf(fmaxf(u, -act.limit), act.limit);
  if (act.kind == 2) return (v > 0.f ? v : 0.f) * (u + act.shift);
  return (v * gt_sigmoid(act.alpha * v)) * (u + act.shift);
}
__device__ __forceinline__ uint2 gt_round4(const float (&y)[4]) {
  bf16x4 r;
#pragma unroll
  for (int x = 0; x < 4; ++x) r[x] = (__bf16)y[x];
  return __builtin_bit_cast(uint2, r);
}

template <int NI, int MJ, int WN, int WM, int NBUF, bool GATED>
__global__ __launch_bounds__(64 * WN * WM, 1) void gemm_tiles_kernel(
    void* __restrict__ C, int64_t ldc, const bf16_t* __restrict__ A, int64_t lda, const bf16_t* __restrict__ W, int M, int cols,
    int K, int m_tiles, int n_tiles, int slabs_per_part, GateAct act) {
  constexpr int WAVES = WN * WM, TN = 32 * NI * WN, TM = 32 * MJ * WM, COLS = GATED ? TN / 2 : TN;
  constexpr int BK = 64, ROW = 2 * BK, RPL = 1024 / ROW;             // bytes a row of a slab, rows a load brings
  constexpr int LW = TN / RPL / WAVES, LA = TM / RPL / WAVES, LOADS = LW + LA, SLAB = (TN + TM) * ROW;
  static_assert(TN % (RPL * WAVES) == 0 && TM % (RPL * WAVES) == 0, "loads");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int total = m_tiles * n_tiles, run = (total + 7) / 8, at8 = blockIdx.x / 8, id = (blockIdx.x % 8) * run + at8;
  if (at8 >= run || id >= total) return;
  const int mt = id % m_tiles, nt = id / m_tiles, m0 = mt * TM, c0 = nt * COLS;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wn = wave / WM;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t*)lds;
  const int slab0 = blockIdx.y * slabs_per_part, slabs = min(slabs_per_part, K / BK - slab0);
  // piece p (16 bytes) of row r lies at place p ^ (r % 8): eight rows' equal pieces in the eight places of 128 bytes
  const int lrow = lane / 8, piece = (lane % 8) ^ lrow;
  uint32_t src_w[LW], src_a[LA];
#pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wave * LW + j) * RPL + lrow;
    int col;
    if (GATED) {
      constexpr int H = 16 * NI;                  // of a wavefront's 32 NI rows, half are gate's
      const int w = r / (2 * H), q = r % (2 * H) / H;
      col = min(c0 + w * H + r % H, cols - 1) + q * cols;
    } else {
      col = min(c0 + r, cols - 1);
    }
    src_w[j] = ((uint32_t)col * (uint32_t)K + 8 * piece) * 2u;
  }
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = (wave * LA + j) * RPL + lrow;
    src_a[j] = ((uint32_t)min(m0 + r, M - 1) * (uint32_t)lda + 8 * piece) * 2u;
  }
  const char* wp = reinterpret_cast<const char*>(W) + (int64_t)slab0 * ROW;
  const char* ap = reinterpret_cast<const char*>(A) + (int64_t)slab0 * ROW;
  uint32_t fill = base;                           // the buffer that the next slab goes to
  auto bring_one = [&](int j) {
    if (j < LW) lds_bring_from(fill + (wave * LW + j) * 1024, src_w[j], wp);
    else lds_bring_from(fill + TN * ROW + (wave * LA + j - LW) * 1024, src_a[j - LW], ap);
  };
  auto brought = [&]() {
    wp += ROW;
    ap += ROW;
    fill = fill == base + (NBUF - 1) * SLAB ? base : fill + SLAB;
  };
  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.f;
  // a wavefront's operands come in halves of a slab: KH steps of 16 elements of K
  constexpr int KH = BK / 32;
  const int turn = c & 7;
  int at[2 * KH];
#pragma unroll
  for (int k = 0; k < 2 * KH; ++k) at[k] = ((2 * k + g) ^ turn) * 16 + c * ROW;
  const unsigned char* cur = lds;
  bf16x8 a[2][KH][NI], b[2][KH][MJ];
  constexpr int READS = KH * (MJ + NI), GROUPS = KH * NI;       // a group: a row of MJ products
  auto read_one = [&](int half, int x) {
    const int k = x / (MJ + NI), y = x % (MJ + NI);
    if (y < MJ) b[half][k][y] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(cur + at[half * KH + k] + TN * ROW + (wm * MJ + y) * 32 * ROW));
    else a[half][k][y - MJ] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(cur + at[half * KH + k] + (wn * NI + y - MJ) * 32 * ROW));
  };
  // the products of one half, beside the reads of the other and the loads of a later slab
  auto half_slab = [&](int half, auto loads) {
#pragma unroll
    for (int x = 0; x < GROUPS; ++x) {
      const int k = x / NI, i = x % NI;
      if (decltype(loads)::value) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j)
          if (j * GROUPS / LOADS == x) bring_one(j);
      }
#pragma unroll
      for (int y = 0; y < READS; ++y)
        if (y * (GROUPS - 1) / READS == x) read_one(1 - half, y);
#pragma unroll
      for (int j = 0; j < MJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[half][k][i], b[half][k][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < NBUF; ++s)
    if (s < slabs) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) bring_one(j);
      brought();
    }
  if (slabs >= NBUF) lds_wait_and_meet<(NBUF - 1) * LOADS>();
  else lds_wait_and_meet<0>();
#pragma unroll
  for (int y = 0; y < READS; ++y) read_one(0, y);
  int s = 0;
  for (; s + NBUF < slabs; ++s) {
    half_slab(0, std::false_type());
    lds_wait_and_meet<(NBUF - 2) * LOADS>();
    cur = cur == lds + (NBUF - 1) * SLAB ? lds : cur + SLAB;
    half_slab(1, std::true_type());
    brought();
  }
  for (; s < slabs; ++s) {
    half_slab(0, std::false_type());
    lds_wait_and_meet<0>();
    cur = cur == lds + (NBUF - 1) * SLAB ? lds : cur + SLAB;
    half_slab(1, std::false_type());
  }
  if constexpr (!GATED) {
    float* P = reinterpret_cast<float*>(C) + (int64_t)blockIdx.y * M * cols;
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      const int m = m0 + (wm * MJ + j) * 32 + c;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = c0 + (wn * NI + i) * 32 + 8 * q + 4 * g;
          if (m < M && n < cols)
            *reinterpret_cast<float4*>(P + (int64_t)m * cols + n) = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
        }
    }
  } else {
    // through LDS, so that rows leave in 16-byte pieces side by side
    constexpr int PITCH = COLS + 8, OI = NI / 2;
    __syncthreads();
    bf16_t* tile = reinterpret_cast<bf16_t*>(lds);
#pragma unroll
    for (int i = 0; i < OI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          float y[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) y[x] = gt_act(acc[i][j][4 * q + x], acc[i + OI][j][4 * q + x], act);
          *reinterpret_cast<uint2*>(tile + ((wm * MJ + j) * 32 + c) * PITCH + (wn * OI + i) * 32 + 8 * q + 4 * g) = gt_round4(y);
        }
    __syncthreads();
    bf16_t* out = reinterpret_cast<bf16_t*>(C);
    for (int idx = tid; idx < TM * COLS / 8; idx += 64 * WAVES) {
      const int m = idx / (COLS / 8), n = idx % (COLS / 8) * 8;
      if (m0 + m < M && c0 + n < cols)
        *reinterpret_cast<uint4*>(out + (int64_t)(m0 + m) * ldc + c0 + n) = *reinterpret_cast<const uint4*>(tile + m * PITCH + n);
    }
  }
}

template <int NI, int MJ, int WN, int WM, int NBUF, bool GATED>
static int gt_launch(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, int M, int cols, int K, int parts,
                     GateAct act, hipStream_t stream) {
  constexpr int TN = 32 * NI * WN, TM = 32 * MJ * WM, COLS = GATED ? TN / 2 : TN;
  constexpr int slabs_bytes = (TN + TM) * 128 * NBUF, out_bytes = GATED ? TM * (COLS + 8) * 2 : 0;
  constexpr int bytes = slabs_bytes > out_bytes ? slabs_bytes : out_bytes;
  const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tiles_kernel<NI, MJ, WN, WM, NBUF, GATED>),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, bytes);       // the current device's
  if (raised != hipSuccess) return (int)raised;
  const int64_t m_tiles = (M + TM - 1) / TM, n_tiles = (cols + COLS - 1) / COLS, groups = (m_tiles * n_tiles + 7) / 8 * 8;
  if (groups > 0x7fffffff / 256) return -2;
  const int per_part = (K / 64 + parts - 1) / parts;
  if ((parts - 1) * per_part >= K / 64) return -4;       // a part without a slab
  hipLaunchKernelGGL((gemm_tiles_kernel<NI, MJ, WN, WM, NBUF, GATED>), dim3((unsigned)groups, parts), dim3(64 * WN * WM), bytes, stream,
                     C, ldc, (const bf16_t*)A, lda, (const bf16_t*)W, M, cols, K, (int)m_tiles, (int)n_tiles, per_part, act);
  return GA_CHECK_LAUNCH();
}

static int gt_check(const void* C, const void* A, int64_t lda, const void* W, int64_t w_rows, int M, int cols, int K) {
  if (cols <= 0 || cols % 8 || K <= 0 || K % 64 || lda < K || lda % 8) return -1;
  if (((uintptr_t)C | (uintptr_t)A | (uintptr_t)W) & 15) return -3;
  if (w_rows * K * 2 >= (1ll << 32) || (int64_t)M * lda * 2 >= (1ll << 32)) return -5;      // offsets are 32-bit
  return 0;
}

// tiling: which tiles, rows of W x rows of A; the caller chooses by sizes and by how full they leave the chip's rounds
// (gated_tiling in kernels/ops.py, tiles_gated in parts/linear.py, the fastest and the library beside each other).  us, product and
// activation by the library's best way -> here, as replays of a graph over several layers' weights: 17,920 rows of W, K 1,536: 64 rows
// 30.6 -> 26.9, 128 rows 35.1 -> 30.2 (tiles of 128 x 256, half of them rows that do not exist, 33.5), 256 rows 43.6 -> 37.2, 384
// rows 45.9 -> 39.9; 37,888 rows, K 3,584: 128 rows 84.0 -> 79.3, 384 rows 133.9 -> 121.4, 1,000 rows 324 -> 272, 1,280 rows 386 ->
// 291, 2,048 rows 552 -> 464; 19,456 rows, K 2,560: 128 rows 46.0 -> 44.0 (128 x 256 tiles 49.1), 384 rows 64.0 -> 57.8.
// Tiles of 192 rows of W stand beside the others (6 to 8) where those leave the chip's rounds emptier (gated_wide_tiling in
// kernels/ops.py has the rule and the figures): many rows run at 1.5 to 1.7 GHz, which is the power they may draw, with the
// matrix cores busy 0.61 (192 x 256, K 1,536) to 0.68 of the time (256 x 256, K 3,584) and wavefronts waiting 0.21 and 0.14 of it, so
// that only less padding, not a busier loop, gains much.
extern "C" int ga_gemm_tiles_gated(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, int M, int cols, int K, int kind,
                                   float limit, float alpha, float shift, int tiling, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = gt_check(C, A, lda, W, 2 * (int64_t)cols, M, cols, K);
  if (rc) return rc;
  if (kind < 0 || kind > 2 || ldc < cols || ldc % 8) return -1;
  const GateAct act = {kind, limit, alpha, shift};
  switch (tiling) {
    case 0: return gt_launch<2, 1, 2, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 64
    case 1: return gt_launch<4, 2, 1, 4, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 256
    case 2: return gt_launch<4, 2, 2, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 256 x 128
    case 3: return gt_launch<4, 4, 2, 2, 2, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 256 x 256
    case 4: return gt_launch<2, 2, 2, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 128
    case 6: return gt_launch<6, 1, 1, 2, 4, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 64
    case 7: return gt_launch<6, 1, 1, 4, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 128
    case 8: return gt_launch<6, 2, 1, 4, 2, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 256
  }
  return -6;
}

// Up to 64 rows tiles of 64 x 64, beyond 128 x 64.  us with the norm that adds the parts, the best other way -> here, with as many
// parts as keep to one round of the chip: 1,536 columns of a K of 8,960: 64 rows 19.5 -> 12.9, 128 rows 20.9 -> 16.7, 256 rows 24.2 ->
// 20.1; 2,048 of 11,008: 25.0 -> 16.9, 27.3 -> 21.2, 35.8 -> 30.6; 3,584 of 3,584: 14.6 -> 13.6, 17.3 -> 15.6, 22.5 -> 19.1.  A workgroup
// more than a round costs it again: 11 parts of the first, 264 workgroups, 16.0.
extern "C" int ga_gemm_tiles_parts(void* C, const void* A, int64_t lda, const void* W, int M, int cols, int K, int parts,
                                   hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = gt_check(C, A, lda, W, cols, M, cols, K);
  if (rc) return rc;
  if (parts < 1 || parts > K / 64 || parts > 65535) return -1;
  const GateAct act = {0, 0.f, 0.f, 0.f};
  if (M <= 64) return gt_launch<2, 1, 1, 2, 4, false>(C, cols, A, lda, W, M, cols, K, parts, act, stream);
  return gt_launch<2, 1, 2, 2, 3, false>(C, cols, A, lda, W, M, cols, K, parts, act, stream);
}
