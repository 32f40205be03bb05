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
// product the first half of a block's rows is the gate's and its second the up matrix's of the same columns, so that both
// sums of a result lie in one lane.  Workgroups that share rows of W are neighbours on one XCD, whose L2 then reads W once.
//
// What bounds it: many rows, the chip's power (products of random numbers run at 1,700 to 1,800 TFLOP/s, 2,400 of zeros) and the
// way of a slab from memory; few rows, the weights' way from memory.  192 x 256 tiles of 2,048 rows, 17,920 rows of W, K 1,536, us: the products
// alone 73, the loads alone 64 (whatever order the tiles come in), both 85, with the LDS reads 95, with the activation 120; the last is a
// third of that where eight wavefronts share it rather than four: 105, though they read a quarter more from LDS.  Tiles beyond 128 x 128
// have eight, us of four and eight: 256 x 256 (37,888 rows, K 3,584, 2,048 rows) 467 -> 455, 128 x 256 (17,920, K 1,536, 1,024 rows) 69.6 -> 65.6, 256 x
// 128 68.9 -> 63.7, 192 x 128 59.1 -> 57.5; 128 x 128 has four, 65.9 against 68.1.  Loads dealt faster than evenly are slower (all at once
// 105 -> 109), W or A read past the caches too (114, 126).
#include "lds_load.h"
#include <type_traits>
#include "ginfer_amd.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// act.kind 0: SiLU(v) * u; 1: g * sigmoid(alpha g) * (u + shift), g = min(v, limit), u = clamp(u, -limit, limit); 2: the same
// with the sigmoid's limit, a step.  Without EXPF, exp2 and the reciprocal are the hardware's: against 64 bits SiLU is off by at most 3 units of
// the 32-bit result's last place for v > -0.5, 6 down to -4, 18 down to -20 and 65 (4e-6 of it) down to -87, below which it is 0;
// with expf and a division (EXPF), as the kernel that streams the weights has it, by at most 3.4 everywhere.  The one rounding that follows is
// 2^-9 of the result.  expf and the division cost 1 us of 27 at 64 rows and 41 of 464 at 2,048 (one tile's 128 results a thread
// are straight code that no one else has fetched yet), a correction of exp2's argument and one step on the reciprocal 21.
struct GateAct {
  int kind;
  float limit, alpha, shift;
};
template <bool EXPF>
__device__ __forceinline__ float gt_sigmoid(float z) {
  if (EXPF) return 1.0f / (1.0f + expf(-z));
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.4426950408889634f));
}
template <bool EXPF = false>
__device__ __forceinline__ float gt_act(float v, float u, const GateAct act) {
  if (act.kind == 0) return (v * gt_sigmoid<EXPF>(v)) * u;
  v = fminf(v, act.limit);
  u = fminf(fmaxf(u, -act.limit), act.limit);
  if (act.kind == 2) return (v > 0.f ? v : 0.f) * (u + act.shift);
  return (v * gt_sigmoid<EXPF>(act.alpha * v)) * (u + act.shift);
}
__device__ __forceinline__ uint2 gt_round4(const float (&y)[4]) {
  bf16x4 r;
#pragma unroll
  for (int x = 0; x < 4; ++x) r[x] = (__bf16)y[x];
  return __builtin_bit_cast(uint2, r);
}

template <int NI, int MJ, int WN, int WM, int NBUF, bool GATED>
__global__ __launch_bounds__(64 * WN * WM, 1) void gemm_tiles_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int64_t lda, int M, int cols, int K, int m_tiles, int n_tiles,
    int slabs_per_part, void* __restrict__ C, int64_t ldc, GateAct act) {
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
    if (GATED) col = min(c0 + r / 32 * 16 + r % 16, cols - 1) + r % 32 / 16 * cols;      // of a block's 32 rows, 16 are the gate's
    else col = min(c0 + r, cols - 1);
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
  // the last slabs: each waits for the next one only
  auto last = [&](auto left) {
    if (s >= slabs) return;
    half_slab(0, std::false_type());
    lds_wait_and_meet<decltype(left)::value * LOADS>();
    cur = cur == lds + (NBUF - 1) * SLAB ? lds : cur + SLAB;
    half_slab(1, std::false_type());
    ++s;
  };
  if constexpr (NBUF >= 4) last(std::integral_constant<int, 2>());
  if constexpr (NBUF >= 3) last(std::integral_constant<int, 1>());
  last(std::integral_constant<int, 0>());
  last(std::integral_constant<int, 0>());
  static_assert(NBUF <= 4, "the last slabs");
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
    constexpr int PITCH = COLS + 8;
    __syncthreads();
    bf16_t* tile = reinterpret_cast<bf16_t*>(lds);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          float y[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) y[x] = gt_act(acc[i][j][4 * q + x], acc[i][j][8 + 4 * q + x], act);
          *reinterpret_cast<uint2*>(tile + ((wm * MJ + j) * 32 + c) * PITCH + (wn * NI + i) * 16 + 8 * q + 4 * g) = gt_round4(y);
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
                     (const bf16_t*)A, (const bf16_t*)W, lda, M, cols, K, (int)m_tiles, (int)n_tiles, per_part, C, ldc, act);
  return GA_CHECK_LAUNCH();
}

static int gt_check(const void* C, const void* A, int64_t lda, const void* W, int64_t w_rows, int M, int cols, int K) {
  if (cols <= 0 || cols % 8 || K <= 0 || K % 64 || lda < K || lda % 8) return -1;
  if (((uintptr_t)C | (uintptr_t)A | (uintptr_t)W) & 15) return -3;
  if (w_rows * K * 2 >= (1ll << 32) || (int64_t)M * lda * 2 >= (1ll << 32)) return -5;      // offsets are 32-bit
  return 0;
}

// ---- up to 512 rows, dealt evenly to the chip
// W's rows come in units of eight: four columns' gates and the same columns' ups.  Column group b of G owns the units [b U / G, (b + 1)
// U / G), row tile t of T the rows [t R, (t + 1) R), and G T workgroups make whole rounds of the chip's compute units, so that each
// takes in the same bytes, whatever the sizes; a tile has room for NB blocks of 16 rows of W and TM rows of A, and what of that
// it does not own is not loaded.  Eight wavefronts, WN x WM of the tile's blocks of v_mfma_f32_16x16x32_bf16 and WK of a slab's K.
//
// What bounds it: few rows, the weights' way from memory (64 rows by 17,920 rows of W, K 1,536: 55 MB in 10.6 us, 5.2 TB/s, where a
// compute unit takes in 39 GB/s).  From about 128 rows on, where most of what a unit takes in comes from its L2: loads return in order, so its stream
// of lines goes at the pace of those from memory, 45 to 50 GB/s a unit (110 with none from memory).  Either way the bytes a compute unit takes in
// are what counts: all 256 at work with a few rows fewer each, not the 188 of tiles of 192 x 128 (256 rows by 17,920 rows of W, K 1,536:
// the loads alone 20.8 us there, 18.0 here, of 26.0 and 22.9 whole).  W is asked for as memory that is read once (nt), so that A
// stays in the L2s: 18.1 -> 17.4 us with a line of W wanted twice, 11.5 -> 10.6 with it wanted once (64 rows).  Slabs of 128 elements
// where the tile leaves room (WK 2): half the meetings, 5 % of the loads' time.
template <int NI, int MJ, int WN, int WM, int WK, int NBUF>
struct SpreadTile {
  static constexpr int WAVES = WN * WM * WK, TM = 16 * MJ * WM, NB = NI * WN, TW = 16 * NB, BK = 64 * WK;
  static constexpr int ROW = 2 * BK, RPL = 1024 / ROW, LPR = ROW / 16;           // bytes a row of a slab; rows a load brings, lanes a row
  static constexpr int LW = (TW / RPL + WAVES - 1) / WAVES, LA = (TM / RPL + WAVES - 1) / WAVES, LOADS = LW + LA, SLAB = (TW + TM) * ROW;
  static constexpr int SUMS = WK == 2 ? (NI * MJ + 1) / 2 * WAVES * 1024 : 0, PITCH = 8 * NB + 4, OUT = TM * PITCH * 2;
  static constexpr int SLABS = SLAB * NBUF, LDS = SLABS > SUMS ? (SLABS > OUT ? SLABS : OUT) : (SUMS > OUT ? SUMS : OUT);
  static_assert(TW % RPL == 0 && TM % RPL == 0 && LDS <= 160 * 1024 && LOADS <= 7 && LOADS * (NBUF - 1) < 64, "tile");
};

// A tile's sums over the slabs [slab0, slab0 + slabs) of K: acc of wavefront (wn, wm, wk), block (i, j) the rows 16 (wn NI + i) of the tile of
// W by the rows 16 (wm MJ + j) of A; with WK 2 block t = i MJ + j is whole in the wavefront with wk = t % 2.  row_of_w(r): which row of W
// is row r of the tile, for r below 8 `own`.  Afterwards the LDS is free.
template <int NI, int MJ, int WN, int WM, int WK, int NBUF, typename RowOfW>
__device__ __forceinline__ void spread_sums(f32x4 (&acc)[NI][MJ], unsigned char* lds, const bf16_t* __restrict__ A, int64_t lda,
                                            const bf16_t* __restrict__ W, int K, int slab0, int slabs, int m0, int live, int own,
                                            RowOfW row_of_w) {
  using S = SpreadTile<NI, MJ, WN, WM, WK, NBUF>;
  constexpr int WAVES = S::WAVES, ROW = S::ROW, RPL = S::RPL, LPR = S::LPR, LW = S::LW, LA = S::LA, LOADS = S::LOADS;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);
  const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t*)lds + wave * 1024;
  // load l of W or of A is wavefront l % WAVES's; how many a slab takes of it
  const int of_w = own * 8 / RPL, of_a = (live + RPL - 1) / RPL;
  const int mine_w = of_w > wave ? (of_w - wave + WAVES - 1) / WAVES : 0, mine_a = of_a > wave ? (of_a - wave + WAVES - 1) / WAVES : 0;
  const int mine = mine_w + mine_a;
  uint32_t src_w[LW], src_a[LA];
#pragma unroll
  for (int j = 0; j < LW; ++j) {      // piece p of row r of a tile lies at place p ^ (r % LPR)
    const int r = min(wave + j * WAVES, of_w - 1) * RPL + lane / LPR, piece = (lane % LPR) ^ (r & (LPR - 1));
    src_w[j] = ((uint32_t)row_of_w(r) * (uint32_t)K + 8 * piece) * 2u;
  }
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int r = (wave + j * WAVES) * RPL + lane / LPR, piece = (lane % LPR) ^ (r & (LPR - 1));
    src_a[j] = ((uint32_t)(m0 + min(r, live - 1)) * (uint32_t)lda + 8 * piece) * 2u;
  }
  const char* wp = reinterpret_cast<const char*>(W) + (int64_t)slab0 * ROW;
  const char* ap = reinterpret_cast<const char*>(A) + (int64_t)slab0 * ROW;
  uint32_t fill = base;                           // the buffer that the next slab goes to
  int fill_at = 0, read_at = 0;
  auto bring_one = [&](int j) {
    if (j < LW) {
      if (j < mine_w) lds_bring_once_from(fill + j * WAVES * 1024, src_w[j], wp);
    } else if (j - LW < mine_a) {
      lds_bring_from(fill + S::TW * ROW + (j - LW) * WAVES * 1024, src_a[j - LW], ap);
    }
  };
  auto brought = [&]() {
    wp += ROW;
    ap += ROW;
    fill_at = fill_at == NBUF - 1 ? 0 : fill_at + 1;
    fill = base + fill_at * S::SLAB;
  };
  // all but the youngest n slabs' loads are in, and all wavefronts meet
  auto wait_for = [&](auto n) {
    constexpr int N = decltype(n)::value;
    switch (mine) {
      case 1: lds_wait_and_meet<N>(); break;
      case 2: lds_wait_and_meet<2 * N>(); break;
      case 3: lds_wait_and_meet<3 * N>(); break;
      case 4: lds_wait_and_meet<4 * N>(); break;
      case 5: lds_wait_and_meet<5 * N>(); break;
      case 6: lds_wait_and_meet<6 * N>(); break;
      case 7: lds_wait_and_meet<7 * N>(); break;
      default: lds_wait_and_meet<0>();
    }
  };
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int at[2];                                      // a wavefront has two steps of 32 of every slab
#pragma unroll
  for (int k = 0; k < 2; ++k) at[k] = (((wk * 2 + k) * 4 + g) ^ (c & (LPR - 1))) * 16 + c * ROW;
  const unsigned char* cur = lds;
  bf16x8 a[2][NI], bb[2][MJ];
  constexpr int READS = MJ + NI;
  auto read_one = [&](int k, int y) {
    if (y < MJ) bb[k][y] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(cur + at[k] + (S::TW + (wm * MJ + y) * 16) * ROW));
    else a[k][y - MJ] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(cur + at[k] + (wn * NI + y - MJ) * 16 * ROW));
  };
  // the products of one step, beside the reads of the next and the loads of a later slab
  auto step = [&](int k, auto loads) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (decltype(loads)::value) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j)
          if (j * NI / LOADS == i) bring_one(j);
      }
#pragma unroll
      for (int y = 0; y < READS; ++y)
        if (y * (NI - 1) / READS == i) read_one(1 - k, y);
#pragma unroll
      for (int j = 0; j < MJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k][i], bb[k][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto turn = [&]() {
    read_at = read_at == NBUF - 1 ? 0 : read_at + 1;
    cur = lds + read_at * S::SLAB;
  };
#pragma unroll
  for (int s = 0; s < NBUF; ++s)
    if (s < slabs) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) bring_one(j);
      brought();
    }
  if (slabs >= NBUF) wait_for(std::integral_constant<int, NBUF - 1>());
  else lds_wait_and_meet<0>();
#pragma unroll
  for (int y = 0; y < READS; ++y) read_one(0, y);
  int s = 0;
  for (; s + NBUF < slabs; ++s) {                 // in mid-slab its operands are all in registers, and its buffer is free
    step(0, std::false_type());
    wait_for(std::integral_constant<int, NBUF - 2>());
    turn();
    step(1, std::true_type());
    brought();
  }
  // the last NBUF slabs (or all, where K has fewer: then all are in): each waits for the next one only
  auto last = [&](auto left) {
    if (s >= slabs) return;
    step(0, std::false_type());
    wait_for(left);
    turn();
    step(1, std::false_type());
    ++s;
  };
  if constexpr (NBUF >= 7) last(std::integral_constant<int, 5>());
  if constexpr (NBUF >= 6) last(std::integral_constant<int, 4>());
  if constexpr (NBUF >= 5) last(std::integral_constant<int, 3>());
  if constexpr (NBUF >= 4) last(std::integral_constant<int, 2>());
  if constexpr (NBUF >= 3) last(std::integral_constant<int, 1>());
  last(std::integral_constant<int, 0>());
  last(std::integral_constant<int, 0>());
  static_assert(NBUF >= 2 && NBUF <= 7, "the last slabs");
  __syncthreads();
  constexpr int T = NI * MJ;
  if constexpr (WK == 2) {                        // the parts of K meet: block t's sums are the wavefront's with wk = t % 2
    constexpr int PER = (T + 1) / 2;
    f32x4* area = reinterpret_cast<f32x4*>(lds);
    const int other = wave ^ (WM * WN);
#pragma unroll
    for (int t = 0; t < T; ++t)
      if (t % 2 != wk) area[(wave * PER + t / 2) * 64 + lane] = acc[t / MJ][t % MJ];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t)
      if (t % 2 == wk) {
        const f32x4 v = area[(other * PER + t / 2) * 64 + lane], h = acc[t / MJ][t % MJ];
        acc[t / MJ][t % MJ] = wk ? v + h : h + v;
      }
    __syncthreads();
  }
}

// What workgroup `id` of m_tiles x groups owns: rows of A from m0 on, `live` of them, and units of W from u0 on, `own` of them.  Workgroups
// that share rows of W are neighbours on one XCD.
struct SpreadShare {
  int m0, live, u0, own;
  // units of W are each * groups + rest; in 32 bits (in 64 the divisions stood in front of the first load for half a microsecond)
  __device__ __forceinline__ bool take(int M, int each, int rest, int m_tiles, int tile_rows, int groups) {
    const int total = m_tiles * groups, run = (total + 7) / 8, at8 = blockIdx.x / 8, id = (blockIdx.x % 8) * run + at8;
    if (at8 >= run || id >= total) return false;
    const int b = id / m_tiles;
    m0 = id % m_tiles * tile_rows;
    live = min(tile_rows, M - m0);
    auto first = [&](int x) {                     // x * units / groups
      return x * each + (groups <= 1 << 16 ? (int)((uint32_t)x * (uint32_t)rest / (uint32_t)groups) : (int)((int64_t)x * rest / groups));
    };
    u0 = __builtin_amdgcn_readfirstlane(first(b));
    own = __builtin_amdgcn_readfirstlane(first(b + 1)) - u0;
    return true;
  }
};
// Lanes of even g hold four columns' first rows of W (gates, a head's lower half), the 16 lanes behind them the second ones: exchanged
// so that every lane has both of two columns, 2 g and 2 g + 1 of the block's eight.
struct SpreadPairs {
  float first[2], second[2];
  __device__ __forceinline__ explicit SpreadPairs(const f32x4& v) {
    const auto even = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[0]), __float_as_uint(v[2]), false, false);
    const auto odd = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[1]), __float_as_uint(v[3]), false, false);
    first[0] = __uint_as_float(even[0]);
    second[0] = __uint_as_float(even[1]);
    first[1] = __uint_as_float(odd[0]);
    second[1] = __uint_as_float(odd[1]);
  }
};
__device__ __forceinline__ uint32_t gt_round2(float a, float b) {
  const bf16x2 r = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, r);
}

// EXPF: products that the kernel streaming the weights would take otherwise (up to 32 rows, or 64 of fewer than 4,096 rows of W) keep its
// activation: 0.3 to 0.4 us of 6 to 16 there; with more rows, whose other tiles have the hardware's too, it would be 0.4 to 2.7.
template <bool EXPF, int NI, int MJ, int WN, int WM, int WK, int NBUF>
__global__ __launch_bounds__(64 * WN * WM * WK, 1) void gemm_spread_gated_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int64_t lda, int M, int cols, int K, int m_tiles, int tile_rows,
    int groups, int each, int rest, bf16_t* __restrict__ C, int64_t ldc, GateAct act) {
  using S = SpreadTile<NI, MJ, WN, WM, WK, NBUF>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  SpreadShare mine;
  if (!mine.take(M, each, rest, m_tiles, tile_rows, groups)) return;
  const int c0 = 4 * mine.u0;
  f32x4 acc[NI][MJ];
  // rows 0 to 3 of a unit are gates, 4 to 7 the same columns' ups
  spread_sums<NI, MJ, WN, WM, WK, NBUF>(acc, lds, A, lda, W, K, 0, K / S::BK, mine.m0, mine.live, mine.own,
                                        [&](int r) { return c0 + (r / 8) * 4 + (r & 3) + ((r & 4) ? cols : 0); });
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);
  bf16_t* tile = reinterpret_cast<bf16_t*>(lds);       // through LDS, so that a row's columns leave side by side
#pragma unroll
  for (int t = 0; t < NI * MJ; ++t)
    if (WK == 1 || t % 2 == wk) {
      const int i = t / MJ, j = t % MJ;
      const SpreadPairs v(acc[i][j]);
      *reinterpret_cast<uint32_t*>(tile + ((wm * MJ + j) * 16 + c) * S::PITCH + (wn * NI + i) * 8 + 2 * g) =
          gt_round2(gt_act<EXPF>(v.first[0], v.second[0], act), gt_act<EXPF>(v.first[1], v.second[1], act));
    }
  __syncthreads();
  for (int idx = threadIdx.x; idx < S::TM * 2 * S::NB; idx += 64 * S::WAVES) {
    const int m = idx / (2 * S::NB), q = idx % (2 * S::NB);
    if (m < mine.live && q < mine.own)
      *reinterpret_cast<uint2*>(C + (int64_t)(mine.m0 + m) * ldc + c0 + 4 * q) = *reinterpret_cast<const uint2*>(tile + m * S::PITCH + 4 * q);
  }
}

// The same for partial sums [parts][M][cols]: the grid's y is the part of K, a unit eight neighbouring columns.
template <int NI, int MJ, int WN, int WM, int WK, int NBUF>
__global__ __launch_bounds__(64 * WN * WM * WK, 1) void gemm_spread_parts_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int M, int cols, int K, int m_tiles, int tile_rows, int groups,
    int each, int rest, int slabs_per_part, float* __restrict__ C) {
  using S = SpreadTile<NI, MJ, WN, WM, WK, NBUF>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  SpreadShare mine;
  if (!mine.take(M, each, rest, m_tiles, tile_rows, groups)) return;
  const int c0 = 8 * mine.u0, slab0 = blockIdx.y * slabs_per_part;
  f32x4 acc[NI][MJ];
  spread_sums<NI, MJ, WN, WM, WK, NBUF>(acc, lds, A, lda, W, K, slab0, min(slabs_per_part, K / S::BK - slab0), mine.m0, mine.live, mine.own,
                                        [&](int r) { return c0 + r; });
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);
  float* P = C + ((int64_t)blockIdx.y * M + mine.m0) * cols + c0;
#pragma unroll
  for (int t = 0; t < NI * MJ; ++t)
    if (WK == 1 || t % 2 == wk) {
      const int i = t / MJ, m = (wm * MJ + t % MJ) * 16 + c, n = (wn * NI + i) * 16 + 4 * g;
      const f32x4 v = acc[i][t % MJ];
      if (m < mine.live && n < 8 * mine.own) *reinterpret_cast<float4*>(P + (int64_t)m * cols + n) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// The fused q|k|v projection of a step of 17 to 512 rows with its epilogue: bias, NeoX rotation of q and k on the 32-bit sums, q to its own
// buffer, k and v into the paged cache (layouts and formula as in rope_kv.hip).  A unit is four columns of a head and their rotation
// partners half a head on, or eight columns of a v head.
struct SpreadQkv {
  const bf16_t* bias;
  const int32_t* positions;
  const float *cos_t, *sin_t;
  const int64_t* slots;
  bf16_t *k_pages, *v_pages;
  int nh, nkv, page_size, write_kv;
};
template <int NI, int MJ, int WN, int WM, int WK, int NBUF>
__global__ __launch_bounds__(64 * WN * WM * WK, 1) void gemm_spread_qkv_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int K, int M, int m_tiles, int tile_rows, int groups, int each,
    int rest, int hd, int turned_heads, bf16_t* __restrict__ q_out, const SpreadQkv x) {
  using S = SpreadTile<NI, MJ, WN, WM, WK, NBUF>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  SpreadShare mine;
  if (!mine.take(M, each, rest, m_tiles, tile_rows, groups)) return;
  const int half = hd / 2, per_head = hd / 8, turned = turned_heads * per_head;      // units of a head; of q and k
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave % WM, wn = wave / WM % WN, wk = wave / (WM * WN);
  // What the epilogue needs from memory: positions and slots of the lane's rows, asked for now (through buffer descriptors: plain loads
  // would be moved down to their use); then, a few blocks at a time, cosines, sines and biases, and the stores.  Block by block each would wait for two
  // ways to memory.
  int pos[MJ];
  int64_t slots[MJ];
  {
    const __amdgpu_buffer_rsrc_t at_pos = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(x.positions + mine.m0), 0, mine.live * 4, 0x00027000);
    const __amdgpu_buffer_rsrc_t at_slot = __builtin_amdgcn_make_buffer_rsrc(const_cast<int64_t*>(x.slots + mine.m0), 0, x.write_kv ? mine.live * 8 : 0, 0x00027000);
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      const int row = min((wm * MJ + j) * 16 + c, mine.live - 1);
      pos[j] = (int)__builtin_amdgcn_raw_buffer_load_b32(at_pos, row * 4, 0, 0);
      slots[j] = __builtin_bit_cast(int64_t, __builtin_amdgcn_raw_buffer_load_b64(at_slot, row * 8, 0, 0));
    }
  }
  // the first row of W of a unit, and how far on its second four rows lie (heads of a power of two: by shifts, a division is some 20 instructions)
  const int shift = (per_head & (per_head - 1)) == 0 ? __builtin_ctz(per_head) : -1;
  auto unit_row = [&](int u) {
    const int head = shift >= 0 ? u >> shift : u / per_head;
    return u < turned ? head * hd + (u - head * per_head) * 4 : u * 8;
  };
  auto unit_step = [&](int u) { return u < turned ? half : 4; };
  f32x4 acc[NI][MJ];
  spread_sums<NI, MJ, WN, WM, WK, NBUF>(acc, lds, A, lda, W, K, 0, K / S::BK, mine.m0, mine.live, mine.own, [&](int r) {
    const int u = mine.u0 + r / 8;
    return unit_row(u) + (r & 3) + ((r & 4) ? unit_step(u) : 0);
  });
  constexpr int BLOCKS = NI * MJ / WK + NI * MJ % WK, TOGETHER = BLOCKS < 4 ? BLOCKS : 4;      // of a wavefront; whose operands are asked for at once
  const bf16_t* biases = x.bias ? x.bias : W;
#pragma unroll
  for (int b0 = 0; b0 < BLOCKS; b0 += TOGETHER) {
    float2 cs[TOGETHER], sn[TOGETHER];
    uint32_t blo[TOGETHER], bhi[TOGETHER];           // two columns' biases as they lie in memory
#pragma unroll
    for (int y = 0; y < TOGETHER; ++y) {
      const int t = min(WK * (b0 + y) + (WK == 2 ? wk : 0), NI * MJ - 1), i = t / MJ;     // (where none is left: dropped below)
      const int u = min(mine.u0 + (wn * NI + i) * 2 + (g >> 1), mine.u0 + mine.own - 1);
      const int n = unit_row(u) + 2 * (g & 1), step = unit_step(u);
      int p = pos[0];
#pragma unroll
      for (int j = 1; j < MJ; ++j) p = t % MJ == j ? pos[j] : p;
      const int64_t at = u < turned ? (int64_t)p * half + (shift >= 0 ? n & (hd - 1) : n % hd) : 0;
      cs[y] = *reinterpret_cast<const float2*>(x.cos_t + at);
      sn[y] = *reinterpret_cast<const float2*>(x.sin_t + at);
      blo[y] = *reinterpret_cast<const uint32_t*>(biases + n);
      bhi[y] = *reinterpret_cast<const uint32_t*>(biases + n + step);
    }
#pragma unroll
    for (int y = 0; y < TOGETHER; ++y)
#pragma unroll
      for (int k = 0; k < WK; ++k) {                 // block t of the two that y stands for is the wavefront's with wk = k
        const int t = WK * (b0 + y) + k;
        if (t >= NI * MJ || (WK == 2 && k != wk)) continue;
        const int i = t / MJ, row = (wm * MJ + t % MJ) * 16 + c, m = mine.m0 + row;
        const int lu = (wn * NI + i) * 2 + (g >> 1), u = mine.u0 + lu;
        const SpreadPairs v(acc[i][t % MJ]);
        if (row >= mine.live || lu >= mine.own) continue;
        const int n = unit_row(u) + 2 * (g & 1), step = unit_step(u);          // columns n, n + 1 and their partners
        float lo[2] = {v.first[0], v.first[1]}, hi[2] = {v.second[0], v.second[1]};
        if (x.bias) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            lo[e] += __uint_as_float(e ? blo[y] & 0xffff0000u : blo[y] << 16);
            hi[e] += __uint_as_float(e ? bhi[y] & 0xffff0000u : bhi[y] << 16);
          }
        }
        const int64_t slot = x.write_kv && u >= x.nh * per_head ? slots[t % MJ] : -1;
        int64_t page = 0, off = 0;
        if (slot >= 0) slot_page(slot, x.page_size, page, off);
        if (u < turned) {
          const int j = shift >= 0 ? n & (hd - 1) : n % hd, head = shift >= 0 ? n >> (shift + 3) : n / hd;
          const float c0 = cs[y].x, c1 = cs[y].y, s0 = sn[y].x, s1 = sn[y].y;
          const uint32_t a = gt_round2(lo[0] * c0 - hi[0] * s0, lo[1] * c1 - hi[1] * s1), b = gt_round2(lo[0] * s0 + hi[0] * c0, lo[1] * s1 + hi[1] * c1);
          bf16_t* o = nullptr;
          if (head < x.nh) o = q_out + ((int64_t)m * x.nh + head) * hd + j;
          else if (slot >= 0) o = x.k_pages + ((page * x.nkv + (head - x.nh)) * x.page_size + off) * hd + j;
          if (o) {
            *reinterpret_cast<uint32_t*>(o) = a;
            *reinterpret_cast<uint32_t*>(o + half) = b;
          }
        } else if (slot >= 0) {
          const int d = n - turned_heads * hd;                         // column of the v heads
          bf16_t* o = x.v_pages + (page * x.nkv * hd + d) * (int64_t)x.page_size + off;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            o[(int64_t)e * x.page_size] = f32_to_bf16(lo[e]);
            o[(int64_t)(step + e) * x.page_size] = f32_to_bf16(hi[e]);
          }
        }
      }
  }
}

// The tiles: NI, MJ, WN, WM, WK, buffers; room for 16 MJ WM rows of A and 16 NI WN of W.  The first ten serve the gated product, all of
// them the others, whose columns are few.
#define GA_SPREAD_GATED(X)                                                                                             \
  X(0, 5, 1, 1, 4, 2, 4) X(1, 5, 2, 1, 4, 2, 3) X(2, 5, 1, 2, 4, 1, 5) X(3, 5, 2, 2, 4, 1, 4) X(4, 5, 3, 2, 4, 1, 3) \
  X(5, 5, 4, 2, 4, 1, 3) X(6, 4, 1, 2, 4, 1, 6) X(7, 4, 2, 2, 4, 1, 5) X(8, 4, 3, 2, 4, 1, 4) X(9, 4, 4, 2, 4, 1, 3)
#define GA_SPREAD_NARROW(X) X(10, 1, 1, 1, 4, 2, 7) X(11, 2, 1, 1, 4, 2, 6) X(12, 2, 2, 1, 4, 2, 4) X(13, 3, 1, 1, 4, 2, 5) X(14, 3, 2, 1, 4, 2, 3)

// Whether a tile holds what a launch deals out; the rows of A of a row tile
template <int NI, int MJ, int WN, int WM, int WK, int NBUF>
static bool spread_fits(int M, int units, int slabs_of_64, int m_tiles, int groups, int& tile_rows) {
  using S = SpreadTile<NI, MJ, WN, WM, WK, NBUF>;
  tile_rows = ((M + m_tiles - 1) / m_tiles + 15) / 16 * 16;
  return slabs_of_64 % WK == 0 && tile_rows <= S::TM && (int64_t)(m_tiles - 1) * tile_rows < M && groups <= units &&
         (units + groups - 1) / groups <= 2 * S::NB;
}
template <typename Kernel>
static int spread_room(Kernel kernel, int bytes) {
  return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);      // the current device's
}
static int spread_check(int M, int m_tiles, int groups) {
  return m_tiles < 1 || m_tiles > M || groups < 1 || (int64_t)m_tiles * groups > 1 << 20 ? -1 : 0;
}
#define GA_SPREAD_GRID(parts) dim3((unsigned)((m_tiles * groups + 7) / 8 * 8), parts)

// tiling: which tiles, rows of W x rows of A; the caller chooses by sizes and by how full they leave the chip's rounds
// (gated_tiling in kernels/ops.py, tiles_gated in parts/linear.py, the fastest and the library beside each other).  us, product and
// activation by the library's best way -> here, as replays of a graph over several layers' weights: 17,920 rows of W, K 1,536: 64 rows
// 30.6 -> 26.9, 128 rows 35.1 -> 30.2 (tiles of 128 x 256, half of them rows that do not exist, 33.5), 256 rows 43.6 -> 37.2, 384
// rows 45.9 -> 39.9; 37,888 rows, K 3,584: 128 rows 84.0 -> 79.3, 384 rows 133.9 -> 121.4, 1,000 rows 324 -> 272, 1,280 rows 386 ->
// 291, 2,048 rows 552 -> 464; 19,456 rows, K 2,560: 128 rows 46.0 -> 44.0 (128 x 256 tiles 49.1), 384 rows 64.0 -> 57.8 (all with four
// wavefronts to a tile; what eight give stands above).
// Tiles of 192 rows of W stand beside the others (6 to 8) where those leave the chip's rounds emptier (gated_wide_tiling in
// kernels/ops.py has the rule and the figures).  17 to 64 rows of up to 81,920 rows of W are dealt evenly (below), so that 0 and 6 are left to calls of up
// to 16 rows, which a step's products make with the kernel that streams the weights.
extern "C" int ga_gemm_tiles_gated(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, int M, int cols, int K, int kind,
                                   float limit, float alpha, float shift, int tiling, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = gt_check(C, A, lda, W, 2 * (int64_t)cols, M, cols, K);
  if (rc) return rc;
  if (kind < 0 || kind > 2 || ldc < cols || ldc % 8) return -1;
  const GateAct act = {kind, limit, alpha, shift};
  switch (tiling) {
    case 0: return gt_launch<2, 1, 2, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 64
    case 1: return gt_launch<2, 2, 2, 4, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 256
    case 2: return gt_launch<2, 2, 4, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 256 x 128
    case 3: return gt_launch<2, 4, 4, 2, 2, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 256 x 256
    case 4: return gt_launch<2, 2, 2, 2, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 128 x 128
    case 6: return gt_launch<6, 1, 1, 2, 4, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 64
    case 7: return gt_launch<3, 1, 2, 4, 3, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 128
    case 8: return gt_launch<3, 2, 2, 4, 2, true>(C, ldc, A, lda, W, M, cols, K, 1, act, stream);     // 192 x 256
  }
  return -6;
}

// shape: the tile, the rows of A and of W that it has room for; m_tiles row tiles of equal numbers of rows times `groups` groups of columns
// (spread_plan in kernels/ops.py chooses them, spread_is_faster in parts/linear.py where the product goes this way at all).  us of the other
// ways -> here, as replays of a graph over weights beyond the 256 MB cache: 17,920 rows of W, K 1,536: 17 rows 15.3 -> 12.5, 64 18.9 -> 13.7, 128
// 22.5 -> 16.7, 256 26.6 -> 23.7, 384 31.4 -> 28.7, 512 43.6 -> 35.2; 37,888, K 3,584: 64 rows 55.9 -> 45.3 (6.0 TB/s of weights), 128 61.3 ->
// 52.3, 192 83.7 -> 61.5, 256 84.1 -> 73.1; 9,728, K 896: 64 11.6 -> 8.1, 256 18.4 -> 11.6.  480 products of 40 sizes of W: 1.22 times as fast
// in the geometric mean.
extern "C" int ga_gemm_spread_gated(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, int M, int cols, int K, int kind,
                                    float limit, float alpha, float shift, int shape, int m_tiles, int groups, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = gt_check(C, A, lda, W, 2 * (int64_t)cols, M, cols, K);
  if (rc) return rc;
  if (kind < 0 || kind > 2 || ldc < cols || ldc % 4 || spread_check(M, m_tiles, groups)) return -1;
  const GateAct act = {kind, limit, alpha, shift};
  int tile_rows;
  switch (shape) {
#define CASE(n, ...)                                                                                                                     \
  case n: {                                                                                                                              \
    if (!spread_fits<__VA_ARGS__>(M, cols / 4, K / 64, m_tiles, groups, tile_rows)) return -7;                                           \
    constexpr int bytes = SpreadTile<__VA_ARGS__>::LDS;                                                                                  \
    constexpr bool few = SpreadTile<__VA_ARGS__>::TM == 64;                                                                              \
    const auto kernel = few && (M <= 32 || cols < 2048) ? gemm_spread_gated_kernel<few, __VA_ARGS__>                                     \
                                                        : gemm_spread_gated_kernel<false, __VA_ARGS__>;                                  \
    if (const int raised = spread_room(kernel, bytes)) return raised;                                                                    \
    hipLaunchKernelGGL(kernel, GA_SPREAD_GRID(1), dim3(64 * SpreadTile<__VA_ARGS__>::WAVES), bytes, stream, (const bf16_t*)A,            \
                       (const bf16_t*)W, lda, M, cols, K, m_tiles, tile_rows, groups, cols / 4 / groups, cols / 4 % groups, (bf16_t*)C, ldc, act); \
    return GA_CHECK_LAUNCH();                                                                                                            \
  }
    GA_SPREAD_GATED(CASE)
#undef CASE
  }
  return -6;
}

// Which shape, row tiles and groups: spread_few_columns in kernels/ops.py; how many parts, and where the other plans are the faster: spread_parts
// in parts/linear.py, with the figures.  570 products of 70 sizes of W with the norm that adds their parts, 17 to 384 rows: 1.18 times as
// fast in the geometric mean.
extern "C" int ga_gemm_spread_parts(void* C, const void* A, int64_t lda, const void* W, int M, int cols, int K, int parts, int shape,
                                    int m_tiles, int groups, hipStream_t stream) {
  if (M <= 0) return 0;
  const int rc = gt_check(C, A, lda, W, cols, M, cols, K);
  if (rc) return rc;
  if (spread_check(M, m_tiles, groups) || parts < 1 || parts > K / 64 || parts > 65535) return -1;
  const int per_part = (K / 64 + parts - 1) / parts;                   // slabs of 64
  if ((parts - 1) * per_part >= K / 64) return -4;       // a part without a slab
  int tile_rows;
  switch (shape) {
#define CASE(n, ...)                                                                                                                     \
  case n: {                                                                                                                              \
    constexpr int slab = SpreadTile<__VA_ARGS__>::BK / 64, bytes = SpreadTile<__VA_ARGS__>::LDS;                                         \
    if (!spread_fits<__VA_ARGS__>(M, cols / 8, K / 64, m_tiles, groups, tile_rows) || (parts > 1 && per_part % slab)) return -7;         \
    if (const int raised = spread_room(gemm_spread_parts_kernel<__VA_ARGS__>, bytes)) return raised;                                     \
    hipLaunchKernelGGL((gemm_spread_parts_kernel<__VA_ARGS__>), GA_SPREAD_GRID(parts), dim3(64 * SpreadTile<__VA_ARGS__>::WAVES), bytes, \
                       stream, (const bf16_t*)A, (const bf16_t*)W, (int)lda, M, cols, K, m_tiles, tile_rows, groups, cols / 8 / groups,  \
                       cols / 8 % groups, per_part / slab, (float*)C);                                                                   \
    return GA_CHECK_LAUNCH();                                                                                                            \
  }
    GA_SPREAD_GATED(CASE) GA_SPREAD_NARROW(CASE)
#undef CASE
  }
  return -6;
}

// us of the fused kernel for few rows (up to 64 rows), or the library and the rotation -> here: 2,048 columns, K 1,536: 17 rows 6.2 -> 6.0, 64
// 8.4 -> 6.8, 128 12.4 -> 7.7, 256 13.5 -> 9.3, 512 14.6 -> 12.9; 4,608, K 3,584: 64 rows 19.2 -> 14.3, 256 40.6 -> 23.4, 512 37.5 -> 32.0; 1,152, K
// 896: 128 rows 10.5 -> 5.5; 10,240, K 8,192: 65 rows 81.9 -> 43.7; of 72 the slowest 2 % behind (6,144, K 4,096 at 512 rows 44.2 -> 45.0).
// W [(nh + 2 nkv) hd, K], bias [the same] or null, hd a multiple of 8 that is rotated whole; the rest as ga_qkv_rope_skinny
extern "C" int ga_qkv_spread(void* q_out, const void* A, int64_t lda, const void* W, const void* bias, const void* positions,
                             const void* cos_t, const void* sin_t, const void* slot_mapping, void* k_pages, void* v_pages, int M, int K,
                             int nh, int nkv, int hd, int page_size, int write_kv, int shape, int m_tiles, int groups,
                             hipStream_t stream) {
  if (M <= 0) return 0;
  if (nh <= 0 || nkv <= 0 || hd <= 0 || hd % 8 || page_size <= 0 || (write_kv && (!slot_mapping || !k_pages || !v_pages))) return -1;
  const int64_t cols = ((int64_t)nh + 2 * nkv) * hd;
  if (cols > 1 << 24) return -1;
  const int rc = gt_check(q_out, A, lda, W, cols, M, (int)cols, K);
  if (rc) return rc;
  if (spread_check(M, m_tiles, groups)) return -1;
  const SpreadQkv x = {(const bf16_t*)bias, (const int32_t*)positions, (const float*)cos_t, (const float*)sin_t, (const int64_t*)slot_mapping,
                       (bf16_t*)k_pages, (bf16_t*)v_pages, nh, nkv, page_size, write_kv};
  int tile_rows;
  switch (shape) {
#define CASE(n, ...)                                                                                                                     \
  case n: {                                                                                                                              \
    if (!spread_fits<__VA_ARGS__>(M, (int)(cols / 8), K / 64, m_tiles, groups, tile_rows)) return -7;                                    \
    constexpr int bytes = SpreadTile<__VA_ARGS__>::LDS;                                                                                  \
    if (const int raised = spread_room(gemm_spread_qkv_kernel<__VA_ARGS__>, bytes)) return raised;                                       \
    hipLaunchKernelGGL((gemm_spread_qkv_kernel<__VA_ARGS__>), GA_SPREAD_GRID(1), dim3(64 * SpreadTile<__VA_ARGS__>::WAVES), bytes,       \
                       stream, (const bf16_t*)A, (const bf16_t*)W, (int)lda, K, M, m_tiles, tile_rows, groups, (int)(cols / 8) / groups, \
                       (int)(cols / 8) % groups, hd, nh + nkv, (bf16_t*)q_out, x);                                                       \
    return GA_CHECK_LAUNCH();                                                                                                            \
  }
    GA_SPREAD_GATED(CASE) GA_SPREAD_NARROW(CASE)
#undef CASE
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
