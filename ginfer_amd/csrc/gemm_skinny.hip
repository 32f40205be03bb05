// C[M, N] = A[M, K] . W[N, K]^T (+ bias) for FEW rows (M <= 64): the decode step's products, where
// every weight is read once and the time is the weight's way from HBM.  bfloat16 operands, 32-bit
// accumulation on the matrix cores, bias added in 32-bit before the one rounding (the reference's
// small-batch kernel is ginfer/core/op/kernels/cuda/gemv_kernel.cu:13-58: one block per output column,
// scalar FMAs; its engine never reaches it, ginfer/core/op/matmul_op.cc:47-50).
//
// A workgroup of 8 wavefronts owns NT*16 rows of W (output columns) and all M rows of A; the wavefronts
// split K and add their parts up through LDS in a fixed order.  v_mfma_f32_16x16x32_bf16 with W as the
// first operand: lane l supplies W[n0 + l%16][k-slots] and A[l%16][k-slots] and receives
// D[n = (l/16)*4+i][m = l%16].  Both operands come from global memory in 16-byte loads, 8 lanes to a row, and turn into
// that layout in the wavefront's own piece of LDS (SkinnyTrip).
#include "common.h"
#include <type_traits>
#include "ginfer_amd.h"   // the entry points below are checked against their declarations

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define SK_WAVES 8
#define GA_FOLD_TARGET 256       // the chip's compute units
#define SK_THREADS (SK_WAVES * 64)


// A root-mean-square norm folded into the two products around it (ginfer/core/op/kernels/cuda/rmsnorm_kernel.cu:27-66
// is the norm itself: y = x * g / sqrtf(sum(x^2) / width + eps)).  The product BEFORE the norm adds its result
// to the 32-bit residual stream, writes h * g rounded once, and one partial sum of h^2 per row and workgroup
// (NormOut).  The product AFTER it runs on h * g and multiplies every sum by 1 / sqrtf(sum / width + eps), the
// partial sums added in a fixed order (NormIn): the same value as normalising first, without the norm's own
// pass over memory.  At most 16 rows.
struct NormIn {
  const float* sumsq;      // [M][parts], or null: the rows are used as they are
  int parts;
  float inv_width, eps;
};
struct NormOut {
  float* residual;         // [M][N] (row stride ldr), read and written; null: a plain product
  int64_t ldr;
  const void* gain;        // [N], bfloat16 or float
  int gain_f32;
  bf16_t* scaled;          // [M][N] (row stride lds): (residual + product) * gain
  int64_t lds;
  float* sumsq;            // [M][gridDim.x]
};
#define NORM_IN_MAX_PARTS 512

// Partial sums of the rows' squares.  With up to 8 rows wavefront w takes row w, else rows 2w and 2w + 1.  Four
// values per lane are asked for at the start of a kernel, so that they arrive while the weights stream (more
// would cost the registers that the weights' loads need): 256 parts of a row, or 128 of each of two; any
// further ones are fetched at the end.
struct NormInLoads {
  float v[4];
  // (no branch stands around a load: what does not exist reads a number of `anything`, or another part, and drops it)
  __device__ __forceinline__ void load(const NormIn& in, const void* anything, int M, int wave, int lane) {
    const float* from = in.sumsq ? in.sumsq : reinterpret_cast<const float*>(anything);
    const int parts = in.sumsq ? in.parts : 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = M <= 8 ? wave : wave * 2 + (j >> 1);
      const int p = M <= 8 ? lane + 64 * j : lane + 64 * (j & 1);
      v[j] = from[(in.sumsq && m < M ? m * parts : 0) + min(p, parts - 1)];
    }
  }
  // the rows' factors; rstd: 16 floats of LDS, a barrier before they are read.  Lane l adds parts l, l + 64, ...
  // in ascending order, then the lanes add up in a butterfly: the order never depends on the data.
  __device__ __forceinline__ void finish(const NormIn& in, float* rstd, int M, int wave, int lane) const {
    if (!in.sumsq) return;
    const int rows = M <= 8 ? 1 : 2, early = M <= 8 ? 4 : 2;
    for (int i = 0; i < rows; ++i) {
      const int m = M <= 8 ? wave : wave * 2 + i;
      float x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = m < M && lane + 64 * (M <= 8 ? j : j & 1) < in.parts ? v[j] : 0.f;
      float t = M <= 8 ? (x[0] + x[1]) + (x[2] + x[3]) : (i == 0 ? x[0] + x[1] : x[2] + x[3]);
      if (m < M)
        for (int p = lane + 64 * early; p < in.parts; p += 64) t += in.sumsq[(int64_t)m * in.parts + p];
      t = wave_sum(t);
      if (lane == 0 && m < 16) rstd[m] = 1.0f / sqrtf(t * in.inv_width + in.eps);
    }
  }
};

// The wavefront's share of the sum over k: UNROLL steps of 64 elements per trip, all loads of a trip issued
// before its products.  The trips run over [0, kend), the same for every lane; a lane's own pointers may be
// shifted (a packed tile, below) and its own range ends at ke: the guard on every 8-element piece makes the
// tail safe (a piece past the end is zeros and touches no memory).  The terms are added in ascending k.
//
// A load brings 8 rows of an operand's tile of 16, 128 bytes of each: lane l brings piece l % 8 of row l / 8.  The matrix cores
// want row l % 16 in lane l, but neighbouring lanes in different rows cost the address unit a cycle a lane, 16 bytes a cycle and
// compute unit, measured from L2 and L1 alike, where 8 lanes to 128 bytes get 56: that rate, of weights and rows of A together, was
// what these products waited for wherever A is not small beside the weights.  So every tile goes through LDS, a wavefront's own
// 2 KB, two of them in turn: written and read by one wavefront, in order, without a barrier; the sums are the same, in the
// same order.  us as replays of a graph over weights beyond the 256 MB cache (0.6 GB; layers that stay in it hide a trip to memory),
// before -> after, at 1, 8 and 16 rows: 1,536 columns of a K of 8,960 with the folded norm 9.1 -> 9.1, 12.4 -> 9.8, 16.7 -> 13.5; 3,584 of
// 18,944 29.2 -> 28.9, 36.0 -> 27.5, 41.1 -> 31.1; 1,536 of 1,536 4.9 -> 4.9, 5.4 -> 5.1, 6.2 -> 5.7; q|k|v of 28 heads and K 3,584
// 14.7 -> 11.4, 17.8 -> 12.4, 16.7 -> 12.1, at 64 rows 28.8 -> 19.2; of 12 heads and K 1,536 5.4 -> 5.4, 6.0 -> 5.7, 7.4 -> 6.3.  With one row,
// whose tiles of A were nearly free, some are behind by up to 5 %: 1,536 of 4,096 6.1 -> 6.4, 1,024 of 3,072 5.2 -> 5.5, 896 of 4,864 6.3 -> 6.5.
// UNROLL is 1 wherever several workgroups share a compute unit: their wavefronts cover each other's trips, and longer trips were up
// to three times slower, spread over fewer of them.  A workgroup alone on its unit asks for more at once (ga_skinny_trip); two trips
// under way at once were slower than one everywhere.
// Loads go through buffer descriptors (a base for all lanes, 32-bit offsets of each): a lane without a row, or past its end of K, names an
// offset beyond the buffer and gets zeros without touching memory, so that no load stands behind a branch and none waits for another.
#define SK_NOTHING 0x80000000u
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sk_buffer(const bf16_t* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), 0, 0x7fffffff, 0x00027000);
}
template <int NT, int MB, int MATS = 1>    // MATS: bases of W, each with NT / MATS tiles
struct SkinnySource {
  __amdgpu_buffer_rsrc_t w[MATS], a[MB];
  uint32_t wat[NT][2], aat[MB][2];         // bytes to the lane's piece of its rows of each tile, l / 8 and 8 more
  int ke[2], kend;
};
// 16 rows of 8 pieces of 16 bytes; piece p of row r lies at p ^ (r / 2): 16 lanes that read one piece of 16 rows meet all banks once
#define SK_TILE_PIECES 128
template <int NT, int MB, int UNROLL>
struct SkinnyTrip {
  u32x4 a[UNROLL][NT][2], b[UNROLL][MB][2];
  template <int MATS>
  __device__ __forceinline__ void load(const SkinnySource<NT, MB, MATS>& src, int k, int lane) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int from = (k + u * 64) * 2;
        const bool ok = k + u * 64 + (lane & 7) * 8 < src.ke[j];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          a[u][nt][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src.w[nt / (NT / MATS)], ok ? src.wat[nt][j] : SK_NOTHING, from, 0));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          b[u][mb][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src.a[mb], ok ? src.aat[mb][j] : SK_NOTHING, from, 0));
      }
  }
  __device__ __forceinline__ void multiply(f32x4 (&acc)[NT][MB], u32x4* area, int lane) const {
    const int row = lane >> 3, piece = lane & 7, m = lane & 15, g = lane >> 4;
    u32x4* const put[2] = {area + row * 8 + (piece ^ (row >> 1)), area + (row + 8) * 8 + (piece ^ ((row + 8) >> 1))};
    const u32x4* const get[2] = {area + m * 8 + (g ^ (m >> 1)), area + m * 8 + ((4 + g) ^ (m >> 1))};
    auto through = [&](const u32x4 (&v)[2], bf16x8 (&out)[2], int slot) {
#pragma unroll
      for (int j = 0; j < 2; ++j) put[j][slot * SK_TILE_PIECES] = v[j];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int h = 0; h < 2; ++h) out[h] = __builtin_bit_cast(bf16x8, get[h][slot * SK_TILE_PIECES]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      bf16x8 y[MB][2];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) through(b[u][mb], y[mb], (u * (NT + MB) + mb) & 1);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        bf16x8 x[2];
        through(a[u][nt], x, (u * (NT + MB) + MB + nt) & 1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) acc[nt][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[h], y[mb][h], acc[nt][mb], 0, 0, 0);
      }
    }
  }
};

// beside(): asks for what the epilogue needs from memory, behind the first trip's loads: nothing may come between a kernel's
// start and those.  (Nothing in it may use what it loads unless that has to be; conversions belong to the epilogue.)  us as replays of a
// graph over weights beyond the 256 MB cache at 1, 8 and 16 rows, before (the norm's and the epilogue's operands first and converted, loads
// behind branches, K dealt out in 64-bit divisions, arguments from memory) -> after: with the folded norm 1,536 columns of 1,536 4.8, 5.0, 5.6 ->
// 4.0, 4.2, 4.7; of 8,960 9.7, 11.1, 14.0 -> 8.4, 10.0, 12.5; 3,584 of 3,584 8.7, 8.7, 9.9 -> 8.4, 8.3, 9.3; of 18,944 28.8, 29.0, 33.3 -> 27.7, 28.3,
// 32.7; gated 17,920 x 1,536 13.9, 13.7, 15.3 -> 12.7, 13.1, 14.9; 37,888 x 3,584 51.1, 51.7, 54.1 -> 50.7, 50.8, 53.6; q|k|v of 2,048 columns of
// 1,536 5.3, 5.5, 6.1 -> 4.9, 5.0, 5.8; the head, 151,936 x 1,536 80.5, 88.6 -> 79.9, 89.0 (figures below that name the same sizes are from before).
template <int NT, int MB, int UNROLL, int MATS, typename Beside>
__device__ __forceinline__ void skinny_accumulate(f32x4 (&acc)[NT][MB], const SkinnySource<NT, MB, MATS>& src, u32x4* area, int lane,
                                                  Beside beside) {
  {
    SkinnyTrip<NT, MB, UNROLL> trip;
    trip.load(src, 0, lane);
    __builtin_amdgcn_sched_barrier(0);
    beside();
    __builtin_amdgcn_sched_barrier(0);         // no load moves behind a product
    trip.multiply(acc, area, lane);
  }
  for (int k = 64 * UNROLL; k < src.kend; k += 64 * UNROLL) {
    SkinnyTrip<NT, MB, UNROLL> trip;
    trip.load(src, k, lane);
    __builtin_amdgcn_sched_barrier(0);
    trip.multiply(acc, area, lane);
  }
}
// a wavefront's LDS: two tiles under way, and in their place, at the end, its sums: [NT * 16][MB * 16 + 1]
template <int NT, int MB>
struct SkinnyArea {
  static constexpr int SUMS = NT * 16 * (MB * 16 + 1) * 4, TILES = 2 * SK_TILE_PIECES * 16;
  static constexpr int BYTES = ((SUMS > TILES ? SUMS : TILES) + 15) / 16 * 16;
};

// A PACKED tile (PACK == 2, at most 8 rows of A): with so few rows half of the matrix core's 16 x 16 tile
// would hold nothing, so the tile takes 8 rows of W twice, for the two halves of the wavefront's K range:
// tile row q * 8 + c is row c of W over half q, tile column q * 8 + m is row m of A over half q, and
// C[m][c] = D[c][m] + D[8 + c][8 + m] (the other entries mix the halves and are dropped).  A workgroup then
// owns half as many columns over the same K: twice the workgroups stream the weights, with every lane still
// loading, which is what a product with few columns lacks to fill the chip.
template <int PACK>
struct Packed {
  static constexpr int CP = 16 / PACK;     // columns of W in a tile = most rows of A
  // row r of a tile: its column of W (and row of A); its half of K is r / CP
  static __device__ __forceinline__ int col(int r) { return r % CP; }
};

// How K is dealt out: in steps of 64 elements, as evenly as whole steps allow, to `units` consumers (the
// wavefronts that split K, over all workgroups of a column, times the halves of a packed tile).  Consumer u
// takes the steps [u * steps / units, (u + 1) * steps / units).  A lane works in its own coordinates, starting
// at 0 at its first element: `shift` is where that lies, `ke` its own end, `kend` the end of the wavefront's
// trips (the longer of its halves).
template <int PACK>
struct KRange {
  int shift[2], ke[2], kend;               // of tile rows 0 to 7 and 8 to 15
  // units: PER_PART (a power of two) times `parts`; in 32 bits, which the launchers see to (in 64 the divisions were some 400
  // instructions in front of the first load)
  template <int PER_PART>
  static __device__ __forceinline__ int first_step(int unit, int steps, int parts) {
    const uint32_t x = (uint32_t)(unit * steps) / PER_PART;
    return (int)(parts == 1 ? x : x / (uint32_t)parts);
  }
  template <int PER_PART>
  __device__ __forceinline__ KRange(int first_unit, int steps, int parts, int K, std::integral_constant<int, PER_PART>) {
    int longest = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int q = PACK == 2 ? j : 0;
      const int b = first_step<PER_PART>(first_unit + q, steps, parts), e = first_step<PER_PART>(first_unit + q + 1, steps, parts);
      longest = e - b > longest ? e - b : longest;
      shift[j] = b * 64;
      ke[j] = (e * 64 < K ? e * 64 : K) - b * 64;
    }
    kend = longest * 64;
  }
};

// NT: tiles of W per wavefront; MB: 16-row blocks of A; KS: wavefronts of a workgroup that split K
// for the same rows (the workgroup's SK_WAVES / KS groups own different rows of W).  The grid's y
// dimension splits K further: then every workgroup writes its part in 32-bit to P[y][M][N] and the
// consumer adds the parts in order (the bias rides on part 0).
// GATED (NT == 2): W holds two stacked matrices of N rows each (gate over up); the wavefront's two tiles
// are rows n0.. of the gate and the same rows of the up matrix, and the epilogue writes
// silu(gate) * up = (g * (1 / (1 + exp(-g)))) * u (ginfer/core/op/kernels/cuda/swiglu_kernel.cu:24-27) for N
// columns: the activation of the feed-forward without a pass over memory of its own.
// The gate of a gated product: out = g * sigmoid(alpha g) * (u + shift) with g = min(gate, limit) and u = clamp(up, -limit,
// limit).  limit = infinity, alpha = 1, shift = 0 is SiLU(gate) * up, bit for bit what stood here before the bounds; alpha =
// infinity stands for the sigmoid's limit, a step at zero: relu(g) * (u + shift).  (From 17 rows on the product over tiles may
// stand here, whose sigmoid is the hardware's exp2 and reciprocal: csrc/gemm_tiles.hip has the two's errors.)
struct GateAct {
  float limit, alpha, shift;
};
__device__ __forceinline__ float gate_act(float v, float u, const GateAct act) {
  v = fminf(v, act.limit);
  u = fminf(fmaxf(u, -act.limit), act.limit);
  if (isinf(act.alpha)) return (v > 0.f ? v : 0.f) * (u + act.shift);     // the sigmoid's limit, a step: relu(g)
  return (v * (1.0f / (1.0f + expf(-(act.alpha * v))))) * (u + act.shift);
}

template <int NT, int MB, int KS, typename TC, bool GATED, int PACK, int UNROLL = 1>
__global__ __launch_bounds__(SK_THREADS) void gemm_skinny_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                 int64_t lda, int M, int N, int K, int parts, int fold_cols,
                                                                 TC* __restrict__ C, int64_t ldc, const bf16_t* __restrict__ bias,
                                                                 NormIn norm_in, NormOut norm_out, GateAct act) {
  static_assert(PACK == 1 || MB == 1, "a packed tile holds at most 8 rows of A");
  using Area = SkinnyArea<NT, MB>;
  __shared__ __attribute__((aligned(16))) unsigned char area[SK_WAVES][Area::BYTES];
  __shared__ float rstd[16];
  using P = Packed<PACK>;
  constexpr int CP = P::CP;
  constexpr int GROUPS = SK_WAVES / KS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  auto red = [&](int w, int n, int m) -> float& { return reinterpret_cast<float*>(area[w])[n * (MB * 16 + 1) + m]; };
  const int grp = wave / KS, ks = wave % KS;
  constexpr int NCOL = GATED ? CP : NT * CP;       // output columns of a group
  // A product that folds the norm after it owns `fold_cols` (<= CP) columns per workgroup: as many as spread the
  // columns over all compute units (every workgroup reads all rows of A, so fewer, larger workgroups cost more
  // than the empty tile rows of more, smaller ones).
  constexpr bool MAY_FUSE = !GATED && NT == 1 && KS == SK_WAVES && MB == 1;
  const bool fuse_out = MAY_FUSE && fold_cols > 0;
  const int my_cols = fuse_out ? fold_cols : NCOL;
  const int n0 = fuse_out ? blockIdx.x * fold_cols : (blockIdx.x * GROUPS + grp) * NCOL;
  const KRange<PACK> kr((blockIdx.y * KS + ks) * PACK, (K + 63) / 64, parts, K, std::integral_constant<int, KS * PACK>());
  SkinnySource<NT, MB, GATED ? 2 : 1> src;
  src.kend = kr.kend;
  src.w[0] = sk_buffer(W + (int64_t)n0 * K);
  if constexpr (GATED) src.w[1] = sk_buffer(W + ((int64_t)N + n0) * K);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) src.a[mb] = sk_buffer(A + mb * 16 * lda);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tr = (lane >> 3) + 8 * j;            // the row of a tile that the lane brings a piece of
    const uint32_t from = (kr.shift[j] + (lane & 7) * 8) * 2;
    src.ke[j] = kr.ke[j];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = P::col(tr) + (GATED ? 0 : nt * CP);
      src.wat[nt][j] = n0 + n < N && (!fuse_out || n < my_cols) ? (uint32_t)n * (uint32_t)K * 2 + from : SK_NOTHING;
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      src.aat[mb][j] = mb * 16 + P::col(tr) < M ? (uint32_t)P::col(tr) * (uint32_t)lda * 2 + from : SK_NOTHING;
  }
  f32x4 acc[NT][MB];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nt][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  NormInLoads in_loads;
  float out_res = 0.f;                       // NormOut: thread t holds row t / CP, column t % CP of the workgroup
  uint32_t out_gain[2] = {0, 0};             // its two halves, or a bfloat16 twice
  skinny_accumulate<NT, MB, UNROLL>(acc, src, reinterpret_cast<u32x4*>(area[wave]), lane, [&]() {
    if constexpr (MB == 1) in_loads.load(norm_in, A, M, wave, lane);
    if constexpr (MAY_FUSE) {                // (threads without a column, and products without a norm, read something else)
      const int m = min((int)threadIdx.x / CP, M - 1), n = min(n0 + (int)threadIdx.x % CP, N - 1), wide = norm_out.gain_f32 ? 2 : 1;
      const float* res = fuse_out ? norm_out.residual : reinterpret_cast<const float*>(A);
      const bf16_t* gain = fuse_out ? reinterpret_cast<const bf16_t*>(norm_out.gain) : A;
      out_res = res[fuse_out ? (int64_t)m * norm_out.ldr + n : 0];
      out_gain[0] = gain[fuse_out ? n * wide : 0];
      out_gain[1] = gain[fuse_out ? n * wide + wide - 1 : 0];
    }
  });
  if (MB == 1) in_loads.finish(norm_in, rstd, M, wave, lane);
  // the KS parts of a group meet in LDS and are added in wavefront order, the halves of a packed tile in theirs
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i) red(wave, nt * 16 + g * 4 + i, mb * 16 + r) = acc[nt][mb][i];
  __syncthreads();
  const bool scale_rows = MB == 1 && norm_in.sumsq != nullptr;
  // element (column nl of tile t, row m) of group gi, summed over its wavefronts and halves
  auto total = [&](int gi, int t, int nl, int m) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w)
#pragma unroll
      for (int q = 0; q < PACK; ++q) v += red(gi * KS + w, t * 16 + q * CP + nl, (m / CP) * 16 + q * CP + m % CP);
    return v;
  };
  if (fuse_out) {
    // CP columns of up to CP rows: the threads of a row are CP neighbouring lanes, which add up their squares
    if (threadIdx.x >= CP * CP) return;
    const int nl = threadIdx.x % CP, m = threadIdx.x / CP, n = n0 + nl;
    const bool ok = m < M && n < N && nl < my_cols;
    float h = 0.f;
    if (ok) {
      float v = total(0, 0, nl, m);
      if (scale_rows) v *= rstd[m];
      if (bias) v += bf16_to_f32(bias[n]);
      h = out_res + v;
      norm_out.residual[(int64_t)m * norm_out.ldr + n] = h;
      norm_out.scaled[(int64_t)m * norm_out.lds + n] = f32_to_bf16(h * __uint_as_float(out_gain[1] << 16 | (norm_out.gain_f32 ? out_gain[0] : 0)));
    }
    float sq = h * h;
#pragma unroll
    for (int o = CP / 2; o > 0; o >>= 1) sq += __shfl_xor(sq, o, WAVE);
    if (nl == 0 && m < M) norm_out.sumsq[(int64_t)m * gridDim.x + blockIdx.x] = sq;
    return;
  }
  const bool partial = parts > 1;
  float* Pp = reinterpret_cast<float*>(C) + (int64_t)blockIdx.y * M * N;      // parts are [y][M][N], dense
  constexpr int MROWS = PACK == 1 ? MB * 16 : CP;
  for (int idx = threadIdx.x; idx < GROUPS * NCOL * MROWS; idx += SK_THREADS) {
    const int nl = idx % NCOL, rest = idx / NCOL;
    const int gi = rest % GROUPS, m = rest / GROUPS;
    const int n = (blockIdx.x * GROUPS + gi) * NCOL + nl;
    if (m >= M || n >= N) continue;
    float v = GATED ? total(gi, 0, nl, m) : total(gi, nl / CP, nl % CP, m);
    if (scale_rows) v *= rstd[m];
    if (GATED) {
      float u = total(gi, 1, nl, m);
      if (scale_rows) u *= rstd[m];
      v = gate_act(v, u, act);
    }
    if (bias && blockIdx.y == 0) v += bf16_to_f32(bias[n]);
    if (partial) Pp[(int64_t)m * N + n] = v;
    else Num<TC>::st(C + (int64_t)m * ldc + n, v);
  }
}

// The gated product of up to 16 rows, dealt EVENLY to the compute units.  A workgroup of the kernel above owns 16
// columns, whatever their number: the 8,960 columns of a 1.5B model make 560 workgroups for 256 compute units, and a
// unit that gets three of them streams half as much again as one that gets two.  Here the grid is a multiple of the
// number of compute units and workgroup b owns the columns [b N / G, (b + 1) N / G), up to NT tiles of 16 of the gate
// and as many of the up matrix: every unit streams the same bytes.  K is dealt to the 8 wavefronts and their parts are
// added exactly as above, so the results are the same bits.  How many columns a workgroup should own is a trade: every
// workgroup reads all rows of A (as much as M / 2 of its columns' weights), while more, smaller workgroups keep more
// loads on their way; the launcher's rule states what was measured.
// The same dealing serves a plain product of many columns (the head): TILES tiles of 16 columns of W a workgroup, the
// bias added to the sums.  GATED: the first half of the tiles is the gate's, the second the up matrix's.
template <int TILES, typename TC, bool GATED>
__global__ __launch_bounds__(SK_THREADS) void gemm_even_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                               int64_t lda, int M, int N, int K, int each, int rest,
                                                               int rounds, TC* __restrict__ C, int64_t ldc, const bf16_t* __restrict__ bias,
                                                               NormIn norm_in, GateAct act) {
  static_assert(!GATED || TILES % 2 == 0, "as many tiles of the gate as of the up matrix");
  constexpr int PER = GATED ? TILES / 2 : TILES;             // tiles of one matrix
  using Area = SkinnyArea<TILES, 1>;
  __shared__ __attribute__((aligned(16))) unsigned char area[SK_WAVES][Area::BYTES];
  __shared__ float rstd[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  auto red = [&](int w, int n, int m) -> float& { return reinterpret_cast<float*>(area[w])[n * 17 + m]; };
  // b N / G = b each + b rest / G, G = GA_FOLD_TARGET rounds: in 32 bits
  auto first = [&](uint32_t b) {
    const uint32_t x = b * (uint32_t)rest / GA_FOLD_TARGET;
    return (int)(b * (uint32_t)each + (rounds == 1 ? x : x / (uint32_t)rounds));
  };
  const int c0 = first(blockIdx.x), cols = first(blockIdx.x + 1) - c0;      // cols <= PER * 16 by the launcher's choice of the grid
  const KRange<1> kr(wave, (K + 63) / 64, 1, K, std::integral_constant<int, SK_WAVES>());
  SkinnySource<TILES, 1, GATED ? 2 : 1> src;
  src.kend = kr.kend;
  src.w[0] = sk_buffer(W + (int64_t)c0 * K);
  if constexpr (GATED) src.w[1] = sk_buffer(W + ((int64_t)N + c0) * K);
  src.a[0] = sk_buffer(A);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tr = (lane >> 3) + 8 * j;                      // the row of a tile that the lane brings a piece of
    const uint32_t from = (kr.shift[j] + (lane & 7) * 8) * 2;
    src.ke[j] = kr.ke[j];
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int cl = (t % PER) * 16 + tr;                    // its column within the workgroup's range
      src.wat[t][j] = cl < cols ? (uint32_t)cl * (uint32_t)K * 2 + from : SK_NOTHING;
    }
    src.aat[0][j] = tr < M ? (uint32_t)tr * (uint32_t)lda * 2 + from : SK_NOTHING;
  }
  f32x4 acc[TILES][1];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t][0] = f32x4{0.f, 0.f, 0.f, 0.f};
  NormInLoads in_loads;
  skinny_accumulate<TILES, 1, 1>(acc, src, reinterpret_cast<u32x4*>(area[wave]), lane, [&]() { in_loads.load(norm_in, A, M, wave, lane); });
  in_loads.finish(norm_in, rstd, M, wave, lane);
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red(wave, t * 16 + g * 4 + i, r) = acc[t][0][i];
  __syncthreads();
  const bool scale_rows = norm_in.sumsq != nullptr;
  for (int idx = threadIdx.x; idx < cols * M; idx += SK_THREADS) {
    const int cl = idx % cols, m = idx / cols;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < SK_WAVES; ++w) v += red(w, cl, m);            // in wavefront order, as in the kernel above
    if (scale_rows) v *= rstd[m];
    if (GATED) {
      float u = 0.f;
#pragma unroll
      for (int w = 0; w < SK_WAVES; ++w) u += red(w, PER * 16 + cl, m);
      if (scale_rows) u *= rstd[m];
      v = gate_act(v, u, act);
    } else if (bias) {
      v += bf16_to_f32(bias[c0 + cl]);
    }
    Num<TC>::st(C + (int64_t)m * ldc + c0 + cl, v);
  }
}

// GaSkinnyNorm, what ga_gemm_skinny takes beside the product itself, is declared in ginfer_amd.h.

// Tiles of a product of M rows when the caller leaves the choice to the library: packed where they can be and full tiles would make
// fewer than 192 workgroups.  Measured on MI355X with the folded norm, weights beyond the 256 MB cache, us at 1 and 8 rows packed and full:
// 1,536 columns of 1,536 (96 workgroups of full tiles) 4.9 and 5.1, 5.0 and 5.2; of 8,960 9.1 and 9.8, 11.7 and 12.0; 2,048 of 2,048 5.4 and
// 5.6, 5.8 and 5.9; the other way 3,584 of 3,584 (224) 8.7 and 9.6, 9.0 and 8.9, of 18,944 29.2 and 33.7, 27.6 and 27.3; 4,096 of 4,096 9.5 and
// 10.3, 9.8 and 9.9; q|k|v of 6,144 columns, K 2,048 (192) 8.4 and 8.9, 8.4 and 8.3.  The gated product was measured slower packed.
static int auto_pack(int M, int workgroups_of_full_tiles) {
  return (M <= 8 && workgroups_of_full_tiles < 192) ? 2 : 1;
}

// Columns that a workgroup of a product that folds the norm after it owns: the columns of a tile (16, or 8 when packed), or fewer
// where that spreads the product over more compute units, each of which then takes in fewer weights beside the rows of A.  Measured as
// above, us with a tile's columns -> as few as make 256 workgroups, at 1, 8 and 16 rows: 1,536 columns of 8,960 9.1 -> 9.1, 10.2 -> 9.8, 15.6 ->
// 13.5; 896 of 4,864 (112 of 8 -> 224 of 4) 6.7 -> 6.7, 7.4 -> 7.0, 11.2 -> 9.8; 2,048 of 11,008 at 16 rows 19.6 -> 17.3; 1,536 of 1,536 level,
// level, 6.3 -> 6.1.  Never more workgroups than GA_FOLD_TARGET.
// The gated product of up to 16 rows goes to the kernel that deals its columns evenly from this many (activation)
// columns on: a workgroup then has at least 8 of them.
#define GA_GATED_EVEN_MIN_COLUMNS 2048
// Its workgroups: the multiple of GA_FOLD_TARGET that comes nearest to 14 columns a workgroup, and never more than 48 (three
// tiles).  Measured on MI355X as replays of a graph that walks many layers' weights, in us, at 1, 8 and 16 rows: 8,960 x 1,536:
// 13.1, 13.3, 13.8 with 35 columns, 13.4, 13.5, 13.8 with 18, 13.0, 12.9, 13.4 with 12, 12.6, 12.9, 14.5 with 9; 11,008 x 2,048:
// 21.4, 21.1, 21.9 with 43, 20.6, 20.1, 20.8 with 22, 18.5, 18.9, 19.8 with 14; 18,944 x 3,584: 48 to 50 from 12 columns to 37, at 16
// rows 52 with 12.  Up to 4 rows no single round of workgroups with more than a tile's 16 columns, the second tile nearly empty: at 1
// and 4 rows in one round and in two, 4,864 x 896 6.8 and 6.9, 6.5 and 6.55; 5,120 x 1,536 9.4 and 9.4, 9.1 and 9.1; 5,120 x 2,048 11.4 and 11.6,
// 10.5 and 10.6; 4,608 x 4,096 17.3 and 17.4, 17.5 and 16.8; at 16 rows it is the other way, 5,120 x 1,536 9.4, 10.0.  (With operands that came straight from memory in the matrix cores' layout: 13.1, 15.9, 17.0; 18.9, 23.3, 26.7;
// 53.1, 59.9, 63.7.)
// The plain product of up to 16 rows and at least this many columns (the head) is dealt the same way, to workgroups of
// up to 6 tiles, of about 64 columns: 151,936 x 1,536 with 32-bit sums out, in us at 1, 8 and 16 rows: 85.3, 88.3, 94.2 with 85
// columns, 81.7, 88.1, 93.9 with 66, 83.2, 91.8, 100.7 with 33 (before: 88.8, 108.6, 115.6); 152,064 x 3,584: 188, 191, 196 with 66,
// 188, 197, 220 with 25 (before: 187, 235, 248).  Up to 4 rows the kernel above keeps it, its thousands of small workgroups being even
// enough by their number: at 1 and 4 rows dealt evenly -> not, 151,936 x 1,536 82.2 -> 80.4, 85.4 -> 80.2; 152,064 x 2,048 112 -> 110, 114 ->
// 111.  With a K of 3,584 or more each asks for 3 steps at a time: 152,064 x 3,584 dealt evenly 188 and 191, a step at a time 186 and 187, 3 182
// and 180; 152,064 x 8,192 424 and 431, 422 and 422, 418 and 416; 32,000 x 4,096 51.0 and 49.9, 50.1 and 48.4, 48.3 and 49.4.
#define GA_PLAIN_EVEN_MIN_COLUMNS 16384
#define GA_PLAIN_EVEN_MIN_ROWS 5
#define GA_PLAIN_TRIP_MIN_STEPS 7
static int even_workgroups(int N, int target, int most, int most_in_one_round) {
  int rounds = (N + GA_FOLD_TARGET * target / 2) / (GA_FOLD_TARGET * target);
  if (rounds < 1) rounds = 1;
  if (rounds == 1 && N > GA_FOLD_TARGET * most_in_one_round) rounds = 2;
  while ((N + GA_FOLD_TARGET * rounds - 1) / (GA_FOLD_TARGET * rounds) > most) ++rounds;
  return GA_FOLD_TARGET * rounds;
}
// Workgroups that the columns of a product of up to 16 rows are dealt evenly to; 0: the kernel above has it.
extern "C" int ga_skinny_even_workgroups(int M, int N, int gated) {
  if (gated) return N >= GA_GATED_EVEN_MIN_COLUMNS ? even_workgroups(N, 14, 48, M <= 4 ? 16 : 48) : 0;
  return M >= GA_PLAIN_EVEN_MIN_ROWS && N >= GA_PLAIN_EVEN_MIN_COLUMNS ? even_workgroups(N, 64, 96, 96) : 0;
}
static int fold_cols(int M, int N) {
  const int cp = 16 / auto_pack(M, (N + 15) / 16);
  const int full = (N + cp - 1) / cp;
  if (full >= GA_FOLD_TARGET) return cp;
  int cols = (N + GA_FOLD_TARGET - 1) / GA_FOLD_TARGET;          // as few columns as make GA_FOLD_TARGET workgroups
  return cols < 1 ? 1 : (cols > cp ? cp : cols);
}

// Partial sums a row gets from a product of M rows and N columns that feeds a norm.
extern "C" int ga_skinny_norm_parts(int M, int N) {
  const int cols = fold_cols(M, N);
  return (N + cols - 1) / cols;
}

// Steps of K in a trip of a workgroup that is alone on its compute unit, where its longest wavefront has `steps`: what it costs is a
// way to memory a trip and about as much a step, also for the steps of the last trip that lie past the end.  So all at once up to 5, in
// two trips up to 8, and 3 at a time beyond.  us with the folded norm at 1 and 8 rows, trips of 1, 2, 3, 4 and 5 steps: 2 steps (1,536
// columns of 1,536) 5.3, 4.9, 5.1, 5.3, 5.5 and 5.4, 5.1, 5.3, 5.5, 5.7; 3 (1,024 of 3,072) 6.0, 5.9, 5.5, 5.6, 5.9 and 6.2, 6.1, 5.9, 6.0, 6.2;
// 4 (1,536 of 4,096) 7.1, 6.4, 6.9, 6.4, 6.6 and 7.3, 6.7, 7.2, 6.8, 7.0; 5 (896 of 4,864) 7.6, 7.0, 6.7, 7.3, 6.5 and 7.7, 7.3, 7.0, 7.7,
// 6.9; 6 (2,048 of 6,144) 9.5, 8.6, 8.4, 8.8, 9.6 and 9.6, 8.9, 8.8, 9.3, 10.2; 7 (3,584 of 3,584) 9.8, 9.1, 9.2, 8.7, 9.1 and 9.7, 8.8, 9.2,
// 8.7, 9.3; 8 (4,096 of 4,096) 11.0, 9.8, 10.1, 9.8, 9.8 and 11.1, 9.9, 10.2, 10.0, 10.3; 9 (1,536 of 8,960) 11.5, 10.0, 9.1, 10.1, 9.2 and 11.6,
// 10.4, 9.8, 10.7, 9.9; 37 (3,584 of 18,944) 39.6, 29.2, 28.8, 28.6, 28.6 and 35.8, 28.0, 27.5, 27.9, 28.3.
extern "C" int ga_skinny_trip(int steps) { return steps <= 5 ? steps : steps <= 8 ? (steps + 1) / 2 : 3; }

// offsets inside a tile's 96 rows, and steps of K times their consumers, are 32-bit
static bool sk_too_far(int64_t K, int64_t lda, int64_t parts = 1) {
  return K >= 1 << 23 || lda >= 1 << 26 || lda < 0 || parts * 16 * ((K + 63) / 64) >= 1ll << 31;
}

// A [M, K] (row stride lda), W [N, K] contiguous, bias [N] or null.  grid_splits == 1: C [M, N] (row
// stride ldc) in bfloat16 or float.  grid_splits > 1: C is float [grid_splits][M][N], parts to be added
// by the consumer.  gated: W is [2N, K] (gate over up), C [M, N] = silu(A.gate^T) * (A.up^T), no bias, no
// grid split.  M <= 64, K a multiple of 8, rows 16-byte aligned.  nt in {1,2,4}, ks in {1,2,4,8}, pack in
// {1,2} (2: at most 8 rows); 0 lets the library choose.
static int gemm_skinny_launch(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, const void* bias,
                              int M, int N, int K, int out_f32, int nt, int ks, int grid_splits, int gated, int pack,
                              const GaSkinnyNorm* norm, GateAct act, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % 8 || lda % 8 || grid_splits < 1 || sk_too_far(K, M > 1 ? lda : 0, grid_splits)) return -1;
  if (M == 1) lda = K;                           // one row has no next one, whatever its stride says
  const int mb = (M + 15) / 16;
  NormIn norm_in = {nullptr, 0, 0.f, 0.f};
  NormOut norm_out = {nullptr, 0, nullptr, 0, nullptr, 0, nullptr};
  if (norm && norm->in_sumsq) {
    if (mb != 1 || norm->in_parts < 1 || norm->in_parts > NORM_IN_MAX_PARTS) return -5;
    norm_in = NormIn{norm->in_sumsq, norm->in_parts, norm->inv_width, norm->eps};
  }
  if (norm && norm->residual) {
    if (mb != 1 || gated || grid_splits != 1 || !norm->gain || !norm->scaled || !norm->out_sumsq) return -6;
    nt = 1;
    ks = SK_WAVES;
    pack = auto_pack(M, (N + 15) / 16);          // what ga_skinny_norm_parts promised
    norm_out = NormOut{norm->residual, norm->ldr, norm->gain, norm->gain_f32, (bf16_t*)norm->scaled, norm->lds,
                       norm->out_sumsq};
  }
  if (gated) nt = 2;
  if (nt == 0) nt = (N >= 4096 && mb > 1) ? 4 : 1;
  if (ks == 0) ks = 8;
  if ((nt != 1 && nt != 2 && nt != 4) || (ks != 1 && ks != 2 && ks != 4 && ks != 8)) return -2;
  if (nt == 4 && mb > 2 && ks < 2) return -2;      // LDS of the reduction
  if (grid_splits > 1 && !out_f32) return -3;
  if (gated && (grid_splits > 1 || bias)) return -4;
  const int groups = SK_WAVES / ks;
  if (pack == 0) pack = (grid_splits == 1 && !gated) ? auto_pack(M, (N + groups * nt * 16 - 1) / (groups * nt * 16)) : 1;
  if (pack != 1 && (pack != 2 || M > 8)) return -2;
  const bool may_be_even = gated || (grid_splits == 1 && !norm_out.residual && ks == SK_WAVES);
  const int workgroups = mb == 1 && pack == 1 && may_be_even ? ga_skinny_even_workgroups(M, N, gated) : 0;
  if (workgroups > 0 && workgroups < 1 << 16) {       // (its columns are counted in 32 bits)
    const int most = (N + workgroups - 1) / workgroups, per = (most + 15) / 16;      // tiles of one matrix
    dim3 grid(workgroups), block(SK_THREADS);
#define LAUNCH_EVEN(TILES, TC, G)                                                                              \
  hipLaunchKernelGGL((gemm_even_kernel<TILES, TC, G>), grid, block, 0, stream, (const bf16_t*)A,  \
                     (const bf16_t*)W, lda, M, N, K, N / workgroups, N % workgroups, workgroups / GA_FOLD_TARGET, (TC*)C, ldc, (const bf16_t*)bias, norm_in, act)
#define PICK_EVEN(TC)                                                                                          \
  if (gated) {                                                                                                 \
    if (per == 1) LAUNCH_EVEN(2, TC, true); else if (per == 2) LAUNCH_EVEN(4, TC, true); else LAUNCH_EVEN(6, TC, true); \
  } else {                                                                                                     \
    if (per <= 2) LAUNCH_EVEN(2, TC, false); else if (per <= 4) LAUNCH_EVEN(4, TC, false); else LAUNCH_EVEN(6, TC, false); \
  }
    if (out_f32) { PICK_EVEN(float) } else { PICK_EVEN(bf16_t) }
#undef PICK_EVEN
#undef LAUNCH_EVEN
    return GA_CHECK_LAUNCH();
  }
  const int cp = 16 / pack;
  const int ncol = gated ? cp : nt * cp;
  const int ksteps = (K + 63) / 64;
  dim3 grid((N + groups * ncol - 1) / (groups * ncol), grid_splits), block(SK_THREADS);
  int fcols = 0;
  if (norm_out.residual) {
    fcols = fold_cols(M, N);
    grid.x = (N + fcols - 1) / fcols;
  }
  // workgroups that are alone on their compute units, and the head of few rows
  const int consumers = SK_WAVES * pack * grid_splits, steps = (ksteps + consumers - 1) / consumers;
  const bool alone = (int64_t)grid.x * grid.y <= GA_FOLD_TARGET;
  const bool head = M < GA_PLAIN_EVEN_MIN_ROWS && N >= GA_PLAIN_EVEN_MIN_COLUMNS && steps >= GA_PLAIN_TRIP_MIN_STEPS && pack == 1;
  const int trip = alone ? ga_skinny_trip(steps) : head ? 3 : 1;
  if (trip > 1 && mb == 1 && nt == 1 && ks == SK_WAVES && !gated) {
#define LAUNCH_TRIP(TC, PK, UNROLL)                                                                                     \
  hipLaunchKernelGGL((gemm_skinny_kernel<1, 1, SK_WAVES, TC, false, PK, UNROLL>), grid, block, 0, stream, (const bf16_t*)A, \
                     (const bf16_t*)W, lda, M, N, K, grid_splits, fcols, (TC*)C, ldc, (const bf16_t*)bias, norm_in, norm_out, act)
#define PICK_TRIP(TC, PK)                        \
  switch (trip) {                                \
    case 2: LAUNCH_TRIP(TC, PK, 2); break;       \
    case 3: LAUNCH_TRIP(TC, PK, 3); break;       \
    case 4: LAUNCH_TRIP(TC, PK, 4); break;       \
    default: LAUNCH_TRIP(TC, PK, 5); break;      \
  }
    if (out_f32) {
      if (pack == 2) { PICK_TRIP(float, 2) } else { PICK_TRIP(float, 1) }
    } else {
      if (pack == 2) { PICK_TRIP(bf16_t, 2) } else { PICK_TRIP(bf16_t, 1) }
    }
#undef PICK_TRIP
#undef LAUNCH_TRIP
    return GA_CHECK_LAUNCH();
  }
#define LAUNCH(NT, MB, KS, TC, G, PK)                                                                     \
  hipLaunchKernelGGL((gemm_skinny_kernel<NT, MB, KS, TC, G, PK>), grid, block, 0, stream, (const bf16_t*)A, \
                     (const bf16_t*)W, lda, M, N, K, grid_splits, fcols, (TC*)C, ldc, (const bf16_t*)bias,     \
                     norm_in, norm_out, act)
#define PICK_KS(NT, MB, TC, G, PK)                                                                        \
  switch (ks) {                                                                                           \
    case 1: LAUNCH(NT, MB, 1, TC, G, PK); break;                                                          \
    case 2: LAUNCH(NT, MB, 2, TC, G, PK); break;                                                          \
    case 4: LAUNCH(NT, MB, 4, TC, G, PK); break;                                                          \
    default: LAUNCH(NT, MB, 8, TC, G, PK); break;                                                         \
  }
#define PICK_MB(NT, TC, G)                                                                                \
  switch (mb) {                                                                                           \
    case 1:                                                                                               \
      if (pack == 2) { PICK_KS(NT, 1, TC, G, 2) } else { PICK_KS(NT, 1, TC, G, 1) }                       \
      break;                                                                                              \
    case 2: PICK_KS(NT, 2, TC, G, 1) break;                                                               \
    case 3: PICK_KS(NT, 3, TC, G, 1) break;                                                               \
    default: PICK_KS(NT, 4, TC, G, 1) break;                                                              \
  }
#define PICK_NT(TC)                                                                                       \
  switch (nt) {                                                                                           \
    case 1: PICK_MB(1, TC, false) break;                                                                  \
    case 2: PICK_MB(2, TC, false) break;                                                                  \
    default: PICK_MB(4, TC, false) break;                                                                 \
  }
  if (gated) {
    if (out_f32) { PICK_MB(2, float, true) } else { PICK_MB(2, bf16_t, true) }
  } else if (out_f32) {
    PICK_NT(float)
  } else {
    PICK_NT(bf16_t)
  }
#undef PICK_NT
#undef PICK_MB
#undef PICK_KS
#undef LAUNCH
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_gemm_skinny(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, const void* bias,
                              int M, int N, int K, int out_f32, int nt, int ks, int grid_splits, int gated, int pack,
                              const GaSkinnyNorm* norm, hipStream_t stream) {
  return gemm_skinny_launch(C, ldc, A, lda, W, bias, M, N, K, out_f32, nt, ks, grid_splits, gated, pack, norm,
                            GateAct{INFINITY, 1.0f, 0.0f}, stream);
}

// The gated product with a bounded gate: C = g * sigmoid(alpha g) * (u + shift), g = min(A.gate^T, limit), u = clamp(A.up^T,
// -limit, limit); everything else as ga_gemm_skinny with gated = 1.
extern "C" int ga_gemm_skinny_bounded_gate(void* C, int64_t ldc, const void* A, int64_t lda, const void* W, int M, int N,
                                           int K, int out_f32, int ks, int pack, float limit, float alpha, float shift,
                                           const GaSkinnyNorm* norm, hipStream_t stream) {
  if (!(limit > 0.f)) return -1;
  return gemm_skinny_launch(C, ldc, A, lda, W, nullptr, M, N, K, out_f32, 2, ks, 1, 1, pack, norm, GateAct{limit, alpha, shift},
                            stream);
}

// The fused q|k|v projection of a decode step with its epilogue: bias, NeoX rotation of q and k
// (ginfer/core/op/kernels/cuda/rope_kernel.cu:83-102, on the 32-bit sums: one rounding fewer than rotating
// the rounded projection), q to its own buffer, k and v straight into the paged cache (v transposed;
// ginfer/core/op/kernels/cuda/store_kvcache_kernel.cu:19-30).  A wavefront group owns a UNIT of 2 CP output
// columns as two tiles of CP (16, or 8 when packed): for a q or k head the columns j0..j0+CP-1 and their
// rotation partners j0+half..; for a v head 2 CP consecutive columns.  head_dim a multiple of 32,
// rotary_dim == head_dim.  HALF (with more than 16 rows of A, where tiles cannot be packed): a tile holds 8 rows
// of W and nothing in its other half, so that twice the workgroups share the product; this product has too few
// columns to fill the chip otherwise, and its K cannot be split over workgroups (the epilogue needs whole sums).
template <int MB, int KS, int PACK, bool HALF, int UNROLL = 1>
__global__ __launch_bounds__(SK_THREADS) void qkv_rope_skinny_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int64_t lda, const int32_t* __restrict__ positions, int M, int K, int nh,
    int nkv, int hd, int ucols, bf16_t* __restrict__ q_out, const bf16_t* __restrict__ bias, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, const int64_t* __restrict__ slot_mapping, bf16_t* __restrict__ k_pages,
    bf16_t* __restrict__ v_pages, int page_size, int write_kv, NormIn norm_in) {
  static_assert(PACK == 1 || MB == 1, "a packed tile holds at most 8 rows of A");
  static_assert(PACK == 1 || !HALF, "a tile is packed or half empty, not both");
  using Area = SkinnyArea<2, MB>;
  __shared__ __attribute__((aligned(16))) unsigned char area[SK_WAVES][Area::BYTES];
  __shared__ float rstd[16];
  auto red = [&](int w, int n, int m) -> float& { return reinterpret_cast<float*>(area[w])[n * (MB * 16 + 1) + m]; };
  using P = Packed<PACK>;
  constexpr int CP = HALF ? 8 : P::CP;
  constexpr int GROUPS = SK_WAVES / KS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int grp = wave / KS, ks = wave % KS;
  // a unit's two tiles hold `ucols` (<= CP) columns each: fewer than a tile's where that spreads the product over more
  // compute units (the lanes of the other columns load nothing)
  const int half = hd >> 1, upq = half / ucols;         // units per q or k head
  const int upv = hd / (2 * ucols);                     // units per v head
  const int qk_units = (nh + nkv) * upq, units = qk_units + nkv * upv;
  const int unit = blockIdx.x * GROUPS + grp;
  const bool unit_ok = unit < units;
  // first rows of the unit's two tiles
  int row0 = 0, row1 = 0;
  if (unit_ok) {
    if (unit < qk_units) {
      row0 = (unit / upq) * hd + (unit % upq) * ucols;
      row1 = row0 + half;
    } else {
      const int u = unit - qk_units;
      row0 = (nh + nkv) * hd + u * 2 * ucols;
      row1 = row0 + ucols;
    }
  }
  const KRange<PACK> kr(ks * PACK, (K + 63) / 64, 1, K, std::integral_constant<int, KS * PACK>());
  SkinnySource<2, MB, 2> src;
  src.kend = kr.kend;
  src.w[0] = sk_buffer(W + (int64_t)row0 * K);
  src.w[1] = sk_buffer(W + (int64_t)row1 * K);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) src.a[mb] = sk_buffer(A + mb * 16 * lda);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tr = (lane >> 3) + 8 * j;            // the row of a tile that the lane brings a piece of
    const uint32_t from = (kr.shift[j] + (lane & 7) * 8) * 2;
    src.ke[j] = kr.ke[j];
    const int wrow = HALF ? (tr & 7) : P::col(tr);
    src.wat[0][j] = src.wat[1][j] = unit_ok && (!HALF || tr < 8) && wrow < ucols ? (uint32_t)wrow * (uint32_t)K * 2 + from : SK_NOTHING;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      src.aat[mb][j] = mb * 16 + P::col(tr) < M ? (uint32_t)P::col(tr) * (uint32_t)lda * 2 + from : SK_NOTHING;
  }
  // What the epilogue needs from memory is asked for while the weights stream: an epilogue item is (unit of the workgroup, column, row of
  // A).  Positions first, before the weights; slots, biases and, where the positions are in by then, cosines and sines beside them.
  constexpr int MROWS = PACK == 1 ? MB * 16 : CP;
  constexpr int ITEMS = (GROUPS * CP * MROWS + SK_THREADS - 1) / SK_THREADS;
  int e_pos[ITEMS];
  int64_t e_slot[ITEMS];
  float e_cos[ITEMS], e_sin[ITEMS];
  uint32_t e_blo[ITEMS], e_bhi[ITEMS];           // biases as they lie in memory
  const bf16_t* biases = bias ? bias : W;        // (a load that stands behind no branch is not waited for at the branch's end)
  const int64_t* slots = write_kv ? slot_mapping : reinterpret_cast<const int64_t*>(W);
  auto item = [&](int it, int& nl, int& m, int& u) {
    const int idx = threadIdx.x + it * SK_THREADS, rest = idx / ucols;
    nl = idx % ucols;
    m = rest / GROUPS;
    u = blockIdx.x * GROUPS + rest % GROUPS;
  };
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    int nl, m, u;
    item(it, nl, m, u);
    e_pos[it] = positions[min(m, M - 1)];
  }
  auto beside = [&]() {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      int nl, m, u;
      item(it, nl, m, u);
      m = min(m, M - 1);
      u = min(u, units - 1);
      const int v = u - qk_units, head = v < 0 ? u / upq : nh + nkv + v / upv, j = v < 0 ? (u % upq) * ucols + nl : (v % upv) * 2 * ucols + nl;
      e_slot[it] = slots[m];
      e_blo[it] = biases[head * hd + j];
      e_bhi[it] = biases[head * hd + j + (v < 0 ? half : ucols)];
      const int64_t at = v < 0 ? (int64_t)e_pos[it] * half + j : 0;
      e_cos[it] = cos_t[at];
      e_sin[it] = sin_t[at];
    }
  };
  f32x4 acc[2][MB];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[nt][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  NormInLoads in_loads;
  skinny_accumulate<2, MB, UNROLL>(acc, src, reinterpret_cast<u32x4*>(area[wave]), lane, [&]() {
    if (MB == 1) in_loads.load(norm_in, A, M, wave, lane);
    beside();
  });
  if (MB == 1) in_loads.finish(norm_in, rstd, M, wave, lane);
  const bool scale_rows = MB == 1 && norm_in.sumsq != nullptr;
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i) red(wave, nt * 16 + g * 4 + i, mb * 16 + r) = acc[nt][mb][i];
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    int nl, m, u;
    item(it, nl, m, u);
    const int gi = u % GROUPS;
    if (m >= M || u >= units) continue;
    float lo = 0.f, hi = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w)
#pragma unroll
      for (int q = 0; q < PACK; ++q) {
        const int col = PACK == 1 ? m : q * CP + m;
        lo += red(gi * KS + w, q * CP + nl, col);
        hi += red(gi * KS + w, 16 + q * CP + nl, col);
      }
    if (scale_rows) {
      lo *= rstd[m];
      hi *= rstd[m];
    }
    lo += bias ? __uint_as_float(e_blo[it] << 16) : 0.f;
    hi += bias ? __uint_as_float(e_bhi[it] << 16) : 0.f;
    const int64_t slot = write_kv ? e_slot[it] : -1;
    int64_t page = 0, off = 0;
    if (slot >= 0) slot_page(slot, page_size, page, off);
    if (u < qk_units) {
      const int head = u / upq, j = (u % upq) * ucols + nl;
      const float c = e_cos[it], sn = e_sin[it];
      const bf16_t olo = f32_to_bf16(lo * c - hi * sn), ohi = f32_to_bf16(lo * sn + hi * c);
      if (head < nh) {
        bf16_t* o = q_out + (int64_t)m * nh * hd + (int64_t)head * hd + j;
        o[0] = olo;
        o[half] = ohi;
      } else if (slot >= 0) {
        bf16_t* o = k_pages + ((page * nkv + (head - nh)) * page_size + off) * hd + j;
        o[0] = olo;
        o[half] = ohi;
      }
    } else if (slot >= 0) {
      const int v = u - qk_units;
      const int gh = v / upv, d = (v % upv) * 2 * ucols + nl;
      bf16_t* o = v_pages + ((page * nkv + gh) * (int64_t)hd + d) * page_size + off;
      o[0] = f32_to_bf16(lo);
      o[(int64_t)ucols * page_size] = f32_to_bf16(hi);
    }
  }
}

// q_out [M, nh*hd]; A [M, K] (row stride lda); W [(nh + 2 nkv) hd, K]; bias [(nh + 2 nkv) hd] or null;
// positions int32 [M]; cos_t, sin_t float [positions, hd/2]; slot_mapping int64 [M] (-1: no cache write);
// k_pages [pages, nkv, page_size, hd], v_pages [pages, nkv, hd, page_size].  norm: null, or the sums of the
// norm whose (h * g) the rows of A are (its in_ fields only).  pack: 0 (the library chooses), 1 or 2.
//
// Columns of a unit's tile: a tile's 16, 8 when packed, and half of those where a packed tile's 8 would leave the product on so few
// workgroups that twice as many still make one round of the chip.  us over weights beyond the 256 MB cache, at 1 and 8 rows, 8 + 8 columns
// and 4 + 4: 2,048 columns of a K of 1,536 (128 workgroups and 256) 5.47 and 5.82, 5.45 and 5.65; the other way 2,560 of 2,048 (160 and
// 320) 5.97 and 6.28, 6.83 and 6.99.
extern "C" int ga_qkv_unit_columns(int columns, int hd, int pack, int half_tiles) {
  const int ucols = half_tiles ? 8 : 16 / pack;
  return pack == 2 && columns / ucols <= GA_FOLD_TARGET && (hd / 2) % (ucols / 2) == 0 ? ucols / 2 : ucols;
}
extern "C" int ga_qkv_rope_skinny(void* q_out, const void* A, int64_t lda, const void* W, const void* bias,
                                  const void* positions, const void* cos_t, const void* sin_t,
                                  const void* slot_mapping, void* k_pages, void* v_pages, int M, int K, int nh,
                                  int nkv, int hd, int page_size, int write_kv, int pack, const GaSkinnyNorm* norm,
                                  hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 64 || K <= 0 || K % 8 || lda % 8 || hd % 32 || nh <= 0 || nkv <= 0 || sk_too_far(K, M > 1 ? lda : 0)) return -1;
  if (M == 1) lda = K;
  const int mb = (M + 15) / 16;
  NormIn norm_in = {nullptr, 0, 0.f, 0.f};
  if (norm && norm->residual) return -6;
  if (norm && norm->in_sumsq) {
    if (mb != 1 || norm->in_parts < 1 || norm->in_parts > NORM_IN_MAX_PARTS) return -5;
    norm_in = NormIn{norm->in_sumsq, norm->in_parts, norm->inv_width, norm->eps};
  }
  if (pack == 0) pack = auto_pack(M, (nh + 2 * nkv) * hd / 32);
  if (pack != 1 && (pack != 2 || M > 8)) return -2;
  const int ks = 8, groups = SK_WAVES / ks;
  // with more than 8 rows and so few columns that full tiles leave most of the chip idle: half tiles (us at 17 and 64 rows, full ->
  // half: 64 workgroups of full tiles (2,048 columns, K 1,536) 7.4 -> 6.8, 10.9 -> 9.2; 80 (2,560, K 2,048) 8.5 -> 7.9, 12.3 -> 10.7; but 144
  // (4,608, K 1,536) 7.8 -> 8.4, 11.4 -> 15.0)
  const bool half_tiles = pack == 1 && M > 8 && (nh + 2 * nkv) * hd / 32 < 128;
  const int ucols = ga_qkv_unit_columns((nh + 2 * nkv) * hd, hd, pack, half_tiles);
  const int units = (nh + 2 * nkv) * hd / (2 * ucols);
  const int ksteps = (K + 63) / 64;
  dim3 grid((units + groups - 1) / groups), block(SK_THREADS);
  // a packed tile's wavefronts with two steps of K ask for both at once: 2,048 columns of a K of 1,536 at 1 and 8 rows 5.65 and 5.83 us in
  // two trips, 5.44 and 5.66 in one, 4,608 columns 7.37 and 7.78, 7.17 and 7.48; with one step (K 896) 4.06 -> 4.44, with four (4,608
  // columns of 3,584) 11.4 -> 11.6 at 1 row, 12.4 -> 11.9 at 8
  const bool both = pack == 2 && (ksteps + 2 * ks - 1) / (2 * ks) == 2;
#define LAUNCH(MB, PK, HF, ...)                                                                           \
  hipLaunchKernelGGL((qkv_rope_skinny_kernel<MB, 8, PK, HF, ##__VA_ARGS__>), grid, block, 0, stream, (const bf16_t*)A,  \
                     (const bf16_t*)W, lda, (const int32_t*)positions, M, K, nh, nkv, hd, ucols, (bf16_t*)q_out, (const bf16_t*)bias, \
                     (const float*)cos_t, (const float*)sin_t, (const int64_t*)slot_mapping, (bf16_t*)k_pages, \
                     (bf16_t*)v_pages, page_size, write_kv, norm_in)
  switch (mb) {
    case 1:
      if (both) LAUNCH(1, 2, false, 2); else if (pack == 2) LAUNCH(1, 2, false); else if (half_tiles) LAUNCH(1, 1, true); else LAUNCH(1, 1, false);
      break;
    case 2:
      if (half_tiles) LAUNCH(2, 1, true); else LAUNCH(2, 1, false);
      break;
    case 3:
      if (half_tiles) LAUNCH(3, 1, true); else LAUNCH(3, 1, false);
      break;
    default:
      if (half_tiles) LAUNCH(4, 1, true); else LAUNCH(4, 1, false);
      break;
  }
#undef LAUNCH
  return GA_CHECK_LAUNCH();
}
