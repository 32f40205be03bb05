// The walk over a request's tokens that the recurrences with a decaying outer-product state share:
//   S <- diag(a_t) S + k_t v_t^T,  o_t = S^T q_t        (S is [dim, vdim], 32-bit; a acts on the rows)
// A workgroup owns one (entry, head, block of COLS value columns): 16 x COLS threads, thread (s, j) keeps the rows s, s + 16,
// ... of column j in registers.  TILE tokens at a time lie in LDS, the R rows of a slice side by side, so that a token's
// operands are three reads of R numbers; results are partial sums per slice, added over the 16 slices in ascending order.
// Tiles and partial sums are double-buffered, one barrier a tile: while a tile is walked, the next is on its way from memory
// in registers (as loaded: what is computed from it waits until it is stored, so that nothing waits for memory), and the
// results of the one before are added up.  The tokens of a full tile are walked without a branch between them.
//
// What bounds it is the chain of tokens: with one wavefront a SIMD a token costs its 3 R + 4 vector instructions and the
// LDS reads of its wavefronts.  Fewer columns a workgroup halve the reads a compute unit makes per token, which is what a
// single prompt wants (its workgroups do not fill the chip anyway); many entries take 16 columns, which read a token's
// operands half as often.  Entries of one token (a decode step) are bound by the way of their state from memory and back: a
// tile of one token leaves its LDS to as many workgroups as the registers allow.  The caller chooses (decay_walk_way in
// kernels/ops.py, with both sides measured).  A result's bits depend on neither COLS nor TILE, nor on how tokens were cut into steps.
#pragma once
#include "common.h"
#include <type_traits>

#define DW_SLICES 16

__host__ __device__ constexpr int dw_threads(int cols) { return cols == 8 ? 384 : DW_SLICES * cols; }

// Source: `Fixed` (what a channel has for all tokens), fixed(channel), `Raw` (what a thread loads for one element of q, k and a),
// load(Raw&, start, token, channel), finish(Raw, Fixed, channel, q, k, a), load_v(start, token, column), finish_v(v); finish and
// finish_v are templates on whether `acts` is set.  `start` is the same for all threads, tokens count from it.  K_OF_A: k is 1 - a,
// and with 16 columns LDS, whose reads are what many entries wait for, does not hold it.  (With 8 columns it does: a chain waits for
// its arithmetic, 2,048 tokens, 8 heads of 192 x 192, 443 us and 499 without.)
template <int R, int COLS, int TILE, class Source>
__device__ __forceinline__ void decay_walk(float* __restrict__ out, const Source& source, float* __restrict__ state, bool fresh,
                                           int n, int heads, int dim, int vdim, int v0) {
  constexpr int WALKERS = DW_SLICES * COLS, THREADS = dw_threads(COLS), SERVERS = THREADS > WALKERS ? THREADS - WALKERS : WALKERS;
  constexpr int DP = DW_SLICES * R, PER = (TILE * DP + SERVERS - 1) / SERVERS;
  constexpr bool K_OF_A = Source::K_OF_A && COLS > 8;
  constexpr int OPS = K_OF_A ? 2 : 3;                        // q, k, unless it is 1 - a, and a
  static_assert(TILE <= DW_SLICES, "tile sizes");
  __shared__ __attribute__((aligned(16))) float ops[2][TILE][OPS][DW_SLICES][R];
  __shared__ float vs[2][TILE][COLS], partial[2][TILE][DW_SLICES][COLS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const bool walks = THREADS == WALKERS || wave < WALKERS / WAVE, serves = THREADS == WALKERS || !walks;
  const int tid = (THREADS == WALKERS || walks) ? threadIdx.x : threadIdx.x - WALKERS, j = tid % COLS, s = tid / COLS;
  const bool col_ok = v0 + j < vdim;
  float* st = state + v0 + j;
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = s + DW_SLICES * r;
    S[r] = (walks && !fresh && col_ok && i < dim) ? st[(int64_t)i * vdim] : 0.f;
  }
  typename Source::Raw raw[PER];
  typename Source::Fixed fixed[PER];
  float raw_v = 0.f;
#pragma unroll
  for (int x = 0; x < PER; ++x) fixed[x] = source.fixed(min((tid + x * SERVERS) % DP, dim - 1));
  // WHOLE, with 8 columns: the last tile starts early enough to end with the last token, and is then walked from `t0 - start`
  // on.  So a thread's places in a tile never change, and an address is a uniform part and a constant one.  With 16, where
  // entries are short and their activations a good part of the time, a tile starts where it stands, its last token is brought
  // again for those behind it, and only what is `left` is worked out (64 entries of 9 tokens, 8 heads of 256 x 256, us: 156 ->
  // 123); but not where a thread has so many addresses to find anew that long entries lose more (a prompt of 2,048, 28 heads of
  // 128 x 128: 492 -> 530).  No load is conditional either way: what is loaded
  // must not be merged with what was there, which would wait for it.  (Channels and columns that do not exist read another and
  // drop it.)
  constexpr bool WHOLE = COLS == 8 || (R >= 6 && R <= 12 && !K_OF_A);
  auto start_of = [&](int t0) { return WHOLE ? max(min(t0, n - TILE), 0) : t0; };
  auto fetch = [&](int t0) {
    const int start = WHOLE ? start_of(t0) : min(t0, n - 1), last = min(TILE, WHOLE ? n : n - start) - 1;    // (WHOLE: of all tiles)
#pragma unroll
    for (int x = 0; x < PER; ++x) {
      const int idx = tid + x * SERVERS;
      source.load(raw[x], start, min(idx / DP, last), min(idx % DP, dim - 1));
    }
    raw_v = source.load_v(start, min(s, last), min(v0 + j, vdim - 1));      // thread (s, j): token s, column j
  };
  auto stage_with = [&](int b, int left, auto act, auto few) {
    constexpr bool ACT = decltype(act)::value;
#pragma unroll
    for (int x = 0; x < PER; ++x) {
      const int idx = tid + x * SERVERS, tt = idx / DP, i = idx % DP;
      float q, k, a;
      if ((TILE * DP % SERVERS != 0 && tt >= TILE) || (decltype(few)::value && tt >= left)) break;
      source.template finish<ACT>(raw[x], fixed[x], min(i, dim - 1), q, k, a);
      ops[b][tt][0][i % DW_SLICES][i / DW_SLICES] = i < dim ? q : 0.f;
      if constexpr (!K_OF_A) ops[b][tt][1][i % DW_SLICES][i / DW_SLICES] = i < dim ? k : 0.f;
      ops[b][tt][OPS - 1][i % DW_SLICES][i / DW_SLICES] = i < dim ? a : 0.f;
    }
    if (s < TILE) vs[b][s][j] = source.template finish_v<ACT>(raw_v);
  };
  auto stage = [&](int b, int left, auto few) {                // FEW: `left` may be less than a tile
    if (source.acts) stage_with(b, left, std::true_type(), few);
    else stage_with(b, left, std::false_type(), few);
  };
  // the operands of AHEAD tokens are asked for from LDS before a token is worked off (none with 16 columns: a step of many
  // entries lives from many workgroups on a compute unit, and registers cost those)
  constexpr int AHEAD = COLS > 8 ? 0 : R <= 4 ? 3 : R <= 8 ? 2 : 1;
  float qx[AHEAD + 1][R], kx[AHEAD + 1][R], ax[AHEAD + 1][R], vx[AHEAD + 1];
  auto read = [&](int b, int tt, int at) {
    vx[at] = vs[b][tt][j];
#pragma unroll
    for (int r = 0; r < R; ++r) kx[at][r] = K_OF_A ? 0.f : ops[b][tt][1][s][r];
#pragma unroll
    for (int r = 0; r < R; ++r) ax[at][r] = ops[b][tt][OPS - 1][s][r];
#pragma unroll
    for (int r = 0; r < R; ++r) qx[at][r] = ops[b][tt][0][s][r];
  };
  auto token = [&](int b, int tt, int at) {
    float acc = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S[r] = fmaf(ax[at][r], S[r], (K_OF_A ? 1.0f - ax[at][r] : kx[at][r]) * vx[at]);
      acc = fmaf(S[r], qx[at][r], acc);
    }
    partial[b][tt][s][j] = acc;
  };
  auto put = [&](int t0, int b) {                            // thread (s, j) adds up token s, column j
    if (s >= TILE || t0 < 0 || t0 + s >= n || !col_ok) return;
    float o = 0.f;
#pragma unroll
    for (int p = 0; p < DW_SLICES; ++p) o += partial[b][s][p][j];
    out[(int64_t)(t0 + s) * heads * vdim + v0 + j] = o;
  };
  if (serves) {
    fetch(0);
    if (n < TILE) {
      stage(0, n, std::true_type());
    } else {
      stage(0, n, std::false_type());
      fetch(TILE);
    }
  }
  int b = 0, t0 = 0;
  for (; t0 + TILE <= n; t0 += TILE, b ^= 1) {               // (behind the last tile 8 columns bring the last one again)
    __syncthreads();                                         // this tile is staged; the partial sums of the one before are in
    if (walks && AHEAD == 0) {
#pragma unroll 1
      for (int tt = 0; tt < TILE; ++tt) {
        read(b, tt, 0);
        token(b, tt, 0);
      }
    } else if (walks) {
#pragma unroll
      for (int tt = 0; tt < AHEAD; ++tt) read(b, tt, tt);
#pragma unroll
      for (int tt = 0; tt < TILE; ++tt) {
        if (tt + AHEAD < TILE) read(b, tt + AHEAD, (tt + AHEAD) % (AHEAD + 1));
        __builtin_amdgcn_sched_barrier(0x0206);              // arithmetic and stores may move past this, reads may not
        token(b, tt, tt % (AHEAD + 1));
      }
    }
    if (serves) {
      put(t0 - TILE, b ^ 1);
      if constexpr (WHOLE) {
        if (COLS == 8 || t0 + TILE < n) {
          stage(b ^ 1, TILE, std::false_type());
          fetch(t0 + 2 * TILE);
        }
      } else {
        if (t0 + TILE < n) stage(b ^ 1, n - t0 - TILE, std::true_type());
        fetch(t0 + 2 * TILE);
      }
    }
  }
  __syncthreads();
  if (serves) put(t0 - TILE, b ^ 1);
  if (t0 < n) {
    const int skip = t0 - start_of(t0);
    for (int tt = 0; walks && tt < n - t0; ++tt) {
      read(b, skip + tt, 0);
      token(b, tt, 0);
    }
    __syncthreads();
    if (serves) put(t0, b);
  }
  if (walks && col_ok) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int i = s + DW_SLICES * r;
      if (i < dim) st[(int64_t)i * vdim] = S[r];
    }
  }
}

// GO(R, COLS, TILE) for a state of up to 16 * rows rows: as many tokens a tile as leave the workgroups of 16 columns (a step's
// many) or one of 8 their LDS; tokens: that many instead.  With up to 16 rows of state 16 tokens leave four workgroups of 16 columns
// a compute unit, 8 leave eight: `many` says that there are more than four (16 heads of 16 x 32, us, 16 -> 8 tokens: 64 entries of
// 64 29 -> 26, 200 of 33 50 -> 43, but 16 entries of 129 22 -> 27).
#define DW_TILE(TOKENS, OWN) (TOKENS > 0 ? TOKENS : OWN)
#define DW_ROWS(rows, COLS, TOKENS, many, GO)                                                    \
  do {                                                                                           \
    if (rows <= 1 && COLS == 16 && many) GO(1, COLS, DW_TILE(TOKENS, 8));                        \
    else if (rows <= 1) GO(1, COLS, DW_TILE(TOKENS, 16));                                        \
    else if (rows <= 2) GO(2, COLS, DW_TILE(TOKENS, (COLS == 8 ? 16 : 8)));                      \
    else if (rows <= 3) GO(3, COLS, DW_TILE(TOKENS, (COLS == 8 ? 16 : 8)));                      \
    else if (rows <= 4) GO(4, COLS, DW_TILE(TOKENS, (COLS == 8 ? 16 : 8)));                      \
    else if (rows <= 6) GO(6, COLS, DW_TILE(TOKENS, 8));                                         \
    else if (rows <= 8) GO(8, COLS, DW_TILE(TOKENS, 8));                                         \
    else if (rows <= 12) GO(12, COLS, DW_TILE(TOKENS, 8));                                       \
    else GO(16, COLS, DW_TILE(TOKENS, 4));                                                       \
  } while (0)
// way: 1 tiles of one token in 16 columns, 8 and 16 that many columns
#define DW_WAY(way, rows, many, GO)                       \
  do {                                                    \
    if (way == 1) DW_ROWS(rows, 16, 1, false, GO);        \
    else if (way == 8) DW_ROWS(rows, 8, 0, false, GO);    \
    else DW_ROWS(rows, 16, 0, many, GO);                  \
  } while (0)
static inline bool dw_many(int entries, int heads, int vdim) { return (int64_t)entries * heads * ((vdim + 15) / 16) > 4 * 256; }
