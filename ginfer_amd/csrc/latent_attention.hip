// Attention over a cached LATENT: per token only c (kv_rank numbers) is kept, in pages; a head's keys and values are
// linear maps of c (k = Wuk c, v = Wuv c), so with the query carried into the latent space (qa = Wuk^T q) a head's score
// is qa . c and its output Wuv (sum_j p_j c_j): every head attends to the same rows c, which serve as keys and as values.
// A cached row may be longer than its latent (`row` >= `rank` elements): what lies behind the latent is a key part of its own
// that all heads share (turned by position, say), met by the query's elements behind the first `rank`; values are the latent
// alone.
//   s_j = scale * qa . row_j  for positions j with 0 <= i - j < window (window 0: all earlier positions)
//   p_j = exp(s_j) / (exp(sink) + sum_j exp(s_j))        the sink is a learned number per head with no key and no value
//   out = gate * sum_j p_j c_j                            gate: a number per token and head (or none)
// Scores, weights and sums are 32-bit.  Keys are taken in tiles that start at absolute multiples of the tile length and
// every sum has a fixed order, so a token's result does not depend on how its request was cut into steps.
//
// latent_prepare: the two RMS norms (each with a weight per coordinate) on the down-projections, the sigmoid of the
// gate logits, and the write of c into its page.
// latent_turned_prepare: the same for rows with a turned key part: RMS norm of the latent, the rotation of the key part and
// of every head's query part, and the write of the row into its page.
#include "lds_load.h"
#include "ginfer_amd.h"

#define LA_MAX_HEADS_PER_WG 8
#define LA_PAD 4
#define LA_MAX_RANK 512
#define LA_MAX_ROW 640

// ---------------------------------------------------------------------------------------------------- prepare
// proj float [T, q_rank + kv_rank + heads]: (down-projection of the queries | of keys and values | gate logits)
template <typename T>
__global__ __launch_bounds__(256) void latent_prepare_kernel(T* __restrict__ cq, T* __restrict__ c_pages, float* __restrict__ gate,
                                                             const float* __restrict__ proj, int64_t proj_stride,
                                                             const float* __restrict__ wq, const float* __restrict__ wkv,
                                                             const int64_t* __restrict__ slot_mapping, int q_rank, int kv_rank,
                                                             int heads, float eps, int write_c) {
  __shared__ float scratch[4];
  const int64_t t = blockIdx.x;
  const float* p = proj + t * proj_stride;
  float ss = 0.f;
  for (int i = threadIdx.x; i < q_rank; i += 256) ss += p[i] * p[i];
  ss = block_sum<4>(ss, scratch);
  float rms = sqrtf(ss / (float)q_rank + eps);
  for (int i = threadIdx.x; i < q_rank; i += 256) Num<T>::st(cq + t * q_rank + i, p[i] / rms * wq[i]);
  const int64_t slot = slot_mapping[t];
  if (write_c && slot >= 0) {                       // uniform over the workgroup
    p += q_rank;
    ss = 0.f;
    for (int i = threadIdx.x; i < kv_rank; i += 256) ss += p[i] * p[i];
    ss = block_sum<4>(ss, scratch);
    rms = sqrtf(ss / (float)kv_rank + eps);
    for (int i = threadIdx.x; i < kv_rank; i += 256) Num<T>::st(c_pages + slot * kv_rank + i, p[i] / rms * wkv[i]);
    p -= q_rank;
  }
  if (gate)
    for (int i = threadIdx.x; i < heads; i += 256) gate[t * heads + i] = 1.0f / (1.0f + expf(-p[q_rank + kv_rank + i]));
}

// Rows with a turned key part.  proj [T, ...] (compute dtype, row stride given): heads * (dim + turned) query columns, head by
// head (plain | to be turned); at down_start (write only) rank columns of the latent before its norm and turned columns of
// the shared key part.  The latent takes rank8 elements of a row and the key part turned8 behind them (each rounded up to
// multiples of 8, zeros between): q's turned part goes to qa[h][t][rank8 ..], the row to its slot in c_pages.  The first `dims` of the turned coordinates are turned by the token's position (tables
// cos, sin float [positions, dims / 2]; pairs (j, j + dims / 2), or (2j, 2j + 1) where `neighbours`), the rest pass.
template <typename T, typename LD>
__device__ __forceinline__ float la_turned(LD load, int j, int dims, int neighbours, const float* cs, const float* sn) {
  if (j >= dims) return load(j);
  const int half = dims >> 1;
  const int i = neighbours ? j >> 1 : (j < half ? j : j - half);
  const bool first = neighbours ? (j & 1) == 0 : j < half;
  const float u = load(neighbours ? 2 * i : i), v = load(neighbours ? 2 * i + 1 : i + half);
  return first ? u * cs[i] - v * sn[i] : v * cs[i] + u * sn[i];
}

// a token's cached row, by a workgroup of 256: p the latent before its norm and the key part behind it
template <typename T>
__device__ __forceinline__ void la_write_row(T* __restrict__ dst, const T* __restrict__ p, const float* __restrict__ wkv, const float* cs,
                                             const float* sn, int turned, int dims, int neighbours, int rank, float eps,
                                             float* scratch) {
  const int rank8 = (rank + 7) & ~7, row = rank8 + ((turned + 7) & ~7);
  float ss = 0.f;
  for (int i = threadIdx.x; i < rank; i += 256) {
    const float z = Num<T>::ld(p + i);
    ss += z * z;
  }
  ss = block_sum<4>(ss, scratch);
  const float rms = sqrtf(ss / (float)rank + eps);
  for (int i = threadIdx.x; i < row; i += 256) {
    float v = 0.f;
    if (i < rank) v = Num<T>::ld(p + i) / rms * wkv[i];
    else if (i >= rank8 && i - rank8 < turned)
      v = la_turned<T>([&](int x) { return Num<T>::ld(p + rank + x); }, i - rank8, dims, neighbours, cs, sn);
    Num<T>::st(dst + i, v);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void latent_turned_prepare_kernel(
    T* __restrict__ qa, int64_t qa_t, int64_t qa_h, T* __restrict__ c_pages, const T* __restrict__ proj, int64_t proj_stride, int down_start, const float* __restrict__ wkv,
    const int32_t* __restrict__ positions, const float* __restrict__ cosines, const float* __restrict__ sines,
    const int64_t* __restrict__ slot_mapping, int heads, int dim, int turned, int dims, int neighbours, int rank, float eps,
    int write) {
  __shared__ float scratch[4];
  const int64_t t = blockIdx.x;
  const T* p = proj + t * proj_stride;
  const int half = dims >> 1, rank8 = (rank + 7) & ~7, turned8 = (turned + 7) & ~7, row = rank8 + turned8;
  const float* cs = cosines + (int64_t)positions[t] * half;
  const float* sn = sines + (int64_t)positions[t] * half;
  for (int i = threadIdx.x; i < heads * turned8; i += 256) {
    const int h = i / turned8, j = i - h * turned8;
    const T* q = p + h * (dim + turned) + dim;
    float v = 0.f;
    if (j < turned) v = la_turned<T>([&](int x) { return Num<T>::ld(q + x); }, j, dims, neighbours, cs, sn);
    Num<T>::st(qa + t * qa_t + h * qa_h + rank8 + j, v);
  }
  const int64_t slot = slot_mapping[t];
  if (!write || slot < 0) return;                     // uniform over the workgroup
  la_write_row<T>(c_pages + slot * row, p + down_start, wkv, cs, sn, turned, dims, neighbours, rank, eps, scratch);
}

extern "C" int ga_latent_turned_prepare(void* qa, int64_t qa_t, int64_t qa_h, void* c_pages, const void* proj,
                                        int64_t proj_stride, int down_start, const void* wkv,
                                        const void* positions, const void* cosines, const void* sines, const void* slot_mapping,
                                        int tokens, int heads, int dim, int turned, int dims, int neighbours, int rank, float eps,
                                        int write, int is_bf16, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (heads <= 0 || dim < 0 || turned <= 0 || dims < 0 || dims % 2 || dims > turned || rank <= 0 ||
      down_start < 0 || (write && (!wkv || !c_pages)))
    return -1;
#define GO(T) hipLaunchKernelGGL(latent_turned_prepare_kernel<T>, dim3(tokens), dim3(256), 0, stream, (T*)qa, qa_t, qa_h,         \
                                 (T*)c_pages, (const T*)proj, proj_stride, down_start, (const float*)wkv, \
                                 (const int32_t*)positions, (const float*)cosines, (const float*)sines,                        \
                                 (const int64_t*)slot_mapping, heads, dim, turned, dims, neighbours, rank, eps, write)
  if (is_bf16) GO(bf16_t); else GO(float);
#undef GO
  return GA_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------------------------------- attention
// One workgroup per token and up to 8 heads (a wavefront each).  A tile of TK keys (rows of c, widened to 32-bit) goes
// through LDS once for all heads.  Scores: a lane takes key lane % TK and a share lane / TK of the rank, the shares meet
// by lane exchanges; outputs: a lane takes the coordinates lane, lane + 64, ... and adds the tile's keys in order.
template <typename T, typename Q, int TK>
__global__ void latent_attention_kernel(T* __restrict__ out, int64_t out_t, int64_t out_h, const Q* __restrict__ qa,
                                        int64_t qa_t, int64_t qa_h, const T* __restrict__ c_pages,
                                        const int32_t* __restrict__ block_table, int table_width,
                                        const int32_t* __restrict__ token_entry, const int32_t* __restrict__ positions,
                                        const float* __restrict__ sink, const float* __restrict__ gate, int heads, int rank,
                                        int row, int page_size, int window, float scale, int heads_per_wg) {
  extern __shared__ float lds[];
  constexpr int G = WAVE / TK;                       // shares of the rank per key
  constexpr int RL = LA_MAX_RANK / WAVE;             // output coordinates per lane, at most
  const int stride = row + LA_PAD;
  float* tile = lds;                                 // [TK][row + pad]
  float* pw = tile + TK * stride;                    // [waves][TK]
  float* qw = pw + heads_per_wg * TK;                // [waves][row]
  const int t = blockIdx.x, w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int h = blockIdx.y * heads_per_wg + w;
  const bool head_ok = h < heads;
  const int e = token_entry[t], pos = positions[t];
  const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  const int32_t* bt = block_table + (int64_t)e * table_width;
  if (head_ok)
    for (int r = lane; r < row; r += WAVE) qw[w * row + r] = Num<Q>::ld(qa + (int64_t)t * qa_t + (int64_t)h * qa_h + r);
  const int key = lane % TK, g = lane / TK;
  const int share = (row + G - 1) / G;
  const int r0 = g * share, r1 = min(row, r0 + share);
  float m = -INFINITY, l = 0.f, acc[RL];
#pragma unroll
  for (int x = 0; x < RL; ++x) acc[x] = 0.f;
  const int nthreads = blockDim.x;
  for (int k0 = (lo / TK) * TK; k0 <= pos; k0 += TK) {
    __syncthreads();                                 // the tile before is used up (and qw is written)
    if ((row & 7) == 0) {
      const int chunks = row >> 3;
      for (int item = threadIdx.x; item < TK * chunks; item += nthreads) {
        const int kk = item / chunks, r = (item - kk * chunks) << 3;
        const int kp = k0 + kk;
        float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (kp >= lo && kp <= pos) {
          const int page = bt[kp / page_size];
          const T* src = c_pages + ((int64_t)page * page_size + kp % page_size) * row + r;
#pragma unroll
          for (int x = 0; x < 8; ++x) v[x] = Num<T>::ld(src + x);
        }
        float* dst = tile + kk * stride + r;
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
      }
    } else {
      for (int item = threadIdx.x; item < TK * row; item += nthreads) {
        const int kk = item / row, r = item - kk * row;
        const int kp = k0 + kk;
        float v = 0.f;
        if (kp >= lo && kp <= pos) {
          const int page = bt[kp / page_size];
          v = Num<T>::ld(c_pages + ((int64_t)page * page_size + kp % page_size) * row + r);
        }
        tile[kk * stride + r] = v;
      }
    }
    __syncthreads();
    float alpha = 1.f;
    if (head_ok) {
      const float* crow = tile + key * stride;
      const float* q = qw + w * row;
      float dot = 0.f;
      for (int r = r0; r < r1; ++r) dot += q[r] * crow[r];
#pragma unroll
      for (int off = TK; off < WAVE; off <<= 1) dot += __shfl_xor(dot, off, WAVE);
      const int kp = k0 + key;
      const bool valid = kp >= lo && kp <= pos;
      const float sc = valid ? dot * scale : -INFINITY;
      const float m_new = fmaxf(m, wave_max(sc));
      const float p = valid ? expf(sc - m_new) : 0.f;
      alpha = expf(m - m_new);
      l = l * alpha + wave_sum(g == 0 ? p : 0.f);
      m = m_new;
      if (g == 0) pw[w * TK + key] = p;
    }
    __syncthreads();
    if (head_ok) {
      const float* pk = pw + w * TK;
      const int kend = min(TK, pos - k0 + 1), kbeg = max(0, lo - k0);
#pragma unroll
      for (int x = 0; x < RL; ++x) {
        const int r = lane + x * WAVE;
        if (r < rank) {
          float a = acc[x] * alpha;
          for (int kk = kbeg; kk < kend; ++kk) a += pk[kk] * tile[kk * stride + r];
          acc[x] = a;
        }
      }
    }
  }
  if (!head_ok) return;
  float top = m, den = l, keep = 1.f;
  if (sink) {
    const float s = sink[h];
    top = fmaxf(m, s);
    keep = expf(m - top);
    den = l * keep + expf(s - top);
  }
  const float f = keep / den * (gate ? gate[(int64_t)t * heads + h] : 1.f);
#pragma unroll
  for (int x = 0; x < RL; ++x) {
    const int r = lane + x * WAVE;
    if (r < rank) Num<T>::st(out + (int64_t)t * out_t + (int64_t)h * out_h + r, acc[x] * f);
  }
}

static int la_tile_keys(int row) { return row <= 128 ? 64 : (row <= 256 ? 32 : 16); }

extern "C" int ga_latent_attention_max_rank() { return LA_MAX_RANK; }
extern "C" int ga_latent_attention_max_row() { return LA_MAX_ROW; }

extern "C" int ga_latent_prepare(void* cq, void* c_pages, void* gate, const void* proj,
                                 int64_t proj_stride, const void* wq, const void* wkv, const void* slot_mapping, int tokens,
                                 int q_rank, int kv_rank, int heads, float eps, int write_c, int is_bf16, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (q_rank <= 0 || kv_rank <= 0 || heads <= 0) return -1;
  dim3 grid(tokens), block(256);
  if (is_bf16)
    hipLaunchKernelGGL(latent_prepare_kernel<bf16_t>, grid, block, 0, stream, (bf16_t*)cq, (bf16_t*)c_pages, (float*)gate,
                       (const float*)proj, proj_stride, (const float*)wq, (const float*)wkv, (const int64_t*)slot_mapping,
                       q_rank, kv_rank, heads, eps, write_c);
  else
    hipLaunchKernelGGL(latent_prepare_kernel<float>, grid, block, 0, stream, (float*)cq, (float*)c_pages, (float*)gate,
                       (const float*)proj, proj_stride, (const float*)wq, (const float*)wkv, (const int64_t*)slot_mapping,
                       q_rank, kv_rank, heads, eps, write_c);
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_latent_attention(void* out, int64_t out_t, int64_t out_h, const void* qa, int64_t qa_t, int64_t qa_h, int qa_bf16,
                                   const void* c_pages, const void* block_table, int table_width, const void* token_entry,
                                   const void* positions, const void* sink, const void* gate, int tokens, int heads, int rank,
                                   int row, int page_size, int window, float scale, int is_bf16, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (heads <= 0 || rank <= 0 || rank > LA_MAX_RANK || row < rank || row > LA_MAX_ROW || page_size <= 0 || table_width <= 0 ||
      window < 0 || (qa_bf16 && !is_bf16))
    return -1;
  const int hpw = heads < LA_MAX_HEADS_PER_WG ? heads : LA_MAX_HEADS_PER_WG;
  const int tk = la_tile_keys(row);
  const size_t bytes = ((size_t)tk * (row + LA_PAD) + (size_t)hpw * (tk + row)) * sizeof(float);
  if (bytes > 64 * 1024) return -2;
  dim3 grid(tokens, (heads + hpw - 1) / hpw), block(WAVE * hpw);
#define GO(T, Q, TK) hipLaunchKernelGGL((latent_attention_kernel<T, Q, TK>), grid, block, bytes, stream, (T*)out, out_t, out_h, \
                                     (const Q*)qa, qa_t, qa_h, (const T*)c_pages, (const int32_t*)block_table,              \
                                     table_width, (const int32_t*)token_entry, (const int32_t*)positions,                   \
                                     (const float*)sink, (const float*)gate, heads, rank, row, page_size, window, scale, hpw)
#define GT(T, Q) do { if (tk == 64) GO(T, Q, 64); else if (tk == 32) GO(T, Q, 32); else GO(T, Q, 16); } while (0)
  if (!is_bf16) GT(float, float); else if (qa_bf16) GT(bf16_t, bf16_t); else GT(bf16_t, float);
#undef GT
#undef GO
  return GA_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------------------------------- matrix cores
// bfloat16 on v_mfma_f32_16x16x32_bf16 (D[m][n] += sum_k A[m][k] B[n][k]; lane l supplies row l % 16 and k-slots
// (l / 16) * 8 .. + 7 of both operands and receives D[(l / 16) * 4 + i][l % 16]).  A column n is a (token, head) pair; every
// column of a request attends to the same cached rows, so a workgroup brings a tile of 32 rows into LDS once for all of its
// wavefronts' columns, the next tile on its way while one is worked on:
//   rows   prompt portions: the step's pairs in the order token, head; 16 NS to a wavefront, whatever the number of heads.  Where
//          a workgroup's tokens belong to several requests they are worked off request by request, the others masked.
//   heads  single tokens (decoding): 16 heads of one token to a wavefront; the token's keys may be dealt to several workgroups,
//          whose partial results a second kernel merges.
//   S^T = C QA^T    A = 16 cached rows x 32 elements; row m of product t holds key 8 (m / 4) + 4 t + m % 4 of the tile, so that a
//                   lane ends up with the scores of the 8 consecutive keys 8 (l / 16) .. + 7 of its column, which is the
//                   k-slot layout of operand B for P:
//   O^T += C^T P^T  A = 16 coordinates x 8 consecutive keys of the same rows: LDS reads that transpose 4 x 16 blocks
//                   (lane l of 16 names the 8 bytes of row l / 4, columns 4 (l % 4) .. + 3, and receives column l, rows 0 .. 3).
// A tile's rows are KP elements apart in LDS (the row rounded up to a multiple of 64), 16-byte pieces; piece q of key r lies at
// place q ^ f(r) within its group of eight, f(r) = 2 (r & 3) | (r >> 3 & 1): the rows that either kind of read touches at a time
// then lie in different banks.  Softmax in 32-bit per column over tiles of 32 keys at absolute multiples of 32, to the base
// 2; the running maximum a column's weights refer to is raised only when a tile exceeds it by more than LT_SLACK.
// RP: the rank rounded up (64, 128, 256, 512); KP: the row rounded up, RP or RP + 64; elements beyond the rank and the row meet
// zeros of the query or are not stored.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;

#define LT_LOG2E 1.4426950408889634f
#define LT_ALL 0x3fffffff    // keys before a position that it sees where there is no window: all of them
#define LT_SLACK 8.0f        // in powers of 2: weights stay below 2^8 of what the running maximum says

__device__ __forceinline__ bf16x8 lt_zero8() {
  const uint4 z = make_uint4(0u, 0u, 0u, 0u);
  return __builtin_bit_cast(bf16x8, z);
}
__device__ __forceinline__ bf16x8 lt_pack8(const float* v) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f32_to_bf16(v[2 * i]) | ((uint32_t)f32_to_bf16(v[2 * i + 1]) << 16);
  return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}
__device__ __forceinline__ int lt_swizzle(int key) { return ((key & 3) << 1) | ((key >> 3) & 1); }

// A tile is brought 8 keys at a time, KP / 64 kilobytes each, which lie in one page.  Where a lane's 16 bytes of such a group come
// from is the same for every tile: the table behind the tile buffers holds it, in elements from the group's first row, for
// groups of an even and of an odd number (the two swizzle differently).
template <int KP>
struct TileLayout {
  static constexpr int PIECES = KP;                             // of 16 bytes in a group: 8 rows of KP / 8
  static constexpr int TILE = 32 * KP * 2, TABLE = 2 * TILE, BYTES = TABLE + 2 * PIECES * 2;
};

template <int KP>
__device__ __forceinline__ void lt_fill_table(unsigned char* lds, int row, int threads) {
  uint16_t* table = reinterpret_cast<uint16_t*>(lds + TileLayout<KP>::TABLE);
  for (int i = threadIdx.x; i < 2 * TileLayout<KP>::PIECES; i += threads) {
    const int odd = i / TileLayout<KP>::PIECES, at = i % TileLayout<KP>::PIECES, r = at / (KP / 8), place = at % (KP / 8);
    int piece = (place & ~7) | ((place & 7) ^ lt_swizzle(8 * odd + r));
    if (piece * 8 >= row) piece = 0;                            // behind the row: anything that can be read
    table[i] = (uint16_t)(r * row + piece * 8);
  }
}

// The page of the tile's group l % 4 of 8 keys, in lane l; a group without a key in [lo_min, hi_max] takes the page of hi_max,
// which is there.  A vector load on purpose: it is asked for behind the loads of the tile before, and what waits for it is the
// wait that those need anyway.
__device__ __forceinline__ int lt_find_pages(const int32_t* __restrict__ bt, int k0, int ps_shift, int lo_min, int hi_max, int lane) {
  const int k = k0 + 8 * (lane & 3);
  return bt[((k <= hi_max && k + 7 >= lo_min) ? k : hi_max) >> ps_shift];
}

// The wavefront's share of the tile at k0: its groups of 8 keys into the buffer at `place`.
template <int KP, int WAVES>
__device__ __forceinline__ void lt_bring_tile(const unsigned char* lds, uint32_t place, int pages, const bf16_t* __restrict__ c_pages,
                                              int k0, int row, int ps_shift, int wave, int lane) {
#pragma unroll
  for (int x = 0; x < 4 / WAVES; ++x) {
    const int group = wave * (4 / WAVES) + x;
    const int page = __builtin_amdgcn_readlane(pages, group), in_page = (k0 + 8 * group) & ((1 << ps_shift) - 1);
    const bf16_t* rows = c_pages + (((int64_t)page << ps_shift) + in_page) * row;
    const uint16_t* table = reinterpret_cast<const uint16_t*>(lds + TileLayout<KP>::TABLE) + (group & 1) * TileLayout<KP>::PIECES + lane;
#pragma unroll
    for (int j = 0; j < KP / 64; ++j) lds_bring(place + group * (8 * KP * 2) + j * 1024, rows + table[64 * j]);
  }
}

// The walk over the tiles [tile_lo, tile_hi] (multiples of 32) of one request for the wavefront's NS sets of 16 columns; all
// wavefronts of the workgroup walk together.  qb: the columns' queries as B operands; pos_c: a column's position (-1: it sees
// nothing), from which it looks back over `back` more keys.  Leaves the running maximum (in powers of 2), the lane's part of the sum of weights
// and the unnormalised O^T in m_run, l_run, acc.
template <int RP, int KP, int NS, int WAVES>
__device__ __forceinline__ void lt_walk(f32x4 (&acc)[NS][RP / 16], float (&m_run)[NS], float (&l_run)[NS],
                                        const bf16x8 (&qb)[NS][KP / 32], unsigned char* lds,
                                        const bf16_t* __restrict__ c_pages, const int32_t* __restrict__ bt, int row, int ps_shift,
                                        const int (&pos_c)[NS], int back, int lo_min, int hi_max, int tile_lo,
                                        int tile_hi, float scale2, int wave, int c, int g) {
  constexpr int TILE = TileLayout<KP>::TILE;
  const uint32_t base = (uint32_t)(uintptr_t)(lds_byte_t*)lds;
  // the lane's addresses inside a tile: scores read key 8 (c / 4) + 4 t + c % 4, piece 4 kb + g; values read key
  // 8 g + 4 u + c / 4, coordinates 16 rt + 4 (c % 4)
  const int skey = 8 * (c >> 2) + (c & 3), sf = lt_swizzle(skey);           // + 4 t leaves the swizzle as it is
  const int s_at = skey * KP * 2 + ((g ^ sf) << 4);                         // piece 4 kb + g: ^ 64 where kb is odd
  const int vkey = 8 * g + (c >> 2), vf = lt_swizzle(vkey);
  const int v_at = vkey * KP * 2 + ((((c & 3) >> 1) ^ vf) << 4) + (c & 1) * 8;      // coordinates 16 rt on: ^ 32 (rt % 4)
  if (tile_lo > tile_hi) return;                                            // the same for all wavefronts
  const int lane = 16 * g + c;
  int pages = lt_find_pages(bt, tile_lo, ps_shift, lo_min, hi_max, lane);
  lds_wait_and_meet();                                                       // nobody reads the buffers of a walk before any more
  lt_bring_tile<KP, WAVES>(lds, base, pages, c_pages, tile_lo, row, ps_shift, wave, lane);
  if (tile_lo + 32 <= tile_hi) pages = lt_find_pages(bt, tile_lo + 32, ps_shift, lo_min, hi_max, lane);
  int buf = 0;
  for (int k0 = tile_lo; k0 <= tile_hi; k0 += 32, buf ^= 1) {
    lds_wait_and_meet();                   // this tile is in, and nobody reads the other buffer any more
    if (k0 + 32 <= tile_hi) {
      lt_bring_tile<KP, WAVES>(lds, base + (buf ^ 1) * TILE, pages, c_pages, k0 + 32, row, ps_shift, wave, lane);
      if (k0 + 64 <= tile_hi) pages = lt_find_pages(bt, k0 + 64, ps_shift, lo_min, hi_max, lane);
    }
    const unsigned char* cur = lds + buf * TILE;
    f32x4 s[NS][2];
#pragma unroll
    for (int k = 0; k < NS; ++k) s[k][0] = s[k][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // scores in steps of 32 elements, values in steps of 32 coordinates, each step's two operands asked for AHEAD steps before
    // they are multiplied; the barriers keep the compiler from asking for more than the registers hold
    constexpr int AHEAD = RP == 512 ? 1 : 4, RING = AHEAD + 1, SS = KP / 32, VS = RP / 32;
    bf16x8 ring[RING][2];
    auto ask_scores = [&](int st) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
        ring[st % RING][t] = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4*>(cur + (s_at ^ ((st & 1) * 64)) + (st >> 1) * 128 + t * 4 * KP * 2));
    };
    auto ask_values = [&](int st) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const unsigned char* at = cur + (v_at ^ ((2 * (st & 1) + x) * 32)) + (st >> 1) * 128;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)at);
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at + 4 * KP * 2));
        ring[st % RING][x] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
#pragma unroll
    for (int st = 0; st < AHEAD && st < SS; ++st) ask_scores(st);
#pragma unroll
    for (int st = 0; st < SS; ++st) {
      if (st + AHEAD < SS) ask_scores(st + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int k = 0; k < NS; ++k) s[k][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[st % RING][t], qb[k][st], s[k][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int st = 0; st < AHEAD && st < VS; ++st) ask_values(st);
    bf16x8 pb[NS];
    bool rescale = false;
    float alpha[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      float sc[8], mt = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int kp = k0 + 8 * g + j;
        sc[j] = (kp <= pos_c[k] && kp >= pos_c[k] - back) ? s[k][j >> 2][j & 3] * scale2 : -INFINITY;
        mt = fmaxf(mt, sc[j]);
      }
      mt = max_across_16(mt);
      mt = max_across_32(mt);
      const bool raise = mt > m_run[k] + LT_SLACK;                          // also where the column has seen no key yet
      const float m_new = raise ? mt : m_run[k];
      alpha[k] = raise ? __builtin_amdgcn_exp2f(m_run[k] - m_new) : 1.f;
      const float ref = m_new == -INFINITY ? 0.f : m_new;
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sc[j] = __builtin_amdgcn_exp2f(sc[j] - ref);
        sum += sc[j];
      }
      l_run[k] = l_run[k] * alpha[k] + sum;
      m_run[k] = m_new;
      pb[k] = lt_pack8(sc);
      rescale = rescale || raise;
    }
    if (__any(rescale)) {
#pragma unroll
      for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int rt = 0; rt < RP / 16; ++rt) acc[k][rt] *= alpha[k];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < VS; ++st) {
      if (st + AHEAD < VS) ask_values(st + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int k = 0; k < NS; ++k)
          acc[k][2 * st + x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[st % RING][x], pb[k], acc[k][2 * st + x], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int KP>
__device__ __forceinline__ void lt_load_query(bf16x8 (&qb)[KP / 32], const bf16_t* __restrict__ q, int row, int g, bool ok) {
#pragma unroll
  for (int ks = 0; ks < KP / 32; ++ks) {
    const int r = 32 * ks + 8 * g;
    qb[ks] = ok && r < row ? __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(q + r)) : lt_zero8();
  }
}
template <int KP>
__device__ __forceinline__ void lt_load_query(bf16x8 (&qb)[KP / 32], const float* __restrict__ q, int row, int g, bool ok) {
#pragma unroll
  for (int ks = 0; ks < KP / 32; ++ks) {
    const int r = 32 * ks + 8 * g;
    if (ok && r < row) {
      float v[8];
      const float4 a = *reinterpret_cast<const float4*>(q + r), b = *reinterpret_cast<const float4*>(q + r + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
      qb[ks] = lt_pack8(v);
    } else {
      qb[ks] = lt_zero8();
    }
  }
}

// the column's factor on its sums: 1 over (sum of weights + the sink's), times the gate; m in powers of 2
__device__ __forceinline__ float lt_finish(float m, float l, const float* sink, const float* gate, int t, int h, int heads) {
  float keep = 1.f, den = l;
  if (sink) {
    const float s = sink[h] * LT_LOG2E, top = fmaxf(m, s);
    keep = exp2f(m - top);
    den = l * keep + exp2f(s - top);
  }
  return keep / den * (gate ? gate[(int64_t)t * heads + h] : 1.f);
}

template <int RP>
__device__ __forceinline__ void lt_store(bf16_t* __restrict__ o, const f32x4 (&acc)[RP / 16], float f, int rank, int g) {
#pragma unroll
  for (int rt = 0; rt < RP / 16; ++rt) {
    const int r = 16 * rt + 4 * g;
    if (r < rank) {
      const uint32_t lo = (uint32_t)f32_to_bf16(acc[rt][0] * f) | ((uint32_t)f32_to_bf16(acc[rt][1] * f) << 16);
      const uint32_t hi = (uint32_t)f32_to_bf16(acc[rt][2] * f) | ((uint32_t)f32_to_bf16(acc[rt][3] * f) << 16);
      *reinterpret_cast<uint2*>(o + r) = make_uint2(lo, hi);
    }
  }
}

// rows: grid (ceil(tokens * heads / (16 NS WAVES))), 64 WAVES threads, the last pairs (the longest walks of a prompt) first
template <int RP, int KP, int NS, int WAVES, typename Q>
__global__ __launch_bounds__(64 * WAVES, 2) void latent_attention_rows_kernel(
    bf16_t* __restrict__ out, int64_t out_t, int64_t out_h, const Q* __restrict__ qa, int64_t qa_t, int64_t qa_h,
    const bf16_t* __restrict__ c_pages, const int32_t* __restrict__ block_table, int table_width,
    const int32_t* __restrict__ token_entry, const int32_t* __restrict__ positions, const int32_t* __restrict__ cu,
    const float* __restrict__ sink, const float* __restrict__ gate, int tokens, int heads, int rank, int row, int ps_shift,
    int window, float scale2, int skip_singles) {
  extern __shared__ __attribute__((aligned(16))) unsigned char tiles_lds[];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int PAIRS = 16 * NS * WAVES;
  const int first = (int)(gridDim.x - 1 - blockIdx.x) * PAIRS;             // the workgroup's first pair
  const int pairs = tokens * heads, back = window > 0 ? window - 1 : LT_ALL;
  // a column's token (-1: none); worked out where it is needed, which costs less than the registers that would keep it
  auto token_of = [&](int k, int& h) {
    int pair = first + (wave * NS + k) * 16 + c;
    asm volatile("" : "+v"(pair));
    const int t = pair / heads;
    h = pair - t * heads;
    return pair < pairs ? t : -1;
  };
  bf16x8 qb[NS][KP / 32];
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    int h;
    const int t = token_of(k, h);
    lt_load_query<KP>(qb[k], qa + (int64_t)h * qa_h + (int64_t)(t < 0 ? 0 : t) * qa_t, row, g, t >= 0);
  }
  lt_fill_table<KP>(tiles_lds, row, 64 * WAVES);
  int t = first / heads;
  const int t_end = min(tokens - 1, (first + PAIRS - 1) / heads);
  while (t <= t_end) {                                   // request by request; the same for all lanes
    const int e = __builtin_amdgcn_readfirstlane(token_entry[t]);
    const int last = __builtin_amdgcn_readfirstlane(min(t_end, cu[e + 1] - 1));
    if (!(skip_singles && cu[e + 1] - cu[e] == 1)) {
      const int p0 = __builtin_amdgcn_readfirstlane(positions[t]), hi_max = __builtin_amdgcn_readfirstlane(positions[last]);
      const int lo_min = (window > 0 && p0 - window + 1 > 0) ? p0 - window + 1 : 0;
      f32x4 acc[NS][RP / 16];
      float m_run[NS], l_run[NS];
      int pos_c[NS];
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        m_run[k] = -INFINITY;
        l_run[k] = 0.f;
        int h;
        const int tc = token_of(k, h);
        pos_c[k] = tc >= t && tc <= last ? positions[tc] : -1;
#pragma unroll
        for (int rt = 0; rt < RP / 16; ++rt) acc[k][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      lt_walk<RP, KP, NS, WAVES>(acc, m_run, l_run, qb, tiles_lds, c_pages, block_table + (int64_t)e * table_width, row, ps_shift,
                             pos_c, back, lo_min, hi_max, (lo_min >> 5) << 5, hi_max, scale2, wave, c, g);
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        float l = l_run[k];
        l = add_across_16(l);
        l = add_across_32(l);
        int h;
        const int tc = token_of(k, h);
        if (tc >= t && tc <= last)
          lt_store<RP>(out + (int64_t)h * out_h + (int64_t)tc * out_t, acc[k], lt_finish(m_run[k], l, sink, gate, tc, h, heads), rank, g);
      }
    }
    t = last + 1;
  }
}

// heads: grid (single tokens, ceil(heads / (16 WAVES)), splits), 64 WAVES threads; info: int32 x 4 per token = (row of the
// step, position, entry, -).  splits == 1: the result goes to out; else the split's unnormalised O (ws_o: [token][head]
// [split][RP] floats) and (maximum, sum) (ws_ml) for the merge kernel.
template <int RP, int KP, int WAVES, typename Q>
__global__ __launch_bounds__(64 * WAVES, 2) void latent_attention_heads_kernel(
    bf16_t* __restrict__ out, int64_t out_t, int64_t out_h, float* __restrict__ ws_o, float* __restrict__ ws_ml,
    const Q* __restrict__ qa, int64_t qa_t, int64_t qa_h, const bf16_t* __restrict__ c_pages,
    const int32_t* __restrict__ block_table, int table_width, const int32_t* __restrict__ info, const float* __restrict__ sink,
    const float* __restrict__ gate, int heads, int rank, int row, int ps_shift, int window, float scale2, int splits,
    int tiles_per_split) {
  extern __shared__ __attribute__((aligned(16))) unsigned char tiles_lds[];
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = (blockIdx.y * WAVES + wave) * 16 + c;
  const int n = blockIdx.x, t = info[4 * n], pos = info[4 * n + 1], e = info[4 * n + 2], z = blockIdx.z;
  const bool head_ok = h < heads;
  const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  bf16x8 qb[1][KP / 32];
  lt_load_query<KP>(qb[0], qa + (int64_t)(head_ok ? h : 0) * qa_h + (int64_t)t * qa_t, row, g, head_ok);
  lt_fill_table<KP>(tiles_lds, row, 64 * WAVES);
  f32x4 acc[1][RP / 16];
  float m_run[1] = {-INFINITY}, l_run[1] = {0.f};
#pragma unroll
  for (int rt = 0; rt < RP / 16; ++rt) acc[0][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int first = ((lo >> 5) + z * tiles_per_split) << 5;
  int last = first + 32 * (tiles_per_split - 1);
  if (last > pos || splits == 1) last = pos;            // the walk takes every tile that starts at or before `last`
  const int pos_c[1] = {head_ok ? pos : -1}, back = window > 0 ? window - 1 : LT_ALL;
  lt_walk<RP, KP, 1, WAVES>(acc, m_run, l_run, qb, tiles_lds, c_pages, block_table + (int64_t)e * table_width, row, ps_shift,
                            pos_c, back, lo, pos, first, last, scale2, wave, c, g);
  float l = l_run[0];
  l = add_across_16(l);
  l = add_across_32(l);
  if (!head_ok) return;
  if (splits == 1) {
    lt_store<RP>(out + (int64_t)h * out_h + (int64_t)t * out_t, acc[0], lt_finish(m_run[0], l, sink, gate, t, h, heads), rank, g);
    return;
  }
  const int64_t slot = ((int64_t)n * heads + h) * splits + z;
  if (g == 0) {
    ws_ml[2 * slot] = m_run[0];
    ws_ml[2 * slot + 1] = l;
  }
#pragma unroll
  for (int rt = 0; rt < RP / 16; ++rt)
    *reinterpret_cast<float4*>(ws_o + slot * RP + 16 * rt + 4 * g) = make_float4(acc[0][rt][0], acc[0][rt][1], acc[0][rt][2], acc[0][rt][3]);
}

// merges the splits of a single token's heads: grid (tokens, heads, ceil(rank / 64)), 64 threads; at most 64 splits.  Lane z works
// out split z's weight once; every lane then adds its coordinate over the splits, eight loads under way at a time.
__global__ __launch_bounds__(64) void latent_attention_merge_kernel(bf16_t* __restrict__ out, int64_t out_t, int64_t out_h,
                                                                    const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                                    const int32_t* __restrict__ info, const float* __restrict__ sink,
                                                                    const float* __restrict__ gate, int heads, int rank, int rp,
                                                                    int splits) {
  const int n = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, r = blockIdx.z * 64 + lane;
  const int t = info[4 * n];
  const int64_t base = ((int64_t)n * heads + h) * splits;
  const float* o_at = ws_o + base * rp + (r < rank ? r : 0);
  const float m = lane < splits ? ws_ml[2 * (base + lane)] : -INFINITY;
  const float l = lane < splits ? ws_ml[2 * (base + lane) + 1] : 0.f;
  constexpr int U = 8;
  float v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = u < splits ? o_at[(int64_t)u * rp] : 0.f;
  const float s2 = sink ? sink[h] * LT_LOG2E : -INFINITY;
  const float top = fmaxf(wave_max(m), s2);
  const float wz = (m == -INFINITY) ? 0.f : exp2f(m - top);
  const float den = wave_sum(wz * l) + (sink ? exp2f(s2 - top) : 0.f);
  const float f = (gate ? gate[(int64_t)t * heads + h] : 1.f) / den;
  float o = 0.f;
  for (int z = 0; z < splits; z += U) {
    float next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) next[u] = z + U + u < splits ? o_at[(int64_t)(z + U + u) * rp] : 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      o += __shfl(wz, (z + u) & 63, WAVE) * v[u];      // splits behind the last have no sum and no weight
      v[u] = next[u];
    }
  }
  if (r < rank) out[(int64_t)h * out_h + (int64_t)t * out_t + r] = f32_to_bf16(o * f);
}

static int lt_padded_rank(int rank, int row) {
  const int by_row = row - 64 > rank ? row - 64 : rank;        // a padded row is at most 64 longer than its padded rank
  return by_row <= 64 ? 64 : by_row <= 128 ? 128 : by_row <= 256 ? 256 : 512;
}

extern "C" int ga_latent_attention_mfma_padded_rank(int rank, int row) { return lt_padded_rank(rank, row); }

// what both entry points below ask of their operands
static bool lt_operands_ok(const void* out, int64_t out_t, int64_t out_h, const void* qa, int64_t qa_t, int64_t qa_h, int qa_bf16,
                           const void* c_pages, int heads, int rank, int row, int page_size, int table_width, int window) {
  const int q16 = qa_bf16 ? 8 : 4;                             // elements in 16 bytes
  return heads > 0 && rank > 0 && rank <= 512 && rank % 8 == 0 && row >= rank && row <= 576 && row % 8 == 0 && page_size >= 8 &&
         (page_size & (page_size - 1)) == 0 && (int64_t)page_size * row < (1 << 30) && table_width > 0 && window >= 0 &&
         qa_t % q16 == 0 && qa_h % q16 == 0 && out_t % 4 == 0 && out_h % 4 == 0 && ((uintptr_t)qa & 15) == 0 &&
         ((uintptr_t)out & 7) == 0 && ((uintptr_t)c_pages & 15) == 0;
}

#define LT_LAUNCH(KERNEL, KP, GRID, THREADS, ...)                                                                             \
  do {                                                                                                                        \
    constexpr int bytes = TileLayout<KP>::BYTES;                                                                                 \
    const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(&KERNEL),                                     \
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, bytes);                         \
    if (raised != hipSuccess) return (int)raised;                                                                             \
    hipLaunchKernelGGL((KERNEL), GRID, dim3(THREADS), bytes, stream, __VA_ARGS__);                                            \
  } while (0)

// Prompt portions (and, unless skip_singles, every token) on the matrix cores.  bfloat16; rank a multiple of 8 up to 512, row
// (what a cached token takes, at least rank) a multiple of 8 up to 576; page_size a power of two >= 8; qa rows (float, or
// bfloat16 where qa_bf16) 16-byte aligned.
template <int RP, int KP, typename Q>
static int lt_rows(void* out, int64_t out_t, int64_t out_h, const void* qa, int64_t qa_t, int64_t qa_h, const void* c_pages,
                   const void* block_table, int table_width, const void* token_entry, const void* positions, const void* cu,
                   const void* sink, const void* gate, int tokens, int heads, int rank, int row, int ps_shift, int window,
                   float scale2, int skip_singles, hipStream_t stream) {
  // two sets of columns a wavefront where the registers hold them beside the queries
  constexpr int NS = RP <= 128 ? 2 : 1, WAVES = 4, PAIRS = 16 * NS * WAVES;
  const int64_t blocks = ((int64_t)tokens * heads + PAIRS - 1) / PAIRS;
  if ((int64_t)tokens * heads > 0x7fffff00) return -2;
  LT_LAUNCH((latent_attention_rows_kernel<RP, KP, NS, WAVES, Q>), KP, dim3((unsigned)blocks), 64 * WAVES, (bf16_t*)out, out_t, out_h, (const Q*)qa, qa_t,
            qa_h, (const bf16_t*)c_pages, (const int32_t*)block_table, table_width, (const int32_t*)token_entry,
            (const int32_t*)positions, (const int32_t*)cu, (const float*)sink, (const float*)gate, tokens, heads, rank, row, ps_shift,
            window, scale2, skip_singles);
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_latent_attention_rows(void* out, int64_t out_t, int64_t out_h, const void* qa, int64_t qa_t, int64_t qa_h, int qa_bf16,
                                        const void* c_pages, const void* block_table, int table_width, const void* token_entry,
                                        const void* positions, const void* cu, const void* sink, const void* gate, int tokens,
                                        int heads, int rank, int row, int page_size, int window, float scale, int skip_singles,
                                        hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (!lt_operands_ok(out, out_t, out_h, qa, qa_t, qa_h, qa_bf16, c_pages, heads, rank, row, page_size, table_width, window)) return -1;
  const int rp = lt_padded_rank(rank, row);
#define GO(RP, KP, Q) return lt_rows<RP, KP, Q>(out, out_t, out_h, qa, qa_t, qa_h, c_pages, block_table, table_width, token_entry,   \
                                                positions, cu, sink, gate, tokens, heads, rank, row, __builtin_ctz(page_size),     \
                                                window, scale * LT_LOG2E, skip_singles, stream)
#define GK(RP, KP) do { if (qa_bf16) GO(RP, KP, bf16_t); else GO(RP, KP, float); } while (0)
#define GR(RP) do { if (row <= RP) GK(RP, RP); else GK(RP, (RP + 64)); } while (0)
  if (rp == 64) GR(64);
  else if (rp == 128) GR(128);
  else if (rp == 256) GR(256);
  else GR(512);
#undef GR
#undef GK
#undef GO
}

// Single tokens on the matrix cores; info int32 [n][4].  splits > 1: ws_o n * heads * splits * padded rank floats, ws_ml
// n * heads * splits * 2 floats; every token's keys are dealt to `splits` workgroups of tiles_per_split tiles of 32 each
// (splits * tiles_per_split must cover the longest walk: the window, or the longest context, in tiles, plus one).
template <int RP, int KP, int WAVES, typename Q>
static int lt_heads(void* out, int64_t out_t, int64_t out_h, void* ws_o, void* ws_ml, const void* qa, int64_t qa_t, int64_t qa_h,
                    const void* c_pages, const void* block_table, int table_width, const void* info, int n, const void* sink,
                    const void* gate, int heads, int rank, int row, int ps_shift, int window, float scale2, int splits,
                    int tiles_per_split, hipStream_t stream) {
  const dim3 grid(n, (heads + 16 * WAVES - 1) / (16 * WAVES), splits);
  LT_LAUNCH((latent_attention_heads_kernel<RP, KP, WAVES, Q>), KP, grid, 64 * WAVES, (bf16_t*)out, out_t, out_h, (float*)ws_o, (float*)ws_ml,
            (const Q*)qa, qa_t, qa_h, (const bf16_t*)c_pages, (const int32_t*)block_table, table_width, (const int32_t*)info,
            (const float*)sink, (const float*)gate, heads, rank, row, ps_shift, window, scale2, splits, tiles_per_split);
  return GA_CHECK_LAUNCH();
}

extern "C" int ga_latent_attention_heads(void* out, int64_t out_t, int64_t out_h, void* ws_o, void* ws_ml, const void* qa,
                                         int64_t qa_t, int64_t qa_h, int qa_bf16, const void* c_pages, const void* block_table,
                                         int table_width, const void* info, int n, const void* sink, const void* gate, int heads,
                                         int rank, int row, int page_size, int window, float scale, int splits,
                                         int tiles_per_split, hipStream_t stream) {
  if (n <= 0) return 0;
  if (!lt_operands_ok(out, out_t, out_h, qa, qa_t, qa_h, qa_bf16, c_pages, heads, rank, row, page_size, table_width, window) ||
      splits < 1 || splits > 64 || tiles_per_split < 1 || (splits > 1 && (ws_o == nullptr || ws_ml == nullptr)) || heads > 65535)
    return -1;
  const int rp = lt_padded_rank(rank, row);
  int rc = 0;
#define GO(RP, KP, WV, Q) rc = lt_heads<RP, KP, WV, Q>(out, out_t, out_h, ws_o, ws_ml, qa, qa_t, qa_h, c_pages, block_table, table_width,  \
                                                       info, n, sink, gate, heads, rank, row, __builtin_ctz(page_size), window,      \
                                                       scale * LT_LOG2E, splits, tiles_per_split, stream)
#define GW(RP, KP, Q) do { if (heads <= 32) GO(RP, KP, 2, Q); else GO(RP, KP, 4, Q); } while (0)
#define GK(RP, KP) do { if (qa_bf16) GW(RP, KP, bf16_t); else GW(RP, KP, float); } while (0)
#define GR(RP) do { if (row <= RP) GK(RP, RP); else GK(RP, (RP + 64)); } while (0)
  if (rp == 64) GR(64);
  else if (rp == 128) GR(128);
  else if (rp == 256) GR(256);
  else GR(512);
#undef GR
#undef GK
#undef GW
#undef GO
  if (rc != 0 || splits == 1) return rc;
  hipLaunchKernelGGL(latent_attention_merge_kernel, dim3(n, heads, (rank + 63) / 64), dim3(64), 0, stream, (bf16_t*)out, out_t, out_h,
                     (const float*)ws_o, (const float*)ws_ml, (const int32_t*)info, (const float*)sink, (const float*)gate,
                     heads, rank, rp, splits);
  return GA_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------------------------------- few rows
// The products of a head's up-projections with up to 64 tokens (bfloat16), around the attention of a decode step:
//   query   qa[h][t][n] = Wuk_h[n] . q[t][h] for the plain coordinates, and in the same launch (workgroups behind the products')
//           what latent_turned_prepare does: the queries' turned parts and the cached rows.  Both read the layer's one projection.
//   output  o[t][h][n] = Wuv_h[n] . a[h][t], times sigmoid of the gate's column where there is one.
// A wavefront takes 16 rows n of one head's matrix (w [head][rows][K], K a multiple of 8) against all tokens, 16 at a time as
// columns; the sums are 32-bit and their order depends on K alone.
template <int NT>
__device__ __forceinline__ void lf_product(f32x4 (&acc)[NT], const bf16_t* __restrict__ w, const bf16_t* const (&x)[NT], int K, int g) {
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int STEPS = 4;                          // operands of 128 elements of K asked for at a time
  for (int k0 = 0; k0 < K; k0 += 32 * STEPS) {
    bf16x8 a[STEPS], b[STEPS][NT];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int k = k0 + 32 * s + 8 * g;
      const bool in = k < K;
      a[s] = in ? __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(w + k)) : lt_zero8();
#pragma unroll
      for (int n = 0; n < NT; ++n) b[s][n] = in ? __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(x[n] + k)) : lt_zero8();
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], b[s][n], acc[n], 0, 0, 0);
  }
}

__device__ __forceinline__ void lf_store4(bf16_t* p, const float (&v)[4], int left, bool wide) {
  if (wide) {
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                                              (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < left) p[i] = f32_to_bf16(v[i]);
  }
}

template <int NT>
__global__ __launch_bounds__(256) void latent_query_few_kernel(
    bf16_t* __restrict__ qa, bf16_t* __restrict__ c_pages, const bf16_t* __restrict__ proj, int64_t proj_stride, int down_start,
    const bf16_t* __restrict__ w_uk, const float* __restrict__ wkv, const int32_t* __restrict__ positions,
    const float* __restrict__ cosines, const float* __restrict__ sines, const int64_t* __restrict__ slot_mapping, int tokens, int heads,
    int dim, int turned, int dims, int neighbours, int rank, float eps, int write, int product_groups) {
  __shared__ float scratch[4];
  const int rank8 = (rank + 7) & ~7, turned8 = (turned + 7) & ~7, row = rank8 + turned8;
  if ((int)blockIdx.x < product_groups) {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, blocks = (rank8 + 15) / 16;
    const int task = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (task >= heads * blocks) return;
    const int h = task / blocks, n0 = (task - h * blocks) * 16;
    const int wr = n0 + c < rank8 ? n0 + c : rank8 - 1;
    const bf16_t* x[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) x[n] = proj + (int64_t)(16 * n + c < tokens ? 16 * n + c : 0) * proj_stride + h * (dim + turned);
    f32x4 acc[NT];
    lf_product<NT>(acc, w_uk + ((int64_t)h * rank8 + wr) * dim, x, dim, g);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int t = 16 * n + c, r = n0 + 4 * g;
      if (t < tokens && r < rank8) {
        const float v[4] = {acc[n][0], acc[n][1], acc[n][2], acc[n][3]};
        lf_store4(qa + ((int64_t)h * tokens + t) * row + r, v, 4, true);
      }
    }
    return;
  }
  // workgroup 0 of a token: the cached row; the others: 256 elements each of the heads' turned parts
  const int parts = 1 + (heads * turned8 + 255) / 256, id = blockIdx.x - product_groups;
  const int64_t t = id / parts;
  const int part = id - (int)t * parts;
  const bf16_t* p = proj + t * proj_stride;
  const int half = dims >> 1;
  const float* cs = cosines + (int64_t)positions[t] * half;
  const float* sn = sines + (int64_t)positions[t] * half;
  if (part > 0) {
    const int i = (part - 1) * 256 + threadIdx.x;
    if (i >= heads * turned8) return;
    const int h = i / turned8, j = i - h * turned8;
    const bf16_t* q = p + h * (dim + turned) + dim;
    float v = 0.f;
    if (j < turned) v = la_turned<bf16_t>([&](int x) { return Num<bf16_t>::ld(q + x); }, j, dims, neighbours, cs, sn);
    qa[((int64_t)h * tokens + t) * row + rank8 + j] = f32_to_bf16(v);
    return;
  }
  const int64_t slot = slot_mapping[t];
  if (!write || slot < 0) return;                     // uniform over the workgroup
  la_write_row<bf16_t>(c_pages + slot * row, p + down_start, wkv, cs, sn, turned, dims, neighbours, rank, eps, scratch);
}

template <int NT>
__global__ __launch_bounds__(256) void latent_output_few_kernel(bf16_t* __restrict__ o, const bf16_t* __restrict__ a,
                                                                const bf16_t* __restrict__ w_uv, const bf16_t* __restrict__ gate,
                                                                int64_t gate_stride, int tokens, int heads, int vdim, int rank8) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, blocks = (vdim + 15) / 16;
  const int task = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (task >= heads * blocks) return;
  const int h = task / blocks, n0 = (task - h * blocks) * 16;
  const int wr = n0 + c < vdim ? n0 + c : vdim - 1;
  const bf16_t* x[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) x[n] = a + ((int64_t)h * tokens + (16 * n + c < tokens ? 16 * n + c : 0)) * rank8;
  f32x4 acc[NT];
  lf_product<NT>(acc, w_uv + ((int64_t)h * vdim + wr) * rank8, x, rank8, g);
  const int r = n0 + 4 * g;
  if (r >= vdim) return;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int t = 16 * n + c;
    if (t >= tokens) continue;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = acc[n][i];
      // rounded before the gate, as where the product is the library's and the gate a launch of its own
      if (gate && r + i < vdim)
        v[i] = bf16_to_f32(f32_to_bf16(v[i])) / (1.0f + expf(-Num<bf16_t>::ld(gate + (int64_t)t * gate_stride + h * vdim + r + i)));
    }
    lf_store4(o + ((int64_t)t * heads + h) * vdim + r, v, vdim - r, vdim % 4 == 0);
  }
}

// qa [heads][tokens][row] whole: the products of w_uk [heads][rank8][dim] (zeros behind the rank) and the turned parts; the cached rows
// where `write`.  tokens <= 64; dim, turned and proj_stride multiples of 8, operands at 16-byte addresses.
extern "C" int ga_latent_query_few(void* qa, void* c_pages, const void* proj, int64_t proj_stride, int down_start, const void* w_uk,
                                   const void* wkv, const void* positions, const void* cosines, const void* sines,
                                   const void* slot_mapping, int tokens, int heads, int dim, int turned, int dims, int neighbours,
                                   int rank, float eps, int write, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (tokens > 64 || heads <= 0 || dim <= 0 || dim % 8 || turned <= 0 || turned % 8 || dims < 0 || dims % 2 || dims > turned || rank <= 0 ||
      proj_stride % 8 || down_start < 0 || (write && (!wkv || !c_pages)) || (((uintptr_t)qa | (uintptr_t)proj | (uintptr_t)w_uk) & 15))
    return -1;
  const int rank8 = (rank + 7) & ~7, products = (heads * ((rank8 + 15) / 16) + 3) / 4;
  const int parts = 1 + (heads * turned + 255) / 256;
  const dim3 grid(products + tokens * parts), block(256);
#define GO(NT) hipLaunchKernelGGL(latent_query_few_kernel<NT>, grid, block, 0, stream, (bf16_t*)qa, (bf16_t*)c_pages, (const bf16_t*)proj,  \
                                  proj_stride, down_start, (const bf16_t*)w_uk, (const float*)wkv, (const int32_t*)positions,          \
                                  (const float*)cosines, (const float*)sines, (const int64_t*)slot_mapping, tokens, heads, dim, turned, \
                                  dims, neighbours, rank, eps, write, products)
  if (tokens <= 16) GO(1); else if (tokens <= 32) GO(2); else GO(4);
#undef GO
  return GA_CHECK_LAUNCH();
}

// o [tokens][heads][vdim] from a [heads][tokens][rank8] and w_uv [heads][vdim][rank8]; gate: null, or the first gate column of the first
// token, rows gate_stride elements apart.  tokens <= 64; rank8 a multiple of 8, a and w_uv at 16-byte addresses.
extern "C" int ga_latent_output_few(void* o, const void* a, const void* w_uv, const void* gate, int64_t gate_stride, int tokens, int heads,
                                    int vdim, int rank8, hipStream_t stream) {
  if (tokens <= 0) return 0;
  if (tokens > 64 || heads <= 0 || vdim <= 0 || rank8 <= 0 || rank8 % 8 || (((uintptr_t)a | (uintptr_t)w_uv) & 15) || ((uintptr_t)o & 7))
    return -1;
  const dim3 grid((heads * ((vdim + 15) / 16) + 3) / 4), block(256);
#define GO(NT) hipLaunchKernelGGL(latent_output_few_kernel<NT>, grid, block, 0, stream, (bf16_t*)o, (const bf16_t*)a, (const bf16_t*)w_uv,  \
                                  (const bf16_t*)gate, gate_stride, tokens, heads, vdim, rank8)
  if (tokens <= 16) GO(1); else if (tokens <= 32) GO(2); else GO(4);
#undef GO
  return GA_CHECK_LAUNCH();
}
