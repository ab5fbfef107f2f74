// Latent attention: the kernels around the attention proper.
//
//   latent_prepare   a token's down-projected row [query latent | key/value latent | key part to turn] -> the RMS
//                    norm of the query latent; the RMS norm of the key/value latent and the turned key part into
//                    the token's cache cell (K page: [latent | turned part], V page, transposed: the latent), and,
//                    if asked for, the heads' query parts turned into their places beside the latent-space queries
//   rotate_heads     a part of every head's row turned by position into another matrix
//   head_gemm        one product per head on the matrix cores (queries into the latent space, attended latents out), with
//                    rotate_heads beside it if asked for
//
// Norms, angles, sines and the turn itself are float32 whatever the activations are.
#include "mfma_tile.h"

// The cosines and sines of a token's turns (times the encoding's magnitude), once for all heads: [rotary_dim / 2] each
// in LDS.  Every thread of the workgroup calls it, and a barrier stands between it and the first use.
#define TURN_MAX_PAIRS 512

__device__ __forceinline__ void lay_turns(float* cosines, float* sines, int rotary_dim, const float* __restrict__ inv_freq,
                                          float position, float magnitude) {
  for (int i = threadIdx.x; i < rotary_dim / 2; i += blockDim.x) {
    float s, c;
    sincosf(position * inv_freq[i], &s, &c);
    cosines[i] = c * magnitude;
    sines[i] = s * magnitude;
  }
}

// Element j of a row of `width` numbers after the turn of its first `rotary_dim`: the pair (u, v) becomes
// (u cos - v sin, v cos + u sin); pairs are (2i, 2i + 1) (interleaved) or (i, i + rotary_dim / 2).
template <typename T>
__device__ __forceinline__ float turned_element(const T* row, int j, int rotary_dim, int interleaved, const float* cosines,
                                                const float* sines) {
  const float own = to_float(row[j]);
  if (j >= rotary_dim) return own;
  const int half = rotary_dim / 2;
  const bool is_first = interleaved ? (j & 1) == 0 : j < half;
  const int pair = interleaved ? j / 2 : is_first ? j : j - half;
  const int partner = interleaved ? (is_first ? j + 1 : j - 1) : (is_first ? j + half : j - half);
  const float other = to_float(row[partner]);
  return is_first ? own * cosines[pair] - other * sines[pair] : own * cosines[pair] + other * sines[pair];
}

// The heads' query parts to turn: element j of head h stands at rows[token * ld + col + h * head_stride + j] and goes to
// out[token * out_ld + out_col + h * out_head_stride + j].
template <typename T>
struct TurnedHeads {
  const T* rows;
  long ld;
  int col, head_stride, heads;
  T* out;
  long out_ld;
  int out_col, out_head_stride;
};

template <typename T>
__device__ __forceinline__ void turn_heads(const TurnedHeads<T>& t, long token, int width, int rotary_dim, int interleaved,
                                           const float* cosines, const float* sines) {
  for (int at = threadIdx.x; at < t.heads * width; at += blockDim.x) {
    const int head = at / width;
    const int j = at - head * width;
    const T* row = t.rows + token * t.ld + t.col + (long)head * t.head_stride;
    t.out[token * t.out_ld + t.out_col + (long)head * t.out_head_stride + j] =
        from_float<T>(turned_element(row, j, rotary_dim, interleaved, cosines, sines));
  }
}

// Two sums over the workgroup, each as block_sum forms it, behind one barrier.
__device__ __forceinline__ void block_sums(float& a, float& b, float (*scratch)[16]) {
  const int wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
  a = wave_sum(a);
  b = wave_sum(b);
  if (threadIdx.x % WAVE == 0) scratch[0][wave] = a, scratch[1][wave] = b;
  __syncthreads();
  a = b = 0.f;
  for (int i = 0; i < waves; ++i) a += scratch[0][i], b += scratch[1][i];
}

// Bound by its chain of round trips: position, cell and the row in one, one barrier for both sums, the stores.  (Sum by sum, each
// element read again behind its sum and the cell last: of 12 rows of 512 + 128 + 32 6.4 us, now 5.9; of 1,554 rows 9.2, now
// 8.3.)
template <typename T>
__global__ void __launch_bounds__(256)
latent_prepare_kernel(const T* __restrict__ down, long ld, int q_rank, int kv_rank, int rope_dim,
                      const float* __restrict__ q_norm, const float* __restrict__ kv_norm, float eps,
                      const int* __restrict__ positions, const float* __restrict__ inv_freq, int rotary_dim,
                      int interleaved, float magnitude, const int* __restrict__ slot_mapping, T* __restrict__ k_cache,
                      T* __restrict__ v_cache, long page_stride, int page_size, T* __restrict__ q_latent, long q_ld,
                      TurnedHeads<T> queries) {
  __shared__ float scratch[2][16];
  __shared__ float cosines[TURN_MAX_PAIRS], sines[TURN_MAX_PAIRS];
  constexpr int KEPT = 4;                             // elements of each latent that a thread keeps, the rest is read twice
  const long token = blockIdx.x;
  const T* row = down + token * ld;
  const float position = (float)positions[token];
  const int cell = slot_mapping ? slot_mapping[token] : 0;
  float q_kept[KEPT], kv_kept[KEPT];
#pragma unroll
  for (int j = 0; j < KEPT; ++j) {
    const int i = threadIdx.x + j * blockDim.x;
    const float q = to_float(row[min(i, max(q_rank - 1, 0))]), kv = to_float(row[q_rank + min(i, kv_rank - 1)]);
    q_kept[j] = i < q_rank ? q : 0.f;
    kv_kept[j] = i < kv_rank ? kv : 0.f;
  }
  lay_turns(cosines, sines, rotary_dim, inv_freq, position, magnitude);
  float q_squares = 0.f, kv_squares = 0.f;
#pragma unroll
  for (int j = 0; j < KEPT; ++j) {
    q_squares += q_kept[j] * q_kept[j];
    kv_squares += kv_kept[j] * kv_kept[j];
  }
  for (int i = threadIdx.x + KEPT * blockDim.x; i < q_rank; i += blockDim.x) {
    const float v = to_float(row[i]);
    q_squares += v * v;
  }
  for (int i = threadIdx.x + KEPT * blockDim.x; i < kv_rank; i += blockDim.x) {
    const float v = to_float(row[q_rank + i]);
    kv_squares += v * v;
  }
  block_sums(q_squares, kv_squares, scratch);         // (its barrier also publishes the turns)
  if (q_rank > 0) {                                   // the same for every thread
    const float q_denominator = sqrtf(q_squares / (float)q_rank + eps);
    T* q_out = q_latent + token * q_ld;
#pragma unroll
    for (int j = 0; j < KEPT; ++j) {
      const int i = threadIdx.x + j * blockDim.x;
      if (i < q_rank) q_out[i] = from_float<T>(q_kept[j] / q_denominator * q_norm[i]);
    }
    for (int i = threadIdx.x + KEPT * blockDim.x; i < q_rank; i += blockDim.x)
      q_out[i] = from_float<T>(to_float(row[i]) / q_denominator * q_norm[i]);
  }
  const float kv_denominator = sqrtf(kv_squares / (float)kv_rank + eps);
  if (queries.rows) turn_heads(queries, token, rope_dim, rotary_dim, interleaved, cosines, sines);
  if (!slot_mapping) return;
  const long page = cell / page_size;
  const int offset = cell % page_size;
  const int width = kv_rank + rope_dim;
  T* k_cell = k_cache + page * page_stride + (long)offset * width;
  T* v_cell = v_cache + page * page_stride + offset;
  auto keep = [&](int i, float latent) {
    const T value = from_float<T>(latent / kv_denominator * kv_norm[i]);
    k_cell[i] = value;
    v_cell[(long)i * page_size] = value;
  };
#pragma unroll
  for (int j = 0; j < KEPT; ++j) {
    const int i = threadIdx.x + j * blockDim.x;
    if (i < kv_rank) keep(i, kv_kept[j]);
  }
  for (int i = threadIdx.x + KEPT * blockDim.x; i < kv_rank; i += blockDim.x) keep(i, to_float(row[q_rank + i]));
  const T* part = row + q_rank + kv_rank;
  for (int j = threadIdx.x; j < rope_dim; j += blockDim.x)
    k_cell[kv_rank + j] = from_float<T>(turned_element(part, j, rotary_dim, interleaved, cosines, sines));
}

// queries (q_rows null: none): q_heads parts of rope_dim numbers, turned like the key part into q_out.
extern "C" int mi_latent_prepare(const void* down, int dtype, long ld, int T, int q_rank, int kv_rank, int rope_dim,
                                 const float* q_norm, const float* kv_norm, float eps, const int* positions,
                                 const float* inv_freq, int rotary_dim, int interleaved, float magnitude,
                                 const int* slot_mapping, void* k_cache, void* v_cache, long page_stride, int page_size,
                                 void* q_latent, long q_ld, const void* q_rows, long q_rows_ld, int q_col,
                                 int q_head_stride, int q_heads, void* q_out, long q_out_ld, int q_out_col,
                                 int q_out_head_stride, hipStream_t stream) {
  // q_rank 0: the row holds no query latent (queries projected directly); q_norm and q_latent are then not read
  if (!down || !kv_norm || !positions || T <= 0 || q_rank < 0 || (q_rank > 0 && (!q_norm || !q_latent)) || kv_rank <= 0 || rope_dim < 0 ||
      ld < q_rank + kv_rank + rope_dim || q_ld < q_rank || rotary_dim < 0 || rotary_dim > rope_dim || rotary_dim % 2 ||
      (rotary_dim > 0 && !inv_freq) || (slot_mapping && (!k_cache || !v_cache || page_size <= 0)))
    return ERR_BAD_ARGUMENT;
  if (q_rows && (!q_out || q_heads <= 0 || q_col < 0 || q_out_col < 0 || q_head_stride < 0 || q_out_head_stride < 0 ||
                 q_rows_ld < q_col + (long)(q_heads - 1) * q_head_stride + rope_dim ||
                 q_out_ld < q_out_col + (long)(q_heads - 1) * q_out_head_stride + rope_dim))
    return ERR_BAD_ARGUMENT;
  if (rotary_dim > 2 * TURN_MAX_PAIRS) return ERR_UNSUPPORTED_SIZE;
#define PREPARE_LAUNCH(T_)                                                                                          \
  latent_prepare_kernel<T_><<<T, 256, 0, stream>>>(                                                                 \
      (const T_*)down, ld, q_rank, kv_rank, rope_dim, q_norm, kv_norm, eps, positions, inv_freq, rotary_dim, interleaved, \
      magnitude, slot_mapping, (T_*)k_cache, (T_*)v_cache, page_stride, page_size, (T_*)q_latent, q_ld,             \
      TurnedHeads<T_>{(const T_*)q_rows, q_rows_ld, q_col, q_head_stride, q_heads, (T_*)q_out, q_out_ld, q_out_col, \
                      q_out_head_stride})
  if (dtype == DT_F32) PREPARE_LAUNCH(float);
  else if (dtype == DT_BF16) PREPARE_LAUNCH(bf16_t);
  else return ERR_BAD_ARGUMENT;
#undef PREPARE_LAUNCH
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// the query parts alone
template <typename T>
__global__ void rotate_heads_kernel(TurnedHeads<T> heads, int width, const int* __restrict__ positions,
                                    const float* __restrict__ inv_freq, int rotary_dim, int interleaved, float magnitude) {
  __shared__ float cosines[TURN_MAX_PAIRS], sines[TURN_MAX_PAIRS];
  const long token = blockIdx.x;
  lay_turns(cosines, sines, rotary_dim, inv_freq, (float)positions[token], magnitude);
  __syncthreads();
  turn_heads(heads, token, width, rotary_dim, interleaved, cosines, sines);
}

extern "C" int mi_rotate_heads(const void* x, int dtype, long ld, int col, int head_stride, int H, int width,
                               const int* positions, const float* inv_freq, int rotary_dim, int interleaved,
                               float magnitude, void* out, long out_ld, int out_col, int out_head_stride, int T,
                               hipStream_t stream) {
  if (!x || !out || !positions || T <= 0 || H <= 0 || width <= 0 || rotary_dim < 0 || rotary_dim > width ||
      rotary_dim % 2 || (rotary_dim > 0 && !inv_freq) || col < 0 || out_col < 0)
    return ERR_BAD_ARGUMENT;
  if (rotary_dim > 2 * TURN_MAX_PAIRS) return ERR_UNSUPPORTED_SIZE;
  const int threads = H * width >= 256 ? 256 : 64;
#define ROTATE_LAUNCH(T_)                                                                                           \
  rotate_heads_kernel<T_><<<T, threads, 0, stream>>>(                                                               \
      TurnedHeads<T_>{(const T_*)x, ld, col, head_stride, H, (T_*)out, out_ld, out_col, out_head_stride}, width,    \
      positions, inv_freq, rotary_dim, interleaved, magnitude)
  if (dtype == DT_F32) ROTATE_LAUNCH(float);
  else if (dtype == DT_BF16) ROTATE_LAUNCH(bf16_t);
  else return ERR_BAD_ARGUMENT;
#undef ROTATE_LAUNCH
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---------------------------------------------------------------- one product per head
// out[m, out_col + h * out_head_stride + n] = sum_k x[m, x_col + h * x_head_stride + k] * W[h, n, k]
// With turned.rows the launch has one slice of workgroups more, which turn the heads' position parts (as rotate_heads does,
// beside the products in place of behind them: it reads and writes other columns).  A decode step of 12 requests over 12
// layers 1,087 -> 1,077 us (a small launch of a graph costs 0.8 us a layer); 1,554 prompt tokens the same either way.
template <typename T>
struct HeadTurns {
  TurnedHeads<T> heads;             // rows null: none
  int width;
  const int* positions;
  const float* inv_freq;
  int rotary_dim, interleaved;
  float magnitude;
};

// The turns of tokens first .. last - 1 by one workgroup: as many tokens at a time as the LDS holds cosines and sines of.
template <typename T>
__device__ __forceinline__ void turn_tokens(const HeadTurns<T>& t, long first, long last) {
  __shared__ float cosines[TURN_MAX_PAIRS], sines[TURN_MAX_PAIRS];
  const int pairs = t.rotary_dim / 2;
  const int together = pairs > 0 ? TURN_MAX_PAIRS / pairs : TURN_MAX_PAIRS;
  const int each = t.heads.heads * t.width;
  for (long from = first; from < last; from += together) {
    const int count = (int)min((long)together, last - from);
    if (from > first) __syncthreads();
    for (int i = threadIdx.x; i < count * pairs; i += blockDim.x) {
      const int token = i / pairs;
      float s, c;
      sincosf((float)t.positions[from + token] * t.inv_freq[i - token * pairs], &s, &c);
      cosines[i] = c * t.magnitude;
      sines[i] = s * t.magnitude;
    }
    __syncthreads();
    // (two elements of a thread are read before the first is written: one round trip in place of two)
    for (int at0 = threadIdx.x; at0 < count * each; at0 += 2 * blockDim.x) {
      float value[2];
      T* to[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int at = min(at0 + u * (int)blockDim.x, count * each - 1);
        const int token = at / each;
        const int head = (at - token * each) / t.width;
        const int j = at - token * each - head * t.width;
        const T* row = t.heads.rows + (from + token) * t.heads.ld + t.heads.col + (long)head * t.heads.head_stride;
        value[u] = turned_element(row, j, t.rotary_dim, t.interleaved, cosines + token * pairs, sines + token * pairs);
        to[u] = t.heads.out + (from + token) * t.heads.out_ld + t.heads.out_col + (long)head * t.heads.out_head_stride + j;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (at0 + u * (int)blockDim.x < count * each) *to[u] = from_float<T>(value[u]);
    }
  }
}

template <typename T, int MT, bool VEC>
__global__ void __launch_bounds__(TILE_THREADS)
head_gemm_kernel(const T* __restrict__ x, long ldx, int x_col, const T* __restrict__ W, int x_head_stride,
                 int out_head_stride, T* out, long ldo, int out_col, int M, int N, int K, int heads, HeadTurns<T> turned) {
  __shared__ float red[TILE_WAVES][256];
  const int tid = threadIdx.x;
  const int r = (tid & (WAVE - 1)) % 16;
  const int head = blockIdx.z;
  const long n0 = (long)blockIdx.x * 16;
  const long m0 = (long)blockIdx.y * 16 * MT;
  if (head == heads) {                               // the slice that turns: its row of workgroups shares the rows of a tile
    const int share = (16 * MT + gridDim.x - 1) / gridDim.x;
    const long first = m0 + (long)blockIdx.x * share;
    turn_tokens(turned, first, min(min(first + share, m0 + 16 * MT), (long)M));
    return;
  }
  const T* w_row[1] = {W + ((long)head * N + min(n0 + r, (long)N - 1)) * K};
  const T* x_row[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    x_row[mt] = x + min(m0 + 16 * mt + r, (long)M - 1) * ldx + x_col + (long)head * x_head_stride;
  tile_floatx4 acc[1][MT];
  tile_accumulate<T, MT, 1, VEC>(w_row, x_row, K, acc);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const float value = tile_reduce(acc[0][mt], red);
    const int l = tid % 64;
    const long n = n0 + 4 * (l / 16) + tid / 64;
    const long m = m0 + 16 * mt + (l % 16);
    if (n < N && m < M) out[m * ldo + out_col + (long)head * out_head_stride + n] = from_float<T>(value);
  }
}

// The same for prompt portions in bfloat16 with K up to 32 CH <= 128 and whole groups of four features: a wave owns 16 rows and
// 32 features and all of K, asked for at once, so no sum crosses a wave, and a lane stores four neighbouring results.  The four
// runs of K that tile_accumulate deals to its waves are a chunk each here: added in their order the results are the same bits.
// What bounds it: a round trip for the fragments, the launch and the stores.  Eight heads of 1,554 rows, 64 -> 128 features with
// the turns and 128 -> 64 (2.4 MB read, 4 written): the tiles through LDS, two bytes a store, 11.4 us on
// average, this 7.7 and 5.4.  (The turns with eight tokens a workgroup in place of two: 9.3.)
template <int CH>
__global__ void __launch_bounds__(TILE_THREADS)
head_gemm_rows_kernel(const bf16_t* __restrict__ x, long ldx, int x_col, const bf16_t* __restrict__ W, int x_head_stride,
                      int out_head_stride, bf16_t* out, long ldo, int out_col, int M, int N, int K, int heads,
                      HeadTurns<bf16_t> turned) {
  typedef __bf16 four_t __attribute__((ext_vector_type(4)));
  const int head = blockIdx.z;
  const long m_block = (long)blockIdx.y * 16 * TILE_WAVES;
  if (head >= heads) {                               // the slices that turn share the rows of the workgroup's tiles
    const int parts = gridDim.x * (gridDim.z - heads);
    const int share = (16 * TILE_WAVES + parts - 1) / parts;
    const long first = m_block + (long)((head - heads) * (int)gridDim.x + (int)blockIdx.x) * share;
    turn_tokens(turned, first, min(min(first + share, m_block + 16 * TILE_WAVES), (long)M));
    return;
  }
  const int lane = threadIdx.x & (WAVE - 1);
  const int q = lane / 16, r = lane % 16;
  const long n0 = (long)blockIdx.x * 32;
  const long m = m_block + 16 * (threadIdx.x / WAVE) + r;
  const bf16_t* const x_row = x + min(m, (long)M - 1) * ldx + x_col + (long)head * x_head_stride;
  const bf16_t* const w_row[2] = {W + ((long)head * N + min(n0 + r, (long)N - 1)) * K,
                                  W + ((long)head * N + min(n0 + 16 + r, (long)N - 1)) * K};
  tile_bf16x8 a[CH][2], b[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    b[c] = tile_load<bf16_t, true>(x_row, 32 * c + 8 * q, K);
#pragma unroll
    for (int t = 0; t < 2; ++t) a[c][t] = tile_load<bf16_t, true>(w_row[t], 32 * c + 8 * q, K);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    tile_floatx4 sum;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const tile_floatx4 run = tile_mfma(a[c][t], b[c], tile_floatx4{0.f, 0.f, 0.f, 0.f});
      sum = c == 0 ? run : sum + run;
    }
    const long n = n0 + 16 * t + 4 * q;
    four_t packed;
#pragma unroll
    for (int i = 0; i < 4; ++i) packed[i] = (bf16_t)sum[i];
    if (n < N && m < M) *reinterpret_cast<four_t*>(out + m * ldo + out_col + (long)head * out_head_stride + n) = packed;
  }
}

template <typename T>
static int launch_head_gemm(const T* x, long ldx, int x_col, const T* W, int x_head_stride, int out_head_stride, T* out,
                            long ldo, int out_col, int M, int N, int K, int H, const HeadTurns<T>& turned, hipStream_t stream) {
  constexpr int PIECE = TileTraits<T>::PIECE;
  const bool vec = K % PIECE == 0 && ldx % PIECE == 0 && x_col % PIECE == 0 && x_head_stride % PIECE == 0 &&
                   ((unsigned long long)x % 16) == 0 && ((unsigned long long)W % 16) == 0;
  const int row_tiles = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const long blocks_y = ((long)M + 16 * row_tiles - 1) / (16 * row_tiles);
  const int slices = H + (turned.heads.rows ? 1 : 0);
  if (blocks_y > 65535 || slices > 65535) return ERR_UNSUPPORTED_SIZE;
  if constexpr (std::is_same<T, bf16_t>::value) {
    const int columns = (N + 31) / 32;
    const int turning = turned.heads.rows ? (32 + columns - 1) / columns : 0;    // two tokens or fewer a workgroup that turns
    if (row_tiles == 4 && vec && K <= 128 && N % 4 == 0 && ldo % 4 == 0 && out_col % 4 == 0 && out_head_stride % 4 == 0 &&
        ((unsigned long long)out % 8) == 0 && H + turning <= 65535) {
      const dim3 rows_grid((unsigned)columns, (unsigned)blocks_y, (unsigned)(H + turning));
#define HEAD_ROWS_LAUNCH(CH_)                                                                                         \
  head_gemm_rows_kernel<CH_><<<rows_grid, TILE_THREADS, 0, stream>>>(x, ldx, x_col, W, x_head_stride, out_head_stride, out, \
                                                                     ldo, out_col, M, N, K, H, turned)
      if (K <= 64) HEAD_ROWS_LAUNCH(2);
      else HEAD_ROWS_LAUNCH(4);
#undef HEAD_ROWS_LAUNCH
      return 0;
    }
  }
  const dim3 grid((unsigned)((N + 15) / 16), (unsigned)blocks_y, (unsigned)slices);
#define HEAD_LAUNCH(MT_, VEC_)                                                                                        \
  head_gemm_kernel<T, MT_, VEC_><<<grid, TILE_THREADS, 0, stream>>>(x, ldx, x_col, W, x_head_stride, out_head_stride, \
                                                                    out, ldo, out_col, M, N, K, H, turned)
#define HEAD_ROWS(MT_)                                                                                                \
  do {                                                                                                                \
    if (vec) HEAD_LAUNCH(MT_, true);                                                                                  \
    else HEAD_LAUNCH(MT_, false);                                                                                     \
  } while (0)
  if (row_tiles == 1) HEAD_ROWS(1);
  else if (row_tiles == 2) HEAD_ROWS(2);
  else HEAD_ROWS(4);
#undef HEAD_ROWS
#undef HEAD_LAUNCH
  return 0;
}

// positions not null: the heads' parts of `turn_width` numbers at x[m, turn_col + h * turn_head_stride] are turned into
// out[m, turn_out_col + h * turn_out_head_stride] too (columns that the products neither read nor write).
extern "C" int mi_head_gemm(const void* x, int dtype, long ldx, long x_col, const void* W, long x_head_stride,
                            long out_head_stride, void* out, long ldo, long out_col, int M, int N, int K, int H,
                            const int* positions, const float* inv_freq, int rotary_dim, int interleaved, float magnitude,
                            int turn_width, int turn_col, int turn_head_stride, int turn_out_col, int turn_out_head_stride,
                            hipStream_t stream) {
  if (!x || !W || !out || M <= 0 || N <= 0 || K <= 0 || H <= 0 || x_col < 0 || out_col < 0 || x_head_stride < 0 ||
      out_head_stride < 0 || ldx < x_col + (H - 1) * x_head_stride + K || ldo < out_col + (H - 1) * out_head_stride + N)
    return ERR_BAD_ARGUMENT;
  if (positions && (turn_width <= 0 || rotary_dim < 0 || rotary_dim > turn_width || rotary_dim % 2 || (rotary_dim > 0 && !inv_freq) ||
                    turn_col < 0 || turn_head_stride < 0 || turn_out_col < 0 || turn_out_head_stride < 0 ||
                    ldx < turn_col + (long)(H - 1) * turn_head_stride + turn_width ||
                    ldo < turn_out_col + (long)(H - 1) * turn_out_head_stride + turn_width))
    return ERR_BAD_ARGUMENT;
  if (positions && rotary_dim > 2 * TURN_MAX_PAIRS) return ERR_UNSUPPORTED_SIZE;
  int code;
#define HEAD_GEMM(T_)                                                                                                 \
  launch_head_gemm<T_>((const T_*)x, ldx, (int)x_col, (const T_*)W, (int)x_head_stride, (int)out_head_stride, (T_*)out, \
                       ldo, (int)out_col, M, N, K, H,                                                                 \
                       HeadTurns<T_>{{positions ? (const T_*)x : nullptr, ldx, turn_col, turn_head_stride, H, (T_*)out, ldo, \
                                      turn_out_col, turn_out_head_stride},                                            \
                                     turn_width, positions, inv_freq, rotary_dim, interleaved, magnitude},            \
                       stream)
  if (dtype == DT_F32) code = HEAD_GEMM(float);
  else if (dtype == DT_BF16) code = HEAD_GEMM(bf16_t);
  else return ERR_BAD_ARGUMENT;
#undef HEAD_GEMM
  if (code) return code;
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---------------------------------------------------------------- prompt portions on the matrix cores
// Attention of a step's prompt portions over the cached rows [latent | turned part] (DK wide, one row a token for
// all heads; the values are the first DV of them, kept a second time transposed as the V pages), bfloat16.  The
// queries are already in the latent space.  A workgroup takes 16 consecutive tokens of one lane and NSET heads,
// which share every key and value fragment; its eight waves split the keys [0, last position] in runs of whole
// 32-key steps and merge through LDS, set by set (the scheme of the grouped-query prompt kernel, with every head in
// the one group).  Softmax in float32, in units of log2; with `sinks` a head's exp(sink) joins the denominator where the
// waves' results are merged.  PADDED: the cached rows are `rank` + `turned` wide with rank a multiple of 16 up to DV and
// the sum a multiple of 8 up to DK; the kernel computes with DK and DV, the queries hold zeros past their width.
#include "attn_mfma.h"

#define LATENT_LOG2E 1.4426950408889634f

template <int DK, int DV, int NSET, int STEPS, bool PADDED, int LATENT_WAVES>
__global__ void __launch_bounds__(LATENT_WAVES * WAVE)
latent_attention_kernel(const bf16_t* __restrict__ q, long q_ld, int H, int rank, int turned,
                        const float* __restrict__ sinks, const bf16_t* __restrict__ k_base,
                        const bf16_t* __restrict__ v_base, long page_stride, int page_size,
                        const int* __restrict__ block_tables, int max_pages, const int* __restrict__ tiles,
                        const int* __restrict__ cu_seqlens, const int* __restrict__ start_pos, float scale, int window,
                        bf16_t* __restrict__ out, long out_ld) {
  constexpr int ITEMS = 2 + 4 * (DV / 16);                    // m, l and the accumulator of one set
  const int key_dim = PADDED ? rank + turned : DK;
  const int value_dim = PADDED ? rank : DV;
  __shared__ float part[LATENT_WAVES][ITEMS][WAVE];
  __shared__ int wave_pages[LATENT_WAVES][WAVE];
  // heavy tiles first; every other head pass the other way round
  const int block = (blockIdx.z & 1) ? blockIdx.x : gridDim.x - 1 - blockIdx.x;
  const int tile = block / 4;
  const int head0 = blockIdx.z * NSET;
  const int request = tiles[2 * tile];
  if (request < 0) return;                                    // a row of the table past the step's own runs
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int qd = lane / 16;
  const int n = lane % 16;
  const int lane_end = cu_seqlens[request + 1];
  const int first_token = tiles[2 * tile + 1] + 16 * (block % 4);
  if (first_token >= lane_end) return;                        // the whole workgroup
  const int token = first_token + n;
  const bool has_query = token < lane_end;
  const int base_position = start_pos[request] - cu_seqlens[request];
  const int position = base_position + token;
  const int last_position = base_position + min(first_token + 15, lane_end - 1);
  const int first_position = base_position + first_token;
  const bool full_tile = first_token + 16 <= lane_end && head0 + NSET <= H;

  mfma_bf16x8 q_frag[NSET][DK / 32];
  int col_pos[NSET];
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const bool valid = has_query && head0 + s < H;
    col_pos[s] = valid ? position : -1;
#pragma unroll
    for (int kk = 0; kk < DK / 32; ++kk) {
      if (valid && (!PADDED || 32 * kk + 8 * qd < key_dim)) {
        q_frag[s][kk] = *reinterpret_cast<const mfma_bf16x8*>(q + (long)token * q_ld + (long)(head0 + s) * key_dim +
                                                               32 * kk + 8 * qd);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) q_frag[s][kk][j] = (bf16_t)0.f;
      }
    }
  }
  AttnAccumulator<DK, NSET, DV> acc;
  acc.clear();
  AttnCache cache;
  cache.k_base = k_base;
  cache.v_base = v_base;
  cache.page_stride = page_stride;
  cache.page_size = page_size;
  cache.kvh = 0;
  cache.key_dim = key_dim;
  cache.value_dim = value_dim;
  const int* cache_pages = block_tables + (long)request * max_pages;
  int key_lo = 0;
  if (window > 0 && first_position - window + 1 > 0) key_lo = ((first_position - window + 1) / 32) * 32;
  const int key_hi = last_position + 1;
  const int steps = (key_hi - key_lo + 31) / 32;
  const int steps_per_wave = (steps + LATENT_WAVES - 1) / LATENT_WAVES;
  const int my_lo = key_lo + 32 * steps_per_wave * wave;
  const int my_hi = min(key_hi, my_lo + 32 * steps_per_wave);
  // the page ids of the run go through LDS, 64 pages at a time (a wave's own corner of it: no barrier)
  for (int part_lo = my_lo; part_lo < my_hi;) {
    const int first_page = part_lo / page_size;
    const int part_hi = min(my_hi, (first_page + WAVE) * page_size);
    wave_pages[wave][lane] = cache_pages[min(first_page + lane, max_pages - 1)];
    cache.pages = wave_pages[wave];
    cache.base_page = first_page;
    attend_keys<DK, NSET, STEPS, false, false, DV, false, PADDED, PADDED>(
        acc, q_frag, col_pos, window, scale, part_lo, part_hi, cache, full_tile ? first_position : -1, last_position);
    part_lo = part_hi;
  }

  // merge: set s is finished by wave s
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    __syncthreads();
    part[wave][0][lane] = acc.m[s];
    part[wave][1][lane] = acc.l[s];
#pragma unroll
    for (int dt = 0; dt < DV / 16; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) part[wave][2 + 4 * dt + i][lane] = acc.o[s][dt][i];
    __syncthreads();
    if (wave != s % LATENT_WAVES) continue;
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < LATENT_WAVES; ++w) m = fmaxf(m, part[w][0][lane]);
    const float sink = sinks ? sinks[min(head0 + s, H - 1)] * LATENT_LOG2E : -INFINITY;
    m = fmaxf(m, sink);
    float factor[LATENT_WAVES];
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < LATENT_WAVES; ++w) {
      const float m_w = part[w][0][lane];
      factor[w] = m_w == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_w - m);
      l += part[w][1][lane] * factor[w];
    }
    l += __shfl_xor(l, 16, WAVE);
    l += __shfl_xor(l, 32, WAVE);
    if (col_pos[s] < 0) continue;
    if (sinks) l += __builtin_amdgcn_exp2f(sink - m);
    const float inverse = 1.f / l;
    bf16_t* o = out + (long)token * out_ld + (long)(head0 + s) * value_dim;
#pragma unroll
    for (int dt = 0; dt < DV / 16; ++dt) {
      if (PADDED && 16 * dt >= value_dim) break;
      mfma_bf16x4 packed;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float value = 0.f;
#pragma unroll
        for (int w = 0; w < LATENT_WAVES; ++w) value += part[w][2 + 4 * dt + i][lane] * factor[w];
        packed[i] = (bf16_t)(value * inverse);
      }
      *reinterpret_cast<mfma_bf16x4*>(o + 16 * dt + 4 * qd) = packed;
    }
  }
}

// The widths the kernels are built for: (latent, turned part) as they are, and the widest that a PADDED form takes.
// most: how many heads share a fragment at most; waves: of a prompt workgroup.
#define LATENT_SHAPES(CASE)                                                                                        \
  CASE(32, 32, 4, 4) CASE(64, 32, 4, 2) CASE(64, 64, 4, 2) CASE(96, 32, 2, 2) CASE(128, 32, 2, 1) CASE(128, 64, 2, 1) \
  CASE(192, 64, 1, 1)
#define LATENT_PADDED_SHAPES(CASE)                                                                                 \
  CASE(32, 32, 4, 4, 8) CASE(64, 32, 4, 2, 8) CASE(96, 32, 2, 2, 8) CASE(128, 32, 2, 1, 8) CASE(128, 64, 2, 1, 8)  \
  CASE(192, 64, 1, 1, 8) CASE(256, 64, 1, 1, 4)

// whether (rank, turned) runs in the PADDED form of (RANK, TURNED)
static bool latent_fits(int rank, int turned, int RANK, int TURNED) {
  return rank > 0 && turned >= 0 && rank % 16 == 0 && (rank + turned) % 8 == 0 && rank <= RANK && rank + turned <= RANK + TURNED;
}

extern "C" int mi_latent_attention_supported(int rank, int turned) {
#define SUPPORTED_CASE(RANK_, TURNED_, ...) \
  if (latent_fits(rank, turned, RANK_, TURNED_)) return 1;
  LATENT_PADDED_SHAPES(SUPPORTED_CASE)
#undef SUPPORTED_CASE
  return 0;
}

template <int DK, int DV, int MOST, int STEPS, bool PADDED, int WAVES>
static int launch_latent_attention(const bf16_t* q, long q_ld, int H, int rank, int turned, const float* sinks,
                                   const bf16_t* k_base, const bf16_t* v_base, long page_stride, int page_size,
                                   const int* block_tables, int max_pages, const int* tiles, int n_tiles,
                                   const int* cu_seqlens, const int* start_pos, float scale, int window, bf16_t* out,
                                   long out_ld, hipStream_t stream) {
  const int passes = (H + MOST - 1) / MOST;
  const int per_pass = (H + passes - 1) / passes;
#define LATENT_LAUNCH(NSET_)                                                                                       \
  latent_attention_kernel<DK, DV, NSET_, STEPS, PADDED, WAVES>                                                     \
      <<<dim3(4 * n_tiles, 1, passes), WAVES * WAVE, 0, stream>>>(                                                \
          q, q_ld, H, rank, turned, sinks, k_base, v_base, page_stride, page_size, block_tables, max_pages, tiles, \
          cu_seqlens, start_pos, scale, window, out, out_ld)
  if (MOST >= 4 && per_pass > 2) LATENT_LAUNCH(MOST >= 4 ? 4 : 1);
  else if (MOST >= 2 && per_pass > 1) LATENT_LAUNCH(MOST >= 2 ? 2 : 1);
  else LATENT_LAUNCH(1);
#undef LATENT_LAUNCH
  return 0;
}

// tiles: int32 [n_tiles, 2] = (lane, first token row) of runs of up to 64 tokens of one lane; the step's own keys
// must be in the cache already.  sinks (optional): float32 [H].  ERR_UNSUPPORTED_SIZE for widths the kernel is not built for.
extern "C" int mi_latent_attention(const void* q, long q_ld, int H, int rank, int turned, const float* sinks,
                                   const void* k_base, const void* v_base, long page_stride, int page_size,
                                   const int* block_tables, int max_pages, const int* tiles, int n_tiles,
                                   const int* cu_seqlens, const int* start_pos, float scale, int window, void* out,
                                   long out_ld, hipStream_t stream) {
  if (!q || !k_base || !v_base || !block_tables || !tiles || !cu_seqlens || !start_pos || !out || n_tiles <= 0 || H <= 0 ||
      page_size <= 0 || max_pages <= 0)
    return ERR_BAD_ARGUMENT;
  if (page_size % 4 != 0 || q_ld % 8 != 0 || out_ld % 4 != 0 || ((unsigned long long)q % 16) != 0 ||
      ((unsigned long long)out % 8) != 0 || n_tiles > (1 << 28) || H > 65535)
    return ERR_UNSUPPORTED_SIZE;
#define LATENT_ARGUMENTS                                                                                           \
  (const bf16_t*)q, q_ld, H, rank, turned, sinks, (const bf16_t*)k_base, (const bf16_t*)v_base, page_stride, page_size, \
      block_tables, max_pages, tiles, n_tiles, cu_seqlens, start_pos, scale, window, (bf16_t*)out, out_ld, stream
#define LATENT_CASE(RANK_, TURNED_, MOST_, STEPS_)                                                                 \
  if (rank == RANK_ && turned == TURNED_) {                                                                        \
    launch_latent_attention<RANK_ + TURNED_, RANK_, MOST_, STEPS_, false, 8>(LATENT_ARGUMENTS);                    \
    RETURN_IF_LAUNCH_FAILED();                                                                                     \
    return 0;                                                                                                      \
  }
  LATENT_SHAPES(LATENT_CASE)
#undef LATENT_CASE
#define LATENT_CASE(RANK_, TURNED_, MOST_, STEPS_, WAVES_)                                                         \
  if (latent_fits(rank, turned, RANK_, TURNED_)) {                                                                 \
    launch_latent_attention<RANK_ + TURNED_, RANK_, MOST_, STEPS_, true, WAVES_>(LATENT_ARGUMENTS);                \
    RETURN_IF_LAUNCH_FAILED();                                                                                     \
    return 0;                                                                                                      \
  }
  LATENT_PADDED_SHAPES(LATENT_CASE)
#undef LATENT_CASE
#undef LATENT_ARGUMENTS
  return ERR_UNSUPPORTED_SIZE;
}

// ---------------------------------------------------------------- single decoded tokens, the context split
// For steps of single-token lanes in bfloat16: a wave takes one run of `split_keys` keys of one request and up to
// 16 heads, which are the columns of the matrix cores' products (all heads read the same cached rows, so a key or
// value fragment is fetched once for the sixteen); it leaves an unnormalized partial result with its maximum and
// normalizer (in units of log2), and a second kernel merges a token's runs in ascending order.  grid = (runs,
// tokens, sets of 16 heads), one wave a workgroup.  PADDED: as above.
template <int DK, int DV, int STEPS, bool PADDED>
__global__ void __launch_bounds__(WAVE)
latent_decode_kernel(const bf16_t* __restrict__ q, long q_ld, int H, int rank, int turned, const bf16_t* __restrict__ k_base,
                     const bf16_t* __restrict__ v_base, long page_stride, int page_size,
                     const int* __restrict__ block_tables, int max_pages, const int* __restrict__ lane_of_token,
                     const int* __restrict__ positions, float scale, int window, int split_keys, int splits,
                     float* __restrict__ partial_o, float* __restrict__ partial_ml) {
  const int key_dim = PADDED ? rank + turned : DK;
  const int value_dim = PADDED ? rank : DV;
  const int split = blockIdx.x;
  const long token = blockIdx.y;
  const int head0 = blockIdx.z * 16;
  const int pos = positions[token];
  int first_key = 0;
  if (window > 0 && pos - window + 1 > 0) first_key = pos - window + 1;
  const int range_lo = (first_key / 32) * 32 + split * split_keys;
  if (range_lo > pos) return;                                 // the merge knows which runs hold keys
  const int range_hi = min(range_lo + split_keys, pos + 1);
  const int lane = threadIdx.x & (WAVE - 1);
  const int qd = lane / 16;
  const int n = lane % 16;
  const int head = head0 + n;
  const bool valid = head < H;
  mfma_bf16x8 q_frag[1][DK / 32];
  int col_pos[1] = {valid ? pos : -1};
#pragma unroll
  for (int kk = 0; kk < DK / 32; ++kk) {
    if (valid && (!PADDED || 32 * kk + 8 * qd < key_dim)) {
      q_frag[0][kk] = *reinterpret_cast<const mfma_bf16x8*>(q + token * q_ld + (long)head * key_dim + 32 * kk + 8 * qd);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) q_frag[0][kk][j] = (bf16_t)0.f;
    }
  }
  AttnAccumulator<DK, 1, DV> acc;
  acc.clear();
  AttnCache cache;
  cache.k_base = k_base;
  cache.v_base = v_base;
  cache.page_stride = page_stride;
  cache.page_size = page_size;
  cache.kvh = 0;
  cache.pages = block_tables + (long)lane_of_token[token] * max_pages;
  cache.base_page = 0;
  cache.key_dim = key_dim;
  cache.value_dim = value_dim;
  attend_keys<DK, 1, STEPS, false, false, DV, false, PADDED, PADDED>(acc, q_frag, col_pos, window, scale, range_lo, range_hi,
                                                                     cache);
  const float l = attn_normalizer<DK, 1, DV>(acc, 0);
  if (!valid) return;
  const long at = (token * H + head) * splits + split;
  if (qd == 0) {
    partial_ml[2 * at] = acc.m[0];
    partial_ml[2 * at + 1] = l;
  }
#pragma unroll
  for (int dt = 0; dt < DV / 16; ++dt)
    if (!PADDED || 16 * dt < value_dim)
      *reinterpret_cast<mfma_floatx4*>(partial_o + at * value_dim + 16 * dt + 4 * qd) = acc.o[0][dt];
}

#define LATENT_MERGE_SPLITS 256
#define LATENT_MERGE_AT_ONCE 16

__global__ void latent_decode_merge_kernel(const float* __restrict__ partial_o, const float* __restrict__ partial_ml,
                                           const int* __restrict__ positions, int window, int split_keys, int splits,
                                           int H, int dv, const float* __restrict__ sinks, bf16_t* __restrict__ out,
                                           long out_ld) {
  __shared__ float factor[LATENT_MERGE_SPLITS];      // exp2(maximum of the run - maximum), 0 for a run without keys
  __shared__ float scratch[16];
  const long token = blockIdx.x;
  const int head = blockIdx.y;
  const float* ml = partial_ml + (token * H + head) * splits * 2;
  const float* o = partial_o + (token * H + head) * (long)splits * dv;
  // The first runs' results are asked for before it is known how many runs there are (a run past the last is not used, whatever
  // its place holds): one round trip in place of four (12 rows of
  // eight heads, up to 24 runs: 6.1 -> 4.5 us).
  const int own = min((int)threadIdx.x, splits - 1), own_dim = min((int)threadIdx.x, dv - 1);
  const float own_maximum = ml[2 * own], own_normalizer = ml[2 * own + 1];
  float ahead[LATENT_MERGE_AT_ONCE];
#pragma unroll
  for (int u = 0; u < LATENT_MERGE_AT_ONCE; ++u) ahead[u] = o[(long)min(u, splits - 1) * dv + own_dim];
  const float sink = sinks ? sinks[head] * LATENT_LOG2E : -INFINITY;
  const int pos = positions[token];
  int first_key = 0;
  if (window > 0 && pos - window + 1 > 0) first_key = pos - window + 1;
  const int used = min(splits, (pos - (first_key / 32) * 32) / split_keys + 1);
  float maximum = (int)threadIdx.x < used ? own_maximum : -INFINITY;
  for (int s = threadIdx.x + blockDim.x; s < used; s += blockDim.x) maximum = fmaxf(maximum, ml[2 * s]);
  maximum = wave_max(maximum);
  if ((threadIdx.x & (WAVE - 1)) == 0) scratch[threadIdx.x / WAVE] = maximum;
  __syncthreads();
  for (int w = 0; w < (int)(blockDim.x + WAVE - 1) / WAVE; ++w) maximum = fmaxf(maximum, scratch[w]);
  maximum = fmaxf(maximum, sink);
  float share = 0.f;
  for (int s = threadIdx.x; s < used; s += blockDim.x) {
    const float m = s == (int)threadIdx.x ? own_maximum : ml[2 * s];
    const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - maximum);
    factor[s] = f;
    share += f * (s == (int)threadIdx.x ? own_normalizer : ml[2 * s + 1]);
  }
  float denominator = block_sum(share, scratch);                 // (its barriers also publish the factors)
  if (sinks) denominator += __builtin_amdgcn_exp2f(sink - maximum);
  for (int dim = threadIdx.x; dim < dv; dim += blockDim.x) {
    float sum = 0.f;
    if (dim != (int)threadIdx.x) {                                // (wider values than threads)
#pragma unroll
      for (int u = 0; u < LATENT_MERGE_AT_ONCE; ++u) ahead[u] = o[(long)min(u, used - 1) * dv + dim];
    }
#pragma unroll
    for (int u = 0; u < LATENT_MERGE_AT_ONCE; ++u)
      if (u < used) sum = fmaf(factor[u], ahead[u], sum);
    for (int s0 = LATENT_MERGE_AT_ONCE; s0 < used; s0 += LATENT_MERGE_AT_ONCE) {      // so many runs asked for at once; past the last, the last again
      float value[LATENT_MERGE_AT_ONCE];
#pragma unroll
      for (int u = 0; u < LATENT_MERGE_AT_ONCE; ++u) value[u] = o[(long)min(s0 + u, used - 1) * dv + dim];
#pragma unroll
      for (int u = 0; u < LATENT_MERGE_AT_ONCE; ++u)
        if (s0 + u < used) sum = fmaf(factor[s0 + u], value[u], sum);
    }
    out[token * out_ld + (long)head * dv + dim] = (bf16_t)(sum / denominator);
  }
}

// partial_o: float32 [T, H, splits, rank]; partial_ml: float32 [T, H, splits, 2].  split_keys: a multiple of 32.
// sinks (optional): float32 [H].
extern "C" int mi_latent_decode_attention(const void* q, long q_ld, int T, int H, int rank, int turned, const float* sinks,
                                          const void* k_base, const void* v_base, long page_stride, int page_size,
                                          const int* block_tables, int max_pages, const int* lane_of_token,
                                          const int* positions, float scale, int window, int split_keys, int splits,
                                          float* partial_o, float* partial_ml, void* out, long out_ld,
                                          hipStream_t stream) {
  if (!q || !k_base || !v_base || !block_tables || !lane_of_token || !positions || !partial_o || !partial_ml || !out ||
      T <= 0 || H <= 0 || page_size <= 0 || max_pages <= 0 || splits <= 0 || split_keys <= 0)
    return ERR_BAD_ARGUMENT;
  if (page_size % 4 != 0 || q_ld % 8 != 0 || ((unsigned long long)q % 16) != 0 || split_keys % 32 != 0 || T > 65535 ||
      (H + 15) / 16 > 65535 || H > 65535 || splits > LATENT_MERGE_SPLITS)
    return ERR_UNSUPPORTED_SIZE;
  const dim3 grid(splits, T, (H + 15) / 16);
#define LATENT_DECODE_LAUNCH(RANK_, TURNED_, PADDED_)                                                              \
  do {                                                                                                             \
    latent_decode_kernel<RANK_ + TURNED_, RANK_, (RANK_ + TURNED_ <= 128 ? 2 : 1), PADDED_><<<grid, WAVE, 0, stream>>>( \
        (const bf16_t*)q, q_ld, H, rank, turned, (const bf16_t*)k_base, (const bf16_t*)v_base, page_stride, page_size, \
        block_tables, max_pages, lane_of_token, positions, scale, window, split_keys, splits, partial_o, partial_ml); \
    RETURN_IF_LAUNCH_FAILED();                                                                                     \
    latent_decode_merge_kernel<<<dim3(T, H), (rank + 63) / 64 * 64, 0, stream>>>(                                  \
        partial_o, partial_ml, positions, window, split_keys, splits, H, rank, sinks, (bf16_t*)out, out_ld);       \
    RETURN_IF_LAUNCH_FAILED();                                                                                     \
    return 0;                                                                                                      \
  } while (0)
#define LATENT_DECODE_CASE(RANK_, TURNED_, ...) \
  if (rank == RANK_ && turned == TURNED_) LATENT_DECODE_LAUNCH(RANK_, TURNED_, false);
  LATENT_SHAPES(LATENT_DECODE_CASE)
#undef LATENT_DECODE_CASE
#define LATENT_DECODE_CASE(RANK_, TURNED_, ...) \
  if (latent_fits(rank, turned, RANK_, TURNED_)) LATENT_DECODE_LAUNCH(RANK_, TURNED_, true);
  LATENT_PADDED_SHAPES(LATENT_DECODE_CASE)
#undef LATENT_DECODE_CASE
#undef LATENT_DECODE_LAUNCH
  return ERR_UNSUPPORTED_SIZE;
}
