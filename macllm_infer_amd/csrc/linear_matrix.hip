// Retention and the generalized delta rule for prompt portions in bfloat16, a run of N tokens at a time on the float32
// matrix cores (v_mfma_f32_16x16x4_f32: products and sums in float32, as in the walk of linear_state.hip):
//     retention    S_t = decay S_(t-1) + k_t v_t^T                                        o_t = S_t^T r_t
//     delta rule   S_t = diag(w_t) S_(t-1) - (a_t * u_t)(u_t^T S_(t-1)) + k_t v_t^T         o_t = S_t^T r_t
// Delta rule inside a run whose starting state is S: let d_t = w_1 * ... * w_t (channel by channel), and
//     B_t = d_(t-1) * u_t    A_t = a_t * u_t / d_t    K_t = k_t / d_t    R_t = d_t * r_t    (rows of N x dk matrices)
// Then S_t = diag(d_t) (S + sum_(s <= t) K_s v_s^T - A_s z_s^T) with z_t = B_t S + sum_(s < t) (B_t . K_s) v_s - (B_t . A_s) z_s,
// so with strict lower triangles L = B A^T and P = B K^T and the triangles RK = R K^T, RA = R A^T (diagonal included)
//     (I + L) [Zk | Zv] = [B | P V]            z = Zk S + Zv
//     O = Ro S + Ov                            Ro = R - RA Zk          Ov = RK V - RA Zv
//     S_end = M S + Nv                         M = diag(d_N)(I - A^T Zk)   Nv = diag(d_N)(K^T V - A^T Zv)
// Retention is the same without A, its powers of the decay laid on the triangle itself (a decay may be zero).
// Two kernels:
//     chunk   a workgroup a (run, head), all runs of a prompt side by side: Ro, M and Nv to memory, Ov to the outputs
//     carry   a workgroup a (lane of the step, head, 16 value channels) walks the lane's runs: O = Ov + Ro S, S <- M S + Nv
//             (retention: S <- decay^N S + Nv), the next runs' matrices on their way meanwhile
// Every w_t is at least exp(-decay_floor), and 1 / d_t at most exp(N decay_floor): the caller keeps that within float32.
// What is in float32 and what in 64 bits: states, operands and the products over tokens are float32.  The d_t are 64-bit
// products of the w_t, so that B, A, K, R (and A and K as they stand at the run's end, for M and Nv) are rounded once; the
// triangles, whose sums over all key channels are the longest, are summed in 64 bits (v_mfma_f64_16x16x4_f64) and rounded
// once; the sums over tokens run from the oldest to the newest, whose terms are as a rule the largest; the carry's sums
// over key channels are chains of 16.  Off 64 bits, in units of the result's norm, outputs and (states) of the walk and of
// this, 300 tokens: delta rule with 16 heads of 64 channels 1.01e-7 (7.4e-8) and 7.4e-8 (5.8e-8), decays near their floor
// of exp(-0.6) 8.4e-8 (4.8e-8) and 6.3e-8 (4.7e-8), near one 5.9e-7 (7.5e-7) and 1.9e-7 (2.1e-7), 8 heads of 128 channels
// 1.07e-7 (7.5e-8) and 7.5e-8 (5.9e-8); retention 3.0e-7 (3.5e-7) and 1.6e-7 (1.5e-7).  (All in float32, one chain a sum:
// 1.6e-7 (1.0e-7), 1.35e-7 (9.4e-8), 2.6e-7 (2.8e-7), 2.0e-7 (1.1e-7), 2.0e-7 (1.5e-7), and 98 instead of the 104 us below.)
// What bounds it: the chunk kernel its products (some 110 matrix instructions a value wave and run of 32 tokens) and the
// waits between its stages; the carry what one compute unit can fetch, 30 KB a run at 28 KB a microsecond, of M alone 16.
// 1,999 tokens, in microseconds with both kernels, the three passes of linear_state.hip and this: delta rule with 16
// heads of 64 channels 244 and 104, retention with 8 heads of 64 and 128 channels 125 and 48; 100 tokens, where the walk
// goes from end to end: 96 and 23, 63 and 21.
#include "common.h"
#include <cstdint>
#include <type_traits>

typedef float lm_floatx4 __attribute__((ext_vector_type(4)));
typedef double lm_doublex4 __attribute__((ext_vector_type(4)));

#define LM_RETENTION 0
#define LM_DELTA 1
#define LM_CHUNK_TOKENS 128         // a row of the table of chunks holds at most this many tokens
#define LM_PREP_WAVES 8             // waves of the chunk kernel that form B, A, K and R
#define LM_MOST_WAVES 16

struct LinearMatrixArgs {
  const bf16_t* u;                  // the projection's rows [T, ld]
  long ld;
  int r_col, k_col, v_col, removal_col;
  int H, dv;
  float* state;                     // [slots, H, dv, dk]
  const int* slot_ids;              // [lanes]
  const int* chunks;                // [chunks, 4] = (lane or -1, first row, tokens, index in the lane)
  const int* lane_chunks;           // [lanes, 2] = (first chunk, chunks)
  const float* head_decay;          // retention: [H]
  float key_scale;
  const int* positions;             // [T]
  const float* inv_freq;            // [rotary_dim / 2] or null
  int rotary_dim;
  const float* decay_logits;        // delta rule: [T, logits_ld]
  long logits_ld;
  const float* decay_bias;          // [H * dk]
  float decay_floor, key_eps;
  float* local;                     // [runs (lm_first_run), H, Ro | Nv | M]
  float* out;                       // [T, out_ld]
  long out_ld;
};

__device__ __forceinline__ float lm_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

__device__ __forceinline__ lm_floatx4 lm_mfma(const lm_floatx4& a, const lm_floatx4& b, lm_floatx4 acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
  return acc;
}

// the same with products and sums in 64 bits
__device__ __forceinline__ lm_doublex4 lm_mfma_double(const lm_floatx4& a, const lm_floatx4& b, lm_doublex4 acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[i], (double)b[i], acc, 0, 0, 0);
  return acc;
}

// 16 x 16 of a matrix in LDS as a left operand: row r, columns 4q .. 4q + 3 from `at` on (rows `stride` apart) ...
__device__ __forceinline__ lm_floatx4 lm_rows(const float* at, int stride, int q, int r) {
  return *reinterpret_cast<const lm_floatx4*>(at + r * stride + 4 * q);
}
// ... and of its transpose: column r, rows 4q .. 4q + 3 (also a right operand, whose index of the sum runs over rows)
__device__ __forceinline__ lm_floatx4 lm_columns(const float* at, int stride, int q, int r) {
  lm_floatx4 value;
#pragma unroll
  for (int i = 0; i < 4; ++i) value[i] = at[(4 * q + i) * stride + r];
  return value;
}

// The rows of LDS that belong to a tile of 16 tokens are permuted (row 4a + b is token 4b + a, and the other way round): one
// matrix instruction then sums four neighbouring tokens, and a product's chain runs from the oldest token to the newest.
__device__ __forceinline__ constexpr int lm_place(int at) { return (at & ~15) + 4 * (at & 3) + ((at >> 2) & 3); }

// acc + a tile on a triangle's diagonal (16 x 16 at `at`, zero above the diagonal, STRICT: and on it) times `right`.  A row
// of the result is a token's and takes the tokens up to its own (STRICT: before it); a later token's infinity or NaN must
// not reach it through a product with zero: such values stay out of the product and are added to their own rows.
template <bool STRICT>
__device__ __forceinline__ lm_floatx4 lm_diagonal(const float* at, int stride, int q, int r, const lm_floatx4& right, lm_floatx4 acc) {
  lm_floatx4 numbers;
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool number = __builtin_isfinite(right[i]);
    finite &= number;
    numbers[i] = number ? right[i] : 0.f;
  }
  acc = lm_mfma(lm_rows(at, stride, q, r), numbers, acc);
  if (__all(finite)) return acc;
#pragma unroll 1
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = 4 * g + j;
      const float value = __shfl(right[j], 16 * g + r, WAVE);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 4 * q + i;
        const bool sees = STRICT ? lm_place(s) < lm_place(t) : lm_place(s) <= lm_place(t);
        if (!__builtin_isfinite(value) && sees) acc[i] = fmaf(at[t * stride + s], value, acc[i]);
      }
    }
  return acc;
}

template <int KIND, int DK, int N>
static constexpr long lm_run_floats(int dv) { return (long)N * DK + (long)dv * DK + (KIND == LM_DELTA ? DK * DK : 0); }

// Where the runs of a lane that begins at token row `row` lie in the work area: a lane of n tokens has ceil(n / N) runs, and
// floor((row + n) / N) + lane + 1 is never before its last.  The area holds floor(tokens / N) + lanes of them.
template <int N>
__device__ __forceinline__ long lm_first_run(int lane, long row) { return row / N + lane; }

template <int KIND, int DK, int N>
static constexpr int lm_chunk_lds_floats() {
  constexpr int KS = DK + 4, TS = N + 4, T = N / 16;
  return KIND == LM_DELTA ? 4 * N * KS + 4 * N * TS + T * 16 * 20 + DK + 2 * LM_PREP_WAVES * DK : 2 * N * KS + N * TS + N + 4;
}

template <int KIND, int DK, int N>
__global__ void __launch_bounds__(LM_MOST_WAVES * WAVE) linear_matrix_chunk_kernel(const LinearMatrixArgs a) {
  constexpr bool DELTA = KIND == LM_DELTA;
  constexpr int KS = DK + 4, TS = N + 4;               // row strides in LDS: the four rows of 16 a wave reads lie in different banks
  constexpr int T = N / 16, KT = DK / 16;
  constexpr int RUNS = LM_CHUNK_TOKENS / N;
  constexpr int PT = N / LM_PREP_WAVES, PC = DK / WAVE; // tokens of a preparing wave, channels of a lane
  extern __shared__ __align__(16) float lds[];
  float* const K = lds;
  float* const R = K + N * KS;
  float* const RK = R + N * KS;
  float* const powers = RK + N * TS;                    // retention: decay^0 .. decay^N
  float* const RA = RK + N * TS;                        // delta rule
  float* const L = RA + N * TS;
  float* const P = L + N * TS;
  float* const B = P + N * TS;
  float* const A = B + N * KS;
  float* const inverse = A + N * KS;                    // [T][16][20]: the inverses of I + L's diagonal blocks
  float* const last = inverse + T * 16 * 20;            // d_N
  double* const products = reinterpret_cast<double*>(last + DK);   // [waves][DK]: of the waves' decays

  const int* row = a.chunks + 4 * (blockIdx.x / RUNS);
  if (row[0] < 0) return;                               // a row past the step's own chunks
  const int part = blockIdx.x % RUNS;
  const int count = min(N, row[2] - part * N);
  if (count <= 0) return;
  const long t0 = (long)row[1] + part * N;
  const int head = blockIdx.y;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = threadIdx.x / WAVE;
  const int waves = blockDim.x / WAVE;
  const int q = lane / 16;
  const int r = lane % 16;
  const int dv = a.dv;
  const int value_tile = wave - (DELTA ? KT : 0);       // this wave's 16 value channels, if it has some
  const bool has_values = value_tile >= 0 && value_tile < dv / 16;
  float* const run = a.local + ((lm_first_run<N>(row[0], row[1] - row[3] * LM_CHUNK_TOKENS) + row[3] * RUNS + part) * a.H + head) * lm_run_floats<KIND, DK, N>(dv);
  float* const Ro = run;                                // [N][DK]
  float* const Nv = Ro + N * DK;                        // [dv][DK], transposed as the state is
  float* const M = Nv + (long)dv * DK;                  // [DK][DK]

  lm_floatx4 v[T];                                      // the values as right operands: row 16j + 4q + i (lm_place), column r
#pragma unroll
  for (int j = 0; j < T; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * j + 4 * i + q;
      const float value = (float)a.u[(t0 + min(t, count - 1)) * a.ld + a.v_col + (long)head * dv + (has_values ? 16 * value_tile + r : 0)];
      v[j][i] = t < count ? value : 0.f;
    }

  // ---- B, A, K and R, a wave PT tokens in a row, a lane PC channels (and A and K as they stand at the run's end)
  float a_end[PT][PC], k_end[PT][PC];
  if (!DELTA) {
    const float decay = a.head_decay[head];
    for (int n = threadIdx.x; n <= N; n += blockDim.x) powers[n] = n == 0 ? 1.f : powf(decay, (float)n);
    __syncthreads();
    if (wave < LM_PREP_WAVES) {
      const int half = a.rotary_dim / 2;
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        const int t = wave * PT + j;
        const bool valid = t < count;
        const long token = t0 + min(t, count - 1);
        const bf16_t* from = a.u + token * a.ld + (long)head * DK;
#pragma unroll
        for (int pc = 0; pc < PC; ++pc) {
          const int c = lane + WAVE * pc;
          float rx = (float)from[a.r_col + c], kx = (float)from[a.k_col + c];
          if (a.inv_freq && c < a.rotary_dim) {
            const bool low = c < half;
            const int pair = low ? c + half : c - half;
            float sine, cosine;
            sincosf((float)a.positions[token] * a.inv_freq[low ? c : c - half], &sine, &cosine);
            const float r_pair = (float)from[a.r_col + pair], k_pair = (float)from[a.k_col + pair];
            rx = low ? rx * cosine - r_pair * sine : rx * cosine + r_pair * sine;
            kx = low ? kx * cosine - k_pair * sine : kx * cosine + k_pair * sine;
          }
          R[lm_place(t) * KS + c] = valid ? rx : 0.f;
          K[lm_place(t) * KS + c] = valid ? kx * a.key_scale : 0.f;
          Ro[t * DK + c] = valid ? rx * powers[t + 1] : 0.f;
        }
      }
    }
  } else {
    float kx[PT][PC], rx[PT][PC], removal[PT][PC], logit[PT][PC];
    double w[PT][PC];
    if (wave < LM_PREP_WAVES) {
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        const long token = t0 + min(wave * PT + j, count - 1);
        const bf16_t* from = a.u + token * a.ld + (long)head * DK;
#pragma unroll
        for (int pc = 0; pc < PC; ++pc) {
          const int c = lane + WAVE * pc;
          kx[j][pc] = (float)from[a.k_col + c];
          rx[j][pc] = (float)from[a.r_col + c];
          removal[j][pc] = (float)from[a.removal_col + c];
          logit[j][pc] = a.decay_logits[token * a.logits_ld + (long)head * DK + c];
        }
      }
      double kept[PC];                                  // of a state over this wave's tokens
#pragma unroll
      for (int pc = 0; pc < PC; ++pc) kept[pc] = 1.0;
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        const bool valid = wave * PT + j < count;
#pragma unroll
        for (int pc = 0; pc < PC; ++pc) {
          const int c = lane + WAVE * pc;
          const float rate = lm_sigmoid(logit[j][pc] + a.decay_bias[head * DK + c]);
          w[j][pc] = valid ? exp((double)(-a.decay_floor * rate)) : 1.0;
          kept[pc] *= w[j][pc];
        }
      }
#pragma unroll
      for (int pc = 0; pc < PC; ++pc) products[wave * DK + lane + WAVE * pc] = kept[pc];
    }
    __syncthreads();
    if (wave < LM_PREP_WAVES) {
      double d[PC], d_last[PC];                         // d_(t-1), d_N
#pragma unroll
      for (int pc = 0; pc < PC; ++pc) {
        d[pc] = d_last[pc] = 1.0;
        for (int other = 0; other < LM_PREP_WAVES; ++other) {
          const double product = products[other * DK + lane + WAVE * pc];
          if (other < wave) d[pc] *= product;
          d_last[pc] *= product;
        }
        if (wave == 0) last[lane + WAVE * pc] = (float)d_last[pc];
      }
#pragma unroll
      for (int j = 0; j < PT; ++j) {
        const int t = wave * PT + j;
        const bool valid = t < count;
        float squares = 0.f;
#pragma unroll
        for (int pc = 0; pc < PC; ++pc) squares = fmaf(kx[j][pc], kx[j][pc], squares);
        const float length = sqrtf(wave_sum(squares) + a.key_eps);
#pragma unroll
        for (int pc = 0; pc < PC; ++pc) {
          const int c = lane + WAVE * pc;
          const float unit = kx[j][pc] / length;
          const double key = kx[j][pc], away = lm_sigmoid(removal[j][pc]) * unit;
          B[lm_place(t) * KS + c] = valid ? (float)(d[pc] * (double)unit) : 0.f;
          d[pc] *= w[j][pc];
          const double grown = 1.0 / d[pc], to_end = d_last[pc] * grown;
          A[lm_place(t) * KS + c] = valid ? (float)(grown * away) : 0.f;
          K[lm_place(t) * KS + c] = valid ? (float)(grown * key) : 0.f;
          R[lm_place(t) * KS + c] = valid ? (float)(d[pc] * (double)rx[j][pc]) : 0.f;
          a_end[j][pc] = valid ? (float)(to_end * away) : 0.f;
          k_end[j][pc] = valid ? (float)(to_end * key) : 0.f;
        }
      }
    }
  }
  __syncthreads();

  // ---- the triangles, a tile of 16 x 16 a turn: rows t of R (B) against rows s of K (A)
  constexpr int KINDS = DELTA ? 4 : 1;
  for (int item = wave; item < KINDS * (T * (T + 1) / 2); item += waves) {
    const int which = item % KINDS, pair = item / KINDS;
    int ti = 0;
    while ((ti + 1) * (ti + 2) / 2 <= pair) ++ti;
    const int tj = pair - ti * (ti + 1) / 2;
    const float* left = (which < 2 ? R : B) + 16 * ti * KS;
    const float* right = ((which & 1) ? A : K) + 16 * tj * KS;
    float* into = which == 0 ? RK : which == 1 ? RA : which == 2 ? P : L;
    lm_doublex4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < KT; ++c) acc = lm_mfma_double(lm_rows(left + 16 * c, KS, q, r), lm_rows(right + 16 * c, KS, q, r), acc);
    const int s = lm_place(16 * tj + r);
#pragma unroll
    for (int i = 0; i < 4; ++i) {                       // (rows of a result in 64 bits lie four apart in a lane)
      const int at = 16 * ti + 4 * i + q, t = lm_place(at);
      if (!DELTA) acc[i] *= (double)powers[max(t - s, 0)];
      into[at * TS + 16 * tj + r] = (which < 2 ? s <= t : s < t) ? (float)acc[i] : 0.f;
    }
  }
  __syncthreads();
  if (DELTA && wave < LM_PREP_WAVES) {                  // (read behind the next barrier)
#pragma unroll
    for (int j = 0; j < PT; ++j)
#pragma unroll
      for (int pc = 0; pc < PC; ++pc) {
        A[lm_place(wave * PT + j) * KS + lane + WAVE * pc] = a_end[j][pc];
        K[lm_place(wave * PT + j) * KS + lane + WAVE * pc] = k_end[j][pc];
      }
  }

  lm_floatx4 z[T];                                      // this wave's 16 columns of [Zk | Zv], rows 16j + 4q + i
  if (DELTA) {
    if (wave < KT) {                                    // columns of B; the first T of these waves invert the diagonal blocks too
#pragma unroll
      for (int ti = 0; ti < T; ++ti) z[ti] = lm_columns(B + 16 * ti * KS + 16 * wave, KS, q, r);
      if (wave < T) {
        float x[16];
        const float* block = L + (16 * wave) * TS + 16 * wave;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float sum = i == lm_place(r) ? 1.f : 0.f;
#pragma unroll
          for (int m = 0; m < i; ++m) sum = fmaf(-block[lm_place(i) * TS + lm_place(m)], x[m], sum);
          x[i] = sum;
        }
        if (q == 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) inverse[(wave * 16 + lm_place(i)) * 20 + r] = x[i];
        }
      }
    } else if (has_values) {
#pragma unroll
      for (int ti = 0; ti < T; ++ti) {
        z[ti] = lm_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tj = 0; tj < ti; ++tj) z[ti] = lm_mfma(lm_rows(P + 16 * ti * TS + 16 * tj, TS, q, r), v[tj], z[ti]);
        z[ti] = lm_diagonal<true>(P + 16 * ti * TS + 16 * ti, TS, q, r, v[ti], z[ti]);
      }
    }
    __syncthreads();
    if (wave >= KT && !has_values) return;
    // forward substitution, block row after block row; a result's layout is that of the next product's right operand
#pragma unroll
    for (int ti = 0; ti < T; ++ti) {
      lm_floatx4 known = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tj = 0; tj < ti; ++tj) known = lm_mfma(lm_rows(L + 16 * ti * TS + 16 * tj, TS, q, r), z[tj], known);
      z[ti] = lm_diagonal<false>(inverse + ti * 16 * 20, 20, q, r, z[ti] - known, lm_floatx4{0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int ti = 0; ti < T; ++ti) z[ti] = -z[ti];      // what is taken away
  } else if (!has_values) {
    return;
  }

  if (DELTA && wave < KT) {
    // 16 columns of Ro and M
#pragma unroll
    for (int ti = 0; ti < T; ++ti) {
      lm_floatx4 taken = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tj = 0; tj < ti; ++tj) taken = lm_mfma(lm_rows(RA + 16 * ti * TS + 16 * tj, TS, q, r), z[tj], taken);
      taken = lm_diagonal<false>(RA + 16 * ti * TS + 16 * ti, TS, q, r, z[ti], taken);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = 16 * ti + 4 * q + i;
        Ro[lm_place(at) * DK + 16 * wave + r] = R[at * KS + 16 * wave + r] + taken[i];
      }
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      lm_floatx4 taken = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int tj = 0; tj < T; ++tj) taken = lm_mfma(lm_columns(A + 16 * tj * KS + 16 * kt, KS, q, r), z[tj], taken);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 16 * kt + 4 * q + i, c = 16 * wave + r;
        M[k * DK + c] = (k == c ? last[k] : 0.f) + taken[i];
      }
    }
    return;
  }

  // ---- 16 value channels of Ov and Nv: one chain of sums each, from the oldest tokens to the newest, whose terms are as a rule
  // the largest
#pragma unroll
  for (int ti = 0; ti < T; ++ti) {
    lm_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tj = 0; tj < ti; ++tj) {
      if (DELTA) sum = lm_mfma(lm_rows(RA + 16 * ti * TS + 16 * tj, TS, q, r), z[tj], sum);
      sum = lm_mfma(lm_rows(RK + 16 * ti * TS + 16 * tj, TS, q, r), v[tj], sum);
    }
    if (DELTA) sum = lm_diagonal<false>(RA + 16 * ti * TS + 16 * ti, TS, q, r, z[ti], sum);
    sum = lm_diagonal<false>(RK + 16 * ti * TS + 16 * ti, TS, q, r, v[ti], sum);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * ti + 4 * i + q;
      if (t < count) a.out[(t0 + t) * a.out_ld + (long)head * dv + 16 * value_tile + r] = sum[i];
    }
  }
  if (!DELTA) {                                         // the keys' way to the run's end, laid on the values
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] *= powers[max(count - 1 - (16 * j + 4 * i + q), 0)];
  }
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    lm_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tj = 0; tj < T; ++tj) {
      if (DELTA) sum = lm_mfma(lm_columns(A + 16 * tj * KS + 16 * kt, KS, q, r), z[tj], sum);
      sum = lm_mfma(lm_columns(K + 16 * tj * KS + 16 * kt, KS, q, r), v[tj], sum);
    }
    *reinterpret_cast<lm_floatx4*>(Nv + (long)(16 * value_tile + r) * DK + 16 * kt + 4 * q) = sum;
  }
}

// A wave owns 16 rows of [Ro ; M] (retention: of Ro, and every thread some elements of the state); the state of the
// workgroup's 16 value channels goes from run to run through LDS.  AHEAD runs' operands are on their way.
template <int KIND, int DK, int N, int AHEAD>
__global__ void __launch_bounds__((KIND == LM_DELTA ? N / 16 + DK / 16 : 4) * WAVE) linear_matrix_carry_kernel(const LinearMatrixArgs a) {
  constexpr bool DELTA = KIND == LM_DELTA;
  constexpr int T = N / 16, KT = DK / 16, KS = DK + 4;
  constexpr int WAVES = DELTA ? T + KT : 4;
  constexpr int FOURS = DELTA ? 1 : 16 * DK / 4 / (WAVES * WAVE);      // retention: groups of four elements of a thread
  static_assert(DELTA || (T <= 4 && FOURS >= 1), "four waves hold the outputs' rows and the state");
  __shared__ __align__(16) float s_lds[2][16 * KS];
  const int lane_of_step = blockIdx.x;
  const int head = blockIdx.y;
  const int value0 = 16 * blockIdx.z;
  const int first = a.lane_chunks[2 * lane_of_step];
  const int chunks = a.lane_chunks[2 * lane_of_step + 1];
  if (chunks <= 0) return;
  const long row0 = a.chunks[4 * first + 1];
  const int tokens = (chunks - 1) * LM_CHUNK_TOKENS + a.chunks[4 * (first + chunks - 1) + 2];
  const int runs = (tokens + N - 1) / N;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int r = lane % 16;
  const int dv = a.dv;
  const bool outputs = wave < T;
  const long run_floats = lm_run_floats<KIND, DK, N>(dv), run_stride = run_floats * a.H;
  const float* const local = a.local + (lm_first_run<N>(lane_of_step, row0) * a.H + head) * run_floats;
  const float* const matrix = local + (outputs ? (long)(16 * wave + r) * DK
                                               : (long)N * DK + (long)dv * DK + (long)(16 * (wave - T) + r) * DK) + 4 * q;
  const float* const Nv = local + N * DK + (long)value0 * DK;
  float* const state = a.state + (((long)a.slot_ids[lane_of_step] * a.H + head) * dv + value0) * DK;
  for (int e = tid; e < 16 * DK; e += WAVES * WAVE) s_lds[0][(e / DK) * KS + e % DK] = state[e];
  float decay_run = 0.f, decay_last = 0.f;              // of a whole run, and of the lane's last
  if (!DELTA) {
    decay_run = powf(a.head_decay[head], (float)N);
    decay_last = powf(a.head_decay[head], (float)(tokens - (runs - 1) * N));
  }

  // `in_flight` runs' operands are on their way (a run past the lane's last is asked for as that run again)
  auto walk = [&](auto in_flight) {
    constexpr int IN_FLIGHT = decltype(in_flight)::value;
    lm_floatx4 rows[IN_FLIGHT][KT], beside[IN_FLIGHT][FOURS], known[IN_FLIGHT];
    auto ask = [&](int at, int j) {
      const int run = min(j, runs - 1);
      const float* from = matrix + run * run_stride;
#pragma unroll
      for (int c = 0; c < KT; ++c) rows[at][c] = *reinterpret_cast<const lm_floatx4*>(from + 16 * c);
      if (DELTA) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          beside[at][0][i] = Nv[run * run_stride + (4 * q + i) * DK + (outputs ? 0 : 16 * (wave - T) + r)];
      } else {
#pragma unroll
        for (int g = 0; g < FOURS; ++g)
          beside[at][g] = *reinterpret_cast<const lm_floatx4*>(Nv + run * run_stride + 4 * (tid + g * WAVES * WAVE));
      }
      const long row = row0 + min(run * N + 16 * (outputs ? wave : 0) + r, tokens - 1);
      known[at] = *reinterpret_cast<const lm_floatx4*>(a.out + row * a.out_ld + (long)head * dv + value0 + 4 * q);
    };
#pragma unroll
    for (int j = 0; j < IN_FLIGHT; ++j) ask(j, j);
    __syncthreads();
    for (int j0 = 0; j0 < runs; j0 += IN_FLIGHT) {
#pragma unroll
      for (int at = 0; at < IN_FLIGHT; ++at) {
        // (no way out of the turns of a round: behind one the compiler waits for every load in flight.  A turn past the
        // last run repeats that run's products, stores nothing and hands the state on)
        const int j = j0 + at;
        const bool live = j < runs;
        const float* const s_now = s_lds[j & 1];
        float* const s_next = s_lds[(j + 1) & 1];
        lm_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
        if (DELTA || outputs) {
#pragma unroll
          for (int c = 0; c < KT; c += 4) {               // a chain for every 16 channels, added in pairs
            lm_floatx4 part[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) part[p] = lm_mfma(lm_rows(s_now + 16 * (c + p), KS, q, r), rows[at][c + p], lm_floatx4{0.f, 0.f, 0.f, 0.f});
            sum += (part[0] + part[1]) + (part[2] + part[3]);
          }
        }
        if (outputs) {                                    // value channels 4q + i of token r
          const int t = j * N + 16 * wave + r;
          if (t < tokens)
            *reinterpret_cast<lm_floatx4*>(a.out + (row0 + t) * a.out_ld + (long)head * dv + value0 + 4 * q) = known[at] + sum;
        } else if (DELTA) {                               // value channels 4q + i of key channel r
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int place = (4 * q + i) * KS + 16 * (wave - T) + r;
            s_next[place] = live ? sum[i] + beside[at][0][i] : s_now[place];
          }
        }
        if (!DELTA) {
          const int own = min(N, tokens - j * N);
          const float shrink = own == N ? decay_run : decay_last;
#pragma unroll
          for (int g = 0; g < FOURS; ++g) {
            const int e = 4 * (tid + g * WAVES * WAVE);
            const int place = (e / DK) * KS + e % DK;
            const lm_floatx4 before = *reinterpret_cast<const lm_floatx4*>(s_now + place);
            *reinterpret_cast<lm_floatx4*>(s_next + place) = live ? shrink * before + beside[at][g] : before;
          }
        }
        ask(at, j + IN_FLIGHT);
        __syncthreads();
      }
    }
    return (runs + IN_FLIGHT - 1) / IN_FLIGHT * IN_FLIGHT;      // turns made
  };
  // a lane of one run or two, as single tokens beside a portion are, does not ask for their operands again and again
  const int turns = runs == 1 ? walk(std::integral_constant<int, 1>()) : runs <= 2 ? walk(std::integral_constant<int, 2>())
                                                                      : walk(std::integral_constant<int, AHEAD>());
  const float* const s_end = s_lds[turns & 1];
  for (int e = tid; e < 16 * DK; e += WAVES * WAVE) state[e] = s_end[(e / DK) * KS + e % DK];
}

// Tokens of a run.  The delta rule at 64 channels takes 60 KB of LDS a workgroup with runs of 32 (two a compute unit) and
// 149 with 64: 37 us against 50 in the chunk kernel and 64 against 46 in the carry for 1,999 tokens and 16 heads, 13 + 8
// against 23 + 9 for 100 tokens.  Retention has no M to carry and half the matrices.
#define LM_DELTA_RUN 32
#define LM_RETENTION_RUN 64

// dk 64 or 128 and whole tiles of 16 value channels, at most as many as there are waves for
extern "C" int mi_linear_matrix_supported(int delta, int dk, int dv) {
  return (dk == 64 || dk == 128) && dv > 0 && dv % 16 == 0 && dv / 16 + (delta ? dk / 16 : 0) <= LM_MOST_WAVES ? 1 : 0;
}
// tokens of a run: the delta rule's decay_floor times this is the logarithm of the largest number it forms
extern "C" int mi_linear_matrix_run(int delta) { return delta ? LM_DELTA_RUN : LM_RETENTION_RUN; }
extern "C" int mi_linear_matrix_chunk_tokens(void) { return LM_CHUNK_TOKENS; }

// of the work area for a step of so many tokens in so many lanes
extern "C" long mi_linear_matrix_floats(int delta, int tokens, int lanes, int H, int dk, int dv) {
  const long run = mi_linear_matrix_run(delta);
  return (tokens / run + lanes) * H * (run * dk + (long)dv * dk + (delta ? (long)dk * dk : 0));
}

template <int KIND, int DK, int N, int AHEAD>
static int launch_linear_matrix(const LinearMatrixArgs& a, int num_chunks, int lanes, hipStream_t stream) {
  const size_t lds = sizeof(float) * lm_chunk_lds_floats<KIND, DK, N>();
  // beyond 64 KiB a kernel has to be told once per device that it may have that much (gfx950 has 160 KiB)
  static bool told[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return ERR_BAD_ARGUMENT;
  if (!told[device]) {
    if (hipFuncSetAttribute((const void*)linear_matrix_chunk_kernel<KIND, DK, N>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess) {
      (void)hipGetLastError();
      return ERR_UNSUPPORTED_SIZE;
    }
    told[device] = true;
  }
  const int tiles = a.dv / 16 + (KIND == LM_DELTA ? DK / 16 : 0);
  const int waves = tiles > LM_PREP_WAVES ? tiles : LM_PREP_WAVES;
  linear_matrix_chunk_kernel<KIND, DK, N><<<dim3(num_chunks * (LM_CHUNK_TOKENS / N), a.H), waves * WAVE, lds, stream>>>(a);
  RETURN_IF_LAUNCH_FAILED();
  const int carry_waves = KIND == LM_DELTA ? N / 16 + DK / 16 : 4;
  linear_matrix_carry_kernel<KIND, DK, N, AHEAD><<<dim3(lanes, a.H, a.dv / 16), carry_waves * WAVE, 0, stream>>>(a);
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// u: bfloat16 rows, any columns; state, local and out float32 and 16-byte aligned, out_ld a multiple of 4; the table's
// chunks hold LM_CHUNK_TOKENS tokens but for a lane's last.  removal_col >= 0: the delta rule.
extern "C" int mi_linear_matrix_scan(const void* u, long ld, int r_col, int k_col, int v_col, int removal_col, int H, int dk,
                                     int dv, float* state, const int* slot_ids, int lanes, const int* chunks,
                                     const int* lane_chunks, int num_chunks, int chunk_tokens, const float* head_decay,
                                     float key_scale, const int* positions, const float* inv_freq, int rotary_dim,
                                     const float* decay_logits, long logits_ld, const float* decay_bias, float decay_floor,
                                     float key_eps, float* local, float* out, long out_ld, hipStream_t stream) {
  const bool delta = removal_col >= 0;
  if (!u || !state || !slot_ids || !chunks || !lane_chunks || !local || !out || H <= 0 || lanes <= 0 || num_chunks <= 0 ||
      r_col < 0 || k_col < 0 || v_col < 0 || out_ld < (long)H * dv || (delta ? !decay_logits || !decay_bias : !head_decay) ||
      (inv_freq && (!positions || rotary_dim <= 0 || rotary_dim > dk || rotary_dim % 2)))
    return ERR_BAD_ARGUMENT;
  if (!mi_linear_matrix_supported(delta, dk, dv) || chunk_tokens != LM_CHUNK_TOKENS || H > 65535 || out_ld % 4 ||
      ((uintptr_t)state | (uintptr_t)local | (uintptr_t)out) % 16)
    return ERR_UNSUPPORTED_SIZE;
  if (delta && !(decay_floor >= 0.f && decay_floor * mi_linear_matrix_run(1) <= 60.f)) return ERR_UNSUPPORTED_SIZE;
  if (ld < r_col + (long)H * dk || ld < k_col + (long)H * dk || ld < v_col + (long)H * dv ||
      (delta && (ld < removal_col + (long)H * dk || logits_ld < (long)H * dk)))
    return ERR_BAD_ARGUMENT;
  const LinearMatrixArgs a = {(const bf16_t*)u, ld, r_col, k_col, v_col, removal_col, H, dv, state, slot_ids, chunks,
                              lane_chunks, head_decay, key_scale, positions, inv_freq, rotary_dim, decay_logits, logits_ld,
                              decay_bias, decay_floor, key_eps, local, out, out_ld};
  if (delta)
    return dk == 64 ? launch_linear_matrix<LM_DELTA, 64, LM_DELTA_RUN, 4>(a, num_chunks, lanes, stream)
                    : launch_linear_matrix<LM_DELTA, 128, LM_DELTA_RUN, 2>(a, num_chunks, lanes, stream);
  return dk == 64 ? launch_linear_matrix<LM_RETENTION, 64, LM_RETENTION_RUN, 4>(a, num_chunks, lanes, stream)
                  : launch_linear_matrix<LM_RETENTION, 128, LM_RETENTION_RUN, 2>(a, num_chunks, lanes, stream);
}
