// Matrix products of the float32 path: out[M, N] = x[M, K] . W[N, K]^T (+ bias[N]), with float32
// operands, products and sums throughout (v_mfma_f32_16x16x4_f32 multiplies and adds in float32; no
// reduced-precision matrix mode).
//
// One kernel serves a decode step of a few rows and a prompt portion of thousands: a workgroup owns
// NT tiles of 16 output features and MT tiles of 16 rows, its four waves split K into four contiguous
// runs of 16-wide chunks, and their partial tiles are added through LDS in the order of the waves.  The
// order in which an output element is summed depends on K alone (which chunks a wave owns, the four
// products of a chunk in turn, wave 0 to 3), never on M, on the tiling or on the rows beside it: a
// row's result is bit for bit the same alone, in a small step and in a large one.
//
// A step of up to 32 rows is bound by reading W once: every wave keeps its 1 KiB fragments in flight.  More rows are
// bound by the matrix cores and go through tiled_f32_kernel and direct_f32_kernel, which share their operands through LDS and keep that
// order of the sums (K a multiple of 32, rows of whole 16-byte pieces; other sizes stay with the first kernel).
#include "common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

#define GF_WAVES 4
#define GF_THREADS (GF_WAVES * WAVE)

// four consecutive k of one row; VEC: one 16-byte load (K, the leading dimension and the base are
// multiples of 4 floats); otherwise four loads, each checked against K.  A k at or past K gives zero.
template <bool VEC>
__device__ __forceinline__ floatx4 load_k4(const float* row, int k, int K) {
  if (VEC) {
    const floatx4 value = *reinterpret_cast<const floatx4*>(row + min(k, K - 4));
    return k < K ? value : floatx4{0.f, 0.f, 0.f, 0.f};
  }
  floatx4 value;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float element = row[min(k + j, K - 1)];
    value[j] = k + j < K ? element : 0.f;
  }
  return value;
}

template <int MT, int NT, int DEPTH, bool VEC>
__global__ void __launch_bounds__(GF_THREADS)
gemm_f32_kernel(const float* __restrict__ x, long ldx, const float* __restrict__ W, long ldw,
                const float* __restrict__ bias, float* __restrict__ out, long ldo, int M, int N, int K) {
  __shared__ float red[GF_WAVES][MT][256];
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int r = lane % 16;
  const long n0 = (long)blockIdx.x * 16 * NT;
  const long m0 = (long)blockIdx.y * 16 * MT;
  const float* w_row[NT];
  const float* x_row[MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) w_row[nt] = W + min(n0 + 16 * nt + r, (long)N - 1) * ldw;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) x_row[mt] = x + min(m0 + 16 * mt + r, (long)M - 1) * ldx;

  const int chunks = (K + 15) / 16;
  const int per_wave = (chunks + GF_WAVES - 1) / GF_WAVES;
  const int first_chunk = wave * per_wave;
  const int iterations = max(0, min(per_wave, chunks - first_chunk));

  floatx4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};

  // DEPTH chunks are asked for before the first is used; no branch between the loads (a chunk past
  // the wave's run reads the run's last one again and is not multiplied)
  for (int first = 0; first < iterations; first += DEPTH) {
    floatx4 a[DEPTH][NT], b[DEPTH][MT];
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      const int k = (first_chunk + min(first + j, iterations - 1)) * 16 + 4 * q;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) a[j][nt] = load_k4<VEC>(w_row[nt], k, K);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[j][mt] = load_k4<VEC>(x_row[mt], k, K);
    }
    // a step of few rows waits for its weights: every load of the round is asked for before its first product (left
    // to itself the scheduler moves each load down to the product that uses it and waits for it there, one round
    // trip to memory after the other; the tiles of many rows, which wait for their products, are better left to it)
    if (NT == 1) __builtin_amdgcn_sched_barrier(0);
    // no branch around the products either (under one the compiler waits for each load where it is used,
    // one at a time): a chunk past the end is multiplied as zeros
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      const bool live = first + j < iterations;
      const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
      floatx4 weights[NT], rows[MT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) weights[nt] = live ? a[j][nt] : zero;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) rows[mt] = live ? b[j][mt] : zero;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(weights[nt][i], rows[mt][i], acc[nt][mt], 0, 0, 0);
    }
  }

  // the waves' partial tiles, added in the order of the waves, one tile of 16 features after the other
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt > 0) __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][mt][i * 64 + lane] = acc[nt][mt][i];
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      // element tid of the tile: feature 4 (l / 16) + i, row l % 16, stored at i * 64 + l
      const int i = tid / 64;
      const int l = tid % 64;
      float value = red[0][mt][tid];
#pragma unroll
      for (int w = 1; w < GF_WAVES; ++w) value += red[w][mt][tid];
      const long n = n0 + 16 * nt + 4 * (l / 16) + i;
      const long m = m0 + 16 * mt + (l % 16);
      if (n < N && m < M) out[m * ldo + n] = bias ? value + bias[n] : value;
    }
  }
}

// Many rows: a group of 2 x 2 waves owns 32 MT rows x 32 NT features, stages 32 columns of both operands in LDS (two
// buffers; the stages behind it are on their way to registers while this one is multiplied) and sums the four runs of chunks
// one after the other, each from zero, adding the runs' sums in their order: bit for bit the sums above.
// GROUPS = 4: four such groups of a workgroup take a run each and group 0 adds their tiles, for products of too few
// tiles to fill 256 compute units one wave a SIMD (a wave's chain of products is then a quarter as long).
// LDS: a row of a stage is eight 16-byte pieces; piece p of row r lies at r * 8 + (p ^ (r & 7)), so that the eight rows
// that a quarter-wave reads at once fall into different banks, and a thread's stores are one run.
// EVEN: the runs are whole stages (K a multiple of 128).
// What bounds it: the matrix cores (v_mfma_f32_16x16x4_f32, 152 TFLOP/s in a large library product) and what the waves
// do between their products, all at once in a workgroup: with the operands fetched where they are used, the stages laid
// down and asked for in a row and the barrier behind, 512 x 4,096 x 1,024 took 47.1 us, 512 x 1,024 x 2,048 29.4, 512 x 768 x
// 1,024 16.6, 512 x 32,784 x 1,024 331; fetched a chunk ahead, one by one between the products, 45.1, 24.2, 14.5, 321 (without
// any of those instructions 35, 18, 11, 252).  64 x 128 tiles in two groups take 43.5, 41.1 (N = 768) and 343, 64 x 64 ones in
// two groups 47.4; a second stage on its way, 128 x 128 tiles and an order of the tiles by die gain nothing.

// The order of a chunk's instructions: stores to LDS, loads from memory and loads from LDS one by one between its products.
template <int PRODUCTS, int STORES, int LOADS, int FETCHES>
__device__ __forceinline__ void interleave() {
  constexpr int OTHERS = STORES + LOADS + FETCHES;
  constexpr int EACH = PRODUCTS / OTHERS > 0 ? PRODUCTS / OTHERS : 1;
#pragma unroll
  for (int i = 0; i < OTHERS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);                        // matrix products
    if (i < STORES) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);           // a store to LDS
    else if (i < STORES + LOADS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);          // a load from memory
    else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      // a load from LDS
  }
}

template <int MT, int NT, int GROUPS, bool EVEN>
__global__ void __launch_bounds__(GF_THREADS * GROUPS)
tiled_f32_kernel(const float* __restrict__ x, long ldx, const float* __restrict__ W, long ldw,
                 const float* __restrict__ bias, float* __restrict__ out, long ldo, bool whole, int M, int N, int K) {
  constexpr int BM = 32 * MT, BN = 32 * NT, ROWS = BM + BN;
  constexpr int PIECES = ROWS * 8 / GF_THREADS;                // 16-byte pieces a thread moves a stage
  constexpr int STAGED = GROUPS * 2 * ROWS * 8, PARTIAL = (GROUPS - 1) * BM * BN / 4;
  __shared__ floatx4 lds[STAGED > PARTIAL ? STAGED : PARTIAL];
  const int group = GROUPS == 1 ? 0 : threadIdx.x / GF_THREADS;
  const int tid = threadIdx.x % GF_THREADS;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int r = lane % 16;
  const int first_m = (wave & 1) * MT * 16, first_n = (wave >> 1) * NT * 16;     // the wave's part of the tile
  const long n0 = (long)blockIdx.x * BN;
  const long m0 = (long)blockIdx.y * BM;
  floatx4* const stage_of_group = lds + group * 2 * ROWS * 8;

  const int chunks = K / 16;
  const int run = (chunks + GF_WAVES - 1) / GF_WAVES;          // chunks of one of the four runs
  const int first_chunk = group * run;
  const int mine = GROUPS == 1 ? chunks : max(0, min(run, chunks - first_chunk));
  const int stages = GROUPS == 1 ? chunks / 2 : (run + 1) / 2;
  const float* source[PIECES];
  int column[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int slot = p * GF_THREADS + tid;
    const int row = slot / 8;
    source[p] = row < BN ? W + min(n0 + row, (long)N - 1) * ldw : x + min(m0 + row - BN, (long)M - 1) * ldx;
    column[p] = first_chunk * 16 + 4 * ((slot % 8) ^ (row & 7));
  }
  floatx4 on_the_way[PIECES];
  auto ask = [&](int stage) {                                  // (columns past the row's end repeat its last ones and are not multiplied)
#pragma unroll
    for (int p = 0; p < PIECES; ++p)
      on_the_way[p] = *reinterpret_cast<const floatx4*>(source[p] + min(column[p] + 32 * stage, K - 4));
  };
  auto lay_down = [&](int buffer) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) stage_of_group[buffer * ROWS * 8 + p * GF_THREADS + tid] = on_the_way[p];
  };

  floatx4 acc[NT][MT], total[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = total[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};
  int left = run;
  floatx4 weights[2][NT], rows[2][MT];                         // the operands of a stage's two chunks
  auto fetch = [&](int stage, int c) {                         // (a row's number and r agree modulo 8)
    const floatx4* const staged = stage_of_group + (stage & 1) * ROWS * 8 + ((4 * c + q) ^ (r & 7));
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) weights[c][nt] = staged[(first_n + nt * 16 + r) * 8];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) rows[c][mt] = staged[(BN + first_m + mt * 16 + r) * 8];
  };
  auto multiply = [&](int stage, int c) {
    if (GROUPS > 1 && !EVEN && 2 * stage + c >= mine) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(weights[c][nt][i], rows[c][mt][i], acc[nt][mt], 0, 0, 0);
    if (GROUPS == 1 && (c == 1 || !EVEN)) {
      left -= EVEN ? 2 : 1;
      if (left == 0) {                                         // a run ends
        left = run;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            total[nt][mt] += acc[nt][mt];
            acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };
  // Every wait has products in front of it: a stage's columns leave memory a whole stage before they are laid down, and
  // a chunk's operands leave LDS while the chunk before is multiplied.  The one barrier a stage stands between its two
  // chunks: behind it the next stage is laid down, and nobody reads the one before any more.
  ask(0);
  lay_down(0);
  ask(1);
  __syncthreads();
  fetch(0, 0);
  for (int stage = 0; stage < stages; ++stage) {
    lay_down((stage + 1) & 1);
    ask(stage + 2);
    fetch(stage, 1);
    multiply(stage, 0);
    interleave<4 * NT * MT, PIECES, PIECES, NT + MT>();
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    fetch(stage + 1, 0);
    multiply(stage, 1);
    interleave<4 * NT * MT, 0, 0, NT + MT>();
    __builtin_amdgcn_sched_barrier(0);
  }

  if (GROUPS > 1) {
    __syncthreads();                                           // the stages are read
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        if (group > 0) lds[((group - 1) * NT * MT + nt * MT + mt) * GF_THREADS + tid] = acc[nt][mt];
    __syncthreads();
    if (group > 0) return;
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      floatx4 value = total[nt][mt] + acc[nt][mt];             // (the last run's sum, or a shorter run's behind it)
#pragma unroll
      for (int g = 1; g < GROUPS; ++g) value += lds[((g - 1) * NT * MT + nt * MT + mt) * GF_THREADS + tid];
      const long n = n0 + first_n + nt * 16 + 4 * q;
      const long m = m0 + first_m + mt * 16 + r;
      if (m >= M) continue;
      if (bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) value[i] += bias[min(n + i, (long)N - 1)];
      }
      if (whole && n + 3 < N) {
        *reinterpret_cast<floatx4*>(out + m * ldo + n) = value;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) out[m * ldo + n + i] = value[i];
      }
    }
}

// The 64 x 64 tile of the above where the runs are whole stages (K a multiple of 128): the stages go from memory to LDS
// without passing through registers (`buffer_load ... lds` writes 64 pieces one after the other, so it is the lanes'
// addresses within a line that are exchanged), and the waves have nothing between their products but the loads of the next
// chunk's operands.  Two stages in LDS: four workgroups a compute unit hide each other's waits (with three stages 280 us in place
// of 273 for 32,784 features; tiles of 64 x 128 and 128 x 64 39.5 to 41.0 for the first).  512 x 4,096 x 1,024 45.2 -> 39.6 us, 512
// x 3,352 x 1,024 43.6 -> 39.1, 512 x 32,784 x 1,024 298 -> 273, 2,048 x 1,024 x 2,048 73.3 -> 68.2; the smaller tiles in four
// groups gain nothing this way (512 x 1,024 x 2,048 22.7 | 24.0).
typedef __attribute__((address_space(3))) void f32_lds;
#define DIRECT_STAGES 2

__global__ void __launch_bounds__(GF_THREADS)
direct_f32_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ W, int ldw, const float* __restrict__ bias,
                  float* __restrict__ out, long ldo, bool whole, int M, int N, int K) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int TILE = 64, ROWS = 2 * TILE, LOADS = ROWS / 8 / GF_WAVES;       // of eight rows that a wave makes a stage
  __shared__ floatx4 lds[DIRECT_STAGES][ROWS * 8];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int q = lane / 16, r = lane % 16;
  const int first_m = (wave & 1) * 32, first_n = (wave >> 1) * 32;             // the wave's part of the tile
  const int n0 = blockIdx.x * TILE, m0 = blockIdx.y * TILE;
  const __amdgpu_buffer_rsrc_t w_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (long)n0 * ldw), 0, 0xffffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t x_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (long)m0 * ldx), 0, 0xffffffff, 0x00020000);
  int offset[LOADS];                                           // (bytes within the tile's rows: the launch keeps them below 2^31)
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (i * GF_WAVES + wave) * 8 + lane / 8;
    const int piece = (lane % 8) ^ (row & 7);
    offset[i] = 4 * (i * GF_WAVES * 8 < TILE ? min(row, N - 1 - n0) * ldw + 4 * piece : min(row - TILE, M - 1 - m0) * ldx + 4 * piece);
  }
  const int stages = K / 32, run = stages / GF_WAVES;          // the sums' four runs
  auto ask = [&](int stage) {                                  // (past the last one: the last again, never multiplied)
    floatx4* const into = lds[stage % DIRECT_STAGES];
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i * GF_WAVES * 8 < TILE ? w_rows : x_rows, (f32_lds*)(into + (i * GF_WAVES + wave) * 64), 16,
                                               offset[i], min(stage, stages - 1) * 128, 0, 0);
  };
  floatx4 acc[2][2], total[2][2];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[n][m] = total[n][m] = floatx4{0.f, 0.f, 0.f, 0.f};
  floatx4 weights[2][2], rows[2][2];                           // the operands of a stage's two chunks
  auto fetch = [&](int stage, int chunk) {
    const floatx4* const from = lds[stage % DIRECT_STAGES] + ((4 * chunk + q) ^ (r & 7));
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      weights[chunk][t] = from[(first_n + 16 * t + r) * 8];
      rows[chunk][t] = from[(TILE + first_m + 16 * t + r) * 8];
    }
  };
  auto multiply = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(weights[chunk][n][i], rows[chunk][m][i], acc[n][m], 0, 0, 0);
  };
#pragma unroll
  for (int stage = 0; stage < DIRECT_STAGES; ++stage) ask(stage);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DIRECT_STAGES - 1) * LOADS) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  fetch(0, 0);
  int left = run;
  for (int stage = 0; stage < stages; ++stage) {
    fetch(stage, 1);
    multiply(0);
    interleave<16, 0, 0, 4>();
    __builtin_amdgcn_sched_barrier(0);
    // this wave has read the stage, and its own part of the next one has arrived: behind the barrier the same holds for all
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((DIRECT_STAGES - 2) * LOADS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    ask(stage + DIRECT_STAGES);
    fetch(stage + 1, 0);
    multiply(1);
    interleave<16, 0, LOADS, 4>();
    __builtin_amdgcn_sched_barrier(0);
    if (--left == 0) {                                         // a run ends
      left = run;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          total[n][m] += acc[n][m];
          acc[n][m] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  // nothing of the stages past the end may still be on its way to LDS when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      floatx4 value = total[nt][mt];
      const int n = n0 + first_n + 16 * nt + 4 * q;
      const long m = m0 + first_m + 16 * mt + r;
      if (m >= M) continue;
      if (bias) {
#pragma unroll
        for (int i = 0; i < 4; ++i) value[i] += bias[min(n + i, N - 1)];
      }
      if (whole && n + 3 < N) {
        *reinterpret_cast<floatx4*>(out + m * ldo + n) = value;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) out[m * ldo + n + i] = value[i];
      }
    }
#endif
}

template <int MT, int NT, int DEPTH>
static void launch_gemm_f32(bool vec, dim3 grid, hipStream_t stream, const float* x, long ldx, const float* W,
                            long ldw, const float* bias, float* out, long ldo, int M, int N, int K) {
  if (vec) gemm_f32_kernel<MT, NT, DEPTH, true><<<grid, GF_THREADS, 0, stream>>>(x, ldx, W, ldw, bias, out, ldo, M, N, K);
  else gemm_f32_kernel<MT, NT, DEPTH, false><<<grid, GF_THREADS, 0, stream>>>(x, ldx, W, ldw, bias, out, ldo, M, N, K);
}

extern "C" int mi_gemm_f32(const float* x, long ldx, const float* W, long ldw, const float* bias, float* out,
                           long ldo, int M, int N, int K, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || ldx < K || ldw < K || ldo < N) return ERR_BAD_ARGUMENT;
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && ((unsigned long long)x % 16) == 0 &&
                   ((unsigned long long)W % 16) == 0;
  if (M > 32 && vec && K % 32 == 0) {
    // The tiling that the rounds of workgroups over 256 compute units make cheapest: microseconds a round at K =
    // 1,024, in tenths, as measured over 40 to 512 rows and 768 to 32,784 features (32 x 32 in four groups: 9.0 to 9.8,
    // 15.8, 22.5, 28.8, 37.1, 41.7 for one to six rounds; 32 x 64 in four groups: 13.4 to 15.3, 28, 38 to 40, 55; 64 x 64 in one
    // group: 22 to 24, 39 to 41, 56, then 18.5 a round: workgroups of a compute unit hide each other's waits).  From 33 rows
    // on the best of them is at least as fast as the first kernel at every size measured.
    auto rounds = [&](long rows, long features) {
      return (((M + rows - 1) / rows) * ((N + features - 1) / features) + 255) / 256;
    };
    const long small = 28 + 66 * rounds(32, 32), middle = 25 + 130 * rounds(32, 64), tall = rounds(64, 64);
    const long large = tall == 1 ? 235 : tall == 2 ? 400 : 185 * tall;
    const bool whole = ldo % 4 == 0 && ((unsigned long long)out % 16) == 0;
    const int bm = large < small && large < middle ? 64 : 32, bn = bm == 64 || middle < small ? 64 : 32;
    const dim3 tiles((unsigned)(((long)N + bn - 1) / bn), (unsigned)(((long)M + bm - 1) / bm));
    if (((long)M + bm - 1) / bm <= 65535) {
      const bool even = K % 128 == 0;
#define TILED(MT_, NT_, GROUPS_)                                                                                       \
  do {                                                                                                                 \
    if (even) tiled_f32_kernel<MT_, NT_, GROUPS_, true><<<tiles, GROUPS_ * GF_THREADS, 0, stream>>>(x, ldx, W, ldw, bias, out, ldo, whole, M, N, K); \
    else tiled_f32_kernel<MT_, NT_, GROUPS_, false><<<tiles, GROUPS_ * GF_THREADS, 0, stream>>>(x, ldx, W, ldw, bias, out, ldo, whole, M, N, K);     \
  } while (0)
      if (bm == 64 && even && ldx <= 1 << 22 && ldw <= 1 << 22)
        direct_f32_kernel<<<tiles, GF_THREADS, 0, stream>>>(x, (int)ldx, W, (int)ldw, bias, out, ldo, whole, M, N, K);
      else if (bm == 64) tiled_f32_kernel<2, 2, 1, false><<<tiles, GF_THREADS, 0, stream>>>(x, ldx, W, ldw, bias, out, ldo, whole, M, N, K);
      else if (bn == 64) TILED(1, 2, 4);
      else TILED(1, 1, 4);
#undef TILED
      RETURN_IF_LAUNCH_FAILED();
      return 0;
    }
  }
  // rows and features of a workgroup: one tile of features while the step is small (W is read once, by as
  // many workgroups as there are tiles of it); 64 x 64 for many rows (x and W come from the caches)
  const int row_tiles = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int feature_tiles = M <= 64 ? 1 : 4;
  const long blocks_x = ((long)N + 16 * feature_tiles - 1) / (16 * feature_tiles);
  const long blocks_y = ((long)M + 16 * row_tiles - 1) / (16 * row_tiles);
  if (blocks_y > 65535 || blocks_x > 0x7fffffffL) return ERR_UNSUPPORTED_SIZE;
  const dim3 grid((unsigned)blocks_x, (unsigned)blocks_y);
  if (feature_tiles == 4) launch_gemm_f32<4, 4, 2>(vec, grid, stream, x, ldx, W, ldw, bias, out, ldo, M, N, K);
  else if (row_tiles == 4) launch_gemm_f32<4, 1, 4>(vec, grid, stream, x, ldx, W, ldw, bias, out, ldo, M, N, K);
  else if (row_tiles == 2) launch_gemm_f32<2, 1, 4>(vec, grid, stream, x, ldx, W, ldw, bias, out, ldo, M, N, K);
  else launch_gemm_f32<1, 1, 8>(vec, grid, stream, x, ldx, W, ldw, bias, out, ldo, M, N, K);
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}
