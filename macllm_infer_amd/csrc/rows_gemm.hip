// Products of many rows in bfloat16 on the matrix cores: out[M, N] = x[M, K] . W[N, K]^T (+ bias[N], float32), rounded once,
// SiLU(gate) * up of the rounded results of a W whose rows lie in tiles of 8 gate rows and 8 up rows, or the float32 sums.
//
// A workgroup owns a tile of BM rows x BN features.  K is walked in stages of 64 columns, whole lines of 128 bytes of every
// row, which go from memory to LDS without passing through registers (`buffer_load ... lds`), STAGES of them on their way;
// one barrier a stage.  A wave holds the fragments of half a stage (small tiles: of a whole one) in registers and reads those of
// the next while it multiplies.  Piece p of row r of a stage lies at 8 r + (p ^ (r & 7)): a load to LDS
// writes 64 pieces one after the other, so it is the lanes' addresses that are exchanged (within a line), and no read of a
// fragment meets a bank conflict.  A row's sum runs in k order in one lane, whatever the tile and the rows beside it.
//
// What bounds it: a stage's reads from LDS, their latency and its barrier (64 x 64 tiles: 400 cycles a stage, 128 of them
// products; with the next half's fragments in place of the next stage's on their way 470, with four waves in place of eight
// 540), the launch and the lines written at its end (2,048 x 4,096 with K = 64: 8.9 us).  So it is at its best where the tiles
// fit the chip once, which is where the library is at its worst: us, library | this, rows and weights from memory: 65 x 1,024 x
// 1,024 8.3 | 6.5, 1,554 x 1,024 x 1,024 10.6 | 8.6, 1,554 x 1,024 x 512 8.6 | 6.4, 640 x 1,024 x 2,048 10.9 | 9.9; with the
// activation (the library's product and the launch behind it) 256 x 4,096 x 1,024 15.1 | 8.0, 640 rows 19.0 | 13.9, 2,048 rows
// 27 | 23.0; and where it is not: 2,048 x 1,024 x 2,048 18.0 | 17.7, 1,999 x 6,144 x 1,024 31 | 40, 2,048 x 24,576 x 3,072 with the
// activation 253 | 310.
#include "common.h"

typedef float g_floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 g_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 g_bf16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void g_lds;

#define GEMM_STAGE 64                // columns of a stage
#define EPI_ROWS_PLAIN 0
#define EPI_ROWS_SWIGLU 1
#define EPI_ROWS_F32 2               // the sums as they are

struct RowsGemm {
  const bf16_t* x;
  const bf16_t* w;
  const float* bias;
  void* out;
  int ldx, ldw;                      // elements
  long ldo;
  int M, N, K, tiles_m, tiles_n;
  int whole;                         // four neighbouring outputs are one aligned piece
};

template <int BM, int BN, int WM, int WN, int STAGES, bool AHEAD, int EPI>
__global__ void __launch_bounds__(WAVE * WM * WN, 2)
rows_gemm_kernel(RowsGemm p) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int WAVES = WM * WN;
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  constexpr int LOADS = (BM + BN) / 8 / WAVES;               // of 1 KiB, eight rows, that a wave makes a stage
  static_assert((BM + BN) % (8 * WAVES) == 0 && BM % (8 * WAVES) == 0, "whole loads, each of x or of W");
  static_assert(EPI != EPI_ROWS_SWIGLU || TN % 2 == 0, "pairs of tiles");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES][(BM + BN) * 2 * GEMM_STAGE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  // Workgroups go round the eight dies by their numbers: a die gets a run of tiles, walked in bands of eight tiles of rows,
  // so that the rows and the features that it reads stay in its cache.
  const int per_die = gridDim.x / 8;
  const int number = (int)(blockIdx.x % 8) * per_die + (int)(blockIdx.x / 8);
  if (number >= p.tiles_m * p.tiles_n) return;
  const int first_of_band = number / (8 * p.tiles_n) * 8;
  const int band = min(8, p.tiles_m - first_of_band);
  const int in_band = number % (8 * p.tiles_n);
  const int m0 = (first_of_band + in_band % band) * BM, n0 = in_band / band * BN;
  // (every offset below is within the tile's rows, which the entry point keeps below 2^31 bytes)
  const __amdgpu_buffer_rsrc_t x_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(p.x + (long)m0 * p.ldx), 0, 0xffffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (long)n0 * p.ldw), 0, 0xffffffff, 0x00020000);
  int offset[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = (i * WAVES + wave) * 8 + lane / 8;
    const int piece = (lane % 8) ^ (row & 7);
    offset[i] = i * WAVES * 8 < BM ? 2 * (min(row, p.M - 1 - m0) * p.ldx + 8 * piece)
                                   : 2 * (min(row - BM, p.N - 1 - n0) * p.ldw + 8 * piece);
  }
  const int stages = p.K / GEMM_STAGE;
  auto ask = [&](int stage) {                                // (past the last one: the last again, never read)
    const int column = min(stage, stages - 1) * 2 * GEMM_STAGE;
    unsigned char* const into = lds[stage % STAGES];
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i * WAVES * 8 < BM ? x_rows : w_rows, (g_lds*)(into + (i * WAVES + wave) * 1024), 16,
                                               offset[i], column, 0, 0);
  };
  const int wm = wave % WM, wn = wave / WM;
  const int q = lane / 16, r = lane % 16;
  g_floatx4 acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = g_floatx4{0.f, 0.f, 0.f, 0.f};
  g_bf16x8 rows[AHEAD ? 2 : 1][2][TM], features[AHEAD ? 2 : 1][2][TN];     // the fragments of a stage's halves
  auto fetch = [&](int set, int stage, int half) {
    const unsigned char* const from = lds[stage % STAGES];
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int row = (wm * TM + m) * 16 + r;
      rows[set][half][m] = *reinterpret_cast<const g_bf16x8*>(from + 128 * row + 16 * ((4 * half + q) ^ (row & 7)));
    }
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int row = BM + (wn * TN + n) * 16 + r;
      features[set][half][n] = *reinterpret_cast<const g_bf16x8*>(from + 128 * row + 16 * ((4 * half + q) ^ (row & 7)));
    }
  };
  auto multiply = [&](int set, int half) {
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m)
        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(features[set][half][n], rows[set][half][m], acc[n][m], 0, 0, 0);
  };
  // this wave has read what it wanted of a stage, and its own part of the next one has arrived: behind the barrier the same
  // holds for all
  auto next_stage = [&]() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * LOADS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int stage = 0; stage < STAGES; ++stage) ask(stage);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * LOADS) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  fetch(0, 0, 0);
  if constexpr (AHEAD) {
    // few products a stage: the next stage's fragments are read, into a second set, while this one is multiplied
    fetch(0, 0, 1);
    for (int stage = 0; stage < stages; stage += 2) {
      next_stage();
      ask(stage + STAGES);
      fetch(1, stage + 1, 0);
      fetch(1, stage + 1, 1);
      multiply(0, 0);
      multiply(0, 1);
      __builtin_amdgcn_sched_barrier(0);
      next_stage();
      ask(stage + 1 + STAGES);
      fetch(0, stage + 2, 0);
      fetch(0, stage + 2, 1);
      if (stage + 1 < stages) {
        multiply(1, 0);
        multiply(1, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    // half a stage ahead, one load between every few products
    constexpr int PRODUCTS = TM * TN, FETCHES = TM + TN;
    constexpr int EACH = PRODUCTS / FETCHES > 0 ? PRODUCTS / FETCHES : 1;
    constexpr int BOTH = PRODUCTS / (FETCHES + LOADS) > 0 ? PRODUCTS / (FETCHES + LOADS) : 1;
    for (int stage = 0; stage < stages; ++stage) {
      fetch(0, stage, 1);
      multiply(0, 0);
#pragma unroll
      for (int i = 0; i < FETCHES; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);  // matrix products
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     // a load from LDS
      }
      __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS, 0);
      __builtin_amdgcn_sched_barrier(0);
      next_stage();
      ask(stage + STAGES);
      fetch(0, stage + 1, 0);
      multiply(0, 1);
#pragma unroll
      for (int i = 0; i < FETCHES + LOADS; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, BOTH, 0);
        if ((i % 2 == 0 && i / 2 < FETCHES) || i - (i + 1) / 2 >= LOADS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        else __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                    // a load from memory
      }
      __builtin_amdgcn_sched_group_barrier(0x008, PRODUCTS, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // nothing of the stages past the end may still be on its way to LDS when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // a lane holds four neighbouring features (4 q ..) of row r of every tile
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const long row = m0 + (wm * TM + m) * 16 + r;
    bf16_t* const out = (bf16_t*)p.out + row * p.ldo;
    if (EPI == EPI_ROWS_SWIGLU) {
#pragma unroll
      for (int n = 0; n < TN; n += 2) {
        // of a tile the lanes below 32 hold gate rows and those above the up rows of the same outputs: exchanged between
        // two tiles, the lower lanes have both of the first and the upper lanes both of the second
        const int first = n0 + (wn * TN + n) * 16;           // of the pair's features
        g_bf16x4 packed;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float a = acc[n][m][i], b = acc[n + 1][m][i];
          if (p.bias) {
            a += p.bias[min(first + 4 * q + i, p.N - 1)];
            b += p.bias[min(first + 16 + 4 * q + i, p.N - 1)];
          }
          const auto swapped = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
          // (rounded as by a product of its own with the activation behind it: the same bits either way, for 0.3 us, 640 x 4,096 x
          // 1,024 11.1 -> 11.4)
          const float gate = (float)(bf16_t)__builtin_bit_cast(float, (unsigned)swapped[0]);
          const float up = (float)(bf16_t)__builtin_bit_cast(float, (unsigned)swapped[1]);
          packed[i] = (bf16_t)(silu_bf16_f(gate) * up);
        }
        const int mine = first + 16 * (q / 2);               // the tile this lane has now (whole, as N is a multiple of 16)
        if (row < p.M && mine < p.N) *reinterpret_cast<g_bf16x4*>(out + mine / 2 + 4 * (q % 2)) = packed;
      }
    } else {
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int feature = n0 + (wn * TN + n) * 16 + 4 * q;
        g_floatx4 value = acc[n][m];
        if (p.bias) {
#pragma unroll
          for (int i = 0; i < 4; ++i) value[i] += p.bias[min(feature + i, p.N - 1)];
        }
        if (row >= p.M) continue;
        if (EPI == EPI_ROWS_F32) {
          float* const sums = (float*)p.out + row * p.ldo;
          if (p.whole && feature + 3 < p.N) {
            *reinterpret_cast<g_floatx4*>(sums + feature) = value;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (feature + i < p.N) sums[feature + i] = value[i];
          }
        } else {
          g_bf16x4 packed;
#pragma unroll
          for (int i = 0; i < 4; ++i) packed[i] = (bf16_t)value[i];
          if (p.whole && feature + 3 < p.N) {
            *reinterpret_cast<g_bf16x4*>(out + feature) = packed;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (feature + i < p.N) out[feature + i] = packed[i];
          }
        }
      }
    }
  }
#endif
}

template <int BM, int BN, int WM, int WN, int STAGES, bool AHEAD>
static void launch_rows_gemm(RowsGemm p, int epilogue, hipStream_t stream) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  const int per_die = (int)(((long)p.tiles_m * p.tiles_n + 7) / 8);
  if (epilogue == EPI_ROWS_SWIGLU) rows_gemm_kernel<BM, BN, WM, WN, STAGES, AHEAD, EPI_ROWS_SWIGLU><<<8 * per_die, WAVE * WM * WN, 0, stream>>>(p);
  else if (epilogue == EPI_ROWS_F32) rows_gemm_kernel<BM, BN, WM, WN, STAGES, AHEAD, EPI_ROWS_F32><<<8 * per_die, WAVE * WM * WN, 0, stream>>>(p);
  else rows_gemm_kernel<BM, BN, WM, WN, STAGES, AHEAD, EPI_ROWS_PLAIN><<<8 * per_die, WAVE * WM * WN, 0, stream>>>(p);
}

// The tile with the least estimate of its time in microseconds: by the workgroups of the fullest compute unit, as measured
// over 33 to 4,096 rows, 256 to 8,192 features and K of 512 to 2,048 (medians).  At K = 1,024, with one / two / three / four of
// them: 64 x 64 6.7 / 9.8 / 15.2 / 18.5, 64 x 128 8.2 / 14.2 / 22 / 28, 128 x 128 with two stages, two of which run beside each
// other, 13.5 / 21.7 / 33 / 40, with four stages, one at a time, 11.4 / 25.  The choice is the fastest of the four or within
// 15 % of it, 0.4 % behind it on average.
static int rows_gemm_tile(int M, int N, int K) {
  auto fullest = [&](long rows, long features) { return (int)(((M + rows - 1) / rows * ((N + features - 1) / features) + 255) / 256); };
  const float k = K / 1024.f;
  const int large = fullest(128, 128);
  const float time[4] = {2.3f + fullest(64, 64) * (0.6f + 3.68f * k), 2.f + fullest(64, 128) * (1.1f + 5.5f * k),
                         large > 1 ? 1e9f : 4.8f + 6.85f * k, 2.5f + (3.5f + 15.6f * k) * (large / 2) + (1.f + 10.5f * k) * (large % 2)};
  int best = 0;
  for (int i = 1; i < 4; ++i)
    if (time[i] < time[best]) best = i;
  return best;
}

// K a multiple of 64; rows of x and W start at 16 bytes.  epilogue 1: N features in tiles of 8 gate and 8 up rows, out
// [M, N / 2] bfloat16; 2: out float32.  tile: 0 .. 3, or -1 for the rule's choice.
extern "C" int mi_rows_gemm(const void* x, long ldx, const void* w, long ldw, const float* bias, void* out, long ldo, int M,
                            int N, int K, int epilogue, int tile, hipStream_t stream) {
  const bool swiglu = epilogue == EPI_ROWS_SWIGLU;
  if (!x || !w || !out || M <= 0 || N <= 0 || K <= 0 || ldx < K || ldw < K || ldo < (swiglu ? N / 2 : N) || tile < -1 || tile > 3 || epilogue < 0 ||
      epilogue > EPI_ROWS_F32)
    return ERR_BAD_ARGUMENT;
  if (K % GEMM_STAGE || ldx % 8 || ldw % 8 || (uintptr_t)x % 16 || (uintptr_t)w % 16 || ldx > (1 << 22) || ldw > (1 << 22) ||
      (long)(M / 64 + 1) * (N / 64 + 1) > (1 << 28) || (swiglu && (N % 16 || ldo % 4 || (uintptr_t)out % 8)))
    return ERR_UNSUPPORTED_SIZE;
  RowsGemm p = {(const bf16_t*)x, (const bf16_t*)w, bias, out, (int)ldx, (int)ldw, ldo, M, N, K, 0, 0,
                ldo % 4 == 0 && (uintptr_t)out % (epilogue == EPI_ROWS_F32 ? 16 : 8) == 0};
  switch (tile < 0 ? rows_gemm_tile(M, N, K) : tile) {
    case 0: launch_rows_gemm<64, 64, 4, 2, 4, true>(p, epilogue, stream); break;
    case 1: launch_rows_gemm<64, 128, 2, 4, 3, true>(p, epilogue, stream); break;
    case 2: launch_rows_gemm<128, 128, 2, 4, 4, false>(p, epilogue, stream); break;
    default: launch_rows_gemm<128, 128, 2, 4, 2, false>(p, epilogue, stream); break;
  }
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}
