// Prompt attention on the matrix cores with keys and values that the waves of a workgroup share through LDS:
// bfloat16, heads of 64 or 128 with values as wide, for portions whose tiles are mostly full.
#include <type_traits>

#include "attn_mfma.h"

// One workgroup: a tile of up to 64 consecutive tokens of one lane x NSET query heads of one kv head.  Its eight waves
// are two groups of four; in a group wave w has the tokens 16 w .. 16 w + 15 of the tile (NSET sets of 16 columns),
// and the two groups take turns at the stages of 64 keys, so each group walks every other stage.  A stage's K and V
// pieces go from the cache pages through registers to the group's half of LDS (two buffers: the pieces of the next
// stage are on their way while this one is worked on; one barrier a stage), in the order in which the matrix
// instructions take them: a fragment is 64 pieces of 16 bytes one after the other, read and written without bank
// conflicts.  The two groups' sums are merged through LDS at the end.
//
// Within a step of 32 keys, row 4 a + b of score tile t is key 8 a + 4 t + b: the probabilities a lane holds after the
// softmax (four of either tile) are then those of eight consecutive keys, and their V piece is one load of 16 bytes.
//
// What bounds it: the instructions of the softmax (about 850 cycles of a wave for 64 keys and 16 columns), the reads of
// the fragments from LDS and the fetches from L2, about a third of the time each; they overlap only in part.  Heads of
// 64 fit two workgroups on a compute unit, heads of 128 one; of those two heads a workgroup halve the reads and the
// fetches of a column.  Measured against the kernel whose waves read their own keys (prefill_attention_kernel) in
// replayed steps, pages of 16: 8 heads of 64 over 2 kv heads, 1,536 tokens 28.4 -> 21.9 us, 4 prompts of 512 28.3 -> 14.1;
// 12 heads of 128 over 2, 1,999 tokens 95 -> 79, 1,536 behind 6,000 249 -> 199; 8 prompts of 256, 32 heads of 128 over 8,
// 123 -> 36.5; with the logarithmic bias 1,999 tokens of 12 of 128 225 -> 90, with a window of 1,024 too 1,536 of 8 of 64
// 30.3 -> 20.6.  Where it is the slower one is at ops.shared_prefill_heads, with both sides.  The error of its
// results against 64 bits is the smaller one (2,048 tokens, scores of deviation one: 0.00195 against 0.00198, relative;
// behind 1,024: 0.00203 against 0.00213), because every step of 32 keys has its own reference.
// Tried without gain: the two groups half a turn apart (the phases only get longer: 36.7 us in place of 28.2), two
// stages on their way; a reference that moves only where a column's maximum does saves 2 us of 28 and costs precision.
#define SHARED_STAGE 64
#define SHARED_WAVES 8
#define SHARED_PAGES 1024            // of a walk's list of pages in LDS; a longer context takes several walks
#define SHARED_SPARE 32              // entries for the four stages that are asked for past the end, in pages of 8

// U: steps of 32 keys whose scores are formed before the softmax.
// BIAS: BIAS_LOG, the scores lose log_bias[head] = (r1, r2) -> r1 * ln(1 + r2 * distance).  sinks (may be null): one more term
// exp(sinks[head]) of the softmax's denominator.
template <int DH, int NSET, int U, int BIAS = BIAS_NONE>
__global__ void __launch_bounds__(SHARED_WAVES * WAVE, DH * NSET == 64 && BIAS == BIAS_NONE ? 4 : 2)
prefill_shared_kernel(const bf16_t* __restrict__ q, long q_ld, int Hq, int Hkv, const bf16_t* __restrict__ k_base,
                      const bf16_t* __restrict__ v_base, long page_stride, int page_shift,
                      const int* __restrict__ block_tables, int max_pages, const int* __restrict__ tiles,
                      const int* __restrict__ cu_seqlens, const int* __restrict__ start_pos, float scale, int window,
                      bf16_t* __restrict__ out, long out_ld, const float* __restrict__ log_bias,
                      const float* __restrict__ sinks) {
  constexpr int FRAGMENTS = DH / 8;              // of K in a stage, and as many of V
  constexpr int PIECES = FRAGMENTS / 4;          // of either that a thread moves
  // two heads of 128: fragments are asked for four at a time, or they would spill
  constexpr bool TIGHT = DH * NSET > 128;
  constexpr int KD = DH / 32, VD = DH / 16;
  constexpr int ITEMS = 2 + 4 * VD;              // m, l and the sums of one set
  constexpr int STAGE_BYTES = 2 * FRAGMENTS * WAVE * 16;
  constexpr int MERGE_BYTES = 4 * NSET * ITEMS * WAVE * 4;
  constexpr int BYTES = 4 * STAGE_BYTES > MERGE_BYTES ? 4 * STAGE_BYTES : MERGE_BYTES;
  __shared__ __attribute__((aligned(16))) unsigned char area[BYTES];
  __shared__ unsigned long long pages[SHARED_PAGES + SHARED_SPARE];
  const int tile = (blockIdx.z & 1) ? blockIdx.x : gridDim.x - 1 - blockIdx.x;
  const int kvh = blockIdx.y;
  const int G = Hq / Hkv;
  const int head0 = kvh * G + blockIdx.z * NSET;
  const int request = tiles[2 * tile];
  if (request < 0) return;
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int group = wave / 4;
  const int w = wave % 4;
  const int qd = lane / 16;
  const int n = lane % 16;
  const int lane_end = cu_seqlens[request + 1];
  const int tile_token = tiles[2 * tile + 1];
  if (tile_token >= lane_end) return;
  const int base_position = start_pos[request] - cu_seqlens[request];
  const int tile_last = base_position + min(tile_token + 63, lane_end - 1);
  const int first_token = tile_token + 16 * w;
  const int token = first_token + n;
  const bool has_query = token < lane_end;
  const int first_position = base_position + first_token;
  const int last_position = base_position + min(first_token + 15, lane_end - 1);     // below first_position: no token
  const bool full = first_token + 16 <= lane_end && (blockIdx.z + 1) * NSET <= G;

  mfma_bf16x8 q_frag[NSET][KD];
  int col_pos[NSET], col_first[NSET];
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const bool valid = has_query && blockIdx.z * NSET + s < G;
    col_pos[s] = valid ? base_position + token : -1;
    col_first[s] = first_visible_key(max(col_pos[s], 0), window);
#pragma unroll
    for (int kk = 0; kk < KD; ++kk) {
      if (valid) {
        q_frag[s][kk] = *reinterpret_cast<const mfma_bf16x8*>(q + (long)token * q_ld + (long)(head0 + s) * DH + 32 * kk + 8 * qd);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) q_frag[s][kk][j] = (bf16_t)0.f;
      }
    }
  }
  AttnAccumulator<DH, NSET> acc;
  acc.clear();
  float highest[NSET];                           // score of a column so far
#pragma unroll
  for (int s = 0; s < NSET; ++s) highest[s] = -INFINITY;
  const float scale_log2 = scale * 1.4426950408889634f;
  const float unit = BIAS == BIAS_NONE ? scale_log2 : 1.f;   // of a score towards units of log2: biased ones are there already
  float bias_r1[NSET], bias_r2[NSET];
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const int head = min(head0 + s, Hq - 1);
    bias_r1[s] = BIAS == BIAS_LOG ? log_bias[2 * head] : 0.f;
    bias_r2[s] = BIAS == BIAS_LOG ? log_bias[2 * head + 1] : 0.f;
  }
  const int page_mask = (1 << page_shift) - 1;
  const int key_lo = first_visible_key(base_position + tile_token, window) / SHARED_STAGE * SHARED_STAGE;
  const int key_hi = tile_last + 1;
  // where a whole wave sees every key from here on (its last column's first key)
  const int wave_lo = first_visible_key(max(first_position, 0), window);
  const int open_lo = first_visible_key(last_position, window);
  const int* request_pages = block_tables + (long)request * max_pages;
  mfma_uintx4* const buffers = reinterpret_cast<mfma_uintx4*>(area) + group * 2 * (STAGE_BYTES / 16);

  // What a thread moves of a stage: piece i of K and of V is fragment w + 4 i.  A piece's address is that of its page (the
  // list in LDS) plus an offset that no stage changes, plus for pages of more than a stage the stage's own place in its
  // page: stages begin at multiples of 64 and pages are powers of two.
  const long to_values = (const char*)v_base - (const char*)k_base;

  // scores, softmax and values of U steps of 32 keys, the first of them step `step` of the stage
  auto attend = [&](auto masked, const mfma_uintx4* buffer, int step, int k0) {
    constexpr bool MASKED = decltype(masked)::value;
    mfma_floatx4 score[NSET][2 * U];              // step st, tile t: [2 * st + t]
#pragma unroll
    for (int s = 0; s < NSET; ++s)
#pragma unroll
      for (int t = 0; t < 2 * U; ++t) score[s][t] = mfma_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2 * U; ++t)
#pragma unroll
      for (int kk = 0; kk < KD; ++kk) {
        const mfma_bf16x8 k = __builtin_bit_cast(mfma_bf16x8, buffer[((2 * step + t) * KD + kk) * WAVE + lane]);
#pragma unroll
        for (int s = 0; s < NSET; ++s)
          score[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, q_frag[s][kk], score[s][t], 0, 0, 0);
        if (TIGHT && kk % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
    // the largest score of every column in every step, in its four lanes
    float top[NSET][U];
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      if (BIAS == BIAS_LOG) {                    // a key past the column's position gets a bias of anything: it is masked
#pragma unroll
        for (int t = 0; t < 2 * U; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float distance = (float)(col_pos[s] - (k0 + 8 * qd + 32 * (t / 2) + 4 * (t % 2) + i));
            score[s][t][i] = fmaf(score[s][t][i], scale_log2, -bias_r1[s] * __log2f(fmaf(bias_r2[s], fmaxf(distance, 0.f), 1.f)));
          }
      }
      if (MASKED) {
        // visible keys of the column relative to the lane's first: lo .. lo + span, one unsigned compare a score (an
        // empty range gets a lo that no offset reaches)
        const bool any = col_pos[s] >= 0;
        const int lo = any ? col_first[s] - (k0 + 8 * qd) : 0x40000000;
        const unsigned span = any ? (unsigned)(col_pos[s] - col_first[s]) : 0u;
#pragma unroll
        for (int t = 0; t < 2 * U; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            score[s][t][i] = (unsigned)(32 * (t / 2) + 4 * (t % 2) + i - lo) <= span ? score[s][t][i] : -INFINITY;
      }
#pragma unroll
      for (int st = 0; st < U; ++st) {
        float most = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; ++i) most = fmaxf(most, score[s][2 * st + i / 4][i % 4]);
        top[s][st] = most;
      }
#pragma unroll
      for (int st = 0; st < U; ++st) top[s][st] = fmaxf(top[s][st], __shfl_xor(top[s][st], 16, WAVE));
#pragma unroll
      for (int st = 0; st < U; ++st) top[s][st] = fmaxf(top[s][st], __shfl_xor(top[s][st], 32, WAVE));
    }
    mfma_bf16x8 p_frag[NSET][U];
    float correction[NSET][U];
#pragma unroll
    for (int s = 0; s < NSET; ++s)
#pragma unroll
      for (int st = 0; st < U; ++st) {
        // The sums are held relative to the largest score of the step's keys, not of all keys so far, as long as that is
        // within 2^16 of it: the largest weight of every step is then one, which bfloat16 holds exactly.
        const float most = top[s][st] * unit;                                   // scale > 0: the maximum stays the maximum
        highest[s] = fmaxf(highest[s], most);
        const float reference = fmaxf(most, highest[s] - 16.f);
        const float m_safe = reference == -INFINITY ? 0.f : reference;          // nothing visible yet
        correction[s][st] = __builtin_amdgcn_exp2f(acc.m[s] - m_safe);
        acc.m[s] = reference;
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = __builtin_amdgcn_exp2f(fmaf(score[s][2 * st + t][i], unit, -m_safe));
            sum += p;
            p_frag[s][st][4 * t + i] = (bf16_t)p;
          }
        acc.l[s] = acc.l[s] * correction[s][st] + sum;
      }
#pragma unroll
    for (int st = 0; st < U; ++st)
#pragma unroll
      for (int dt = 0; dt < VD; ++dt) {
        mfma_uintx4 v = buffer[(FRAGMENTS + (step + st) * VD + dt) * WAVE + lane];
        if (MASKED) {
          // cells outside the wave's keys (not written yet, not for its columns, or behind their windows in pages that
          // were given back) stay out of the product
          const int key = k0 + 32 * st + 8 * qd;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (key + 2 * j < wave_lo || key + 2 * j > last_position) v[j] &= 0xffff0000u;
            if (key + 2 * j + 1 < wave_lo || key + 2 * j + 1 > last_position) v[j] &= 0x0000ffffu;
          }
        }
#pragma unroll
        for (int s = 0; s < NSET; ++s) {
#pragma unroll
          for (int i = 0; i < 4; ++i) acc.o[s][dt][i] *= correction[s][st];
          acc.o[s][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mfma_bf16x8, v), p_frag[s][st],
                                                                 acc.o[s][dt], 0, 0, 0);
        }
        if (TIGHT && dt % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
  };

  for (int from = key_lo; from < key_hi;) {
    const int first_page = from >> page_shift;
    const int room = ((first_page + SHARED_PAGES) << page_shift) - from;
    const int to = min(key_hi, from + room / SHARED_STAGE * SHARED_STAGE);
    const int listed = ((to - 1) >> page_shift) - first_page;
    __syncthreads();
    for (int i = threadIdx.x; i <= listed + SHARED_SPARE; i += SHARED_WAVES * WAVE)
      pages[i] = (unsigned long long)(k_base + (long)max(request_pages[min(first_page + min(i, listed), max_pages - 1)], 0) * page_stride);
    __syncthreads();
    const int stages = (to - from + SHARED_STAGE - 1) / SHARED_STAGE;
    const int turns = (stages + 1) / 2;
    mfma_uintx4 held[2 * PIECES];
    auto fetch = [&](int k0) {
      const unsigned long long* const list = pages + (k0 >> page_shift) - first_page;
      const unsigned within = 2 * (k0 & page_mask);
      // formed anew for every stage: kept, these offsets would take the registers of the sums
      int at = lane;
      asm volatile("" : "+v"(at));
      const int row = at % 16, piece = 8 * (at / 16);
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int f = w + 4 * i;
        const int key = 32 * (f / (2 * KD)) + 8 * (row / 4) + 4 * (f / KD % 2) + row % 4;
        const unsigned offset = 2 * ((((unsigned)kvh << page_shift) + (key & page_mask)) * DH + 32 * (f % KD) + piece);
        held[i] = *reinterpret_cast<const mfma_uintx4*>(list[key >> page_shift] + (offset + within * DH));
      }
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        const int f = w + 4 * i;
        const int key = 32 * (f / VD) + piece;
        const unsigned offset = 2 * ((((unsigned)kvh * DH + 16 * (f % VD) + row) << page_shift) + (key & page_mask));
        held[PIECES + i] = *reinterpret_cast<const mfma_uintx4*>(list[key >> page_shift] + to_values + (offset + within));
      }
    };
    auto lay = [&](mfma_uintx4* buffer) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) buffer[(w + 4 * i) * WAVE + lane] = held[i];
#pragma unroll
      for (int i = 0; i < PIECES; ++i) buffer[(FRAGMENTS + w + 4 * i) * WAVE + lane] = held[PIECES + i];
    };
    auto work = [&](const mfma_uintx4* buffer, int stage_key) {
#pragma unroll 1
      for (int step = 0; step < 2; step += U) {
        const int k0 = stage_key + 32 * step;
        if (k0 > last_position || k0 >= to || k0 + 32 * U <= wave_lo) continue;
        if (!full || k0 + 32 * U - 1 > first_position || k0 < open_lo)
          attend(std::true_type(), buffer, step, k0);
        else
          attend(std::false_type(), buffer, step, k0);
      }
    };
    // the next stage is on its way while one is worked on; past the end it holds cells of the last page, never used
    fetch(from + SHARED_STAGE * group);
    for (int turn = 0; turn < turns; ++turn) {
      const int key = from + SHARED_STAGE * (2 * turn + group);
      const mfma_uintx4* const buffer = buffers + (turn & 1) * (STAGE_BYTES / 16);
      lay(buffers + (turn & 1) * (STAGE_BYTES / 16));
      __syncthreads();
      fetch(key + 2 * SHARED_STAGE);
      __builtin_amdgcn_sched_barrier(0);
      work(buffer, key);
    }
    from = to;
  }

  // merge: the second group's sums through LDS to the first
  float* const part = reinterpret_cast<float*>(area);
  __syncthreads();
  if (group == 1) {
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      float* const mine = part + (w * NSET + s) * ITEMS * WAVE + lane;
      mine[0] = acc.m[s];
      mine[WAVE] = acc.l[s];
#pragma unroll
      for (int dt = 0; dt < VD; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[(2 + 4 * dt + i) * WAVE] = acc.o[s][dt][i];
    }
  }
  __syncthreads();
  if (group == 1) return;
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    const float* const other = part + (w * NSET + s) * ITEMS * WAVE + lane;
    const float m_other = other[0];
    // the sink, in the scores' units of log2: it may be the largest term
    const float sink = sinks ? sinks[min(head0 + s, Hq - 1)] * 1.4426950408889634f : -INFINITY;
    const float m = fmaxf(fmaxf(acc.m[s], m_other), sink);
    const float factor = acc.m[s] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(acc.m[s] - m);
    const float factor_other = m_other == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_other - m);
    float l = acc.l[s] * factor + other[WAVE] * factor_other;
    l += __shfl_xor(l, 16, WAVE);
    l += __shfl_xor(l, 32, WAVE);
    if (sinks) l += __builtin_amdgcn_exp2f(sink - m);       // once for the column: no key, no value
    if (col_pos[s] < 0) continue;
    const float inverse = 1.f / l;
    bf16_t* const o = out + (long)token * out_ld + (long)(head0 + s) * DH;
#pragma unroll
    for (int dt = 0; dt < VD; ++dt) {
      mfma_bf16x4 packed;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        packed[i] = (bf16_t)((acc.o[s][dt][i] * factor + other[(2 + 4 * dt + i) * WAVE] * factor_other) * inverse);
      *reinterpret_cast<mfma_bf16x4*>(o + 16 * dt + 4 * qd) = packed;
    }
  }
}

// tiles: int32 [n_tiles, 2] = (lane or -1, first token row) of runs of up to 64 tokens of one lane.
// Returns ERR_UNSUPPORTED_SIZE for shapes it does not cover (the caller uses mi_prefill_attention).
extern "C" int mi_prefill_attention_shared(const void* q, long q_ld, int Hq, int Hkv, int dh, const void* k_base,
                                           const void* v_base, long page_stride, int page_size, const int* block_tables,
                                           int max_pages, const int* tiles, int n_tiles, const int* cu_seqlens,
                                           const int* start_pos, float scale, int window, int nset, void* out,
                                           long out_ld, const float* log_bias, const float* sinks, hipStream_t stream) {
  if (n_tiles <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0 || page_size <= 0 || max_pages <= 0)
    return ERR_BAD_ARGUMENT;
  const int G = Hq / Hkv;
  if ((dh != 64 && dh != 128) || page_size < 8 || (page_size & (page_size - 1)) != 0 || page_stride % 8 != 0 ||
      (uintptr_t)k_base % 16 != 0 || (uintptr_t)v_base % 16 != 0 || q_ld % 8 != 0 || (uintptr_t)q % 16 != 0 ||
      out_ld % 4 != 0 || (uintptr_t)out % 8 != 0 || Hkv > 65535 || G > 64 || n_tiles > (1 << 28) ||
      2L * Hkv * dh * page_size > (1L << 32))      // (offsets into a page are 32 bits)
    return ERR_UNSUPPORTED_SIZE;
  if (nset != 1 && (nset != 2 || dh != 128)) return ERR_BAD_ARGUMENT;
  int page_shift = 0;
  while ((1 << page_shift) < page_size) ++page_shift;
  const dim3 grid(n_tiles, Hkv, (G + nset - 1) / nset);
#define SHARED_LAUNCH(DH_, NSET_, U_, BIAS_)                                                                      \
  prefill_shared_kernel<DH_, NSET_, U_, BIAS_><<<grid, SHARED_WAVES * WAVE, 0, stream>>>(                        \
      (const bf16_t*)q, q_ld, Hq, Hkv, (const bf16_t*)k_base, (const bf16_t*)v_base, page_stride, page_shift,    \
      block_tables, max_pages, tiles, cu_seqlens, start_pos, scale, window, (bf16_t*)out, out_ld, log_bias, sinks)
#define SHARED_CASE(DH_, NSET_, U_)                                                                              \
  if (dh == DH_ && nset == NSET_) {                                                                              \
    if (log_bias) SHARED_LAUNCH(DH_, NSET_, U_, BIAS_LOG);                                                       \
    else SHARED_LAUNCH(DH_, NSET_, U_, BIAS_NONE);                                                               \
  }
  SHARED_CASE(64, 1, 2) SHARED_CASE(128, 1, 2) SHARED_CASE(128, 2, 1)
#undef SHARED_LAUNCH
#undef SHARED_CASE
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}
