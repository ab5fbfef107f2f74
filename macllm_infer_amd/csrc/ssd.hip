// The Mamba2 selective scan for prompt portions in bfloat16, in chunks on the matrix cores
// (the "state space duality" form).  Per lane (consecutive tokens of one request), head h,
// group g of the head, with delta_t = softplus(dt_t + dt_bias), a_t = delta_t * A_h and the
// recurrence of mamba2.hip
//     S_t = exp(a_t) S_{t-1} + delta_t x_t (outer) B_t,   y_t = S_t . C_t + D_h x_t,
// cut the lane into chunks of Q tokens and let L_t be the running sum of a inside a chunk:
//     y_t   = exp(L_t) (S_in . C_t) + sum_{s<=t} exp(L_t - L_s) delta_s (C_t . B_s) x_s + D_h x_t
//     S_out = exp(L_end) S_in + sum_s exp(L_end - L_s) delta_s x_s (outer) B_s
// Every exponent is a difference of a non-increasing sequence taken forwards, so it is <= 0 and
// nothing overflows.  The result does not depend on Q beyond rounding.  Five kernels (the last three are one launch
// where every lane is one chunk, see ssd_single_kernel):
//     prepare     delta, L                                    (one workgroup per chunk and head)
//     transpose   x and B of each chunk, token-contiguous and zero-padded to Q: [chunk, E + G*N, Q]
//     chunk_state sum_s exp(L_end - L_s) delta_s x_s (outer) B_s  per chunk and head (matrix cores)
//     state_pass  S_in of every chunk from the slot's state, serially over a lane's chunks; the
//                 lane's final state goes back to the slot (float32 throughout)
//     chunk_scan  y: the two sums above on the matrix cores, (C . B^T) shared by the heads of a group;
//                 optionally the gate y * SiLU(z) on the way out
// Operand layouts follow attn_mfma.h: a matrix-core operand wants its contraction index
// contiguous, which is the state index n for C . B^T and S_in . C, and the token for the other
// two products, hence the transposed copies.
// (reference recurrence: crates/macllm-kernels/src/mamba2.rs:259-288; the reference scans token by token.)
#include "attn_prefill.h"
#include "read_ahead.h"
#include "rope_rows.h"

typedef __bf16 s_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 s_bf16x4 __attribute__((ext_vector_type(4)));
typedef float s_floatx4 __attribute__((ext_vector_type(4)));

#define SSD_MAX_Q 256
#define SSD_HEADS_PER_BLOCK 1

// chunk table: int32 [n_chunks, 4] = (lane, first token row, length, index of the chunk within its lane)

// ---------------------------------------------------------------- prepare
// delta[t, h] = softplus(dt + bias); cum[t, h] = sum of delta*A over the chunk up to t (inclusive).
__device__ __forceinline__ void ssd_prepare_block(const bf16_t* __restrict__ dt, long dt_ld, const float* __restrict__ dt_bias,
                                  const float* __restrict__ A, const int* __restrict__ chunks, int H,
                                  float* __restrict__ delta, float* __restrict__ cum, int chunk, int head,
                                  float* wave_total) {
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  const int s = threadIdx.x;
  const int lane = s & (WAVE - 1);
  const int wave = s / WAVE;
  float step = 0.f, a = 0.f;
  if (s < length) {
    step = softplus_f((float)dt[(long)(t0 + s) * dt_ld + head] + dt_bias[head]);
    a = step * A[head];
  }
  float running = a;                       // inclusive scan inside the wave
#pragma unroll
  for (int offset = 1; offset < WAVE; offset <<= 1) {
    const float other = __shfl_up(running, offset, WAVE);
    if (lane >= offset) running += other;
  }
  if (lane == WAVE - 1) wave_total[wave] = running;
  __syncthreads();
  float before = 0.f;
  for (int w = 0; w < wave; ++w) before += wave_total[w];
  if (s < length) {
    delta[(long)(t0 + s) * H + head] = step;
    cum[(long)(t0 + s) * H + head] = running + before;
  }
}

// ---------------------------------------------------------------- transpose
// out[chunk, channel, s] = xbc[t0 + s, channel] for s < length, 0 for the padding up to Q.
// 64 channels of a chunk per workgroup: 16-byte loads along the channels, 2-byte stores into a
// transposed LDS tile whose row stride (Q + 2 elements = an odd number of banks) keeps them
// apart, 4-byte LDS reads and 16-byte stores along the tokens.
__device__ __forceinline__ void ssd_transpose_block(const bf16_t* __restrict__ xbc, long ld, int channels, const int* __restrict__ chunks,
                                    int Q, bf16_t* __restrict__ out, int chunk, int c0, bf16_t* tile) {
  const int stride = Q + 2;
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  for (int index = threadIdx.x; index < Q * 8; index += 256) {
    const int s = index / 8;
    const int c = (index % 8) * 8;
    s_bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16_t)0.f;
    if (s < length && c0 + c < channels) v = *reinterpret_cast<const s_bf16x8*>(xbc + (long)(t0 + s) * ld + c0 + c);
#pragma unroll
    for (int j = 0; j < 8; ++j) tile[(c + j) * stride + s] = v[j];
  }
  __syncthreads();
  const int vectors = Q / 8;
  for (int index = threadIdx.x; index < 64 * vectors; index += 256) {
    const int c = index / vectors;
    const int s = (index % vectors) * 8;
    if (c0 + c >= channels) continue;
    const unsigned* words = reinterpret_cast<const unsigned*>(tile + c * stride + s);
    uint4 v;
    v.x = words[0];
    v.y = words[1];
    v.z = words[2];
    v.w = words[3];
    *reinterpret_cast<uint4*>(out + ((long)chunk * channels + c0 + c) * Q + s) = v;
  }
}

// Both in one launch (they do not depend on each other and each is too small to fill the GPU): rows
// 0 .. H-1 of the grid prepare a head, the rows after transpose 64 channels.
__global__ void __launch_bounds__(256)
ssd_prepare_transpose_kernel(const bf16_t* __restrict__ dt, long dt_ld, const float* __restrict__ dt_bias,
                             const float* __restrict__ A, const int* __restrict__ chunks, int H, float* __restrict__ delta,
                             float* __restrict__ cum, const bf16_t* __restrict__ xbc, long xbc_ld, int channels, int Q,
                             bf16_t* __restrict__ TT) {
  __shared__ __align__(4) bf16_t tile[64 * (SSD_MAX_Q + 2)];
  __shared__ float wave_total[SSD_MAX_Q / WAVE];
  if ((int)blockIdx.y < H)
    ssd_prepare_block(dt, dt_ld, dt_bias, A, chunks, H, delta, cum, blockIdx.x, blockIdx.y, wave_total);
  else
    ssd_transpose_block(xbc, xbc_ld, channels, chunks, Q, TT, blockIdx.x, ((int)blockIdx.y - H) * 64, tile);
}

// ---------------------------------------------------------------- conv, fused with the transpose
// The causal depthwise conv + SiLU of mamba2.hip (conv1d_silu) on a chunk's tokens and 64 channels, from the
// raw projection rows: the result goes to xbc[t, channel] (row-major, what the chunk scan reads for C, B and
// the skip) and, for the channels of x and B, into the transposed copy as well.  A thread takes 8 channels and
// 4 consecutive tokens; the K-1 rows before a chunk are the lane's previous tokens, or the request's conv
// tail when the chunk opens the lane.  All loads first, none under a condition (rows and channels that do
// not exist are clamped and dropped).  The tail itself is updated later, by ssd_tail_block, once every
// chunk has read it.
template <int K>
__device__ __forceinline__ void ssd_conv_block(const bf16_t* __restrict__ u, long u_ld, int C, const float* __restrict__ conv_w,
                               const float* __restrict__ conv_b, const bf16_t* __restrict__ conv_state,
                               const int* __restrict__ chunks, const int* __restrict__ slot_ids, int Q,
                               bf16_t* __restrict__ xbc, long xbc_ld, int tt_channels, bf16_t* __restrict__ TT,
                               int chunk, int c0, bf16_t* tile) {
  constexpr int ROWS = 4;
  const int stride = Q + 2;
  const int lane_id = chunks[4 * chunk];
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  const bool opens = chunks[4 * chunk + 3] == 0;
  const bf16_t* tail = conv_state + (long)slot_ids[lane_id] * (K - 1) * C;
  const long first_row = opens ? (long)t0 : (long)t0 - (K - 1);
  const float* bias_or_taps = conv_b ? conv_b : conv_w;
  for (int item = threadIdx.x; item < (Q / ROWS) * 8; item += 256) {
    const int s0 = (item / 8) * ROWS;
    const int c = (item % 8) * 8;
    const bool real = c0 + c < C;
    const int channel = real ? c0 + c : C - 8;
    s_bf16x8 window[ROWS + K - 1], before[K - 1];
#pragma unroll
    for (int j = 0; j < ROWS + K - 1; ++j) {
      const long row = min(max((long)t0 + s0 - (K - 1) + j, first_row), (long)t0 + length - 1);
      window[j] = *reinterpret_cast<const s_bf16x8*>(u + row * u_ld + channel);
    }
#pragma unroll
    for (int j = 0; j < K - 1; ++j) before[j] = *reinterpret_cast<const s_bf16x8*>(tail + (long)j * C + channel);
    s_floatx4 taps[2 * K];                          // conv_w[channel .. channel+8, 0 .. K): 8K contiguous floats
#pragma unroll
    for (int j = 0; j < 2 * K; ++j) taps[j] = *reinterpret_cast<const s_floatx4*>(conv_w + (long)channel * K + 4 * j);
    const s_floatx4 b_lo = *reinterpret_cast<const s_floatx4*>(bias_or_taps + channel);
    const s_floatx4 b_hi = *reinterpret_cast<const s_floatx4*>(bias_or_taps + channel + 4);
    if (opens && s0 == 0) {
#pragma unroll
      for (int j = 0; j < K - 1; ++j) window[j] = before[j];
    }
    auto tap = [&](int cc, int k) { return taps[(cc * K + k) / 4][(cc * K + k) % 4]; };
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int position = s0 + i;
      float sum[8];
#pragma unroll
      for (int cc = 0; cc < 8; ++cc) sum[cc] = conv_b ? (cc < 4 ? b_lo[cc] : b_hi[cc - 4]) : 0.f;
#pragma unroll
      for (int k = 0; k < K; ++k)
#pragma unroll
        for (int cc = 0; cc < 8; ++cc) sum[cc] += tap(cc, k) * (float)window[i + k][cc];
      s_bf16x8 result;
      const bool live = real && position < length;
#pragma unroll
      for (int cc = 0; cc < 8; ++cc) result[cc] = live ? (bf16_t)silu_bf16_f(sum[cc]) : (bf16_t)0.f;
      if (live) *reinterpret_cast<s_bf16x8*>(xbc + (long)(t0 + position) * xbc_ld + channel) = result;
#pragma unroll
      for (int cc = 0; cc < 8; ++cc) tile[(c + cc) * stride + position] = result[cc];
    }
  }
  __syncthreads();
  const int vectors = Q / 8;
  for (int index = threadIdx.x; index < 64 * vectors; index += 256) {
    const int c = index / vectors;
    const int position = (index % vectors) * 8;
    if (c0 + c >= tt_channels) continue;
    const unsigned* words = reinterpret_cast<const unsigned*>(tile + c * stride + position);
    uint4 v;
    v.x = words[0];
    v.y = words[1];
    v.z = words[2];
    v.w = words[3];
    *reinterpret_cast<uint4*>(TT + ((long)chunk * tt_channels + c0 + c) * Q + position) = v;
  }
}

// ---------------------------------------------------------------- attention beside the scan
// A layer whose attention and state-space mixer read the same projected rows runs two chains of small launches that do
// not depend on each other: rotation and cache write, then the attention; conv and prepare, then the scan.  In a short
// prompt none of them fills the GPU and each costs its launch and its round trips, so the attention's two run as further
// workgroups of the scan's two, or in chunks of the first and the last of its four.  37 tokens of the 0.5B shape through 36 layers: 2,314 us in four launches, 1,954 in two; 128 tokens of
// twelve layers of the 7B shape 3,100 and 2,872.
struct PromptBeside {
  void* qkv;                       // rows [q | k | v] of T tokens, bfloat16
  long ld;
  int T, Hq, Hkv, dh;
  const int* positions;
  const float* inv_freq;
  int rotary_dim;
  const int* slot_mapping;
  void* k_base;
  void* v_base;
  long page_stride;
  int page_size;
  const int* block_tables;
  int max_pages;
  const int* tiles;
  int n_tiles;
  const int* cu_seqlens;
  const int* start_pos;
  float scale;
  int window, max_seq_len;
  void* out;
  long out_ld;
  AheadWeight ahead[AHEAD_MOST];   // weights that the launches behind read, brought into the caches by the second launch
  int ahead_count;
};
#define BESIDE_AHEAD_BLOCKS 128    // by so many workgroups, a multiple of 8

// workgroup `index` of the attention's
template <int DH, int NSET>
__device__ __forceinline__ void prompt_attention_beside(unsigned char* __restrict__ smem, const int index, const PromptBeside& beside) {
  const int places = 4 * beside.n_tiles;
  prefill_attention_block<DH, NSET>(smem, index % places, places, index / places % beside.Hkv, index / places / beside.Hkv,
                                    (const bf16_t*)beside.qkv, beside.ld, beside.Hq, beside.Hkv, (const bf16_t*)beside.k_base,
                                    (const bf16_t*)beside.v_base, beside.page_stride, beside.page_size, beside.block_tables,
                                    beside.max_pages, beside.tiles, beside.cu_seqlens, beside.start_pos, beside.scale,
                                    beside.window, (bf16_t*)beside.out, beside.out_ld, nullptr, nullptr, DH, nullptr, nullptr, 0,
                                    nullptr, nullptr, 0, DH);
}

// prepare (rows 0 .. H-1 of the grid) and the conv with the transpose (the rows after) in one launch (their code inlined in
// both instances: as a function called from two kernels the conv took 30 us where it takes 16); with BESIDE the rows
// from `first_beside` on rotate and store a token each
template <int K, bool BESIDE>
__global__ void __launch_bounds__(256)
ssd_prepare_conv_kernel(const bf16_t* __restrict__ dt, long dt_ld, const float* __restrict__ dt_bias,
                        const float* __restrict__ A, const int* __restrict__ chunks, int H, float* __restrict__ delta,
                        float* __restrict__ cum, const bf16_t* __restrict__ u, long u_ld, int C,
                        const float* __restrict__ conv_w, const float* __restrict__ conv_b,
                        const bf16_t* __restrict__ conv_state, const int* __restrict__ slot_ids, int Q,
                        bf16_t* __restrict__ xbc, long xbc_ld, int tt_channels, bf16_t* __restrict__ TT, int first_beside,
                        PromptBeside beside) {
  __shared__ __align__(4) bf16_t tile[64 * (SSD_MAX_Q + 2)];
  __shared__ float wave_total[SSD_MAX_Q / WAVE];
  if ((int)blockIdx.y < H)
    ssd_prepare_block(dt, dt_ld, dt_bias, A, chunks, H, delta, cum, blockIdx.x, blockIdx.y, wave_total);
  else if (!BESIDE || (int)blockIdx.y < first_beside)
    ssd_conv_block<K>(u, u_ld, C, conv_w, conv_b, conv_state, chunks, slot_ids, Q, xbc, xbc_ld, tt_channels, TT,
                      blockIdx.x, ((int)blockIdx.y - H) * 64, tile);
  else {
    const long token = (long)((int)blockIdx.y - first_beside) * gridDim.x + blockIdx.x;
    if (token < beside.T)
      rope_kv_store_row<bf16_t>(token, (bf16_t*)beside.qkv, beside.ld, beside.Hq, beside.Hkv, beside.dh, beside.dh, beside.positions,
                                beside.inv_freq, beside.rotary_dim, beside.slot_mapping, (bf16_t*)beside.k_base,
                                (bf16_t*)beside.v_base, beside.page_stride, beside.page_size);
  }
}

// The conv tail of a lane after its tokens: the last K-1 rows of [old tail ; the lane's raw rows]
// (conv_state_update of mamba2.hip), one thread per channel; every old value is read before the first is written.
__device__ __forceinline__ void ssd_tail_block(const bf16_t* __restrict__ u, long u_ld, int C, int K, bf16_t* __restrict__ conv_state,
                               const int* __restrict__ chunks, const int* __restrict__ lane_chunks,
                               const int* __restrict__ slot_ids, int Q, int lane, int channel) {
  if (channel >= C) return;
  const int first = lane_chunks[2 * lane];
  const int count = lane_chunks[2 * lane + 1];
  const long start = chunks[4 * first + 1];
  const long total = (long)(count - 1) * Q + chunks[4 * (first + count - 1) + 2];
  bf16_t* tail = conv_state + (long)slot_ids[lane] * (K - 1) * C + channel;
  bf16_t kept[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (j < K - 1) {
      const long source = total + j;                 // row of the (K-1 + total)-row window
      kept[j] = source < K - 1 ? tail[source * C] : u[(start + source - (K - 1)) * u_ld + channel];
    }
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (j < K - 1) tail[(long)j * C] = kept[j];
}

// ---------------------------------------------------------------- chunk state
// chunk_state[chunk, h, p, n] = sum_s xT[h*P + p, s] * (BT[g*N + n, s] * exp(L_end - L_s) * delta_s)
// computed as its transpose on the matrix cores: A = weighted BT rows (n), B = xT rows (p),
// contraction over the Q tokens; a lane ends up with 4 consecutive n of one p.
// chunk_decay[chunk, h] = exp(L_end).  TT is the transposed copy [chunk, E + G*N, Q]: x rows
// first, B rows after.  QK = Q / 32 is a template parameter and a tile of rows that does not
// exist is clamped, so that all fragments of a tile are asked for at once.
template <int QK>
__global__ void __launch_bounds__(512)
ssd_chunk_state_kernel(const bf16_t* __restrict__ TT, int E, int GN, const float* __restrict__ delta,
                       const float* __restrict__ cum, const int* __restrict__ chunks, int H, int P, int N, int G,
                       float* __restrict__ chunk_state, float* __restrict__ chunk_decay) {
  constexpr int Q = 32 * QK;
  __shared__ float weight[Q];
  const int chunk = blockIdx.x;
  const int head = blockIdx.y;
  const int group = head / (H / G);
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int r = lane % 16;
  const float total = cum[(long)(t0 + length - 1) * H + head];
  for (int s = tid; s < Q; s += 512) {
    const long at = (long)(t0 + min(s, length - 1)) * H + head;
    const float value = __expf(total - cum[at]) * delta[at];
    weight[s] = s < length ? value : 0.f;
  }
  if (tid == 0) chunk_decay[(long)chunk * H + head] = __expf(total);
  __syncthreads();
  const bf16_t* x_rows = TT + ((long)chunk * (E + GN) + (long)head * P) * Q;
  const bf16_t* b_rows = TT + ((long)chunk * (E + GN) + E + (long)group * N) * Q;
  float* out = chunk_state + ((long)chunk * H + head) * P * N;
  const int p_tiles = P / 16;
  for (int nt = wave; nt < N / 16; nt += 8) {
    for (int pt0 = 0; pt0 < p_tiles; pt0 += 4) {            // four p-tiles share the weighted B fragments
      s_bf16x8 b_raw[QK], x[4][QK];
#pragma unroll
      for (int ks = 0; ks < QK; ++ks)
        b_raw[ks] = *reinterpret_cast<const s_bf16x8*>(b_rows + (long)(nt * 16 + r) * Q + 32 * ks + 8 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pt = min(pt0 + i, p_tiles - 1);
#pragma unroll
        for (int ks = 0; ks < QK; ++ks)
          x[i][ks] = *reinterpret_cast<const s_bf16x8*>(x_rows + (long)(pt * 16 + r) * Q + 32 * ks + 8 * q);
      }
      s_floatx4 acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = s_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < QK; ++ks) {
        s_bf16x8 a;
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = (bf16_t)((float)b_raw[ks][j] * weight[32 * ks + 8 * q + j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, x[i][ks], acc[i], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (pt0 + i < p_tiles)
          *reinterpret_cast<s_floatx4*>(out + (long)((pt0 + i) * 16 + r) * N + nt * 16 + 4 * q) = acc[i];
    }
  }
}

// ---------------------------------------------------------------- state pass
// Per lane, serially over its chunks: state_in[chunk] = running (rounded to bfloat16: it is a
// matrix-core operand); running = decay[chunk] * running + chunk_state[chunk].  The running state
// starts from the request's slot and goes back to it, in float32.
// V neighbouring elements a thread.  An element of a chunk's state is 6 bytes, float32 in and bfloat16 out; four elements a
// thread ask for 16 bytes a load and write 8 (one element a thread: 4 and 2), in workgroups of one wave so that small
// states still reach every compute unit.  A lane's chunks come in rounds of AT_ONCE whose loads are all asked for
// before the recurrence; lanes of up to four chunks take the short round, which asks for nothing twice over.  Few chunks
// are bound by the launch and the round trips, many by their bytes, which come from the caches that the launch before
// filled.  Alone, 24 heads, in us: 64 x 128, 1 chunk 3.0, 4 3.8, 16 7.6 (2.5 TB/s), 32 12.4, so 0.29 for each chunk more
// (4.1 TB/s); 128 x 256, 1 chunk 5.2, 16 14.3 (5.3 TB/s), 32 26.1.  Beside the prompt attention (one element a thread ->
// now): 16 chunks of 64 x 128 12.4 -> 8.4, of 128 x 256 55 -> 25; 25 lanes of one to five chunks of 64 x 128 67 -> 25.
template <int V, int AT_ONCE>
__device__ __forceinline__ void ssd_pass_rounds(const float* __restrict__ chunk_state, const float* __restrict__ chunk_decay,
                                                bf16_t* __restrict__ state_in, int first, int count, int H, int head,
                                                long per_head, long element, float (&running)[V]) {
  typedef float floats __attribute__((ext_vector_type(V)));
  typedef __bf16 halves __attribute__((ext_vector_type(V)));
  for (int c0 = first; c0 < first + count; c0 += AT_ONCE) {
    floats added[AT_ONCE];
    float decay[AT_ONCE];
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      const int c = min(c0 + j, first + count - 1);
      added[j] = *reinterpret_cast<const floats*>(chunk_state + ((long)c * H + head) * per_head + element);
      decay[j] = chunk_decay[(long)c * H + head];
    }
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      if (c0 + j < first + count) {
        halves entering;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          entering[i] = (bf16_t)running[i];
          running[i] = decay[j] * running[i] + added[j][i];
        }
        *reinterpret_cast<halves*>(state_in + ((long)(c0 + j) * H + head) * per_head + element) = entering;
      }
    }
  }
}

template <int V>
__global__ void ssd_state_pass_kernel(const float* __restrict__ chunk_state, const float* __restrict__ chunk_decay,
                                      const int* __restrict__ lane_chunks, const int* __restrict__ slot_ids, int H,
                                      long per_head, float* __restrict__ ssm_state, bf16_t* __restrict__ state_in,
                                      const bf16_t* __restrict__ u, long u_ld, int C, int K,
                                      bf16_t* __restrict__ conv_state, const int* __restrict__ chunks, int Q) {
  typedef float floats __attribute__((ext_vector_type(V)));
  const int lane = blockIdx.z;
  if ((int)blockIdx.y >= H) {                // rows past the heads (when the conv ran here): the lane's conv tail
    if (blockIdx.x == 0)
      ssd_tail_block(u, u_ld, C, K, conv_state, chunks, lane_chunks, slot_ids, Q, lane,
                     ((int)blockIdx.y - H) * blockDim.x + threadIdx.x);
    return;
  }
  const int head = blockIdx.y;
  const long element = V * ((long)blockIdx.x * blockDim.x + threadIdx.x);
  if (element >= per_head) return;
  const int first = lane_chunks[2 * lane];
  const int count = lane_chunks[2 * lane + 1];
  float* slot = ssm_state + ((long)slot_ids[lane] * H + head) * per_head + element;
  floats state = *reinterpret_cast<const floats*>(slot);
  float running[V];
#pragma unroll
  for (int i = 0; i < V; ++i) running[i] = state[i];
  if (count <= 4)
    ssd_pass_rounds<V, 4>(chunk_state, chunk_decay, state_in, first, count, H, head, per_head, element, running);
  else
    ssd_pass_rounds<V, 16>(chunk_state, chunk_decay, state_in, first, count, H, head, per_head, element, running);
#pragma unroll
  for (int i = 0; i < V; ++i) state[i] = running[i];
  *reinterpret_cast<floats*>(slot) = state;
}

// ---------------------------------------------------------------- chunk scan
// One workgroup per (chunk, group, up to HB heads of the group, 64 tokens); each of its waves
// takes a tile of 16 tokens t.  For a tile, with lane (q, n) holding column t = tile*16 + n:
//   inter:  O^T[p, t] = S_in[p, :] . C[t, :]         A = S_in rows (bfloat16), B = C rows; then * exp(L_t)
//   intra:  for 32 tokens s at a time, W^T[s, t] = B[s, :] . C[t, :] (shared by the heads), then per
//           head  P^T[s, t] = W^T exp(L_t - L_s) delta_s [s <= t]  and  O^T += xT[p, s] . P^T[s, t]
//   y[t, p] = O^T[p, t] + D x[t, p];  with z given, gated[t, p] = y * SiLU(z[t, p]) is written instead.
// 64 state rows p (4 tiles of 16) are held at a time; a larger head repeats the pass.  NK = N / 32
// is a template parameter and no load stands under a condition (a head or a tile of rows that
// does not exist is clamped to the last that does, computed and not stored): loads come back in
// order and a condition between them would make each wait for the one before.
template <int HB, int NK>
__global__ void __launch_bounds__(256)
ssd_chunk_scan_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                      const bf16_t* __restrict__ state_in, const float* __restrict__ delta,
                      const float* __restrict__ cum, const float* __restrict__ D, const int* __restrict__ chunks,
                      int Q, int H, int P, int G, float* __restrict__ y, long y_ld,
                      const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated, long gated_ld) {
  constexpr int PT = 4;
  constexpr int N = 32 * NK;
  __shared__ float L[HB][SSD_MAX_Q];
  __shared__ float step[HB][SSD_MAX_Q];
  const int chunk = blockIdx.x;
  const int heads_per_group = H / G;
  const int subsets = (heads_per_group + HB - 1) / HB;
  const int group = blockIdx.y / subsets;
  const int head0 = group * heads_per_group + (blockIdx.y % subsets) * HB;
  const int heads = min(HB, group * heads_per_group + heads_per_group - head0);
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int tile = (gridDim.z - 1 - blockIdx.z) * 4 + wave;    // the tiles with the most tokens before them first
  if ((tile - wave) * 16 >= length) return;                      // the whole workgroup
  const int q = lane / 16;
  const int n = lane % 16;
  const int end_s = min(length, (tile - wave) * 16 + 64);        // tokens any wave of the workgroup looks at
  for (int index = tid; index < HB * end_s; index += 256) {
    const int hb = index / end_s;
    const int s = index % end_s;
    const int head = head0 + min(hb, heads - 1);
    L[hb][s] = cum[(long)(t0 + s) * H + head];
    step[hb][s] = delta[(long)(t0 + s) * H + head];
  }
  __syncthreads();
  if (tile * 16 >= length) return;
  const int b_col = E + group * N;                 // columns of B and C in a row of xbc
  const int c_col = E + G * N + group * N;
  const int last_row = t0 + length - 1;
  const int t = tile * 16 + n;                     // this lane's column
  const bool has_t = t < length;
  const int t_safe = min(t, length - 1);
  const long t_row = t0 + t_safe;
  const int p_tiles = P / 16;
  // C of the column, all of N: the B operand of both score products
  s_bf16x8 c_frag[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    c_frag[kk] = *reinterpret_cast<const s_bf16x8*>(xbc + t_row * xbc_ld + c_col + 32 * kk + 8 * q);
  if (!has_t) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
#pragma unroll
      for (int j = 0; j < 8; ++j) c_frag[kk][j] = (bf16_t)0.f;
  }
  for (int pt0 = 0; pt0 < p_tiles; pt0 += PT) {
    s_floatx4 acc[HB][PT];
    // inter-chunk term
#pragma unroll
    for (int hb = 0; hb < HB; ++hb) {
      const int head = head0 + min(hb, heads - 1);
      const float carry = __expf(L[hb][t_safe]);
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        const int pt = min(pt0 + pi, p_tiles - 1);
        const bf16_t* s_rows = state_in + (((long)chunk * H + head) * P + pt * 16 + n) * N + 8 * q;
        s_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(s_rows + 32 * kk);
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], sum, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[hb][pi][i] = sum[i] * carry;
      }
    }
    // intra-chunk term
    for (int s0 = 0; s0 <= tile * 16 + 15 && s0 < length; s0 += 32) {
      s_floatx4 w[2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        w[half] = s_floatx4{0.f, 0.f, 0.f, 0.f};
        const long s_row = min((long)t0 + s0 + 16 * half + n, (long)last_row);
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(xbc + s_row * xbc_ld + b_col + 32 * kk + 8 * q);
          w[half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], w[half], 0, 0, 0);
        }
      }
      // the A operands of all heads and row tiles of this step: asked for before the exponentials
      s_bf16x4 x_lo[HB][PT], x_hi[HB][PT];
#pragma unroll
      for (int hb = 0; hb < HB; ++hb) {
        const int head = head0 + min(hb, heads - 1);
#pragma unroll
        for (int pi = 0; pi < PT; ++pi) {
          const int pt = min(pt0 + pi, p_tiles - 1);
          const bf16_t* x_row = TT + ((long)chunk * (E + G * N) + (long)head * P + pt * 16 + n) * Q + s0 + 4 * q;
          x_lo[hb][pi] = *reinterpret_cast<const s_bf16x4*>(x_row);
          x_hi[hb][pi] = *reinterpret_cast<const s_bf16x4*>(x_row + 16);
        }
      }
#pragma unroll
      for (int hb = 0; hb < HB; ++hb) {
        s_bf16x8 p_frag;
        const float l_t = L[hb][t_safe];
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int s = s0 + 16 * half + 4 * q + i;
            const int s_safe = min(s, length - 1);
            const bool visible = has_t && s <= t && s < length;
            const float value = visible ? w[half][i] * __expf(l_t - L[hb][s_safe]) * step[hb][s_safe] : 0.f;
            p_frag[4 * half + i] = (bf16_t)value;
          }
#pragma unroll
        for (int pi = 0; pi < PT; ++pi) {
          s_bf16x8 a;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            a[j] = x_lo[hb][pi][j];
            a[4 + j] = x_hi[hb][pi][j];
          }
          acc[hb][pi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p_frag, acc[hb][pi], 0, 0, 0);
        }
      }
    }
    // y[t, h*P + 16 pt + 4q + i] = acc + D x: the skip and gate operands first, then the stores
    s_bf16x4 x_skip[HB][PT], gate[HB][PT];
#pragma unroll
    for (int hb = 0; hb < HB; ++hb)
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        const long column = (long)(head0 + min(hb, heads - 1)) * P + min(pt0 + pi, p_tiles - 1) * 16 + 4 * q;
        x_skip[hb][pi] = *reinterpret_cast<const s_bf16x4*>(xbc + t_row * xbc_ld + column);
        gate[hb][pi] = *reinterpret_cast<const s_bf16x4*>((z != nullptr ? z + t_row * z_ld : xbc + t_row * xbc_ld) + column);
      }
#pragma unroll
    for (int hb = 0; hb < HB; ++hb) {
      const float skip = D[head0 + min(hb, heads - 1)];
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        if (!has_t || hb >= heads || pt0 + pi >= p_tiles) continue;
        const long column = (long)(head0 + hb) * P + (pt0 + pi) * 16 + 4 * q;
        s_floatx4 out;
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = acc[hb][pi][i] + skip * (float)x_skip[hb][pi][i];
        if (z != nullptr) {
          s_bf16x4 packed;
#pragma unroll
          for (int i = 0; i < 4; ++i) packed[i] = (bf16_t)(out[i] * silu_bf16_f((float)gate[hb][pi][i]));
          *reinterpret_cast<s_bf16x4*>(gated + t_row * gated_ld + column) = packed;
        } else {
          *reinterpret_cast<s_floatx4*>(y + t_row * y_ld + column) = out;
        }
      }
    }
  }
}

#define SSD_SCAN_WAVES 8
static_assert(SSD_SCAN_WAVES == PREFILL_WAVES, "workgroups of one launch");
// The same with the operands that the eight tiles of 128 tokens share staged in LDS: one
// workgroup of eight waves per (chunk, head, 128 tokens), a tile of 16 tokens a wave.  S_in of
// the head (64 rows at a time), then, 64 tokens s at a time, the rows of B and the columns of
// x^T go through LDS once for all tiles instead of once per tile from the caches; only C, the
// skip and the gate are read per tile.  Rows are padded by 16 bytes so that the 16 rows a
// matrix-core operand reads fall in different banks.  Head sizes up to 128.
template <int NK, int PT>
__device__ __forceinline__ void
ssd_chunk_scan_block(unsigned char* __restrict__ scan_smem, const int chunk, const int head, const int part,
                     const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                     const bf16_t* __restrict__ state_in, const float* __restrict__ delta,
                     const float* __restrict__ cum, const float* __restrict__ D,
                     const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y,
                     long y_ld, const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated,
                     long gated_ld) {
  constexpr int N = 32 * NK;
  constexpr int P = 16 * PT;
  constexpr int LD1 = N + 8;                     // row stride of the S / B buffer
  constexpr int LDX = 64 + 8;                    // row stride of the x^T buffer
  constexpr int THREADS = SSD_SCAN_WAVES * WAVE;
  bf16_t* buf1 = reinterpret_cast<bf16_t*>(scan_smem);                 // [64][LD1]: S_in rows, then B rows
  bf16_t* buf_x = buf1 + 64 * LD1;                                     // [P][LDX]
  float* L = reinterpret_cast<float*>(buf_x + (long)P * LDX);          // [Q]
  float* step = L + Q;                                                 // [Q]
  const int group = head / (H / G);
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  if (part * 128 >= length) return;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int n = lane % 16;
  const int tile = part * 8 + wave;
  const int end_s = min(length, part * 128 + 128);
  const int GN = G * N;
  const int b_col = E + group * N;
  const int c_col = E + GN + group * N;
  const int last_row = t0 + length - 1;
  const int t = tile * 16 + n;
  const bool tile_live = tile * 16 < length;
  const bool has_t = t < length;
  const int t_safe = min(t, length - 1);
  const long t_row = t0 + t_safe;

  for (int s = tid; s < end_s; s += THREADS) {
    L[s] = cum[(long)(t0 + s) * H + head];
    step[s] = delta[(long)(t0 + s) * H + head];
  }
  // per tile: C of the column, the skip and the gate operands (asked for now, used at the end)
  s_bf16x8 c_frag[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    c_frag[kk] = *reinterpret_cast<const s_bf16x8*>(xbc + t_row * xbc_ld + c_col + 32 * kk + 8 * q);
  if (!has_t) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
#pragma unroll
      for (int j = 0; j < 8; ++j) c_frag[kk][j] = (bf16_t)0.f;
  }

  s_floatx4 acc[PT];
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) acc[pi] = s_floatx4{0.f, 0.f, 0.f, 0.f};

  // ---- inter-chunk term: S_in through LDS, 64 rows at a time
  const bf16_t* s_head = state_in + ((long)chunk * H + head) * P * N;
  for (int pb = 0; pb * 64 < P; ++pb) {
    __syncthreads();
    for (int index = tid; index < 64 * (N / 8); index += THREADS) {
      const int row = index / (N / 8);
      const int v = index % (N / 8);
      const int p = min(pb * 64 + row, P - 1);
      *reinterpret_cast<s_bf16x8*>(buf1 + row * LD1 + 8 * v) =
          *reinterpret_cast<const s_bf16x8*>(s_head + (long)p * N + 8 * v);
    }
    __syncthreads();
    if (tile_live) {
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        if (pi / 4 == pb) {
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) {
            const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(buf1 + ((pi % 4) * 16 + n) * LD1 + 32 * kk + 8 * q);
            acc[pi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], acc[pi], 0, 0, 0);
          }
        }
      }
    }
  }
  {
    const float carry = __expf(L[min(t_safe, end_s - 1)]);
#pragma unroll
    for (int pi = 0; pi < PT; ++pi)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[pi][i] *= carry;
  }

  // ---- intra-chunk term: 64 tokens s at a time, B rows and x^T columns through LDS
  const bf16_t* x_head = TT + ((long)chunk * (E + GN) + (long)head * P) * Q;
  for (int sb = 0; sb * 64 < end_s; ++sb) {
    __syncthreads();
    for (int index = tid; index < 64 * (N / 8); index += THREADS) {
      const int row = index / (N / 8);
      const int v = index % (N / 8);
      const long s_row = min((long)t0 + sb * 64 + row, (long)last_row);
      *reinterpret_cast<s_bf16x8*>(buf1 + row * LD1 + 8 * v) =
          *reinterpret_cast<const s_bf16x8*>(xbc + s_row * xbc_ld + b_col + 8 * v);
    }
    for (int index = tid; index < P * 8; index += THREADS) {
      const int row = index / 8;
      const int v = index % 8;
      s_bf16x8 value;
#pragma unroll
      for (int j = 0; j < 8; ++j) value[j] = (bf16_t)0.f;
      if (sb * 64 + 8 * v < Q) value = *reinterpret_cast<const s_bf16x8*>(x_head + (long)row * Q + sb * 64 + 8 * v);
      *reinterpret_cast<s_bf16x8*>(buf_x + row * LDX + 8 * v) = value;
    }
    __syncthreads();
    if (!tile_live) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int s0 = sb * 64 + 32 * j;
      if (s0 > tile * 16 + 15 || s0 >= length) continue;
      s_floatx4 w[2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        w[half] = s_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(buf1 + (32 * j + 16 * half + n) * LD1 + 32 * kk + 8 * q);
          w[half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], w[half], 0, 0, 0);
        }
      }
      s_bf16x8 p_frag;
      const float l_t = L[min(t_safe, end_s - 1)];
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = s0 + 16 * half + 4 * q + i;
          const int s_safe = min(s, end_s - 1);
          const bool visible = has_t && s <= t && s < length;
          const float value = visible ? w[half][i] * __expf(l_t - L[s_safe]) * step[s_safe] : 0.f;
          p_frag[4 * half + i] = (bf16_t)value;
        }
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        const bf16_t* x_row = buf_x + (pi * 16 + n) * LDX + 32 * j + 4 * q;
        const s_bf16x4 lo = *reinterpret_cast<const s_bf16x4*>(x_row);
        const s_bf16x4 hi = *reinterpret_cast<const s_bf16x4*>(x_row + 16);
        s_bf16x8 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] = lo[e];
          a[4 + e] = hi[e];
        }
        acc[pi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p_frag, acc[pi], 0, 0, 0);
      }
    }
  }

  // ---- y[t, h*P + 16 pi + 4q + i] = acc + D x
  if (!has_t) return;
  const float skip = D[head];
  s_bf16x4 x_skip[PT], gate[PT];
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) {
    const long column = (long)head * P + pi * 16 + 4 * q;
    x_skip[pi] = *reinterpret_cast<const s_bf16x4*>(xbc + t_row * xbc_ld + column);
    gate[pi] = *reinterpret_cast<const s_bf16x4*>((z != nullptr ? z + t_row * z_ld : xbc + t_row * xbc_ld) + column);
  }
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) {
    const long column = (long)head * P + pi * 16 + 4 * q;
    s_floatx4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = acc[pi][i] + skip * (float)x_skip[pi][i];
    if (z != nullptr) {
      s_bf16x4 packed;
#pragma unroll
      for (int i = 0; i < 4; ++i) packed[i] = (bf16_t)(out[i] * silu_bf16_f((float)gate[pi][i]));
      *reinterpret_cast<s_bf16x4*>(gated + t_row * gated_ld + column) = packed;
    } else {
      *reinterpret_cast<s_floatx4*>(y + t_row * y_ld + column) = out;
    }
  }
}

#define SCAN_OPERANDS xbc, xbc_ld, TT, E, state_in, delta, cum, D, chunks, Q, H, G, y, y_ld, z, z_ld, gated, gated_ld
template <int NK, int PT>
__global__ void __launch_bounds__(SSD_SCAN_WAVES * WAVE)
ssd_chunk_scan_lds_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                          const bf16_t* __restrict__ state_in, const float* __restrict__ delta,
                          const float* __restrict__ cum, const float* __restrict__ D,
                          const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y,
                          long y_ld, const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated,
                          long gated_ld) {
  extern __shared__ __align__(16) unsigned char scan_smem[];
  // the later 128 tokens first: they have more before them
  ssd_chunk_scan_block<NK, PT>(scan_smem, blockIdx.x, blockIdx.y, gridDim.z - 1 - blockIdx.z, SCAN_OPERANDS);
}

// The same beside the prompt attention of the layer (see PromptBeside): workgroups 0 .. scan_groups - 1 are the scan's, those
// after them the attention's.  Heads of 64: one a workgroup of the attention, in 128 registers (two would take 191, and the
// compute unit one workgroup of either kind: 18 us for 515 tokens, where the whole prompt gained nothing, 12 for 300); of 128
// two, of which none fits beside another.  Which rows share a workgroup changes no sum.
template <int NK, int PT, int DH, int NSET>
__global__ void __launch_bounds__(SSD_SCAN_WAVES * WAVE, DH == 64 ? 4 : 2)
ssd_chunk_scan_beside_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                             const bf16_t* __restrict__ state_in, const float* __restrict__ delta,
                             const float* __restrict__ cum, const float* __restrict__ D,
                             const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y,
                             long y_ld, const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated,
                             long gated_ld, int n_chunks, int parts, int scan_groups, const PromptBeside beside) {
  extern __shared__ __align__(16) unsigned char scan_smem[];
  const int number = blockIdx.x;
  if (number < scan_groups) {
    ssd_chunk_scan_block<NK, PT>(scan_smem, number % n_chunks, number / n_chunks % H, parts - 1 - number / n_chunks / H, SCAN_OPERANDS);
    return;
  }
  prompt_attention_beside<DH, NSET>(scan_smem, number - scan_groups, beside);
}
#undef SCAN_OPERANDS

// ---------------------------------------------------------------- lanes of one chunk
// Every lane of the step is one chunk of at most SSD_SINGLE_TOKENS tokens, so that a chunk starts from its request's state
// and leaves it: the chunk's state, the pass and the scan in one launch, with their products and sums in their order (the
// state read in float32, rounded to bfloat16 where it is an operand of the outputs, as the pass rounds it).  One workgroup
// of eight waves a (lane, head), a tile of 16 tokens a wave; rows of the grid past the heads update the lanes' conv tails,
// as in the pass.  A short prompt waits for round trips, not for bytes: everything that the first 64 tokens need, the old
// state and the operands of the new one are asked for at the top and laid in LDS behind one barrier.  37 tokens, 24 heads
// of 64 x 128: 8.0 + 7.0 + 7.8 us in three launches, 13.5 in this one (14.7 with every stage asking for its own); with the
// conv's launch before, replayed alone, 23.6 -> 19.2 (100 tokens 27.5 -> 23.1, 128 27.9 -> 24.0; 37 of 128 x 256 44.7 -> 40.2).
#define SSD_SINGLE_TOKENS (SSD_SCAN_WAVES * 16)
struct SsdSingle {
  float* state;                    // [slots, H, P, N]
  const int* slot_ids;
  const bf16_t* u;                 // the conv's raw rows and tails, where the conv ran in the launch before
  long u_ld;
  int C, K;
  bf16_t* conv_state;
  const int* lane_chunks;
};
template <int NK, int PT>
__device__ __forceinline__ void ssd_single_block(
    unsigned char* __restrict__ scan_smem, const int chunk, const int head, const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                  const float* __restrict__ delta, const float* __restrict__ cum, const float* __restrict__ D,
                  const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y, long y_ld,
                  const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated, long gated_ld, const SsdSingle one) {

  constexpr int N = 32 * NK;
  constexpr int P = 16 * PT;
  constexpr int LD1 = N + 8;                     // row stride of the S and B buffers
  constexpr int LDX = 64 + 8;                    // row stride of the x^T buffer
  constexpr int THREADS = SSD_SCAN_WAVES * WAVE;
  constexpr int S_PIECES = (P * (N / 8) + THREADS - 1) / THREADS;      // eight elements a piece
  constexpr int B_PIECES = (64 * (N / 8) + THREADS - 1) / THREADS;
  constexpr int X_PIECES = (P * 8 + THREADS - 1) / THREADS;
  constexpr int QK = SSD_SINGLE_TOKENS / 32;
  constexpr int PB = PT < 4 ? PT : 4;            // tiles of state rows that share the weighted B fragments
  constexpr int ITEMS = (N / 16) * (PT / PB);
  bf16_t* s_rows = reinterpret_cast<bf16_t*>(scan_smem);               // [P][LD1]
  bf16_t* b_lds = s_rows + P * LD1;                                    // [64][LD1]
  bf16_t* x_lds = b_lds + 64 * LD1;                                    // [P][LDX]
  float* L = reinterpret_cast<float*>(x_lds + P * LDX);                // [SSD_SINGLE_TOKENS] each
  float* step = L + SSD_SINGLE_TOKENS;
  float* weight = step + SSD_SINGLE_TOKENS;
  const int step_lane = chunks[4 * chunk];
  const int t0 = chunks[4 * chunk + 1];
  const int length = chunks[4 * chunk + 2];
  if (length <= 0) return;                    // a row of the table past the step's own chunks: the whole workgroup leaves
  const int tid = threadIdx.x;
  if (head >= H) {
    ssd_tail_block(one.u, one.u_ld, one.C, one.K, one.conv_state, chunks, one.lane_chunks, one.slot_ids, Q, step_lane,
                   (head - H) * THREADS + tid);
    return;
  }
  const int group = head / (H / G);
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int q = lane / 16;
  const int n = lane % 16;
  const int GN = G * N;
  const int b_col = E + group * N;
  const int c_col = E + GN + group * N;
  const int t = wave * 16 + n;
  const bool tile_live = wave * 16 < length;
  const bool has_t = t < length;
  const long t_row = t0 + min(t, length - 1);
  float* const slot = one.state + ((long)one.slot_ids[step_lane] * H + head) * P * N;
  const bf16_t* x_rows = TT + ((long)chunk * (E + GN) + (long)head * P) * Q;
  const bf16_t* b_rows = TT + ((long)chunk * (E + GN) + E + (long)group * N) * Q;

  // ---- everything is asked for
  const int token = min(tid, length - 1);
  const float own_cum = cum[(long)(t0 + token) * H + head];            // (the first 128 threads' count)
  const float own_delta = delta[(long)(t0 + token) * H + head];
  s_bf16x8 c_frag[NK], b_piece[B_PIECES], x_piece[X_PIECES];
  s_floatx4 s_piece[S_PIECES][2];
#pragma unroll
  for (int i = 0; i < S_PIECES; ++i) {
    const int at = min(tid + i * THREADS, P * (N / 8) - 1) * 8;        // (the state of a head is one run)
    s_piece[i][0] = *reinterpret_cast<const s_floatx4*>(slot + at);
    s_piece[i][1] = *reinterpret_cast<const s_floatx4*>(slot + at + 4);
  }
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    c_frag[kk] = *reinterpret_cast<const s_bf16x8*>(xbc + t_row * xbc_ld + c_col + 32 * kk + 8 * q);
  auto ask_block = [&](int sb) {                                       // 64 tokens s: B's rows and x^T's columns
#pragma unroll
    for (int i = 0; i < B_PIECES; ++i) {
      const int index = min(tid + i * THREADS, 64 * (N / 8) - 1);
      const long row = t0 + min(64 * sb + index / (N / 8), length - 1);
      b_piece[i] = *reinterpret_cast<const s_bf16x8*>(xbc + row * xbc_ld + b_col + 8 * (index % (N / 8)));
    }
#pragma unroll
    for (int i = 0; i < X_PIECES; ++i) {
      const int index = min(tid + i * THREADS, P * 8 - 1);
      const int at = 64 * sb + 8 * (index % 8);                        // (past Q: the last there are, whose weights are zero)
      x_piece[i] = *reinterpret_cast<const s_bf16x8*>(x_rows + (long)(index / 8) * Q + min(at, Q - 8));
    }
  };
  auto lay_block = [&]() {
#pragma unroll
    for (int i = 0; i < B_PIECES; ++i) {
      const int index = tid + i * THREADS;
      if (index < 64 * (N / 8)) *reinterpret_cast<s_bf16x8*>(b_lds + (index / (N / 8)) * LD1 + 8 * (index % (N / 8))) = b_piece[i];
    }
#pragma unroll
    for (int i = 0; i < X_PIECES; ++i) {
      const int index = tid + i * THREADS;
      if (index < P * 8) *reinterpret_cast<s_bf16x8*>(x_lds + (index / 8) * LDX + 8 * (index % 8)) = x_piece[i];
    }
  };
  ask_block(0);
  s_bf16x8 b_raw[QK], x[PB][QK];
  s_floatx4 before[PB];
  auto ask_state = [&](int item) {
    const int nt = item % (N / 16), pt0 = item / (N / 16) * PB;
#pragma unroll
    for (int ks = 0; ks < QK; ++ks)
      b_raw[ks] = *reinterpret_cast<const s_bf16x8*>(b_rows + (long)(nt * 16 + n) * Q + min(32 * ks, Q - 32) + 8 * q);
#pragma unroll
    for (int i = 0; i < PB; ++i) {
#pragma unroll
      for (int ks = 0; ks < QK; ++ks)
        x[i][ks] = *reinterpret_cast<const s_bf16x8*>(x_rows + (long)((pt0 + i) * 16 + n) * Q + min(32 * ks, Q - 32) + 8 * q);
      before[i] = *reinterpret_cast<const s_floatx4*>(slot + (long)((pt0 + i) * 16 + n) * N + nt * 16 + 4 * q);
    }
  };
  constexpr bool EARLY = NK <= 4;                // (256 state columns and the operands of the new state do not fit the registers)
  if (EARLY) ask_state(min(wave, ITEMS - 1));
  s_bf16x4 x_skip[PT], gate[PT];
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) {
    const long column = (long)head * P + pi * 16 + 4 * q;
    x_skip[pi] = *reinterpret_cast<const s_bf16x4*>(xbc + t_row * xbc_ld + column);
    gate[pi] = *reinterpret_cast<const s_bf16x4*>((z != nullptr ? z + t_row * z_ld : xbc + t_row * xbc_ld) + column);
  }

  // ---- and laid down
  if (tid < SSD_SINGLE_TOKENS) {
    L[tid] = own_cum;
    step[tid] = own_delta;
  }
#pragma unroll
  for (int i = 0; i < S_PIECES; ++i) {
    const int index = tid + i * THREADS;
    s_bf16x8 value;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      value[e] = (bf16_t)s_piece[i][0][e];
      value[4 + e] = (bf16_t)s_piece[i][1][e];
    }
    if (index < P * (N / 8)) *reinterpret_cast<s_bf16x8*>(s_rows + (index / (N / 8)) * LD1 + 8 * (index % (N / 8))) = value;
  }
  lay_block();
  if (!has_t) {
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
#pragma unroll
      for (int j = 0; j < 8; ++j) c_frag[kk][j] = (bf16_t)0.f;
  }
  __syncthreads();
  const float total = L[length - 1];
  if (tid < SSD_SINGLE_TOKENS) weight[tid] = tid < length ? __expf(total - own_cum) * own_delta : 0.f;

  // ---- the state's part of the outputs, then the chunk's own tokens, 64 at a time
  s_floatx4 acc[PT];
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) acc[pi] = s_floatx4{0.f, 0.f, 0.f, 0.f};
  const float l_t = L[min(t, length - 1)];
  if (tile_live) {
    const float carry = __expf(l_t);
#pragma unroll
    for (int pi = 0; pi < PT; ++pi) {
#pragma unroll
      for (int kk = 0; kk < NK; ++kk) {
        const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(s_rows + (pi * 16 + n) * LD1 + 32 * kk + 8 * q);
        acc[pi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], acc[pi], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[pi][i] *= carry;
    }
  }
  for (int sb = 0; sb * 64 < length; ++sb) {
    if (sb > 0) {
      ask_block(sb);
      __syncthreads();                                                 // the block before is read
      lay_block();
      __syncthreads();
    }
    if (!tile_live) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int s0 = sb * 64 + 32 * j;
      if (s0 > wave * 16 + 15 || s0 >= length) continue;
      s_floatx4 w[2];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        w[half] = s_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) {
          const s_bf16x8 a = *reinterpret_cast<const s_bf16x8*>(b_lds + (32 * j + 16 * half + n) * LD1 + 32 * kk + 8 * q);
          w[half] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, c_frag[kk], w[half], 0, 0, 0);
        }
      }
      s_bf16x8 p_frag;
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = s0 + 16 * half + 4 * q + i;
          const int s_safe = min(s, length - 1);
          const bool visible = has_t && s <= t && s < length;
          const float value = visible ? w[half][i] * __expf(l_t - L[s_safe]) * step[s_safe] : 0.f;
          p_frag[4 * half + i] = (bf16_t)value;
        }
#pragma unroll
      for (int pi = 0; pi < PT; ++pi) {
        const bf16_t* x_row = x_lds + (pi * 16 + n) * LDX + 32 * j + 4 * q;
        const s_bf16x4 lo = *reinterpret_cast<const s_bf16x4*>(x_row);
        const s_bf16x4 hi = *reinterpret_cast<const s_bf16x4*>(x_row + 16);
        s_bf16x8 a;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[e] = lo[e];
          a[4 + e] = hi[e];
        }
        acc[pi] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p_frag, acc[pi], 0, 0, 0);
      }
    }
  }
  __syncthreads();                                                     // the weights are there

  // ---- the state the chunk leaves: sum_s weight_s x_s (outer) B_s beside what is left of the old one
  const float decay = __expf(total);
  for (int item = wave; item < ITEMS; item += SSD_SCAN_WAVES) {
    const int nt = item % (N / 16), pt0 = item / (N / 16) * PB;
    if (!EARLY || item != wave) ask_state(item);
    s_floatx4 sum[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) sum[i] = s_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < QK; ++ks) {
      if (32 * ks >= Q) continue;              // (a chunk's own columns once more, whose infinities a weight of zero would not stop)
      s_bf16x8 a;
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = (bf16_t)((float)b_raw[ks][j] * weight[32 * ks + 8 * q + j]);
#pragma unroll
      for (int i = 0; i < PB; ++i) sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, x[i][ks], sum[i], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) before[i][j] = decay * before[i][j] + sum[i][j];
      *reinterpret_cast<s_floatx4*>(slot + (long)((pt0 + i) * 16 + n) * N + nt * 16 + 4 * q) = before[i];
    }
  }

  // ---- y[t, h*P + 16 pi + 4q + i] = acc + D x
  if (!has_t) return;
  const float skip = D[head];
#pragma unroll
  for (int pi = 0; pi < PT; ++pi) {
    const long column = (long)head * P + pi * 16 + 4 * q;
    s_floatx4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = acc[pi][i] + skip * (float)x_skip[pi][i];
    if (z != nullptr) {
      s_bf16x4 packed;
#pragma unroll
      for (int i = 0; i < 4; ++i) packed[i] = (bf16_t)(out[i] * silu_bf16_f((float)gate[pi][i]));
      *reinterpret_cast<s_bf16x4*>(gated + t_row * gated_ld + column) = packed;
    } else {
      *reinterpret_cast<s_floatx4*>(y + t_row * y_ld + column) = out;
    }
  }
}

template <int NK, int PT>
__global__ void __launch_bounds__(SSD_SCAN_WAVES * WAVE)
ssd_single_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                  const float* __restrict__ delta, const float* __restrict__ cum, const float* __restrict__ D,
                  const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y, long y_ld,
                  const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated, long gated_ld, const SsdSingle one) {
  extern __shared__ __align__(16) unsigned char scan_smem[];
  ssd_single_block<NK, PT>(scan_smem, blockIdx.x, blockIdx.y, xbc, xbc_ld, TT, E, delta, cum, D, chunks, Q, H, G, y, y_ld, z, z_ld, gated, gated_ld, one);
}

// The same beside the prompt attention of the layer (see PromptBeside): workgroups 0 .. scan_groups - 1 are the scan's, the
// longer ones, and those after them the attention's, of as many threads; either uses the workgroup's LDS.
// Heads that share their keys and states of 64 x 128 and more: two launches are the faster way at every such size, by what the
// launches and the attention behind the scan cost.  37 tokens | 128 | five lanes of 16 behind 700 keys, four launches and two in us, 24 heads
// of the scan: states of 64 x 128 beside 8 / 2 heads of 64 28.5, 19.2 | 33.8, 24.2 | 33.5, 19.0; 64 x 256 beside 6 / 2 of
// 64 31.2, 22.5 | 37.5, 28.5 | 36.8, 22.7; 128 x 128 beside 12 / 2 of 128 41.5, 26.6 | 49.8, 33.6 | 53.4, 29.9; 128 x 256
// beside 8 / 2 of 64 50.6, 41.4 | 58.7, 48.9 | 59.7, 43.9.  (Smaller states, and a key for every query head, are in no shape of this
// framework and would be six times the instances: 100 s to compile and 5.3 MB, 31 and 1.7 with these.)
#define BESIDE_LEAST_P 64
#define BESIDE_LEAST_N 128
template <int NK, int PT, int DH, int NSET>
__global__ void __launch_bounds__(SSD_SCAN_WAVES * WAVE)
ssd_single_beside_kernel(const bf16_t* __restrict__ xbc, long xbc_ld, const bf16_t* __restrict__ TT, int E,
                  const float* __restrict__ delta, const float* __restrict__ cum, const float* __restrict__ D,
                  const int* __restrict__ chunks, int Q, int H, int G, float* __restrict__ y, long y_ld,
                  const bf16_t* __restrict__ z, long z_ld, bf16_t* __restrict__ gated, long gated_ld, const SsdSingle one,
                         int n_chunks, int scan_groups, int passes, int ahead_from, const PromptBeside beside, const AheadList ahead) {
  extern __shared__ __align__(16) unsigned char scan_smem[];
  if ((int)blockIdx.x < scan_groups) {
    ssd_single_block<NK, PT>(scan_smem, blockIdx.x % n_chunks, blockIdx.x / n_chunks, xbc, xbc_ld, TT, E, delta, cum, D, chunks, Q, H, G, y, y_ld, z, z_ld, gated, gated_ld, one);
    return;
  }
  if ((int)blockIdx.x >= ahead_from) {
    read_ahead_block<SSD_SCAN_WAVES * WAVE>(ahead, blockIdx.x - ahead_from);
    return;
  }
  prompt_attention_beside<DH, NSET>(scan_smem, blockIdx.x - scan_groups, beside);
}

static size_t ssd_single_lds_bytes(int P, int N) {
  return (size_t)(P + 64) * (N + 8) * 2 + (size_t)P * (64 + 8) * 2 + (size_t)3 * SSD_SINGLE_TOKENS * 4;
}

static bool ssd_staged_sizes(int P, int N) {
  return (P == 16 || P == 32 || P == 64 || P == 128) && (N == 32 || N == 64 || N == 128 || N == 256);
}

// Whether a step whose longest lane holds `longest` tokens (0: not known) is worked on in one launch behind the conv: with
// states that begin at whole 16-byte pieces, as that launch moves them.
extern "C" int mi_ssd_single(int Q, int P, int N, int longest, const float* ssm_state) {
  return (uintptr_t)ssm_state % 16 == 0 && longest > 0 && longest <= Q && longest <= SSD_SINGLE_TOKENS && ssd_staged_sizes(P, N) ? 1 : 0;
}

// beyond 64 KiB a kernel has to be told once per device that it may have that much (gfx950 has 160 KiB)
template <typename Kernel>
static int allow_lds(Kernel kernel, size_t lds, bool (&told)[64]) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return ERR_BAD_ARGUMENT;
  if (lds <= 64 * 1024 || told[device]) return 0;
  if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
    (void)hipGetLastError();
    return ERR_UNSUPPORTED_SIZE;
  }
  told[device] = true;
  return 0;
}

#define SINGLE_ARGUMENTS xbc, xbc_ld, TT, E, delta, cum, D, chunks, Q, H, G, y, y_ld, z, z_ld, gated, gated_ld, one
template <int NK, int PT>
static int launch_ssd_single(dim3 grid, hipStream_t stream, const bf16_t* xbc, long xbc_ld, const bf16_t* TT, int E,
                             const float* delta, const float* cum, const float* D, const int* chunks, int Q, int H, int G,
                             float* y, long y_ld, const bf16_t* z, long z_ld, bf16_t* gated, long gated_ld,
                             const SsdSingle& one, const PromptBeside* beside, int nset) {
  const size_t lds = ssd_single_lds_bytes(16 * PT, 32 * NK);
  if constexpr (32 * NK >= BESIDE_LEAST_N && 16 * PT >= BESIDE_LEAST_P) {
    if (beside) {
      const int passes = (beside->Hq / beside->Hkv + nset - 1) / nset;
      const long all = (long)grid.x * grid.y + 4L * beside->n_tiles * beside->Hkv * passes;
      if (all > 0x7fffffffL) return ERR_UNSUPPORTED_SIZE;
      AheadList ahead;
      if (!read_ahead_list(ahead, beside->ahead, beside->ahead_count, BESIDE_AHEAD_BLOCKS, SSD_SCAN_WAVES * WAVE)) return ERR_BAD_ARGUMENT;
      const int scan_groups = (int)(grid.x * grid.y);
      const unsigned groups = (unsigned)all + (beside->ahead_count && all < 0x7fffffffL - BESIDE_AHEAD_BLOCKS ? BESIDE_AHEAD_BLOCKS : 0);
#define BESIDE_CASE(DH_, NSET_)                                                                                             \
  if (beside->dh == DH_ && nset == NSET_) {                                                                                 \
    static bool told[64] = {};                                                                                              \
    const size_t both = lds > (size_t)prefill_lds_bytes(DH_) ? lds : (size_t)prefill_lds_bytes(DH_);                        \
    const int code = allow_lds(ssd_single_beside_kernel<NK, PT, DH_, NSET_>, both, told);                                   \
    if (code) return code;                                                                                                  \
    ssd_single_beside_kernel<NK, PT, DH_, NSET_><<<groups, SSD_SCAN_WAVES * WAVE, both, stream>>>(                          \
        SINGLE_ARGUMENTS, (int)grid.x, scan_groups, passes, (int)all, *beside, ahead);                                                       \
    return 0;                                                                                                               \
  }
      BESIDE_CASE(64, 2) BESIDE_CASE(64, 3) BESIDE_CASE(64, 4) BESIDE_CASE(128, 2)
#undef BESIDE_CASE
    }
  }
  if (beside) return ERR_UNSUPPORTED_SIZE;
  static bool told[64] = {};
  const int code = allow_lds(ssd_single_kernel<NK, PT>, lds, told);
  if (code) return code;
  ssd_single_kernel<NK, PT><<<grid, SSD_SCAN_WAVES * WAVE, lds, stream>>>(SINGLE_ARGUMENTS);
  return 0;
}
#undef SINGLE_ARGUMENTS

// Whether mi_ssd_prefill takes the attention of such heads beside its last launch (of a step that mi_ssd_single or, in chunks,
// mi_ssd_staged covers, whose H heads of the scan may have a group each): what it would refuse is refused here, before anything is launched.
extern "C" int mi_ssd_beside(int H, int P, int N, int Hq, int Hkv, int dh, int n_tiles, int max_seq_len) {
  if (H <= 0 || Hkv <= 0 || Hkv > 256 || Hq <= Hkv || Hq % Hkv != 0 || n_tiles <= 0 || n_tiles > (1 << 20) || (dh != 64 && dh != 128) ||
      !ssd_staged_sizes(P, N) || P < BESIDE_LEAST_P || N < BESIDE_LEAST_N)
    return 0;
  const int nset = prefill_head_set(dh, Hq / Hkv, n_tiles, Hkv, max_seq_len);
  // rows of the first launch, with a lane's tokens beside each chunk; workgroups of the second (a lane of one chunk has a tile)
  const long own_rows = H + ((long)H * (P + 2 * N) + 63) / 64;
  const long passes = (Hq / Hkv + nset - 1) / nset;
  return own_rows + SSD_MAX_Q <= 65535 && n_tiles * (2 * own_rows + 4 * Hkv * passes) <= 0x7fffffffL ? 1 : 0;
}

static size_t ssd_scan_lds_bytes(int Q, int P, int N) {
  return (size_t)64 * (N + 8) * 2 + (size_t)P * (64 + 8) * 2 + (size_t)2 * Q * 4;
}

// Whether the scan of chunks of Q tokens stages its operands in LDS: it then takes an attention beside it too.
extern "C" int mi_ssd_staged(int Q, int P, int N) { return ssd_staged_sizes(P, N) && ssd_scan_lds_bytes(Q, P, N) <= 64 * 1024 ? 1 : 0; }

// query heads of a workgroup of the attention beside the scan of chunks (see there)
static int scan_beside_heads(int dh) { return dh == 64 ? 1 : 2; }

// Whether the attention of `tokens` tokens beside the scan of n_chunks chunks is faster than on a stream of its own, whose fork and
// join cost about 12 us a layer: two streams | one launch in us a prompt, eight layers or more, at the workgroups of the launch in brackets.
// Heads of 64, two workgroups on a compute unit; 24 heads of the scan beside 8 / 2 of the attention (A), 48 and 96 beside 8 / 2 (B, C), 24
// beside 16 / 2 and 32 / 2 (D, E), 48 beside 16 / 4 (F), 96 beside 32 / 8 (G).
// Behind contexts of up to 2,048 the line lies by the tokens, as the longest rows of keys end the launch: to 768 the one launch is
// the faster at every number of heads (640 tokens A (496) 3,723 | 3,529, C (928) 1,727 | 1,674, E (1,552) 1,346 | 1,276; 768 A (584) 3,822 |
// 3,768, B (752) 1,358 | 1,347, C (1,088) 1,758 | 1,753, E (1,832) 1,426 | 1,361; 150 G (1,024) 1,249 | 1,187; four lanes of 200 A (1,064)
// 4,295 | 4,139, C (2,144) 2,196 | 2,148), to 896 where the scan's workgroups have a compute unit each (A (672) 3,912 | 3,896, two lanes of
// 400 4,200 | 4,038, D (1,152) 2,055 | 2,032, E (2,112) 1,518 | 1,477, but B 1,359 | 1,384, C 1,791 | 1,828; 1,024 A 4,128 | 4,199, D
// 2,125 | 2,142).  Far more
// workgroups than that gain nothing (five lanes of 150 E (2,896) 1,431 | 1,447, four of 200 beside 192 heads (3,584) 3,497 | 3,531).
// Behind longer ones a workgroup of the attention takes longer than one of the scan, and the line lies by their number: 4,096 tokens
// in portions of 256 A (232) 12,508 | 10,929, F (464) 13,711 | 12,843, G (928) 20,892 | 22,592; of 384 D (392) 19,762 | 19,185, C (608) 15,459 |
// 15,825, E (992) 14,043 | 15,073; of 512 A (408) 32,450 | 31,932, B (528) 9,909 | 9,648, D (696) 15,180 | 16,026; of 576 A (552) 32,550 |
// 32,070; of 640 A (496) 29,093 | 27,746, B (640) 9,510 | 9,767, F (992) 15,080 | 16,531.  (States of 64 x 256 and 128 x 128 have the lines of A.)
// Heads of 128, one on a compute unit (twelve layers of the 7B shape): 144 tokens 2,777 | 2,677, 256 3,190 | 3,102, 300 (216)
// 3,268 | 3,213, 400 (288) 3,702 | 3,710; 4,096 in portions of 256 51,570 | 52,090, 200 beside four tokens behind 4,000 keys (528)
// 3,750 | 3,959.
extern "C" int mi_ssd_chunks_beside(int Q, int H, int P, int N, int n_chunks, int tokens, int Hq, int Hkv, int dh, int n_tiles,
                                    int max_seq_len) {
  if (n_chunks <= 0 || !mi_ssd_staged(Q, P, N) || !mi_ssd_beside(H, P, N, Hq, Hkv, dh, n_tiles, max_seq_len)) return 0;
  const int nset = scan_beside_heads(dh);
  const long groups = (long)n_chunks * H * ((Q + 127) / 128) + 4L * n_tiles * Hkv * ((Hq / Hkv + nset - 1) / nset);
  const long scan = (long)((tokens + Q - 1) / Q) * H * ((Q + 127) / 128);      // that work: chunks past the step's own leave at once
  const bool near = max_seq_len > 0 && max_seq_len <= 2048;
  if (dh != 64) return near && groups <= 256 ? 1 : 0;
  return near ? groups <= 2304 && tokens <= (scan <= 256 ? 896 : 768) : groups <= 560;
}

template <int NK, int PT>
static int launch_ssd_scan_beside(hipStream_t stream, const bf16_t* xbc, long xbc_ld, const bf16_t* TT, int E, const bf16_t* state_in,
                                  const float* delta, const float* cum, const float* D, const int* chunks, int n_chunks, int Q,
                                  int H, int G, float* y, long y_ld, const bf16_t* z, long z_ld, bf16_t* gated, long gated_ld,
                                  const PromptBeside& beside) {
  const int nset = scan_beside_heads(beside.dh);
  if constexpr (32 * NK >= BESIDE_LEAST_N && 16 * PT >= BESIDE_LEAST_P) {
    const size_t lds = ssd_scan_lds_bytes(Q, 16 * PT, 32 * NK);
    const int parts = (Q + 127) / 128, passes = (beside.Hq / beside.Hkv + nset - 1) / nset;
    const long scan_groups = (long)n_chunks * H * parts, all = scan_groups + 4L * beside.n_tiles * beside.Hkv * passes;
    if (all > 0x7fffffffL) return ERR_UNSUPPORTED_SIZE;
#define BESIDE_CASE(DH_, NSET_)                                                                                             \
  if (beside.dh == DH_ && nset == NSET_) {                                                                                  \
    static bool told[64] = {};                                                                                              \
    const size_t most = ssd_scan_lds_bytes(SSD_MAX_Q, 16 * PT, 32 * NK);                                                    \
    const size_t both = most > (size_t)prefill_lds_bytes(DH_) ? most : (size_t)prefill_lds_bytes(DH_);                      \
    const int code = allow_lds(ssd_chunk_scan_beside_kernel<NK, PT, DH_, NSET_>, both, told);                               \
    if (code) return code;                                                                                                  \
    ssd_chunk_scan_beside_kernel<NK, PT, DH_, NSET_>                                                                        \
        <<<(unsigned)all, SSD_SCAN_WAVES * WAVE, lds > (size_t)prefill_lds_bytes(DH_) ? lds : (size_t)prefill_lds_bytes(DH_), stream>>>( \
            xbc, xbc_ld, TT, E, state_in, delta, cum, D, chunks, Q, H, G, y, y_ld, z, z_ld, gated, gated_ld, n_chunks, parts, \
            (int)scan_groups, beside);                                                                                      \
    return 0;                                                                                                               \
  }
    BESIDE_CASE(64, 1) BESIDE_CASE(128, 2)
#undef BESIDE_CASE
  }
  return ERR_UNSUPPORTED_SIZE;
}

// Sizes: bfloat16; Q a multiple of 32 and at most 256; head_dim P a multiple of 16; state size N a
// multiple of 32 and at most 256; row strides multiples of 8 elements.  Otherwise
// ERR_UNSUPPORTED_SIZE (the caller uses mi_ssm_scan).
extern "C" int mi_ssd_supported(int Q, int P, int N, int G, int E) {
  return (Q % 32 == 0 && Q > 0 && Q <= SSD_MAX_Q && P % 16 == 0 && N % 32 == 0 && N <= 256 &&
          (E % 8) == 0 && ((long)G * N) % 8 == 0) ? 1 : 0;
}

// beside: null, or the attention that reads the same step's rows (bfloat16, values as wide as the keys, a cache to write to
// or none): needs the conv here and a step that mi_ssd_single or mi_ssd_staged, and mi_ssd_beside, cover.
extern "C" int mi_ssd_prefill(const void* xbc, long xbc_ld, const void* dt, long dt_ld, const float* dt_bias,
                              const float* A, const float* D, float* ssm_state, const int* chunks, int n_chunks,
                              const int* lane_chunks, const int* slot_ids, int n_lanes, int Q, int H, int P, int N,
                              int G, float* delta, float* cum, void* TT, float* chunk_state,
                              float* chunk_decay, void* state_in, float* y, long y_ld, const void* z, long z_ld,
                              void* gated, long gated_ld, const void* u, long u_ld, const float* conv_w,
                              const float* conv_b, void* conv_state, int conv_k, int longest, const PromptBeside* beside, hipStream_t stream) {
  if (n_chunks <= 0 || n_lanes <= 0 || H <= 0 || G <= 0 || H % G != 0) return ERR_BAD_ARGUMENT;
  const int E = H * P;
  const int GN = G * N;
  const int C = E + 2 * GN;
  const bool conv_here = u != nullptr;       // xbc is then written here, from the raw rows u [T, C] (+ u_ld)
  if (conv_here && (!conv_w || !conv_state || conv_k < 2 || conv_k > 4 || u_ld % 8 != 0 || C % 8 != 0 ||
                    ((uintptr_t)u % 16) != 0 || ((uintptr_t)conv_state % 16) != 0 || ((uintptr_t)conv_w % 16) != 0 ||
                    ((uintptr_t)conv_b % 16) != 0 || H + (C + 63) / 64 > 65535 || H + (C + 255) / 256 > 65535))
    return ERR_UNSUPPORTED_SIZE;
  if ((z == nullptr) != (gated == nullptr) || (z == nullptr && y == nullptr)) return ERR_BAD_ARGUMENT;
  if (!mi_ssd_supported(Q, P, N, G, E) || xbc_ld % 8 != 0 || y_ld % 4 != 0 || z_ld % 4 != 0 || gated_ld % 4 != 0 ||
      n_chunks > 65535 * 32 ||
      H + (E + GN + 63) / 64 > 65535 || n_lanes > 65535)
    return ERR_UNSUPPORTED_SIZE;
  int nset = 0;
  if (beside) {
    const PromptBeside& b = *beside;
    if (!conv_here || !b.qkv || b.T <= 0 || b.Hq <= 0 || b.Hkv <= 0 || b.Hq % b.Hkv != 0 || b.dh <= 0 || (b.dh & 1) || !b.positions ||
        b.ld < (long)(b.Hq + 2 * b.Hkv) * b.dh || b.rotary_dim < 0 || b.rotary_dim > b.dh || (b.rotary_dim & 1) ||
        (b.rotary_dim > 0 && !b.inv_freq))
      return ERR_BAD_ARGUMENT;
    if (!b.block_tables || b.max_pages <= 0 || !b.tiles || b.n_tiles <= 0 || !b.cu_seqlens || !b.start_pos || !b.out || !b.k_base ||
        !b.v_base || b.page_size <= 0)
      return ERR_BAD_ARGUMENT;
    if (!(mi_ssd_single(Q, P, N, longest, ssm_state) || mi_ssd_staged(Q, P, N)) || !mi_ssd_beside(H, P, N, b.Hq, b.Hkv, b.dh, b.n_tiles, b.max_seq_len) ||
        b.page_size % 4 != 0 || b.ld % 8 != 0 || b.out_ld % 4 != 0 || (uintptr_t)b.qkv % 16 != 0 || (uintptr_t)b.out % 8 != 0)
      return ERR_UNSUPPORTED_SIZE;
    nset = prefill_head_set(b.dh, b.Hq / b.Hkv, b.n_tiles, b.Hkv, b.max_seq_len);
  }
  if (conv_here) {
    const int own_rows = H + (C + 63) / 64;
    const int rows = own_rows + (beside ? (beside->T + n_chunks - 1) / n_chunks : 0);
    if (rows > 65535) return ERR_UNSUPPORTED_SIZE;
    const dim3 grid(n_chunks, rows);
    const PromptBeside none = {};
#define CONV_LAUNCH(K_, BESIDE_)                                                                                   \
  ssd_prepare_conv_kernel<K_, BESIDE_><<<grid, 256, 0, stream>>>(                                                  \
      (const bf16_t*)dt, dt_ld, dt_bias, A, chunks, H, delta, cum, (const bf16_t*)u, u_ld, C, conv_w, conv_b,      \
      (const bf16_t*)conv_state, slot_ids, Q, (bf16_t*)xbc, xbc_ld, E + GN, (bf16_t*)TT, own_rows, beside ? *beside : none)
#define CONV_CASE(K_)                                                                                              \
  do {                                                                                                             \
    if (beside) CONV_LAUNCH(K_, true);                                                                             \
    else CONV_LAUNCH(K_, false);                                                                                   \
  } while (0)
    if (conv_k == 2) CONV_CASE(2);
    else if (conv_k == 3) CONV_CASE(3);
    else CONV_CASE(4);
#undef CONV_CASE
#undef CONV_LAUNCH
    RETURN_IF_LAUNCH_FAILED();
  } else {
    const dim3 grid(n_chunks, H + (E + GN + 63) / 64);       // x and B are neighbours in a row of xbc
    ssd_prepare_transpose_kernel<<<grid, 256, 0, stream>>>((const bf16_t*)dt, dt_ld, dt_bias, A, chunks, H, delta, cum,
                                                           (const bf16_t*)xbc, xbc_ld, E + GN, Q, (bf16_t*)TT);
    RETURN_IF_LAUNCH_FAILED();
  }
  if (mi_ssd_single(Q, P, N, longest, ssm_state)) {
    const int tail_rows = conv_here ? (C + SSD_SCAN_WAVES * WAVE - 1) / (SSD_SCAN_WAVES * WAVE) : 0;
    const SsdSingle one = {ssm_state, slot_ids, (const bf16_t*)u, u_ld, C, conv_k, (bf16_t*)conv_state, lane_chunks};
    int status = ERR_UNSUPPORTED_SIZE;
#define SINGLE_CASE(NK_, PT_)                                                                                     \
  if (N == 32 * NK_ && P == 16 * PT_)                                                                             \
    status = launch_ssd_single<NK_, PT_>(dim3(n_chunks, H + tail_rows), stream, (const bf16_t*)xbc, xbc_ld,       \
                                         (const bf16_t*)TT, E, delta, cum, D, chunks, Q, H, G, y, y_ld,           \
                                         (const bf16_t*)z, z_ld, (bf16_t*)gated, gated_ld, one, beside, nset);
    SINGLE_CASE(1, 1) SINGLE_CASE(1, 2) SINGLE_CASE(1, 4) SINGLE_CASE(1, 8)
    SINGLE_CASE(2, 1) SINGLE_CASE(2, 2) SINGLE_CASE(2, 4) SINGLE_CASE(2, 8)
    SINGLE_CASE(4, 1) SINGLE_CASE(4, 2) SINGLE_CASE(4, 4) SINGLE_CASE(4, 8)
    SINGLE_CASE(8, 1) SINGLE_CASE(8, 2) SINGLE_CASE(8, 4) SINGLE_CASE(8, 8)
#undef SINGLE_CASE
    if (status != 0) return status;
    RETURN_IF_LAUNCH_FAILED();
    return 0;
  }
  if (!chunk_state || !chunk_decay || !state_in) return ERR_BAD_ARGUMENT;
  {
    const dim3 grid(n_chunks, H);
#define STATE_CASE(QK_)                                                                                         \
  case QK_:                                                                                                     \
    ssd_chunk_state_kernel<QK_><<<grid, 512, 0, stream>>>((const bf16_t*)TT, E, GN, delta, cum, chunks, H, P, N, G, \
                                                          chunk_state, chunk_decay);                          \
    break;
    switch (Q / 32) {
      STATE_CASE(1) STATE_CASE(2) STATE_CASE(3) STATE_CASE(4) STATE_CASE(5) STATE_CASE(6) STATE_CASE(7) STATE_CASE(8)
      default: return ERR_UNSUPPORTED_SIZE;
    }
#undef STATE_CASE
    RETURN_IF_LAUNCH_FAILED();
  }
  {
    // states and their areas are whole pieces of four (P * N is a multiple of 512) unless a caller's view begins
    // in the middle of one
    const long per_head = (long)P * N;
    const bool pieces = (((uintptr_t)chunk_state | (uintptr_t)ssm_state) % 16) == 0 && ((uintptr_t)state_in % 8) == 0;
    const int threads = pieces ? 64 : 256, each = pieces ? 4 : 1;
    const dim3 grid((unsigned)((per_head / each + threads - 1) / threads),
                    H + (conv_here ? (C + threads - 1) / threads : 0), n_lanes);
#define PASS_CASE(V_)                                                                                              \
  ssd_state_pass_kernel<V_><<<grid, threads, 0, stream>>>(chunk_state, chunk_decay, lane_chunks, slot_ids, H, per_head, \
                                                          ssm_state, (bf16_t*)state_in, (const bf16_t*)u, u_ld, C,     \
                                                          conv_k, (bf16_t*)conv_state, chunks, Q)
    if (pieces) PASS_CASE(4);
    else PASS_CASE(1);
#undef PASS_CASE
    RETURN_IF_LAUNCH_FAILED();
  }
  if (beside) {
    int status = ERR_UNSUPPORTED_SIZE;
#define SCAN_BESIDE_CASE(NK_, PT_)                                                                                \
  if (N == 32 * NK_ && P == 16 * PT_)                                                                             \
    status = launch_ssd_scan_beside<NK_, PT_>(stream, (const bf16_t*)xbc, xbc_ld, (const bf16_t*)TT, E, (const bf16_t*)state_in, \
                                              delta, cum, D, chunks, n_chunks, Q, H, G, y, y_ld, (const bf16_t*)z, z_ld, \
                                              (bf16_t*)gated, gated_ld, *beside);
    SCAN_BESIDE_CASE(4, 4) SCAN_BESIDE_CASE(4, 8) SCAN_BESIDE_CASE(8, 4) SCAN_BESIDE_CASE(8, 8)
#undef SCAN_BESIDE_CASE
    if (status != 0) return status;
    RETURN_IF_LAUNCH_FAILED();
    return 0;
  }
  if (mi_ssd_staged(Q, P, N)) {
    const dim3 grid(n_chunks, H, (Q + 127) / 128);
    const size_t lds = ssd_scan_lds_bytes(Q, P, N);
#define SCAN_LDS_CASE(NK_, PT_)                                                                                   \
  if (N == 32 * NK_ && P == 16 * PT_)                                                                             \
    ssd_chunk_scan_lds_kernel<NK_, PT_><<<grid, SSD_SCAN_WAVES * WAVE, lds, stream>>>(                            \
        (const bf16_t*)xbc, xbc_ld, (const bf16_t*)TT, E, (const bf16_t*)state_in, delta, cum, D, chunks, Q, H, G, \
        y, y_ld, (const bf16_t*)z, z_ld, (bf16_t*)gated, gated_ld);
    SCAN_LDS_CASE(1, 1) SCAN_LDS_CASE(1, 2) SCAN_LDS_CASE(1, 4) SCAN_LDS_CASE(1, 8)
    SCAN_LDS_CASE(2, 1) SCAN_LDS_CASE(2, 2) SCAN_LDS_CASE(2, 4) SCAN_LDS_CASE(2, 8)
    SCAN_LDS_CASE(4, 1) SCAN_LDS_CASE(4, 2) SCAN_LDS_CASE(4, 4) SCAN_LDS_CASE(4, 8)
    SCAN_LDS_CASE(8, 1) SCAN_LDS_CASE(8, 2) SCAN_LDS_CASE(8, 4) SCAN_LDS_CASE(8, 8)
#undef SCAN_LDS_CASE
    RETURN_IF_LAUNCH_FAILED();
  } else {
    const int subsets = (H / G + SSD_HEADS_PER_BLOCK - 1) / SSD_HEADS_PER_BLOCK;
    const dim3 grid(n_chunks, G * subsets, (Q + 63) / 64);
#define SCAN_CASE(NK_)                                                                                            \
  case NK_:                                                                                                       \
    ssd_chunk_scan_kernel<SSD_HEADS_PER_BLOCK, NK_><<<grid, 256, 0, stream>>>(                                    \
        (const bf16_t*)xbc, xbc_ld, (const bf16_t*)TT, E, (const bf16_t*)state_in, delta, cum, D, chunks, Q, H, P, \
        G, y, y_ld, (const bf16_t*)z, z_ld, (bf16_t*)gated, gated_ld);                                          \
    break;
    switch (N / 32) {
      SCAN_CASE(1) SCAN_CASE(2) SCAN_CASE(3) SCAN_CASE(4) SCAN_CASE(5) SCAN_CASE(6) SCAN_CASE(7) SCAN_CASE(8)
      default: return ERR_UNSUPPORTED_SIZE;
    }
#undef SCAN_CASE
    RETURN_IF_LAUNCH_FAILED();
  }
  return 0;
}
