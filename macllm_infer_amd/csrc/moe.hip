// A feed-forward of many small experts of which a token uses a few.
//
//   moe_route        float32 router logits -> softmax, correction, the token's experts and their weights (one wave
//                    a token), and the sigmoid of the shared expert's gate logit; or (mode 1) logits + bias -> the
//                    largest ones and the softmax over those alone; groups of neighbouring experts may restrict
//                    the choice to the best groups
//   moe_plan         the step's (token, choice) rows grouped by expert, every expert's rows starting a tile of 16
//                    places: built on the device by one workgroup, so that no count has to travel to the host and
//                    the launches that follow depend on the number of tokens alone; a shared expert's rows may stand
//                    in front of them, as one expert more
//   moe_expert_gemm  the grouped product on the matrix cores: a tile's rows (gathered from the tokens' rows, or
//                    the places themselves) with its expert's matrix; epilogue: plain, or the clamped gated
//                    activation of a gate tile and an up tile
//   moe_combine      a token's weighted sum over its choices, in their order, plus the (gated) shared expert
//
// The router may have more outputs than there are experts with matrices: the last ones are identity experts, whose
// output is the token's own row.  The plan gives their choices no place, the sum takes the row itself.
//
// A row of a tile is summed on its own (a column of the matrix cores' result), so a token's numbers do not depend
// on which other rows share its tile or on the place it was given.
#include "mfma_tile.h"

#define MOE_MAX_EXPERTS 1024
#define MOE_PER_LANE (MOE_MAX_EXPERTS / WAVE)

// ---------------------------------------------------------------- router
// The largest number of a wave and the smallest, in every lane: shifts within the rows of 16 lanes, then across them
// (data-parallel primitives: no trips through the LDS crossbar; neither depends on the order it is taken in).
template <int CONTROL, int ROW_MASK>
__device__ __forceinline__ int moved_or(int x, int otherwise) {
  return __builtin_amdgcn_update_dpp(otherwise, x, CONTROL, ROW_MASK, 0xf, false);
}
__device__ __forceinline__ float wave_most(float v) {
  const int none = __builtin_bit_cast(int, -INFINITY);
#define MOST_STEP(C_, M_) v = fmaxf(v, __builtin_bit_cast(float, moved_or<C_, M_>(__builtin_bit_cast(int, v), none)))
  MOST_STEP(0x111, 0xf); MOST_STEP(0x112, 0xf); MOST_STEP(0x114, 0xf); MOST_STEP(0x118, 0xf); MOST_STEP(0x142, 0xa); MOST_STEP(0x143, 0xc);
#undef MOST_STEP
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ int wave_least(int v) {
#define LEAST_STEP(C_, M_) v = min(v, moved_or<C_, M_>(v, 0x7fffffff))
  LEAST_STEP(0x111, 0xf); LEAST_STEP(0x112, 0xf); LEAST_STEP(0x114, 0xf); LEAST_STEP(0x118, 0xf); LEAST_STEP(0x142, 0xa); LEAST_STEP(0x143, 0xc);
#undef LEAST_STEP
  return __builtin_amdgcn_readlane(v, 63);
}

struct RouteArgs {
  const float* logits;
  long ld;
  int T, E, top;
  const float* correction;
  float scale, eps;
  int mode, renormalize, groups, kept_groups;
  int* chosen;
  float* weights;
  float* gate;
};

// One wave routes one token.  PER_LANE: the most experts a lane holds.
template <int PER_LANE>
__device__ __forceinline__ void route_token(const RouteArgs& a, int token) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int E = a.E, top = a.top;
  const float* row = a.logits + (long)token * a.ld;
  float score[PER_LANE], choice[PER_LANE];
  const int held = (E + WAVE - 1) / WAVE;          // experts a lane holds: the loops below end there (the same in every lane)
  float most = -INFINITY;
#pragma unroll
  for (int j = 0; j < PER_LANE; ++j) {
    if (j >= held) break;
    const int e = lane + WAVE * j;
    score[j] = e < E ? row[e] : -INFINITY;
    choice[j] = (a.correction && e < E) ? a.correction[e] : 0.f;     // (asked for beside the logits)
    most = fmaxf(most, score[j]);
  }
  if (a.mode == 0) {
    most = wave_most(most);
    float total = 0.f;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      if (j >= held) break;
      const int e = lane + WAVE * j;
      score[j] = e < E ? expf(score[j] - most) : 0.f;
      total += score[j];
    }
    total = wave_sum(total);
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      if (j >= held) break;
      const int e = lane + WAVE * j;
      score[j] = score[j] / total;
      choice[j] = e < E ? score[j] + choice[j] : -INFINITY;
    }
  } else if (a.mode == 2) {
    // every output on its own: s = sigmoid(z).  Without a correction the logits decide, whose order is that of the s
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      if (j >= held) break;
      const int e = lane + WAVE * j;
      const float logit = score[j];
      score[j] = e < E ? 1.0f / (1.0f + expf(-logit)) : 0.f;
      choice[j] = e < E ? (a.correction ? score[j] + choice[j] : logit) : -INFINITY;
    }
  } else {
    // the logits with their bias are what is chosen by and what is weighted
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      if (j >= held) break;
      const int e = lane + WAVE * j;
      score[j] = e < E ? score[j] + choice[j] : -INFINITY;
      choice[j] = score[j];
    }
  }
  // the expert with the largest number among those whose bit is not set in `out`: ties go to the lower expert
  auto best_of = [&](unsigned out) {
    float best = -INFINITY;
    int best_id = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j) {
      if (j >= held) break;
      const int e = lane + WAVE * j;
      if (e < E && !(out >> j & 1) && (choice[j] > best || (choice[j] == best && e < best_id))) {
        best = choice[j];
        best_id = e;
      }
    }
    const float largest = wave_most(best);
    return wave_least(best == largest ? best_id : 0x7fffffff);
  };
  if (a.groups > 0) {
    // the best groups, one round each: the largest choice score outside the groups kept so far is its group's score.
    // Everything outside the kept groups ends at minus infinity.
    const int group_size = E / a.groups;
    unsigned kept = 0;                 // bit j: this lane's j-th expert belongs to a kept group
    for (int k = 0; k < a.kept_groups; ++k) {
      const int group = best_of(kept) / group_size;
#pragma unroll
      for (int j = 0; j < PER_LANE; ++j) {
        if (j >= held) break;
        if ((lane + WAVE * j) / group_size == group) kept |= 1u << j;
      }
    }
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j)
      if (j < held && !(kept >> j & 1)) choice[j] = -INFINITY;
  }
  float first_picked = 0.f;        // mode 1: the largest chosen logit, which is the first one picked
  float picked_sum = 0.f;
  float mine = 0.f;            // lane k keeps the score of the k-th choice
  int mine_id = 0;
  for (int k = 0; k < top; ++k) {
    const int best_id = min(best_of(0), E - 1);     // scores that are no numbers pick nothing: whatever is chosen is an expert
    float own = 0.f;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j)
      if (j < held && lane + WAVE * j == best_id) {
        choice[j] = -INFINITY;
        own = score[j];
      }
    float best_score = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, own), best_id & (WAVE - 1)));
    if (a.mode == 1) {
      if (k == 0) first_picked = best_score;
      best_score = expf(best_score - first_picked);
    }
    picked_sum += best_score;
    if ((k & (WAVE - 1)) == lane) {
      mine = best_score;
      mine_id = best_id;
    }
    if (top > WAVE && lane == 0) {       // more choices than lanes: written as they come
      a.chosen[(long)token * top + k] = best_id;
      a.weights[(long)token * top + k] = best_score;      // divided below
    }
  }
  const float denominator = a.renormalize ? picked_sum + a.eps : 1.0f;
  if (top <= WAVE) {
    if (lane < top) {
      a.chosen[(long)token * top + lane] = mine_id;
      a.weights[(long)token * top + lane] = mine / denominator * a.scale;
    }
  } else if (lane == 0) {
    for (int k = 0; k < top; ++k) a.weights[(long)token * top + k] = a.weights[(long)token * top + k] / denominator * a.scale;
  }
  if (a.gate && lane == 0) a.gate[token] = 1.0f / (1.0f + expf(-row[E]));
}

template <int PER_LANE>
__global__ void __launch_bounds__(256) moe_route_kernel(RouteArgs a) {
  const int token = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
  if (token < a.T) route_token<PER_LANE>(a, token);
}

static int check_route(const RouteArgs& a) {
  if (!a.logits || !a.chosen || !a.weights || a.T <= 0 || a.E <= 0 || a.top <= 0 || a.top > a.E || a.ld < a.E + (a.gate ? 1 : 0))
    return ERR_BAD_ARGUMENT;
  if (a.E > MOE_MAX_EXPERTS) return ERR_UNSUPPORTED_SIZE;
  if (a.mode < 0 || a.mode > 2) return ERR_BAD_ARGUMENT;
  if (a.mode == 1 && (!a.renormalize || a.groups != 0)) return ERR_BAD_ARGUMENT;
  if (a.groups < 0 || (a.groups > 0 && (a.E % a.groups != 0 || a.kept_groups <= 0 || a.kept_groups > a.groups ||
                                        a.kept_groups * (a.E / a.groups) < a.top)))
    return ERR_BAD_ARGUMENT;
  return 0;
}

// mode 0: softmax over all experts, choice by score + correction, weights score / (sum of the chosen + eps) * scale,
// or without `renormalize` score * scale.  groups > 0 (mode 0): E / groups neighbouring experts form a group, its score
// is its largest score + correction, and only experts of the `kept_groups` best groups can be chosen.
// mode 1: choice by logit + correction (a bias), weights the softmax over the chosen (logit + correction) * scale.
// mode 2: as mode 0 with the sigmoid of each logit in place of the softmax.  correction may be null (nothing is added).
extern "C" int mi_moe_route(const float* logits, long ld, int T, int E, int top, const float* correction, float scale,
                            float eps, int mode, int renormalize, int groups, int kept_groups, int* chosen, float* weights,
                            float* gate, hipStream_t stream) {
  const RouteArgs a = {logits, ld, T, E, top, correction, scale, eps, mode, renormalize, groups, kept_groups, chosen, weights, gate};
  const int code = check_route(a);
  if (code) return code;
  if (E <= 2 * WAVE) moe_route_kernel<2><<<(T + 3) / 4, 256, 0, stream>>>(a);
  else moe_route_kernel<MOE_PER_LANE><<<(T + 3) / 4, 256, 0, stream>>>(a);
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---------------------------------------------------------------- rows grouped by expert
struct PlanArgs {
  const int* chosen;
  int entries, top, E, pad, capacity;
  int* source;
  int* place;
  int* tile_expert;
  int* ranks;
  const float* weights;             // with place_weight: the choices' weights, laid beside the places (padding gets 0)
  float* place_weight;
  int shared;                       // a shared expert's rows: rows 0 .. shared - 1 of the step stand at the places of these numbers, as expert E
};

// By one workgroup; a choice of E or beyond is an identity expert and gets the place -1.  Bound by its chain of round trips:
// what a thread has read and counted of its first PLAN_KEPT entries stays in registers (4,662 of 16 experts 7.8 -> 5.6 us; in the
// launch that routes small steps too it costs them 2 to 6 us in twelve layers, so there none).
template <int PLAN_KEPT>
__device__ __forceinline__ void plan_rows(const PlanArgs& a, int* counts, int* offsets) {
  const int tid = threadIdx.x;
  const int threads = blockDim.x;
  const int shared_tiles = (a.shared + a.pad - 1) / a.pad;
  int expert[PLAN_KEPT + 1], rank[PLAN_KEPT + 1];           // of the entries that this thread keeps; the rest goes through memory
#pragma unroll
  for (int j = 0; j < PLAN_KEPT; ++j) {
    expert[j] = -1;
    rank[j] = 0;
    if (j * threads < a.entries && tid + j * threads < a.entries) expert[j] = a.chosen[tid + j * threads];
  }
  for (int e = tid; e < a.E; e += threads) counts[e] = 0;
  for (int i = tid; i < a.capacity; i += threads) {
    a.source[i] = i < a.shared ? i : -1;
    if (a.place_weight) a.place_weight[i] = 0.f;
  }
  for (int t = tid; t < a.capacity / a.pad; t += threads) a.tile_expert[t] = t < shared_tiles ? a.E : -1;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PLAN_KEPT; ++j)
    if ((unsigned)expert[j] < (unsigned)a.E) rank[j] = atomicAdd(&counts[expert[j]], 1);      // (an identity expert's choice stands nowhere)
  for (int i = tid + PLAN_KEPT * threads; i < a.entries; i += threads) {
    const int one = a.chosen[i];
    if (one < a.E) a.ranks[i] = atomicAdd(&counts[one], 1);
  }
  __syncthreads();
  // where every expert's places begin: whole tiles, an inclusive sum over the wave in turns of 64 experts
  if (tid < WAVE) {
    int before = shared_tiles * a.pad;
    for (int e0 = 0; e0 < a.E; e0 += WAVE) {
      const int e = e0 + tid;
      const int places = e < a.E ? (counts[e] + a.pad - 1) / a.pad * a.pad : 0;
      int running = places;
#pragma unroll
      for (int offset = 1; offset < WAVE; offset <<= 1) {
        const int other = __shfl_up(running, offset, WAVE);
        if (tid >= offset) running += other;
      }
      if (e < a.E) offsets[e] = before + running - places;
      before += __shfl(running, WAVE - 1, WAVE);
    }
  }
  __syncthreads();
  for (int e = tid; e < a.E; e += threads) {
    const int first = offsets[e] / a.pad;
    const int tiles = (counts[e] + a.pad - 1) / a.pad;
    for (int t = 0; t < tiles; ++t) a.tile_expert[first + t] = e;
  }
#pragma unroll
  for (int j = 0; j < PLAN_KEPT; ++j) {
    const int i = tid + j * threads;
    if (expert[j] < 0) continue;
    const int at = expert[j] < a.E ? offsets[expert[j]] + rank[j] : -1;
    a.place[i] = at;
    if (at < 0) continue;
    a.source[at] = i / a.top;
    if (a.place_weight) a.place_weight[at] = a.weights[i];
  }
  for (int i = tid + PLAN_KEPT * threads; i < a.entries; i += threads) {
    const int one = a.chosen[i];
    if (one >= a.E) {
      a.place[i] = -1;
      continue;
    }
    const int at = offsets[one] + a.ranks[i];
    a.source[at] = i / a.top;
    a.place[i] = at;
    if (a.place_weight) a.place_weight[at] = a.weights[i];
  }
}

__global__ void __launch_bounds__(1024) moe_plan_kernel(PlanArgs a) {
  __shared__ int counts[MOE_MAX_EXPERTS];
  __shared__ int offsets[MOE_MAX_EXPERTS];
  plan_rows<8>(a, counts, offsets);
}

static int check_plan(const PlanArgs& a) {
  if (a.place_weight && !a.weights) return ERR_BAD_ARGUMENT;
  if (!a.chosen || !a.source || !a.place || !a.tile_expert || !a.ranks || a.entries <= 0 || a.top <= 0 || a.E <= 0 || a.pad <= 0 ||
      a.capacity % a.pad != 0 || a.shared < 0 || (a.shared > 0 && a.place_weight) ||
      a.capacity < (a.shared + a.pad - 1) / a.pad * a.pad + a.entries + a.E * (a.pad - 1))
    return ERR_BAD_ARGUMENT;
  return a.E > MOE_MAX_EXPERTS ? ERR_UNSUPPORTED_SIZE : 0;
}

extern "C" int mi_moe_plan(const int* chosen, int entries, int top, int E, int pad, int capacity, int* source, int* place,
                           int* tile_expert, int* ranks, const float* weights, float* place_weight, int shared,
                           hipStream_t stream) {
  const PlanArgs a = {chosen, entries, top, E, pad, capacity, source, place, tile_expert, ranks, weights, place_weight, shared};
  const int code = check_plan(a);
  if (code) return code;
  moe_plan_kernel<<<1, 1024, 0, stream>>>(a);
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// Choice and grouping of a step of few tokens in one launch: a wave a token, then the workgroup groups what its waves
// chose (the same workgroup: a barrier makes its own writes visible).
#define ROUTE_PLAN_TOKENS 64
template <int PER_LANE>
__global__ void __launch_bounds__(1024) moe_route_plan_kernel(RouteArgs route, PlanArgs plan) {
  __shared__ int counts[MOE_MAX_EXPERTS];
  __shared__ int offsets[MOE_MAX_EXPERTS];
  for (int token = threadIdx.x / WAVE; token < route.T; token += blockDim.x / WAVE) route_token<PER_LANE>(route, token);
  __threadfence_block();
  __syncthreads();
  plan_rows<0>(plan, counts, offsets);
}

// experts: those with matrices, at most route's E.
extern "C" int mi_moe_route_plan(const float* logits, long ld, int T, int E, int top, const float* correction, float scale,
                                 float eps, int mode, int renormalize, int groups, int kept_groups, int* chosen,
                                 float* weights, float* gate, int experts, int pad, int capacity, int* source, int* place,
                                 int* tile_expert, int* ranks, float* place_weight, int shared, hipStream_t stream) {
  const RouteArgs route = {logits, ld, T, E, top, correction, scale, eps, mode, renormalize, groups, kept_groups, chosen, weights, gate};
  const PlanArgs plan = {chosen, T * top, top, experts, pad, capacity, source, place, tile_expert, ranks, weights, place_weight, shared};
  int code = check_route(route);
  if (!code) code = check_plan(plan);
  if (code) return code;
  if (T > ROUTE_PLAN_TOKENS || experts > E) return ERR_UNSUPPORTED_SIZE;
  const int threads = T >= 16 ? 1024 : (T > 4 ? T * WAVE : 4 * WAVE);
  if (E <= 2 * WAVE) moe_route_plan_kernel<2><<<1, threads, 0, stream>>>(route, plan);
  else moe_route_plan_kernel<MOE_PER_LANE><<<1, threads, 0, stream>>>(route, plan);
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---------------------------------------------------------------- the grouped product
// The sums of the expert `rounded` (-1: none) are rounded to bfloat16 before anything else is done with them, as those of a product
// of its own are, and in the same order: an expert gets the same bits in a launch with others as in launches of its own.  In tiles
// of 16 places that is the order of the product of few rows, four runs of K (K up to 1,024), or with in_k_order that of the
// product of many rows, which the tiles of 64 and 128 places have anyway.  In k order a wave walks all of K, eight chunks at a time,
// beside the routed experts' tiles: steps of twelve layers with the shared expert apart | so, us: 32 decoded tokens 1,372 | 1,253,
// 64 1,638 | 1,477, a prompt of 40 1,391 | 1,236, 100 1,403 | 1,310.
__device__ __forceinline__ float sum_as(float sum, bool rounded) { return rounded ? (float)(bf16_t)sum : sum; }

// Tile t of 16 MT places belongs to expert tile_expert[t] (none: the workgroup leaves).  A workgroup owns the
// tile's rows and PAIRS tiles of 16 output features.  GLU: the expert's matrix is [2 I, K], gate rows then up
// rows; out[place, n] = act(gate tile, up tile), n < I.  Places without a row get zeros.  Steps of few rows take
// MT = 1 (every expert's matrix is read once, by as many workgroups as it has tiles of features); prompt portions,
// whose experts get dozens of rows each, MT = 4 and four tiles of features (the rows and the matrix come from the
// caches, 64 x 64 results a workgroup).  Steps of few rows are bound by the matrices (12 tokens, 16 of 17 experts of 512 x 1,024: 33 MB
// in 9.8 us, 17 in 8.1, launch and two round trips of the tables among it); a wave's whole run of up to eight chunks is on its way
// at once (two of them: a prompt of 40 1,254 -> 1,236 us, of 64 1,359 -> 1,343, 12 decoded tokens the same).
template <typename T, typename TO, bool VEC, bool GLU, int MT, int PAIRS>
__global__ void __launch_bounds__(TILE_THREADS)
moe_expert_gemm_kernel(const T* __restrict__ x, long ldx, int x_rows, const T* __restrict__ W, long expert_stride, long ldw,
                       int N, int K, const int* __restrict__ source, const int* __restrict__ tile_expert, int gather,
                       float limit, float alpha, float offset, int squared_relu,
                       const float* __restrict__ row_scale, int rounded, int in_k_order, TO* __restrict__ out, long ldo) {
  __shared__ float red[TILE_WAVES][256];
  const int tile = blockIdx.y;
  const int tid = threadIdx.x;
  const int r = (tid & (WAVE - 1)) % 16;
  const int expert = tile_expert[tile];
  int from[MT];                                      // the rows that stand at the tile's places, beside the expert's number
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) from[mt] = source[(tile * MT + mt) * 16 + r];
  if (expert < 0) return;
  const int width = GLU ? N / 2 : N;
  const long n0 = (long)blockIdx.x * 16 * PAIRS;
  const T* matrix = W + (long)expert * expert_stride;
  constexpr int NT = GLU ? 2 * PAIRS : PAIRS;
  const T* w_row[NT];
  const T* x_row[MT];
#pragma unroll
  for (int p = 0; p < PAIRS; ++p) {
    const long n_row = min(n0 + 16 * p + r, (long)width - 1);
    w_row[p] = matrix + n_row * ldw;
    if (GLU) w_row[NT - PAIRS + p] = matrix + (width + n_row) * ldw;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const long x_at = gather ? max(from[mt], 0) : (tile * MT + mt) * 16 + r;
    x_row[mt] = x + min(x_at, (long)x_rows - 1) * ldx;
  }
  tile_floatx4 acc[NT][MT];
  const int l = tid % 64;
  bool serial = false;                               // the tiles of `rounded` whose sums run through K in one wave each
  if constexpr (MT == 1 && PAIRS == 1 && VEC) {
    serial = in_k_order && expert == rounded;
    if (serial) {
      // the NT tiles of features by as many waves, eight chunks asked for at once; the sums to where tile_reduce would read them
      constexpr int CHUNK = TileTraits<T>::CHUNK, PIECE = TileTraits<T>::PIECE;
      const int wave = tid / WAVE, q = (tid & (WAVE - 1)) / 16;
      const T* const mine = w_row[NT > 1 && wave == 1 ? NT - 1 : 0];
      tile_floatx4 sum = {0.f, 0.f, 0.f, 0.f};
      if (wave < NT)
        for (int k0 = 0; k0 < K; k0 += 8 * CHUNK) {
          typename TileTraits<T>::Piece a[8], b[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            a[j] = tile_load<T, true>(mine, k0 + j * CHUNK + PIECE * q, K);
            b[j] = tile_load<T, true>(x_row[0], k0 + j * CHUNK + PIECE * q, K);
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) sum = tile_mfma(a[j], b[j], sum);
        }
      if (wave < NT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][i * 64 + (tid & (WAVE - 1))] = sum[i];
      }
      __syncthreads();
    }
  }
  if constexpr (MT == 1 && PAIRS == 1 && VEC) {
    if (serial) {
    } else if (K <= TILE_WAVES * 4 * TileTraits<T>::CHUNK) {
      tile_accumulate<T, MT, NT, VEC, 4>(w_row, x_row, K, acc);
    } else {
      tile_accumulate<T, MT, NT, VEC, 8>(w_row, x_row, K, acc);
    }
  } else {
    tile_accumulate<T, MT, NT, VEC>(w_row, x_row, K, acc);
  }
#pragma unroll
  for (int p = 0; p < PAIRS; ++p)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int place = (tile * MT + mt) * 16 + (l % 16);
      const float scale = row_scale ? row_scale[place] : 1.0f;
      float value = sum_as((serial ? red[0][tid] : tile_reduce(acc[p][mt], red)) * scale, expert == rounded);
      if (GLU) {
        const float up = sum_as((serial ? red[1][tid] : tile_reduce(acc[NT - PAIRS + p][mt], red)) * scale, expert == rounded);
        const float g = fminf(value, limit);
        const float u = fminf(fmaxf(up, -limit), limit);
        value = g / (1.0f + expf(-alpha * g)) * (u + offset);
      } else if (squared_relu) {
        value = fmaxf(value, 0.f);
        value *= value;
      }
      const long n = n0 + 16 * p + 4 * (l / 16) + tid / 64;
      if (n < width) out[(long)place * ldo + n] = from_float<TO>(from[mt] >= 0 ? value : 0.f);
    }
}

// Four neighbouring results of one place: in one store where the rows of the output are whole groups of four.
template <typename TO>
__device__ __forceinline__ void store_four(TO* row, long n, int width, bool whole, const float (&value)[4]) {
  typedef TO four_t __attribute__((ext_vector_type(4)));
  if (whole && n + 3 < width) {
    four_t packed;
#pragma unroll
    for (int i = 0; i < 4; ++i) packed[i] = from_float<TO>(value[i]);
    *reinterpret_cast<four_t*>(row + n) = packed;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n + i < width) row[n + i] = from_float<TO>(value[i]);
}

// The same product for prompt portions whose rows and matrices are whole 16-byte pieces: a workgroup owns a tile
// of ROWS places (128 where experts get hundreds of rows each, else 64) and 128 rows of its expert's matrix (GLU: 64
// gate rows and the 64 up rows that go with them, which make 64 outputs; else 128 outputs), every one of its four waves
// half the places and half the features (GLU: 32 gate rows and their 32 up rows): no sum crosses a wave, a row's result
// is summed in k order by one lane's accumulator.  K is walked in stages of eight pieces a row, whole lines of 128 bytes
// (64 columns of bfloat16, 32 of float32), through two LDS stages; the next stage's pieces are asked for before the
// current one's products.  Piece p of row r of a stage lies at r * 8 + (p ^ (r & 7)): the eight rows that a quarter of a
// wave reads at once fall into different groups of banks, and a thread's stores are one run.
// What bounds it: the bytes in flight of a compute unit (a stage a workgroup, 24 or 32 KB).  Three of sixteen experts of
// 512 x 1,024 in bfloat16, us for the two products of 1,554 / 700 tokens: stages of 64 bytes a row 75 / 50 with
// tiles of 128 / 64 places; now 51 / 41 with 128 and 45 / 35 with 64.  (Bounds of two workgroups a compute unit keep the
// sums out of the accumulator registers, whose moves cost 20 us; two or three stages on their way: 55 and 62 with 128.)
template <typename T, typename TO, bool GLU, int ROWS>
__global__ void __launch_bounds__(TILE_THREADS, 2)
moe_expert_gemm_wide_kernel(const T* __restrict__ x, long ldx, int x_rows, const T* __restrict__ W, long expert_stride,
                            long ldw, int N, int K, const int* __restrict__ source, const int* __restrict__ tile_expert,
                            int gather, float limit, float alpha, float offset, int squared_relu,
                            const float* __restrict__ row_scale, int rounded, TO* __restrict__ out, long ldo, int whole) {
  typedef typename TileTraits<T>::Piece Piece;
  constexpr int PIECE = TileTraits<T>::PIECE;
  constexpr int STAGE_K = 8 * PIECE;
  constexpr int FEATURES = 128;
  constexpr int MT = ROWS / 32;                                // tiles of 16 places a wave
  constexpr int X_PIECES = ROWS * 8 / TILE_THREADS, W_PIECES = FEATURES * 8 / TILE_THREADS;
  __shared__ Piece stage[2][(ROWS + FEATURES) * 8];
  const int tile = blockIdx.y;
  const int expert = tile_expert[tile];
  if (expert < 0) return;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE - 1);
  const int wave = tid / WAVE;
  const int wm = wave / 2;                                     // which half of the places
  const int wn = wave % 2;                                     // which half of the features
  const int q = lane / 16;
  const int r = lane % 16;
  const int width = GLU ? N / 2 : N;
  const long n0 = (long)blockIdx.x * (GLU ? 64 : 128);
  const T* matrix = W + (long)expert * expert_stride;
  // what this thread brings into a stage: one piece each of X_PIECES rows of x and W_PIECES of the matrix, 32 rows apart
  const int lrow = tid / 8;
  const int column = PIECE * ((tid % 8) ^ (lrow & 7));
  const T* x_from[X_PIECES];
  const T* w_from[W_PIECES];
#pragma unroll
  for (int j = 0; j < X_PIECES; ++j) {
    const int place_in = tile * ROWS + lrow + 32 * j;
    const long x_at = gather ? max(source[place_in], 0) : place_in;
    x_from[j] = x + min(x_at, (long)x_rows - 1) * ldx;
  }
#pragma unroll
  for (int j = 0; j < W_PIECES; ++j) {
    const int row = lrow + 32 * j;                             // of the stage's matrix part
    const long feature = GLU ? (row < 64 ? 0 : width) + min(n0 + row % 64, (long)width - 1) : min(n0 + row, (long)width - 1);
    w_from[j] = matrix + feature * ldw;
  }
  tile_floatx4 acc[4][MT];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = tile_floatx4{0.f, 0.f, 0.f, 0.f};
  const int stages = (K + STAGE_K - 1) / STAGE_K;
  Piece gx[X_PIECES], gw[W_PIECES];
  auto ask = [&](int stage_number) {                           // (a piece past the end: the row's last one, laid as zeros)
    const int k = min(stage_number * STAGE_K + column, K - PIECE);
#pragma unroll
    for (int j = 0; j < X_PIECES; ++j) gx[j] = *reinterpret_cast<const Piece*>(x_from[j] + k);
#pragma unroll
    for (int j = 0; j < W_PIECES; ++j) gw[j] = *reinterpret_cast<const Piece*>(w_from[j] + k);
  };
  auto lay = [&](int stage_number) {
    const bool there = stage_number * STAGE_K + column < K;
    Piece* const into = stage[stage_number & 1];
    const Piece none = {};
#pragma unroll
    for (int j = 0; j < X_PIECES; ++j) into[tid + TILE_THREADS * j] = there ? gx[j] : none;
#pragma unroll
    for (int j = 0; j < W_PIECES; ++j) into[ROWS * 8 + tid + TILE_THREADS * j] = there ? gw[j] : none;
  };
  auto multiply = [&](const Piece* staged) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      Piece a[4], b[MT];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        // GLU: nt 0, 1 are gate rows, nt 2, 3 the up rows of the same outputs (the stage's second 64 rows)
        const int row = GLU ? 64 * (nt / 2) + 32 * wn + 16 * (nt % 2) + r : 64 * wn + 16 * nt + r;
        a[nt] = staged[(ROWS + row) * 8 + ((4 * c + q) ^ (row & 7))];
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int row = 16 * MT * wm + 16 * mt + r;
        b[mt] = staged[row * 8 + ((4 * c + q) ^ (row & 7))];
      }
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = tile_mfma(a[nt], b[mt], acc[nt][mt]);
    }
  };
  ask(0);
  lay(0);
  __syncthreads();
  for (int s = 0; s < stages; ++s) {
    ask(s + 1);
    __builtin_amdgcn_sched_barrier(0);                         // (left to itself the scheduler moves the loads behind the products)
    multiply(stage[s & 1]);
    __builtin_amdgcn_sched_barrier(0);
    lay(s + 1);
    __syncthreads();
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int place = tile * ROWS + 16 * MT * wm + 16 * mt + r;
    const bool live = source[place] >= 0;
    const float scale = row_scale ? row_scale[place] : 1.0f;
    TO* row = out + (long)place * ldo;
    if (GLU) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float value[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = fminf(sum_as(acc[h][mt][i] * scale, expert == rounded), limit);
          const float u = fminf(fmaxf(sum_as(acc[2 + h][mt][i] * scale, expert == rounded), -limit), limit);
          value[i] = live ? g / (1.0f + expf(-alpha * g)) * (u + offset) : 0.f;
        }
        store_four<TO>(row, n0 + 32 * wn + 16 * h + 4 * q, width, whole != 0, value);
      }
    } else {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        float value[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          value[i] = sum_as(acc[nt][mt][i] * scale, expert == rounded);
          if (squared_relu) {
            value[i] = fmaxf(value[i], 0.f);
            value[i] *= value[i];
          }
          if (!live) value[i] = 0.f;
        }
        store_four<TO>(row, n0 + 64 * wn + 16 * nt + 4 * q, width, whole != 0, value);
      }
    }
  }
}

template <typename T, typename TO>
static void launch_expert_gemm(const T* x, long ldx, int x_rows, const T* W, long expert_stride, long ldw, int N, int K,
                               const int* source, const int* tile_expert, int tiles, int pad, int gather, int activation,
                               float limit, float alpha, float offset, const float* row_scale, int rounded, int in_k_order, TO* out, long ldo,
                               hipStream_t stream) {
  const int glu = activation == 1;
  const int squared_relu = activation == 2;
  constexpr int PIECE = TileTraits<T>::PIECE;
  const bool vec = K % PIECE == 0 && ldx % PIECE == 0 && ldw % PIECE == 0 && expert_stride % PIECE == 0 &&
                   ((unsigned long long)x % 16) == 0 && ((unsigned long long)W % 16) == 0;
  const int width = glu ? N / 2 : N;
#define EXPERT_LAUNCH(VEC_, GLU_, MT_, PAIRS_)                                                                           moe_expert_gemm_kernel<T, TO, VEC_, GLU_, MT_, PAIRS_>                                                                    <<<dim3((unsigned)((width + 16 * PAIRS_ - 1) / (16 * PAIRS_)), (unsigned)tiles), TILE_THREADS, 0, stream>>>(               x, ldx, x_rows, W, expert_stride, ldw, N, K, source, tile_expert, gather, limit, alpha, offset, squared_relu, row_scale, rounded, in_k_order, out, ldo)
#define EXPERT_SHAPE(MT_, PAIRS_GLU_, PAIRS_PLAIN_)                                                                      do {                                                                                                                    if (vec && glu) EXPERT_LAUNCH(true, true, MT_, PAIRS_GLU_);                                                            else if (vec) EXPERT_LAUNCH(true, false, MT_, PAIRS_PLAIN_);                                                           else if (glu) EXPERT_LAUNCH(false, true, MT_, PAIRS_GLU_);                                                             else EXPERT_LAUNCH(false, false, MT_, PAIRS_PLAIN_);                                                                 } while (0)
  if ((pad == 128 || pad == 64) && vec) {      // (plans of 128 places are made of rows and matrices in whole pieces only)
    const dim3 grid((unsigned)((width + (glu ? 64 : 128) - 1) / (glu ? 64 : 128)), (unsigned)tiles);
    const int whole = ldo % 4 == 0 && ((unsigned long long)out % 16) == 0;
#define EXPERT_WIDE(GLU_, ROWS_)                                                                                  \
  moe_expert_gemm_wide_kernel<T, TO, GLU_, ROWS_><<<grid, TILE_THREADS, 0, stream>>>(                             \
      x, ldx, x_rows, W, expert_stride, ldw, N, K, source, tile_expert, gather, limit, alpha, offset, squared_relu, \
      row_scale, rounded, out, ldo, whole)
    if (pad == 128 && glu) EXPERT_WIDE(true, 128);
    else if (pad == 128) EXPERT_WIDE(false, 128);
    else if (glu) EXPERT_WIDE(true, 64);
    else EXPERT_WIDE(false, 64);
#undef EXPERT_WIDE
  } else if (pad == 64) {
    EXPERT_SHAPE(4, 2, 4);
  } else {
    EXPERT_SHAPE(1, 1, 1);
  }
#undef EXPERT_SHAPE
#undef EXPERT_LAUNCH
}

extern "C" int mi_moe_expert_gemm(const void* x, int dtype, long ldx, int x_rows, const void* W, long expert_stride,
                                  long ldw, int N, int K, const int* source, const int* tile_expert, int tiles, int pad,
                                  int gather, int activation, float limit, float alpha, float offset,
                                  const float* row_scale, int rounded, int in_k_order, void* out, int out_dtype, long ldo, hipStream_t stream) {
  // row_scale (or null): a number for every place that multiplies its row before the product (as the products are linear
  // in the row, the sums before the activation)
  // activation: 0 none, 1 the clamped gated one (the matrix holds gate rows then up rows), 2 max(z, 0)^2
  const int glu = activation == 1;
  if (activation < 0 || activation > 2) return ERR_BAD_ARGUMENT;
  if (!x || !W || !source || !tile_expert || !out || x_rows <= 0 || N <= 0 || K <= 0 || tiles <= 0 || ldx < K || ldw < K ||
      (glu && N % 2) || ldo < (glu ? N / 2 : N))
    return ERR_BAD_ARGUMENT;
  if ((pad != 16 && pad != 64 && pad != 128) || tiles > 65535) return ERR_UNSUPPORTED_SIZE;
  if (pad == 128) {
    const long piece = dtype == DT_F32 ? 4 : 8;
    if (K % piece || ldx % piece || ldw % piece || expert_stride % piece || ((unsigned long long)x % 16) ||
        ((unsigned long long)W % 16))
      return ERR_UNSUPPORTED_SIZE;
  }
  if (dtype == DT_F32 && out_dtype == DT_F32)
    launch_expert_gemm<float, float>((const float*)x, ldx, x_rows, (const float*)W, expert_stride, ldw, N, K, source,
                                     tile_expert, tiles, pad, gather, activation, limit, alpha, offset, row_scale, rounded, in_k_order, (float*)out, ldo, stream);
  else if (dtype == DT_BF16 && out_dtype == DT_BF16)
    launch_expert_gemm<bf16_t, bf16_t>((const bf16_t*)x, ldx, x_rows, (const bf16_t*)W, expert_stride, ldw, N, K, source,
                                       tile_expert, tiles, pad, gather, activation, limit, alpha, offset, row_scale, rounded, in_k_order, (bf16_t*)out, ldo, stream);
  else if (dtype == DT_BF16 && out_dtype == DT_F32)
    launch_expert_gemm<bf16_t, float>((const bf16_t*)x, ldx, x_rows, (const bf16_t*)W, expert_stride, ldw, N, K, source,
                                      tile_expert, tiles, pad, gather, activation, limit, alpha, offset, row_scale, rounded, in_k_order, (float*)out, ldo, stream);
  else
    return ERR_BAD_ARGUMENT;
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}

// ---------------------------------------------------------------- a token's weighted sum
// total[t, i] = sum over the choices k of weights[t, k] * (down[place[t, k], i], or x[t, i] where the place is negative),
// + (gate[t], or one) * shared[t, i]; weights null: every choice counts once.  Without a tail out = total.  With one the sum goes on into the residual stream in
// the same launch: h += tanh(post_alpha total) * post_w + post_b, and (next_w not null) the new rows through the next
// tanh norm, next_out = tanh(next_alpha h) * next_w + next_b.  A thread takes PIECE neighbouring features of a token.
struct CombineTail {
  float* h;
  const float* post_w;
  const float* post_b;
  const float* next_w;
  const float* next_b;
  float post_alpha, next_alpha;
  void* next_out;                   // [T, d] of x's type
};

template <int PIECE>
__device__ __forceinline__ void piece_of(const float* from, float (&to)[PIECE]) {
  if constexpr (PIECE == 1) {
    to[0] = from[0];
  } else {
    const tile_floatx4 piece = *reinterpret_cast<const tile_floatx4*>(from);
#pragma unroll
    for (int j = 0; j < PIECE; ++j) to[j] = piece[j];
  }
}

template <int PIECE>
__device__ __forceinline__ void piece_of(const bf16_t* from, float (&to)[PIECE]) {
  typedef __bf16 four __attribute__((ext_vector_type(4)));
  if constexpr (PIECE == 1) {
    to[0] = (float)from[0];
  } else {
    const four piece = *reinterpret_cast<const four*>(from);
#pragma unroll
    for (int j = 0; j < PIECE; ++j) to[j] = (float)piece[j];
  }
}

template <typename TS, typename TX, int PIECE>
__global__ void __launch_bounds__(256)
moe_combine_kernel(const float* __restrict__ down, long ld, const int* __restrict__ place, const float* __restrict__ weights,
                   int top, const TX* __restrict__ x, long x_ld, const TS* __restrict__ shared, long shared_ld,
                   const float* __restrict__ gate, float* __restrict__ out, int d, long total_pieces, CombineTail tail) {
  const long index = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (index >= total_pieces) return;
  const int pieces = d / PIECE;
  const long token = index / pieces;
  const int i = (int)(index - token * pieces) * PIECE;
  float own[PIECE], extra[PIECE], total[PIECE], stream[PIECE], pw[PIECE], pb[PIECE], nw[PIECE], nb[PIECE];
#pragma unroll
  for (int j = 0; j < PIECE; ++j) own[j] = extra[j] = total[j] = 0.f;
  if (x) piece_of<PIECE>(x + token * x_ld + i, own);
  if (shared) piece_of<PIECE>(shared + token * shared_ld + i, extra);
  if (tail.h) {
    piece_of<PIECE>(tail.h + token * d + i, stream);
    piece_of<PIECE>(tail.post_w + i, pw);
    piece_of<PIECE>(tail.post_b + i, pb);
    if (tail.next_w) {
      piece_of<PIECE>(tail.next_w + i, nw);
      piece_of<PIECE>(tail.next_b + i, nb);
    }
  }
  for (int k0 = 0; k0 < top; k0 += 4) {
    // four choices' rows asked for at once; a choice past the last reads the last again and weighs nothing
    float value[4][PIECE], weight[4];
    int at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = min(k0 + u, top - 1);
      at[u] = place[token * top + k];
      weight[u] = k0 + u < top ? (weights ? weights[token * top + k] : 1.0f) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) piece_of<PIECE>(down + (long)max(at[u], 0) * ld + i, value[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + u < top) {
#pragma unroll
        for (int j = 0; j < PIECE; ++j) total[j] = fmaf(weight[u], at[u] < 0 ? own[j] : value[u][j], total[j]);
      }
  }
  if (shared) {
    const float share = gate ? gate[token] : 1.0f;
#pragma unroll
    for (int j = 0; j < PIECE; ++j) total[j] = fmaf(share, extra[j], total[j]);
  }
  if (!tail.h) {
    if constexpr (PIECE == 1) out[token * d + i] = total[0];
    else *reinterpret_cast<tile_floatx4*>(out + token * d + i) = tile_floatx4{total[0], total[1], total[2], total[3]};
    return;
  }
#pragma unroll
  for (int j = 0; j < PIECE; ++j) stream[j] += tanh_norm_f(total[j], tail.post_alpha, pw[j], pb[j]);
  if constexpr (PIECE == 1) tail.h[token * d + i] = stream[0];
  else *reinterpret_cast<tile_floatx4*>(tail.h + token * d + i) = tile_floatx4{stream[0], stream[1], stream[2], stream[3]};
  if (!tail.next_w) return;
  TX* next = (TX*)tail.next_out + token * d + i;
  if constexpr (PIECE == 1) {
    next[0] = from_float<TX>(tanh_norm_f(stream[0], tail.next_alpha, nw[0], nb[0]));
  } else {
    typedef TX four __attribute__((ext_vector_type(4)));
    four piece;
#pragma unroll
    for (int j = 0; j < 4; ++j) piece[j] = from_float<TX>(tanh_norm_f(stream[j], tail.next_alpha, nw[j], nb[j]));
    *reinterpret_cast<four*>(next) = piece;
  }
}

// out, or (h not null) the tail, whose next rows have x_dtype.
extern "C" int mi_moe_combine(const float* down, long ld, const int* place, const float* weights, int top, const void* x,
                              int x_dtype, long x_ld, const void* shared, int shared_dtype, long shared_ld,
                              const float* gate, float* out, int T, int d, float* h, const float* post_w,
                              const float* post_b, float post_alpha, const float* next_w, const float* next_b,
                              float next_alpha, void* next_out, hipStream_t stream) {
  if (!down || !place || T <= 0 || d <= 0 || top <= 0 || ld < d || (shared && shared_ld < d) || (x && x_ld < d))
    return ERR_BAD_ARGUMENT;
  if (h ? (!post_w || !post_b || (next_w && (!next_b || !next_out))) : !out) return ERR_BAD_ARGUMENT;
  const CombineTail tail = {h, post_w, post_b, next_w, next_b, post_alpha, next_alpha, next_out};
  const uintptr_t addresses = (uintptr_t)down | (uintptr_t)x | (uintptr_t)shared | (uintptr_t)out | (uintptr_t)h | (uintptr_t)post_w |
                              (uintptr_t)post_b | (uintptr_t)next_w | (uintptr_t)next_b | (uintptr_t)next_out;
  const bool fours = d % 4 == 0 && ld % 4 == 0 && x_ld % 4 == 0 && shared_ld % 4 == 0 && addresses % 16 == 0;
  const long pieces = (long)T * d / (fours ? 4 : 1);
  const int block = pieces <= 64 * 1024 ? WAVE : 256;
  const long blocks = (pieces + block - 1) / block;
  if (blocks > 0x7fffffffL) return ERR_UNSUPPORTED_SIZE;
#define COMBINE_PIECE(TS_, TX_, PIECE_)                                                                                \
  moe_combine_kernel<TS_, TX_, PIECE_><<<(unsigned)blocks, block, 0, stream>>>(                                        \
      down, ld, place, weights, top, (const TX_*)x, x_ld, (const TS_*)shared, shared_ld, gate, out, d, pieces, tail)
#define COMBINE_LAUNCH(TS_, TX_)                                                                                       \
  do {                                                                                                                 \
    if (fours) COMBINE_PIECE(TS_, TX_, 4);                                                                             \
    else COMBINE_PIECE(TS_, TX_, 1);                                                                                   \
  } while (0)
  if (shared_dtype == DT_F32 && x_dtype == DT_F32) COMBINE_LAUNCH(float, float);
  else if (shared_dtype == DT_F32 && x_dtype == DT_BF16) COMBINE_LAUNCH(float, bf16_t);
  else if (shared_dtype == DT_BF16 && x_dtype == DT_F32) COMBINE_LAUNCH(bf16_t, float);
  else if (shared_dtype == DT_BF16 && x_dtype == DT_BF16) COMBINE_LAUNCH(bf16_t, bf16_t);
  else return ERR_BAD_ARGUMENT;
#undef COMBINE_LAUNCH
#undef COMBINE_PIECE
  RETURN_IF_LAUNCH_FAILED();
  return 0;
}
