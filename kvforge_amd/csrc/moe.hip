// Routed experts: the router's choice per token, and the row-wise steps around the experts'
// matrix products.  Router arithmetic is fp32 throughout.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {
constexpr int MAX_PER_LANE = 8;   // router outputs per lane: up to 512 of them
constexpr int MAX_TOP = 16;

// A wave per token; z gets a bias per output first (null: none).  SCORE_SOFTMAX: s = softmax(z) over all R
// router outputs; SCORE_SIGMOID: s = sigmoid(z) of each by itself; the `top` outputs with the largest
// s + correction (null: none) are chosen (the lowest index among equals), and weighted by their s
// alone, divided (`renorm`) by the sum of the chosen s (+ 1e-20).  SCORE_CHOSEN: the outputs with the
// largest z are chosen, and weighted by the softmax over the chosen z.  The weights are then
// multiplied by `scale`.  sel [N, top], wgt [N, top].
enum { SCORE_SOFTMAX = 0, SCORE_SIGMOID = 1, SCORE_CHOSEN = 2 };
// PER: router outputs a lane holds.  What bounds a token is the chain of sums and maxima over the lanes: a choice
// takes one maximum, its index (one output a lane: from the lanes that hold the maximum) and its score are read
// off the lane.  8 tokens of 34 outputs, 4 choices: 6.7 us with eight outputs a lane and three chains a choice; now
// 5.8 with the plan behind them (moe_choose_plan_kernel).
template <int PER>
__device__ __forceinline__ void choose(const float* __restrict__ zr, const float* __restrict__ bias,
                                       const float* __restrict__ correction, int R, int top, int score, int renorm,
                                       float scale, int& picked, float& weight) {
  const int lane = threadIdx.x % KVF_WAVE;
  float s[PER], c[PER];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + KVF_WAVE * j;
    c[j] = correction && e < R ? correction[e] : 0.f;
    s[j] = e < R ? zr[e] + (bias ? bias[e] : 0.f) : -INFINITY;
    mx = fmaxf(mx, s[j]);
  }
  if (score == SCORE_SIGMOID) {
#pragma unroll
    for (int j = 0; j < PER; ++j) s[j] = 1.f / (1.f + expf(-s[j]));
  } else if (score == SCORE_SOFTMAX) {
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = lane + KVF_WAVE * j;
      s[j] = e < R ? expf(s[j] - mx) : 0.f;
      sum += s[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PER; ++j) s[j] = s[j] / sum;
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + KVF_WAVE * j;
    c[j] = e < R ? s[j] + c[j] : -INFINITY;
  }
  constexpr int NONE = 0x7fffffff;
  float picked_s = 0.f, total = 0.f;   // lane k keeps the k-th choice
  picked = -1;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY, mine = 0.f;
    int at = NONE;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if (c[j] > best) {   // a lane's own candidates come in rising index: '>' keeps the lowest
        best = c[j];
        mine = s[j];
        at = lane + KVF_WAVE * j;
      }
    }
    const float wbest = wave_max(best);
    int cand = best == wbest ? at : NONE;
    if (PER == 1) {
      const unsigned long long who = __ballot(cand != NONE);
      cand = who ? __builtin_ctzll(who) : NONE;
    } else {
#pragma unroll
      for (int o = KVF_WAVE / 2; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, KVF_WAVE));
    }
    // the owner hands over its score and retires the choice
    const float sv = cand == NONE ? 0.f : __shfl(mine, cand % KVF_WAVE, KVF_WAVE);
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + KVF_WAVE * j == cand) c[j] = -INFINITY;
    total += sv;
    if (lane == k) {
      picked_s = sv;
      picked = cand;
    }
  }
  if (score == SCORE_CHOSEN) {   // the first choice has the largest z
    picked_s = lane < top ? expf(picked_s - __shfl(picked_s, 0, KVF_WAVE)) : 0.f;
    total = wave_sum(picked_s);
  }
  weight = (score == SCORE_CHOSEN ? picked_s / total : renorm ? picked_s / (total + 1e-20f) : picked_s) * scale;
}

template <int PER>
__global__ __launch_bounds__(KVF_WAVE) void moe_topk_kernel(const float* __restrict__ z, int z_stride,
                                                            const float* __restrict__ bias,
                                                            const float* __restrict__ correction,
                                                            int* __restrict__ sel, float* __restrict__ wgt,
                                                            int R, int top, int score, int renorm, float scale) {
  const int n = blockIdx.x, lane = threadIdx.x;
  int picked;
  float weight;
  choose<PER>(z + static_cast<size_t>(n) * z_stride, bias, correction, R, top, score, renorm, scale, picked, weight);
  if (lane < top) {
    sel[static_cast<size_t>(n) * top + lane] = picked;
    wgt[static_cast<size_t>(n) * top + lane] = weight;
  }
}

__device__ __forceinline__ float silu(float g) { return g / (1.f + expf(-g)); }
// an expert's (gate, up) pair joined: silu(g) u, or the limited form (GateForm)
__device__ __forceinline__ float joined(const GateForm& f, float g, float u) {
  return f.act == GATE_LIMITED ? limited_pair_exact(g, u, f.limit) : silu(g) * u;
}

// Every expert's gate/up pair for every token is there (one product over all experts, columns
// 2 (e ff + j) and 2 (e ff + j) + 1): act[n, e ff + j] = weight(n, e) * silu(gate) * up where the
// token chose expert e, and an exact zero elsewhere, so that one product with the experts' down
// matrices side by side along K is the weighted sum over the chosen experts.  `weigh_input`: the weight
// belongs to the expert's input, act = silu(w gate) * (w up) (gate and up are linear in it).  `f`: how a
// pair is joined where it is not by silu.
template <typename T>
__global__ void moe_dense_act_kernel(const T* __restrict__ gu, const int* __restrict__ sel,
                                     const float* __restrict__ wgt, T* __restrict__ act, int E, int ff,
                                     int top, int weigh_input, GateForm f, long total) {
  const long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const long cols = static_cast<long>(E) * ff;
  const long n = i / cols;
  const int col = static_cast<int>(i - n * cols), e = col / ff;
  float w = 0.f;
  bool chosen = false;
  for (int k = 0; k < top; ++k)
    if (sel[n * top + k] == e) {
      w = wgt[n * top + k];
      chosen = true;
    }
  float y = 0.f;
  if (chosen) {
    const float g = Elem<T>::load(gu + 2 * i), u = Elem<T>::load(gu + 2 * i + 1);
    y = weigh_input ? joined(f, w * g, w * u) : w * joined(f, g, u);
  }
  Elem<T>::store(act + i, y);
}

// x[n, :] += (sum of the weights of the token's choices at or beyond `first`) * h[n, :]: router
// outputs that stand for "pass the input on".  x fp32, h of type T.
template <typename T>
__global__ __launch_bounds__(256) void moe_identity_kernel(float* __restrict__ x, const T* __restrict__ h,
                                                           const int* __restrict__ sel,
                                                           const float* __restrict__ wgt, int width,
                                                           int top, int first) {
  const int n = blockIdx.x;
  float w = 0.f;
  for (int k = 0; k < top; ++k)
    if (sel[static_cast<size_t>(n) * top + k] >= first) w += wgt[static_cast<size_t>(n) * top + k];
  if (w == 0.f) return;
  float* xr = x + static_cast<size_t>(n) * width;
  const T* hr = h + static_cast<size_t>(n) * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) xr[i] = fmaf(w, Elem<T>::load(hr + i), xr[i]);
}

// ---------------------------------------------------------------------------------------------
// The experts' products over only the rows that chose them (bf16, matrix cores).
//
// moe_plan: the (token, choice) pairs are grouped by expert: where[pair] is the pair's place in
// that order (-1 for a choice that names no expert), order[place] the pair; every expert's rows
// are cut into tiles of up to 2^tile_shift: tiles[t] = (expert | the tile's place among the expert's tiles << 9, first
// place, rows | how many tiles the expert has << 8).  One workgroup; the order of
// an expert's rows among themselves is whatever the atomics give, which no result depends on
// (a row's products do not depend on its neighbours).  What bounds it is one workgroup's chain of trips: choices,
// counters in LDS, sums over the experts, stores.  Up to 8,192 pairs the choices and their places stay in
// registers in between, and a lane adds up no more experts than there are; plan to sum at 4 experts (512 x 1,024)
// and 24 pairs 19.4 us (20.3 with both passes over memory and sums over all 512 places).
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int PLAN_EXPERT_BITS = 9, PLAN_MAX_EXPERTS = 1 << PLAN_EXPERT_BITS, PLAN_ROWS_BITS = 8;
constexpr int PLAN_BATCH = 8;      // choices a thread of the plan has in flight
constexpr int PREFETCH_SETS = 3;   // sets of operand registers in flight in the kernels of few rows
constexpr int DEEP_SETS = 8;       // the same in deep_product
constexpr long EXPERTS_STREAM_BYTES = 32l << 20;   // the eight L2s

__device__ __forceinline__ int tile_expert(const int* tiles, int t) { return tiles[3 * t] & (PLAN_MAX_EXPERTS - 1); }
__device__ __forceinline__ int tile_in_expert(const int* tiles, int t) { return tiles[3 * t] >> PLAN_EXPERT_BITS; }
__device__ __forceinline__ int tile_rows(const int* tiles, int t) { return tiles[3 * t + 2] & ((1 << PLAN_ROWS_BITS) - 1); }
__device__ __forceinline__ int tiles_in_expert(const int* tiles, int t) { return tiles[3 * t + 2] >> PLAN_ROWS_BITS; }

__device__ __forceinline__ uint2 pack4(const f32x4& a) {
  return make_uint2(static_cast<uint32_t>(f32_to_bf16(a[0])) | (static_cast<uint32_t>(f32_to_bf16(a[1])) << 16),
                    static_cast<uint32_t>(f32_to_bf16(a[2])) | (static_cast<uint32_t>(f32_to_bf16(a[3])) << 16));
}

// All threads of the one workgroup; sel in LDS or memory.
__device__ __forceinline__ void plan(const int* sel, int pairs, int E, int* __restrict__ where, int* __restrict__ order,
                                     int* __restrict__ tiles, int* __restrict__ num_tiles, int max_tiles, int tile_shift) {
  __shared__ int cnt[PLAN_MAX_EXPERTS], off[PLAN_MAX_EXPERTS], first_tile[PLAN_MAX_EXPERTS];
  const int tid = threadIdx.x, step = static_cast<int>(blockDim.x);
  const int per = (E + KVF_WAVE - 1) / KVF_WAVE;   // experts a lane of the first wave adds up
  auto tiles_of = [&](int rows) { return (rows + (1 << tile_shift) - 1) >> tile_shift; };
  for (int e = tid; e < per * KVF_WAVE; e += step) cnt[e] = 0;
  // A thread's choices are asked for together: one trip to memory for PLAN_BATCH of them.  One round of
  // them stays in registers up to the end, more are read again.
  int e[PLAN_BATCH], at[PLAN_BATCH];
  const bool once = pairs <= PLAN_BATCH * step;
  auto ask = [&](int p0) {
#pragma unroll
    for (int i = 0; i < PLAN_BATCH; ++i)
      if (i * step < pairs) e[i] = sel[min(p0 + i * step, pairs - 1)];
  };
  auto each = [&](int p0, auto&& go) {
#pragma unroll
    for (int i = 0; i < PLAN_BATCH; ++i)
      if (i * step < pairs && p0 + i * step < pairs) go(p0 + i * step, e[i], at[i]);
  };
  if (tid < pairs) ask(tid);
  __syncthreads();
  for (int p0 = tid; p0 < pairs; p0 += PLAN_BATCH * step) {
    if (p0 != tid) ask(p0);
    each(p0, [&](int p, int expert, int& place) {
      place = expert >= 0 && expert < E ? atomicAdd(&cnt[expert], 1) : -1;
      if (!once) where[p] = place;
    });
  }
  __syncthreads();
  if (tid < KVF_WAVE) {   // where every expert's rows and tiles begin: sums over the lanes before
    int rows = 0, nt = 0;
    for (int i = 0; i < per; ++i) {
      rows += cnt[per * tid + i];
      nt += tiles_of(cnt[per * tid + i]);
    }
    int rows_upto = rows, nt_upto = nt;
#pragma unroll
    for (int o = 1; o < KVF_WAVE; o *= 2) {
      const int r = __shfl_up(rows_upto, o, KVF_WAVE), t = __shfl_up(nt_upto, o, KVF_WAVE);
      if (tid >= o) {
        rows_upto += r;
        nt_upto += t;
      }
    }
    if (tid == KVF_WAVE - 1) *num_tiles = min(nt_upto, max_tiles);
    rows_upto -= rows;
    nt_upto -= nt;
    for (int i = 0; i < per; ++i) {
      off[per * tid + i] = rows_upto;
      first_tile[per * tid + i] = nt_upto;
      rows_upto += cnt[per * tid + i];
      nt_upto += tiles_of(cnt[per * tid + i]);
    }
  }
  __syncthreads();
  if (tid < E && cnt[tid] > 0) {   // an expert's tiles hold about equally many rows, in whole sixteens
    const int c = cnt[tid], nt = tiles_of(c);
    int each_has = c;
    if (nt > 1) each_has = ((c + nt - 1) / nt + 15) / 16 * 16;
    for (int i = 0; i < nt && first_tile[tid] + i < max_tiles; ++i) {
      int* t = tiles + 3 * (first_tile[tid] + i);
      t[0] = tid | i << PLAN_EXPERT_BITS;
      t[1] = off[tid] + i * each_has;
      t[2] = min(each_has, c - i * each_has) | nt << PLAN_ROWS_BITS;
    }
  }
  for (int p0 = tid; p0 < pairs; p0 += PLAN_BATCH * step) {
    if (!once) {
      ask(p0);
#pragma unroll
      for (int i = 0; i < PLAN_BATCH; ++i) at[i] = where[min(p0 + i * step, pairs - 1)];
    }
    each(p0, [&](int p, int expert, int place) {
      const bool named = expert >= 0 && expert < E;
      if (named) order[off[expert] + place] = p;
      if (named || once) where[p] = named ? off[expert] + place : -1;
    });
  }
}

__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ sel, int pairs, int E,
                                                        int* __restrict__ where, int* __restrict__ order,
                                                        int* __restrict__ tiles, int* __restrict__ num_tiles,
                                                        int max_tiles, int tile_shift) {
  plan(sel, pairs, E, where, order, tiles, num_tiles, max_tiles, tile_shift);
}

// The choices of a few tokens, a wave each, and their plan in one kernel: up to CHOOSE_TOKENS tokens a launch
// and a trip of the choices through memory cost more than the waves of one workgroup do (8 tokens of 34 outputs:
// 5.8 us, two kernels of 6.7 and 3.9 before).
constexpr int CHOOSE_TOKENS = 16;
template <int PER>
__global__ __launch_bounds__(CHOOSE_TOKENS * KVF_WAVE) void moe_choose_plan_kernel(
    const float* __restrict__ z, int z_stride, const float* __restrict__ bias, const float* __restrict__ correction,
    int* __restrict__ sel, float* __restrict__ wgt, int n, int R, int top, int score, int renorm, float scale, int E,
    int* __restrict__ where, int* __restrict__ order, int* __restrict__ tiles, int* __restrict__ num_tiles, int max_tiles,
    int tile_shift) {
  __shared__ int chosen[CHOOSE_TOKENS * MAX_TOP];
  const int lane = threadIdx.x % KVF_WAVE, token = threadIdx.x / KVF_WAVE;
  if (token < n) {
    int picked;
    float weight;
    choose<PER>(z + static_cast<size_t>(token) * z_stride, bias, correction, R, top, score, renorm, scale, picked, weight);
    if (lane < top) {
      chosen[token * top + lane] = picked;
      sel[token * top + lane] = picked;
      wgt[token * top + lane] = weight;
    }
  }
  __syncthreads();
  plan(chosen, n * top, E, where, order, tiles, num_tiles, max_tiles, tile_shift);
}

// v_mfma_f32_16x16x32_bf16 computes D[i][j] += sum_k A[i][k] B[j][k]; lane 16 c + r gives row r,
// elements 8c..8c+7 of the step's 32 of either operand, and holds D[4 (l / 16) + v][l % 16].
// A is a tile of the weight (1 KB in lane order, as ``StreamedWeight`` keeps it), B the tile's 16
// rows: a lane ends with four neighbouring output columns of one row.
//
// The kernels of few rows (a decode step): a wave takes 16 rows of one expert and 16 weight rows, so that
// the experts' matrices, which bound it, come in through as many workgroups as there are.  Two ways:
// narrow_product: a step's two fragments are asked for two steps ahead of the matrix instruction that uses them
// (PREFETCH_SETS sets of registers take turns), and lanes without a row ask for none.  deep_product: a wave's own chain
// of trips is what takes the time where there are few workgroups, so eight steps are on their way, and no load is predicated
// (lanes without a row read the last one).  See goes_deep for which is taken.
// STREAMED (see load_16): up to 16 tokens, of whose experts each is read by one tile alone, over layers whose experts take
// more than the L2s.  Four kernels and no branch in one: that was 3 to 10 us slower than either way by itself.
// Plan, up and down (us; tokens, experts, 4 chosen, ff, K; matrices from memory), cached and streamed, both narrow:
//   8, 32, 1,024, 2,048: 51.3, 46.4      13: 70.3, 63.3      5, 32, 2,048, 2,048: 74.8, 67.8      16, 16, 512, 1,024: 22.2, 20.4
template <class Load>
__device__ __forceinline__ f32x4 narrow_product(int S, const Load& load) {
  constexpr int NB = PREFETCH_SETS;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  bf16x8 x[NB], w[NB];
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < S) load(i, x[i], w[i]);
  for (int s = 0; s < S; s += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (s + i < S) {
        if (s + i + NB - 1 < S) load(s + i + NB - 1, x[(i + NB - 1) % NB], w[(i + NB - 1) % NB]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[i], acc, 0, 0, 0);
      }
    }
  }
  return acc;
}
template <class Load>
__device__ __forceinline__ f32x4 deep_product(int S, const Load& load) {
  constexpr int NB = DEEP_SETS;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  bf16x8 x[NB], w[NB];
  if (S < NB) return narrow_product(S, load);
#pragma unroll
  for (int i = 0; i < NB; ++i) load(i, x[i], w[i]);
  int s = 0;
  for (; s + 2 * NB <= S; s += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[i], acc, 0, 0, 0);
      load(s + NB + i, x[i], w[i]);
    }
  }
  const int left = S - s - NB;   // steps not asked for yet, fewer than NB
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[i], acc, 0, 0, 0);
    if (i < left) load(s + NB + i, x[i], w[i]);
  }
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < left) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[i], acc, 0, 0, 0);
  return acc;
}

// moe_up: act[place, :] = silu(gate) * up for the tile's rows with their expert's matrices; the
// weight holds every expert's gate and up rows interleaved (gate_j, up_j neighbours), so a lane's
// four columns are two whole pairs.  Grid (column blocks, tiles).  in_wgt (or null): the choice's weight
// belongs to the expert's input; gate and up are linear in it, so it is multiplied into both sums ahead
// of the activation.
template <bool DEEP, bool STREAMED>
__global__ __launch_bounds__(256) void moe_up_kernel(const bf16_t* __restrict__ x, int ldx, int K,
                                                     const uint4* __restrict__ wt, int S,
                                                     const int* __restrict__ order,
                                                     const int* __restrict__ tiles,
                                                     const int* __restrict__ num_tiles, int top, int ff,
                                                     const float* __restrict__ in_wgt, GateForm f,
                                                     bf16_t* __restrict__ act) {
  const int tile = blockIdx.y;
  if (tile >= *num_tiles) return;
  const int e = tile_expert(tiles, tile), row0 = tiles[3 * tile + 1], rows = tile_rows(tiles, tile);
  const int lane = threadIdx.x % KVF_WAVE, wave = threadIdx.x / KVF_WAVE;
  const int j = lane % 16, c = lane / 16;
  const int groups = ff / 8, g = blockIdx.x * 4 + wave;   // groups of 16 interleaved rows per expert
  if (g >= groups) return;
  const uint4* wbase = wt + (static_cast<size_t>(e) * groups + g) * S * KVF_WAVE + lane;
  const int s_full = K / 32;   // steps whose 32 elements all lie inside a row
  f32x4 acc;
  if constexpr (DEEP) {
    const bf16_t* own = x + static_cast<size_t>(order[row0 + min(j, rows - 1)] / top) * ldx;
    acc = deep_product(S, [&](int s, bf16x8& xs, bf16x8& ws) {
      const bool in = s < s_full || 32 * s + 8 * c + 8 <= K;
      uint4 xf = *reinterpret_cast<const uint4*>(own + (in ? 32 * s + 8 * c : 0));
      if (!in) xf = make_uint4(0u, 0u, 0u, 0u);
      xs = __builtin_bit_cast(bf16x8, xf);
      ws = __builtin_bit_cast(bf16x8, load_16<STREAMED>(wbase + static_cast<size_t>(s) * KVF_WAVE));
    });
  } else {
    const bf16_t* xr = j < rows ? x + static_cast<size_t>(order[row0 + j] / top) * ldx + 8 * c : nullptr;
    acc = narrow_product(S, [&](int s, bf16x8& xs, bf16x8& ws) {
      uint4 xf = make_uint4(0u, 0u, 0u, 0u);
      if (xr && (s < s_full || 32 * s + 8 * c + 8 <= K)) xf = *reinterpret_cast<const uint4*>(xr + 32 * s);
      xs = __builtin_bit_cast(bf16x8, xf);
      ws = __builtin_bit_cast(bf16x8, load_16<STREAMED>(wbase + static_cast<size_t>(s) * KVF_WAVE));
    });
  }
  if (j >= rows) return;
  const float w = in_wgt ? in_wgt[order[row0 + j]] : 1.f;
  const float y0 = joined(f, w * acc[0], w * acc[1]), y1 = joined(f, w * acc[2], w * acc[3]);
  *reinterpret_cast<uint32_t*>(act + static_cast<size_t>(row0 + j) * ff + g * 8 + 2 * c) =
      static_cast<uint32_t>(f32_to_bf16(y0)) | (static_cast<uint32_t>(f32_to_bf16(y1)) << 16);
}

// moe_down: y[place, :] = act[place, :] W_down[expert]^T (bf16, not yet weighted).  The weight
// holds the experts' down matrices side by side along K: expert e owns the steps e ff/32 ...
template <bool DEEP, bool STREAMED>
__global__ __launch_bounds__(256) void moe_down_kernel(const bf16_t* __restrict__ act, int ff,
                                                       const uint4* __restrict__ wt, int S_all,
                                                       const int* __restrict__ tiles,
                                                       const int* __restrict__ num_tiles,
                                                       bf16_t* __restrict__ y, int hidden) {
  const int tile = blockIdx.y;
  if (tile >= *num_tiles) return;
  const int e = tile_expert(tiles, tile), row0 = tiles[3 * tile + 1], rows = tile_rows(tiles, tile);
  const int lane = threadIdx.x % KVF_WAVE, wave = threadIdx.x / KVF_WAVE;
  const int j = lane % 16, c = lane / 16;
  const int groups = (hidden + 15) / 16, g = blockIdx.x * 4 + wave;
  if (g >= groups) return;
  const int S = ff / 32;
  const uint4* wbase = wt + (static_cast<size_t>(g) * S_all + static_cast<size_t>(e) * S) * KVF_WAVE + lane;
  f32x4 acc;
  if constexpr (DEEP) {
    const bf16_t* own = act + static_cast<size_t>(row0 + min(j, rows - 1)) * ff + 8 * c;
    acc = deep_product(S, [&](int s, bf16x8& xs, bf16x8& ws) {
      xs = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(own + 32 * s));
      ws = __builtin_bit_cast(bf16x8, load_16<STREAMED>(wbase + static_cast<size_t>(s) * KVF_WAVE));
    });
  } else {
    const bf16_t* ar = j < rows ? act + static_cast<size_t>(row0 + j) * ff + 8 * c : nullptr;
    acc = narrow_product(S, [&](int s, bf16x8& xs, bf16x8& ws) {
      uint4 af = make_uint4(0u, 0u, 0u, 0u);
      if (ar) af = *reinterpret_cast<const uint4*>(ar + 32 * s);
      xs = __builtin_bit_cast(bf16x8, af);
      ws = __builtin_bit_cast(bf16x8, load_16<STREAMED>(wbase + static_cast<size_t>(s) * KVF_WAVE));
    });
  }
  const int col = g * 16 + 4 * c;
  if (j >= rows || col >= hidden) return;   // hidden is a multiple of 8
  *reinterpret_cast<uint2*>(y + static_cast<size_t>(row0 + j) * hidden + col) = pack4(acc);
}

// ---------------------------------------------------------------------------------------------
// The same two products for more rows: tiles of up to 128 rows of one expert against 128 of its weight
// rows, four waves of 32 weight rows each.
//
// What bounds it: the experts' matrices come from memory once (32 experts of 2,048 x 1,024: 403 MB, 80 us
// at the 5 TB/s of a large copy), the other tiles of an expert find them in their XCD's L2 (see
// wide_item).  A wave needs its own weight fragments only, so they go straight into registers; the rows, which
// all four waves need, are gathered through LDS, 64 elements of K at a time in two buffers.  Weights are asked for
// two passes ahead, into the registers of those just used, rows three, and each of these loads stands between
// two products.  Rows past an expert's last are read as its last and not stored; tiles of up to 96, 64 and 32
// rows leave the other matrix instructions out.
//
// Up and down together with plan and sum, 32 experts, 4 chosen, 2,048 wide.  2,047 tokens: 304 us at ff 2,048, 171 at
// 1,024 (333 and 173 with an expert's tiles one behind the other, where both came from memory anew: 1.26 GB read
// instead of 0.63; 307 and 170 with that mended alone).  180 tokens at 2,048: 148 (161), 5.4 TB/s.  On the way: 256 weight rows
// a workgroup in 512 registers a lane 360 / 228; two workgroups a compute unit instead of three the same.
constexpr int WIDE_SHIFT = 7, WIDE_ROWS = 1 << WIDE_SHIFT, WIDE_GW = 2;

// What a workgroup takes: tile and block of columns.  Workgroups go to the eight XCDs in turn, and each
// XCD gets an unbroken eighth of the (expert, block, tile) triples: the tiles of an expert that read the same weight rows
// start together and walk K side by side, so the L2 (4 MB, a fifth of an expert's matrices at ff 2,048) brings those in
// once, and the expert's rows stay there over its blocks.
__device__ __forceinline__ bool wide_item(const int* tiles, int num_tiles, int blocks, int& tile, int& block) {
  const int total = num_tiles * blocks, share = (total + 7) / 8, at = blockIdx.x / 8;
  const int item = static_cast<int>(blockIdx.x % 8) * share + at;
  if (at >= share || item >= total) return false;
  const int some = item / blocks;                    // a tile of the item's expert
  const int first = some - tile_in_expert(tiles, some), count = tiles_in_expert(tiles, some);
  const int in = item - first * blocks;
  block = in / count;
  tile = first + in % count;
  return true;
}
template <int N> struct Rows { static constexpr int value = N; };
template <class F> __device__ __forceinline__ void wide_rows(int rows, const F& go) {
  if (rows > 96) go(Rows<8>{});
  else if (rows > 64) go(Rows<6>{});
  else if (rows > 32) go(Rows<4>{});
  else go(Rows<2>{});
}

// For the scheduler, N times: a row fragment's products, the read of another fragment, an instruction of a third kind.
template <int N, int MASK>
__device__ __forceinline__ void beside_products() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, WIDE_GW, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(MASK, 1, 0);
  }
}

template <int RT> struct WideAcc { f32x4 v[RT][WIDE_GW]; };

// row_of(r): where row r of the tile starts (r below 16 RT).  wbase, goff: the
// fragment of group g and step s begins at wbase + goff[g] + s * KVF_WAVE (the same for the whole wave).
template <int RT, class RowOf>
__device__ __forceinline__ void wide_product(const RowOf& row_of, int K, const uint4* __restrict__ wbase,
                                             const size_t (&goff)[WIDE_GW], int S, uint4* lds, WideAcc<RT>& acc) {
  constexpr int PASSES = RT / 2;                     // 32 rows of 128 bytes are staged at a time
  const int tid = threadIdx.x, lane = tid % KVF_WAVE;
  const int ch = tid % 8, sr = tid / 8;              // staged: the 8 elements at 8 ch of rows sr + 32 p
  const bf16_t* src[PASSES];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) src[p] = row_of(sr + 32 * p) + 8 * ch;
  // A fragment (16 rows x 32 elements) is 64 pieces of 16 bytes.  Piece (row j, c) lies at 4 j + c, c turned
  // over for rows 8..15: a 16-byte access serves lanes 0-3, 12-15 and 20-27 together, then 4-11, 16-19 and
  // 28-31, and either sixteen then fall on all banks, read (row lane % 16) or written (row lane / 8).
  auto place = [](int j, int c) { return 4 * j + (c ^ (j >= 8 ? 3 : 0)); };
  const int put_at = ((sr / 16) * 2 + ch / 4) * KVF_WAVE + place(sr % 16, ch % 4);
  const int get_at = place(lane % 16, lane / 16);
  // No load stands under a condition: where paths with and without one meet, the compiler waits for the
  // newest loads before the first product, and nothing is ahead of anything any more.  WHOLE: the pass lies inside K.
  using Stage = uint4[PASSES];
  auto fetch = [&](auto whole, int it, Stage& stage) {
    const int k = decltype(whole)::value ? 64 * it : min(64 * it, K - 8 - 8 * ch);   // K is a multiple of 8: past it a row's last 8, see put
#pragma unroll
    for (int p = 0; p < PASSES; ++p) stage[p] = *reinterpret_cast<const uint4*>(src[p] + k);
  };
  auto put = [&](auto whole, int it, const Stage& stage) {
    const bool in = decltype(whole)::value || 64 * it + 8 * ch < K;
    uint4* to = lds + (it & 1) * RT * 2 * KVF_WAVE + put_at;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) to[p * 4 * KVF_WAVE] = in ? stage[p] : make_uint4(0u, 0u, 0u, 0u);
  };
  using Weights = uint4[2][WIDE_GW];
  auto weights = [&](int it, int h, Weights& w) {
#pragma unroll
    for (int g = 0; g < WIDE_GW; ++g) w[h][g] = (wbase + goff[g] + static_cast<size_t>(min(2 * it + h, S - 1)) * KVF_WAVE)[lane];
  };
  auto product = [&](int it, int h, const Weights& w) {
    const uint4* frag = lds + (it & 1) * RT * 2 * KVF_WAVE + get_at;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const bf16x8 x = __builtin_bit_cast(bf16x8, frag[(2 * r + h) * KVF_WAVE]);
#pragma unroll
      for (int g = 0; g < WIDE_GW; ++g)
        acc.v[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[h][g]), x, acc.v[r][g], 0, 0, 0);
    }
  };
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int g = 0; g < WIDE_GW; ++g) acc.v[r][g] = f32x4{0.f, 0.f, 0.f, 0.f};
  // A pass: rows of the next go from registers to LDS, those of the third from here are asked for, and so are the
  // weights of the one after the next as soon as these have been used.
  auto pass = [&](auto whole, int it, Weights& w, Stage& stage) {
    __syncthreads();                                 // this pass's rows are there, the other buffer is free
    put(whole, it + 1, stage);
    fetch(whole, it + 3, stage);
    product(it, 0, w);
    weights(it + 2, 0, w);
    product(it, 1, w);
    weights(it + 2, 1, w);
    // row fragments two ahead of the one in use, then everything else one by one between the products
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    beside_products<PASSES, 0x200>();
    beside_products<RT - PASSES, 0x020>();
    beside_products<RT - 2, 0x020>();
    __builtin_amdgcn_sched_group_barrier(0x008, 2 * WIDE_GW, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::true_type WHOLE{};
  constexpr std::false_type PART{};
  Weights w0, w1;
  Stage s0, s1;
  fetch(PART, 0, s0);
  fetch(PART, 1, s1);
  weights(0, 0, w0);
  weights(0, 1, w0);
  weights(1, 0, w1);
  weights(1, 1, w1);
  put(PART, 0, s0);
  fetch(PART, 2, s0);
  const int passes = S / 2;                          // whole ones; an odd step is left over
  int it = 0;
#pragma unroll 1
  for (; 64 * (it + 5) <= K; it += 2) {
    pass(WHOLE, it, w0, s1);
    pass(WHOLE, it + 1, w1, s0);
  }
#pragma unroll 1
  for (; it < passes; it += 2) {
    pass(PART, it, w0, s1);
    if (it + 1 < passes) pass(PART, it + 1, w1, s0);
  }
  if (S % 2) {
    __syncthreads();
    if (passes % 2) product(passes, 0, w1);
    else product(passes, 0, w0);
  }
}

// A lane holds four neighbouring weight rows' products of row lane % 16 of every sub-tile.
template <int RT>
__device__ __forceinline__ void wide_up_tile(const bf16_t* __restrict__ x, int ldx, int K, const uint4* __restrict__ wt,
                                             int S, const int* __restrict__ order, int e, int row0, int rows, int block,
                                             int top, int ff, const float* __restrict__ in_wgt, const GateForm& f,
                                             bf16_t* __restrict__ act, uint4* lds) {
  const int lane = threadIdx.x % KVF_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVF_WAVE);
  const int j = lane % 16, c = lane / 16;
  const int groups = ff / 8, g_first = (block * 4 + wave) * WIDE_GW;
  const int g_read = min(g_first, groups - WIDE_GW);   // groups come in whole fours: all of a wave's or none
  size_t goff[WIDE_GW];
#pragma unroll
  for (int g = 0; g < WIDE_GW; ++g) goff[g] = static_cast<size_t>(g) * S * KVF_WAVE;
  WideAcc<RT> acc;
  wide_product<RT>([&](int r) { return x + static_cast<size_t>(order[row0 + min(r, rows - 1)] / top) * ldx; }, K,
                   wt + (static_cast<size_t>(e) * groups + g_read) * S * KVF_WAVE, goff, S, lds, acc);
  if (g_first >= groups) return;
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = 16 * r + j;
    if (row >= rows) continue;
    bf16_t* out = act + static_cast<size_t>(row0 + row) * ff;
    const float w = in_wgt ? in_wgt[order[row0 + row]] : 1.f;
#pragma unroll
    for (int g = 0; g < WIDE_GW; ++g) {
      const f32x4 a = acc.v[r][g];
      const float y0 = joined(f, w * a[0], w * a[1]), y1 = joined(f, w * a[2], w * a[3]);
      *reinterpret_cast<uint32_t*>(out + (g_first + g) * 8 + 2 * c) =
          static_cast<uint32_t>(f32_to_bf16(y0)) | (static_cast<uint32_t>(f32_to_bf16(y1)) << 16);
    }
  }
}

__global__ __launch_bounds__(256, 3) void moe_up_wide_kernel(const bf16_t* __restrict__ x, int ldx, int K,
                                                             const uint4* __restrict__ wt, int S,
                                                             const int* __restrict__ order,
                                                             const int* __restrict__ tiles,
                                                             const int* __restrict__ num_tiles, int top, int ff,
                                                             const float* __restrict__ in_wgt, GateForm f,
                                                             bf16_t* __restrict__ act) {
  __shared__ uint4 lds[2 * WIDE_ROWS * 8];
  int tile, block;
  if (!wide_item(tiles, *num_tiles, (ff / 8 + 4 * WIDE_GW - 1) / (4 * WIDE_GW), tile, block)) return;
  const int e = tile_expert(tiles, tile), row0 = tiles[3 * tile + 1], rows = tile_rows(tiles, tile);
  auto go = [&](auto rt) { wide_up_tile<decltype(rt)::value>(x, ldx, K, wt, S, order, e, row0, rows, block, top, ff, in_wgt, f, act, lds); };
  wide_rows(rows, go);
}

template <int RT>
__device__ __forceinline__ void wide_down_tile(const bf16_t* __restrict__ act, int ff, const uint4* __restrict__ wt,
                                               int S_all, int e, int row0, int rows, int block,
                                               bf16_t* __restrict__ y, int hidden,
                                               uint4* lds) {
  const int lane = threadIdx.x % KVF_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVF_WAVE);
  const int j = lane % 16, c = lane / 16;
  const int groups = (hidden + 15) / 16, g_first = (block * 4 + wave) * WIDE_GW, S = ff / 32;
  size_t goff[WIDE_GW];   // a group past the last is read as the last and not stored
#pragma unroll
  for (int g = 0; g < WIDE_GW; ++g) goff[g] = static_cast<size_t>(min(g_first + g, groups - 1)) * S_all * KVF_WAVE;
  WideAcc<RT> acc;
  wide_product<RT>([&](int r) { return act + static_cast<size_t>(row0 + min(r, rows - 1)) * ff; }, ff,
                   wt + static_cast<size_t>(e) * S * KVF_WAVE, goff, S, lds, acc);
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = 16 * r + j;
    if (row >= rows) continue;
    bf16_t* out = y + static_cast<size_t>(row0 + row) * hidden;
#pragma unroll
    for (int g = 0; g < WIDE_GW; ++g) {
      const int col = (g_first + g) * 16 + 4 * c;
      if (col >= hidden) continue;                     // hidden is a multiple of 8
      *reinterpret_cast<uint2*>(out + col) = pack4(acc.v[r][g]);
    }
  }
}

__global__ __launch_bounds__(256, 3) void moe_down_wide_kernel(const bf16_t* __restrict__ act, int ff,
                                                               const uint4* __restrict__ wt, int S_all,
                                                               const int* __restrict__ tiles,
                                                               const int* __restrict__ num_tiles,
                                                               bf16_t* __restrict__ y, int hidden) {
  __shared__ uint4 lds[2 * WIDE_ROWS * 8];
  int tile, block;
  if (!wide_item(tiles, *num_tiles, ((hidden + 15) / 16 + 4 * WIDE_GW - 1) / (4 * WIDE_GW), tile, block)) return;
  const int e = tile_expert(tiles, tile), row0 = tiles[3 * tile + 1], rows = tile_rows(tiles, tile);
  auto go = [&](auto rt) { wide_down_tile<decltype(rt)::value>(act, ff, wt, S_all, e, row0, rows, block, y, hidden, lds); };
  wide_rows(rows, go);
}

// x[n, :] += sum over the token's choices, in their order, of weight * (the expert's row of y, or
// the token's own input h for a choice that names no expert): fp32 sums into the fp32 stream.
// A thread takes eight neighbouring elements (hidden is a multiple of 8 here): per choice one
// 16-byte load, the choice itself being the same for the whole workgroup.  wgt null: weights of one
// (they went into the experts' inputs).  `fresh`: x is written, not added to.
__device__ __forceinline__ void load8_any(const bf16_t* p, float (&v)[8]) { load8(p, v); }
__device__ __forceinline__ void load8_any(const float* p, float (&v)[8]) { load8(p, v); }

template <typename T>
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ x, const bf16_t* __restrict__ y,
                                                          const T* __restrict__ h, const int* __restrict__ sel,
                                                          const float* __restrict__ wgt,
                                                          const int* __restrict__ where, int hidden, int top,
                                                          int E, int fresh) {
  const int n = blockIdx.x;
  float* xr = x + static_cast<size_t>(n) * hidden;
  const T* hr = h + static_cast<size_t>(n) * hidden;
  for (int i = 8 * threadIdx.x; i < hidden; i += 8 * blockDim.x) {
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < top; ++k) {
      const int p = n * top + k, e = sel[p];
      const float w = wgt ? wgt[p] : 1.f;
      float v[8];
      if (e >= E) load8_any(hr + i, v);
      else if (e >= 0) load8(y + static_cast<size_t>(where[p]) * hidden + i, v);
      else continue;
#pragma unroll
      for (int u = 0; u < 8; ++u) sum[u] = fmaf(w, v[u], sum[u]);
    }
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (!fresh) {
      a = *reinterpret_cast<const float4*>(xr + i);
      b = *reinterpret_cast<const float4*>(xr + i + 4);
    }
    a.x += sum[0]; a.y += sum[1]; a.z += sum[2]; a.w += sum[3];
    b.x += sum[4]; b.y += sum[5]; b.z += sum[6]; b.w += sum[7];
    *reinterpret_cast<float4*>(xr + i) = a;
    *reinterpret_cast<float4*>(xr + i + 4) = b;
  }
}
// A choice that a table makes: token id t uses the experts table[t, 0 .. top-1] (a row's entries
// differ), each with weight 1 / top.  An id outside the table, or an entry that names no expert,
// gives the pair (expert 0, weight 0): such a token adds nothing.
__global__ void moe_table_kernel(const int* __restrict__ tokens, const int* __restrict__ table, int* __restrict__ sel,
                                 float* __restrict__ wgt, int n, int vocab, int top, int E) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * top) return;
  const int t = tokens[i / top];
  const int e = t >= 0 && t < vocab ? table[static_cast<size_t>(t) * top + i % top] : -1;
  const bool ok = e >= 0 && e < E;
  sel[i] = ok ? e : 0;
  wgt[i] = ok ? 1.f / static_cast<float>(top) : 0.f;
}
}  // namespace

static bool form_ok(int act, float limit) { return act == 0 || (act == GATE_LIMITED && limit > 0.f); }

KVF_EXPORT int kvf_moe_topk(const float* z, int z_stride, const float* bias, const float* correction, int* sel,
                            float* wgt, int n, int R, int top, int score, int renorm, float scale, hipStream_t s) {
  if (n <= 0) return 0;
  if (score < SCORE_SOFTMAX || score > SCORE_CHOSEN || (score == SCORE_CHOSEN && correction) ||
      R <= 0 || R > MAX_PER_LANE * KVF_WAVE || top <= 0 || top > MAX_TOP || top > R)
    return static_cast<int>(hipErrorInvalidValue);
#define GO(PER)                                                                                                    \
  hipLaunchKernelGGL(moe_topk_kernel<PER>, dim3(n), dim3(KVF_WAVE), 0, s, z, z_stride, bias, correction, sel, wgt, R, \
                     top, score, renorm, scale)
  if (R <= KVF_WAVE) GO(1);
  else if (R <= 2 * KVF_WAVE) GO(2);
  else GO(MAX_PER_LANE);
#undef GO
  return kvf_last_error();
}

KVF_EXPORT int kvf_moe_table(const int* tokens, const int* table, int* sel, float* wgt, int n, int vocab, int top,
                             int E, hipStream_t s) {
  if (n <= 0) return 0;
  if (vocab <= 0 || top <= 0 || top > MAX_TOP || E <= 0) return static_cast<int>(hipErrorInvalidValue);
  hipLaunchKernelGGL(moe_table_kernel, dim3((n * top + 255) / 256), dim3(256), 0, s, tokens, table, sel, wgt, n,
                     vocab, top, E);
  return kvf_last_error();
}

KVF_EXPORT int kvf_moe_dense_act(int dtype, const void* gu, const int* sel, const float* wgt, void* act,
                                 int n, int E, int ff, int top, int weigh_input, int form, float limit, hipStream_t s) {
  const long total = static_cast<long>(n) * E * ff;
  if (total <= 0) return 0;
  if (!form_ok(form, limit)) return static_cast<int>(hipErrorInvalidValue);
  const GateForm f{form, limit, 1.f};
  const dim3 grid(static_cast<unsigned>((total + 255) / 256));
  if (dtype == 0)
    hipLaunchKernelGGL(moe_dense_act_kernel<float>, grid, dim3(256), 0, s, static_cast<const float*>(gu), sel,
                       wgt, static_cast<float*>(act), E, ff, top, weigh_input, f, total);
  else if (dtype == 1)
    hipLaunchKernelGGL(moe_dense_act_kernel<bf16_t>, grid, dim3(256), 0, s, static_cast<const bf16_t*>(gu), sel,
                       wgt, static_cast<bf16_t*>(act), E, ff, top, weigh_input, f, total);
  else
    return static_cast<int>(hipErrorInvalidValue);
  return kvf_last_error();
}

KVF_EXPORT int kvf_moe_identity(int dtype, float* x, const void* h, const int* sel, const float* wgt, int n,
                                int width, int top, int first, hipStream_t s) {
  if (n <= 0) return 0;
  if (dtype == 0)
    hipLaunchKernelGGL(moe_identity_kernel<float>, dim3(n), dim3(256), 0, s, x, static_cast<const float*>(h),
                       sel, wgt, width, top, first);
  else if (dtype == 1)
    hipLaunchKernelGGL(moe_identity_kernel<bf16_t>, dim3(n), dim3(256), 0, s, x, static_cast<const bf16_t*>(h),
                       sel, wgt, width, top, first);
  else
    return static_cast<int>(hipErrorInvalidValue);
  return kvf_last_error();
}

// Whether kvf_moe_grouped takes the kernels of more rows.  Those of few rows bring an expert's 6 ff K bytes in anew
// for every tile of 16 rows, in all about pairs / 16 + E / 2 tiles, at 7 TB/s where the matrices lie in the caches;
// the others walk along K and ff in passes of 64 elements, 0.7 us each however few workgroups there are.  The
// line is where the first takes longer than the second,
//   (pairs / 16 + E / 2) 6 ff K / 7 TB/s > (K + ff) / 64 * 0.7 us, fitted: pairs / 16 + E / 2 >= 15,500 (1 / ff + 1 / K),
// and six rows an expert, for below that either is bound by the matrices' way from memory.  Plan to sum, us, few
// against more (experts, ff, K):
//   4, 512, 1,024: 64 rows an expert 26 / 31, 192 41 / 35       8, 1,024, 1,024: 40 rows 36 / 42, 64 50 / 46
//   8, 3,584, 2,048: 12 rows 92 / 100, 20 108 / 101             16, 512, 1,024: 32 rows 34 / 35, 48 42 / 37
//   32, 1,024, 2,048: 6 rows 89 / 83, 32 163 / 87               64, 256, 1,024: 6 rows 33 / 36, 20 45 / 39
// over 19 shapes and 2 to 512 rows an expert at most 10% off the better one.  (Six rows an expert alone sent the few
// and small experts' steps to the wrong side, up to 33% slower.)  Pairs that name no expert are counted like
// the others: the device alone knows them, and a router with such outputs changes sides that much early.
KVF_EXPORT int kvf_moe_grouped_many_rows(int pairs, int E, int ff, int K) {
  return pairs >= 6ll * E && (pairs + 8ll * E) * ff * K >= 248000ll * (ff + K);
}

// kvf_moe_topk of up to CHOOSE_TOKENS tokens together with the plan of kvf_moe_grouped, which is then called with
// `planned`; arguments as there.
KVF_EXPORT int kvf_moe_topk_plan(const float* z, int z_stride, const float* bias, const float* correction, int* sel,
                                 float* wgt, int n, int R, int top, int score, int renorm, float scale, int E, int ff, int K,
                                 int* where, int* order, int* tiles, int* num_tiles, int max_tiles, hipStream_t s) {
  if (n <= 0) return 0;
  const int pairs = n * top;
  if (n > CHOOSE_TOKENS || score < SCORE_SOFTMAX || score > SCORE_CHOSEN || (score == SCORE_CHOSEN && correction) ||
      R <= 0 || R > MAX_PER_LANE * KVF_WAVE || top <= 0 || top > MAX_TOP || top > R || E <= 0 || E > PLAN_MAX_EXPERTS ||
      max_tiles < (pairs + 15) / 16 + E)
    return static_cast<int>(hipErrorInvalidValue);
  const bool many = kvf_moe_grouped_many_rows(pairs, E, ff, K) != 0;
  // the plan has a thread for every expert
  const int threads = n * KVF_WAVE > E ? n * KVF_WAVE : (E + KVF_WAVE - 1) / KVF_WAVE * KVF_WAVE;
#define GO(PER)                                                                                                      \
  hipLaunchKernelGGL(moe_choose_plan_kernel<PER>, dim3(1), dim3(threads), 0, s, z, z_stride, bias, correction, sel, wgt, n, \
                     R, top, score, renorm, scale, E, where, order, tiles, num_tiles, max_tiles, many ? WIDE_SHIFT : 4)
  if (R <= KVF_WAVE) GO(1);
  else if (R <= 2 * KVF_WAVE) GO(2);
  else GO(MAX_PER_LANE);
#undef GO
  return kvf_last_error();
}

// Whether one of the kernels of few rows that can have so many workgroups takes deep_product.  What was measured over 13 layers
// (8 to 128 experts, ff 256 to 3,584, K 1,024 to 4,096) and 1 to 41 tokens, each kernel by itself, narrow less deep in us:
// up to two workgroups a compute unit (256 of them) faster or the same (0 to 18: up of 32 experts of 1,024 x 2,048, one token 8.3, four
// 3.0; down of 8 of 3,584 x 2,048, ten tokens 11.7); from there to four either way, as few of the compute units have a third
// one to wait for (5 tokens of the first -3.5, 8 of them 0.8; 4 of the second's up -2.7, 10 of them 3.0); beyond that faster
// again or the same (down of the first at 13 tokens 0.8, up of 128 of 768 x 2,048, 13 tokens 3.6; worst -1.8 of 95).
// Whole layers, deep up to 384 workgroups of the larger kernel / this: 4 tokens, 32 of 1,024 x 2,048 39.9 / 35.3; 5 tokens, 32 of
// 2,048 x 2,048 64.7 / 63.3; 8 tokens, 8 of 3,584 x 2,048 76.6 / 66.0; of 168 none slower by more than runs differ (1.4%).
static bool goes_deep(long blocks) { return blocks <= 512 || blocks > 1024; }

// The routed experts of a bf16 step without the rows that did not choose them.  x [n, K] (row
// stride ldx), w_gate_up / w_down: the tiled forms of [E 2 ff, K] (gate and up rows interleaved)
// and [K, E ff]; sel / wgt [n, top]; scratch: where, order [n top], tiles [3 max_tiles],
// num_tiles [1], act [n top, ff], y [n top, K].  Needs K % 8 == 0 and ff % 32 == 0.  The outputs' rows stay in y, which
// kvf_moe_combine adds up.  weigh_input: the weights go into the experts' inputs instead of the sum over their outputs.  form, limit: how an expert's pairs are joined (GateForm's act 0 or 2).  many_rows: below
// 0, or which kernels are taken whatever the sizes (0: those of few rows, else those of more).  planned: where,
// order, tiles and num_tiles hold the plan already (kvf_moe_topk_plan).  cached: the matrices are not to go past the caches, whatever
// their size.
KVF_EXPORT int kvf_moe_grouped(const void* x, int ldx, int n, int K, int E, int ff, int top,
                               const void* w_gate_up, const void* w_down, const int* sel, const float* wgt,
                               int* where, int* order, int* tiles, int* num_tiles, int max_tiles, void* act,
                               void* y, int weigh_input, int form, float limit,
                               int many_rows, int planned, int cached, hipStream_t s) {
  if (n <= 0) return 0;
  const int pairs = n * top;
  const bool many = many_rows < 0 ? kvf_moe_grouped_many_rows(pairs, E, ff, K) != 0 : many_rows != 0;
  const GateForm f{form, limit, 1.f};
  if (!form_ok(form, limit) || E <= 0 || E > PLAN_MAX_EXPERTS || K % 8 != 0 || ff % 32 != 0 || ldx % 8 != 0 || max_tiles > 65535 ||
      max_tiles < (pairs + 15) / 16 + E)
    return static_cast<int>(hipErrorInvalidValue);
  if (!planned)
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(1024), 0, s, sel, pairs, E, where, order, tiles, num_tiles,
                       max_tiles, many ? WIDE_SHIFT : 4);
  const int S = (K + 31) / 32, up_groups = ff / 8, down_groups = (K + 15) / 16;
  const bf16_t* xb = static_cast<const bf16_t*>(x);
  const uint4 *up = static_cast<const uint4*>(w_gate_up), *down = static_cast<const uint4*>(w_down);
  const float* in_wgt = weigh_input ? wgt : nullptr;
  bf16_t *a = static_cast<bf16_t*>(act), *out = static_cast<bf16_t*>(y);
  const int gw = many ? 4 * WIDE_GW : 4;   // groups a workgroup takes
  const unsigned up_blocks = (up_groups + gw - 1) / gw, down_blocks = (down_groups + gw - 1) / gw;
  if (many) {   // (tile, block) pairs in one dimension, whole eighths of them
    const unsigned most = (pairs + WIDE_ROWS - 1) / WIDE_ROWS + E;
    hipLaunchKernelGGL(moe_up_wide_kernel, dim3((up_blocks * most + 7) / 8 * 8), dim3(256), 0, s, xb, ldx, K, up, S, order,
                       tiles, num_tiles, top, ff, in_wgt, f, a);
    hipLaunchKernelGGL(moe_down_wide_kernel, dim3((down_blocks * most + 7) / 8 * 8), dim3(256), 0, s, a, ff, down,
                       E * (ff / 32), tiles, num_tiles, out, K);
  } else {
    const bool streamed = n <= 16 && !cached && 6l * E * ff * K >= EXPERTS_STREAM_BYTES;
    // (up to 16 tokens make one tile of every expert they choose)
    const long most = std::min(pairs, n <= 16 ? E : pairs / 16 + E);
    const auto go = [&](auto st) {
      constexpr bool ST = decltype(st)::value;
      const auto up_as = [&](auto deep) {
        hipLaunchKernelGGL((moe_up_kernel<decltype(deep)::value, ST>), dim3(up_blocks, max_tiles), dim3(256), 0, s, xb, ldx, K, up, S,
                           order, tiles, num_tiles, top, ff, in_wgt, f, a);
      };
      const auto down_as = [&](auto deep) {
        hipLaunchKernelGGL((moe_down_kernel<decltype(deep)::value, ST>), dim3(down_blocks, max_tiles), dim3(256), 0, s, a, ff, down,
                           E * (ff / 32), tiles, num_tiles, out, K);
      };
      if (goes_deep(most * up_blocks)) up_as(Flag<true>{});
      else up_as(Flag<false>{});
      if (goes_deep(most * down_blocks)) down_as(Flag<true>{});
      else down_as(Flag<false>{});
    };
    if (streamed) go(Flag<true>{});
    else go(Flag<false>{});
  }
  return kvf_last_error();
}

// The sum over the choices behind kvf_moe_grouped, arguments as there: x [n, K] is the residual stream; wgt null: the weights went
// into the experts' inputs.
KVF_EXPORT int kvf_moe_combine(float* x, const void* y, const void* h, const int* sel, const float* wgt, const int* where, int n,
                               int K, int top, int E, int fresh, hipStream_t s) {
  if (n <= 0) return 0;
  if (K <= 0 || K % 8 != 0 || top <= 0 || top > MAX_TOP || E <= 0) return static_cast<int>(hipErrorInvalidValue);
  hipLaunchKernelGGL(moe_combine_kernel<bf16_t>, dim3(n), dim3(256), 0, s, x, static_cast<const bf16_t*>(y),
                     static_cast<const bf16_t*>(h), sel, wgt, where, K, top, E, fresh);
  return kvf_last_error();
}
