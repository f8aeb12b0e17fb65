// Products of many rows: C = A * W^T for bf16 rows and bf16 weights in tiles (see the head of gemm_bf16.hip), fp32 sums.
// Two kernels over the walk of tile_walk.h: plain and gated products (gemm_tile_kernel), and the fused q/k/v projection with
// rotary and the cache write in its epilogue (qkv_tile_kernel, RopeEpi).
//
// Sums run along K in steps of 32 on one accumulator, and are rounded to bf16 before they are rotated or joined, as a stored product
// is.  The library's product does the same at most sizes, to the bit; it cuts K at some, where 3 to 7 in 100,000 of the result turn a rounding: of 713 sizes of
// plain and gated products that were compared, of 66 to 2,048 rows, at three (1,771 rows of 28,672 columns), of 306 of the fused projection at 14
// (65 to 128 rows).
#include <type_traits>

#include "tile_walk.h"

namespace {
constexpr int MAX_ROT = 128;

// How far the tiles of one band of rows go before the next column: tiles that run at the same time share rows and weights in L2.
constexpr int BAND = 4;
__device__ __forceinline__ void place_of(int item, int tm, int tn, int& row_tile, int& col_tile) {
  const int band = item / (BAND * tn), in = item - band * BAND * tn, rows = min(BAND, tm - band * BAND);
  row_tile = band * BAND + in % rows;
  col_tile = in / rows;
}

// What a product's tiles are read from: rows and weights of the tile `item`, then of the one `step` behind it, up to `last`.
struct Product {
  const bf16_t* A;
  const bf16_t* W;
  int M, N, K, lda, tm, tn, last, step, row_item, weight_item;
  template <class W_> __device__ __forceinline__ void rows(W_& walk) {
    int row_tile, col_tile;
    place_of(row_item, tm, tn, row_tile, col_tile);
    const int m0 = row_tile * W_::BM;
    walk.aim_rows(reinterpret_cast<const char*>(A + static_cast<size_t>(m0) * lda),
                  [&](int r) { return static_cast<uint32_t>(min(r, M - 1 - m0)) * lda * 2; }, K / 32);
    if (row_item + step < last) row_item += step;
  }
  template <class W_> __device__ __forceinline__ void weights(W_& walk) {
    int row_tile, col_tile;
    place_of(weight_item, tm, tn, row_tile, col_tile);
    const int g0 = col_tile * W_::WC, S = K / 32, groups = (N + 15) / 16;
    walk.aim_weights(reinterpret_cast<const char*>(W) + static_cast<size_t>(g0) * S * 1024,
                     [&](int g) { return static_cast<uint32_t>(min(g, groups - 1 - g0)) * S * 1024; }, S);
    if (weight_item + step < last) weight_item += step;
  }
};

// An unbroken eighth of `total` tiles for every XCD (workgroups go to the eight of them in turn): the workgroup's first and
// the end of its XCD's.
__device__ __forceinline__ bool share_of(int total, int& first, int& last) {
  const int share = (total + 7) / 8, begin = static_cast<int>(blockIdx.x % 8) * share;
  first = begin + static_cast<int>(blockIdx.x / 8);
  last = min(total, begin + share);
  return first < last;
}

// What becomes of a sum: stored as bf16 or fp32, or neighbouring columns are (gate, up) pairs (GateForm, with fp32 biases by
// pair or null) and their join is stored as bf16; SILU_PAIRS: joined by silu, without biases and scale.
enum Kind { STORE_BF16 = 0, STORE_F32 = 1, PAIRS = 2, SILU_PAIRS = 3 };
struct TileEpi {
  void* out;
  int ldc;
  GateForm form;
  const float* gate_bias;
  const float* up_bias;
};

// a (gate, up) pair joined, without the scale, as gated_act does it.  (Its division is rounded: a reciprocal and one step took 112.6 us in place of 114.7 for
// 2,048 rows of 16,384 x 2,048, and lost what 1 + exp(-g) above 2^126 divides.)
template <int ACT> __device__ __forceinline__ float join(const GateForm& f, float g, float u) {
  if constexpr (ACT == GATE_LIMITED) {
    return limited_pair(g, u, f.limit);
  } else if constexpr (ACT == 1) {   // tanh(t) = 1 - 2 / (1 + exp(2 t)); exp overflows to +inf for large t, which gives 1
    const float t = 0.7978845608028654f * (g + 0.044715f * g * g * g);
    return 0.5f * g * (2.f - 2.f / (1.f + __expf(2.f * t))) * u;
  } else {
    return g / (1.f + __expf(-g)) * u;
  }
}
// as a stored product is read again
__device__ __forceinline__ float stored(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// bf16 results leave through the wave's own rows in LDS, as whole pieces of 16 bytes: N, ldc in whole 8s of them.
template <class T, int KIND> constexpr int own_bytes() {
  return KIND == STORE_F32 ? 0 : OwnRows<KIND == STORE_BF16 ? 2 * T::CT : T::CT>::BYTES;
}

// between a wave's writes of its own rows in LDS and its reads of them: a wave's accesses go in order, the compiler's must too
__device__ __forceinline__ void wave_rows() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Whole rows of bf16: value(r, c, where the lane's four columns go).
template <class T, int PIECES, class Value>
__device__ __forceinline__ void store_rows(const T& w, void* out, int ldc, char* own, int m0, int M, int col0, int cols, const Value& value) {
  using Own = OwnRows<PIECES>;
#pragma unroll
  for (int r = 0; r < T::RT; ++r) {
#pragma unroll
    for (int c = 0; c < T::CT; ++c) value(r, c);
    wave_rows();
    Own::each(own, w.lane, [&](int row, int piece, const uint4& v) {
      const int m = m0 + (w.wm * T::RT + r) * 16 + row, n = col0 + piece * 8;
      if (m < M && n < cols) *reinterpret_cast<uint4*>(static_cast<bf16_t*>(out) + static_cast<size_t>(m) * ldc + n) = v;
    });
    wave_rows();
  }
}

// (a form at a time: with the forms told apart pair by pair the code outgrows the instruction cache)
template <class T, int ACT, bool BIASED>
__device__ __forceinline__ void store_pairs(const T& w, const TileEpi& e, char* own, int m0, int n0, int M, int N) {
  using Own = OwnRows<T::CT>;
  const int r16 = w.lane % 16, kg = w.lane / 16, cols = N / 2, col0 = (n0 + w.wn * T::CT * 16) / 2;
  float gb[T::CT][2], ub[T::CT][2];
  if constexpr (BIASED) {
#pragma unroll
    for (int c = 0; c < T::CT; ++c)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int at = min(col0 + c * 8 + 2 * kg + i, cols - 1);
        gb[c][i] = e.gate_bias ? e.gate_bias[at] : 0.f;
        ub[c][i] = e.up_bias ? e.up_bias[at] : 0.f;
      }
  }
  store_rows<T, T::CT>(w, e.out, e.ldc, own, m0, M, col0, cols, [&](int r, int c) {
    const f32x4 a = w.acc[r][c];
    float y[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      y[i] = BIASED ? join<ACT>(e.form, stored(a[2 * i]) + gb[c][i], stored(a[2 * i + 1]) + ub[c][i]) * e.form.scale
                    : join<ACT>(e.form, stored(a[2 * i]), stored(a[2 * i + 1]));
    *reinterpret_cast<uint32_t*>(own + Own::place(r16, c) + kg * 4) = f32_to_bf16(y[0]) | static_cast<uint32_t>(f32_to_bf16(y[1])) << 16;
  });
}

template <class T, int KIND>
__device__ __forceinline__ void store_tile(const T& w, const TileEpi& e, char* own, int m0, int n0, int M, int N) {
  const int r16 = w.lane % 16, kg = w.lane / 16;
  if constexpr (KIND == STORE_F32) {
#pragma unroll
    for (int r = 0; r < T::RT; ++r)
#pragma unroll
      for (int c = 0; c < T::CT; ++c) {
        const int m = m0 + (w.wm * T::RT + r) * 16 + r16, n = n0 + (w.wn * T::CT + c) * 16 + kg * 4;
        if (m >= M || n >= N) continue;
        *reinterpret_cast<f32x4*>(static_cast<float*>(e.out) + static_cast<size_t>(m) * e.ldc + n) = w.acc[r][c];
      }
  } else if constexpr (KIND == SILU_PAIRS) {
    store_pairs<T, 0, false>(w, e, own, m0, n0, M, N);
  } else if constexpr (KIND == PAIRS) {
    if (e.form.act == GATE_LIMITED) store_pairs<T, GATE_LIMITED, true>(w, e, own, m0, n0, M, N);
    else if (e.form.act == 1) store_pairs<T, 1, true>(w, e, own, m0, n0, M, N);
    else store_pairs<T, 0, true>(w, e, own, m0, n0, M, N);
  } else {
    using Own = OwnRows<2 * T::CT>;
    const int col0 = n0 + w.wn * T::CT * 16;
    store_rows<T, 2 * T::CT>(w, e.out, e.ldc, own, m0, M, col0, N, [&](int r, int c) {
      const f32x4 a = w.acc[r][c];
      *reinterpret_cast<uint2*>(own + Own::place(r16, 2 * c + kg / 2) + (kg % 2) * 8) =
          make_uint2(f32_to_bf16(a[0]) | static_cast<uint32_t>(f32_to_bf16(a[1])) << 16,
                     f32_to_bf16(a[2]) | static_cast<uint32_t>(f32_to_bf16(a[3])) << 16);
    });
  }
}

template <class T, int KIND>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_tile_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int M, int N,
                                                                  int K, int lda, int tm, int tn, int step, TileEpi e) {
  constexpr int OWN = own_bytes<T, KIND>();
  __shared__ __attribute__((aligned(1024))) char lds[T::BYTES + T::WAVES * OWN];
  int item, last;
  if (!share_of(tm * tn, item, last)) return;
  Product src{A, W, M, N, K, lda, tm, tn, last, step, item, item};
  T walk;
  walk.template start<false>(lds, K / 32, src);
  char* own = lds + T::BYTES + walk.wave * OWN;
  const auto tile = [&](auto is_last, bool first) {
    walk.template run<decltype(is_last)::value>(K / 32, first, src);
    int row_tile, col_tile;
    place_of(item, tm, tn, row_tile, col_tile);
    store_tile<T, KIND>(walk, e, own, row_tile * T::BM, col_tile * T::BN, M, N);
  };
  bool first = true;
  for (; item + step < last; item += step, first = false) tile(std::false_type{}, first);
  tile(std::true_type{}, first);
}

// One tile a workgroup (FEW: see Walk::start).
template <class T, bool FEW>
__global__ __launch_bounds__(T::THREADS, 2) void qkv_tile_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                 bf16_t* __restrict__ q_out, int M, int N, int K, int lda, int ldq,
                                                                 int tm, int tn, RopeEpi rp) {
  constexpr int BM = T::BM, BN = T::BN, RT = T::RT, CT = T::CT, WM = T::WM, WAVES = T::WAVES;
  constexpr int ANGLES = BM * (MAX_ROT * 4 + 16);
  __shared__ __attribute__((aligned(1024))) char lds[T::BYTES > ANGLES ? T::BYTES : ANGLES];
  int item, last;
  if (!share_of(tm * tn, item, last)) return;
  int row_tile, col_tile;
  place_of(item, tm, tn, row_tile, col_tile);
  const int m0 = row_tile * BM, n0 = col_tile * BN;
  T walk;
  const int lane = threadIdx.x % KVF_WAVE, r16 = lane % 16, kg = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVF_WAVE), wm = wave % WM, wn = wave / WM;
  // What the epilogue needs of a lane's tokens is asked for ahead of the walk over K: position and sequence before the first
  // stages, the page they lead to behind those.
  int pos[RT], page[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = min(m0 + (wm * RT + r) * 16 + r16, M - 1);
    pos[r] = rp.positions[m];
    page[r] = rp.write_kv ? rp.seq_of_token[m] : -1;   // the sequence for now
  }
  Product src{A, W, M, N, K, lda, tm, tn, item + 1, 1, item, item};
  walk.template start<FEW>(lds, K / 32, src);
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int blk = pos[r] / rp.block_size;
    const bool has = pos[r] >= 0 && pos[r] < rp.table_len && page[r] >= 0 && page[r] < rp.n_seqs && blk < rp.table_stride;
    page[r] = has ? rp.block_table[static_cast<size_t>(page[r]) * rp.table_stride + blk] : -1;
  }
  if constexpr (FEW) walk.run_few(K / 32);
  else walk.template run<true>(K / 32, true, src);
  const auto& acc = walk.acc;
  // The angles of the tile's tokens go through LDS, a cosine and a sine side by side: a lane would read them 4 bytes at
  // a time from 16 rows of the tables otherwise, for every head anew (10 of 42 us at 2,048 x 3,072).
  const int rot8 = rp.rot / 8, pitch = rp.rot * 4 + 16;   // 16 more bytes a row: 16 rows lie on all banks
  if (rp.rot > 0 && n0 < (rp.H + rp.KV) * rp.d) {
    __syncthreads();                                      // nobody reads a stage any more
    for (int i = threadIdx.x; i < BM * rot8; i += WAVES * KVF_WAVE) {
      const int row = i / rot8, j = i - row * rot8, p = rp.positions[min(m0 + row, M - 1)];
      const size_t at = static_cast<size_t>(p >= 0 && p < rp.table_len ? p : 0) * (rp.rot / 2) + 4 * j;
      const float4 cs = *reinterpret_cast<const float4*>(rp.cos_t + at), sn = *reinterpret_cast<const float4*>(rp.sin_t + at);
      float4* to = reinterpret_cast<float4*>(lds + row * pitch + j * 32);
      to[0] = make_float4(cs.x, sn.x, cs.y, sn.y);
      to[1] = make_float4(cs.z, sn.z, cs.w, sn.w);
    }
    __syncthreads();
  }
  // A lane holds four neighbouring columns (N and d are multiples of 4: they lie in one head) of RT x CT rows and heads.
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int n = n0 + (wn * CT + c) * 16 + kg * 4, head = n / rp.d, e = n - head * rp.d;
    if (n >= N) continue;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int m = m0 + (wm * RT + r) * 16 + r16;
      if (m >= M) continue;
      uint16_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = f32_to_bf16(acc[r][c][i]);
      if (head < rp.H + rp.KV && e < rp.rot && pos[r] >= 0 && pos[r] < rp.table_len) {   // rot is a multiple of 8 here
        const f32x4 turn = *reinterpret_cast<const f32x4*>(lds + ((wm * RT + r) * 16 + r16) * pitch + e * 4);
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          // (which product is rounded before the sum is as in rope_kvwrite_tile_kernel)
          const float cs = turn[i], sn = turn[i + 1], x1 = bf16_to_f32(b[i]), x2 = bf16_to_f32(b[i + 1]);
          b[i] = f32_to_bf16(fmaf(x1, cs, -(x2 * sn)));
          b[i + 1] = f32_to_bf16(fmaf(x1, sn, x2 * cs));
        }
      }
      const uint2 packed = make_uint2(b[0] | static_cast<uint32_t>(b[1]) << 16, b[2] | static_cast<uint32_t>(b[3]) << 16);
      if (head < rp.H || head >= rp.H + 2 * rp.KV) {   // q, and columns behind q, k and v, which follow q as they are
        const int col = head < rp.H ? n : n - 2 * rp.KV * rp.d;
        *reinterpret_cast<uint2*>(q_out + static_cast<size_t>(m) * ldq + col) = packed;
      } else if (page[r] >= 0 && page[r] < rp.num_blocks) {
        const int off = pos[r] % rp.block_size;
        if (head < rp.H + rp.KV) {
          *reinterpret_cast<uint2*>(rp.k_pages + ((static_cast<size_t>(page[r]) * rp.KV + head - rp.H) * rp.block_size + off) * rp.d + e) = packed;
        } else {   // V pages are [num_blocks, KV, d, block_size]: neighbouring tokens are neighbouring elements
          bf16_t* dst = rp.v_pages + ((static_cast<size_t>(page[r]) * rp.KV + head - rp.H - rp.KV) * rp.d + e) * rp.block_size + off;
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[static_cast<size_t>(i) * rp.block_size].bits = b[i];
        }
      }
    }
  }
}

// Tiles that are tried and what they take, in us: once a launch, once a round of them over the chip (weights from memory), and with
// K, a round at K = 2,048.  Those of plain and gated products were fitted to 244 sizes of 66 to 2,048 rows, 1,024 to
// 28,672 columns and K of 512 to 14,336: within 8% (64 x 64: 12%) in the mean.
struct Tile {
  int bm, bn, per_cu;
  float once, round, k2048;
};
constexpr Tile TILES[] = {{256, 256, 1, -7.1f, 13.3f, 37.3f}, {192, 256, 1, -2.4f, 7.5f, 29.6f}, {128, 256, 1, -1.0f, 5.1f, 23.7f},
                          {128, 128, 1, 0.9f, 2.6f, 17.1f},   {64, 128, 1, 1.4f, 1.6f, 12.0f},   {192, 128, 1, 0.4f, 3.5f, 20.2f},
                          {256, 128, 1, -0.8f, 5.0f, 24.4f},  {64, 64, 2, 2.4f, 0.7f, 12.7f}};
constexpr Tile PLAIN_TILES[] = {{192, 256, 1, -3.6f, 8.7f, 29.0f}, {128, 256, 1, -2.2f, 6.3f, 23.3f}, {128, 128, 1, 0.1f, 3.3f, 16.6f},
                                {64, 128, 1, 1.2f, 1.9f, 11.9f},   {192, 128, 1, -0.4f, 4.2f, 19.8f}, {256, 128, 1, -1.9f, 6.1f, 23.9f},
                                {64, 64, 2, 2.4f, 0.8f, 12.6f}};
// (with rotation and cache write; fitted to 72 sizes of 66 to 2,048 rows, 1,024 to 6,144 columns and K of 512 to 4,096, the two smallest anew with 231 of
// 65 to 2,100 rows, 192 to 10,240 columns and K from 64: over those the tile it names takes at most 3% more than the best of the six, 0.05% in the mean.
// With a round of 64 x 64 at 0.5 us as the larger K asked for, many rounds of short ones took that tile: 1,434 rows of 4,096 x 192 18.5 us,
// 13.2 in tiles of 192 x 128, 1,705 of 6,144 x 512 37.5 and 27.9)
constexpr Tile QKV_TILES[] = {{128, 192, 1, -0.2f, 8.4f, 20.5f}, {192, 128, 1, -1.7f, 10.3f, 18.9f}, {128, 128, 1, 0.8f, 6.1f, 15.4f},
                              {64, 192, 1, 1.1f, 4.6f, 14.7f},   {64, 128, 1, 1.7f, 2.9f, 11.0f},    {64, 64, 2, 3.0f, 2.5f, 11.7f}};

template <int COUNT> int best_tile(const Tile (&tiles)[COUNT], int M, int N, int K, int cus, float& us) {
  int best = 0;
  us = 0.f;
  for (int i = 0; i < COUNT; ++i) {
    const Tile& t = tiles[i];
    const long of = static_cast<long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const long at_once = static_cast<long>(cus) * t.per_cu, rounds = (of + at_once - 1) / at_once;
    const float cost = (t.once + rounds * (t.round + t.k2048 * K / 2048.f)) * (t.per_cu == 2 && of <= cus ? 0.82f : 1.f);
    if (i == 0 || cost < us) {
      best = i;
      us = cost;
    }
  }
  return best;
}
template <int N> constexpr int count_of(const Tile (&)[N]) { return N; }

template <class T>
int launch_qkv(const bf16_t* A, const bf16_t* W, bf16_t* q_out, int M, int N, int K, int lda, int ldq, const RopeEpi& rp, hipStream_t s) {
  const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN;
  const auto go = [&](auto few) {
    hipLaunchKernelGGL((qkv_tile_kernel<T, decltype(few)::value>), dim3((tm * tn + 7) / 8 * 8), dim3(T::THREADS), 0, s, A, W, q_out, M, N, K,
                       lda, ldq, tm, tn, rp);
    return kvf_last_error();
  };
  return K / 32 < T::NW + 2 ? go(std::true_type{}) : go(std::false_type{});
}

int launch_qkv_tile(int tile, const bf16_t* A, const bf16_t* W, bf16_t* q_out, int M, int N, int K, int lda, int ldq, const RopeEpi& rp, hipStream_t s) {
  switch (tile) {
    case 0: return launch_qkv<Walk<2, 4, 4, 3, 4>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 1: return launch_qkv<Walk<4, 2, 3, 4, 3>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 2: return launch_qkv<Walk<2, 4, 4, 2, 4>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 3: return launch_qkv<Walk<2, 4, 2, 3, 4>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 4: return launch_qkv<Walk<2, 4, 2, 2, 4>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 5: return launch_qkv<Walk<2, 2, 2, 2, 4>>(A, W, q_out, M, N, K, lda, ldq, rp, s);
  }
  return static_cast<int>(hipErrorInvalidValue);
}

template <class T, int... KINDS>
int launch_tiles(int kind, int per_cu, const bf16_t* A, const bf16_t* W, int M, int N, int K, int lda, const TileEpi& e, hipStream_t s) {
  const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN;
  const int share = (tm * tn + 7) / 8, room = compute_units() / 8 * per_cu, step = share < room ? share : room;
  int code = static_cast<int>(hipErrorInvalidValue);
  const auto go = [&](auto k) {
    if (kind != decltype(k)::value) return;
    hipLaunchKernelGGL((gemm_tile_kernel<T, decltype(k)::value>), dim3(8 * step), dim3(T::THREADS), 0, s, A, W, M, N, K, lda, tm, tn, step, e);
    code = kvf_last_error();
  };
  (go(std::integral_constant<int, KINDS>{}), ...);
  return code;
}
template <class T>
int launch_pairs(int kind, int per_cu, const bf16_t* A, const bf16_t* W, int M, int N, int K, int lda, const TileEpi& e, hipStream_t s) {
  return launch_tiles<T, PAIRS, SILU_PAIRS>(kind, per_cu, A, W, M, N, K, lda, e, s);
}
template <class T>
int launch_plain(int kind, int per_cu, const bf16_t* A, const bf16_t* W, int M, int N, int K, int lda, const TileEpi& e, hipStream_t s) {
  return launch_tiles<T, STORE_BF16, STORE_F32>(kind, per_cu, A, W, M, N, K, lda, e, s);
}

int launch_tile(int tile, int kind, const bf16_t* A, const bf16_t* W, int M, int N, int K, int lda, const TileEpi& e, hipStream_t s) {
  using Launch = int (*)(int, int, const bf16_t*, const bf16_t*, int, int, int, int, const TileEpi&, hipStream_t);
  static constexpr Launch pairs[] = {launch_pairs<Walk<4, 2, 4, 8, 2>>, launch_pairs<Walk<4, 2, 3, 8, 2>>, launch_pairs<Walk<2, 4, 4, 4, 3>>,
                                     launch_pairs<Walk<2, 4, 4, 2, 4>>, launch_pairs<Walk<2, 4, 2, 2, 4>>, launch_pairs<Walk<4, 2, 3, 4, 3>>,
                                     launch_pairs<Walk<4, 2, 4, 4, 3>>, launch_pairs<Walk<2, 2, 2, 2, 4>>};
  static constexpr Launch plain[] = {launch_plain<Walk<4, 2, 3, 8, 2>>, launch_plain<Walk<2, 4, 4, 4, 3>>, launch_plain<Walk<2, 4, 4, 2, 4>>,
                                     launch_plain<Walk<2, 4, 2, 2, 4>>, launch_plain<Walk<4, 2, 3, 4, 3>>, launch_plain<Walk<4, 2, 4, 4, 3>>,
                                     launch_plain<Walk<2, 2, 2, 2, 4>>};
  static_assert(sizeof(pairs) / sizeof(pairs[0]) == count_of(TILES) && sizeof(plain) / sizeof(plain[0]) == count_of(PLAIN_TILES), "one for each tile");
  return kind == PAIRS || kind == SILU_PAIRS ? pairs[tile](kind, TILES[tile].per_cu, A, W, M, N, K, lda, e, s)
                                             : plain[tile](kind, PLAIN_TILES[tile].per_cu, A, W, M, N, K, lda, e, s);
}
}  // namespace

// Whether the fused projection takes M rows of [N, K]: where it is expected to be faster than a product of its own (the library's, or one in
// tiles) and rope_kvwrite, which take 9 us, K / 285, 5.3 TB/s over the weights, 1.75 PFLOP/s, and 3.5 TB/s over 4 M N bytes (within 10% of
// what was measured at six widths and twelve row counts).  Both measured, those two / this, at 3,072 x 2,048: 2,048 rows 39.6 / 32.6,
// 1,024 30.6 / 21.0, 512 21.6 / 16.2, 100 18.1 / 12.2; 1,024 x 512: 2,048 rows 13.3 / 9.1, 66 8.6 / 6.5; 6,144 x 4,096: 1,024 rows 61.5 /
// 55.0, 333 44.8 / 37.8.  Large ones with a part of a round of tiles left over stay there: 1,500 rows of 6,144 x 4,096 83 / 97,
// 2,048 of 5,120 x 3,072 66 / 76.
KVF_EXPORT int kvf_gemm_tile_qkv_takes(int M, int N, int K, int rot) {
  if (rot < 0 || rot % 8 != 0 || rot > MAX_ROT) return 0;
  if (M <= 0 || N <= 0 || N % 4 != 0 || K <= 0 || K % 64 != 0) return 0;
  float us;
  best_tile(QKV_TILES, M, N, K, compute_units(), us);
  const double two = 9.0 + K / 285.0 + 2.0 * N * K / 5.3e6 + 2.0 * M * N * K / 1.75e9 + 4.0 * M * N / 3.5e6;
  return K <= 512 || us <= 0.92 * two;   // (short K: what the two store and read again is most of it, 2,091 rows of 8,192 x 256 50 / 35)
}

// Which of QKV_TILES M rows of [N, K] take.
KVF_EXPORT int kvf_gemm_tile_qkv_tile(int M, int N, int K) {
  float us;
  return best_tile(QKV_TILES, M, N, K, compute_units(), us);
}

// Arguments as kvf_gemm_bf16_qkv_rope with bf16 rows and tiled weights; K % 64 == 0.  tile: which of QKV_TILES,
// or -1 for the one that the rule takes.
KVF_EXPORT int kvf_gemm_tile_qkv_rope(const void* A, const void* W, void* q_out, int M, int K, int lda, int ldq, const int* positions,
                                      const int* seq_of_token, const float* cos_t, const float* sin_t, const int* block_table,
                                      void* k_pages, void* v_pages, int H, int KV, int d, int rot, int table_len, int block_size,
                                      int table_stride, int num_blocks, int write_kv, int n_seqs, int extra_cols, int tile,
                                      hipStream_t s) {
  if (M <= 0) return 0;
  if (K <= 0 || K % 64 != 0 || lda % 8 != 0 || reinterpret_cast<uintptr_t>(A) % 16 != 0 || reinterpret_cast<uintptr_t>(W) % 16 != 0 ||
      d % 4 != 0 || rot < 0 || rot % 8 != 0 || rot > d || rot > MAX_ROT || ldq % 4 != 0 || reinterpret_cast<uintptr_t>(q_out) % 8 != 0 || extra_cols < 0 ||
      extra_cols % 4 != 0 || KV < 0 || ldq < H * d + extra_cols || block_size <= 0 ||
      (rot > 0 && (table_len <= 0 || reinterpret_cast<uintptr_t>(cos_t) % 16 != 0 || reinterpret_cast<uintptr_t>(sin_t) % 16 != 0)) || (write_kv && KV == 0) || lda > (1 << 23))
    return static_cast<int>(hipErrorInvalidValue);
  const RopeEpi rp{positions, seq_of_token, cos_t, sin_t, block_table, static_cast<bf16_t*>(k_pages), static_cast<bf16_t*>(v_pages),
                   H, KV, d, rot, table_len, block_size, table_stride, num_blocks, write_kv, n_seqs, 0, 0.f, 1.f, nullptr, nullptr};
  const int N = (H + 2 * KV) * d + extra_cols;
  if (N <= 0) return 0;
  float us;
  if (tile < 0) tile = best_tile(QKV_TILES, M, N, K, compute_units(), us);
  return launch_qkv_tile(tile, static_cast<const bf16_t*>(A), static_cast<const bf16_t*>(W), static_cast<bf16_t*>(q_out), M, N, K, lda, ldq, rp, s);
}

constexpr int MIN_K = 320;   // ten stages: eight on their way and one pair more

// What the library's product of M rows of [N, K] takes, in us, in two ways.  By its work: 5.5 us, 1.34 with 1,000 of K, 8 TB/s over the weights,
// 1.57 PFLOP/s, 5 TB/s over what is stored; the pass behind it that joins pairs 1 us and 5 TB/s.
double library_by_work(int M, int N, int K, bool pairs) {
  const double mn = 1e-6 * M * N;
  return 5.5 + 1.34e-3 * K + 0.25e-6 * N * K + 1.28e-3 * mn * K + 0.4 * mn + (pairs ? 1.0 + 0.6 * mn : 0.0);
}
// By the rounds of its tiles over the chip, which the first does not see: 2,048 rows of 8,192 x 4,096 are one round of 256 x 256.  Fitted to
// 2,113 times of 66 to 8,192 rows, 512 to 33,000 columns, K of 320 to 14,336: within 11% in the mean.
double library_by_rounds(int M, int N, int K, int cus, bool pairs) {
  constexpr int tiles[][2] = {{256, 256}, {256, 128}, {128, 128}, {64, 64}};
  const double k = K / 2048.0;
  double best = 0.0;
  for (const auto& t : tiles) {
    const long of = static_cast<long>((M + t[0] - 1) / t[0]) * ((N + t[1] - 1) / t[1]), rounds = (of + cus - 1) / cus;
    const double area = t[0] * t[1] / 65536.0, us = rounds * (6.4 * area + (40.2 * area + 1.25 * (t[0] + t[1]) / 512.0) * k);
    if (best == 0.0 || us < best) best = us;
  }
  return 8.7 + 1.9 * k + 0.12e-6 * N * K + best + (pairs ? 3.3 + 0.4e-6 * M * N : 0.0);
}

// Whether kvf_gemm_tile takes M rows of [N, K]: where it is expected to be faster than the library's product, and, with `pairs`, a pass over
// it that joins the pairs, by both of the above, and below MOST products of two elements.  Of 1,111 sizes of gated products that were
// measured it takes 721, in 0.63 of the time of the two, two of them more than 5% slower; of 1,002 of plain ones 470, in 0.71 of the
// library's, four more than 5% slower.  (By the first alone it took 17 and 57 such, up to 36% slower: plain products of one round of 256 x 256, 2,048 rows
// of 8,192 x 2,048 52 -> 67 us, and gated ones of large weights, 1,013 rows of 28,672 x 4,096 193 -> 214.)  Both measured, library / this in us.
// Gated: 2,048 rows of 16,384 x 2,048 120 / 115, 512 42 / 36, 66 20 / 17; of 4,096 x 2,048 38 / 32.  Plain: 2,048 rows of 2,048 x 1,024
// 13.3 / 12.8, 320 of 3,072 x 2,048 13.1 / 11.6, of 1,024 x 512 8.8 / 6.8, 66 6.1 / 4.4.  The library's: 2,048 rows of 2,048 x 8,192 73 / 78, of
// 6,144 x 4,096 80 / 93, gated ones of 28,672 x 4,096 377 / 391.
// Above MOST the two take the same within some percent whichever is faster, and the library's is left alone.
// (Tiles of 256 x 256 are not for plain products: of 22 sizes at which they would be the best, the library is faster at 17.)
constexpr double MOST = 1.1e11;
KVF_EXPORT int kvf_gemm_tile_takes(int M, int N, int K, int pairs) {
  if (M <= 0 || N <= 0 || N % (pairs ? 16 : 8) != 0 || K < MIN_K || K % 64 != 0 || 1.0 * M * N * K > MOST) return 0;
  const int cus = compute_units();
  float us;
  if (pairs) best_tile(TILES, M, N, K, cus, us);
  else best_tile(PLAIN_TILES, M, N, K, cus, us);
  return us <= 0.95 * library_by_work(M, N, K, pairs) && us <= 0.86 * library_by_rounds(M, N, K, cus, pairs);
}

// The product of many rows: arguments as kvf_gemm_bf16 with bf16 rows and tiled weights.  kind: what becomes of it (Kind), `form`, limit, scale
// and the biases (null: none) with PAIRS.  K in whole 64s from MIN_K; N and ldc in whole 8s (PAIRS: N in 16s, ldc counted in pairs),
// out at 16 bytes.  tile: which of TILES (PAIRS) or PLAIN_TILES, or -1 for the one that the rule takes.
KVF_EXPORT int kvf_gemm_tile(const void* A, const void* W, void* out, int kind, int M, int N, int K, int lda, int ldc, int form, float limit,
                             float scale, const float* gate_bias, const float* up_bias, int tile, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  const bool pairs = kind == PAIRS;
  if (K < MIN_K || K % 64 != 0 || lda % 8 != 0 || lda < K || lda > (1 << 23) || reinterpret_cast<uintptr_t>(A) % 16 != 0 ||
      reinterpret_cast<uintptr_t>(W) % 16 != 0 || reinterpret_cast<uintptr_t>(out) % 16 != 0 || kind < STORE_BF16 || kind > PAIRS ||
      N % (pairs ? 16 : 8) != 0 || ldc % 8 != 0 || ldc < (pairs ? N / 2 : N) || form < 0 || form > GATE_LIMITED ||
      (form == GATE_LIMITED && !(limit > 0.f)) || tile < -1 || tile >= (pairs ? count_of(TILES) : count_of(PLAIN_TILES)))
    return static_cast<int>(hipErrorInvalidValue);
  const TileEpi e{out, ldc, GateForm{form, limit, scale}, gate_bias, up_bias};
  float us;
  if (tile < 0) tile = pairs ? best_tile(TILES, M, N, K, compute_units(), us) : best_tile(PLAIN_TILES, M, N, K, compute_units(), us);
  const bool silu = pairs && form == 0 && scale == 1.f && !gate_bias && !up_bias;
  return launch_tile(tile, silu ? static_cast<int>(SILU_PAIRS) : kind, static_cast<const bf16_t*>(A), static_cast<const bf16_t*>(W), M, N, K, lda, e, s);
}
