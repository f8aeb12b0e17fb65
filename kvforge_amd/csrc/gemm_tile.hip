// The fused q/k/v projection of many rows: C = A * W^T for bf16 rows and bf16 weights in tiles (see the head of
// gemm_bf16.hip), fp32 sums, with rotary and the cache write in its epilogue (RopeEpi).
//
// Sums run along K in steps of 32 on one accumulator and are rounded to bf16 before they are rotated, as a stored product is.
// The library's product, which stood here with rope_kvwrite behind it, does the same at most sizes, to the bit; it cuts K at 14 of
// 306 that were compared (65 to 77 rows over 3,072 and 3,136 columns, 128 rows over 1,024 and 2,048), where 3 in 100,000 of the
// result turn a rounding.
//
// A workgroup takes a tile of BM rows x BN columns, 64 of K a stage.  Rows and weights go from memory straight
// into LDS, NB stages side by side, without passing through registers, and are asked for NB - 1.5 stages ahead.  A
// stage has one barrier, in its middle: before it come the products of the stage's first half, beside which the
// second half's operands are read from LDS and the last loads of an earlier stage are asked for; behind it
// those of the second half, beside which the next stage's operands are read (they have arrived by
// then) and the first loads of the stage that takes the place of the one before are asked for.  Loads stand one by one between products:
// asked for in one go behind the barrier they block the waves for as long as a product of the
// stage takes (2,048 x 2,048 x 2,048: 28.5 us on four waves, 19.9 spread out).
//
// What bounds it: a stage of 128 x 128 takes 0.5 us where its matrix instructions take 0.21, its loads from L2 0.32 and its
// reads of LDS 0.16; they overlap in part, and weights from memory add 0.08.  Without
// the epilogue it is as fast as the library's product, 28.5 us for 2,048 rows of 3,072 x 2,048 (0.9 PFLOP/s); with it 33, where
// product and rope_kvwrite took 42.
#include <type_traits>

#include "gemm_common.h"

namespace {
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// 64 lanes x 16 bytes from memory straight into LDS: base + off (per lane) -> lds + 16 * lane.  Written by hand because
// the compiler, which cannot tell the stages of a buffer apart, waits for every such load before any read of
// LDS.  The loads have no output register; whoever reads the bytes waits for vmcnt and the barrier first, in loads_left, which
// says to the compiler that memory has changed: here it would order every read of LDS beside the load behind it.
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "m0");
}
// At most N of the wave's own loads are still on their way, and the other waves have come as far.
template <int N> __device__ __forceinline__ void loads_left() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory"); }

constexpr int MAX_ROT = 128;

template <int WM, int WN, int RT, int CT, int NB>
__global__ __launch_bounds__(WM * WN * KVF_WAVE, 2) void gemm_tile_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, bf16_t* __restrict__ q_out, int M, int N, int K, int lda,
    int ldq, int tm, int tn, RopeEpi rp) {
  constexpr int WAVES = WM * WN, BM = 16 * RT * WM, BN = 16 * CT * WN;
  constexpr int AC = BM / 8, WC = BN / 8;             // KB of a stage
  constexpr int AL = AC / WAVES, WL = WC / WAVES, LOADS = AL + WL;
  static_assert(AC % WAVES == 0 && WC % WAVES == 0 && NB >= 3, "a wave asks for whole KB of rows and of weights");
  constexpr uint32_t STAGE = (AC + WC) * 1024;
  static_assert(NB * STAGE >= BM * (MAX_ROT * 4 + 16), "the angles take the place of the stages");
  __shared__ __attribute__((aligned(1024))) char lds[NB * STAGE];
  const int lane = threadIdx.x % KVF_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVF_WAVE);
  const int r16 = lane % 16, kg = lane / 16;
  const int total = tm * tn, share = (total + 7) / 8;
  const int item = static_cast<int>(blockIdx.x % 8) * share + static_cast<int>(blockIdx.x / 8);
  if (static_cast<int>(blockIdx.x / 8) >= share || item >= total) return;
  constexpr int GM = 4;
  const int band = item / (GM * tn), in = item - band * GM * tn, gm = min(GM, tm - band * GM);
  const int m0 = (band * GM + in % gm) * BM, n0 = in / gm * BN;
  const int S = K / 64, ksteps = K / 32, groups = (N + 15) / 16;
  uint32_t aoff[AL], woff[WL];
  const char* abase = reinterpret_cast<const char*>(A + static_cast<size_t>(m0) * lda);
  const char* wbase = reinterpret_cast<const char*>(W) + static_cast<size_t>(n0 / 16) * ksteps * 1024;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u32*)lds));
#pragma unroll
  for (int i = 0; i < AL; ++i)
    aoff[i] = static_cast<uint32_t>(min((wave * AL + i) * 8 + lane / 8, M - 1 - m0)) * lda * 2 + ((lane % 8) ^ (lane / 8)) * 16;
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int w = wave * WL + i;
    woff[i] = (static_cast<uint32_t>(min(w / 2, groups - 1 - n0 / 16)) * ksteps + w % 2) * 1024 + lane * 16;
  }
  auto issue1 = [&](int i, uint32_t buf, int s) {
    if (i < AL) load_to_lds(abase + static_cast<size_t>(s) * 128, aoff[i < AL ? i : 0], lds0 + buf + (wave * AL + i) * 1024);
    else load_to_lds(wbase + static_cast<size_t>(s) * 2048, woff[i >= AL ? i - AL : 0], lds0 + buf + (AC + wave * WL + i - AL) * 1024);
  };
  const int wm = wave % WM, wn = wave / WM;
  const int a_at = wm * RT * 2048 + (r16 / 8) * 1024 + (r16 % 8) * 128, x0 = (kg ^ (r16 % 8)) * 16;
  const int w_at = AC * 1024 + wn * CT * 2048 + lane * 16;
  f32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frags { bf16x8 a[RT], w[CT]; } f0, f1;
  constexpr int PR = RT * CT, RD = RT + CT;
  auto read1 = [&](Frags& f, int i, uint32_t buf, int h) {
    if (i < CT) f.w[i < CT ? i : 0] = *reinterpret_cast<const bf16x8*>(lds + buf + w_at + i * 2048 + h * 1024);
    else f.a[i >= CT ? i - CT : 0] = *reinterpret_cast<const bf16x8*>(lds + buf + (a_at + (x0 ^ (h * 64))) + (i - CT) * 2048);
  };
  auto half = [&](const Frags& f, Frags& g, uint32_t gbuf, int gh, auto lo, auto hi, uint32_t to, int ts) {
    constexpr int LO = decltype(lo)::value, HI = decltype(hi)::value;
    __builtin_amdgcn_sched_barrier(0);
    int rd = 0, ld = LO;
#pragma unroll
    for (int p = 0; p < PR; ++p) {
#pragma unroll
      for (; rd < RD && rd < (p + 1) * RD * 2 / PR; ++rd) read1(g, rd, gbuf, gh);
      __builtin_amdgcn_sched_barrier(0);
      acc[p / CT][p % CT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[p % CT], f.a[p / CT], acc[p / CT][p % CT], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (; ld < HI && ld - LO < (p + 1) * (HI - LO) / PR; ++ld)
        if (ts < S) issue1(ld, to, ts);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // What the epilogue needs of a lane's tokens is asked for ahead of the walk over K: position and sequence before the first
  // stages, the page they lead to behind those.
  int pos[RT], page[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = min(m0 + (wm * RT + r) * 16 + r16, M - 1);
    pos[r] = rp.positions[m];
    page[r] = rp.write_kv ? rp.seq_of_token[m] : -1;   // the sequence for now
  }
  using Int0 = std::integral_constant<int, 0>;
  using IntH = std::integral_constant<int, LOADS / 2>;
  using IntL = std::integral_constant<int, LOADS>;
#pragma unroll
  for (int i = 0; i < NB - 2; ++i)
#pragma unroll
    for (int j = 0; j < LOADS; ++j)
      if (i < S) issue1(j, i * STAGE, i);
#pragma unroll
  for (int j = 0; j < LOADS / 2; ++j)
    if (NB - 2 < S) issue1(j, (NB - 2) * STAGE, NB - 2);
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int blk = pos[r] / rp.block_size;
    const bool has = pos[r] >= 0 && pos[r] < rp.table_len && page[r] >= 0 && page[r] < rp.n_seqs && blk < rp.table_stride;
    page[r] = has ? rp.block_table[static_cast<size_t>(page[r]) * rp.table_stride + blk] : -1;
  }
  if (NB - 2 < S) loads_left<LOADS * (NB - 3) + LOADS / 2>();
  else loads_left<0>();
#pragma unroll
  for (int i = 0; i < RD; ++i) read1(f0, i, 0, 0);
  uint32_t cur = 0, last = (NB - 1) * STAGE, fill = (NB - 2) * STAGE;
#pragma unroll 1
  for (int s = 0; s < S; ++s) {
    half(f0, f1, cur, 1, IntH{}, IntL{}, fill, s + NB - 2);
    if (s + NB - 2 < S) loads_left<LOADS * (NB - 3)>();
    else loads_left<0>();
    fill = last;
    last = cur;
    cur = cur == (NB - 1) * STAGE ? 0 : cur + STAGE;
    half(f1, f0, cur, 0, Int0{}, IntH{}, fill, s + NB - 1);
  }
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

// Tiles that are tried, and what one round of them over the chip takes at K = 2,048, and how much of that does not grow with K (us,
// weights from memory, with rotation and cache write; two of 64 x 64 fit beside each other on a compute unit).  3,072
// columns: 2,048 rows as 128 x 192 33.9, 1,876 as 192 x 128 30.2, 1,024 as 128 x 128 23.5 and as 64 x 192 24.6, 512 as 64 x 128 18.2
// and as 64 x 64 19.8, 100 as 64 x 64 16.3.  6,144 columns at K = 4,096: 1,024 rows as 128 x 192 56.9, 512 as 128 x 128 42.0,
// 200 as 64 x 128 28.7.  The rule takes the least over the rounds that M x N has of each.
struct Tile {
  int bm, bn, per_cu;
  float us, start;
};
constexpr Tile TILES[] = {{128, 192, 1, 33.f, 9.f}, {192, 128, 1, 31.f, 5.f}, {128, 128, 1, 24.f, 5.f},
                          {64, 192, 1, 24.f, 4.f}, {64, 128, 1, 18.5f, 7.f}, {64, 64, 2, 20.f, 4.f}};

int best_tile(int M, int N, int K, int cus, float& us) {
  int best = 0;
  us = 0.f;
  for (int i = 0; i < static_cast<int>(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const Tile& t = TILES[i];
    const long tiles = static_cast<long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const long rounds = (tiles + static_cast<long>(cus) * t.per_cu - 1) / (static_cast<long>(cus) * t.per_cu);
    const float cost = rounds * (t.start + (t.us - t.start) * K / 2048.f) * (t.per_cu == 2 && tiles <= cus ? 0.82f : 1.f);
    if (i == 0 || cost < us) {
      best = i;
      us = cost;
    }
  }
  return best;
}

template <int WM, int WN, int RT, int CT, int NB>
int launch(const bf16_t* A, const bf16_t* W, bf16_t* q_out, int M, int N, int K, int lda, int ldq, const RopeEpi& rp, hipStream_t s) {
  constexpr int BM = 16 * RT * WM, BN = 16 * CT * WN;
  const int tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_tile_kernel<WM, WN, RT, CT, NB>), dim3((tm * tn + 7) / 8 * 8), dim3(WM * WN * KVF_WAVE), 0, s, A, W, q_out, M, N, K,
                     lda, ldq, tm, tn, rp);
  return kvf_last_error();
}

int launch_tile(int tile, const bf16_t* A, const bf16_t* W, bf16_t* q_out, int M, int N, int K, int lda, int ldq, const RopeEpi& rp, hipStream_t s) {
  switch (tile) {
    case 0: return launch<2, 4, 4, 3, 4>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 1: return launch<4, 2, 3, 4, 4>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 2: return launch<2, 4, 4, 2, 4>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 3: return launch<2, 4, 2, 3, 5>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 4: return launch<2, 4, 2, 2, 6>(A, W, q_out, M, N, K, lda, ldq, rp, s);
    case 5: return launch<2, 2, 2, 2, 4>(A, W, q_out, M, N, K, lda, ldq, rp, s);
  }
  return static_cast<int>(hipErrorInvalidValue);
}
}  // namespace

// Whether the fused projection takes M rows of [N, K]: where it is expected to be faster than the library's product and
// rope_kvwrite, which take 9 us, K / 285, 5.3 TB/s over the weights, 1.5 PFLOP/s, and 3.5 TB/s over 4 M N bytes (within 10% of
// what was measured at five widths and nine row counts).  Both measured, those two / this, at 3,072 x 2,048: 2,048 rows 41.6 / 32.6,
// 1,024 31.3 / 23.5, 512 23.4 / 18.0, 100 18.4 / 16.2; 1,024 x 512: 2,048 rows 16.2 / 9.4, 66 10.5 / 6.9; 6,144 x 4,096: 1,024 rows 63.3 /
// 55.6, 333 46.0 / 39.5.  Large ones with a part of a round of tiles left over stay there: 1,500 rows of 6,144 x 4,096 89 / 101,
// 2,048 of 5,120 x 3,072 77 / 82.
KVF_EXPORT int kvf_gemm_tile_qkv_takes(int M, int N, int K, int rot) {
  if (rot < 0 || rot % 8 != 0 || rot > MAX_ROT) return 0;
  if (M <= 0 || N <= 0 || N % 4 != 0 || K <= 0 || K % 64 != 0) return 0;
  float us;
  best_tile(M, N, K, compute_units(), us);
  const double two = 9.0 + K / 285.0 + 2.0 * N * K / 5.3e6 + 2.0 * M * N * K / 1.5e9 + 4.0 * M * N / 3.5e6;
  return us <= 0.97 * two;
}

// Arguments as kvf_gemm_bf16_qkv_rope with bf16 rows and tiled weights; K % 64 == 0.  tile: which of TILES, or
// -1 for the one that the rule takes.
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
  if (tile < 0) tile = best_tile(M, N, K, compute_units(), us);
  return launch_tile(tile, static_cast<const bf16_t*>(A), static_cast<const bf16_t*>(W), static_cast<bf16_t*>(q_out), M, N, K, lda, ldq, rp, s);
}
