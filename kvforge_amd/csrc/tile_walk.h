// Products of many rows in tiles: how a workgroup of gemm_tile.hip walks along K.
//
// A workgroup of WM x WN waves takes tiles of BM = 16 RT WM rows by BN = 16 CT WN columns (rows of a weight in the tiled form of
// gemm_bf16.hip), 32 of K a stage.  Rows and weights go from memory straight into LDS without passing through
// registers: weights by stages, NW of them side by side, rows by pairs of stages, NA pairs, because a compute unit asks for
// whole lines of 128 bytes (by stages, 64 bytes a row, 2,048 x 4,096 x 8,192 takes 136 us in place of 112).  A stage has one
// barrier, at its beginning: the next stage's operands have arrived by then and are read beside this one's products (their
// registers alternate), and the loads that take the place of what was read in the stage before are asked for, one by one between
// products: asked for in one go they block the waves for as long as a product of the stage takes.
//
// A workgroup that takes several tiles does not stop between them: the loads run on into the next tile (Source says
// where it lies) while the last stages of one are multiplied and while its results are stored, and the first stages of a tile do
// not wait for the stores before them.  No load stands under a condition: the last stages of the last tile, behind which nothing is
// asked for, are code of their own.
//
// What bounds it: 2,048 x 16,384 x 2,048 in tiles of 256 x 256 takes 107 us (1.28 PFLOP/s).  Its matrix instructions alone are 65 at the 2.0
// GHz that the chip holds under them; with the loads left out it took 18 us less, with the reads of LDS left out 8, with
// both left out, 28.  About 10 us are the results' way out, two tiles one behind the other.  Small tiles are bound by what comes out of
// L2: about 14 TB/s over the chip.  The instruction of 32 x 32 x 16 in place of 16 x 16 x 32, which reads a third less
// from registers, was 5% slower.
#pragma once
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
// At most N of the wave's own loads are still on their way, its reads of LDS are done, and the other waves have come as far.
template <int N> __device__ __forceinline__ void loads_left() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

template <int WM_, int WN_, int RT_, int CT_, int NA_>
struct Walk {
  static constexpr int WM = WM_, WN = WN_, RT = RT_, CT = CT_, NA = NA_, NW = 2 * NA;
  static constexpr int WAVES = WM * WN, THREADS = WAVES * KVF_WAVE, BM = 16 * RT * WM, BN = 16 * CT * WN;
  static constexpr int AC = BM / 8, WC = BN / 16;                     // KB: 8 rows of 128 bytes (two stages), 16 weight rows of 64
  static constexpr int AL = AC / WAVES, WL = (WC + WAVES - 1) / WAVES;   // of a wave (where WC does not divide, the last KB several times)
  static constexpr uint32_t ROWS = AC * 1024, WEIGHTS = WC * 1024, W0 = NA * ROWS, BYTES = W0 + NW * WEIGHTS;
  static_assert(AC % WAVES == 0 && NA >= 2, "a wave asks for whole KB of rows, one pair ahead of that in use");
  struct Frags { bf16x8 a[RT], w[CT]; };

  // Stage t asks for the weights of stage t + NW and, if it is odd, ahead of those for the rows of the pair (t - 1) / 2 + NA.
  // How many loads may be on their way at the beginning of stage h, which reads the operands of stage h + 1; `odd`: h is.
  static constexpr int asked(int t) { return WL + (t % 2 != 0 ? AL : 0); }
  static constexpr int between(int from, int to) {
    int n = 0;
    for (int t = from; t <= to; ++t) n += asked(t);
    return n;
  }
  static constexpr int in_flight(bool odd, int last) {   // `last`: the last stage that asked, of an even h = 64 or the odd one behind it
    const int h = 64 + (odd ? 1 : 0), weights = between(h + 2 - NW, last), rows = WL + between(h + 3 - NW, last);
    return odd && rows < weights ? rows : weights;
  }
  static constexpr int in_flight(bool odd) { return in_flight(odd, odd ? 64 : 63); }
  static constexpr int ARRIVED = NW - 1;   // stages whose next operands have been asked for before a tile begins

  const char* lds;
  int lane, wave, wm, wn;
  int left_a, left_w;              // pairs and stages that are still to be asked for where the loads are now
  uint32_t lds0, a_nxt, w_nxt, a_fill, w_fill;
  int a_at, x0, w_at;
  const char *rows_at, *weights_at;
  uint32_t a_off[AL], w_off[WL];
  Frags f0, f1;
  f32x4 acc[RT][CT];

  // Loads of rows now come from base + off(row of the tile), S / 2 pairs of stages; of weights from base + off(group of 16 of the tile's
  // columns), S stages; offsets in bytes.  Piece c (8 elements) of a row lies at place c ^ row % 8 of its 128 bytes: reads of fragments
  // are free of bank conflicts.
  template <class Off> __device__ __forceinline__ void aim_rows(const char* base, const Off& off, int S) {
    rows_at = base;
#pragma unroll
    for (int i = 0; i < AL; ++i) a_off[i] = off((wave * AL + i) * 8 + lane / 8) + ((lane % 8) ^ (lane / 8)) * 16;
    left_a = S / 2;
  }
  template <class Off> __device__ __forceinline__ void aim_weights(const char* base, const Off& off, int S) {
    weights_at = base;
#pragma unroll
    for (int i = 0; i < WL; ++i) w_off[i] = off(min(wave * WL + i, WC - 1)) + lane * 16;
    left_w = S;
  }

  __device__ __forceinline__ void ask_rows(int i) { load_to_lds(rows_at, a_off[i], lds0 + a_fill + (wave * AL + i) * 1024); }
  __device__ __forceinline__ void ask_weights(int i) { load_to_lds(weights_at, w_off[i], lds0 + W0 + w_fill + min(wave * WL + i, WC - 1) * 1024); }
  __device__ __forceinline__ void rows_asked() {
    rows_at += 128;
    a_fill = a_fill == (NA - 1) * ROWS ? 0 : a_fill + ROWS;
  }
  __device__ __forceinline__ void weights_asked() {
    weights_at += 1024;
    w_fill = w_fill == (NW - 1) * WEIGHTS ? 0 : w_fill + WEIGHTS;
  }

  // operand i of half h of the pair at a_nxt and the stage at w_nxt
  __device__ __forceinline__ void read(Frags& f, int i, int h) {
    if (i < CT) f.w[i < CT ? i : 0] = *reinterpret_cast<const bf16x8*>(lds + W0 + w_nxt + w_at + i * 1024);
    else f.a[i >= CT ? i - CT : 0] = *reinterpret_cast<const bf16x8*>(lds + a_nxt + (a_at + (x0 ^ (h * 64))) + (i - CT) * 2048);
  }
  // what is read next; h: the half that was read
  __device__ __forceinline__ void read_on(int h) {
    w_nxt = w_nxt == (NW - 1) * WEIGHTS ? 0 : w_nxt + WEIGHTS;
    if (h == 1) a_nxt = a_nxt == (NA - 1) * ROWS ? 0 : a_nxt + ROWS;
  }

  // src.rows and src.weights aim at the first tile, then at the next ones.  FEW: a tile may have fewer than NW + 2 stages (S of
  // them): what is past them is asked for from its last ones, for nobody.  (Without FEW there are no branches here: each
  // would be a trip to memory for instructions, 3 us a launch.)
  template <bool FEW, class Source>
  __device__ __forceinline__ void start(const char* shared, int S, Source& src) {
    lds = shared;
    lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u32*)shared));
    lane = threadIdx.x % KVF_WAVE;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVF_WAVE);
    wm = wave % WM;
    wn = wave / WM;
    const int r16 = lane % 16, kg = lane / 16;
    a_at = wm * RT * 2048 + (r16 / 8) * 1024 + (r16 % 8) * 128;
    x0 = (kg ^ (r16 % 8)) * 16;
    w_at = wn * CT * 1024 + lane * 16;
    a_nxt = w_nxt = a_fill = w_fill = 0;
    src.rows(*this);
    src.weights(*this);
#pragma unroll
    for (int t = 0; t < NW; ++t) {            // what stages -NW to -1 would have asked for
      if (t % 2 == 1) {
#pragma unroll
        for (int i = 0; i < AL; ++i) ask_rows(i);
        rows_asked();
        if (FEW && t + 1 >= S) rows_at -= 128;
      }
#pragma unroll
      for (int i = 0; i < WL; ++i) ask_weights(i);
      weights_asked();
      if (FEW && t + 1 >= S) weights_at -= 1024;
    }
    left_a -= NA;
    left_w -= NW;
    if constexpr (FEW) loads_left<0>();
    else loads_left<in_flight(true)>();
#pragma unroll
    for (int i = 0; i < RT + CT; ++i) read(f0, i, 0);
    read_on(0);
  }

  // Stage h of a tile, H its parity: its products, from f; the next stage's operands go to g (READ), and later ones are asked for (ASK).
  template <int H, bool READ, bool ASK>
  __device__ __forceinline__ void products(const Frags& f, Frags& g) {
    constexpr int PR = RT * CT, RD = READ ? RT + CT : 0, LOADS = !ASK ? 0 : H == 1 ? AL + WL : WL;
    __builtin_amdgcn_sched_barrier(0);
    int rd = 0, ld = 0;
#pragma unroll
    for (int p = 0; p < PR; ++p) {
#pragma unroll
      for (; rd < RD && rd < ((p + 1) * RD * 3 + 2 * PR - 1) / (2 * PR); ++rd) read(g, rd, 1 - H);
      __builtin_amdgcn_sched_barrier(0);
      acc[p / CT][p % CT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[p % CT], f.a[p / CT], acc[p / CT][p % CT], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (; ld < LOADS && ld < (p + 1) * LOADS / PR; ++ld) {
        if (H == 1 && ld < AL) ask_rows(ld < AL ? ld : 0);
        else ask_weights(H == 1 ? ld - AL : ld);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (READ) read_on(1 - H);
  }
  // `arrived`: the next stage's operands are known to be in LDS (this wave's part of them).
  template <int H, bool LAST, class Source>
  __device__ __forceinline__ void stage(const Frags& f, Frags& g, bool arrived, Source& src) {
    if (arrived) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else loads_left<in_flight(H == 1)>();
    products<H, true, true>(f, g);
    if (H == 1) {
      rows_asked();
      if (!LAST && --left_a == 0) src.rows(*this);
    }
    weights_asked();
    if (!LAST && --left_w == 0) src.weights(*this);
  }
  // The last NW stages of the last tile, behind which nothing is asked for.
  template <int J>
  __device__ __forceinline__ void last_stages() {
    if constexpr (J < NW) {
      constexpr bool odd = J % 2 == 1, more = J + 1 < NW;
      if constexpr (more) loads_left<in_flight(odd, 64 + odd - 1 - J)>();
      products<J % 2, more, false>(odd ? f1 : f0, odd ? f0 : f1);
      last_stages<J + 1>();
    }
  }

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // A tile: S stages, an even number of at least NW + 2.  LAST: no tile comes behind it (a constant: where both ways meet, registers
  // are copied or spilled).  `first`: nothing was stored since start().
  template <bool LAST, class Source>
  __device__ __forceinline__ void run(int S, bool first, Source& src) {
    clear();
    const int arrived = first ? 0 : ARRIVED;   // settle() has seen them arrive
    const int asks = LAST ? S - NW : S;
#pragma unroll 1
    for (int s = 0; s < asks; s += 2) {
      stage<0, LAST>(f0, f1, s < arrived, src);
      stage<1, LAST>(f1, f0, s + 1 < arrived, src);
    }
    if constexpr (LAST) last_stages<0>();
    else settle();
  }
  // The only tile, of fewer stages, all of which have arrived (start<true>).
  __device__ __forceinline__ void run_few(int S) {
    clear();
#pragma unroll 1
    for (int s = 0; s < S; s += 2) {
      products<0, true, false>(f0, f1);
      products<1, true, false>(f1, f0);
    }
  }

  // Ahead of a tile's stores: every load of the wave has arrived.  (Behind the last stages they have.)
  __device__ __forceinline__ static void settle() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
};

// A wave's own place in LDS where 16 rows of PIECES pieces of 16 bytes are turned from fragments into rows.  A row's
// pieces are mixed by its number against bank conflicts.
template <int PIECES> struct OwnRows {
  static_assert((PIECES & (PIECES - 1)) == 0, "pieces are mixed by the bits of a row's number");
  static constexpr int PITCH = PIECES * 16, BYTES = 16 * PITCH;
  __device__ __forceinline__ static int place(int row, int piece) { return row * PITCH + (piece ^ (row & (PIECES - 1))) * 16; }
  // go(row, piece, its 16 bytes) for all of them, 64 at a time
  template <class Go> __device__ __forceinline__ static void each(const char* own, int lane, const Go& go) {
#pragma unroll
    for (int i = 0; i < (16 * PIECES + KVF_WAVE - 1) / KVF_WAVE; ++i) {
      const int at = lane + i * KVF_WAVE;
      if (16 * PIECES % KVF_WAVE == 0 || at < 16 * PIECES)
        go(at / PIECES, at % PIECES, *reinterpret_cast<const uint4*>(own + place(at / PIECES, at % PIECES)));
    }
  }
};
}  // namespace
