// C[M, N] = A[M, K] * W[N, K]^T with fp32 multiply and fp32 accumulate.
// This is the matrix product of the 32-bit path and the fallback for operand types the
// bf16 MFMA kernels do not take (for instance a weight that the checkpoint stores in fp32 while
// activations are bf16).  Operands stored in bf16 are widened (exactly) before they are multiplied.
//
// Many rows of fp32 by fp32 where there are enough of them: the bf16 matrix cores over operands split in three
// (gemm_split_kernel below), whose sums are nearer to 64 bits than those of fp32 instructions.
// Many rows (a portion of a prompt) otherwise, rows of K that start on 16 bytes: tiles of 16 to 128 rows x 64
// outputs on the matrix cores with v_mfma_f32_16x16x4_f32, which multiplies and adds in fp32
// (gemm_mfma32_kernel below).  Many rows otherwise, and kept for comparison: tiles of 64 x 64
// outputs on the vector ALUs, every output summed
// over k = 0..K-1 in that order by one thread.  Few rows (decode steps), where the product is
// bound by reading W once: a wave owns one to four columns of W for all rows, its lanes walk K side by
// side with 16-byte loads (a wave reads 1 KB of a row of W at a time, several such loads in
// flight), every lane keeps a partial sum per output and the 64 partial sums are added in a fixed
// tree at the end.  Within either kernel a row's result does not depend on the number of rows, on
// the row's place in the batch or on the grid; between the kernels the order of the sums differs,
// so results agree to rounding.
//
// Output modes: 0 = store as TO;  1 = add into a fp32 matrix (the residual stream).
#include <type_traits>

#include "common.h"

namespace {
constexpr int BM = 64, BN = 64, BK = 16, TM = 4, TN = 4;

template <typename TA, typename TW, typename TO, int MODE>
__global__ __launch_bounds__(256) void gemm_tile_kernel(const TA* __restrict__ A,
                                                        const TW* __restrict__ W,
                                                        TO* __restrict__ C, int M, int N, int K,
                                                        int lda, int ldc) {
  __shared__ float As[BK][BM + 4];
  __shared__ float Ws[BK][BN + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int tr = tid / 16, tc = tid % 16;  // micro-tile rows tr*4.., cols tc*4..
  float acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;

  const int lrow = tid / 4, lk = (tid % 4) * 4;  // this thread stages 4 consecutive k of one row
  for (int k0 = 0; k0 < K; k0 += BK) {
    {
      const int m = m0 + lrow;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + lk + e;
        As[lk + e][lrow] = (m < M && k < K) ? Elem<TA>::load(A + static_cast<size_t>(m) * lda + k)
                                            : 0.f;
      }
      const int n = n0 + lrow;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + lk + e;
        Ws[lk + e][lrow] = (n < N && k < K) ? Elem<TW>::load(W + static_cast<size_t>(n) * K + k)
                                            : 0.f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float a[TM], w[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = As[kk][tr * TM + i];
#pragma unroll
      for (int j = 0; j < TN; ++j) w[j] = Ws[kk][tc * TN + j];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + tr * TM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + tc * TN + j;
      if (n >= N) continue;
      TO* c = C + static_cast<size_t>(m) * ldc + n;
      if (MODE == 1) {
        Elem<TO>::store(c, Elem<TO>::load(c) + acc[i][j]);
      } else {
        Elem<TO>::store(c, acc[i][j]);
      }
    }
  }
}

// Few rows of A (decode steps): a tile of 64 x 64 outputs would leave N / 64 workgroups to stream
// all of W.  Here a workgroup owns 16 columns and 16 rows, one output per thread, and walks K in
// steps of 64 through LDS; every output is still accumulated over k = 0..K-1 in that order by
// one thread with the same fused multiply-adds, so it has the same bits as from the kernel above.
constexpr int RN = 16, RM = 16, RK = 64;

template <typename TA, typename TW, typename TO, int MODE>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const TA* __restrict__ A,
                                                        const TW* __restrict__ W,
                                                        TO* __restrict__ C, int M, int N, int K,
                                                        int lda, int ldc) {
  __shared__ __align__(16) float As[RM][RK + 4];  // rows 16 bytes apart in banks: no conflicts
  __shared__ __align__(16) float Ws[RN][RK + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * RM, n0 = blockIdx.x * RN;
  const int r = tid / RN, c = tid % RN;          // this thread's output
  const int lrow = tid / 16, lk = (tid % 16) * 4;  // and what it stages: 4 consecutive k of a row
  // whole 16-byte loads where both operands are fp32 and every row starts on 16 bytes
  const bool vec = sizeof(TA) == 4 && sizeof(TW) == 4 && K % 4 == 0 && lda % 4 == 0 &&
                   reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0;
  float acc = 0.f;
  for (int k0 = 0; k0 < K; k0 += RK) {
    {
      const int m = m0 + lrow, n = n0 + lrow, k = k0 + lk;
      if (vec) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f), w = a;
        if (m < M && k < K) a = *reinterpret_cast<const float4*>(A + static_cast<size_t>(m) * lda + k);
        if (n < N && k < K) w = *reinterpret_cast<const float4*>(W + static_cast<size_t>(n) * K + k);
        *reinterpret_cast<float4*>(&As[lrow][lk]) = a;
        *reinterpret_cast<float4*>(&Ws[lrow][lk]) = w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          As[lrow][lk + e] = (m < M && k + e < K) ? Elem<TA>::load(A + static_cast<size_t>(m) * lda + k + e) : 0.f;
          Ws[lrow][lk + e] = (n < N && k + e < K) ? Elem<TW>::load(W + static_cast<size_t>(n) * K + k + e) : 0.f;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < RK; kk += 4) {
      const float4 a = *reinterpret_cast<const float4*>(&As[r][kk]);
      const float4 w = *reinterpret_cast<const float4*>(&Ws[c][kk]);
      acc = fmaf(a.x, w.x, acc);
      acc = fmaf(a.y, w.y, acc);
      acc = fmaf(a.z, w.z, acc);
      acc = fmaf(a.w, w.w, acc);
    }
    __syncthreads();
  }
  const int m = m0 + r, n = n0 + c;
  if (m >= M || n >= N) return;
  TO* o = C + static_cast<size_t>(m) * ldc + n;
  if (MODE == 1) {
    Elem<TO>::store(o, Elem<TO>::load(o) + acc);
  } else {
    Elem<TO>::store(o, acc);
  }
}

// ---- few rows, W streamed once: see the head of the file.
constexpr int SKC = 1024;    // elements of K per staged chunk of A
constexpr int SQ = 4 * KVF_WAVE;  // elements of K a wave reads per step (16 bytes a lane)

// four neighbouring elements: as they lie in memory, and as floats
template <typename T> struct Quad;
template <> struct Quad<float> {
  typedef float4 Raw;
  static __device__ __forceinline__ Raw raw(const float* p) { return *reinterpret_cast<const float4*>(p); }
  static __device__ __forceinline__ float4 wide(const Raw& r) { return r; }
  static __device__ __forceinline__ float4 load(const float* p) { return raw(p); }
  static __device__ __forceinline__ void store(float* p, const float (&v)[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
};
template <> struct Quad<bf16_t> {
  typedef uint2 Raw;
  static __device__ __forceinline__ Raw raw(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }
  static __device__ __forceinline__ float4 wide(const Raw& r) {
    return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u),
                       __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
  }
  static __device__ __forceinline__ float4 load(const bf16_t* p) { return wide(raw(p)); }
  static __device__ __forceinline__ void store(bf16_t* p, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(p) =
        make_uint2(static_cast<uint32_t>(f32_to_bf16(v[0])) | (static_cast<uint32_t>(f32_to_bf16(v[1])) << 16),
                   static_cast<uint32_t>(f32_to_bf16(v[2])) | (static_cast<uint32_t>(f32_to_bf16(v[3])) << 16));
  }
};

// ---- many rows on the matrix cores, true fp32.
// A workgroup of four waves owns 16 RT rows x 64 columns of outputs; a wave owns 16 of the columns, as RT tiles of
// v_mfma_f32_16x16x4_f32 with W as the first operand (lane 16 c + r supplies W[column r][k = c] and
// A[row r][k = c], and holds columns 4 c .. 4 c + 3 of row r).  K is walked in tiles of 32.  A lane reads its operands
// from LDS 16 bytes at a time, k = 16 u + 4 c .. + 3, so instruction (u, e) sums k = 16 u + e, + 4, + 8 and + 12: the
// order of the sums is fixed by K alone, whatever the tile.  Rows of A and W start on 16 bytes (8 for bf16) and K is a
// multiple of 4: the caller checks.
//
// What bounds it: the matrix cores (32 cycles an instruction, 154 TFLOP/s when nothing else is done).  A k-tile's elements
// are asked for three k-tiles ahead, two k-tiles lie in LDS, a wave holds the fragments of half a k-tile ahead, and what
// is loaded, written and read is spread among the matrix instructions one by one: with the same work ahead of them
// instead, 777 rows by 16,384 columns of 2,048 took 462 us, and now 386 (135 TFLOP/s; whole loads from 64-bit addresses
// made anew for each and 32 x 32 tiles of v_mfma_f32_32x32x2_f32 on four separate waves 451).  The other products of such
// a step: 3,072 and 2,048 x 2,048, 2,048 x 8,192: 82, 58 and 220 us, 108, 80 and 297 before.  2,048 rows: 997, 191, 127
// and 492 us (135 to 140 TFLOP/s), 1,061, 224, 149 and 564 before.
// Rows and columns past the end are read as the last and not stored.  Consecutive workgroups go to the eight XCDs in
// turn; each XCD gets an unbroken eighth of the tiles, the tiles that share columns of W side by side.
constexpr int XK = 32, XN = 64, XQ = XK / 4;   // elements of K and columns a tile, 16-byte pieces of a row
typedef float f32x4 __attribute__((ext_vector_type(4)));

// N times one matrix instruction and one of another kind, for the scheduler.
template <int N, int MASK>
__device__ __forceinline__ void spread() {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(MASK, 1, 0);
  }
}

template <typename TA, typename TW, typename TO, int MODE, int RT>
__global__ __launch_bounds__(256, 2) void gemm_mfma32_kernel(const TA* __restrict__ A,
                                                          const TW* __restrict__ W,
                                                          TO* __restrict__ C, int M, int N, int K,
                                                          int lda, int ldc) {
  constexpr int XM = 16 * RT;
  constexpr int AQ = (XM + 31) / 32, WQ = XN / 32;   // 16-byte pieces of A and W a thread stages per k-tile
  __shared__ float4 As[2][32 * AQ * XQ];
  __shared__ float4 Ws[2][XN * XQ];
  const int down = (M + XM - 1) / XM, total = down * ((N + XN - 1) / XN), share = (total + 7) / 8;
  const int at = static_cast<int>(blockIdx.x / 8), item = static_cast<int>(blockIdx.x % 8) * share + at;
  if (at >= share || item >= total) return;
  const int tid = threadIdx.x, lane = tid % KVF_WAVE, wave = tid / KVF_WAVE;
  const int m0 = item % down * XM, n0 = item / down * XN;
  const int r16 = lane % 16, kg = lane / 16;

  // two sums an output, of either half of every k-tile: shorter chains, less rounding (8,192 elements: 1.6e-6 of the
  // result against 64 bits with one, 1.1e-6 with two)
  f32x4 acc[2][RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[0][i] = acc[1][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Piece q of row r lies at 8 r + (q ^ (r / 2 % 8)).  A 16-byte access serves lanes 0-3, 12-15 and 20-27 together,
  // then 4-11, 16-19 and 28-31: either sixteen fall on all banks, written (row lane / 8, piece lane % 8) or read (row
  // lane % 16, piece 4 u + lane / 16).
  auto place = [](int row, int q) { return row * XQ + (q ^ (row / 2 % XQ)); };
  const int srow = tid / XQ, sq = tid % XQ;        // staged: elements 4 sq .. + 3 of rows srow + 32 i
  // a thread's pieces begin so many elements behind the tile's first row: 32 bits, the rest of an address is the same
  // for all threads
  uint32_t aoff[AQ], woff[WQ];
#pragma unroll
  for (int i = 0; i < AQ; ++i) aoff[i] = static_cast<uint32_t>(min(srow + 32 * i, M - 1 - m0)) * lda + 4 * sq;
#pragma unroll
  for (int i = 0; i < WQ; ++i) woff[i] = static_cast<uint32_t>(min(srow + 32 * i, N - 1 - n0)) * K + 4 * sq;
  const TA* abase = A + static_cast<size_t>(m0) * lda;
  const TW* wbase = W + static_cast<size_t>(n0) * K;
  struct Staged { typename Quad<TA>::Raw a[AQ]; typename Quad<TW>::Raw w[WQ]; };
  // WHOLE: the k-tile lies inside K.  Otherwise what lies past K is read inside the row and staged as zeros.
  auto fetch = [&](auto whole, int k0, Staged& f) {
    const int back = decltype(whole)::value ? 0 : max(k0 + 4 * sq - (K - 4), 0);
#pragma unroll
    for (int i = 0; i < AQ; ++i) f.a[i] = Quad<TA>::raw(abase + k0 + aoff[i] - back);
#pragma unroll
    for (int i = 0; i < WQ; ++i) f.w[i] = Quad<TW>::raw(wbase + k0 + woff[i] - back);
  };
  const int put_at = place(srow, sq);              // rows 32 apart are turned over alike
  auto stage = [&](auto whole, int k0, const Staged& f, int buf) {
    const bool in = decltype(whole)::value || k0 + 4 * sq < K;
    auto kept = [&](const float4& v) { return make_float4(in ? v.x : 0.f, in ? v.y : 0.f, in ? v.z : 0.f, in ? v.w : 0.f); };
#pragma unroll
    for (int i = 0; i < AQ; ++i) As[buf][put_at + 32 * XQ * i] = kept(Quad<TA>::wide(f.a[i]));
#pragma unroll
    for (int i = 0; i < WQ; ++i) Ws[buf][put_at + 32 * XQ * i] = kept(Quad<TW>::wide(f.w[i]));
  };
  struct Frags { float4 a[RT], w; };
  auto read = [&](int buf, int u, Frags& f) {
    f.w = Ws[buf][place(16 * wave + r16, 4 * u + kg)];
#pragma unroll
    for (int i = 0; i < RT; ++i) f.a[i] = As[buf][place(r16, 4 * u + kg) + 16 * XQ * i];
  };
  auto product = [&](const Frags& f, f32x4 (&sum)[RT]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float wv = e == 0 ? f.w.x : e == 1 ? f.w.y : e == 2 ? f.w.z : f.w.w;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const float av = e == 0 ? f.a[i].x : e == 1 ? f.a[i].y : e == 2 ? f.a[i].z : f.a[i].w;
        sum[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, av, sum[i], 0, 0, 0);
      }
    }
  };

  Frags f0, f1;
  Staged s0, s1;
  // One k-tile: its first fragments are in registers, the next k-tile's elements in `next` on their way.  What is read,
  // written and asked for is spread among the matrix instructions, which are what takes the time.
  auto tile = [&](auto whole, int k0, Staged& next, int buf) {
    read(buf, 1, f1);
    stage(whole, k0 + XK, next, buf ^ 1);   // its readers are past the last barrier
    fetch(whole, k0 + 3 * XK, next);
    product(f0, acc[0]);
    spread<RT + 1, 0x100>();
    spread<AQ + WQ, 0x200>();
    spread<AQ + WQ, 0x020>();
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * RT, 0);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    read(buf ^ 1, 0, f0);
    product(f1, acc[1]);
    spread<RT + 1, 0x100>();
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * RT, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::true_type WHOLE{};
  constexpr std::false_type PART{};
  fetch(PART, 0, s0);
  fetch(PART, XK, s1);
  stage(PART, 0, s0, 0);
  fetch(PART, 2 * XK, s0);
  __syncthreads();
  read(0, 0, f0);
  int k0 = 0;
#pragma unroll 1
  for (; k0 + 5 * XK <= K; k0 += 2 * XK) {
    tile(WHOLE, k0, s1, 0);
    tile(WHOLE, k0 + XK, s0, 1);
  }
#pragma unroll 1
  for (; k0 < K; k0 += 2 * XK) {
    tile(PART, k0, s1, 0);
    if (k0 + XK < K) tile(PART, k0 + XK, s0, 1);
  }
  const int n = n0 + 16 * wave + 4 * kg;
  if (n >= N) return;
  // four neighbouring columns at once where they exist and start on their size
  const bool whole = n + 4 <= N && ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % (4 * sizeof(TO)) == 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + 16 * i + r16;
    if (m >= M) continue;
    TO* c = C + static_cast<size_t>(m) * ldc + n;
    const f32x4 sum = acc[0][i] + acc[1][i];
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    if (whole) {
      if (MODE == 1) {
        const float4 old = Quad<TO>::load(c);
        v[0] += old.x; v[1] += old.y; v[2] += old.z; v[3] += old.w;
      }
      Quad<TO>::store(c, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= N) break;
        Elem<TO>::store(c + e, MODE == 1 ? Elem<TO>::load(c + e) + v[e] : v[e]);
      }
    }
  }
}

// Many rows, both operands fp32: every element is the sum of three bf16 numbers (x = h + m + l, each the rest of the one before rounded to nearest: 24
// bits but for |x| below 2^-110, whose last bits lie under the least number of the type), and the product is six products of such parts on the
// bf16 matrix cores, exact each, with fp32 sums: h h in one accumulator, h m, m h, m m, h l and l h in another (Henry, Tang and Heinecke, "Leveraging
// the bfloat16 artificial intelligence datatype for higher-precision computations", 2019).  What is left out (m l, l m, l l) is below 2^-24 of a product of
// two elements, as much as the rounding of one fp32 product at most.
//
// Against 64 bits (2-norm; this / the fp32 instruction it takes the place of): normal rows and weights, K 512 1.3e-7 / 2.9e-7, 2,048 2.7e-7 / 5.8e-7,
// 8,192 5.7e-7 / 1.1e-6, 28,672 1.1e-6 / 2.2e-6; all positive 0.7 of it; rows as they leave a gate, 0.5; all elements 1 + 2^-8 - 2^-17, which leave
// out the most, 5.9e-8 both.
// A result is in doubt that is not finite (an element that is none, or more than bf16 can round, makes its row or column NaN here), or that the
// last parts of elements below 2^-110 might change, by the largest elements of its row and column.  A wave that holds one walks along K once more with the fp32
// instruction, and results in doubt take its sums: which they are follows from their own row and column alone.  777 rows of 16,384 x 2,048 360 us, 510
// with one NaN, 960 all NaN (790 and 17,900 where lanes summed theirs one by one); of 2,048 x 8,192 200, 500 and 630.
//
// What bounds it: 777 rows of 16,384 x 2,048 take 310 us (fp32 instruction 414), 168 TFLOP/s; the matrix instructions of a stage of 128 x 128 are
// 1,536 cycles a SIMD, what splits its elements 700, reads and writes of LDS 1,500 at 128 bytes a cycle, in 2,600.  Tried: three buffers
// and the first operands read a stage ahead 328 us; four waves of 64 x 64 379; 128 x 256 a workgroup 609 (registers spilled); conversions one by one in place of pairs 370.
//
// A workgroup of eight waves takes BM = 16 RT WM rows by BN = 16 CT WN columns, 32 of K a stage.  Elements come through registers, two stages
// ahead, where they are split, into three planes of LDS, double-buffered, with one barrier a stage; splitting, reads, writes and loads stand
// between the matrix instructions.
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
constexpr int SPLIT_K = 32;

// For the scheduler: PRODUCTS matrix instructions with READS reads of LDS behind the first ones, WRITES writes and LOADS loads behind the last, and
// the vector instructions that split elements between all of them.
template <int PRODUCTS, int READS, int WRITES, int LOADS>
__device__ __forceinline__ void spread_with() {
#pragma unroll
  for (int i = 0; i < PRODUCTS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (i < READS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    if (i >= PRODUCTS - WRITES - LOADS && i < PRODUCTS - LOADS) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    if (i >= PRODUCTS - LOADS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
  }
}
// (two workgroups of the smaller tile share a compute unit: 300 rows of 16,384 x 2,048 149 us, 174 with one)
template <int WM, int WN, int RT, int CT, int MODE>
__global__ __launch_bounds__(WM * WN * KVF_WAVE, RT * CT > 4 ? WM * WN / 4 : WM * WN / 2) void gemm_split_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C,
                                                            int M, int N, int K, int lda, int ldc) {
  constexpr int TM_ = 16 * RT * WM, TN_ = 16 * CT * WN, ROWS = TM_ + TN_, PLANE = ROWS * 64, BUF = 3 * PLANE;
  constexpr int PASS = WM * WN * 8;                  // rows that are staged at a time
  constexpr int Q = ROWS / PASS, AQ = TM_ / PASS;    // 16-byte pieces a thread stages, and how many of them are of A
  static_assert(TM_ % PASS == 0 && TN_ % PASS == 0, "whole passes");
  __shared__ __attribute__((aligned(1024))) char lds[2 * BUF];
  const int down = (M + TM_ - 1) / TM_, total = down * ((N + TN_ - 1) / TN_), share = (total + 7) / 8;
  const int at = blockIdx.x / 8, item = static_cast<int>(blockIdx.x % 8) * share + at;   // an unbroken eighth for every XCD
  if (at >= share || item >= total) return;
  const int tid = threadIdx.x, lane = tid % KVF_WAVE, wave = tid / KVF_WAVE, wm = wave % WM, wn = wave / WM;
  const int r16 = lane % 16, kg = lane / 16;
  const int m0 = item % down * TM_, n0 = item / down * TN_;
  // Piece c (8 elements) of row j of sixteen lies at 4 j + c, c turned over for rows 8..15: no bank conflicts, read or written.
  auto place = [](int row, int c) { return row / 16 * 1024 + (4 * (row % 16) + (c ^ (row % 16 >= 8 ? 3 : 0))) * 16; };
  const int srow = tid / 8, sq = tid % 8;            // staged: elements 4 sq .. + 3 of rows srow + PASS i
  const int put_at = place(srow, sq / 2) + sq % 2 * 8;
  const float* src[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i)
    src[i] = i < AQ ? A + static_cast<size_t>(min(m0 + srow + PASS * i, M - 1)) * lda + 4 * sq
                    : W + static_cast<size_t>(min(n0 + srow + PASS * (i - AQ), N - 1)) * K + 4 * sq;
  struct Staged { float4 v[Q]; };
  const int stages = K / SPLIT_K;
  auto fetch = [&](int s, Staged& f) {
    const int k = min(s, stages - 1) * SPLIT_K;      // past the end the last once more, for nobody
#pragma unroll
    for (int i = 0; i < Q; ++i) f.v[i] = *reinterpret_cast<const float4*>(src[i] + k);
  };
  // of the thread's elements of each row, the largest magnitude; of A's in two chains (one: 1% slower at 777 rows of 16,384 x 2,048; two for both:
  // a register too many for two workgroups a compute unit)
  float top[Q], top2[AQ];
#pragma unroll
  for (int i = 0; i < Q; ++i) top[i] = top2[min(i, AQ - 1)] = 0.f;
  auto put = [&](const Staged& f, uint32_t buf) {
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      top[i] = fmaxf(fmaxf(top[i], fabsf(f.v[i].x)), fabsf(f.v[i].y));
      float& other = i < AQ ? top2[min(i, AQ - 1)] : top[i];
      other = fmaxf(fmaxf(other, fabsf(f.v[i].z)), fabsf(f.v[i].w));
      f32x2 x[2] = {{f.v[i].x, f.v[i].y}, {f.v[i].z, f.v[i].w}};
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        uint32_t b[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          b[p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x[p], bf16x2));
          if (part < 2) {
            x[p][0] -= __uint_as_float(b[p] << 16);
            x[p][1] -= __uint_as_float(b[p] & 0xffff0000u);
          }
        }
        *reinterpret_cast<uint2*>(lds + buf + part * PLANE + put_at + i * PASS * 64) = make_uint2(b[0], b[1]);
      }
    }
  };
  const int a_in = place(16 * wm * RT + r16, kg), w_in = place(TM_ + 16 * wn * CT + r16, kg);
  f32x4 big[RT][CT], small[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) big[r][c] = small[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Frags { bf16x8 a[RT], w[CT]; };
  auto read = [&](uint32_t plane, Frags& f) {
#pragma unroll
    for (int c = 0; c < CT; ++c) f.w[c] = *reinterpret_cast<const bf16x8*>(lds + plane + w_in + c * 1024);
#pragma unroll
    for (int r = 0; r < RT; ++r) f.a[r] = *reinterpret_cast<const bf16x8*>(lds + plane + a_in + r * 1024);
  };
  auto product = [&](const Frags& w, const Frags& a, f32x4 (&sum)[RT][CT]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) sum[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.w[c], a.a[r], sum[r][c], 0, 0, 0);
  };
  auto stage = [&](int s, Staged& staged, uint32_t buf) {
    Frags h, m, l;
    read(buf, h);
    read(buf + PLANE, m);
    read(buf + 2 * PLANE, l);
    put(staged, BUF - buf);                          // its readers are past the last barrier
    fetch(s + 3, staged);
    product(h, h, big);
    product(m, h, small);
    product(h, m, small);
    product(m, m, small);
    product(l, h, small);
    product(h, l, small);
    __builtin_amdgcn_sched_group_barrier(0x100, RT + CT, 0);
    spread_with<6 * RT * CT, 2 * (RT + CT), 3 * Q, Q>();
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
  };
  Staged s0, s1;
  fetch(0, s0);
  fetch(1, s1);
  put(s0, 0);
  fetch(2, s0);
  __syncthreads();
  int s = 0;
#pragma unroll 1
  for (; s + 1 < stages; s += 2) {
    stage(s, s1, 0);
    stage(s + 1, s0, BUF);
  }
  if (s < stages) stage(s, s1, 0);
  float* tops = reinterpret_cast<float*>(lds);       // nobody reads a stage any more
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    if (i < AQ) top[i] = fmaxf(top[i], top2[min(i, AQ - 1)]);
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) top[i] = fmaxf(top[i], __shfl_xor(top[i], o, KVF_WAVE));
    if (sq == 0) tops[srow + PASS * i] = top[i];
  }
  __syncthreads();
  // What the parts cannot hold of an element is less than 3 * 2^-126, and so is what a product of parts loses: results below 2^24 of the sum of
  // these are in doubt.  (A row or column of zeros loses nothing.)
  const float least = 0x1p-100f * K;
  const float *row_tops = tops + 16 * wm * RT + r16, *col_tops = tops + TM_ + 16 * wn * CT + 4 * kg;
  float most = 1.f, lowest = INFINITY, all = 0.f;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const f32x4 col = *reinterpret_cast<const f32x4*>(col_tops + 16 * c);
    most = fmaxf(fmaxf(fmaxf(most, col[0]), col[1]), fmaxf(col[2], col[3]));
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    most = fmaxf(most, row_tops[16 * r]);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      big[r][c] += small[r][c];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        all += fabsf(big[r][c][e]);
        lowest = fminf(lowest, fabsf(big[r][c][e]));
      }
    }
  }
  // (a launch fetches its code anew: what is seldom needed stands apart, and what asks for it is short; a prompt of 777 rows 11,740 us, 12,020 where
  // every lane tested its 32 results one by one)
  uint32_t doubt = 0;
  if (__builtin_expect(__any(!(lowest >= 3.f * least * most && all <= 3.402823466e38f)), 0)) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = fabsf(big[r][c][e]), row = row_tops[16 * r], col = col_tops[16 * c + e];
          const float lost = row > 0.f && col > 0.f ? least * (row + col + 1.f) : 0.f;
          doubt |= static_cast<uint32_t>(!(v <= 3.402823466e38f) || v < lost) << ((r * CT + c) * 4 + e);
        }
  }
  if (__builtin_expect(__any(doubt != 0), 0)) {
    // as gemm_mfma32_kernel sums, to the bit, with operands straight from memory
    const float *a_at[RT], *w_at[CT];
#pragma unroll
    for (int r = 0; r < RT; ++r) a_at[r] = A + static_cast<size_t>(min(m0 + 16 * (wm * RT + r) + r16, M - 1)) * lda + 4 * kg;
#pragma unroll
    for (int c = 0; c < CT; ++c) w_at[c] = W + static_cast<size_t>(min(n0 + 16 * (wn * CT + c) + r16, N - 1)) * K + 4 * kg;
    f32x4 sum[2][RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) sum[0][r][c] = sum[1][r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k = 0; k < K; k += XK) {
      f32x4 a[2][RT], w[2][CT];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int r = 0; r < RT; ++r) a[u][r] = *reinterpret_cast<const f32x4*>(a_at[r] + k + 16 * u);
#pragma unroll
        for (int c = 0; c < CT; ++c) w[u][c] = *reinterpret_cast<const f32x4*>(w_at[c] + k + 16 * u);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c) sum[u][r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][c][e], a[u][r][e], sum[u][r][c], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const f32x4 v = sum[0][r][c] + sum[1][r][c];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (doubt >> ((r * CT + c) * 4 + e) & 1) big[r][c][e] = v[e];
      }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int m = m0 + 16 * (wm * RT + r) + r16;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int n = n0 + 16 * (wn * CT + c) + 4 * kg;
      if (m >= M || n >= N) continue;                // N is a multiple of 4
      f32x4* to = reinterpret_cast<f32x4*>(C + static_cast<size_t>(m) * ldc + n);
      *to = MODE == 1 ? *to + big[r][c] : big[r][c];
    }
  }
}

// MT rows per workgroup (1, 2, 4, 8 or 16); SN columns of W per wave, each read DEPTH steps
// ahead, so that SN * DEPTH loads of 16 bytes are in flight per lane: narrow outputs (few
// columns, hence few waves) take one column per wave and look far ahead, wide ones four columns.
// SW waves per workgroup share the staged rows of A: with one column per wave a workgroup of four
// waves would stage all of A for four columns of W and move twice the bytes of W through LDS,
// so narrow outputs get sixteen waves per workgroup.
// The sums do not depend on MT, SN, DEPTH or SW.  Needs K % 4 == 0 and rows of A and W that start on
// 16 bytes (8 for bf16): the caller checks.
template <typename TA, typename TW, typename TO, int MODE, int MT, int SN, int DEPTH, int SW>
__global__ __launch_bounds__(SW * KVF_WAVE) void gemm_stream_kernel(
    const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ C, int M, int N, int K,
    int lda, int ldc) {
  __shared__ __align__(16) float As[MT][SKC];
  const int tid = threadIdx.x, lane = tid % KVF_WAVE, wave = tid / KVF_WAVE;
  const int n0 = (blockIdx.x * SW + wave) * SN, m0 = blockIdx.y * MT;
  float acc[MT][SN];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j) acc[i][j] = 0.f;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  // rows of W this wave reads; columns past N read row N - 1 and are dropped at the end
  const TW* wrow[SN];
#pragma unroll
  for (int j = 0; j < SN; ++j) wrow[j] = W + static_cast<size_t>(min(n0 + j, N - 1)) * K + lane * 4;

  float4 w[DEPTH][SN];   // w[t % DEPTH]: step t of this wave's walk along K
#pragma unroll
  for (int t = 0; t < DEPTH; ++t)
#pragma unroll
    for (int j = 0; j < SN; ++j) w[t][j] = t * SQ + lane * 4 < K ? Quad<TW>::load(wrow[j] + t * SQ) : zero;

  const int steps = (K + SQ - 1) / SQ;
  for (int t0 = 0; t0 < steps; t0 += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const int t = t0 + u, k = t * SQ;      // uniform
      if (k >= K) break;
      if (k % SKC == 0) {
        __syncthreads();  // the chunk before has been read by every wave
        for (int idx = tid; idx < MT * (SKC / 4); idx += SW * KVF_WAVE) {
          const int row = idx / (SKC / 4), kq = k + (idx % (SKC / 4)) * 4;
          float4 a = zero;
          if (m0 + row < M && kq < K) a = Quad<TA>::load(A + static_cast<size_t>(m0 + row) * lda + kq);
          *reinterpret_cast<float4*>(&As[row][kq - k]) = a;
        }
        __syncthreads();
      }
      float4 cur[SN];
#pragma unroll
      for (int j = 0; j < SN; ++j) cur[j] = w[u][j];
      const int ahead = k + DEPTH * SQ;
#pragma unroll
      for (int j = 0; j < SN; ++j) w[u][j] = ahead + lane * 4 < K ? Quad<TW>::load(wrow[j] + ahead) : zero;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float4 a = *reinterpret_cast<const float4*>(&As[i][k % SKC + lane * 4]);
#pragma unroll
        for (int j = 0; j < SN; ++j) {
          float v = acc[i][j];
          v = fmaf(a.x, cur[j].x, v);
          v = fmaf(a.y, cur[j].y, v);
          v = fmaf(a.z, cur[j].z, v);
          v = fmaf(a.w, cur[j].w, v);
          acc[i][j] = v;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j) {
      const float total = wave_sum(acc[i][j]);
      const int m = m0 + i, n = n0 + j;
      if (lane == 0 && m < M && n < N) {
        TO* o = C + static_cast<size_t>(m) * ldc + n;
        if (MODE == 1) {
          Elem<TO>::store(o, Elem<TO>::load(o) + total);
        } else {
          Elem<TO>::store(o, total);
        }
      }
    }
}

template <typename TA, typename TW, typename TO, int MODE, int MT>
int launch_stream(const TA* A, const TW* W, TO* C, int M, int N, int K, int lda, int ldc, hipStream_t s) {
#define GO(SN, DEPTH, SW)                                                                        \
  do {                                                                                           \
    dim3 grid((N + SN * SW - 1) / (SN * SW), (M + MT - 1) / MT);                                 \
    hipLaunchKernelGGL((gemm_stream_kernel<TA, TW, TO, MODE, MT, SN, DEPTH, SW>), grid,          \
                       dim3(SW * KVF_WAVE), 0, s, A, W, C, M, N, K, lda, ldc);                   \
  } while (0)
  // about four waves or more per compute unit's SIMD at the widest choice that allows it
  if (N >= 16384) GO(4, 2, 4);
  else if (N >= 6144) GO(2, 4, 8);
  else GO(1, 8, 16);
#undef GO
  return kvf_last_error();
}

constexpr int STREAM_MAX_M = 32;
int g_vector_alus_only = 0;   // tests: many rows through the 64 x 64 tiles of the vector ALUs

// Compute units of the current device, asked once per device.
int compute_units() {
  static int known[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (known[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    known[dev] = n;
  }
  return known[dev];
}

// Rows a tile holds of the fp32 product on the matrix cores, in sixteens: the fewest rounds of tiles over the compute
// units, a tile's time being its rows' matrix instructions and about those of another sixteen rows for the walk along
// K itself (one tile a compute unit, K 2,048: 20 us for 32 rows, 64 for 128).  Among equals the most rows, which read W
// least often.  777 rows by 16,384 columns: 386 us with the 112 rows it chooses, 394 to 437 with 32 to 128; by 2,048:
// 58, against 59 to 94.
constexpr int MFMA32_MAX_ROW = 1 << 24;
int mfma32_row_tiles(int M, int N) {
  const long cus = compute_units(), across = (N + XN - 1) / XN;
  int best = 8;
  long least = -1;
  for (int rt = 8; rt >= 1; --rt) {
    const long cost = (across * ((M + 16 * rt - 1) / (16 * rt)) + cus - 1) / cus * (rt + 1);
    if (least < 0 || cost < least) {
      least = cost;
      best = rt;
    }
  }
  return best;
}

// Tiles of the split product, and what a round of them over the chip takes at K = 2,048 (us).
struct SplitTile { int bm, bn; float us; };
constexpr SplitTile SPLIT_TILES[] = {{128, 128, 73.f}, {128, 64, 46.f}};
constexpr int SPLIT_COUNT = 2;
int g_split_tile = -1;        // tests: which of SPLIT_TILES is taken whatever the size; SPLIT_COUNT: none
// Which of SPLIT_TILES an fp32 product of many rows takes (both give the same bits), or -1: the fp32 instruction, whose tiles are smaller, up to 64 rows, where
// there are not tiles of 128 x 64 for three quarters of the compute units, and for short K.  One line in the rows for every weight, so that a row has the
// same bits among any number of rows on its side of it.  Both measured, us (fp32 / split): 777 rows of 16,384 x 2,048 414 / 310, of 2,048 x 2,048 70 /
// 55, of 2,048 x 8,192 229 / 182, of 3,072 x 2,048 87 / 77, 2,048 rows of 16,384 x 2,048 1,016 / 655, 300 of them 186 / 143, 65 rows of 128,256 x 2,048 381 /
// 343; on the other side 65 rows of 16,384 x 2,048 44 / 50, 300 rows of 2,048 x 8,192 111 / 165, 777 of 1,536 x 512 14.4 / 15.4, 48 and 64 rows of 128,256 x
// 2,048 248 and 307 / 355.  (Tiles of 32 or 64 rows and 64 columns do not move the line: 64 rows of 16,384 x 2,048 37 / 45, 300 of 2,048 x 8,192 111 / 160:
// a stage has its waits whatever the tile.)
constexpr int SPLIT_MIN_K = 512, SPLIT_MIN_M = 65;
int split_tile(int M, int N, int K) {
  if (g_split_tile >= 0) return g_split_tile < SPLIT_COUNT ? g_split_tile : -1;
  const long cus = compute_units();
  if (M < SPLIT_MIN_M || K < SPLIT_MIN_K || static_cast<long>(M) * N < cus * (128 * 64 * 3 / 4)) return -1;
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < SPLIT_COUNT; ++i) {
    const SplitTile& t = SPLIT_TILES[i];
    const long tiles = static_cast<long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const float cost = (tiles + cus - 1) / cus * t.us;
    if (i == 0 || cost < least) {
      best = i;
      least = cost;
    }
  }
  return best;
}
template <int MODE>
int launch_split(int tile, const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldc, hipStream_t s) {
  const SplitTile& t = SPLIT_TILES[tile];
  const dim3 grid(static_cast<unsigned>((static_cast<long>((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) + 7) / 8 * 8));
  if (tile == 0) hipLaunchKernelGGL((gemm_split_kernel<2, 4, 4, 2, MODE>), grid, dim3(512), 0, s, A, W, C, M, N, K, lda, ldc);
  else hipLaunchKernelGGL((gemm_split_kernel<4, 2, 2, 2, MODE>), grid, dim3(512), 0, s, A, W, C, M, N, K, lda, ldc);
  return kvf_last_error();
}

template <typename TA, typename TW, typename TO, int MODE>
int launch(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldc,
           hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  const bool quads = K % 4 == 0 && lda % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(A) % (4 * sizeof(TA)) == 0 &&
                     reinterpret_cast<uintptr_t>(W) % (4 * sizeof(TW)) == 0;
  if (M <= STREAM_MAX_M && quads) {
    const TA* a = static_cast<const TA*>(A);
    const TW* w = static_cast<const TW*>(W);
    TO* c = static_cast<TO*>(C);
    if (M == 1) return launch_stream<TA, TW, TO, MODE, 1>(a, w, c, M, N, K, lda, ldc, s);
    if (M == 2) return launch_stream<TA, TW, TO, MODE, 2>(a, w, c, M, N, K, lda, ldc, s);
    if (M <= 4) return launch_stream<TA, TW, TO, MODE, 4>(a, w, c, M, N, K, lda, ldc, s);
    if (M <= 8) return launch_stream<TA, TW, TO, MODE, 8>(a, w, c, M, N, K, lda, ldc, s);
    return launch_stream<TA, TW, TO, MODE, 16>(a, w, c, M, N, K, lda, ldc, s);
  }
  if (M <= 2 * RM) {
    dim3 rows_grid((N + RN - 1) / RN, (M + RM - 1) / RM);
    hipLaunchKernelGGL((gemm_rows_kernel<TA, TW, TO, MODE>), rows_grid, dim3(256), 0, s,
                       static_cast<const TA*>(A), static_cast<const TW*>(W), static_cast<TO*>(C), M,
                       N, K, lda, ldc);
    return kvf_last_error();
  }
  if constexpr (std::is_same_v<TA, float> && std::is_same_v<TW, float> && std::is_same_v<TO, float>) {
    if (quads && K >= SPLIT_K && K % SPLIT_K == 0 && N % 4 == 0 && ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0 && !g_vector_alus_only) {
      const int tile = split_tile(M, N, K);
      if (tile >= 0)
        return launch_split<MODE>(tile, static_cast<const float*>(A), static_cast<const float*>(W), static_cast<float*>(C), M, N, K, lda, ldc, s);
    }
  }
  // (its loads need an element of K to be clamped to, and a tile's rows within 32 bits of each other)
  if (quads && K > 0 && K < MFMA32_MAX_ROW && lda < MFMA32_MAX_ROW && !g_vector_alus_only) {
#define TILES(RT)                                                                                \
  case RT: {                                                                                     \
    const int total = ((N + XN - 1) / XN) * ((M + 16 * RT - 1) / (16 * RT));                     \
    hipLaunchKernelGGL((gemm_mfma32_kernel<TA, TW, TO, MODE, RT>), dim3((total + 7) / 8 * 8),    \
                       dim3(256), 0, s, static_cast<const TA*>(A), static_cast<const TW*>(W),    \
                       static_cast<TO*>(C), M, N, K, lda, ldc);                                  \
    break;                                                                                       \
  }
    switch (mfma32_row_tiles(M, N)) {
      TILES(1) TILES(2) TILES(3) TILES(4) TILES(5) TILES(6) TILES(7) TILES(8)
    }
#undef TILES
    return kvf_last_error();
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  hipLaunchKernelGGL((gemm_tile_kernel<TA, TW, TO, MODE>), grid, dim3(256), 0, s,
                     static_cast<const TA*>(A), static_cast<const TW*>(W), static_cast<TO*>(C), M,
                     N, K, lda, ldc);
  return kvf_last_error();
}
}  // namespace

// For tests that compare the two many-row kernels: nonzero keeps products of many rows on the
// vector ALUs.  Returns the setting before.
KVF_EXPORT int kvf_gemm_generic_vector_alus_only(int on) {
  const int before = g_vector_alus_only;
  g_vector_alus_only = on;
  return before;
}

// For tests: which tile of the split product fp32 products of many rows take (0, 1), none (2), or the one that their size asks
// for (-1).  Returns the setting before.
KVF_EXPORT int kvf_gemm_generic_split_tile(int tile) {
  const int before = g_split_tile;
  g_split_tile = tile;
  return before;
}

// Which tile of the split product M fp32 rows of [N, K] take, or -1.
KVF_EXPORT int kvf_gemm_generic_split_takes(int M, int N, int K) { return split_tile(M, N, K); }

// a_type / w_type: 0 = fp32, 1 = bf16.  out_mode: 0 = store in a_type... see table below.
//   out_kind 0: store fp32      out_kind 1: store bf16      out_kind 2: add into fp32
KVF_EXPORT int kvf_gemm_generic(const void* A, int a_type, const void* W, int w_type, void* C,
                                int out_kind, int M, int N, int K, int lda, int ldc,
                                hipStream_t s) {
#define CASE(AT, WT, TA, TW)                                                                      \
  if (a_type == AT && w_type == WT) {                                                             \
    if (out_kind == 0) return launch<TA, TW, float, 0>(A, W, C, M, N, K, lda, ldc, s);            \
    if (out_kind == 1) return launch<TA, TW, bf16_t, 0>(A, W, C, M, N, K, lda, ldc, s);           \
    if (out_kind == 2) return launch<TA, TW, float, 1>(A, W, C, M, N, K, lda, ldc, s);            \
  }
  CASE(0, 0, float, float)
  CASE(0, 1, float, bf16_t)
  CASE(1, 0, bf16_t, float)
  CASE(1, 1, bf16_t, bf16_t)
#undef CASE
  return static_cast<int>(hipErrorInvalidValue);
}
