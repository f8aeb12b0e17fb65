// C[M, N] = A[M, K] * W[N, K]^T for bf16 weights on the matrix cores (fp32 accumulation),
// built for few rows of A: the weight matrix is streamed once per pass of up to 16*MT rows and
// the kernel is bound by HBM, so all of the chip has to pull on W at once.
//
// One workgroup owns 16 rows of W (16 output columns).  Its waves split K: wave w takes the
// 32-wide k-steps w, w + nw, w + 2nw, ... so neighbouring waves read neighbouring 64-byte pieces
// of the same rows.  Per k-step a lane loads 16 B of W (row lane%16, k-offset 8*(lane/16)) and
// the matching 8 elements of each 16-row tile of A and issues one v_mfma_f32_16x16x32_bf16 per
// tile with W as the first operand, so a lane ends up holding four consecutive output columns of
// one row of C.  Partial sums of the waves are added in wave order through LDS.  With several
// row tiles of A (more than 16 rows) a wave takes NT neighbouring 16-row groups of W per k-step
// and reuses its A fragments for them, which divides the traffic for A (served by L2) by NT.
// The launch shape depends on N, K and on how many 16-row tiles a pass holds (1, 2, 4 or 8),
// never on the rows themselves.
//
// Left operand (AT): 0 = bf16 activations; 1 = the fp32 residual stream with the RMS norm folded
// in: y = x * rsqrt(mean(x^2) + eps) is applied as a per-row factor on the accumulators (the
// norm's weight vector is folded into W's columns when the model is loaded); the sum of squares
// is taken in fp32 from the same loads that feed the matrix cores.
//
// Epilogues (EPI): 0 store fp32; 1 store bf16; 2 add into fp32 (the residual stream);
// 3 SwiGLU gate: columns come in (gate, up) pairs, out[m, j] = silu(c[2j]) * c[2j+1] as bf16;
// 4 rotary + cache write for a fused q/k/v projection: neighbouring columns of q and k heads are
//   rotary pairs; rotated q goes to the output (bf16, q heads only), rotated k and plain v go
//   straight into the pages of the token's sequence (K pages [nb, KV, block, d], V pages
//   transposed [nb, KV, d, block]).
// 5 greedy pick for the output head of a decode step (at most 16 bf16 rows, already normalised:
//   with the norm folded in, each of the head's thousands of workgroups would read the fp32 rows
//   and their sums of squares again, as many bytes as the matrix itself): no logits are stored;
//   every workgroup leaves the best (value, column) of its columns per row in a workspace and
//   takes a ticket, and the workgroup that takes the last one picks every row's best over all
//   workgroups (the lowest column among equal values), then does what the step's tail would
//   need kernels of their own for: it hands the tokens out, makes each sequence's token its
//   next input (token id, position and context length move on by one), keeps the tokens in the
//   ring row of this step for the host, and writes the tokens' embedding rows into the residual
//   stream for the next step.
// K must be a multiple of 8 (16-byte loads); a k-step that passes K loads zeros.
//
// A product that is added to a narrow C over a long K (the down projection) has fewer workgroups
// than the chip has compute units, and a compute unit keeps only so many bytes in flight.  It
// may be cut into two halves of K (`Riders::half_out`): a second layer of workgroups stores its
// half beside C (rounded to bf16, as a product that is stored is), and the caller owes that half
// to C.  The next consumers add it on their way:
// the fused q/k/v projection in its loads (`a_add`), the output projection in its sum (`c_add`).
//
// Layout of W.  In the checkpoint's row-major [N, K] a wave's load of one operand fragment
// touches 16 rows, 64 bytes each: 16 cache lines per group of 16 lanes, and the L1 looks lines up
// one at a time, which bounds the kernel far below what HBM delivers.  The engine therefore also
// keeps W in tiles (`w_tiled`): [ceil(N/16)][ceil(K/32)][64 lanes][8 elements], tile (g, s) being
// rows 16g..16g+15, columns 32s..32s+31 in the order the instruction wants them (lane
// 16*c + r holds row r, columns 8c..8c+7), zero-padded.  A fragment is then 1 KB of consecutive
// bytes.  Both layouts give the same bits.
#include "gemm_common.h"

namespace {
// Sums that ride along, all bf16 (a workgroup of the fused projection reads every row of A and
// of a_add: with the addend in fp32 that was as many bytes again as A, 1.8 us of a 8.6 us kernel
// at eight rows).  `a_add` (kernels built with ADD): the left operand is A + a_add, A in fp32,
// the same row stride counted in elements.  `c_add` (with EPI 2): C += product + c_add, row
// stride of C.
// `half_out` (with EPI 2): the grid is two deep; workgroups of the second layer walk the second
// half of K and store their product there (fp32, row stride of C) instead of adding it to C, so
// that a narrow C still puts a workgroup on every compute unit; the caller owes half_out to C.
struct Riders {
  const bf16_t* a_add;
  const bf16_t* c_add;
  bf16_t* half_out;
};

// Operands of the greedy pick (EPI 5).  part_val / part_idx: [16][workgroups] and behind them
// [16][PICK_LANES] scratch; ticket:
// PICK_TICKET_INTS ints, zero between launches (atomics on one address are served one after the
// other, some 65 ns each on this chip, and thousands of workgroups on one counter would queue
// for longer than the product takes: the workgroups are spread over PICK_LANES counters, a
// cache line apart, and the last arrival at each takes a ticket of a second counter).  tokens: [M] out.  token_ids / positions / ctx_lens: the step's
// inputs, advanced in place; ring [ring_rows][ring_stride] and run_counter as decode_advance
// takes them.  embed [vocab][hidden] bf16 -> residual [M][ld_res] fp32 for the next step.
struct PickEpi {
  float* part_val;
  int* part_idx;
  int* ticket;
  int* tokens;
  int* token_ids;
  int* positions;
  int* ctx_lens;
  int* ring;
  int* run_counter;
  const bf16_t* embed;
  float* residual;
  int ring_stride, ring_rows, hidden, ld_res;
};

constexpr int PICK_LANES = 64, PICK_STRIDE = 16;   // counters, and ints between two of them
constexpr int PICK_TICKET_INTS = (PICK_LANES + 1) * PICK_STRIDE;

// True in the caller (one thread asks) that arrives last of `expected` at `counter`, which it
// leaves zero.  Every caller has made its results visible before.
__device__ __forceinline__ bool pick_last_at(int* counter, int expected) {
  if (atomicAdd(counter, 1) != expected - 1) return false;
  __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
  return v > bv || (v == bv && i < bi);
}

// Results that other workgroups are going to read are stored past this XCD's L2 (an atomic store
// at device scope is written through); before a ticket is taken they have to be complete.
// A device-scope release fence would also write the whole L2's dirty lines back, and thousands
// of workgroups doing that made the head's product take 275 us instead of 90.  What orders the
// results before the ticket instead: every wave that published waits until its stores have been
// acknowledged (the vector memory counter at zero: a written-through store is acknowledged from
// where the device's other L2s read it), then comes the workgroup's barrier, and only then does
// thread 0 add to the ticket.  A fence of workgroup scope alone would not do: it lets stores to
// global memory stay in flight, since all waves of a workgroup share one L1.
__device__ __forceinline__ void pick_publish(float* val, int* idx, size_t at, float v, int i) {
  __hip_atomic_store(val + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(idx + at, i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void pick_stores_done() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The last arrival at counter `lane`: the best per row over the workgroups lane, lane + 64, ...
// into the second level of the scratch ([16][PICK_LANES] behind the first).  All threads of the
// workgroup; plain loads after the caller's acquire fence.
__device__ __forceinline__ void pick_merge_lane(const PickEpi& pk, int M, int groups, int lane) {
  const int tid = threadIdx.x, sub = tid % 32;    // 32 threads per row, rows in turn
  for (int row = tid / 32; row < 16; row += blockDim.x / 32) {   // the same trips in every thread
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    if (row < M) {
      for (int c = lane + sub * PICK_LANES; c < groups; c += 32 * PICK_LANES) {
        const float v = pk.part_val[row * groups + c];
        const int i = pk.part_idx[row * groups + c];
        if (better(v, i, bv, bi)) { bv = v; bi = i; }
      }
    }
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, KVF_WAVE);
      const int oi = __shfl_xor(bi, o, KVF_WAVE);
      if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
    }
    if (sub == 0 && row < M)
      pick_publish(pk.part_val + 16 * groups, pk.part_idx + 16 * groups, row * PICK_LANES + lane, bv, bi);
  }
  pick_stores_done();
}

// The last workgroup of a greedy pick: see EPI 5 at the head of the file.  `lds` holds at least
// 16 ints.
__device__ __forceinline__ void pick_finish(const PickEpi& pk, int M, int groups, float* lds) {
  const int tid = threadIdx.x;
  const int lanes = groups < PICK_LANES ? groups : PICK_LANES;
  int* tok = reinterpret_cast<int*>(lds);   // [16]
  // 16 threads per row over the second level's (at most 64) candidates, rows in turn
  for (int row = tid / 16; row < 16; row += blockDim.x / 16) {
    const int sub = tid % 16;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    if (row < M) {
      for (int c = sub; c < lanes; c += 16) {
        const float v = pk.part_val[16 * groups + row * PICK_LANES + c];
        const int i = pk.part_idx[16 * groups + row * PICK_LANES + c];
        if (better(v, i, bv, bi)) { bv = v; bi = i; }
      }
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, KVF_WAVE);
      const int oi = __shfl_xor(bi, o, KVF_WAVE);
      if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
    }
    if (sub == 0 && row < M) tok[row] = bi == 0x7fffffff ? 0 : bi;
  }
  const int step = *pk.run_counter;   // read by every thread before it moves
  __syncthreads();
  if (tid < M) {
    const int t = tok[tid];
    pk.tokens[tid] = t;
    if (step >= 0 && step < pk.ring_rows) pk.ring[step * pk.ring_stride + tid] = t;
    if (pk.ctx_lens[tid] > 0) {     // padding sequences stay empty
      pk.token_ids[tid] = t;
      pk.positions[tid] += 1;
      pk.ctx_lens[tid] += 1;
    }
  }
  if (tid == 0) *pk.run_counter = step + 1;
  __syncthreads();
  // the tokens' embedding rows, widened, are the next step's residual stream
  const int per_row = pk.hidden / 8;
  for (int idx = tid; idx < M * per_row; idx += blockDim.x) {
    const int r = idx / per_row, k = (idx - r * per_row) * 8;
    float v[8];
    load8(pk.embed + static_cast<size_t>(tok[r]) * pk.hidden + k, v);
    float* dst = pk.residual + static_cast<size_t>(r) * pk.ld_res + k;
    *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(dst + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
}

__device__ __forceinline__ bf16x8 load_frag(const bf16_t* p, bool ok) {
  uint4 r = make_uint4(0u, 0u, 0u, 0u);
  if (ok) r = *reinterpret_cast<const uint4*>(p);
  return __builtin_bit_cast(bf16x8, r);
}

template <bool STREAMED> __device__ __forceinline__ bf16x8 load_weight(const bf16_t* p, bool ok) {
  uint4 r = make_uint4(0u, 0u, 0u, 0u);
  if (ok) r = load_16<STREAMED>(p);
  return __builtin_bit_cast(bf16x8, r);
}

// Whether a matrix in tiles goes past the caches: one launch of few rows reads each of its bytes once, in whole lines, so
// nothing is lost where it cannot lie there from the last step, and what can (activations, keys and values) stays.
// Eight rows (us, cached and streamed): output head of 525 MB 89.5 and 76.6, gated pair of 67 MB 15.3 and 14.6, q/k/v
// of 12.6 MB 8.4 and 7.8 and the attention behind them 8.8 and 7.7; 41 rows over 12.6 MB 11.3 and 10.3.  The line is at what
// an XCD's L2 holds: the matrices of a decoder 512 wide (0.5 to 2.9 MB), which do lie in the caches, took 0.2 to 0.6 us longer
// streamed, one of 8 MB the same.  (gemm_mid_kernel, whose workgroups share lines: 15.7 and 16.9, so it does not.)  A matrix of
// a model that lies in the last-level cache as a whole does come from there the next step: the caller says so (CACHED), see
// StreamedWeight.
constexpr long STREAM_BYTES = 4l << 20;
constexpr int CACHED = 2;          // w_tiled: in tiles, and through the caches whatever its size
constexpr int GROUP_CACHED = 8;    // the same in an item of a launch of several
__host__ __device__ inline bool streams(int N, int K) { return 2l * N * K >= STREAM_BYTES; }

// 8 fp32 (with ADD plus 8 of `q`) -> 8 bf16 (round to nearest even); adds their squares to ss.
// Nothing inside the branches uses what they load, so no branch ends in a wait and the loads of
// a whole pass stay in flight together.
template <bool ADD>
__device__ __forceinline__ bf16x8 load_frag_f32(const float* p, const bf16_t* q, bool ok, float& ss) {
  typedef __attribute__((ext_vector_type(8))) float f32x8;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  uint4 raw = make_uint4(0u, 0u, 0u, 0u);   // eight bf16 of q, widened after the branch
  if (ok) {
    load8(p, v);
    if (ADD) raw = *reinterpret_cast<const uint4*>(q);
  }
  const float w[8] = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u),
                      __uint_as_float(raw.y << 16), __uint_as_float(raw.y & 0xffff0000u),
                      __uint_as_float(raw.z << 16), __uint_as_float(raw.z & 0xffff0000u),
                      __uint_as_float(raw.w << 16), __uint_as_float(raw.w & 0xffff0000u)};
  f32x8 x;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float t = ADD ? v[i] + w[i] : v[i];
    ss = fmaf(t, t, ss);
    x[i] = t;
  }
  return __builtin_convertvector(x, bf16x8);
}

// What an epilogue reads besides the accumulators.  With one row tile the lanes of wave 0 finish
// the workgroup's tile and know their row and columns from the start, so they ask for these
// operands before the walk over K and find them in registers afterwards, instead of paying
// their latencies (up to three dependent loads for the cache write) at the end.
struct EpiOperands {
  f32x4 c;            // EPI 2: the four values the product is added to
  int pos, page;      // EPI 4: the token's position; the page its key and value go to (or -1)
  float cs[2], sn[2]; // EPI 4: rotation of the lane's two pairs
  bool have;
};

// 16-byte accesses to C are possible where rows and base are aligned and all four columns exist
__device__ __forceinline__ bool vec4_ok(const void* Cv, int ldc, int n, int N, int elem) {
  return n + 3 < N && (ldc * elem) % 16 == 0 && n % 4 == 0 &&
         reinterpret_cast<uintptr_t>(Cv) % 16 == 0;
}

// First stage: loads that need only (m, n).
template <int EPI>
__device__ __forceinline__ void epi_prefetch_a(EpiOperands& op, int m, int n, int N, int ldc, const void* Cv,
                                               const bf16_t* c_add, const RopeEpi& rp) {
  op.have = true;
  if (EPI == 2) {
    const size_t idx = static_cast<size_t>(m) * ldc + n;
    const float* c = static_cast<const float*>(Cv) + idx;
    if (vec4_ok(Cv, ldc, n, N, 4) && vec4_ok(c_add, ldc, n, N, 2)) {
      op.c = *reinterpret_cast<const f32x4*>(c);
      if (c_add) {
        const uint2 packed = *reinterpret_cast<const uint2*>(c_add + idx);
        op.c += f32x4{__uint_as_float(packed.x << 16), __uint_as_float(packed.x & 0xffff0000u),
                      __uint_as_float(packed.y << 16), __uint_as_float(packed.y & 0xffff0000u)};
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        op.c[r] = n + r < N ? c[r] + (c_add ? bf16_to_f32(c_add[idx + r].bits) : 0.f) : 0.f;
    }
  }
  if (EPI == 4) {
    op.pos = rp.positions[m];
    op.page = rp.write_kv ? rp.seq_of_token[m] : -1;  // the sequence for now
  }
}
// Second stage: loads that need what the first brought (position -> angles, sequence -> page).
template <int EPI>
__device__ __forceinline__ void epi_prefetch_b(EpiOperands& op, int n, const RopeEpi& rp) {
  if (EPI != 4) return;
  const int head = n / rp.d, e = n - head * rp.d;
  const int p = op.pos;
  const bool pos_ok = p >= 0 && p < rp.table_len;
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    const int j = (e + 2 * pr) / 2;
    const bool rotate = head < rp.H + rp.KV && pos_ok && 2 * j + 1 < rp.rot;
    op.cs[pr] = rotate ? rp.cos_t[static_cast<size_t>(p) * (rp.rot / 2) + j] : 1.f;
    op.sn[pr] = rotate ? rp.sin_t[static_cast<size_t>(p) * (rp.rot / 2) + j] : 0.f;
  }
  const int seq = op.page;
  int page = -1;
  if (head >= rp.H && head < rp.H + 2 * rp.KV && rp.write_kv && pos_ok) {
    const int blk = p / rp.block_size;
    if (seq >= 0 && seq < rp.n_seqs && blk < rp.table_stride)
      page = rp.block_table[static_cast<size_t>(seq) * rp.table_stride + blk];
  }
  op.page = page;
}

// One lane's four neighbouring columns n..n+3 of row m, after the waves' partial sums are added.
template <int EPI>
__device__ __forceinline__ void store_tile(const f32x4& s, int m, int n, int N, int ldc, void* Cv,
                                           const bf16_t* c_add, const RopeEpi& rp, EpiOperands& op) {
  if (EPI == 2 || EPI == 4) {
    if (!op.have) {
      epi_prefetch_a<EPI>(op, m, n, N, ldc, Cv, c_add, rp);
      epi_prefetch_b<EPI>(op, n, rp);
    }
  }
  if (EPI <= 2) {
    const size_t idx = static_cast<size_t>(m) * ldc + n;
    if (EPI == 0 && vec4_ok(Cv, ldc, n, N, 4)) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(Cv) + idx) = s;
    } else if (EPI == 2 && vec4_ok(Cv, ldc, n, N, 4)) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(Cv) + idx) = op.c + s;
    } else if (EPI == 1 && vec4_ok(Cv, ldc, n, N, 2)) {
      uint2 packed;
      packed.x = static_cast<uint32_t>(f32_to_bf16(s[0])) | (static_cast<uint32_t>(f32_to_bf16(s[1])) << 16);
      packed.y = static_cast<uint32_t>(f32_to_bf16(s[2])) | (static_cast<uint32_t>(f32_to_bf16(s[3])) << 16);
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(Cv) + idx) = packed;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (n + r >= N) break;
        if (EPI == 0) static_cast<float*>(Cv)[idx + r] = s[r];
        if (EPI == 1) static_cast<bf16_t*>(Cv)[idx + r].bits = f32_to_bf16(s[r]);
        if (EPI == 2) static_cast<float*>(Cv)[idx + r] = op.c[r] + s[r];
      }
    }
  } else if (EPI == 3) {
    // N is even and n a multiple of 4: two (gate, up) pairs
    bf16_t* o = static_cast<bf16_t*>(Cv) + static_cast<size_t>(m) * ldc + n / 2;
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      if (n + 2 * pr >= N) break;
      float g = s[2 * pr], u = s[2 * pr + 1];
      if (rp.gate_bias) g += rp.gate_bias[n / 2 + pr];
      if (rp.up_bias) u += rp.up_bias[n / 2 + pr];
      float y;
      if (rp.act == GATE_LIMITED) {
        y = limited_pair(g, u, rp.act_limit) * rp.act_scale;
      } else if (rp.act == 1) {
        const float t = 0.7978845608028654f * (g + 0.044715f * g * g * g);
        y = 0.5f * g * (1.f + tanhf(t)) * u * rp.act_scale;
      } else {
        y = g / (1.f + __expf(-g)) * u * rp.act_scale;
      }
      o[pr].bits = f32_to_bf16(y);
    }
  } else {
    // fused q/k/v projection: d is a multiple of 4, so the four columns lie in one head; pairs
    // that are not rotated (v heads, elements past the rotary width, positions off the table)
    // carry the identity
    const int head = n / rp.d, e = n - head * rp.d;
    float o[4];
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      const float x1 = s[2 * pr], x2 = s[2 * pr + 1];
      o[2 * pr] = x1 * op.cs[pr] - x2 * op.sn[pr];
      o[2 * pr + 1] = x2 * op.cs[pr] + x1 * op.sn[pr];
    }
    uint2 packed;
    packed.x = static_cast<uint32_t>(f32_to_bf16(o[0])) | (static_cast<uint32_t>(f32_to_bf16(o[1])) << 16);
    packed.y = static_cast<uint32_t>(f32_to_bf16(o[2])) | (static_cast<uint32_t>(f32_to_bf16(o[3])) << 16);
    if (head < rp.H) {
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(Cv) + static_cast<size_t>(m) * ldc + n) = packed;
    } else if (head >= rp.H + 2 * rp.KV) {
      // columns behind q, k and v (an output gate, say): stored behind q, as they are
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(Cv) + static_cast<size_t>(m) * ldc + n -
                                2 * rp.KV * rp.d) = packed;
    } else if (op.page >= 0 && op.page < rp.num_blocks) {
      const int off = op.pos % rp.block_size;
      if (head < rp.H + rp.KV) {
        const int kvh = head - rp.H;
        *reinterpret_cast<uint2*>(
            rp.k_pages + ((static_cast<size_t>(op.page) * rp.KV + kvh) * rp.block_size + off) * rp.d + e) =
            packed;
      } else {
        // V pages are [num_blocks, KV, d, block_size]: one element per key row
        const int kvh = head - rp.H - rp.KV;
        bf16_t* dst =
            rp.v_pages + ((static_cast<size_t>(op.page) * rp.KV + kvh) * rp.d + e) * rp.block_size + off;
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[static_cast<size_t>(r) * rp.block_size].bits = f32_to_bf16(o[r]);
      }
    }
  }
}

// more tiles per wave mean more registers per lane and more LDS per wave: fewer waves; fp32
// rows take twice the registers while in flight
constexpr int max_waves(int mt, int nt, int at) {
  return (mt * nt >= 8 || (at && mt >= 4)) ? 4 : (mt * nt >= 4 || (at && mt >= 2)) ? 8 : 16;
}
// k-steps whose loads are in flight together in one wave
constexpr int depth(int mt, int nt, int at) {
  return at ? (mt == 1 ? 4 : mt <= 4 ? 2 : 1) : (mt * nt == 1 ? 8 : mt * nt <= 4 ? 4 : 2);
}

// ST: W is streamed past the caches (see streams); a kernel of its own, so that either has the other's arithmetic.
template <int MT, int NT, int AT, int EPI, bool ADD, bool ST>
__global__ __launch_bounds__(max_waves(MT, NT, AT) * KVF_WAVE) void gemm_skinny_kernel(
    const void* __restrict__ Av, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M, int N,
    int K, int lda, int ldc, int m_base, float eps, int w_tiled, Riders rd, RopeEpi rp, PickEpi pk) {
  constexpr int RW = 16;  // rows of W per group
  extern __shared__ float red[];  // [nw][MT][64 lanes][4], then [nw][MT][16] sums of squares
  const int lane = threadIdx.x % KVF_WAVE, wave = threadIdx.x / KVF_WAVE;
  const int nw = blockDim.x / KVF_WAVE;
  const int n0 = blockIdx.x * RW * NT;
  const int r16 = lane % 16, kg = lane / 16;
  const int ksteps = (K + 31) / 32;
  // the k-steps this workgroup walks: all, or one half of them (see Riders::half_out)
  const bool halves = EPI == 2 && rd.half_out != nullptr;
  const bool second = halves && blockIdx.y == 1;
  const int ks_cut = halves ? (ksteps + 1) / 2 : ksteps;
  const int ks_lo = second ? ks_cut : 0, ks_hi = second ? ksteps : ks_cut;
  // where this lane's fragment of k-step 0 lies, and how far the next k-step is
  const bf16_t* wp[NT];
  const size_t w_step = w_tiled ? KVF_WAVE * 8 : 32;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if (w_tiled) {
      const int group = min(static_cast<int>(blockIdx.x) * NT + j, (N + RW - 1) / RW - 1);
      wp[j] = W + (static_cast<size_t>(group) * ksteps * KVF_WAVE + lane) * 8;
    } else {
      int wrow = n0 + j * RW + r16;
      if (wrow >= N) wrow = N - 1;  // clamped rows are computed and never stored
      wp[j] = W + static_cast<size_t>(wrow) * K + kg * 8;
    }
  }
  size_t aoff[MT];
  bool a_live[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    // Rows past M are not loaded at all (their lanes hold zeros and are never stored): a wave's
    // load touches one cache line per row it reads, and the L1 looks lines up one at a time.
    const int arow = m_base + t * 16 + r16;
    a_live[t] = arow < M;
    aoff[t] = static_cast<size_t>(a_live[t] ? arow : 0) * lda + kg * 8;
  }
  const bf16_t* Ab = static_cast<const bf16_t*>(Av);
  const float* Af = static_cast<const float*>(Av);
  const bf16_t* a_add = ADD ? rd.a_add : nullptr;
  const bf16_t* c_add = EPI == 2 && !second ? rd.c_add : nullptr;
  f32x4 acc[NT][MT];
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    ss[t] = 0.f;
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // With one row tile, lane l of wave 0 will finish C[m_base + l%16][n0 + j*RW + 4*(l/16) ..+3]:
  // it asks for what its epilogue reads now, and for what depends on that after its first pass.
  constexpr bool PRE = MT == 1 && (EPI == 2 || EPI == 4);
  EpiOperands pre[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) pre[j].have = false;
  const int pre_m = m_base + r16, pre_n = n0 + 4 * kg;
  const bool pre_mine = PRE && wave == 0 && pre_m < M && !second;
  if (pre_mine) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (pre_n + j * RW < N) epi_prefetch_a<EPI>(pre[j], pre_m, pre_n + j * RW, N, ldc, Cv, c_add, rp);
  }

  constexpr int U = depth(MT, NT, AT);
  int ks = ks_lo + wave;
  bool first = true;
  for (; ks + (U - 1) * nw < ks_hi; ks += U * nw) {
    bf16x8 wf[U][NT], af[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (ks + u * nw) * 32;
      const bool ok = k + kg * 8 + 8 <= K;
#pragma unroll
      for (int j = 0; j < NT; ++j) wf[u][j] = load_weight<ST>(wp[j] + (ks + u * nw) * w_step, ok || w_tiled);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        af[u][t] = AT ? load_frag_f32<ADD>(Af + aoff[t] + k, a_add + aoff[t] + k, ok && a_live[t], ss[t])
                      : load_frag(Ab + aoff[t] + k, ok && a_live[t]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][j], af[u][t], acc[j][t], 0, 0, 0);
    if (PRE && first) {  // the first stage has arrived with this pass's loads
      first = false;
      if (pre_mine) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (pre[j].have) epi_prefetch_b<EPI>(pre[j], pre_n + j * RW, rp);
      }
    }
  }
  if (PRE && first && pre_mine) {  // K too short for a full pass
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (pre[j].have) epi_prefetch_b<EPI>(pre[j], pre_n + j * RW, rp);
  }
  for (; ks < ks_hi; ks += nw) {
    const int k = ks * 32;
    const bool ok = k + kg * 8 + 8 <= K;
    bf16x8 af[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
      af[t] = AT ? load_frag_f32<ADD>(Af + aoff[t] + k, a_add + aoff[t] + k, ok && a_live[t], ss[t])
                 : load_frag(Ab + aoff[t] + k, ok && a_live[t]);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const bf16x8 wf = load_weight<ST>(wp[j] + ks * w_step, ok || w_tiled);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, af[t], acc[j][t], 0, 0, 0);
    }
  }
  // lane holds C[row r16][cols n0 + 16*j + 4*kg .. +3] of each tile
  float pick_v = -INFINITY;   // EPI 5: the best of this thread's columns of its row so far
  int pick_i = 0x7fffffff;
  float* red_ss = red + nw * MT * KVF_WAVE * 4;
  if (AT) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      float v = ss[t];
      v += __shfl_xor(v, 16, KVF_WAVE);
      v += __shfl_xor(v, 32, KVF_WAVE);
      if (kg == 0) red_ss[(wave * MT + t) * 16 + r16] = v;
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    if (j > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t)
      *reinterpret_cast<f32x4*>(red + ((wave * MT + t) * KVF_WAVE + lane) * 4) = acc[j][t];
    __syncthreads();
    for (int item = threadIdx.x; item < MT * KVF_WAVE; item += blockDim.x) {
      const int t = item / KVF_WAVE, l = item % KVF_WAVE;
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int w = 0; w < nw; ++w)
        s += *reinterpret_cast<const f32x4*>(red + ((w * MT + t) * KVF_WAVE + l) * 4);
      const int m = m_base + t * 16 + l % 16;
      const int n = n0 + j * RW + 4 * (l / 16);
      if (m >= M || n >= N) continue;
      if (AT) {
        float tot = 0.f;
        for (int w = 0; w < nw; ++w) tot += red_ss[(w * MT + t) * 16 + l % 16];
        s *= rsqrtf(tot / static_cast<float>(K) + eps);
      }
      if (EPI == 5) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N && better(s[r], n + r, pick_v, pick_i)) { pick_v = s[r]; pick_i = n + r; }
        continue;
      }
      EpiOperands fresh;
      fresh.have = false;
      if (EPI == 2 && second)
        store_tile<1>(s, m, n, N, ldc, rd.half_out, nullptr, rp, fresh);
      else
        store_tile<EPI>(s, m, n, N, ldc, Cv, c_add, rp, PRE ? pre[j] : fresh);
    }
  }
  if (EPI == 5) {
    // one row tile: the first 64 threads hold row r16's best over their four columns of every
    // group of this workgroup
    if (wave == 0) {
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1) {
        const float ov = __shfl_xor(pick_v, o, KVF_WAVE);
        const int oi = __shfl_xor(pick_i, o, KVF_WAVE);
        if (better(ov, oi, pick_v, pick_i)) { pick_v = ov; pick_i = oi; }
      }
      const int m = m_base + r16;
      if (kg == 0 && m < M)
        pick_publish(pk.part_val, pk.part_idx, static_cast<size_t>(m) * gridDim.x + blockIdx.x, pick_v, pick_i);
      pick_stores_done();
    }
    // Two levels of tickets: the workgroups are spread over PICK_LANES counters; the last
    // arrival at a counter merges that counter's workgroups and takes a ticket of the top
    // counter; the last arrival there finishes.
    const int groups = static_cast<int>(gridDim.x), lane_id = static_cast<int>(blockIdx.x) % PICK_LANES;
    int* flag = reinterpret_cast<int*>(red);
    __syncthreads();     // (and nobody reads `red` any more)
    if (threadIdx.x == 0)
      flag[0] = pick_last_at(pk.ticket + lane_id * PICK_STRIDE, (groups - lane_id + PICK_LANES - 1) / PICK_LANES);
    __syncthreads();
    if (flag[0] == 0) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // what the others published, not this XCD's stale copy
    pick_merge_lane(pk, M, groups, lane_id);
    __syncthreads();
    if (threadIdx.x == 0)
      flag[1] = pick_last_at(pk.ticket + PICK_LANES * PICK_STRIDE, groups < PICK_LANES ? groups : PICK_LANES);
    __syncthreads();
    if (flag[1] == 0) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    pick_finish(pk, M, groups, red + 64);
  }
}

// 17 to 64 rows of bf16 over tiled weights (EPI 0, 1 and 3).
//
// What bounded gemm_skinny_kernel here: every wave read its own fragments of A through the L1, 16
// rows of 64 bytes each, as many bytes as of W at 64 rows, and a pass over its few k-steps ended in a
// wait for all of them (2,048 x 16,384 with the gate: 23.6 us at 41 rows, 2.8 TB/s).  Here A goes
// through LDS once for the workgroup, 128 columns a stage (whole cache lines), and W straight into
// registers, both MID_AHEAD stages before they are used, so that the memory always has 48 to 96 KB of
// a workgroup's requests (by rows and groups); two workgroups fit a compute unit (128 registers a lane) and cover each
// other's barriers.  Four or six stages ahead were no faster (17.6 / 18.4 us) and cost registers.
// Eight waves: NG groups of 16 columns, the k-steps of a stage shared by 8 / NG waves whose sums are
// added in LDS.  41 rows: 17.5 us; 20 and 61 rows 21.2 -> 16.1, 25.0 -> 18.3; a head of
// 128,256 columns at 41 rows 131 -> 109 us, where the library took 128.
//
// `parts`: K is cut over gridDim.y and every cut stores its sums in fp32 as a plane of [M][N] of its
// own, which the reader adds (rmsnorm_parts_kernel): a narrow C has too few workgroups otherwise.
// 8,192 x 2,048 in 8 cuts at 41 / 61 rows: 10.5 / 11.0 us (the library 14.4 / 15.7 with a result
// rounded to bf16), 2,048 x 2,048 in 4: 4.9 / 5.2 us (8.4).
constexpr int MID_WAVES = 8;     // waves of a workgroup
constexpr int MID_STEPS = 4;     // k-steps of 32 in a stage
constexpr int MID_AHEAD = 3;     // stages whose loads are on their way
template <int MT, int NG, int EPI>
__global__ __launch_bounds__(MID_WAVES * KVF_WAVE, 4) void gemm_mid_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M, int N, int K,
    int lda, int ldc, RopeEpi rp, float* __restrict__ parts, int stages_each) {
  constexpr int D = MID_AHEAD;
  constexpr int KW = MID_WAVES / NG;            // waves that share a group of columns, by k-steps
  constexpr int FR = MID_STEPS / KW;            // k-steps of a stage that one wave takes
  constexpr int XROWS = MT * 16;
  constexpr int XL = (XROWS * 16 + MID_WAVES * KVF_WAVE - 1) / (MID_WAVES * KVF_WAVE);   // 16-byte pieces a thread
  static_assert(NG >= 2 && NG <= 8, "a wave takes whole k-steps of one group");
  static_assert(2 * XROWS * 256 == MID_WAVES * MT * 1024, "the sums of the waves take the place of both stages of A");
  __shared__ __attribute__((aligned(16))) char lds[2 * XROWS * 256];
  const int tid = threadIdx.x, lane = tid % KVF_WAVE, wave = tid / KVF_WAVE;
  const int r16 = lane % 16, kg = lane / 16;
  const int ksteps = (K + 31) / 32;
  const int groups = (N + 15) / 16;
  const int grp = blockIdx.x * NG + wave % NG;
  const int stages = (ksteps + MID_STEPS - 1) / MID_STEPS;
  const int s_lo = blockIdx.y * stages_each, s_hi = min(stages, s_lo + stages_each);
  const int kw = wave / NG;
  const bf16_t* wp = W + (static_cast<size_t>(min(grp, groups - 1)) * ksteps * KVF_WAVE + lane) * 8;
  // A thread's pieces of a stage of A: rows tid / 16 (+ 32), 8 columns at tid % 16.  In LDS a row's
  // pieces are turned by the row, so that neither the rows of a fragment nor a row's pieces share a bank.
  const int xc = tid % 16;
  const bf16_t* xp[XL];
  int xo[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = tid / 16 + i * 32;
    xp[i] = A + static_cast<size_t>(min(row, M - 1)) * lda + xc * 8;
    xo[i] = row * 256 + ((xc ^ (row & 15)) * 16);
  }
  uint4 wr[D][FR], xr[D][XL];
  auto load_w = [&](int slot, int s) {
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      const int ks = min(s * MID_STEPS + kw * FR + f, ksteps - 1);
      wr[slot][f] = *reinterpret_cast<const uint4*>(wp + static_cast<size_t>(ks) * (KVF_WAVE * 8));
    }
  };
  auto load_x = [&](int slot, int s) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      if (XROWS % 32 != 0 && i == XL - 1 && wave >= 4) continue;
      const int k = s * (MID_STEPS * 32);
      const bool in = k + xc * 8 + 8 <= K;
      const uint4 v = *reinterpret_cast<const uint4*>(xp[i] + (in ? k : -xc * 8));
      xr[slot][i] = in ? v : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto put_x = [&](int slot, int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      if (XROWS % 32 != 0 && i == XL - 1 && wave >= 4) continue;
      *reinterpret_cast<uint4*>(lds + buf * (XROWS * 256) + xo[i]) = xr[slot][i];
    }
  };
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Loads past the last stage repeat it (no load stands under a condition) and are never used.
#pragma unroll
  for (int d = 0; d < D; ++d) {
    load_x(d, min(s_lo + d, s_hi - 1));
    load_w(d, min(s_lo + d, s_hi - 1));
  }
  put_x(0, 0);
  load_x(0, min(s_lo + D, s_hi - 1));
  __syncthreads();
  for (int s0 = s_lo; s0 < s_hi; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int s = s0 + d;
      if (s < s_hi) {
        const char* buf = lds + ((s - s_lo) & 1) * (XROWS * 256);
#pragma unroll
        for (int f = 0; f < FR; ++f) {
          const int kl = kw * FR + f;
          if (s * MID_STEPS + kl < ksteps) {   // the same for all lanes
            const bf16x8 wf = __builtin_bit_cast(bf16x8, wr[d][f]);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              const uint4 xv = *reinterpret_cast<const uint4*>(buf + (t * 16 + r16) * 256 + (((kl * 4 + kg) ^ r16) * 16));
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(bf16x8, xv), acc[t], 0, 0, 0);
            }
          }
        }
        load_w(d, min(s + D, s_hi - 1));
        put_x((d + 1) % D, (s + 1 - s_lo) & 1);
        load_x((d + 1) % D, min(s + 1 + D, s_hi - 1));
        __syncthreads();
      }
    }
  }
  float* red = reinterpret_cast<float*>(lds);   // behind the last stage's barrier
#pragma unroll
  for (int t = 0; t < MT; ++t)
    *reinterpret_cast<f32x4*>(red + ((wave * MT + t) * KVF_WAVE + lane) * 4) = acc[t];
  __syncthreads();
  for (int item = tid; item < NG * MT * KVF_WAVE; item += MID_WAVES * KVF_WAVE) {
    const int l = item % KVF_WAVE, t = item / KVF_WAVE % MT, g = item / KVF_WAVE / MT;
    f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < KW; ++q)
      sum += *reinterpret_cast<const f32x4*>(red + (((q * NG + g) * MT + t) * KVF_WAVE + l) * 4);
    const int m = t * 16 + l % 16, n = (blockIdx.x * NG + g) * 16 + 4 * (l / 16);
    if (m >= M || n >= N) continue;
    EpiOperands fresh;
    fresh.have = false;
    if (EPI == 0 && parts)
      store_tile<0>(sum, m, n, N, N, parts + static_cast<size_t>(blockIdx.y) * M * N, nullptr, rp, fresh);
    else
      store_tile<EPI>(sum, m, n, N, ldc, Cv, nullptr, rp, fresh);
  }
}

// Several products of at most 16 bf16 rows over tiled weights in one launch (EPI 0 to 3 each, inputs of their own):
// the projections that a step's parts begin with.  In a decode step each is a kernel of 4 to 7 us whose time is its
// launch and two trips to memory; together those come once.  Eight rows of 2,048, a recurrence's rows, its gates, a router
// and a gated pair of 4,096 columns: 7.0 + 4.6 + 4.6 + 6.0 us apart, 9.7 together.  A workgroup takes 16 columns of one product as gemm_skinny_kernel<1, 1, 0,
// EPI> on eight waves does, with the same sums in the same order, so that the results are the same to the bit.
struct GroupItem {
  const bf16_t* A;
  const bf16_t* W;
  void* C;
  int N, K, lda, ldc, epi, first;   // first: its first workgroup
  bool streamed;
};
constexpr int GROUP_MAX = 8, GROUP_WAVES = 8;
struct Group {
  GroupItem item[GROUP_MAX];
  int count;
};

__global__ __launch_bounds__(GROUP_WAVES * KVF_WAVE) void gemm_group_kernel(Group group, int M, RopeEpi rp) {
  __shared__ __attribute__((aligned(16))) float red[GROUP_WAVES * KVF_WAVE * 4];
  int which = 0;
  for (int i = 1; i < group.count; ++i)
    if (static_cast<int>(blockIdx.x) >= group.item[i].first) which = i;   // the same for the whole workgroup
  const GroupItem it = group.item[which];
  const int lane = threadIdx.x % KVF_WAVE, wave = threadIdx.x / KVF_WAVE, r16 = lane % 16, kg = lane / 16;
  const int grp = blockIdx.x - it.first, n0 = grp * 16, ksteps = (it.K + 31) / 32;
  const bf16_t* wp = it.W + (static_cast<size_t>(grp) * ksteps * KVF_WAVE + lane) * 8;
  const bool live = r16 < M;
  const bf16_t* ap = it.A + static_cast<size_t>(live ? r16 : 0) * it.lda + kg * 8;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  EpiOperands pre;                     // what the product is added to, asked for now (see EpiOperands)
  pre.have = false;
  if (it.epi == 2 && wave == 0 && live && n0 + 4 * kg < it.N)
    epi_prefetch_a<2>(pre, r16, n0 + 4 * kg, it.N, it.ldc, it.C, nullptr, rp);
  constexpr int U = depth(1, 1, 0), nw = GROUP_WAVES;
  auto walk = [&](auto streamed) {
    constexpr bool S = decltype(streamed)::value;
    int ks = wave;
    for (; ks + (U - 1) * nw < ksteps; ks += U * nw) {
      bf16x8 wf[U], af[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = (ks + u * nw) * 32;
        wf[u] = load_weight<S>(wp + static_cast<size_t>(ks + u * nw) * (KVF_WAVE * 8), true);
        af[u] = load_frag(ap + k, live && k + kg * 8 + 8 <= it.K);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u], af[u], acc, 0, 0, 0);
    }
    for (; ks < ksteps; ks += nw) {
      const bf16x8 wf = load_weight<S>(wp + static_cast<size_t>(ks) * (KVF_WAVE * 8), true);
      const bf16x8 af = load_frag(ap + ks * 32, live && ks * 32 + kg * 8 + 8 <= it.K);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, af, acc, 0, 0, 0);
    }
  };
  if (it.streamed) walk(Flag<true>{});
  else walk(Flag<false>{});
  *reinterpret_cast<f32x4*>(red + (wave * KVF_WAVE + lane) * 4) = acc;
  __syncthreads();
  const int n = n0 + 4 * kg;
  if (wave != 0 || !live || n >= it.N) return;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < nw; ++w) s += *reinterpret_cast<const f32x4*>(red + (w * KVF_WAVE + lane) * 4);
  EpiOperands none;
  none.have = false;
  if (it.epi == 0) store_tile<0>(s, r16, n, it.N, it.ldc, it.C, nullptr, rp, none);
  else if (it.epi == 1) store_tile<1>(s, r16, n, it.N, it.ldc, it.C, nullptr, rp, none);
  else if (it.epi == 2) store_tile<2>(s, r16, n, it.N, it.ldc, it.C, nullptr, rp, pre);
  else store_tile<3>(s, r16, n, it.N, it.ldc, it.C, nullptr, rp, none);
}

int g_waves_override = 0;
int g_rows_override = 0;

// Waves per workgroup, as measured on the shapes of a 1B-parameter decoder: eight (fewer leave
// loads unhidden, sixteen crowd the CU); at least one k-step per wave.
int pick_waves(int K) {
  const int ksteps = (K + 31) / 32;
  int nw = g_waves_override > 0 ? g_waves_override : 8;
  if (nw > 16) nw = 16;
  if (nw > ksteps) nw = ksteps;
  if (nw < 1) nw = 1;
  return nw;
}

template <int MT, int NT, int AT, int EPI, bool ADD>
int launch_as(dim3 grid, dim3 block, size_t lds, const void* A, const bf16_t* W, void* C, int M, int N, int K, int lda,
              int ldc, int m_base, float eps, int w_tiled, const Riders& rd, const RopeEpi& rp, const PickEpi& pk,
              hipStream_t s) {
  if (w_tiled && w_tiled != CACHED && streams(N, K))
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, AT, EPI, ADD, true>), grid, block, lds, s, A, W, C, M, N, K, lda,
                       ldc, m_base, eps, w_tiled, rd, rp, pk);
  else
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, NT, AT, EPI, ADD, false>), grid, block, lds, s, A, W, C, M, N, K, lda,
                       ldc, m_base, eps, w_tiled, rd, rp, pk);
  return kvf_last_error();
}

template <int MT, int NT, int AT, int EPI>
int launch_one(const void* A, const bf16_t* W, void* C, int M, int N, int K, int lda, int ldc,
               int m_base, float eps, int w_tiled, const Riders& rd, const RopeEpi& rp, hipStream_t s,
               const PickEpi& pk = PickEpi{}) {
  const int groups = (N + 16 * NT - 1) / (16 * NT);
  int nw = pick_waves(K);
  if (nw > max_waves(MT, NT, AT)) nw = max_waves(MT, NT, AT);
  const dim3 grid(groups, EPI == 2 && rd.half_out ? 2 : 1), block(nw * KVF_WAVE);
  size_t lds = static_cast<size_t>(nw) * MT * (KVF_WAVE * 4 + 16) * sizeof(float);
  if (EPI == 5 && lds < (64 + 2 * 16 * 16 + 16) * sizeof(float)) lds = (64 + 2 * 16 * 16 + 16) * sizeof(float);
  if (rd.a_add) {
    // the sum that rides in the left operand's loads: only the fused q/k/v projection of one
    // tile of rows is built with it
    if constexpr (MT == 1 && AT == 1 && EPI == 4)
      return launch_as<MT, NT, AT, EPI, true>(grid, block, lds, A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp,
                                              pk, s);
    return static_cast<int>(hipErrorInvalidValue);
  }
  return launch_as<MT, NT, AT, EPI, false>(grid, block, lds, A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp,
                                           pk, s);
}

// How 17 to 64 rows are cut: groups of columns a workgroup and cuts of K.  The rule takes the least
// bytes through a compute unit's L1, over the rounds of workgroups: rows and columns over the cut's K,
// and 16 bytes for every sum that is stored in fp32, added to the stream and read back (measured: 2,048 x
// 2,048 at 61 rows 5.2 us as 2 x 4, 5.9 as 4 x 8; 8,192 x 2,048 11.0 as 4 x 8, 12.9 as 2 x 8; without
// cuts 2,048 x 8,192 at 48 rows 12.7 with 2 groups, 14.2 with 4, and x 16,384 18.1 and 17.4).
struct MidCut {
  int groups, splits;
};
MidCut mid_cut(int M, int N, int K, bool may_split) {
  const int tiles = (N + 15) / 16, stages = ((K + 31) / 32 + MID_STEPS - 1) / MID_STEPS, cus = compute_units();
  MidCut best{4, 1};
  long least = -1;
  for (int ng = 2; ng <= 4; ng *= 2) {
    for (int sp = may_split ? 2 : 1; sp <= (may_split ? 8 : 1); sp *= 2) {
      if (sp > stages) break;
      const int each = (stages + sp - 1) / sp;
      if ((stages + each - 1) / each != sp) continue;    // a cut would be empty
      const long wgs = static_cast<long>((tiles + ng - 1) / ng) * sp;
      const long bytes = (wgs + cus - 1) / cus * (2l * MID_STEPS * 32 * each * (M + 16 * ng) + (may_split ? 16l * M * 16 * ng : 0));
      if (least < 0 || bytes < least) {
        least = bytes;
        best = MidCut{ng, sp};
      }
    }
  }
  return best;
}

// Whether 17 to 64 rows without cuts of K take gemm_mid_kernel instead of gemm_skinny_kernel, which takes
// fewer columns a workgroup and so reaches more of the chip where there are few: up to 32 rows from three
// groups of 16 columns for each compute unit on (12,288 columns x 2,048: 16.5 -> 14.0 us; 8,192: 11.1
// and 11.1; 4,096: 7.5 and 9.6), above, where it also re-reads more rows, from one and a half on (6,144 x
// 2,048: 13.8 -> 12.2; 4,096: 9.8 and 11.2).
bool mid_pays(int M, int N, int epi, int w_tiled) {
  if (M <= 16 || M > 64 || !w_tiled || (epi != 0 && epi != 1 && epi != 3)) return false;
  const long tiles = (N + 15) / 16, cus = compute_units();
  return M <= 32 ? tiles >= 3 * cus : 2 * tiles >= 3 * cus;
}

template <int MT, int EPI>
int launch_mid_mt(const bf16_t* A, const bf16_t* W, void* C, int M, int N, int K, int lda, int ldc, const RopeEpi& rp,
                  float* parts, const MidCut& cut, hipStream_t s) {
  const int stages = ((K + 31) / 32 + MID_STEPS - 1) / MID_STEPS, each = (stages + cut.splits - 1) / cut.splits;
  const dim3 grid(((N + 15) / 16 + cut.groups - 1) / cut.groups, cut.splits), block(MID_WAVES * KVF_WAVE);
  if (cut.groups == 2)
    hipLaunchKernelGGL((gemm_mid_kernel<MT, 2, EPI>), grid, block, 0, s, A, W, C, M, N, K, lda, ldc, rp, parts, each);
  else
    hipLaunchKernelGGL((gemm_mid_kernel<MT, 4, EPI>), grid, block, 0, s, A, W, C, M, N, K, lda, ldc, rp, parts, each);
  return kvf_last_error();
}

template <int EPI>
int launch_mid(const void* A, const bf16_t* W, void* C, int M, int N, int K, int lda, int ldc, const RopeEpi& rp,
               float* parts, const MidCut& cut, hipStream_t s) {
  const bf16_t* a = static_cast<const bf16_t*>(A);
  if (M <= 32) return launch_mid_mt<2, EPI>(a, W, C, M, N, K, lda, ldc, rp, parts, cut, s);
  if (M <= 48) return launch_mid_mt<3, EPI>(a, W, C, M, N, K, lda, ldc, rp, parts, cut, s);
  return launch_mid_mt<4, EPI>(a, W, C, M, N, K, lda, ldc, rp, parts, cut, s);
}

// How many 16-row groups of W a wave takes when A has several row tiles.  With 17 to 64 rows the
// product is bound by what every compute unit has to bring in through its L1, which keeps only
// some fifty lines in flight: all rows of A for each of its workgroups, and their columns of W.
// A wave that takes more groups shares A's rows among more columns, but leaves fewer
// workgroups; the choice is the one with the least to fill per compute unit, in rounds of
// workgroups over the chip (measured at 32 rows: [5120, 3072] 15.2 us with one group, 10.9 with
// two; [28672, 4096] 62.8 with two, 53.3 with four).
template <int MT, int AT, int EPI>
int launch_nt(const void* A, const bf16_t* W, void* C, int M, int N, int K, int lda, int ldc,
              int m_base, float eps, int w_tiled, const Riders& rd, const RopeEpi& rp, hipStream_t s) {
  const int tiles = (N + 15) / 16;
  if constexpr (MT >= 2 && MT <= 4 && !AT) {
    const int cus = compute_units(), rows = M - m_base < MT * 16 ? M - m_base : MT * 16;
    int best = 1, least = 0x7fffffff;
    for (int nt = 1; nt <= 4; nt *= 2) {
      const int groups = (tiles + nt - 1) / nt;
      const int fill = ((groups + cus - 1) / cus) * (rows + 16 * nt);
      if (fill < least) {
        least = fill;
        best = nt;
      }
    }
    if (best == 4)
      return launch_one<MT, 4, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
    if (best == 2)
      return launch_one<MT, 2, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
  }
  if (MT == 1) {
    // Every workgroup reads all of A, so with several rows of A and many rows of W a workgroup
    // takes 32 rows of W and halves that traffic; fp32 rows weigh twice as much and make it pay
    // with fewer rows of W.
    const int rw = g_rows_override > 0 ? g_rows_override : (M - m_base > 4 && tiles >= (AT ? 256 : 512) ? 32 : 16);
    if (rw == 32) return launch_one<1, 2, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
    if (rw == 64) return launch_one<1, 4, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
  }
  return launch_one<MT, 1, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
}

template <int AT, int EPI>
int launch_rows(const void* A, const bf16_t* W, void* C, int M, int N, int K, int lda, int ldc,
                float eps, int w_tiled, const Riders& rd, const RopeEpi& rp, hipStream_t s) {
  if constexpr (AT == 0 && (EPI == 0 || EPI == 1 || EPI == 3)) {
    if (mid_pays(M, N, EPI, w_tiled))
      return launch_mid<EPI>(A, W, C, M, N, K, lda, ldc, rp, nullptr, mid_cut(M, N, K, false), s);
  }
  int err = 0;
  for (int m_base = 0; m_base < M && !err; m_base += 128) {
    const int rows = M - m_base < 128 ? M - m_base : 128;
    if (rows <= 16) err = launch_nt<1, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
    else if (rows <= 32) err = launch_nt<2, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
    else if (rows <= 64) err = launch_nt<4, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
    else err = launch_nt<8, AT, EPI>(A, W, C, M, N, K, lda, ldc, m_base, eps, w_tiled, rd, rp, s);
  }
  return err;
}

template <int AT>
int launch_epi(const void* A, const bf16_t* W, void* C, int epi, int M, int N, int K, int lda,
               int ldc, float eps, int w_tiled, const Riders& rd, const RopeEpi& rp, hipStream_t s) {
  switch (epi) {
    case 0: return launch_rows<AT, 0>(A, W, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
    case 1: return launch_rows<AT, 1>(A, W, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
    case 2: return launch_rows<AT, 2>(A, W, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
    case 3: return launch_rows<AT, 3>(A, W, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
    case 4: return launch_rows<AT, 4>(A, W, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
  }
  return static_cast<int>(hipErrorInvalidValue);
}
}  // namespace

// For measurements: force the number of waves per workgroup and the rows of W per workgroup
// (0 = choose by shape).
KVF_EXPORT void kvf_gemm_bf16_set_waves(int waves) { g_waves_override = waves; }
KVF_EXPORT void kvf_gemm_bf16_set_rows(int rows) { g_rows_override = rows; }

// a_type: 0 = bf16 rows, 1 = fp32 rows normalised by rsqrt(mean(x^2) + eps) in the kernel.
// epi: 0 store fp32, 1 store bf16, 2 add into fp32, 3 SwiGLU pairs -> bf16 [M, N/2].
// w_tiled: W is [N, K] row-major (0) or in tiles of 16 x 32 (1, see the head of this file; CACHED: and not to go past the caches).
// c_add (epi 2 only, may be null): bf16 [M, ldc], added to C together with the product.
// half_out (epi 2 with bf16 rows only, may be null): bf16 [M, ldc]; the product over the second
//   half of K is stored there instead of being added to C, by a second layer of workgroups.
KVF_EXPORT int kvf_gemm_bf16(const void* A, int a_type, const void* W, int w_tiled, void* C, int epi,
                             int M, int N, int K, int lda, int ldc, float eps, const void* c_add,
                             void* half_out, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 8 != 0 || lda % 8 != 0 || epi < 0 || epi > 3 || (epi == 3 && N % 4 != 0))
    return static_cast<int>(hipErrorInvalidValue);
  if (((c_add || half_out) && epi != 2) || (half_out && (a_type != 0 || K < 64)))
    return static_cast<int>(hipErrorInvalidValue);
  RopeEpi none{};
  none.act_scale = 1.f;
  const Riders rd{nullptr, static_cast<const bf16_t*>(c_add), static_cast<bf16_t*>(half_out)};
  const bf16_t* w = static_cast<const bf16_t*>(W);
  if (a_type == 0) return launch_epi<0>(A, w, C, epi, M, N, K, lda, ldc, eps, w_tiled, rd, none, s);
  if (a_type == 1) return launch_epi<1>(A, w, C, epi, M, N, K, lda, ldc, eps, w_tiled, rd, none, s);
  return static_cast<int>(hipErrorInvalidValue);
}

// Whether no product of a launch of several (items and M as kvf_gemm_bf16_group) reads or writes what another one writes, since they run
// at the same time.  Results that are blocks of columns of rows of one length are apart.
KVF_EXPORT int kvf_gemm_bf16_group_apart(const long long* items, int count, int M) {
  struct Rows { long long at, pitch, width, end; };
  const auto rows = [M](long long at, long long pitch, long long width) { return Rows{at, pitch, width, at + (M - 1) * pitch + width}; };
  const auto meet = [](const Rows& a, const Rows& b) { return a.at < b.end && b.at < a.end; };
  for (int i = 0; i < count; ++i) {
    const long long *v = items + 8 * i, epi = v[7] & ~GROUP_CACHED, size = epi == 0 || epi == 2 ? 4 : 2;
    const Rows out = rows(v[2], v[6] * size, (epi == 3 ? v[3] / 2 : v[3]) * size);
    for (int j = 0; j < count; ++j) {
      const long long *u = items + 8 * j, its = u[7] & ~GROUP_CACHED, other = its == 0 || its == 2 ? 4 : 2;
      if (meet(out, rows(u[0], 2 * u[5], 2 * u[4]))) return 0;
      const Rows to = rows(u[2], u[6] * other, (its == 3 ? u[3] / 2 : u[3]) * other);
      if (j >= i || !meet(out, to)) continue;
      if (out.pitch != to.pitch || out.pitch <= 0) return 0;
      const long long away = ((to.at - out.at) % out.pitch + out.pitch) % out.pitch;
      if (away < out.width || away + to.width > out.pitch) return 0;
    }
  }
  return 1;
}

// Several products of M <= 16 rows in one launch (see gemm_group_kernel).  items: for each A, W, C (addresses), N, K, lda, ldc
// and epi (0 store fp32, 1 store bf16, 2 add into fp32, 3 SwiGLU pairs -> bf16 [M, N/2]; with GROUP_CACHED: W not past the caches); W in
// tiles, K beyond 224 (a k-step for every wave).
KVF_EXPORT int kvf_gemm_bf16_group(const long long* items, int count, int M, hipStream_t s) {
  if (M <= 0 || count <= 0) return 0;
  if (M > 16 || count > GROUP_MAX || !kvf_gemm_bf16_group_apart(items, count, M)) return static_cast<int>(hipErrorInvalidValue);
  Group g{};
  int blocks = 0;
  for (int i = 0; i < count; ++i) {
    const long long* v = items + 8 * i;
    GroupItem& it = g.item[i];
    it = GroupItem{reinterpret_cast<const bf16_t*>(v[0]), reinterpret_cast<const bf16_t*>(v[1]), reinterpret_cast<void*>(v[2]),
                   static_cast<int>(v[3]), static_cast<int>(v[4]), static_cast<int>(v[5]), static_cast<int>(v[6]),
                   static_cast<int>(v[7] & ~GROUP_CACHED), blocks, false};
    it.streamed = !(v[7] & GROUP_CACHED) && streams(it.N, it.K);
    if (!it.A || !it.W || !it.C || it.N <= 0 || it.K <= 224 || it.K % 8 != 0 || it.lda % 8 != 0 || v[0] % 16 != 0 || v[1] % 16 != 0 ||
        !(it.epi >= 0 && (it.epi <= 2 || (it.epi == 3 && it.N % 4 == 0))))
      return static_cast<int>(hipErrorInvalidValue);
    blocks += (it.N + 15) / 16;
  }
  g.count = count;
  RopeEpi rp{};
  rp.act_scale = 1.f;
  hipLaunchKernelGGL(gemm_group_kernel, dim3(blocks), dim3(GROUP_WAVES * KVF_WAVE), 0, s, g, M, rp);
  return kvf_last_error();
}

// A product of 17 to 64 bf16 rows cut over K, see gemm_mid_kernel.  How many parts M rows over W [N, K]
// are stored in, or 0 where they had better be one product: wide outputs fill the chip by themselves, and
// up to 32 rows over a matrix with fewer rows than columns gemm_skinny_kernel is as fast (4,096 x 2,048 at
// 17 rows: 6.1 us both).  A shorter K would gain a microsecond a product (1,024 x 2,048 at 33 rows 5.5 and 4.2).  It is left
// out because cuts sum in another order: models of such layers, whose steps are mostly bound by the host's launches (0.56 ms
// and 0.58 with cuts for 50 tokens of layers 512 wide), would give other tokens near ties for next to nothing.
KVF_EXPORT int kvf_gemm_bf16_parts_count(int M, int N, int K) {
  if (M <= 16 || M > 64 || N <= 0 || N % 16 != 0 || N > 4096 || K < 2048 || K % 8 != 0 || (M <= 32 && K < N)) return 0;
  return mid_cut(M, N, K, true).splits;
}

// parts: fp32 [kvf_gemm_bf16_parts_count(M, N, K)][M][N], whose sum is A * W^T; W in tiles.
KVF_EXPORT int kvf_gemm_bf16_parts(const void* A, const void* W, float* parts, int count, int M, int N, int K,
                                   int lda, hipStream_t s) {
  if (count <= 0 || count != kvf_gemm_bf16_parts_count(M, N, K) || lda % 8 != 0 || reinterpret_cast<uintptr_t>(parts) % 16 != 0)
    return static_cast<int>(hipErrorInvalidValue);
  RopeEpi none{};
  none.act_scale = 1.f;
  return launch_mid<0>(A, static_cast<const bf16_t*>(W), nullptr, M, N, K, lda, N, none, parts, mid_cut(M, N, K, true), s);
}

// The gated pair epilogue (epi 3) with its activation chosen and biases: out[m, j] =
// act(c[2j] + gate_bias[j]) * (c[2j+1] + up_bias[j]) as bf16 [M, N/2]; act 0 silu, 1 the tanh form
// of gelu, 2 the limited form (GateForm), the whole times `scale`; the biases are fp32 [N/2] and may be null.
KVF_EXPORT int kvf_gemm_bf16_gated(const void* A, int a_type, const void* W, int w_tiled, void* C,
                                   int M, int N, int K, int lda, int ldc, float eps, int act,
                                   float limit, float scale, const float* gate_bias, const float* up_bias, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 8 != 0 || lda % 8 != 0 || N % 4 != 0 || act < 0 || act > GATE_LIMITED ||
      (act == GATE_LIMITED && !(limit > 0.f)))
    return static_cast<int>(hipErrorInvalidValue);
  RopeEpi rp{};
  rp.act = act;
  rp.act_limit = limit;
  rp.act_scale = scale;
  rp.gate_bias = gate_bias;
  rp.up_bias = up_bias;
  const Riders rd{nullptr, nullptr, nullptr};
  const bf16_t* w = static_cast<const bf16_t*>(W);
  if (a_type == 0) return launch_rows<0, 3>(A, w, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
  if (a_type == 1) return launch_rows<1, 3>(A, w, C, M, N, K, lda, ldc, eps, w_tiled, rd, rp, s);
  return static_cast<int>(hipErrorInvalidValue);
}

// Fused q/k/v projection with rotary and cache write.  W: [(H + 2*KV) * d, K] with q and k rows
// permuted so that rotary pairs are neighbouring rows.  q_out: [M, ldq >= H * d] bf16.
// extra_cols (a multiple of 4): further rows of W behind q, k and v, whose columns of the product
// are stored behind q in q_out as they are (ldq >= H * d + extra_cols); KV may then be 0 for a
// projection without keys and values.
// a_add (a_type 1 and at most 16 rows only, may be null): bf16 [M, lda], added to A before the
// norm.
KVF_EXPORT int kvf_gemm_bf16_qkv_rope(const void* A, int a_type, const void* W, int w_tiled,
                                      void* q_out, int M, int K, int lda, int ldq, float eps,
                                      const void* a_add, const int* positions,
                                      const int* seq_of_token, const float* cos_t,
                                      const float* sin_t, const int* block_table, void* k_pages,
                                      void* v_pages, int H, int KV, int d, int rot, int table_len,
                                      int block_size, int table_stride, int num_blocks,
                                      int write_kv, int n_seqs, int extra_cols, hipStream_t s) {
  if (M <= 0) return 0;
  if (K <= 0 || K % 8 != 0 || lda % 8 != 0 || d % 4 != 0 || rot % 2 != 0 || rot > d || ldq % 4 != 0 ||
      (a_add && (a_type != 1 || M > 16)) || extra_cols < 0 || extra_cols % 4 != 0 || KV < 0 ||
      ldq < H * d + extra_cols)
    return static_cast<int>(hipErrorInvalidValue);
  const Riders rd{static_cast<const bf16_t*>(a_add), nullptr, nullptr};
  const RopeEpi rp{positions, seq_of_token, cos_t, sin_t, block_table,
                   static_cast<bf16_t*>(k_pages), static_cast<bf16_t*>(v_pages), H, KV, d, rot,
                   table_len, block_size, table_stride, num_blocks, write_kv, n_seqs, 0, 0.f, 1.f, nullptr, nullptr};
  const int N = (H + 2 * KV) * d + extra_cols;
  const bf16_t* w = static_cast<const bf16_t*>(W);
  if (a_type == 0) return launch_rows<0, 4>(A, w, q_out, M, N, K, lda, ldq, eps, w_tiled, rd, rp, s);
  if (a_type == 1) return launch_rows<1, 4>(A, w, q_out, M, N, K, lda, ldq, eps, w_tiled, rd, rp, s);
  return static_cast<int>(hipErrorInvalidValue);
}


// How many workgroups the greedy pick of M rows over N columns launches: the caller sizes
// part_val / part_idx as 16 * that many.
KVF_EXPORT int kvf_gemm_bf16_pick_ticket_ints() { return PICK_TICKET_INTS; }
KVF_EXPORT int kvf_gemm_bf16_pick_groups(int M, int N) {
  const int tiles = (N + 15) / 16;
  const int nt = (M > 4 && tiles >= 512) ? 2 : 1;
  return (N + 16 * nt - 1) / (16 * nt);
}

// Output head of a decode step with the greedy pick and the step's tail folded in (EPI 5 at the
// head of the file).  A: the normalised rows [M <= 16, lda] bf16.  W: [N, K] bf16, row-major or
// tiled.  residual: [M, ld_res] fp32, receives the picked tokens' rows of `embed` [>= N, hidden].
// See PickEpi for the rest.
KVF_EXPORT int kvf_gemm_bf16_pick(const void* A, const void* W, int w_tiled, int M, int N, int K,
                                  int lda, float* part_val, int* part_idx, int* ticket, int* tokens,
                                  int* token_ids, int* positions, int* ctx_lens, int* ring,
                                  int* run_counter, int ring_stride, int ring_rows, const void* embed,
                                  float* residual, int hidden, int ld_res, hipStream_t s) {
  if (M <= 0) return 0;
  if (M > 16 || N <= 0 || K <= 0 || K % 8 != 0 || lda % 8 != 0 || hidden % 8 != 0 || ld_res % 4 != 0 ||
      ring_stride < M || ring_rows <= 0 || !part_val || !part_idx || !ticket)
    return static_cast<int>(hipErrorInvalidValue);
  const Riders rd{nullptr, nullptr, nullptr};
  const RopeEpi none{};
  const PickEpi pk{part_val, part_idx, ticket, tokens, token_ids, positions, ctx_lens, ring, run_counter,
                   static_cast<const bf16_t*>(embed), residual, ring_stride, ring_rows, hidden, ld_res};
  const bf16_t* w = static_cast<const bf16_t*>(W);
  if (M > 4 && (N + 15) / 16 >= 512)   // two groups of 16 columns per workgroup, as pick_groups counts
    return launch_one<1, 2, 0, 5>(A, w, nullptr, M, N, K, lda, 0, 0, 0.f, w_tiled, rd, none, s, pk);
  return launch_one<1, 1, 0, 5>(A, w, nullptr, M, N, K, lda, 0, 0, 0.f, w_tiled, rd, none, s, pk);
}
