// states-form attention over the KV state slots for gfx950.
//
// Contract (packages/runtime/src/kernels/state-attention.ts:1-113, docs/ir-v1.md:296-351):
// logical columns [0, P+Q); column c < P is read from the slot at physical row c (or c % W for
// a sliding window), column c >= P from this step's ins row c - P; output row r attends to
// c <= P + r and, with a window, P + r - c < W; kv plane = floor((b*H + h) / r); rows >= Q
// are written as exact 0; the half-scale multiplies q and k.
//
// The reference materialises S, reduces row statistics and multiplies by V in three
// dispatches.  Here one launch streams K and V once with an online softmax:
//  * decode (Q = 1, M = 1): split-K.  A workgroup owns one KV head and one range of past
//    columns, loads that range's K and V with 16-byte coalesced loads, scores all r query
//    heads of the KV head against it (the KV bytes are read once, not r times), and writes
//    (max, sum, weighted V) partials that a second small kernel merges in split order.
//    The column partition depends only on the number of past columns, the head dim and the
//    slot dtype, so a sequence gives the same bits alone or inside a ragged batch.
//  * everything else (prefill chunks, pad rows, head dims the fast path does not cover):
//    a generic kernel, one workgroup per (plane, row).
#include "krm_internal.h"

#include <cmath>
#include <type_traits>

using namespace krm;

namespace {

constexpr int kThreads = 256;
constexpr int kDecodeIter = 8;  // K/V rows each lane group walks per split

template <typename T>
__device__ inline float ld_f32(const T* p, size_t i);
template <>
__device__ inline float ld_f32<float>(const float* p, size_t i) { return p[i]; }
template <>
__device__ inline float ld_f32<__half>(const __half* p, size_t i) { return __half2float(p[i]); }
template <typename T>
__device__ inline void st_f32(T* p, size_t i, float v);
template <>
__device__ inline void st_f32<float>(float* p, size_t i, float v) { p[i] = v; }
template <>
__device__ inline void st_f32<__half>(__half* p, size_t i, float v) { p[i] = __float2half_rn(v); }

// first logical column a row with causal limit `limit` may see (0 for a full context)
__host__ __device__ inline uint64_t window_low(uint32_t window, uint64_t limit) {
  return (window && limit + 1 > window) ? limit + 1 - window : 0;
}

// ------------------------------------------------------------------------------ generic

struct GenericArgs {
  uint32_t heads, kv_heads, chunk_rows, depth, capacity, window, past, query;
  float scale;
  uint32_t* lengths;  // device {past, query, fault} overriding past / query when not null
};

// Run-time lengths read on the device (the reference carries them in a uniform buffer the
// generation context rewrites every run, packages/runtime/src/kernels/state-attention.ts:
// 190-193).  The host checks of the scalar form are repeated here; a violation raises the
// fault word instead of touching memory.
__device__ inline bool device_lengths(uint32_t* lengths, uint32_t chunk_rows, uint32_t capacity,
                                      uint32_t window, uint32_t& past, uint32_t& query) {
  if (!lengths) return true;
  past = lengths[0];
  query = lengths[1];
  const bool ok = query >= 1 && query <= chunk_rows &&
                  (uint64_t)past + query <= 0xffffffffull &&
                  (window != 0 || (uint64_t)past + query <= capacity);
  if (!ok && threadIdx.x == 0) lengths[2] = 1u;
  return ok;
}

// One workgroup per (plane z = b*H + h, row).  Columns are walked 256 at a time: a thread
// scores one column (serial dot over D), the block folds the chunk into the running
// (max, sum), then threads switch to one output dim each and add the chunk's P*V.
template <typename XT, typename ST>
__global__ __launch_bounds__(kThreads) void attention_generic_kernel(
    const XT* __restrict__ q, const XT* __restrict__ ins_k, const XT* __restrict__ ins_v,
    const ST* __restrict__ slot_k, const ST* __restrict__ slot_v, XT* __restrict__ out,
    GenericArgs a) {
  __shared__ float s_q[1024];
  __shared__ float s_p[kThreads];
  __shared__ float s_red[kThreads / kWave];
  __shared__ float s_bcast;

  const uint32_t z = blockIdx.x;
  const uint32_t row = blockIdx.y;
  const uint32_t tid = threadIdx.x;
  const uint32_t D = a.depth;
  const size_t q_base = ((size_t)z * a.chunk_rows + row) * D;
  if (!device_lengths(a.lengths, a.chunk_rows, a.capacity, a.window, a.past, a.query)) return;

  if (row >= a.query) {  // pad row: exact zeros, nothing is read
    for (uint32_t d = tid; d < D; d += kThreads) st_f32<XT>(out, q_base + d, 0.0f);
    return;
  }
  const uint32_t kv_plane = z / (a.heads / a.kv_heads);
  const uint64_t limit = (uint64_t)a.past + row;
  const uint64_t lo = window_low(a.window, limit);
  const uint64_t count = limit - lo + 1;  // >= 1: the row always sees its own column

  for (uint32_t d = tid; d < D; d += kThreads) s_q[d] = ld_f32<XT>(q, q_base + d) * a.scale;
  __syncthreads();

  float run_max = -INFINITY, run_sum = 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};  // output dims tid, tid+256, ... (D <= 1024)

  for (uint64_t c0 = 0; c0 < count; c0 += kThreads) {
    const uint64_t col = lo + c0 + tid;
    const bool valid = c0 + tid < count;
    float score = -INFINITY;
    if (valid) {
      float dot = 0.f;
      if (col < a.past) {
        // (a slot column is below `past`, a u32: the ring row is a 32-bit modulo)
        const uint32_t prow = a.window ? (uint32_t)col % a.window : (uint32_t)col;
        const ST* kp = slot_k + ((size_t)kv_plane * a.capacity + prow) * D;
        for (uint32_t d = 0; d < D; ++d) dot = fmaf(s_q[d], ld_f32<ST>(kp, d) * a.scale, dot);
      } else {
        const XT* kp = ins_k + ((size_t)kv_plane * a.chunk_rows + (col - a.past)) * D;
        for (uint32_t d = 0; d < D; ++d) dot = fmaf(s_q[d], ld_f32<XT>(kp, d) * a.scale, dot);
      }
      score = dot;
    }
    // chunk max
    float m = score;
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, kWave));
    if ((tid & (kWave - 1)) == 0) s_red[tid >> 6] = m;
    __syncthreads();
    if (tid == 0) {
      float t = s_red[0];
      for (int i = 1; i < kThreads / kWave; ++i) t = fmaxf(t, s_red[i]);
      s_bcast = fmaxf(t, run_max);
    }
    __syncthreads();
    const float new_max = s_bcast;  // finite: every chunk holds at least one valid column
    const float alpha = expf(run_max - new_max);  // exp(-inf) = 0 on the first chunk
    const float p = valid ? expf(score - new_max) : 0.f;
    s_p[tid] = p;
    float s = p;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
    __syncthreads();  // s_p complete; s_red free to reuse
    if ((tid & (kWave - 1)) == 0) s_red[tid >> 6] = s;
    __syncthreads();
    float chunk_sum = 0.f;
    for (int i = 0; i < kThreads / kWave; ++i) chunk_sum += s_red[i];
    run_sum = run_sum * alpha + chunk_sum;
    run_max = new_max;

    const uint32_t ncols = (uint32_t)((count - c0) < kThreads ? (count - c0) : kThreads);
#pragma unroll
    for (int slot = 0; slot < 4; ++slot) {
      const uint32_t d = tid + slot * kThreads;
      if (d >= D) break;
      float sum = 0.f;
      for (uint32_t c = 0; c < ncols; ++c) {
        const uint64_t vc = lo + c0 + c;
        float v;
        if (vc < a.past) {
          const uint32_t prow = a.window ? (uint32_t)vc % a.window : (uint32_t)vc;
          v = ld_f32<ST>(slot_v, ((size_t)kv_plane * a.capacity + prow) * D + d);
        } else {
          v = ld_f32<XT>(ins_v, ((size_t)kv_plane * a.chunk_rows + (vc - a.past)) * D + d);
        }
        sum = fmaf(s_p[c], v, sum);
      }
      acc[slot] = acc[slot] * alpha + sum;
    }
    __syncthreads();  // before s_p / s_red are overwritten
  }
  const float inv = 1.0f / run_sum;  // run_sum >= 1: the max column contributes exp(0)
#pragma unroll
  for (int slot = 0; slot < 4; ++slot) {
    const uint32_t d = tid + slot * kThreads;
    if (d < D) st_f32<XT>(out, q_base + d, acc[slot] * inv);
  }
}

// ------------------------------------------------------------------- chunks of rows, MFMA
//
// A chunk of M > 1 rows with D = 64 or 128 (a prefill step): workgroup = (plane z, 16 query
// rows), WAVES waves; the key columns the 16 rows can see are walked in blocks of 32 and wave w
// takes blocks w, w + WAVES, ...  Products and sums are f32's.  Rows of f32 (the state's, or this step's
// beside an fp16 state) run on v_mfma_f32_16x16x4_f32 with the generic kernel's operand roundings: q *
// scale and k * scale are rounded before the product.  Blocks of fp16 rows run on
// v_mfma_f32_16x16x32_f16, sixteen times that rate: K and V are fp16 as they are, q is fp16 or three fp16 parts
// of the row times powers of two (all bits of an entry down to 2^-36 of the row's largest magnitude; a row with
// smaller ones is formed with f32 operands), a probability from 2^-16 on three parts of p 2^15 (all its bits; a row
// with a smaller one in the block multiplies V with f32 operands there), products are exact, sums f32, scale^2
// multiplies the f32 sum.
// Error against 64 bits (2-norm, f32 queries, normal values; all in f32 operands): D = 64 behind 1024
// 2.3e-7 (3.6e-7), D = 128 2.4e-7 (4.4e-7), D = 256 3.1e-7 (6.3e-7); queries four times as large 4.6e-7 (9.0e-7),
// 6.3e-7 (1.2e-6), 7.9e-7 (1.7e-6).  A part of zero beside an infinity
// of the state is a NaN that the value itself would not give, and 2^15 times a sum of this step's f32 rows
// can be infinite where the sum is not: a row whose sums are not finite is formed anew with f32 operands and
// without the factor, alone.  With g = lane / 16:
//   S^T = K Q^T    two tiles of 16 keys; A = the K tile (row = key, lane group g walks dims
//                  g D/4 ..), B = Q^T (column = query row): a lane ends up with the scores of
//                  ONE query row (lane % 16) against keys 16 t + 4 g + i (t < 2, i < 4), so the
//                  running maximum and sum of the online softmax are per lane, plus an
//                  exchange between the four lane groups;
//   O^T += V^T P^T the scores a lane holds are exactly a B operand if MFMA step (t, i) is
//                  given the keys 16 t + 4 g + i, so the probabilities never move; V^T is the A
//                  operand with the same key per step: 16 lanes take that key's row 16 bytes each
//                  and keep it in registers (a piece's four dims feed four output tiles), so V
//                  needs no LDS at all (fp16: the eight keys of a dim, two to a register, are one
//                  operand of 32 keys).
// The K block is parked in the wave's own LDS area (coalesced 16-byte loads; a block may straddle
// the state slot and this step's rows): read as an operand from memory it came in half lines,
// half as fast.  D = 64: the next block's rows are asked for as soon as this one's are used.  The
// waves' (max, sum, O) are merged in LDS at the end; rows >= query are written as +0.  Sixteen
// rows a workgroup (not 32) so that a 128-row chunk of 32 heads is 256 workgroups, one per CU.
// What bounds f32 rows is their matrix rate with two waves a SIMD to cover softmax and waits (D = 64,
// r = 8, 128 rows behind 1024: 8 us of MFMA), fp16 rows the vector instructions of softmax and operands.
// us with f32 operands / with fp16 ones / with fp16 ones where rows hold probabilities below 2^-16 (queries
// four times as large), 128 rows behind 1024 and 512 behind 2048: fp16 D = 64 19.1 / 10.5 / 15.2, 118 / 53 / 89; D =
// 128, r = 4 32 / 17 / 25, 234 / 106 / 166; D = 256, 16 heads, r = 8 71 / 36 / 56, 272 / 133 / 216; f32 queries D = 64
// 20.8 / 14.8 / 19.0, 130 / 80 / 115; D = 128 36 / 21 / 29, 265 / 140 / 207; D = 256 76 / 50 / 70, 302 / 196 / 275.
// (Two parts for every probability, 22 bits and nothing below 2^-40, and q's parts at one scale took 0 to 11 %
// less.)  Before those f32 forms, with V parked as well, rows looked up one by one (two element types: a wait
// at each), expf and no requests ahead, us before / with f32 operands: the case of 8 us of MFMA
// 22.7 / 19.3; fp16, D = 128, r = 4: 49.4 / 32.6; f32 over fp16 slots 106.5 / 36.8; D = 256, r = 8
// (two waves then, four now that LDS holds K alone): 172 / 71.
typedef float float4v_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

template <typename T>
__device__ inline float4 load4_f32(const T* p);
template <>
__device__ inline float4 load4_f32<float>(const float* p) {
  return *reinterpret_cast<const float4*>(p);
}
template <>
__device__ inline float4 load4_f32<__half>(const __half* p) {
  const uint2 raw = *reinterpret_cast<const uint2*>(p);
  const __half2 a = __builtin_bit_cast(__half2, raw.x), b = __builtin_bit_cast(__half2, raw.y);
  return make_float4(__low2float(a), __high2float(a), __low2float(b), __high2float(b));
}

// Halves (x = 32) or neighbouring rows (x = 16) of a wave trade places in one instruction: {a of
// the lanes whose bit x is clear | b of the same lanes, x further on} and the same of the lanes
// whose bit is set.
struct Exchanged {
  float clear, set;
};
__device__ inline Exchanged exchange(float a, float b, int x) {
  const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
  const auto s = x == 32 ? __builtin_amdgcn_permlane32_swap(ua, ub, false, false)
                         : __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
  return {__uint_as_float(s[0]), __uint_as_float(s[1])};
}
__device__ inline float exchange_max(float v, int x) {
  const Exchanged s = exchange(v, v, x);
  return fmaxf(s.clear, s.set);
}
// A 4-element piece of a row as it arrives: 16 bytes of f32 or 8 of fp16.
template <typename T>
__device__ inline uint4 load4_raw(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const uint4*>(p);
  } else {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_uint4(v.x, v.y, 0u, 0u);
  }
}
template <typename T>
__device__ inline float4 raw4_f32(const uint4& v) {
  if constexpr (sizeof(T) == 4) {
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                       __uint_as_float(v.w));
  } else {
    const __half2 a = __builtin_bit_cast(__half2, v.x), b = __builtin_bit_cast(__half2, v.y);
    return make_float4(__low2float(a), __high2float(a), __low2float(b), __high2float(b));
  }
}

// e^d for d <= 0 (or -inf: 0) with one v_exp_f32.  2^t with t = d log2 e rounded alone is off by up
// to |d| 2^-24 of itself; e^d = 2^t e^r with r = d - t ln 2, and r is so small that 1 + r is its
// exponential.  ln 2 in two parts, the first of 24 bits: the first difference is exact.  (The bounds
// hold r finite where 2^t is 0 anyway.)  2^t alone took 1 to 2 % less of a long chunk (512 rows behind
// 2048, D = 128, f32: 233 us, 237 so).
__device__ inline float exp_of_difference(float d) {
  const float t = d * 1.4426950408889634f;
  const float high = 0.69314718055994531f;
  const float low = (float)(0.693147180559945309417 - (double)0.69314718055994531f);
  const float r = __builtin_amdgcn_fmed3f(fmaf(-t, low, fmaf(-t, high, d)), -1.0f, 1.0f);
  const float p = __builtin_amdgcn_exp2f(t);
  return fmaf(p, r, p);
}

template <typename XT, typename ST, int D, int WAVES, int RB>
__global__ __launch_bounds__(64 * WAVES) void attention_rows_kernel(
    const XT* __restrict__ q, const XT* __restrict__ ins_k, const XT* __restrict__ ins_v,
    ST* __restrict__ slot_k, ST* __restrict__ slot_v, XT* __restrict__ out,
    GenericArgs a, uint32_t flags) {
  constexpr uint32_t kBlock = 64u * WAVES;
  constexpr int kRows = 16 * RB;              // query rows of a workgroup: RB blocks of 16
  constexpr int kRow = D + 4;                 // floats of a parked row
  constexpr int DT = D / 16;                  // output tiles of 16 dims
  constexpr int kQuarter = D / 4;             // dims a lane group walks
  constexpr int kVPieces = D / 64;            // 16-byte pieces of a V row a lane takes
  constexpr int kPieces = D / 4;              // 4-element pieces of a row
  constexpr int kRowsPerLoad = 64 / kPieces;
  constexpr int kLoads = 32 / kRowsPerLoad;
  // State rows of fp16 are products of fp16 operands: see `half_block` below.
  constexpr bool kHalf = sizeof(ST) == 2;
  constexpr int kHalfRow = D + 8;             // halves of a parked row
  // A probability from 2^-16 on is three fp16 parts of p 2^15, all its 24 bits: below that the last of them
  // lie under fp16's smallest step, and a row with such a probability takes f32 operands in that block.
  constexpr int kPParts = 3;
  constexpr float kPScale = 32768.0f, kPLeast = 1.0f / 65536.0f;
  constexpr int kQParts = sizeof(XT) == 2 ? 1 : 3, kSteps = D / 32;
  constexpr float kQNext = 2048.0f;
  __shared__ __align__(16) float s_k[WAVES][32 * kRow];
  constexpr bool kSplitQ = kHalf && sizeof(XT) == 4;
  __shared__ __align__(16) __half s_q[kSplitQ ? kQParts * kRows * kHalfRow : 8];  // the parts of Q
  __shared__ float s_factor[kSplitQ ? kRows : 1];                                // scale^2 2^-e of a row
  __shared__ float s_m[WAVES][kRows], s_l[WAVES][kRows];
  __shared__ uint32_t s_lost[WAVES];

  const uint32_t z = blockIdx.x, row0 = blockIdx.y * (uint32_t)kRows;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // key blocks are a wave's: scalar
  const int r = lane & 15, g = lane >> 4;
  uint32_t past = a.past, query = a.query;
  if (!device_lengths(a.lengths, a.chunk_rows, a.capacity, a.window, past, query)) return;

  const bool row_major = (flags & KRM_CHUNK_OUT_ROW_MAJOR) != 0;
  const bool out_f16 = (flags & KRM_CHUNK_OUT_F16) != 0;  // fp16 `out` beside f32 q / k / v
  auto out_index = [&](uint32_t row, uint32_t d) -> size_t {
    if (row_major) {  // [B, M, H, D]
      const uint32_t b = z / a.heads, head = z - b * a.heads;
      return (((size_t)b * a.chunk_rows + row) * a.heads + head) * D + d;
    }
    return ((size_t)z * a.chunk_rows + row) * D + d;
  };
  if (row0 >= query) {  // a block of pad rows: exact zeros, nothing is read
    for (uint32_t i = tid; i < (uint32_t)kRows * D; i += kBlock) {
      const uint32_t row = row0 + i / D;
      if (row >= a.chunk_rows) continue;
      if (out_f16)
        st_f32<__half>(reinterpret_cast<__half*>(out), out_index(row, i % D), 0.0f);
      else
        st_f32<XT>(out, out_index(row, i % D), 0.0f);
    }
    return;
  }
  // (scalar, which the compiler's division is not: the planes' addresses take no vector registers)
  const uint32_t kv_plane = __builtin_amdgcn_readfirstlane(z / (a.heads / a.kv_heads));

  // Q block: asked for first, parked (scaled) behind the request of the wave's first key block
  // (fp16 beside fp16 state rows: each lane's operand pieces instead, which never see the LDS)
  constexpr int kQUnits = kRows * kPieces, kQPer = (kQUnits + (int)kBlock - 1) / (int)kBlock;
  constexpr bool kQDirect = kHalf && sizeof(XT) == 2;
  half8_t qh[kQDirect ? RB : 1][kQDirect ? kSteps : 1];
  if constexpr (kQDirect) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const uint32_t row = min(row0 + 16u * rb + r, a.chunk_rows - 1);
#pragma unroll
      for (int i = 0; i < kSteps; ++i)
        qh[rb][i] = *reinterpret_cast<const half8_t*>(q + ((size_t)z * a.chunk_rows + row) * D + 32 * i + 8 * g);
    }
  }
  uint4 qraw[kQPer];
#pragma unroll
  for (int j = 0; j < kQPer && !kQDirect; ++j) {
    const uint32_t i = min((uint32_t)tid + j * kBlock, (uint32_t)kQUnits - 1u);
    const uint32_t row = min(row0 + i / kPieces, a.chunk_rows - 1);
    qraw[j] = load4_raw<XT>(q + ((size_t)z * a.chunk_rows + row) * D + 4 * (i % kPieces));
  }

  // columns the block's rows can see: [c_lo, limit_hi]
  const uint32_t last_row = min(row0 + (uint32_t)kRows - 1u, query - 1u);
  const uint64_t limit_hi = (uint64_t)past + last_row;
  const uint64_t c_lo = window_low(a.window, (uint64_t)past + row0);
  const uint32_t blocks = (uint32_t)((limit_hi - c_lo) / 32u) + 1u;
  uint64_t my_limit[RB], my_low[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    my_limit[rb] = (uint64_t)past + row0 + (uint32_t)(16 * rb + r);
    my_low[rb] = window_low(a.window, my_limit[rb]);
  }

  float* mk = s_k[wave];
  auto wave_sync = [] {  // the areas are the wave's own: its LDS queue orders them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  // Requests only: the K rows of key block kb (whole rows, parked in LDS later) and its V rows (in
  // the operand layout: step j of lane group g carries the key 16 (j / 4) + 4 g + j % 4, and 16
  // lanes take that row 16 bytes each).  Columns below `past` are slot rows, the rest this step's;
  // a column beyond the last one is the last one again, masked when used.  A block on one side of
  // `past` whose slot rows do not wrap is 32-bit offsets from one base; only the others look every
  // row up.
  const uint32_t load_key = lane / kPieces, load_piece = 4u * (lane % kPieces);
  // A lane's key number inside a block, from which its rows' numbers are formed anew for every block
  // where two element types meet: there every row keeps one of its own, and held over the walk these
  // took the state's registers to spilling.
  auto lane_number = [](uint32_t number) {
    if constexpr (sizeof(ST) != sizeof(XT)) asm volatile("" : "+v"(number));
    return number;
  };
  const size_t slot_plane = (size_t)kv_plane * a.capacity * D;
  const size_t ins_plane = (size_t)kv_plane * a.chunk_rows * D;
  auto slot_columns = [&](uint64_t c0) -> uint32_t {  // of the block's 32
    return c0 >= past ? 0u : (uint32_t)(past - c0 < 32u ? past - c0 : 32u);
  };
  // `keys` lane rows, row i the block's key lane_key + step_of(i), `pieces` pieces of 4 elements 64
  // apart
  auto request = [&](uint32_t kb, const ST* slot, const XT* ins, auto keys, uint32_t lane_key,
                     auto step_of, uint32_t lane_dim, auto pieces, auto& raw) __attribute__((always_inline)) {
    lane_key = lane_number(lane_key);
    constexpr int kKeys = decltype(keys)::value, kPer = decltype(pieces)::value;
    const uint64_t c0 = c_lo + (uint64_t)kb * 32u;
    const uint32_t slots = slot_columns(c0);
    const uint32_t first = a.window ? (uint32_t)c0 % a.window : (uint32_t)c0;
    if (slots == 32u && (a.window == 0 || first + 32u <= a.window)) {
      const ST* base = slot + slot_plane + (size_t)first * D;
#pragma unroll
      for (int i = 0; i < kKeys; ++i)
#pragma unroll
        for (int j = 0; j < kPer; ++j)
          raw[i * kPer + j] = load4_raw<ST>(base + ((lane_key + step_of(i)) * D + lane_dim + 64 * j));
    } else if (slots == 0u) {
      const XT* base = ins + ins_plane + (size_t)(c0 - past) * D;
      const uint32_t most = limit_hi - c0 < 31u ? (uint32_t)(limit_hi - c0) : 31u;
#pragma unroll
      for (int i = 0; i < kKeys; ++i)
#pragma unroll
        for (int j = 0; j < kPer; ++j)
          raw[i * kPer + j] = load4_raw<XT>(
              base + (min(lane_key + step_of(i), most) * D + lane_dim + 64 * j));
    } else {
#pragma unroll
      for (int i = 0; i < kKeys; ++i) {
        const uint32_t key = min(lane_key + step_of(i), (uint32_t)(limit_hi - c0 < 31u ? limit_hi - c0 : 31u));
        const bool in_slot = key < slots;
        uint32_t at = first + key;  // (a block of 32 wraps once, unless the window is shorter)
        if (a.window && at >= a.window) at = a.window >= 32u ? at - a.window : at % a.window;
        const size_t row = lane_dim + (in_slot ? slot_plane + (size_t)at * D
                                               : ins_plane + (size_t)(c0 + key - past) * D);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
          if constexpr (sizeof(ST) == sizeof(XT))
            raw[i * kPer + j] = load4_raw<XT>((in_slot ? reinterpret_cast<const XT*>(slot) : ins) + row + 64 * j);
          else
            raw[i * kPer + j] = in_slot ? load4_raw<ST>(slot + row + 64 * j) : load4_raw<XT>(ins + row + 64 * j);
        }
      }
    }
  };
  auto v_step = [](int j) -> uint32_t { return (uint32_t)(16 * (j / 4) + j % 4); };
  uint4 kraw[kLoads], vraw[8 * kVPieces];
  auto request_k = [&](uint32_t kb) __attribute__((always_inline)) {
    request(kb, slot_k, ins_k, std::integral_constant<int, kLoads>{}, load_key,
            [](int i) { return (uint32_t)(i * kRowsPerLoad); }, load_piece,
            std::integral_constant<int, 1>{}, kraw);
  };
  auto request_v = [&](uint32_t kb) __attribute__((always_inline)) {
    request(kb, slot_v, ins_v, std::integral_constant<int, 8>{}, 4u * g, v_step, 4u * r,
            std::integral_constant<int, kVPieces>{}, vraw);
  };
  // f32 of what arrived
  auto element4 = [&](const uint4& v, uint32_t key, uint32_t slots) {
    if constexpr (sizeof(ST) == sizeof(XT)) {
      return raw4_f32<XT>(v);
    } else {
      const float4 s4 = raw4_f32<ST>(v), x4 = raw4_f32<XT>(v);
      const bool in_slot = key < slots;
      return make_float4(in_slot ? s4.x : x4.x, in_slot ? s4.y : x4.y, in_slot ? s4.z : x4.z,
                         in_slot ? s4.w : x4.w);
    }
  };
  // (longer rows: the next block's beside this one's would take the registers of the state; f32 queries
  // beside fp16 rows of 128 spill with it, 128 rows behind 1024 24.7 us, 22.1 without)
  constexpr bool kAhead = D * sizeof(XT) * sizeof(ST) <= 64 * 16 && !(kSplitQ && D > 64);
  if (kAhead && (uint32_t)wave < blocks) {
    request_k((uint32_t)wave);
    request_v((uint32_t)wave);
  }

  // each lane's B operands: Q[r][g * D/4 + s]
  float qf[RB][kQDirect ? 1 : kQuarter];
  if constexpr (!kQDirect) {
    const bool split = kSplitQ && slot_columns(c_lo) == 32u;  // (no fp16 block, nothing to split)
#pragma unroll
    for (int j = 0; j < kQPer; ++j) {
      const uint32_t i = (uint32_t)tid + j * kBlock;
      float4 v = raw4_f32<XT>(qraw[j]);
      if (split) {
        // The row times 2^e, its largest magnitude in [2^13, 2^14), as three fp16 parts, each what the one
        // before it leaves times 2^11: all 24 bits of an entry down to 2^-36 of the largest, in sums of their
        // own that are put together at the end (at one scale the parts ended at 2^-24, and entries below 2^-14
        // of the largest lost bits).  A row with an entry that they do not hold gets a NaN for its factor, and
        // with it the second turn.  A row lies in kPieces neighbouring lanes.
        float top = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
#pragma unroll
        for (int off = 1; off < kPieces; off <<= 1) top = fmaxf(top, __shfl_xor(top, off, kWave));
        const int biased = (int)(__float_as_uint(top) >> 23);
        float up = 1.f, down = 1.f;
        if (top != 0.f && biased != 255) {
          int power = 13 - (biased - 127);
          power = power > 100 ? 100 : power < -100 ? -100 : power;  // (2^-e scale^2 stays normal)
          up = __uint_as_float((uint32_t)(127 + power) << 23);
          down = __uint_as_float((uint32_t)(127 - power) << 23);
        }
        float left[4] = {v.x * up, v.y * up, v.z * up, v.w * up};  // exact: a power of two
        __half parts[kQParts][4];
        bool whole = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int p = 0; p < kQParts; ++p) {
            parts[p][e] = __float2half_rn(left[e]);
            left[e] = (left[e] - __half2float(parts[p][e])) * kQNext;
          }
          whole = whole && left[e] == 0.f;
        }
        const uint64_t row_lanes = (kPieces == 64 ? ~0ull : (1ull << (kPieces % 64)) - 1ull) << (lane & ~(kPieces - 1));
        whole = (~__ballot(whole) & row_lanes) == 0;
        if (i < (uint32_t)kQUnits) {
          if (i % kPieces == 0) s_factor[i / kPieces] = whole ? a.scale * a.scale * down : NAN;
#pragma unroll
          for (int p = 0; p < kQParts; ++p)
            __builtin_memcpy(__builtin_assume_aligned(
                s_q + (p * kRows + i / kPieces) * kHalfRow + 4 * (i % kPieces), 8), parts[p], 8);
        }
      }
      v.x *= a.scale; v.y *= a.scale; v.z *= a.scale; v.w *= a.scale;
      if (i < (uint32_t)kQUnits)
        *reinterpret_cast<float4*>(&s_k[0][(i / kPieces) * kRow + 4 * (i % kPieces)]) = v;
    }
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < kQuarter / 4; ++i) {
        const float4 v = *reinterpret_cast<const float4*>(
            &s_k[0][(16 * rb + r) * kRow + g * kQuarter + 4 * i]);
        qf[rb][4 * i] = v.x; qf[rb][4 * i + 1] = v.y; qf[rb][4 * i + 2] = v.z; qf[rb][4 * i + 3] = v.w;
      }
    __syncthreads();
  }

  float run_m[RB], run_l[RB];
  float4v_t acc[RB][DT];
  // The end of a turn: the waves' states are merged, the rows `due` and not `lost` in any wave written, the
  // chunk's own rows stored by the first turn.  Returns the rows lost in any wave.
  auto finish = [&](uint32_t due, uint32_t lost, bool first) __attribute__((always_inline)) -> uint32_t {
  // The chunk's own K / V rows of this block go to the state slots when asked for (the first query
  // head of each kv plane does it; asked for here, stored behind the merge).  Without a window no
  // reader of this launch touches them: slot rows are read for columns < past only, these are
  // rows past + row.
  const bool append = (flags & KRM_CHUNK_APPEND) && z % (a.heads / a.kv_heads) == 0;
  uint4 own_k[kQPer], own_v[kQPer];
#pragma unroll
  for (int j = 0; j < kQPer; ++j) {
    const uint32_t i = min((uint32_t)tid + j * kBlock, (uint32_t)kQUnits - 1u);
    const uint32_t row = min(row0 + i / kPieces, query - 1u);
    const size_t src = ((size_t)kv_plane * a.chunk_rows + row) * D + 4 * (i % kPieces);
    if (append && first) {
      own_k[j] = load4_raw<XT>(ins_k + src);
      own_v[j] = load4_raw<XT>(ins_v + src);
    }
  }

  // the wave's state: (max, sum) per query row and O[row][d] in its own area
  if (kHalf && lane == 0) s_lost[wave] = lost;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    for (int x = 16; x <= 32; x <<= 1) {
      const Exchanged both = exchange(run_l[rb], run_l[rb], x);
      run_l[rb] = both.clear + both.set;
    }
    if (g == 0) {
      s_m[wave][16 * rb + r] = run_m[rb];
      s_l[wave][16 * rb + r] = run_l[rb];
    }
#pragma unroll
    for (int i = 0; i < kVPieces; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)  // register j of tiles 4 i + 0..3: dims 64 i + 16 g + 4 j + 0..3
        *reinterpret_cast<float4*>(&mk[(16 * rb + r) * kRow + 64 * i + 16 * g + 4 * j]) =
            make_float4(acc[rb][4 * i][j], acc[rb][4 * i + 1][j], acc[rb][4 * i + 2][j],
                        acc[rb][4 * i + 3][j]);
  }
  __syncthreads();

  if constexpr (kHalf) {
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv) lost |= s_lost[wv];
  }

  // merge of the waves, wave order: a row's dims dealt over the threads of its block of 16 rows (a
  // workgroup of two waves takes two rounds)
  constexpr uint32_t kUnits = kBlock < 256u ? 256u : kBlock;
  for (uint32_t unit = tid; unit < kUnits; unit += kBlock) {
   for (uint32_t rb = 0; rb < (uint32_t)RB; ++rb) {
    constexpr int kPer = 16 * D / (int)kUnits, kParts = D / kPer;
    const uint32_t rr = 16u * rb + unit / kParts, d0 = (unit % kParts) * kPer;
    const uint32_t row = row0 + rr;
    float top = s_m[0][rr];
#pragma unroll
    for (int wv = 1; wv < WAVES; ++wv) top = fmaxf(top, s_m[wv][rr]);  // finite: the own column
    float wgt[WAVES], total_l = 0.f;
#pragma unroll
    for (int wv = 0; wv < WAVES; ++wv) {
      wgt[wv] = expf(s_m[wv][rr] - top);
      total_l = fmaf(wgt[wv], s_l[wv][rr], total_l);
    }
    const float inv = 1.0f / total_l;
    if (row < a.chunk_rows && (!kHalf || (due & ~lost) >> rr & 1u)) {
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        float o = 0.f;
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) o = fmaf(wgt[wv], s_k[wv][rr * kRow + d0 + e], o);
        float value = row < query ? o * inv : 0.0f;
        if (out_f16 && sizeof(XT) == 4) value = rounded_f32(value);  // the f32 result, rounded again
        if (out_f16)
          st_f32<__half>(reinterpret_cast<__half*>(out), out_index(row, d0 + e), value);
        else
          st_f32<XT>(out, out_index(row, d0 + e), value);
      }
    }
   }
  }
  if (append && first) {
#pragma unroll
    for (int j = 0; j < kQPer; ++j) {
      const uint32_t i = (uint32_t)tid + j * kBlock, row = row0 + i / kPieces;
      if (i >= (uint32_t)kQUnits || row >= query) continue;
      const size_t dst = ((size_t)kv_plane * a.capacity + past + row) * D + 4 * (i % kPieces);
      const float4 kv = raw4_f32<XT>(own_k[j]), vv = raw4_f32<XT>(own_v[j]);
      st_f32<ST>(slot_k, dst, kv.x); st_f32<ST>(slot_k, dst + 1, kv.y);
      st_f32<ST>(slot_k, dst + 2, kv.z); st_f32<ST>(slot_k, dst + 3, kv.w);
      st_f32<ST>(slot_v, dst, vv.x); st_f32<ST>(slot_v, dst + 1, vv.y);
      st_f32<ST>(slot_v, dst + 2, vv.z); st_f32<ST>(slot_v, dst + 3, vv.w);
    }
  }
  return lost;
  };

  // One walk over the wave's key blocks: kNever, kAlways or (f32 queries: this step's own rows are f32)
  // kSlotBlocks with fp16 operands.
  enum { kNever, kAlways, kSlotBlocks };
  auto walk = [&](auto mode_tag) __attribute__((always_inline)) {
    constexpr int kMode = decltype(mode_tag)::value;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    run_m[rb] = -INFINITY;
    run_l[rb] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[rb][dt][i] = 0.f;
  }

  for (uint32_t kb = (uint32_t)wave; kb < blocks; kb += (uint32_t)WAVES) {
    const uint64_t c0 = c_lo + (uint64_t)kb * 32u;
    // park the K rows of the block (scaled), then ask for the next one's
    const bool more = kb + (uint32_t)WAVES < blocks;
    if constexpr (!kAhead) request_k(kb);
    const uint32_t slots = slot_columns(c0);
    const uint32_t parked_key = lane_number(load_key);
    // Every key of the block is fp16 as it lies in memory: it is parked so, and K Q^T and V^T P^T run
    // on v_mfma_f32_16x16x32_f16, sixteen times the rate of f32 operands.
    const bool half_block = kMode == kAlways || (kMode == kSlotBlocks && slots == 32u);
    if (half_block) {
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        *reinterpret_cast<uint2*>(reinterpret_cast<__half*>(mk) +
                                  (j * kRowsPerLoad + parked_key) * kHalfRow + load_piece) =
            make_uint2(kraw[j].x, kraw[j].y);
    } else
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const uint32_t key = j * kRowsPerLoad + parked_key;
      float4 kv = element4(kraw[j], key, slots);
      kv.x *= a.scale; kv.y *= a.scale; kv.z *= a.scale; kv.w *= a.scale;
      *reinterpret_cast<float4*>(&mk[key * kRow + load_piece]) = kv;
    }
    if constexpr (!kAhead) request_v(kb);
    if (kAhead && more) request_k(kb + (uint32_t)WAVES);
    wave_sync();

#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      // (a block past every column these 16 rows can see is skipped: the workgroup's other
      // rows see further)
      if (c0 > (uint64_t)past + row0 + (uint32_t)(16 * rb + 15)) continue;
      // S^T[key][query row], tile t = keys 16 t ..: A = K[16 t + r][g * D/4 + s], B = Q^T
      // (the two tiles, and below the dims, in turn: neighbouring MFMAs do not wait for each other)
      float4v_t st[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) st[t][i] = 0.f;
      if (half_block) {
        const __half* keys = reinterpret_cast<const __half*>(mk) + r * kHalfRow + 8 * g;
        const float factor = kQDirect ? a.scale * a.scale : s_factor[kSplitQ ? 16 * rb + r : 0];
        float4v_t sums[kQParts][2];  // of a part of q each
#pragma unroll
        for (int p = 0; p < kQParts; ++p) sums[p][0] = sums[p][1] = st[0];
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
          half8_t qs[kQParts];
#pragma unroll
          for (int p = 0; p < kQParts; ++p)
            qs[p] = kQDirect ? qh[kQDirect ? rb : 0][kQDirect ? i : 0]
                             : *reinterpret_cast<const half8_t*>(
                                   s_q + (p * kRows + 16 * rb + r) * kHalfRow + 32 * i + 8 * g);
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const half8_t kh = *reinterpret_cast<const half8_t*>(keys + 16 * t * kHalfRow + 32 * i);
#pragma unroll
            for (int p = 0; p < kQParts; ++p)
              sums[p][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qs[p], sums[p][t], 0, 0, 0);
          }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float sum = sums[kQParts - 1][t][i];
#pragma unroll
            for (int p = kQParts - 2; p >= 0; --p) sum = fmaf(sum, 1.0f / kQNext, sums[p][t][i]);
            st[t][i] = sum * factor;
          }
      } else {
        // The keys' next piece is read beside the products of this one where it gains (f32 rows, D = 64, 128
        // rows behind 1024 17.7 us left to the compiler, 17.5 so; D = 256 70.8 and 68.8; D = 128, 512 behind
        // 2048 234 and 235).
        constexpr bool kKeysAhead = !kHalf && D != 128;
        auto read_keys = [&](int i, float (&to)[2][4]) {
#pragma unroll
          for (int t = 0; t < 2; ++t)
            *reinterpret_cast<float4*>(to[t]) =
                *reinterpret_cast<const float4*>(&mk[(16 * t + r) * kRow + g * kQuarter + 4 * i]);
        };
        float next[2][4];
        if constexpr (kKeysAhead) {
          read_keys(0, next);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
#pragma unroll
        for (int i = 0; i < kQuarter / 4; ++i) {
          float qs[4];
          if constexpr (kQDirect) {  // (the second walk)
            const uint32_t row = min(row0 + (uint32_t)(16 * rb + r), a.chunk_rows - 1);
            const float4 v = load4_f32<XT>(q + ((size_t)z * a.chunk_rows + row) * D + g * kQuarter + 4 * i);
            qs[0] = v.x * a.scale; qs[1] = v.y * a.scale; qs[2] = v.z * a.scale; qs[3] = v.w * a.scale;
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) qs[j] = qf[rb][4 * i + j];
          }
          float kf[2][4];
          if constexpr (kKeysAhead) {
            __builtin_memcpy(kf, next, sizeof(kf));
            if (i + 1 < kQuarter / 4) read_keys(i + 1, next);
          } else {
            read_keys(i, kf);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t)
              st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t][j], qs[j], st[t], 0, 0, 0);
          if constexpr (kKeysAhead) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
          }
        }
      }
      // this lane: query row 16 rb + r, keys 16 t + 4 g + i
      // (uniform: a block that every one of these rows sees whole needs no mask)
      const uint64_t first_limit = (uint64_t)past + row0 + 16u * (uint32_t)rb;
      if (c0 + 31u > first_limit || window_low(a.window, first_limit + 15u) > c0) {
        const int last_key = my_limit[rb] < c0 ? -1 : (int)(my_limit[rb] - c0 < 32u ? my_limit[rb] - c0 : 32u);
        const int first_key = my_low[rb] <= c0 ? 0 : (int)(my_low[rb] - c0 < 32u ? my_low[rb] - c0 : 32u);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = 16 * t + 4 * g + i;
            if (key > last_key || key < first_key) st[t][i] = -INFINITY;
          }
      }
      float block_max = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) block_max = fmaxf(block_max, st[t][i]);
      block_max = exchange_max(exchange_max(block_max, 16), 32);
      const float new_m = fmaxf(run_m[rb], block_max);
      const float ref = new_m == -INFINITY ? 0.f : new_m;  // nothing seen yet: exp(-inf - 0) = 0
      // (expf's own range handling was a quarter of the loop's instructions)
      const float alpha = exp_of_difference(run_m[rb] - ref);
      float p[2][4], sum = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[t][i] = exp_of_difference(st[t][i] - ref);  // 0 where masked
          sum += p[t][i];
        }
      run_l[rb] = run_l[rb] * alpha + sum;
      run_m[rb] = new_m;
      // O^T[d][query row] = alpha * O^T + V^T P^T: step (t, i) carries the keys 16 t + 4 g + i
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rb][dt][i] *= alpha;
      // (tile dt = 4 i + e holds the dims 64 i + 4 r + e: a 16-byte piece feeds four tiles)
      const uint32_t pv_key = lane_number(4u * g);
      if constexpr (kMode != kNever) {  // (the sums of V are kept times 2^15: small probabilities keep their bits)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) p[t][i] *= kPScale;
      }
      // Rows with such a small probability in the block take f32 operands, the others of the sixteen see zeros
      // there: a row's sums do not depend on its neighbours.
      bool small = !half_block, some_small = small, all_small = small;
      if (kMode != kNever && half_block) {
        uint32_t least = 0xffffffffu;  // (of the bits less one: a zero comes out on top)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) least = min(least, __float_as_uint(p[t][i]) - 1u);
        small = least < __float_as_uint(kPLeast * kPScale) - 1u;
        const uint64_t lanes = __ballot(small);  // (a row's keys lie in four lanes)
        some_small = lanes != 0;
        if (some_small) {
          const uint64_t pairs = lanes | lanes >> 32;
          const uint32_t rows = (uint32_t)(pairs | pairs >> 16) & 0xffffu;
          small = (rows >> r & 1u) != 0;
          all_small = rows == 0xffffu;
        }
      }
      if (some_small)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float weight = small ? p[j / 4][j % 4] : 0.f;
        p[j / 4][j % 4] = small ? 0.f : p[j / 4][j % 4];
#pragma unroll
        for (int i = 0; i < kVPieces; ++i) {
          const float4 v4 = element4(vraw[j * kVPieces + i], pv_key + v_step(j), slots);
          const float vf[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[rb][4 * i + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[e], weight, acc[rb][4 * i + e], 0, 0, 0);
        }
      }
      if (!all_small) {
        half8_t ph[kPParts];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float left = p[j / 4][j % 4];
#pragma unroll
          for (int q = 0; q < kPParts; ++q) {
            const _Float16 part = (_Float16)left;
            ph[q][j] = part;
            left -= (float)part;
          }
        }
#pragma unroll
        for (int i = 0; i < kVPieces; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            uint32_t pair[4];  // dim e of the pieces of keys 2 q, 2 q + 1
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const uint4& v0 = vraw[2 * q * kVPieces + i];
              const uint4& v1 = vraw[(2 * q + 1) * kVPieces + i];
              pair[q] = __builtin_amdgcn_perm(e < 2 ? v1.x : v1.y, e < 2 ? v0.x : v0.y,
                                              e % 2 ? 0x07060302u : 0x05040100u);
            }
            const half8_t vh = __builtin_bit_cast(half8_t, make_uint4(pair[0], pair[1], pair[2], pair[3]));
#pragma unroll
            for (int q = kPParts - 1; q >= 0; --q)
              acc[rb][4 * i + e] =
                  __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[q], acc[rb][4 * i + e], 0, 0, 0);
          }
      }
    }
    if (kAhead && more) request_v(kb + (uint32_t)WAVES);
    wave_sync();  // the block's rows have been read: the next block may be parked
  }
  };
  // One turn writes every row.  Over an fp16 state a row whose sums are not finite in some wave is written by a
  // second turn, with f32 operands and without the factor: parts of a value meet an infinity of the state
  // as 0 * inf, the value itself does not, and 2^15 takes sums of this step's f32 rows past f32's range from
  // 1e34 on.  The other rows keep what the first turn wrote, whatever stands beside them.
  constexpr uint32_t kEvery = 0xffffffffu;  // a bit for each row of the workgroup
  uint32_t due = kEvery;
  bool first = true;
  if constexpr (kHalf) {
    if (!kSplitQ || slot_columns(c_lo) == 32u) {  // (else there is no block of fp16 keys)
      walk(std::integral_constant<int, sizeof(XT) == 2 ? kAlways : kSlotBlocks>{});
      uint32_t lost = 0;  // of the wave's rows
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        bool here = !(fabsf(run_l[rb]) < INFINITY);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            here = here || !(fabsf(acc[rb][dt][i]) < INFINITY);
            acc[rb][dt][i] *= 1.0f / kPScale;
          }
        const uint64_t lanes = __ballot(here && row0 + (uint32_t)(16 * rb + r) < query);
        const uint64_t pairs = lanes | lanes >> 32;
        lost |= ((uint32_t)(pairs | pairs >> 16) & 0xffffu) << (16 * rb);
      }
      due = finish(kEvery, lost, true);
      if (due == 0) return;  // (the same rows in every thread)
      first = false;
      __syncthreads();  // the waves' states have been read: their areas take key blocks again
      if (kAhead && (uint32_t)wave < blocks) {
        request_k((uint32_t)wave);
        request_v((uint32_t)wave);
      }
    }
  }
  walk(std::integral_constant<int, kNever>{});
  finish(due, 0u, first);
}

// ------------------------------------------------------------------------------ decode

typedef float float4_t __attribute__((ext_vector_type(4)));

// Value of lane `src` (0..15) of the caller's 16-lane row, in every lane of that row.
template <int SRC>
__device__ inline float row_broadcast_from(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + SRC, 0xf, 0xf, true));
}
__device__ inline float row_broadcast(float v, int src) {  // `src` is a constant after unrolling
  switch (src) {
    case 0: return row_broadcast_from<0>(v);
    case 1: return row_broadcast_from<1>(v);
    case 2: return row_broadcast_from<2>(v);
    case 3: return row_broadcast_from<3>(v);
    case 4: return row_broadcast_from<4>(v);
    case 5: return row_broadcast_from<5>(v);
    case 6: return row_broadcast_from<6>(v);
    default: return row_broadcast_from<7>(v);
  }
}

// Sum over the LPR consecutive lanes that share one K/V row; all of them get the total.
template <int LPR>
__device__ inline float group_sum(float v) {
  if constexpr (LPR >= 2) {
    int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true);
    v += __builtin_bit_cast(float, t);  // quad_perm [1,0,3,2]
  }
  if constexpr (LPR >= 4) {
    int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true);
    v += __builtin_bit_cast(float, t);  // quad_perm [2,3,0,1]
  }
  if constexpr (LPR >= 8) {
    int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true);
    v += __builtin_bit_cast(float, t);  // row_half_mirror
  }
  if constexpr (LPR >= 16) {
    int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true);
    v += __builtin_bit_cast(float, t);  // row_mirror
  }
  if constexpr (LPR >= 32) v += __shfl_xor(v, 16, kWave);
  if constexpr (LPR >= 64) v += __shfl_xor(v, 32, kWave);
  return v;
}

// Sums of N values (a power of two) over the four 16-lane rows of a wave, each lane left with its
// share of them: returns the index of the first and leaves max(1, N / 4) totals in v[0..].  A
// value's tree is the same for every N.
template <int N>
__device__ inline int sum_rows(float (&v)[N], int lane) {
  int n = N, first = 0;
#pragma unroll
  for (int x = 32; x >= 16; x >>= 1) {
    if (n > 1) {
      n >>= 1;
#pragma unroll
      for (int i = 0; i < N / 2; ++i) {
        if (i >= n) continue;
        const Exchanged s = exchange(v[i], v[i + n], x);
        v[i] = s.clear + s.set;
      }
      first += (lane & x) ? n : 0;
    } else {
      const Exchanged s = exchange(v[0], v[0], x);
      v[0] = s.clear + s.set;
    }
  }
  return first;
}

template <typename ST>
struct RowChunk;  // 16 bytes of a K/V row
template <>
struct RowChunk<__half> {
  static constexpr int E = 8;
  __device__ static inline void unpack(const uint4& raw, float (&f)[8]) {
    const __half2* h = reinterpret_cast<const __half2*>(&raw);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 v = __half22float2(h[i]);
      f[2 * i] = v.x;
      f[2 * i + 1] = v.y;
    }
  }
};
template <>
struct RowChunk<float> {
  static constexpr int E = 4;
  __device__ static inline void unpack(const uint4& raw, float (&f)[4]) {
    f[0] = __uint_as_float(raw.x);
    f[1] = __uint_as_float(raw.y);
    f[2] = __uint_as_float(raw.z);
    f[3] = __uint_as_float(raw.w);
  }
};

struct DecodeArgs {
  uint32_t heads, kv_heads;
  uint32_t repeat;           // query heads per kv head (H / Hkv)
  uint32_t head_groups;      // workgroups one kv head's query heads are spread over
  uint32_t window;           // 0 = full context
  uint32_t past;             // single sequence: P.  ragged batch: unused
  uint64_t slot_batch_stride;  // elements between batches of the slot (0 for a ragged batch)
  uint64_t slot_plane_stride;  // elements between kv heads of the slot
  float scale;
  uint32_t nseq;             // ragged batch: sequences; single: batch
  const int32_t* cu_rows;    // ragged batch: [nseq+1] first slot row of each sequence
  const int32_t* split_prefix;  // ragged batch: [nseq+1] first global split of each sequence
  uint32_t* tickets;         // arrival counter (sequence, head unit) at index * kTicketStride, zero between launches
  uint32_t* lengths;         // single sequence: device {past, query, fault} or null
  uint32_t capacity;         // single sequence: slot rows (checked against device lengths)
  uint32_t splits;           // that the grid and the workspace are sized for
  uint32_t units;            // kv heads * head_groups
  // Not 0: the grid is (8 units, splits / 8, batch), else (splits, units, batch).  Bits 4 and 8: XCDs by which the last
  // splits of a kv head and of a batch entry begin behind those of the one before.
  uint32_t folded;
};

// Columns are walked in chunks of kDecodeIter * G rows (G = 256 / lanes-per-row groups, each
// owning one row per iteration).  Short pasts (<= kSingleSplitChunks chunks) stay in ONE split
// that loops over its chunks — no partials, no merge; longer ones get one chunk per split.
// The rule is a pure function of the number of past columns and the chunk size, so a sequence
// is partitioned the same way alone and inside a ragged batch.
constexpr uint32_t kSingleSplitChunks = 4;
__host__ __device__ inline uint32_t decode_split_columns(uint32_t lanes_per_row) {
  return kDecodeIter * (kThreads / lanes_per_row);
}
__host__ __device__ inline uint32_t decode_chunks(uint64_t slot_columns, uint32_t chunk_columns) {
  return (uint32_t)((slot_columns + chunk_columns - 1) / chunk_columns);
}
// Chunks a split of a long past walks.  Two (both requested before the first is scored) halve
// the partials and help a launch that is bandwidth-bound — the 16-sequence ragged batch went
// from 36.7 to 33.9 us — but a single 4096-column sequence then has 256 workgroups instead of
// 512 and went from 10.1 to 12.6 us; the partition has to be the same function of a
// sequence's columns in both launches (a sequence gives the same bits alone and in a batch),
// so it stays at one.
#ifndef KRM_SPLIT_CHUNKS
#define KRM_SPLIT_CHUNKS 1
#endif
constexpr uint32_t kSplitChunks = KRM_SPLIT_CHUNKS;
__host__ __device__ inline uint32_t decode_splits(uint64_t slot_columns, uint32_t chunk_columns) {
  const uint32_t chunks = decode_chunks(slot_columns, chunk_columns);
  return chunks <= kSingleSplitChunks ? 1u : (chunks + kSplitChunks - 1) / kSplitChunks;
}

constexpr float kLog2e = 1.4426950408889634f;

// Device-scope store / load of one float: written through to (read from) memory that every
// XCD sees, without touching the rest of the cache.
__device__ inline void publish(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float observe(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
constexpr int kMergeChunk = 32;  // split partials merged per pass (all requested at once)
constexpr int kMergeBlock = 8;   // rows of a pass that are asked for or left out together

// Workgroup = (split, kv head, batch | -): 256 threads = G groups of LPR lanes; a group owns
// one K/V row per iteration, a lane 16 bytes of it.  Every group keeps its own running
// (max, sum, weighted V) over the rows it sees — no workgroup barrier inside the column walk —
// and the group states (where the scores run on the matrix cores: four wave states) are merged
// once at the end, in ascending order.  Scores live in the base-2 domain (q carries
// scale^2 * log2 e), so exponentials are single v_exp_f32.
// With several splits every workgroup publishes its merged partial; the one that arrives last
// at the (sequence, kv head) counter merges the partials of its r heads in ascending split
// order — the result does not depend on which workgroup that is.
// What bounds a long launch is the chain of one workgroup (addresses, rows, scores, P * V, merge,
// publish: half of a wave's time is waiting) against how many of them a CU holds.  fp16, r = 4,
// D = 128, sixteen ragged sequences of 4096 columns at most: held to two waves a SIMD and with
// every head's exponentials in every lane 178 us for four layers (3.1 TB/s); at three waves a SIMD
// 158; with a wave's softmax shared by its lanes and its groups summed in registers 151
// (3.7 TB/s).  Forced to four waves it spills: 168.
template <typename XT, typename ST, int R, int LPR, bool RAGGED>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 4)))
void attention_decode_kernel(
    const XT* __restrict__ q, const XT* __restrict__ ins_k, const XT* __restrict__ ins_v,
    const ST* __restrict__ slot_k, const ST* __restrict__ slot_v, XT* __restrict__ out,
    float* ws_ml, float* ws_acc, DecodeArgs a) {
  constexpr int E = RowChunk<ST>::E;
  constexpr int D = LPR * E;
  constexpr int G = kThreads / LPR;
  constexpr int kChunkCols = kDecodeIter * G;
  // fp16 queries and fp16 rows of 128 dims: the scores run on the matrix cores
  constexpr bool kMfma = sizeof(XT) == 2 && sizeof(ST) == 2 && LPR == 16 && kDecodeIter == 8;
  constexpr int kParts = kMfma ? kThreads / kWave : G;  // states merged through LDS
  constexpr int kOuts = (R * D + kThreads - 1) / kThreads;
  __shared__ float s_m[kParts][R];
  __shared__ float s_l[kParts][R];
  __shared__ __align__(16) float s_acc[kParts][R * D];
  __shared__ float s_w[R][kMergeChunk];
  __shared__ float s_wl[R][kMergeChunk];
  __shared__ uint32_t s_ticket;

  const int tid = threadIdx.x;
  const int sub = tid % LPR;   // which 16 bytes of the row
  const int group = tid / LPR;
  // Workgroups that share a split's rows (head groups of a kv head) follow each other on one XCD, whose L2 then has
  // the rows for all of them: workgroups go to the eight XCDs in turn.  (Splits and head groups as the two sides of the grid:
  // the same XCD where the splits are a multiple of eight, every XCD reading every row elsewhere.)  us before / now:
  // f32 32 heads of 8, D = 128, 4000 columns (63 splits) 17.3 / 12.1, 600 8.4 / 6.8; 8 heads of 2 11.7 / 8.3; 8 heads of 1,
  // D = 256, 4000 20.9 / 14.7, fp16 12.2 / 8.6, ragged 25 sequences up to 2602 51.2 / 43.9; fp16 32 of 8, D = 128, 4095 (32
  // splits) 8.71 / 8.48.
  const uint32_t unit = a.folded ? blockIdx.x >> 3 : blockIdx.y;
  const uint32_t hk = unit / a.head_groups;
  // Each kv head's splits begin on the XCD behind the one before it; the last ones, fewer than eight, begin behind the
  // last one of the head before, or some XCDs would have up to one more of every head.
  uint32_t at_split = blockIdx.x;
  if (a.folded) {
    const uint32_t first_xcd =
        blockIdx.y == a.splits >> 3 ? blockIdx.z * (a.folded >> 8) + hk * (a.folded >> 4) : hk;  // (modulo eight)
    at_split = blockIdx.y * 8u + ((blockIdx.x - first_xcd) & 7u);
  }
  const uint32_t head0 = hk * a.repeat + (unit - hk * a.head_groups) * R;  // first head

  // The rows of a chunk as they arrive: K pieces (row-owner layout, or the MFMA A-operand
  // layout: piece tile*4 + t) and V pieces (row-owner layout).
  struct ChunkRows {
    uint4 k[kDecodeIter];
    uint4 v[kDecodeIter];
  };
  const int wave = tid >> 6, lane = tid & 63;
  const int frag_row = lane & 15, frag_g = lane >> 4;
  // offset inside a chunk of the column that (lane group, iteration) owns
  auto column_of = [&](int it) -> uint32_t {
    if constexpr (kMfma)
      return (uint32_t)((wave * 2 + it / 4) * 16 + 4 * frag_g + (it & 3));
    else
      return (uint32_t)(it * G + group);
  };
  // Requests only: every K row, then every V row of the `width` columns from c_begin of a slot;
  // unconditional (a column past the end re-reads the first column and is masked when used).
  auto request_rows = [&](const ST* kslot, const ST* vslot, uint32_t first_row, uint32_t c_begin,
                          uint32_t width, ChunkRows& rows) {
    // Physical row of column c_begin, found once; the columns of a chunk follow it and wrap
    // at most once (a launch's live slot columns number fewer than the window).  A modulo per
    // request cost about 35 instructions and a branch each: 0.9 us to ask for a chunk's rows.
    const uint32_t r_begin = a.window ? c_begin % a.window : c_begin;
    const uint32_t wrap = a.window ? a.window : 0xFFFFFFFFu;
    auto slot_row = [&](uint32_t offset) {  // element offset of the row's first dim
      const uint32_t r = r_begin + (offset < width ? offset : 0u);
      return (size_t)(first_row + (r >= wrap ? r - wrap : r)) * D;
    };
    if constexpr (kMfma) {
      // lane (r = lane % 16, g = lane / 16) takes 16 bytes of K row r of each 16-row tile at
      // dims 32t + 8g..: the A-operand layout of v_mfma_f32_16x16x32_f16
#pragma unroll
      for (int tile = 0; tile < 2; ++tile) {
        const size_t at = slot_row((uint32_t)((wave * 2 + tile) * 16 + frag_row));
#pragma unroll
        for (int t = 0; t < 4; ++t)
          rows.k[tile * 4 + t] =
              *reinterpret_cast<const uint4*>(kslot + at + 32 * t + 8 * frag_g);
      }
    } else {
#pragma unroll
      for (int it = 0; it < kDecodeIter; ++it)
        rows.k[it] = *reinterpret_cast<const uint4*>(kslot + slot_row(column_of(it)) + sub * E);
    }
#pragma unroll
    for (int it = 0; it < kDecodeIter; ++it)
      rows.v[it] = *reinterpret_cast<const uint4*>(vslot + slot_row(column_of(it)) + sub * E);
  };

  // Lengths that live on the device (a recorded decode step) cost a dependent round trip before
  // the first address is known.  Without a window the first chunk of a split does not depend
  // on them — only how many of its columns count does — so its rows are asked for right away,
  // bounded by the slot's capacity instead of the past; columns that turn out to lie beyond
  // the past are masked when the chunk is used, like any ragged end.
  ChunkRows rows0;
  bool early = false;
  if constexpr (!RAGGED) {
    early = a.lengths != nullptr && a.window == 0;
    if (early) {
      const size_t base = (size_t)blockIdx.z * a.slot_batch_stride + (size_t)hk * a.slot_plane_stride;
      const uint32_t want = at_split * (kSplitChunks * (uint32_t)kChunkCols);
      const uint32_t c_begin = want < a.capacity ? want : a.capacity - 1u;
      const uint32_t room = a.capacity - c_begin;
      request_rows(slot_k + base, slot_v + base, 0u, c_begin,
                   room < (uint32_t)kChunkCols ? room : (uint32_t)kChunkCols, rows0);
    }
  }

  // Columns and slot rows are 32-bit (pastLength is a u32, a ragged batch holds < 2^31 rows);
  // only the final byte address is 64-bit: 64-bit index math per load costs more than the
  // attention arithmetic of a short past.
  uint32_t seq, split, nsplit, first_split;
  uint32_t past, row_base;
  if constexpr (RAGGED) {
    // The last sequence whose first split is <= at_split, 64 sequences at a time: every lane
    // asks for one sequence's entries at once, so the tables cost one round trip (a binary search
    // cost log2(nseq) of them in a row, 0.6 us each, in front of the first row's address).
    uint32_t first_of = 0, next_of = 0, row_of = 0, row_end_of = 0;
    seq = 0;
    for (uint32_t base = 0;; base += kWave) {
      const uint32_t i = min(base + (uint32_t)lane, a.nseq - 1u);
      first_of = (uint32_t)a.split_prefix[i];
      next_of = (uint32_t)a.split_prefix[i + 1];
      row_of = (uint32_t)a.cu_rows[i];
      row_end_of = (uint32_t)a.cu_rows[i + 1];
      const uint64_t mine = __ballot(base + (uint32_t)lane < a.nseq && first_of <= at_split &&
                                     at_split < next_of);
      if (mine) {
        const int owner = __builtin_ctzll(mine);
        seq = base + owner;
        first_of = __builtin_amdgcn_readlane(first_of, owner);
        next_of = __builtin_amdgcn_readlane(next_of, owner);
        row_of = __builtin_amdgcn_readlane(row_of, owner);
        row_end_of = __builtin_amdgcn_readlane(row_end_of, owner);
        break;
      }
      if (base + kWave >= a.nseq) return;  // a grid sized for the most splits the batch may need
    }
    first_split = first_of;
    nsplit = next_of - first_of;
    split = at_split - first_split;
    row_base = row_of;
    past = row_end_of - row_of;
  } else {
    seq = blockIdx.z;
    uint32_t p32 = a.past, q32 = 1;
    if (!device_lengths(a.lengths, 1, a.capacity, a.window, p32, q32)) return;
    past = p32;
    row_base = 0;
    nsplit = decode_splits(past - window_low(a.window, past), kChunkCols);
    split = at_split;
    // The grid and the workspace were sized on the host for the longest past the launch may
    // see.  A replay whose device-side past needs more splits than that would never complete a
    // ticket round and would index partials beyond the workspace: raise the fault word and
    // leave everything untouched instead.
    if (nsplit > a.splits) {
      if (a.lengths && at_split == 0 && unit == 0 && tid == 0) a.lengths[2] = 1u;
      return;
    }
    if (split >= nsplit) return;  // the grid is sized for the longest past it may see
    first_split = seq * nsplit;
  }
  const uint32_t low = (uint32_t)window_low(a.window, past);  // limit of row 0 is `past`
  const uint32_t total_chunks = decode_chunks(past - low, kChunkCols);
  const uint32_t my_chunks =
      nsplit == 1 ? total_chunks : min(kSplitChunks, total_chunks - split * kSplitChunks);
  const uint32_t c_first = low + split * (kSplitChunks * kChunkCols);  // < past (split 0 alone)
  const bool last = split + 1 == nsplit;

  const size_t slot_base = (size_t)seq * a.slot_batch_stride + (size_t)hk * a.slot_plane_stride;
  const ST* kslot = slot_k + slot_base;
  const ST* vslot = slot_v + slot_base;

  const bool own = last && group == 0;  // the lanes that also take this step's own column
  // This step's own row and the query heads (valid addresses for every lane)
  const size_t ins_base = ((size_t)seq * a.kv_heads + hk) * D;
  float kx[kMfma ? 1 : E], vx[kMfma ? 1 : E], qf[kMfma ? 1 : R][E];
  if constexpr (!kMfma) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      kx[e] = ld_f32<XT>(ins_k, ins_base + sub * E + e);
      vx[e] = ld_f32<XT>(ins_v, ins_base + sub * E + e);
    }
#pragma unroll
    for (int h = 0; h < R; ++h) {
      const size_t q_base = ((size_t)seq * a.heads + head0 + h) * D + sub * E;
#pragma unroll
      for (int e = 0; e < E; ++e)
        qf[h][e] = ((ld_f32<XT>(q, q_base + e) * a.scale) * a.scale) * kLog2e;
    }
  }

  // (this step's rows may start at any element: 16 bytes at once, but not 16-byte aligned)
  struct __attribute__((packed, aligned(2))) ElementAligned {
    uint32_t x, y, z, w;
  };
  auto load_own = [](const XT* p) {
    const ElementAligned v = *reinterpret_cast<const ElementAligned*>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
  };
  // B operand of the score MFMAs: lane (n = lane % 16, g = lane / 16) holds head n's query at
  // dims 32t + 8g.. as raw fp16 (exact products; the scale is applied to the f32 score)
  half8_t qb[kMfma ? 4 : 1];
  // ... and the A operand whose 16 rows are all this step's own K row: its products are the own
  // column's scores, head n's in every register of lane n.
  half8_t own_k[kMfma ? 4 : 1];
  uint4 own_v;
  if constexpr (kMfma) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      own_k[t] = __builtin_bit_cast(half8_t, load_own(ins_k + ins_base + 32 * t + 8 * frag_g));
    own_v = load_own(ins_v + ins_base + sub * E);
    const int n = tid & 15, g = (tid & 63) >> 4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const size_t at = ((size_t)seq * a.heads + head0 + (n < R ? n : 0)) * D + 32 * t + 8 * g;
      uint4 raw = *reinterpret_cast<const uint4*>(reinterpret_cast<const __half*>(q) + at);
      const uint32_t keep_bits = n < R ? 0xFFFFFFFFu : 0u;
      raw.x &= keep_bits; raw.y &= keep_bits; raw.z &= keep_bits; raw.w &= keep_bits;
      qb[t] = __builtin_bit_cast(half8_t, raw);
    }
  }

  // Running state.  Where the scores run on the matrix cores, lane n of every 16-lane row keeps
  // head n's maximum (one for the whole wave) and its own groups' sum, so a chunk costs a lane
  // eight exponentials whatever the number of heads; elsewhere a group keeps every head's.
  constexpr int kStates = kMfma ? 1 : R;
  float run_m[kStates], run_l[kStates], acc[R][E];
#pragma unroll
  for (int h = 0; h < kStates; ++h) {
    run_m[h] = -INFINITY;
    run_l[h] = 0.f;
  }
#pragma unroll
  for (int h = 0; h < R; ++h)
#pragma unroll
    for (int e = 0; e < E; ++e) acc[h][e] = 0.f;

  auto chunk_begin = [&](uint32_t chunk) { return c_first + chunk * kChunkCols; };
  auto chunk_end = [&](uint32_t c_begin) {  // c_begin < past: no overflow
    return past - c_begin > (uint32_t)kChunkCols ? c_begin + kChunkCols : past;
  };
  auto load_chunk = [&](uint32_t chunk, ChunkRows& rows) {
    const uint32_t c_begin = chunk_begin(chunk);
    request_rows(kslot, vslot, row_base, c_begin, chunk_end(c_begin) - c_begin, rows);
  };
  auto consume_chunk = [&](uint32_t chunk, ChunkRows& rows) {
    const uint32_t c_begin = chunk_begin(chunk), width = chunk_end(c_begin) - c_begin;
    bool valid[kDecodeIter];
#pragma unroll
    for (int it = 0; it < kDecodeIter; ++it) valid[it] = column_of(it) < width;
    float sc[kDecodeIter][kStates];  // score, then probability
    float cm[kStates];
#pragma unroll
    for (int h = 0; h < kStates; ++h) cm[h] = -INFINITY;
    if constexpr (kMfma) {
      // Scores on the matrix cores: the query heads are the B operand (one column per head);
      // lane (h, g) receives the scores of columns 4g..4g+3 of a tile for head h, and lane
      // group g owns exactly those columns for P*V, so a score reaches its group with one
      // broadcast inside the 16-lane row.
      float4_t scores[2];
#pragma unroll
      for (int tile = 0; tile < 2; ++tile) {
        scores[tile] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t)
          scores[tile] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(half8_t, rows.k[tile * 4 + t]), qb[t], scores[tile], 0, 0, 0);
      }
      const float qscale = (a.scale * a.scale) * kLog2e;
#pragma unroll
      for (int it = 0; it < kDecodeIter; ++it) {
        // (column of `it`, head lane % 16)
        sc[it][0] = valid[it] ? scores[it / 4][it & 3] * qscale : -INFINITY;
        cm[0] = fmaxf(cm[0], sc[it][0]);
      }
      cm[0] = exchange_max(exchange_max(cm[0], 32), 16);
    } else {
#pragma unroll
      for (int it = 0; it < kDecodeIter; ++it) {
        float kf[E];
        RowChunk<ST>::unpack(rows.k[it], kf);
#pragma unroll
        for (int h = 0; h < R; ++h) {
          float part = 0.f;
#pragma unroll
          for (int e = 0; e < E; ++e) part = fmaf(qf[h][e], kf[e], part);
          part = group_sum<LPR>(part);
          sc[it][h] = valid[it] ? part : -INFINITY;
          cm[h] = fmaxf(cm[h], sc[it][h]);
        }
      }
    }
    float keep[kStates];
#pragma unroll
    for (int h = 0; h < kStates; ++h) {
      const float m_new = fmaxf(run_m[h], cm[h]);
      const float ref = m_new == -INFINITY ? 0.f : m_new;  // nothing seen yet: 2^(-inf - 0) = 0
      keep[h] = __builtin_amdgcn_exp2f(run_m[h] - ref);
      run_m[h] = m_new;
      run_l[h] *= keep[h];
#pragma unroll
      for (int it = 0; it < kDecodeIter; ++it) {
        sc[it][h] = __builtin_amdgcn_exp2f(sc[it][h] - ref);  // 0 outside the chunk
        run_l[h] += sc[it][h];
      }
    }
    auto of_head = [&](const float (&v)[kStates], int h) {
      if constexpr (kMfma) return row_broadcast(v[0], h);
      else return v[h];
    };
#pragma unroll
    for (int h = 0; h < R; ++h) {
      const float scale = of_head(keep, h);
#pragma unroll
      for (int e = 0; e < E; ++e) acc[h][e] *= scale;
    }
#pragma unroll
    for (int it = 0; it < kDecodeIter; ++it) {
      uint4 raw = rows.v[it];
      const uint32_t keep_bits = valid[it] ? 0xFFFFFFFFu : 0u;  // a masked column: no Inf * 0
      raw.x &= keep_bits; raw.y &= keep_bits; raw.z &= keep_bits; raw.w &= keep_bits;
      float vf[E];
      RowChunk<ST>::unpack(raw, vf);
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const float p = of_head(sc[it], h);
#pragma unroll
        for (int e = 0; e < E; ++e) acc[h][e] = fmaf(p, vf[e], acc[h][e]);
      }
    }
  };
  // One head, a short past walked by this workgroup alone: the rows of the first two or three
  // chunks are requested together (a chunk costs 0.95 us when each waits for its own round
  // trip; 3 x 32 registers of rows fit beside one head's state).  Each case holds its loads and
  // their uses in one branch: a branch between a load and its use makes the compiler wait
  // inside it.  Two chunks where three would pass 256 registers, i.e. one workgroup a CU for
  // launches of many splits: the variant that scores on the matrix cores, and ragged batches whose
  // f32 queries meet fp16 rows (178 registers, 263 with three; 24 sequences up to 3000 columns of 16
  // heads, D = 64, two layers: 77.6 us, 110.6 with three).
  constexpr bool kThreeChunks = !kMfma && !(RAGGED && sizeof(XT) > sizeof(ST));
  if (!early) load_chunk(0, rows0);  // harmless when the split has no column at all
  // The own column's scores, as soon as every row is asked for: the operand's registers go.
  float own_dot = 0.f;
  if constexpr (kMfma) {
    __builtin_amdgcn_sched_barrier(0);
    float4_t dots = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t)
      dots = __builtin_amdgcn_mfma_f32_16x16x32_f16(own_k[t], qb[t], dots, 0, 0, 0);
    own_dot = dots[0] * ((a.scale * a.scale) * kLog2e);
  }
  bool walked = false;
  if constexpr (R == 1) {
    if (nsplit == 1 && total_chunks == 2) {
      ChunkRows rows1;
      load_chunk(1, rows1);
      consume_chunk(0, rows0);
      consume_chunk(1, rows1);
      walked = true;
    } else if (nsplit == 1 && total_chunks > 2) {
      ChunkRows rows1;
      load_chunk(1, rows1);
      if constexpr (kThreeChunks) {
        ChunkRows rows2;
        load_chunk(2, rows2);
        consume_chunk(0, rows0);
        consume_chunk(1, rows1);
        consume_chunk(2, rows2);
      } else {
        consume_chunk(0, rows0);
        consume_chunk(1, rows1);
      }
      for (uint32_t chunk = kThreeChunks ? 3 : 2; chunk < total_chunks; ++chunk) {
        load_chunk(chunk, rows0);
        consume_chunk(chunk, rows0);
      }
      walked = true;
    }
  }
  if (!walked && my_chunks > 0) {
    if (kSplitChunks == 2 && nsplit > 1 && my_chunks == 2) {
      // a split of a long past: both chunks requested before the first is scored
      ChunkRows rows1;
      load_chunk(1, rows1);
      consume_chunk(0, rows0);
      consume_chunk(1, rows1);
    } else {
      consume_chunk(0, rows0);
      for (uint32_t chunk = 1; chunk < my_chunks; ++chunk) {
        load_chunk(chunk, rows0);
        consume_chunk(chunk, rows0);
      }
    }
  }
  // this step's own column: one more row for group 0 of the last split (for every other lane
  // the update below is the identity, so the other splits skip it)
  if (last) {
    float s_own[kStates], vo[E];
    if constexpr (kMfma) {
      s_own[0] = wave == 0 ? own_dot : -INFINITY;
      RowChunk<ST>::unpack(own_v, vo);
    } else {
#pragma unroll
      for (int h = 0; h < R; ++h) {
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) part = fmaf(qf[h][e], kx[e], part);
        part = group_sum<LPR>(part);
        s_own[h] = own ? part : -INFINITY;
      }
#pragma unroll
      for (int e = 0; e < E; ++e) vo[e] = vx[e];
    }
    float keep[kStates], p_own[kStates];
#pragma unroll
    for (int h = 0; h < kStates; ++h) {
      const float m_new = fmaxf(run_m[h], s_own[h]);
      const float ref = m_new == -INFINITY ? 0.f : m_new;
      keep[h] = __builtin_amdgcn_exp2f(run_m[h] - ref);
      p_own[h] = own ? __builtin_amdgcn_exp2f(s_own[h] - ref) : 0.f;
      run_m[h] = m_new;
      run_l[h] = run_l[h] * keep[h] + p_own[h];
    }
#pragma unroll
    for (int h = 0; h < R; ++h) {
      float k = keep[kMfma ? 0 : h], p = p_own[kMfma ? 0 : h];
      if constexpr (kMfma) {
        k = row_broadcast(k, h);
        p = row_broadcast(p, h);
      }
#pragma unroll
      for (int e = 0; e < E; ++e)
        acc[h][e] = fmaf(p, own ? vo[e] : 0.f, acc[h][e] * k);  // 0 * NaN must not leak
    }
  }

  // The states are merged in ascending order.  A wave that keeps one maximum for its groups sums
  // them in registers first, a quarter of the outputs left to each lane (sixteen group states
  // through LDS cost 32 KB and every output sixteen exponentials).
  if constexpr (kMfma) {
    constexpr int kHeld = R * E / 4;  // consecutive dims of one head
    float flat[R * E];
#pragma unroll
    for (int i = 0; i < R * E; ++i) flat[i] = acc[i / E][i % E];
    const int first = sum_rows(flat, lane);
    float* mine = &s_acc[wave][(first / E) * D + sub * E + first % E];
#pragma unroll
    for (int i = 0; i < kHeld; i += 2)
      *reinterpret_cast<float2*>(mine + i) = make_float2(flat[i], flat[i + 1]);
    sum_rows(run_l, lane);
    if (lane < R) {
      s_m[wave][lane] = run_m[0];
      s_l[wave][lane] = run_l[0];
    }
  } else {
#pragma unroll
    for (int h = 0; h < R; ++h) {
#pragma unroll
      for (int e = 0; e < E; ++e) s_acc[group][h * D + sub * E + e] = acc[h][e];
      if (sub == 0) {
        s_m[group][h] = run_m[h];
        s_l[group][h] = run_l[h];
      }
    }
  }
  __syncthreads();
  const uint32_t gsplit = first_split + split;
  float part_o[kOuts], part_l[kOuts], part_m[kOuts];
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = tid + i * kThreads;
    part_o[i] = part_l[i] = 0.f;
    part_m[i] = -INFINITY;
    if (o >= R * D) continue;
    const int h = o / D, d = o - h * D;
    float m = s_m[0][h];
#pragma unroll
    for (int w = 1; w < kParts; ++w) m = fmaxf(m, s_m[w][h]);  // finite: the split holds a column
    float total = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kParts; ++w) {
      const float wgt = __builtin_amdgcn_exp2f(s_m[w][h] - m);
      total = fmaf(wgt, s_acc[w][o], total);
      l = fmaf(wgt, s_l[w][h], l);
    }
    part_o[i] = total;
    part_l[i] = l;
    part_m[i] = m;
    if (nsplit == 1) {
      st_f32<XT>(out, ((size_t)seq * a.heads + head0 + h) * D + d, total / l);
    } else {
      const size_t slot_index = (size_t)gsplit * a.heads + head0 + h;
      publish(&ws_acc[slot_index * D + d], total);
      if (d == 0) {
        publish(&ws_ml[slot_index * 2], m);
        publish(&ws_ml[slot_index * 2 + 1], l);
      }
    }
  }
  if (nsplit == 1) return;

  // Arrival: the partial was written through to memory (device-scope stores); once every
  // thread's stores have completed, take a ticket.  The last arrival merges, reading the
  // partials with device-scope loads.  No cache-wide write-back or invalidate is involved.
  // The wait is spelled out: a workgroup-scope release fence does not wait for global stores
  // on this target, and a device-scope one writes the whole L2 back.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* ticket = &a.tickets[(size_t)(seq * a.units + unit) * kTicketStride];
  if (tid == 0)
    s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (s_ticket + 1 != nsplit) return;

  // Merge nsplit partials of each of the R heads, kMergeChunk at a time, ascending order; the
  // partial rows of a pass are all requested before any is used.
  // Every output element tracks the running (max, sum) of its own head: the same numbers in
  // all elements of a head, and one exponential per partial instead of one per use.
  float tot_m[kOuts], tot_l[kOuts], tot_o[kOuts];
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    tot_m[i] = -INFINITY;
    tot_l[i] = 0.f;
    tot_o[i] = 0.f;
  }
  for (uint32_t s0 = 0; s0 < nsplit; s0 += kMergeChunk) {
    const uint32_t cnt = nsplit - s0 < (uint32_t)kMergeChunk ? nsplit - s0 : (uint32_t)kMergeChunk;
    // the weighted rows first (long latency), the small (max, sum) pairs next
    float rows[kOuts][kMergeChunk];
    auto request = [&](int j0, int j1) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kOuts; ++i) {
        const int o = tid + i * kThreads;
        const int oo = o < R * D ? o : 0;
        const int h = oo / D, d = oo - h * D;
        const float* src = ws_acc + ((size_t)(first_split + s0) * a.heads + head0 + h) * D + d;
        const size_t stride = (size_t)a.heads * D;
#pragma unroll
        for (int j = j0; j < j1; ++j)
          rows[i][j] = observe(&src[(size_t)((uint32_t)j < cnt ? j : 0) * stride]);
      }
    };
    // A nearly full pass is one block of loads; of a shorter one only the blocks of eight that hold a split.  us with 32
    // rows always / so: 5 splits of 8 x 256 dims 6.2 / 5.8, ragged 22 sequences up to 1478 columns 43.7 / 42.5; blocks
    // alone took 8.7 for 32 splits that take 8.5.
    const bool full = cnt > (uint32_t)(kMergeChunk - kMergeBlock);
    if (full) {
      request(0, kMergeChunk);
    } else {
#pragma unroll
      for (int j0 = 0; j0 < kMergeChunk - kMergeBlock; j0 += kMergeBlock) {
        if ((uint32_t)j0 >= cnt) break;
        request(j0, j0 + kMergeBlock);
      }
    }
    __syncthreads();
    for (uint32_t i = tid; i < R * kMergeChunk; i += kThreads) {
      const uint32_t h = i / kMergeChunk, s = i - h * kMergeChunk;
      const size_t slot_index = (size_t)(first_split + s0 + (s < cnt ? s : 0)) * a.heads + head0 + h;
      s_w[h][s] = s < cnt ? observe(&ws_ml[slot_index * 2]) : -INFINITY;
      s_wl[h][s] = s < cnt ? observe(&ws_ml[slot_index * 2 + 1]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOuts; ++i) {
      const int o = tid + i * kThreads;
      const int h = (o < R * D ? o : 0) / D;
      float m = tot_m[i];
#pragma unroll
      for (int j = 0; j < kMergeChunk; ++j) m = fmaxf(m, s_w[h][j]);
      const float keep = __builtin_amdgcn_exp2f(tot_m[i] - m);  // 0 on the first pass
      float l = tot_l[i] * keep, total = tot_o[i] * keep;
      auto add = [&](int j0, int j1) __attribute__((always_inline)) {
#pragma unroll
        for (int j = j0; j < j1; ++j) {
          const float wgt = __builtin_amdgcn_exp2f(s_w[h][j] - m);
          l = fmaf(wgt, s_wl[h][j], l);
          total = fmaf(wgt, rows[i][j], total);
        }
      };
      if (full) {
        add(0, kMergeChunk);
      } else {
#pragma unroll
        for (int j0 = 0; j0 < kMergeChunk - kMergeBlock; j0 += kMergeBlock) {
          if ((uint32_t)j0 >= cnt) break;
          add(j0, j0 + kMergeBlock);
        }
      }
      tot_m[i] = m;
      tot_l[i] = l;
      tot_o[i] = total;
    }
  }
#pragma unroll
  for (int i = 0; i < kOuts; ++i) {
    const int o = tid + i * kThreads;
    if (o >= R * D) break;
    const int h = o / D, d = o - h * D;
    st_f32<XT>(out, ((size_t)seq * a.heads + head0 + h) * D + d, tot_o[i] / tot_l[i]);
  }
  if (tid == 0)  // ready for the next launch
    __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct DecodeLaunch {
  krm_buf q, ins_k, ins_v, slot_k, slot_v, out;
  float* ws_ml;
  float* ws_acc;
  DecodeArgs args;
  uint32_t grid_x, grid_z;     // splits (or total splits), batch
  uint32_t ticket_slots = kTicketSlots;  // counters behind args.tickets
  bool clear_tickets = false;  // zero the counters this launch uses before it runs
};

// Fill kernel for arrival counters (a kernel, not a memset, so that a caller may record it).
__global__ void clear_tickets_kernel(uint32_t* tickets, uint32_t count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) tickets[(size_t)i * kTicketStride] = 0u;
}

template <typename XT, typename ST, int R, int LPR, bool RAGGED>
int32_t launch_decode(krm_ctx* ctx, const DecodeLaunch& L) {
  attention_decode_kernel<XT, ST, R, LPR, RAGGED>
      <<<L.args.folded ? dim3(8 * L.args.units, (L.grid_x + 7) / 8, L.grid_z) : dim3(L.grid_x, L.args.units, L.grid_z),
         dim3(kThreads), 0, ctx->stream>>>(
          ptr<const XT>(L.q), ptr<const XT>(L.ins_k), ptr<const XT>(L.ins_v),
          ptr<const ST>(L.slot_k), ptr<const ST>(L.slot_v), ptr<XT>(L.out), L.ws_ml, L.ws_acc,
          L.args);
  return launched(ctx, "attention_decode_kernel");
}

// `per_block` = query heads one workgroup carries (a divisor of H / Hkv).  A head's result
// does not depend on it: every head keeps its own running state and its own merge.
template <typename XT, typename ST, int LPR, bool RAGGED>
int32_t decode_by_repeat(krm_ctx* ctx, const DecodeLaunch& L, uint32_t per_block) {
  switch (per_block) {
    case 1: return launch_decode<XT, ST, 1, LPR, RAGGED>(ctx, L);
    case 2: return launch_decode<XT, ST, 2, LPR, RAGGED>(ctx, L);
    case 4: return launch_decode<XT, ST, 4, LPR, RAGGED>(ctx, L);
    default: return fail(ctx, KRM_ERR_VALIDATION, "decode attention: %u heads per block", per_block);
  }
}

template <typename XT, typename ST, bool RAGGED>
int32_t decode_by_depth(krm_ctx* ctx, const DecodeLaunch& L, uint32_t per_block, uint32_t lpr) {
  switch (lpr) {
    case 4: return decode_by_repeat<XT, ST, 4, RAGGED>(ctx, L, per_block);
    case 8: return decode_by_repeat<XT, ST, 8, RAGGED>(ctx, L, per_block);
    case 16: return decode_by_repeat<XT, ST, 16, RAGGED>(ctx, L, per_block);
    case 32: return decode_by_repeat<XT, ST, 32, RAGGED>(ctx, L, per_block);
    case 64: return decode_by_repeat<XT, ST, 64, RAGGED>(ctx, L, per_block);
    default: return fail(ctx, KRM_ERR_VALIDATION, "decode attention: %u lanes per row", lpr);
  }
}

// Few (split, kv head) pairs leave most of the chip idle while each workgroup walks its
// columns once per query head; the query heads of a kv head are then spread over several
// workgroups (each re-reads the K/V rows, which the L2 serves) until the grid covers the CUs.
// Four heads at most: the state of eight takes a SIMD's registers to one wave or two, and sixteen
// sequences of eight heads of D = 256 then took 198 us where two groups of four take 133
// (D = 64: 134 and 105).
template <bool RAGGED>
int32_t decode_dispatch(krm_ctx* ctx, DecodeLaunch& L, uint32_t repeat, uint32_t lpr,
                        int32_t io_dtype, int32_t kv_dtype) {
  uint32_t per_block = repeat;
  uint64_t blocks = (uint64_t)L.grid_x * L.grid_z * L.args.kv_heads;
  while (per_block > 4 || (per_block > 1 && blocks < 2ull * (uint64_t)ctx->num_cus)) {
    per_block >>= 1;
    blocks <<= 1;
  }

  L.args.repeat = repeat;
  L.args.head_groups = repeat / per_block;
  L.args.splits = L.grid_x;
  L.args.units = L.args.kv_heads * L.args.head_groups;
  // (one split: the head groups lie on neighbouring XCDs, and seven of eight workgroups of the other grid had no work)
  // (eight kv heads share the XCDs evenly whatever the splits)
  const bool even = L.args.kv_heads % 8 == 0;
  const uint32_t rest = L.grid_x % 8, behind_head = even ? 1u : rest, behind_batch = even ? 0u : L.args.kv_heads * rest % 8;
  L.args.folded = L.grid_x > 1 && L.args.head_groups > 1 && (L.grid_x + 7) / 8 <= 65535
                      ? 1u | behind_head << 4 | behind_batch << 8
                      : 0u;
  const uint64_t counters = (uint64_t)L.args.nseq * L.args.kv_heads * L.args.head_groups;
  if ((uint64_t)L.args.kv_heads * L.args.head_groups > 65535 || counters > L.ticket_slots)
    return fail(ctx, KRM_ERR_VALIDATION, "decode attention: B * H = %llu exceeds %u",
                (unsigned long long)counters, L.ticket_slots);
  if (L.clear_tickets) {
    clear_tickets_kernel<<<dim3(((uint32_t)counters + 255) / 256), dim3(256), 0, ctx->stream>>>(
        L.args.tickets, (uint32_t)counters);
    KRM_TRY(launched(ctx, "clear_tickets_kernel"));
  }
  if (io_dtype == KRM_F16 && kv_dtype == KRM_F16)
    return decode_by_depth<__half, __half, RAGGED>(ctx, L, per_block, lpr);
  if (io_dtype == KRM_F32 && kv_dtype == KRM_F32)
    return decode_by_depth<float, float, RAGGED>(ctx, L, per_block, lpr);
  if (io_dtype == KRM_F32 && kv_dtype == KRM_F16)
    return decode_by_depth<float, __half, RAGGED>(ctx, L, per_block, lpr);
  return decode_by_depth<__half, float, RAGGED>(ctx, L, per_block, lpr);
}

// lanes a K/V row of `depth` elements spans with 16-byte pieces; 0 = not covered
uint32_t decode_lanes_per_row(uint32_t depth, int32_t kv_dtype) {
  const uint32_t row_bytes = depth * (uint32_t)dtype_bytes(kv_dtype);
  if (row_bytes % 16) return 0;
  const uint32_t lpr = row_bytes / 16;
  return (lpr == 4 || lpr == 8 || lpr == 16 || lpr == 32 || lpr == 64) ? lpr : 0;
}

bool decode_repeat_ok(uint32_t repeat) {
  return repeat == 1 || repeat == 2 || repeat == 4 || repeat == 8;
}

template <typename XT, typename ST>
int32_t launch_generic(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v, krm_buf slot_k,
                       krm_buf slot_v, krm_buf out, uint32_t batch, const GenericArgs& a) {
  attention_generic_kernel<XT, ST>
      <<<dim3(batch * a.heads, a.chunk_rows), dim3(kThreads), 0, ctx->stream>>>(
          ptr<const XT>(q), ptr<const XT>(ins_k), ptr<const XT>(ins_v), ptr<const ST>(slot_k),
          ptr<const ST>(slot_v), ptr<XT>(out), a);
  return launched(ctx, "attention_generic_kernel");
}

template <typename XT, typename ST>
int32_t launch_rows(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v, krm_buf slot_k,
                    krm_buf slot_v, krm_buf out, uint32_t batch, const GenericArgs& a,
                    uint32_t flags) {
  // Eight waves, two a SIMD, so that one wave's softmax and LDS traffic run under the other's
  // MFMAs; D = 256: four (the state of a wave takes a SIMD's registers).  A workgroup takes one
  // block of 16 query rows; with D = 64, whose second block fits the registers, two (the K / V
  // blocks then serve both) once that still leaves two workgroups per CU.  (D = 128 in two blocks
  // had to park V as well: 512 rows behind 2048, r = 4, in f32 303 us, 233 in single blocks; 585
  // and 261 in f32 over fp16 slots.)  A row's arithmetic is
  // the same in both forms and the wave count depends on D only, so its bits depend neither on the
  // chunk length, the batch, the past or the capacity nor on the lengths form.
  const uint32_t row_blocks = (a.chunk_rows + 15) / 16;
  // (with a window the key blocks start at the first row's lower bound, which a second row
  // block would not share: one block a workgroup there)
  const bool two = a.window == 0 && a.depth == 64 &&
                   (uint64_t)batch * a.heads * ((row_blocks + 1) / 2) >= 2ull * ctx->num_cus;
  const dim3 grid(batch * a.heads, two ? (row_blocks + 1) / 2 : row_blocks);
#define KRM_ROWS_ATTENTION(DEPTH, WAVES, RB)                                                   \
  attention_rows_kernel<XT, ST, DEPTH, WAVES, RB><<<grid, dim3(64 * WAVES), 0, ctx->stream>>>( \
      ptr<const XT>(q), ptr<const XT>(ins_k), ptr<const XT>(ins_v), ptr<ST>(slot_k),           \
      ptr<ST>(slot_v), ptr<XT>(out), a, flags)
  if (a.depth == 256) {
    KRM_ROWS_ATTENTION(256, 4, 1);
  } else if (a.depth == 64) {
    if (two) KRM_ROWS_ATTENTION(64, 8, 2); else KRM_ROWS_ATTENTION(64, 8, 1);
  } else {
    KRM_ROWS_ATTENTION(128, 8, 1);
  }
#undef KRM_ROWS_ATTENTION
  return launched(ctx, "attention_rows_kernel");
}

// smallest split any dtype uses for this head dim (f32 rows span the most lanes)
uint32_t min_split_columns(uint32_t depth) {
  uint32_t lpr = decode_lanes_per_row(depth, KRM_F32);
  if (!lpr) lpr = decode_lanes_per_row(depth, KRM_F16);
  return lpr ? decode_split_columns(lpr) : 0;
}

}  // namespace

extern "C" {

int32_t krm_attention_state_workspace(uint32_t batch, uint32_t heads, uint32_t kv_heads,
                                      uint32_t chunk_rows, uint32_t depth, uint32_t window,
                                      uint32_t max_past, uint32_t max_query, size_t* bytes) {
  (void)kv_heads;
  (void)chunk_rows;
  (void)max_query;
  if (!bytes) return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_state_workspace: NULL");
  const uint32_t sc = min_split_columns(depth);
  uint64_t columns = max_past;
  if (window && columns > window - 1) columns = window - 1;
  const uint64_t nsplit = sc ? decode_splits(columns, sc) : 1;
  *bytes = (size_t)batch * heads * nsplit * ((size_t)depth + 2) * sizeof(float) + 256;
  return KRM_OK;
}

// `lengths` == 0: past / query are this run's values.  Otherwise they are read on the device
// and `past` is the largest pastLength the launch has to be sized for.
// `tickets` == nullptr: the context's arrival counters.  Otherwise counters supplied by the
// caller (`ticket_slots` of them, kTicketStride words apart), which this call clears first.
static int32_t attention_state_impl(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                                    krm_buf slot_k, krm_buf slot_v, krm_buf out, uint32_t batch,
                                    uint32_t heads, uint32_t kv_heads, uint32_t chunk_rows,
                                    uint32_t depth, uint32_t capacity, uint32_t window,
                                    float half_scale, uint32_t past, uint32_t query,
                                    krm_buf lengths, int32_t io_dtype, int32_t kv_dtype,
                                    krm_buf workspace, size_t workspace_bytes,
                                    uint32_t* tickets = nullptr, uint32_t ticket_slots = 0,
                                    uint32_t chunk_flags = 0, bool chunk_only = false) {
  KRM_TRY(enter(ctx));
  const bool dyn = lengths != 0;
  KRM_REQUIRE(ctx, aligned(lengths, 4), "krm_attention_state: misaligned lengths buffer");
  KRM_REQUIRE(ctx, valid_dtype(io_dtype) && valid_dtype(kv_dtype),
              "krm_attention_state: io_dtype %d / kv_dtype %d", io_dtype, kv_dtype);
  KRM_REQUIRE(ctx,
              batch >= 1 && heads >= 1 && kv_heads >= 1 && chunk_rows >= 1 && depth >= 1 &&
                  capacity >= 1,
              "krm_attention_state: B / H / Hkv / M / D / C must be positive "
              "(%u / %u / %u / %u / %u / %u)",
              batch, heads, kv_heads, chunk_rows, depth, capacity);
  KRM_REQUIRE(ctx, heads % kv_heads == 0, "krm_attention_state: H = %u is not a multiple of Hkv = %u",
              heads, kv_heads);
  KRM_REQUIRE(ctx, window <= capacity, "krm_attention_state: window %u exceeds capacity %u",
              window, capacity);
  KRM_REQUIRE(ctx, std::isfinite(half_scale), "krm_attention_state: scale is not finite");
  KRM_REQUIRE(ctx, depth <= 1024, "krm_attention_state: D = %u exceeds 1024", depth);
  KRM_REQUIRE(ctx, (uint64_t)batch * heads <= 0x7fffffffull && chunk_rows <= 65535,
              "krm_attention_state: B*H = %llu or M = %u exceeds the launch grid",
              (unsigned long long)batch * heads, chunk_rows);
  if (!dyn && (query < 1 || query > chunk_rows))
    return fail(ctx, KRM_ERR_EXECUTION, "krm_attention_state: queryLength %u is outside 1..%u",
                query, chunk_rows);
  if (!dyn && (uint64_t)past + query > 0xffffffffull)
    return fail(ctx, KRM_ERR_EXECUTION,
                "krm_attention_state: pastLength %u + queryLength %u does not fit in 32 bits",
                past, query);
  if (!dyn && window == 0 && (uint64_t)past + query > capacity)
    return fail(ctx, KRM_ERR_EXECUTION,
                "krm_attention_state: pastLength %u + queryLength %u exceeds capacity %u", past,
                query, capacity);
  KRM_REQUIRE(ctx, q && ins_k && ins_v && slot_k && slot_v && out,
              "krm_attention_state: NULL buffer");
  const size_t io_b = dtype_bytes(io_dtype), kv_b = dtype_bytes(kv_dtype);
  KRM_REQUIRE(ctx,
              aligned(q, io_b) && aligned(ins_k, io_b) && aligned(ins_v, io_b) &&
                  aligned(out, io_b) && aligned(slot_k, kv_b) && aligned(slot_v, kv_b),
              "krm_attention_state: misaligned buffer");

  const uint32_t repeat = heads / kv_heads;
  const uint32_t lpr = decode_lanes_per_row(depth, kv_dtype);
  const bool fast = !chunk_only && (dyn || query == 1) && chunk_rows == 1 && lpr &&
                    decode_repeat_ok(repeat) &&
                    aligned(slot_k, 16) && aligned(slot_v, 16) && aligned(q, 16) && batch <= 65535 &&
                    heads <= 65535 &&
                    (uint64_t)batch * heads <= (tickets ? ticket_slots : kTicketSlots);
  if (fast) {
    const uint64_t low = window_low(window, past);
    const uint32_t nsplit = decode_splits((uint64_t)past - low, decode_split_columns(lpr));
    DecodeLaunch L{};
    L.q = q; L.ins_k = ins_k; L.ins_v = ins_v; L.slot_k = slot_k; L.slot_v = slot_v; L.out = out;
    L.args.heads = heads;
    L.args.kv_heads = kv_heads;
    L.args.window = window;
    L.args.past = past;
    L.args.slot_batch_stride = (uint64_t)kv_heads * capacity * depth;
    L.args.slot_plane_stride = (uint64_t)capacity * depth;
    L.args.scale = half_scale;
    L.args.nseq = batch;
    L.grid_x = nsplit;
    L.grid_z = batch;
    L.args.tickets = tickets ? tickets : ctx->tickets;
    L.ticket_slots = tickets ? ticket_slots : kTicketSlots;
    L.clear_tickets = tickets != nullptr;
    L.args.lengths = ptr<uint32_t>(lengths);
    L.args.capacity = capacity;
    if (nsplit > 1) {
      // split partials + arrival counters: the context's counters assume launch order
      if (!tickets) KRM_TRY(needs_serial_scratch(ctx, "the split decode attention"));
      const size_t ml_floats = (size_t)batch * nsplit * heads * 2;
      const size_t need = (ml_floats + (size_t)batch * nsplit * heads * depth) * sizeof(float);
      if (tickets && workspace_bytes < need + 16)
        return fail(ctx, KRM_ERR_VALIDATION,
                    "krm_attention_state_noalloc: this call needs %zu bytes of split partials, the "
                    "built-in scratch holds %zu (use krm_attention_state with a workspace)",
                    need + 16, workspace_bytes);
      KRM_REQUIRE(ctx, workspace && aligned(workspace, 16) && workspace_bytes >= need,
                  "krm_attention_state: workspace of %zu bytes, %zu needed", workspace_bytes,
                  need);
      L.ws_ml = ptr<float>(workspace);
      L.ws_acc = L.ws_ml + ((ml_floats + 3) & ~(size_t)3);
      KRM_REQUIRE(ctx, workspace_bytes >= (size_t)((char*)(L.ws_acc + (size_t)batch * nsplit *
                                                           heads * depth) - (char*)L.ws_ml),
                  "krm_attention_state: workspace of %zu bytes is too small", workspace_bytes);
    }
    return decode_dispatch<false>(ctx, L, repeat, lpr, io_dtype, kv_dtype);
  }

  GenericArgs a{heads, kv_heads, chunk_rows, depth, capacity, window, past, query, half_scale,
                ptr<uint32_t>(lengths)};
  // chunks of rows with the usual head dims: the MFMA form
  if ((chunk_rows > 1 || chunk_only) && (depth == 64 || depth == 128 || depth == 256) &&
      aligned(q, 16) &&
      aligned(ins_k, 16) && aligned(ins_v, 16) && aligned(slot_k, 16) && aligned(slot_v, 16) &&
      (uint64_t)batch * heads <= 0x7fffffffull && (chunk_rows + 31) / 32 <= 65535) {
    const uint32_t f = chunk_flags;
    if (io_dtype == KRM_F32 && kv_dtype == KRM_F32)
      return launch_rows<float, float>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a, f);
    if (io_dtype == KRM_F16 && kv_dtype == KRM_F16)
      return launch_rows<__half, __half>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a, f);
    if (io_dtype == KRM_F32 && kv_dtype == KRM_F16)
      return launch_rows<float, __half>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a, f);
    return launch_rows<__half, float>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a, f);
  }
  if (chunk_only)
    return fail(ctx, KRM_ERR_VALIDATION,
                "krm_attention_chunk: covers D = 64, 128 or 256 and 16-byte aligned buffers (D = %u); "
                "use krm_attention_state, krm_state_append and krm_transpose_01", depth);
  if (io_dtype == KRM_F32 && kv_dtype == KRM_F32)
    return launch_generic<float, float>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a);
  if (io_dtype == KRM_F16 && kv_dtype == KRM_F16)
    return launch_generic<__half, __half>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a);
  if (io_dtype == KRM_F32 && kv_dtype == KRM_F16)
    return launch_generic<float, __half>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a);
  return launch_generic<__half, float>(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, a);
}

int32_t krm_attention_state(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                            krm_buf slot_k, krm_buf slot_v, krm_buf out, uint32_t batch,
                            uint32_t heads, uint32_t kv_heads, uint32_t chunk_rows,
                            uint32_t depth, uint32_t capacity, uint32_t window,
                            float half_scale, uint32_t past, uint32_t query, int32_t io_dtype,
                            int32_t kv_dtype, krm_buf workspace, size_t workspace_bytes) {
  return attention_state_impl(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, heads, kv_heads,
                              chunk_rows, depth, capacity, window, half_scale, past, query, 0,
                              io_dtype, kv_dtype, workspace, workspace_bytes);
}

int32_t krm_attention_state_lengths(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                                    krm_buf slot_k, krm_buf slot_v, krm_buf out, uint32_t batch,
                                    uint32_t heads, uint32_t kv_heads, uint32_t chunk_rows,
                                    uint32_t depth, uint32_t capacity, uint32_t window,
                                    float half_scale, krm_buf lengths, uint32_t max_past,
                                    int32_t io_dtype, int32_t kv_dtype, krm_buf workspace,
                                    size_t workspace_bytes) {
  if (!lengths) return fail(ctx, KRM_ERR_VALIDATION, "krm_attention_state_lengths: NULL lengths");
  return attention_state_impl(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, heads, kv_heads,
                              chunk_rows, depth, capacity, window, half_scale, max_past,
                              chunk_rows, lengths, io_dtype, kv_dtype, workspace, workspace_bytes);
}

int32_t krm_attention_chunk(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v, krm_buf slot_k,
                            krm_buf slot_v, krm_buf out, uint32_t batch, uint32_t heads,
                            uint32_t kv_heads, uint32_t chunk_rows, uint32_t depth,
                            uint32_t capacity, uint32_t window, float half_scale, uint32_t past,
                            uint32_t query, krm_buf lengths, int32_t io_dtype, int32_t kv_dtype,
                            uint32_t flags) {
  KRM_REQUIRE(ctx, (flags & ~(uint32_t)(KRM_CHUNK_OUT_ROW_MAJOR | KRM_CHUNK_APPEND |
                                        KRM_CHUNK_OUT_F16)) == 0,
              "krm_attention_chunk: unknown flags 0x%x", flags);
  KRM_REQUIRE(ctx, !(flags & KRM_CHUNK_APPEND) || window == 0,
              "krm_attention_chunk: the fused append needs window == 0 (a ring overwrites rows "
              "this launch still reads); call krm_state_append after the attention");
  return attention_state_impl(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, heads, kv_heads,
                              chunk_rows, depth, capacity, window, half_scale,
                              lengths ? capacity - 1 : past, lengths ? chunk_rows : query, lengths,
                              io_dtype, kv_dtype, 0, 0, nullptr, 0, flags, true);
}

int32_t krm_attention_varlen_workspace(uint32_t nseq, uint32_t heads, uint32_t kv_heads,
                                       uint32_t depth, uint64_t total_rows, size_t* bytes) {
  (void)kv_heads;
  if (!bytes) return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_varlen_workspace: NULL");
  const uint32_t sc = min_split_columns(depth);
  // every sequence rounds its split count up, so at most total/sc + nseq splits
  const uint64_t splits = sc ? total_rows / sc + nseq : nseq;
  *bytes = 2 * ((size_t)nseq + 1) * sizeof(int32_t) + 64 +
           (size_t)splits * heads * ((size_t)depth + 2) * sizeof(float) + 256;
  return KRM_OK;
}

int32_t krm_attention_varlen(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                             krm_buf slot_k, krm_buf slot_v, krm_buf out,
                             const int32_t* cu_seqlens, uint32_t nseq, uint32_t heads,
                             uint32_t kv_heads, uint32_t depth, uint64_t total_rows,
                             float half_scale, int32_t io_dtype, int32_t kv_dtype,
                             krm_buf workspace, size_t workspace_bytes) {
  KRM_TRY(enter(ctx));
  KRM_REQUIRE(ctx, valid_dtype(io_dtype) && valid_dtype(kv_dtype),
              "krm_attention_varlen: io_dtype %d / kv_dtype %d", io_dtype, kv_dtype);
  KRM_REQUIRE(ctx, nseq >= 1 && heads >= 1 && kv_heads >= 1 && depth >= 1,
              "krm_attention_varlen: nseq / H / Hkv / D must be positive");
  KRM_REQUIRE(ctx, heads % kv_heads == 0, "krm_attention_varlen: H = %u is not a multiple of Hkv = %u",
              heads, kv_heads);
  KRM_REQUIRE(ctx, std::isfinite(half_scale), "krm_attention_varlen: scale is not finite");
  KRM_REQUIRE(ctx, cu_seqlens != nullptr, "krm_attention_varlen: cu_seqlens is NULL");
  KRM_REQUIRE(ctx, total_rows <= 0x7fffffffull, "krm_attention_varlen: total_rows too large");
  KRM_REQUIRE(ctx, heads <= 65535 && (uint64_t)nseq * heads <= kTicketSlots,
              "krm_attention_varlen: nseq * H = %llu exceeds %u", (unsigned long long)nseq * heads,
              kTicketSlots);
  const uint32_t repeat = heads / kv_heads;
  const uint32_t lpr = decode_lanes_per_row(depth, kv_dtype);
  KRM_REQUIRE(ctx, lpr && decode_repeat_ok(repeat),
              "krm_attention_varlen: D = %u with this slot dtype or H/Hkv = %u is not covered "
              "by the split-K decode kernel",
              depth, repeat);
  KRM_REQUIRE(ctx, q && ins_k && ins_v && slot_k && slot_v && out && workspace,
              "krm_attention_varlen: NULL buffer");
  KRM_REQUIRE(ctx, aligned(slot_k, 16) && aligned(slot_v, 16) && aligned(workspace, 16) &&
                       aligned(q, 16),
              "krm_attention_varlen: q, slots and workspace must be 16-byte aligned");
  KRM_REQUIRE(ctx, cu_seqlens[0] >= 0, "krm_attention_varlen: cu_seqlens[0] is negative");

  // Host-side tables: slot row offsets and the first global split of each sequence.
  const size_t table_ints = 2 * ((size_t)nseq + 1);
  KRM_REQUIRE(ctx, table_ints * sizeof(int32_t) <= ctx->pinned_bytes,
              "krm_attention_varlen: %u sequences exceed the staging table", nseq);
  KRM_TRY(not_recording(ctx, "krm_attention_varlen"));
  // The staging area may still feed the previous call's copy.
  KRM_TRY(hip_status(ctx, hipStreamSynchronize(ctx->stream), "hipStreamSynchronize"));
  int32_t* stage = static_cast<int32_t*>(ctx->pinned);
  int32_t* cu = stage;
  int32_t* prefix = stage + nseq + 1;
  const uint32_t sc = decode_split_columns(lpr);
  uint64_t splits = 0;
  for (uint32_t i = 0; i <= nseq; ++i) {
    cu[i] = cu_seqlens[i];
    if (i > 0) {
      KRM_REQUIRE(ctx, cu_seqlens[i] >= cu_seqlens[i - 1],
                  "krm_attention_varlen: cu_seqlens is not ascending at %u", i);
      prefix[i - 1] = (int32_t)splits;
      const uint32_t ns = decode_splits((uint64_t)(cu_seqlens[i] - cu_seqlens[i - 1]), sc);
      splits += ns;
    }
  }
  prefix[nseq] = (int32_t)splits;
  KRM_REQUIRE(ctx, (uint64_t)cu_seqlens[nseq] <= total_rows,
              "krm_attention_varlen: cu_seqlens[%u] = %d exceeds total_rows %llu", nseq,
              cu_seqlens[nseq], (unsigned long long)total_rows);
  KRM_REQUIRE(ctx, splits <= 0x7fffffffull, "krm_attention_varlen: too many splits");

  const size_t table_bytes = (table_ints * sizeof(int32_t) + 63) & ~(size_t)63;
  const size_t ml_floats = ((size_t)splits * heads * 2 + 3) & ~(size_t)3;
  const size_t need = table_bytes + (ml_floats + (size_t)splits * heads * depth) * sizeof(float);
  KRM_REQUIRE(ctx, workspace_bytes >= need, "krm_attention_varlen: workspace of %zu bytes, %zu needed",
              workspace_bytes, need);
  KRM_TRY(hip_status(ctx,
                     hipMemcpyAsync(ptr<void>(workspace), stage, table_ints * sizeof(int32_t),
                                    hipMemcpyHostToDevice, ctx->stream),
                     "hipMemcpyAsync(tables)"));

  DecodeLaunch L{};
  L.q = q; L.ins_k = ins_k; L.ins_v = ins_v; L.slot_k = slot_k; L.slot_v = slot_v; L.out = out;
  L.args.heads = heads;
  L.args.kv_heads = kv_heads;
  L.args.window = 0;
  L.args.past = 0;
  L.args.slot_batch_stride = 0;
  L.args.slot_plane_stride = total_rows * depth;
  L.args.scale = half_scale;
  L.args.nseq = nseq;
  L.args.cu_rows = ptr<const int32_t>(workspace);
  L.args.split_prefix = L.args.cu_rows + nseq + 1;
  L.ws_ml = ptr<float>(workspace + table_bytes);
  L.ws_acc = L.ws_ml + ml_floats;
  L.grid_x = (uint32_t)splits;
  L.grid_z = 1;
  KRM_TRY(needs_serial_scratch(ctx, "krm_attention_varlen"));
  L.args.tickets = ctx->tickets;
  return decode_dispatch<true>(ctx, L, repeat, lpr, io_dtype, kv_dtype);
}

}  // extern "C"

// ---- ragged batch whose tables are built on the device -------------------------------------

// plan layout (int32): cu_rows[nseq + 1], split_prefix[nseq + 1], fault
//
// One wave, a sequence a lane: 64 offsets are read together and their splits summed over the lanes.  A single
// lane's loop over the sequences is a chain of memory latencies: 16 sequences took
// 3.4 us, now 1.8; 64 10.2, now 2.2; 1000 142, now 9.5 (an empty launch of a replay is 1.8).
__global__ __launch_bounds__(kWave) void varlen_plan_kernel(const int32_t* __restrict__ cu_seqlens,
                                                            int32_t* __restrict__ plan, uint32_t nseq,
                                                            uint32_t chunk_columns, uint64_t total_rows,
                                                            uint32_t max_splits) {
  int32_t* cu = plan;
  int32_t* prefix = plan + nseq + 1;
  const uint32_t lane = threadIdx.x;
  bool ok = true;
  uint64_t before = 0;  // splits of the sequences before this step's
  for (uint64_t base = 0; base <= nseq; base += kWave) {
    const uint64_t i = base + lane;
    const int32_t lo = cu_seqlens[min(i, (uint64_t)nseq)], hi = cu_seqlens[min(i + 1, (uint64_t)nseq)];
    // A step's splits fit 32 bits: those of ascending offsets are at most 2^31 / 32 + 64, other ones count as none.
    const bool ascending = lo >= 0 && hi >= lo;
    ok = ok && ascending;
    const uint32_t own = i < nseq && ascending ? decode_splits((uint64_t)(hi - lo), chunk_columns) : 0u;
    // Sums through each lane: within rows of 16 lanes, then of the row before into odd rows, of the lower half into
    // the upper one (operands of the vector ALU; six shuffles through LDS were 0.3 us of a plan and the attention
    // behind it).
    uint32_t through = own;
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x111, 0xf, 0xf, false);  // row_shr:1
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x112, 0xf, 0xf, false);
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x114, 0xf, 0xf, false);
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x118, 0xf, 0xf, false);
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x142, 0xa, 0xf, false);  // row_bcast:15
    through += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)through, 0x143, 0xc, 0xf, false);  // row_bcast:31
    if (i <= nseq) {
      cu[i] = lo;
      prefix[i] = (int32_t)(before + through - own);
      if (i == nseq) ok = ok && (uint64_t)lo <= total_rows;
    }
    before += (uint32_t)__builtin_amdgcn_readlane((int)through, kWave - 1);
  }
  ok = __all(ok) && before <= max_splits;
  if (!ok)  // no workgroup of the attention launch finds a split: nothing is read or written
    for (uint64_t i = lane; i <= nseq; i += kWave) prefix[i] = 0;
  if (lane == 0) plan[2 * (nseq + 1)] = ok ? 0 : 1;
}

extern "C" {

int32_t krm_attention_varlen_plan_bytes(uint32_t nseq, size_t* bytes) {
  if (!bytes) return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_varlen_plan_bytes: NULL");
  *bytes = ((2 * ((size_t)nseq + 1) + 1) * sizeof(int32_t) + 63) & ~(size_t)63;
  return KRM_OK;
}

int32_t krm_attention_varlen_max_splits(uint32_t nseq, uint32_t depth, int32_t kv_dtype,
                                        uint64_t total_rows, uint32_t* max_splits) {
  if (!max_splits) return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_varlen_max_splits: NULL");
  if (!valid_dtype(kv_dtype))
    return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_varlen_max_splits: kv_dtype %d", kv_dtype);
  const uint32_t lpr = decode_lanes_per_row(depth, kv_dtype);
  if (!lpr)
    return fail(nullptr, KRM_ERR_VALIDATION,
                "krm_attention_varlen_max_splits: D = %u is not covered by the decode kernel", depth);
  // every sequence rounds its split count up
  const uint64_t splits = total_rows / decode_split_columns(lpr) + nseq;
  if (splits > 0x7fffffffull)
    return fail(nullptr, KRM_ERR_VALIDATION, "krm_attention_varlen_max_splits: too many splits");
  *max_splits = (uint32_t)splits;
  return KRM_OK;
}

int32_t krm_attention_varlen_plan(krm_ctx* ctx, krm_buf cu_seqlens_i32, krm_buf plan,
                                  uint32_t nseq, uint32_t depth, int32_t kv_dtype,
                                  uint64_t total_rows, uint32_t max_splits) {
  KRM_TRY(enter(ctx));
  KRM_REQUIRE(ctx, valid_dtype(kv_dtype), "krm_attention_varlen_plan: kv_dtype %d", kv_dtype);
  KRM_REQUIRE(ctx, nseq >= 1 && total_rows <= 0x7fffffffull,
              "krm_attention_varlen_plan: nseq must be positive and total_rows < 2^31");
  const uint32_t lpr = decode_lanes_per_row(depth, kv_dtype);
  KRM_REQUIRE(ctx, lpr, "krm_attention_varlen_plan: D = %u with this slot dtype is not covered",
              depth);
  KRM_REQUIRE(ctx, cu_seqlens_i32 && plan && aligned(cu_seqlens_i32, 4) && aligned(plan, 4),
              "krm_attention_varlen_plan: NULL or misaligned buffer");
  varlen_plan_kernel<<<dim3(1), dim3(kWave), 0, ctx->stream>>>(
      ptr<const int32_t>(cu_seqlens_i32), ptr<int32_t>(plan), nseq, decode_split_columns(lpr),
      total_rows, max_splits);
  return launched(ctx, "varlen_plan_kernel");
}

int32_t krm_attention_varlen_planned(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                                     krm_buf slot_k, krm_buf slot_v, krm_buf out, krm_buf plan,
                                     uint32_t nseq, uint32_t heads, uint32_t kv_heads,
                                     uint32_t depth, uint64_t total_rows, uint32_t max_splits,
                                     float half_scale, int32_t io_dtype, int32_t kv_dtype,
                                     krm_buf workspace, size_t workspace_bytes) {
  KRM_TRY(enter(ctx));
  KRM_REQUIRE(ctx, valid_dtype(io_dtype) && valid_dtype(kv_dtype),
              "krm_attention_varlen_planned: io_dtype %d / kv_dtype %d", io_dtype, kv_dtype);
  KRM_REQUIRE(ctx, nseq >= 1 && heads >= 1 && kv_heads >= 1 && depth >= 1 && max_splits >= 1,
              "krm_attention_varlen_planned: nseq / H / Hkv / D / max_splits must be positive");
  KRM_REQUIRE(ctx, heads % kv_heads == 0,
              "krm_attention_varlen_planned: H = %u is not a multiple of Hkv = %u", heads, kv_heads);
  KRM_REQUIRE(ctx, std::isfinite(half_scale), "krm_attention_varlen_planned: scale is not finite");
  KRM_REQUIRE(ctx, total_rows <= 0x7fffffffull && max_splits <= 0x7fffffffu,
              "krm_attention_varlen_planned: total_rows or max_splits too large");
  KRM_REQUIRE(ctx, heads <= 65535 && (uint64_t)nseq * heads <= kTicketSlots,
              "krm_attention_varlen_planned: nseq * H = %llu exceeds %u",
              (unsigned long long)nseq * heads, kTicketSlots);
  const uint32_t repeat = heads / kv_heads;
  const uint32_t lpr = decode_lanes_per_row(depth, kv_dtype);
  KRM_REQUIRE(ctx, lpr && decode_repeat_ok(repeat),
              "krm_attention_varlen_planned: D = %u with this slot dtype or H/Hkv = %u is not "
              "covered by the split-K decode kernel", depth, repeat);
  KRM_REQUIRE(ctx, q && ins_k && ins_v && slot_k && slot_v && out && workspace && plan,
              "krm_attention_varlen_planned: NULL buffer");
  KRM_REQUIRE(ctx, aligned(slot_k, 16) && aligned(slot_v, 16) && aligned(workspace, 16) &&
                       aligned(q, 16) && aligned(plan, 4),
              "krm_attention_varlen_planned: q, slots and workspace must be 16-byte aligned");
  const size_t ml_floats = ((size_t)max_splits * heads * 2 + 3) & ~(size_t)3;
  const size_t need = (ml_floats + (size_t)max_splits * heads * depth) * sizeof(float);
  KRM_REQUIRE(ctx, workspace_bytes >= need,
              "krm_attention_varlen_planned: workspace of %zu bytes, %zu needed", workspace_bytes,
              need);
  DecodeLaunch L{};
  L.q = q; L.ins_k = ins_k; L.ins_v = ins_v; L.slot_k = slot_k; L.slot_v = slot_v; L.out = out;
  L.args.heads = heads;
  L.args.kv_heads = kv_heads;
  L.args.window = 0;
  L.args.past = 0;
  L.args.slot_batch_stride = 0;
  L.args.slot_plane_stride = total_rows * depth;
  L.args.scale = half_scale;
  L.args.nseq = nseq;
  L.args.cu_rows = ptr<const int32_t>(plan);
  L.args.split_prefix = L.args.cu_rows + nseq + 1;
  L.ws_ml = ptr<float>(workspace);
  L.ws_acc = L.ws_ml + ml_floats;
  L.grid_x = max_splits;
  L.grid_z = 1;
  KRM_TRY(needs_serial_scratch(ctx, "krm_attention_varlen_planned"));
  L.args.tickets = ctx->tickets;
  return decode_dispatch<true>(ctx, L, repeat, lpr, io_dtype, kv_dtype);
}

}  // extern "C"
// ---- the decode attention for callers that cannot allocate ----------------------------------
//
// Split partials and arrival counters live in one file-scope device array instead of a
// caller-supplied workspace and the context's counters.  Each GPU holds its own copy of the
// array at its own address; the address is looked up once per device and that pointer — never
// the array's name, which in host code is only a stand-in — is what kernels and fills receive.
namespace {

constexpr size_t kStaticTicketSlots = 512;
constexpr size_t kStaticTicketBytes = kStaticTicketSlots * kTicketStride * sizeof(uint32_t);
constexpr size_t kStaticScratchBytes = 4u << 20;  // counters + split partials, per GPU
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Device address of this device's copy of `scratch` (the context's device is current).
int32_t static_scratch(krm_ctx* ctx, unsigned char** out) {
  KRM_REQUIRE(ctx, ctx->device >= 0 && ctx->device < kMaxDevices,
              "krm_attention_state_noalloc: device %d is outside 0..%d", ctx->device,
              kMaxDevices - 1);
  unsigned char* p = __atomic_load_n(&g_scratch_ptr[ctx->device], __ATOMIC_ACQUIRE);
  if (!p) {
    void* address = nullptr;
    KRM_TRY(hip_status(ctx, hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)),
                       "hipGetSymbolAddress(scratch)"));
    KRM_REQUIRE(ctx, address != nullptr, "krm_attention_state_noalloc: scratch has no address");
    p = static_cast<unsigned char*>(address);
    __atomic_store_n(&g_scratch_ptr[ctx->device], p, __ATOMIC_RELEASE);
  }
  *out = p;
  return KRM_OK;
}

}  // namespace

namespace krm {
// Called when a context is created on a device, so that the address is known before any caller
// starts recording a graph (the lookup is a runtime call that does not belong in a capture).
int32_t resolve_static_scratch(krm_ctx* ctx) {
  unsigned char* unused = nullptr;
  return static_scratch(ctx, &unused);
}
}  // namespace krm

extern "C" {

int32_t krm_attention_state_noalloc(krm_ctx* ctx, krm_buf q, krm_buf ins_k, krm_buf ins_v,
                                    krm_buf slot_k, krm_buf slot_v, krm_buf out, uint32_t batch,
                                    uint32_t heads, uint32_t kv_heads, uint32_t chunk_rows,
                                    uint32_t depth, uint32_t capacity, uint32_t window,
                                    float half_scale, uint32_t past, uint32_t query,
                                    int32_t io_dtype, int32_t kv_dtype) {
  KRM_TRY(enter(ctx));
  unsigned char* base = nullptr;
  KRM_TRY(static_scratch(ctx, &base));
  // Only the split decode form needs scratch; it checks its partials against `room` and words
  // the error for this entry.  Chunks of rows and head dims the decode form does not cover run
  // without any, and a call with more heads than the array has counters takes the generic
  // kernel.
  const size_t room = kStaticScratchBytes - kStaticTicketBytes;
  return attention_state_impl(ctx, q, ins_k, ins_v, slot_k, slot_v, out, batch, heads, kv_heads,
                              chunk_rows, depth, capacity, window, half_scale, past, query, 0,
                              io_dtype, kv_dtype,
                              static_cast<krm_buf>(reinterpret_cast<uintptr_t>(
                                  base + kStaticTicketBytes)),
                              room, reinterpret_cast<uint32_t*>(base),
                              (uint32_t)kStaticTicketSlots);
}

}  // extern "C"
