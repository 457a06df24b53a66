// int4 `linear` for M > 16 rows (prefill) on the gfx950 matrix cores.
//
// out[m, n] = sum_k x[m,k] * dequant(w)[n,k] + bias[n], same operands and layouts as the GEMV
// (packages/runtime/src/kernels/linear.ts:34-64, packages/runtime/src/kernels/gemm.ts:1187-1237).
// The reference computes this op in f32 and rejects f16 compute with int4 weights
// (packages/runtime/src/kernels/gemm.ts:1204-1209), so this kernel has no same-numerics
// counterpart there: activations are rounded to fp16 (exact when they already are fp16), each
// weight is dequantised to fp16 as fp16(u - 8) * fp16(scale) — one fp16 rounding of a value
// the reference holds exactly — and products are accumulated in f32 by
// v_mfma_f32_32x32x16_f16.  The caller opts in with KRM_COMPUTE_F16.
//
// Workgroup tile BM x BN (waves in a WM x WN grid, 64 x 64 outputs per wave = 2 x 2 MFMA
// tiles, optionally KS wave groups that split each chunk's K and add their sums at the end);
// K is walked KC (64 or 128) codes at a time through LDS:
//   A tile  x[BM rows][KC]  fp16, each group of 8 stored as (x0,x4,x1,x5,x2,x6,x3,x7)
//   B tile  w[BN rows][KC]  fp16 dequantised, the same order within each group of 8 — the
//           order the nibble trick produces (code i pairs with code i+4), so no shuffle is
//           spent on the weights; the k index inside an MFMA is a free permutation as long as
//           both operands use the same one.
// Rows are padded by 16 bytes so the 16-byte fragment reads of 32 consecutive rows spread over
// all LDS banks.  Chunks travel memory -> registers (several in flight, no use of a loaded
// value before it is parked, so the waits are counted) -> LDS -> fragments.  Pipelined form:
// two LDS copies (distinct objects, so fragment reads may pass the parking writes), the
// dequantisation of chunk c + 1 interleaved with the MFMAs of chunk c, one barrier a chunk.
#include "gemm_i4_deal.h"
#include "i4_codes.h"

using namespace krm;

namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));

// A K chunk of KC codes is staged per pass; rows are padded by 16 bytes so the 16-byte
// fragment reads of 32 consecutive rows spread over all LDS banks.
template <int KC>
struct ChunkGeometry {
  static constexpr int kRowBytes = KC * 2 + 16;
};

// A scale as it arrives from memory, kept in a whole 32-bit register until the chunk is parked
// (narrowing it on arrival would be an ALU op that has to wait for the load).
template <typename ST>
__device__ inline uint32_t scale_bits(const ST* s, size_t i);
template <>
__device__ inline uint32_t scale_bits<__half>(const __half* s, size_t i) {
  return reinterpret_cast<const uint16_t*>(s)[i];
}
template <>
__device__ inline uint32_t scale_bits<float>(const float* s, size_t i) {
  return reinterpret_cast<const uint32_t*>(s)[i];
}
template <typename ST>
__device__ inline float load_scale_f32(const ST* s, size_t i);
template <>
__device__ inline float load_scale_f32<__half>(const __half* s, size_t i) {
  return __half2float(s[i]);
}
template <>
__device__ inline float load_scale_f32<float>(const float* s, size_t i) { return s[i]; }
template <typename ST>
__device__ inline _Float16 scale_from_bits(uint32_t bits);
template <>
__device__ inline _Float16 scale_from_bits<__half>(uint32_t bits) {
  return __builtin_bit_cast(_Float16, (uint16_t)bits);
}
template <>
__device__ inline _Float16 scale_from_bits<float>(uint32_t bits) {
  return (_Float16)__uint_as_float(bits);
}

// 8 codes of a word -> 8 fp16 values (u - 8) * scale, order (c0,c4,c1,c5,c2,c6,c3,c7).
__device__ inline uint4 dequant_word(uint32_t word, _Float16 scale) {
  const uint32_t magic = 0x64006400u;  // (1024, 1024)
  const half2_t off_lo = {(_Float16)1032.0f, (_Float16)1032.0f};
  const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const half2_t off_hi = {(_Float16)-72.0f, (_Float16)-72.0f};
  const half2_t s2 = {scale, scale};
  const uint32_t upper = word >> 8;
  const half2_t q0 = (__builtin_bit_cast(half2_t, and_or(word, 0x000F000Fu, magic)) - off_lo) * s2;
  const half2_t q1 = (__builtin_elementwise_fma(
                         __builtin_bit_cast(half2_t, and_or(word, 0x00F000F0u, magic)), sixteenth,
                         off_hi)) * s2;
  const half2_t q2 = (__builtin_bit_cast(half2_t, and_or(upper, 0x000F000Fu, magic)) - off_lo) * s2;
  const half2_t q3 = (__builtin_elementwise_fma(
                         __builtin_bit_cast(half2_t, and_or(upper, 0x00F000F0u, magic)), sixteenth,
                         off_hi)) * s2;
  return make_uint4(__builtin_bit_cast(uint32_t, q0), __builtin_bit_cast(uint32_t, q1),
                    __builtin_bit_cast(uint32_t, q2), __builtin_bit_cast(uint32_t, q3));
}

// 8 consecutive activations as they arrive from memory; converted to fp16 in the order
// (x0,x4,x1,x5,x2,x6,x3,x7) only when they are parked in LDS, so the loads stay in flight.
template <typename XT>
struct Acts8;
template <>
struct Acts8<__half> {
  uint4 raw;
  __device__ inline void load(const __half* p) { raw = *reinterpret_cast<const uint4*>(p); }
  __device__ inline void keep(uint32_t bits) {
    raw.x &= bits; raw.y &= bits; raw.z &= bits; raw.w &= bits;
  }
  __device__ inline uint4 paired() const {
    return make_uint4(__builtin_amdgcn_perm(raw.z, raw.x, 0x05040100u),
                      __builtin_amdgcn_perm(raw.z, raw.x, 0x07060302u),
                      __builtin_amdgcn_perm(raw.w, raw.y, 0x05040100u),
                      __builtin_amdgcn_perm(raw.w, raw.y, 0x07060302u));
  }
};
template <>
struct Acts8<float> {
  uint4 a, b;  // raw bits of x0..x3, x4..x7
  __device__ inline void load(const float* p) {
    a = reinterpret_cast<const uint4*>(p)[0];
    b = reinterpret_cast<const uint4*>(p)[1];
  }
  __device__ inline void keep(uint32_t bits) {
    a.x &= bits; a.y &= bits; a.z &= bits; a.w &= bits;
    b.x &= bits; b.y &= bits; b.z &= bits; b.w &= bits;
  }
  __device__ inline uint4 paired() const {
    auto pack = [](uint32_t lo, uint32_t hi) {
      const half2_t h = {(_Float16)__uint_as_float(lo), (_Float16)__uint_as_float(hi)};  // RNE
      return __builtin_bit_cast(uint32_t, h);
    };
    return make_uint4(pack(a.x, b.x), pack(a.y, b.y), pack(a.z, b.z), pack(a.w, b.w));
  }
};

template <typename T>
__device__ inline float bias_f32(const T* p, size_t i);
template <>
__device__ inline float bias_f32<float>(const float* p, size_t i) { return p[i]; }
template <>
__device__ inline float bias_f32<__half>(const __half* p, size_t i) { return __half2float(p[i]); }
template <typename T>
__device__ inline void store_out(T* p, size_t i, float v);
template <>
__device__ inline void store_out<float>(float* p, size_t i, float v) { p[i] = v; }
template <>
__device__ inline void store_out<__half>(__half* p, size_t i, float v) {
  p[i] = __float2half_rn(v);
}

template <typename XT, typename ST, int WM, int WN, int KC, int KS, int DEPTH, bool PIPE, bool FAST>
__global__ __launch_bounds__(WM * WN * KS * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_i4_f16_kernel(const XT* __restrict__ x, const uint32_t* __restrict__ w,
                        const ST* __restrict__ scales, const XT* __restrict__ bias,
                        XT* __restrict__ out, uint32_t m, uint32_t n, uint32_t k,
                        uint32_t group_shift, uint32_t m_blocks, uint32_t n_blocks,
                        uint32_t wide_rows) {
  // KS wave groups share the tile and split every chunk's K between them (their sums are
  // added once at the end): more waves per output, so more work in flight per CU.
  constexpr int kThreads = WM * WN * KS * 64;
  constexpr int BM = WM * 64, BN = WN * 64;
  constexpr int kRowBytes = ChunkGeometry<KC>::kRowBytes;
  constexpr int kStepsPerGroup = KC / 16 / KS;
  static_assert(KC % (16 * KS) == 0, "the K split divides the chunk");
  constexpr int kRowPieces = KC / 8;                 // 16-byte pieces (or weight words) a row
  constexpr int kAPieces = BM * kRowPieces;          // 16-byte pieces of the A tile
  constexpr int kAPer = kAPieces / kThreads;         // per thread
  constexpr int kBPieces = BN * kRowPieces;          // words of the B tile
  constexpr int kBPer = kBPieces / kThreads;         // words per thread (consecutive in a row)
  static_assert(kAPieces % kThreads == 0 && kBPieces % kThreads == 0, "tile / thread mismatch");
  static_assert(kBPer == 1 || kBPer == 2 || kBPer == 4 || kBPer == 8 || kBPer == 16,
                "B words per thread");
  static_assert(kRowPieces % kBPer == 0, "a thread's weight words stay inside one row");

  // One LDS copy of the chunk; the NEXT chunk waits in registers (its loads are issued right
  // after this chunk is parked), and several workgroups share a CU, so a workgroup that sits
  // at a barrier or waits for memory leaves the matrix cores to the others.
  // PIPE: two LDS copies; while the matrix cores work on chunk c out of one copy, the same
  // wave parks chunk c + 1 in the other (the two instruction streams interleave), one barrier
  // per chunk.
  constexpr int kStageBytes = (BM + BN) * kRowBytes;
  constexpr int kStageValuPerMfma = (kAPer * 4 + kBPer * 13 + kStepsPerGroup * 4 - 1) / (kStepsPerGroup * 4);
  constexpr int kReduceBytes = KS > 1 ? WM * WN * (KS - 1) * 64 * 64 * 4 : 0;
  // two separate objects, so the compiler knows that parking into one copy cannot touch the
  // other and may move the fragment reads past those writes
  __shared__ __attribute__((aligned(16)))
  unsigned char lds[kStageBytes > kReduceBytes ? kStageBytes : kReduceBytes];
  __shared__ __attribute__((aligned(16))) unsigned char lds_other[PIPE ? kStageBytes : 16];
  constexpr int kOffB = BM * kRowBytes;

  // Workgroup ids are dealt round-robin over the 8 XCDs, each with its own L2.  The row panels
  // of one column block get consecutive slots of ONE XCD, so its weights cross the fabric once
  // and the other panels find them in that L2 (x, the smaller operand, is re-read instead).
  uint32_t mb, nb;
  {
    const uint32_t id = blockIdx.x;
    if (8 % m_blocks == 0) {
      const uint32_t xcd = id & 7, slot = id >> 3;
      mb = slot % m_blocks;
      nb = (slot / m_blocks) * 8 + xcd;
    } else {
      mb = id % m_blocks;
      nb = id / m_blocks;
    }
    if (nb >= n_blocks) return;
  }
  const uint32_t m0 = mb * BM, n0 = nb * BN;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = (wave / WM) % WN, kg = wave / (WM * WN);

  const uint32_t words_per_row = k >> 3;
  const uint32_t groups_per_row = k >> group_shift;
  const uint32_t chunks = (k + KC - 1) / KC;

  // staging assignment: element offsets of the thread's pieces at chunk 0 (rows past M or N
  // re-read the last row; their products are never stored)
  uint32_t a_off[kAPer], a_lds[kAPer], a_k[kAPer];
#pragma unroll
  for (int i = 0; i < kAPer; ++i) {
    const int p = tid + i * kThreads;
    const uint32_t row = p / kRowPieces, pc = p % kRowPieces;
    a_off[i] = min(row, m - 1 - m0) * k + pc * 8;  // relative to the tile's first row
    a_k[i] = pc * 8;
    a_lds[i] = row * kRowBytes + pc * 16;
  }
  const uint32_t b_row = (tid * kBPer) / kRowPieces;
  const uint32_t b_w0 = (tid * kBPer) % kRowPieces;
  const uint32_t b_grow = min(n0 + b_row, n - 1);
  const uint32_t* b_src = w + (size_t)b_grow * words_per_row + b_w0;
  const size_t b_scale_row = (size_t)b_grow * groups_per_row;

  const XT* x_tile = x + (size_t)m0 * k;
  // A chunk's operands as they arrive from memory.  DEPTH of them are in flight: chunk c + DEPTH
  // is requested as soon as chunk c has been parked in LDS.
  struct Slot {
    Acts8<XT> a[kAPer];
    uint32_t b[kBPer];
    uint32_t scale[kBPer];  // raw bits, see scale_bits
  };
  // a thread's words are consecutive and aligned to their count, so they share one scale
  // whenever a group covers them all
  const bool one_scale = ((uint32_t)(kBPer * 8 - 1) >> group_shift) == 0;

  // FAST (16-byte aligned rows, one scale per thread, K a multiple of KC): a fetch is the same
  // straight run of loads for every chunk, so waits on an older chunk can be counted and the
  // younger requests stay in flight.  Any branch here would cost that.
  auto fetch = [&](uint32_t chunk, Slot& slot) {
    const uint32_t k0 = chunk * KC;
    if constexpr (FAST) {
#pragma unroll
      for (int i = 0; i < kAPer; ++i) slot.a[i].load(x_tile + a_off[i] + k0);
#pragma unroll
      for (int j = 0; j + 3 < kBPer; j += 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(b_src + (k0 >> 3) + j);
        slot.b[j] = v.x; slot.b[j + 1] = v.y; slot.b[j + 2] = v.z; slot.b[j + 3] = v.w;
      }
      slot.scale[0] = scale_bits<ST>(scales, b_scale_row + ((k0 + b_w0 * 8) >> group_shift));
    } else if (k0 + KC <= k) {  // uniform: the whole chunk lies inside K
#pragma unroll
      for (int i = 0; i < kAPer; ++i) slot.a[i].load(x_tile + a_off[i] + k0);
      if (kBPer >= 4 && wide_rows) {
#pragma unroll
        for (int j = 0; j + 3 < kBPer; j += 4) {
          const uint4 v = *reinterpret_cast<const uint4*>(b_src + (k0 >> 3) + j);
          slot.b[j] = v.x; slot.b[j + 1] = v.y; slot.b[j + 2] = v.z; slot.b[j + 3] = v.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < kBPer; ++j) slot.b[j] = b_src[(k0 >> 3) + j];
      }
      if (one_scale) {  // only scale[0] is loaded (no copies: a copy would wait for the load)
        slot.scale[0] = scale_bits<ST>(scales, b_scale_row + ((k0 + b_w0 * 8) >> group_shift));
      } else {
#pragma unroll
        for (int j = 0; j < kBPer; ++j)
          slot.scale[j] =
              scale_bits<ST>(scales, b_scale_row + ((k0 + (b_w0 + j) * 8) >> group_shift));
      }
    } else {  // last chunk of a K that is not a multiple of KC: zero activations past K
#pragma unroll
      for (int i = 0; i < kAPer; ++i) {
        const bool inside = k0 + a_k[i] < k;
        slot.a[i].load(x_tile + a_off[i] + (inside ? k0 : 0u));
        slot.a[i].keep(inside ? 0xFFFFFFFFu : 0u);
      }
#pragma unroll
      for (int j = 0; j < kBPer; ++j) {
        const uint32_t kk = k0 + (b_w0 + j) * 8;
        const uint32_t kc = kk < k ? kk : 0u;  // x is zero there; any finite weight will do
        slot.b[j] = w[(size_t)b_grow * words_per_row + (kc >> 3)];
        slot.scale[j] = scale_bits<ST>(scales, b_scale_row + (kc >> group_shift));
      }
    }
  };
  float16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int frag_row = lane & 31, frag_g = lane >> 5;
  const int a_frag = (wm * 64 + frag_row) * kRowBytes + frag_g * 16 + kg * kStepsPerGroup * 32;
  const int b_frag =
      kOffB + (wn * 64 + frag_row) * kRowBytes + frag_g * 16 + kg * kStepsPerGroup * 32;

  // `ragged`: the chunk reaches past K and carries one scale per word
  auto stage = [&](const Slot& slot, bool ragged, int buf) {
#pragma unroll
    for (int i = 0; i < kAPer; ++i)
      *reinterpret_cast<uint4*>(&(buf ? lds_other : lds)[a_lds[i]]) = slot.a[i].paired();
#pragma unroll
    for (int j = 0; j < kBPer; ++j)
      *reinterpret_cast<uint4*>(&(buf ? lds_other : lds)[kOffB + b_row * kRowBytes + (b_w0 + j) * 16]) =
          dequant_word(slot.b[j], scale_from_bits<ST>(
                                      slot.scale[(FAST || (one_scale && !ragged)) ? 0 : j]));
  };
  // All fragments of the chunk are requested before the first matrix instruction, so only the
  // first one waits for LDS.
  auto compute = [&](int buf) {
    half8_t af[kStepsPerGroup][2], bf[kStepsPerGroup][2];
#pragma unroll
    for (int ks = 0; ks < kStepsPerGroup; ++ks) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[ks][i] = *reinterpret_cast<const half8_t*>(
            &(buf ? lds_other : lds)[a_frag + i * 32 * kRowBytes + ks * 32]);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        bf[ks][j] = *reinterpret_cast<const half8_t*>(
            &(buf ? lds_other : lds)[b_frag + j * 32 * kRowBytes + ks * 32]);
    }
#pragma unroll
    for (int ks = 0; ks < kStepsPerGroup; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] =
              __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks][i], bf[ks][j], acc[i][j], 0, 0, 0);
  };
  if constexpr (PIPE) {
    // chunk c travels slot[c % DEPTH] -> LDS copy c % 2 (DEPTH is even); DEPTH - 1 chunks are
    // in flight behind the one being parked
    static_assert(DEPTH % 2 == 0, "the LDS copy of a slot is fixed");
    Slot slots[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if constexpr (FAST) {
        fetch(min((uint32_t)d, chunks - 1), slots[d]);
      } else {
        if ((uint32_t)d < chunks) fetch(d, slots[d]);
      }
    }
    stage(slots[0], KC > k, 0);
    if constexpr (FAST) {
      fetch(min((uint32_t)DEPTH, chunks - 1), slots[0]);
    } else {
      if ((uint32_t)DEPTH < chunks) fetch(DEPTH, slots[0]);
    }
    __syncthreads();
    // steady state: every body parks its successor; straight-line code so the staging and the
    // matrix instructions can be interleaved
    auto body = [&](uint32_t chunk, int d) {
      const int nd = (d + 1) % DEPTH;
      stage(slots[nd], (chunk + 1) * KC + KC > k, nd % 2);
      compute(d % 2);
      // one matrix instruction, then a share of the staging work, in turn
      constexpr int kMfmas = kStepsPerGroup * 4;
      constexpr int kLead = kMfmas >= 8 ? 8 : kMfmas;  // fragment reads ahead of the first MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, kLead, 0);
#pragma unroll
      for (int i = 0; i < kMfmas; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, kStageValuPerMfma, 0);
        if (i < kMfmas - kLead) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (i % 2) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
      if constexpr (FAST) {
        fetch(min(chunk + 1 + DEPTH, chunks - 1), slots[nd]);  // past the end: a harmless re-read
      } else {
        if (chunk + 1 + DEPTH < chunks) fetch(chunk + 1 + DEPTH, slots[nd]);
      }
      __syncthreads();
    };
    uint32_t chunk = 0;
    for (; chunk + DEPTH < chunks; chunk += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) body(chunk + d, d);
    }
    // the last 1..DEPTH chunks: the final one has no successor to park
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (chunk + d + 1 < chunks) {
        body(chunk + d, d);
      } else if (chunk + d < chunks) {
        compute(d % 2);
      }
    }
    __syncthreads();
  } else {
    Slot slots[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if constexpr (FAST) {
        fetch(min((uint32_t)d, chunks - 1), slots[d]);
      } else {
        if ((uint32_t)d < chunks) fetch(d, slots[d]);
      }
    }
    for (uint32_t base = 0; base < chunks; base += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {  // unrolled: every slot has fixed registers
        const uint32_t chunk = base + d;
        if (chunk >= chunks) break;
        stage(slots[d], chunk * KC + KC > k, 0);
        __syncthreads();
        if constexpr (FAST) {
          fetch(min(chunk + DEPTH, chunks - 1), slots[d]);  // past the end: a harmless re-read
        } else {
          if (chunk + DEPTH < chunks) fetch(chunk + DEPTH, slots[d]);
        }
        compute(0);
        __syncthreads();  // every wave is done with this chunk before the next one is parked
      }
    }
  }

  if constexpr (KS > 1) {
    // Sum of the K groups, group 0 + 1 + ... in that order; the tile's LDS is free again (the
    // loop ended on a barrier).  Word (r, lane) of a wave's 64 x 64 block: conflict-free.
    float* red = reinterpret_cast<float*>(lds);
    if (kg > 0) {
      float* dst = red + (size_t)(((kg - 1) * WN + wn) * WM + wm) * 64 * 64;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) dst[((i * 2 + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g) {
      const float* src = red + (size_t)(((g - 1) * WN + wn) * WM + wm) * 64 * 64;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += src[((i * 2 + j) * 16 + r) * 64 + lane];
    }
  }

  // epilogue: lane holds column (lane % 32); register r holds row 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t col = n0 + wn * 64 + j * 32 + frag_row;
    if (col >= n) continue;
    const float add = bias ? bias_f32<XT>(bias, col) : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm * 64 + i * 32 + 8 * (r / 4) + 4 * frag_g + (r % 4);
        if (row < m) store_out<XT>(out, (size_t)row * n + col, acc[i][j][r] + add);
      }
    }
  }
}

// ---------------------------------------------------------------- packed weights in LDS
//
// Eight waves, workgroup tile (64 * MT) x 256, wave (wm, wn) = 32 * MT rows x 64 columns, K in
// stages of 128 codes.  The weight bytes are staged as they are — coalesced 16-byte loads, a
// quarter of the LDS bytes the dequantised fp16 tile takes — and every wave dequantises the
// words of its own 64 columns after reading them back: lane (n = lane % 32, h = lane / 32)
// reads 16 bytes = codes 64c + 32h .. + 31 of column n per 64-code chunk, word j of which is
// the B operand of the chunk's MFMA step j (fp16(u - 8) * fp16(scale), order
// c0,c4,c1,c5,c2,c6,c3,c7); the A operand of that step is x[m][64c + 32h + 8j ..] in the
// same order, 16 bytes of the staged x row.  The same arithmetic as the kernel above, so the
// two agree up to the order of the f32 additions.  Two waves share a SIMD: one wave's
// dequantisation runs under the other's MFMAs.  Every stage issues the same loads whatever K
// is (clamped addresses; x past K is parked as zeros).
template <typename XT, typename ST, int MT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_i4_f16_packed_kernel(const XT* __restrict__ x, const uint8_t* __restrict__ w,
                               const ST* __restrict__ scales, const XT* __restrict__ bias,
                               XT* __restrict__ out, uint32_t m, uint32_t n, uint32_t k,
                               uint32_t group_shift, uint32_t m_blocks, uint32_t n_blocks) {
  constexpr int WN = 2;
  constexpr int BM = 2 * 32 * MT, BN = 256;
  constexpr int kStage = 128;                 // codes per LDS stage
  constexpr int kRowA = kStage * 2 + 16;      // bytes per LDS row of fp16 x
  constexpr int kRowB = kStage / 2 + 16;      // bytes per LDS row of packed weights
  constexpr int kAUnits = BM * (kStage / 8) / 512;  // 8-element units of x per thread and stage
  __shared__ __align__(16) uint8_t s_a[2][BM * kRowA];
  __shared__ __align__(16) uint8_t s_b[2][BN * kRowB];
  __shared__ _Float16 s_s[2][BN][2];

  const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
  const uint32_t mb = slot % m_blocks, nb = (slot / m_blocks) * 8u + xcd;
  if (nb >= n_blocks) return;  // the whole workgroup leaves before any barrier
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int frag_row = lane & 31, frag_h = lane >> 5;
  const uint32_t m0 = mb * BM, n0 = nb * BN;
  const uint32_t groups = k >> group_shift;
  const uint32_t stages = (k + kStage - 1) / kStage;

  // staging roles: x rows in 16 units of 8 elements (rows tid / 16 + 32 i), weight rows in 4
  // units of 16 bytes (rows tid / 4 + 128 i), one scale row per thread of the first four waves
  const uint32_t arow0 = tid >> 4, aunit = (tid & 15u) * 8u;      // element offset in the stage
  const uint32_t brow0 = tid >> 2, bunit = (tid & 3u) * 16u;      // byte offset in the stage
  const ST* ssrc = scales + (size_t)min(n0 + (uint32_t)(tid & 255), n - 1) * groups;

  struct Staged {
    Acts8<XT> a[kAUnits];
    uint4 b[2];
  };
  auto load_stage = [&](uint32_t stage, Staged& d) {
    const uint32_t a_at = stage * kStage + aunit, b_at = stage * (kStage / 2) + bunit;
    const uint32_t a_off = a_at < k ? a_at : 0u, b_off = b_at < (k >> 1) ? b_at : 0u;
#pragma unroll
    for (int i = 0; i < kAUnits; ++i)
      d.a[i].load(x + (size_t)min(m0 + arow0 + 32u * i, m - 1) * k + a_off);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      d.b[i] = *reinterpret_cast<const uint4*>(
          w + (size_t)min(n0 + brow0 + 128u * i, n - 1) * (k >> 1) + b_off);
  };
  auto park_stage = [&](uint32_t stage, int buf, Staged& d) {
    const uint32_t keep = stage * kStage + aunit < k ? 0xFFFFFFFFu : 0u;
#pragma unroll
    for (int i = 0; i < kAUnits; ++i) {
      uint4 v = d.a[i].paired();
      v.x &= keep; v.y &= keep; v.z &= keep; v.w &= keep;  // past K: zeros, whatever B holds
      *reinterpret_cast<uint4*>(&s_a[buf][(arow0 + 32u * i) * kRowA + aunit * 2u]) = v;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<uint4*>(&s_b[buf][(brow0 + 128u * i) * kRowB + bunit]) = d.b[i];
    // The stage's (at most two) group scales of this thread's column, fetched here by the first
    // four waves.  (Requested a stage ahead like the tiles, or all at once into an LDS table,
    // measured 5-8 % slower: every lane's scale sits in another cache line.)
    if (tid < 256) {
      const uint32_t c0 = stage * kStage, c1 = stage * kStage + 64u;
      s_s[buf][tid][0] = scale_from_bits<ST>(scale_bits<ST>(ssrc, (c0 < k ? c0 : 0u) >> group_shift));
      s_s[buf][tid][1] = scale_from_bits<ST>(scale_bits<ST>(ssrc, (c1 < k ? c1 : 0u) >> group_shift));
    }
  };

  float16_t acc[MT][WN];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < WN; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.f;

  Staged staged;
  load_stage(0, staged);
  park_stage(0, 0, staged);
  __syncthreads();

  const uint32_t a_base = (uint32_t)((wm * 32 * MT + frag_row) * kRowA + 64 * frag_h);
  const uint32_t b_base = (uint32_t)((wn * 64 + frag_row) * kRowB + 16 * frag_h);
  auto run_stage = [&](uint32_t stage, int buf) {
    load_stage(stage + 1, staged);
    // the requests stay here, a whole stage ahead of their use (left alone, the scheduler
    // moves them down to the parking code, where their latency is in the open)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      uint4 braw[WN];
      _Float16 ws[WN];
#pragma unroll
      for (int nt = 0; nt < WN; ++nt) {
        braw[nt] = *reinterpret_cast<const uint4*>(&s_b[buf][b_base + nt * 32 * kRowB + 32 * c]);
        ws[nt] = s_s[buf][wn * 64 + nt * 32 + frag_row][c];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        half8_t a[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          a[mt] = *reinterpret_cast<const half8_t*>(
              &s_a[buf][a_base + mt * 32 * kRowA + 128 * c + 16 * j]);
#pragma unroll
        for (int nt = 0; nt < WN; ++nt) {
          const uint32_t word = j == 0 ? braw[nt].x : j == 1 ? braw[nt].y : j == 2 ? braw[nt].z
                                                                                  : braw[nt].w;
          const half8_t b = __builtin_bit_cast(half8_t, dequant_word(word, ws[nt]));
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt], b, acc[mt][nt], 0, 0, 0);
        }
      }
    }
    park_stage(stage + 1, buf ^ 1, staged);
    __syncthreads();
  };
  for (uint32_t stage = 0; stage < stages; stage += 2) {
    run_stage(stage, 0);
    run_stage(stage + 1, 1);  // past the last stage: x is zeros
  }

#pragma unroll
  for (int nt = 0; nt < WN; ++nt) {
    const uint32_t col = n0 + wn * 64 + nt * 32 + frag_row;
    const float b = (bias && col < n) ? bias_f32<XT>(bias, col) : 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm * 32 * MT + mt * 32 + 8 * (r / 4) + 4 * frag_h + (r % 4);
        if (row < m && col < n) store_out<XT>(out, (size_t)row * n + col, acc[mt][nt][r] + b);
      }
  }
}

// ------------------------------------------------ packed weights in LDS, K dealt by units
//
// The same 128 x 256 tile and stage loop as above, for outputs whose tiles do not fill the
// chip evenly (172 tiles on 256 CUs leave a third idle; 64 tiles three quarters).  The work is
// the list of (tile, stage) units, tiles in column-block-major order; it is cut into one
// contiguous range per workgroup (the grid is one workgroup per CU, ranges differ by at most
// one unit), so a tile is computed by up to a few workgroups, each over a slice of K.  A
// workgroup that computes a whole tile stores it.  Otherwise it writes its 128 x 256 f32
// partial (device-scope stores, each thread its own registers, 16 bytes at a time), waits for
// the stores, and takes a ticket on the tile's counter; the workgroup that arrives last adds
// the partials in ascending K order — its own from registers — so the bits do not depend on
// who arrives last.  No workgroup ever waits for another.
// WM = 2 (the one in use): eight waves, wave = 64 x 64, two waves a SIMD, as above.  WM = 1: four
// waves, wave = 128 x 64, every weight word dequantised once for four MFMAs instead of twice for
// two — measured 101 us against 78 us on the 512 x 11008 x 4096 product: the single wave of a
// SIMD does not hide its own LDS reads and dequantisation under its MFMAs as compiled (and
// spills 31 registers).
template <typename XT, typename ST, int WM>
__global__ __launch_bounds__(WM * 256) __attribute__((amdgpu_waves_per_eu(WM, WM)))
void gemm_i4_f16_dealt_kernel(const XT* __restrict__ x, const uint8_t* __restrict__ w,
                              const ST* __restrict__ scales, const XT* __restrict__ bias,
                              XT* __restrict__ out, uint32_t m, uint32_t n, uint32_t k,
                              uint32_t group_shift, uint32_t m_blocks, UnitDeal deal) {
  constexpr int MT = 4 / WM, WN = 2;
  constexpr int T = WM * 256;  // threads
  constexpr int BM = WM * 32 * MT, BN = 256;
  static_assert(BM == 128, "the partial layout and the deal assume 128 x 256 tiles");
  constexpr int kStage = 128;
  constexpr int kRowA = kStage * 2 + 16;
  constexpr int kRowB = kStage / 2 + 16;
  constexpr int kAUnits = BM * (kStage / 8) / T;
  constexpr int kBUnits = BN * (kStage / 32) / T;
  __shared__ __align__(16) uint8_t s_a[2][BM * kRowA];
  __shared__ __align__(16) uint8_t s_b[2][BN * kRowB];
  __shared__ _Float16 s_s[2][BN][2];
  __shared__ uint32_t s_ticket;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int frag_row = lane & 31, frag_h = lane >> 5;
  const uint32_t groups = k >> group_shift;
  const uint32_t spt = deal.stages_per_tile;
  const uint32_t arow0 = tid >> 4, aunit = (tid & 15u) * 8u;
  const uint32_t brow0 = tid >> 2, bunit = (tid & 3u) * 16u;
  const uint32_t a_base = (uint32_t)((wm * 32 * MT + frag_row) * kRowA + 64 * frag_h);
  const uint32_t b_base = (uint32_t)((wn * 64 + frag_row) * kRowB + 16 * frag_h);

  // the workgroups of one XCD (ids equal mod 8) take neighbouring ranges: the row panels of a
  // column block then mostly share an L2
  uint32_t v = blockIdx.x;
  if ((gridDim.x & 7u) == 0) v = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const uint32_t my_begin = deal_begin(deal, v);
  uint32_t left = deal_units(deal, v);

  // The tiles of the range are taken last to first: a range usually ends with the first stages
  // of a tile and begins with the last stages of the one before, so every workgroup then walks
  // K upwards from (about) stage 0 and, at any moment, the chip reads few distinct K slices of
  // x, which stay in the L2s.
  while (left > 0) {
    const uint32_t range_end = my_begin + left;
    const uint32_t tile = (range_end - 1u) / spt;
    const uint32_t tile_first = tile * spt;
    const uint32_t s0 = my_begin > tile_first ? my_begin - tile_first : 0u;
    const uint32_t s1 = range_end - tile_first;
    const uint32_t nb = tile / m_blocks, mb = tile - nb * m_blocks;
    const uint32_t m0 = mb * BM, n0 = nb * BN;
    const ST* ssrc = scales + (size_t)min(n0 + (uint32_t)(tid & 255), n - 1) * groups;

    struct Staged {
      Acts8<XT> a[kAUnits];
      uint4 b[kBUnits];
    };
    auto load_stage = [&](uint32_t stage, Staged& d) {
      const uint32_t a_at = stage * kStage + aunit, b_at = stage * (kStage / 2) + bunit;
      const uint32_t a_off = a_at < k ? a_at : 0u, b_off = b_at < (k >> 1) ? b_at : 0u;
#pragma unroll
      for (int i = 0; i < kAUnits; ++i)
        d.a[i].load(x + (size_t)min(m0 + arow0 + (uint32_t)(T / 16) * i, m - 1) * k + a_off);
#pragma unroll
      for (int i = 0; i < kBUnits; ++i)
        d.b[i] = *reinterpret_cast<const uint4*>(
            w + (size_t)min(n0 + brow0 + (uint32_t)(T / 4) * i, n - 1) * (k >> 1) + b_off);
    };
    auto park_stage = [&](uint32_t stage, int buf, Staged& d) {
      const uint32_t keep = stage * kStage + aunit < k ? 0xFFFFFFFFu : 0u;
#pragma unroll
      for (int i = 0; i < kAUnits; ++i) {
        uint4 pv = d.a[i].paired();
        pv.x &= keep; pv.y &= keep; pv.z &= keep; pv.w &= keep;
        *reinterpret_cast<uint4*>(&s_a[buf][(arow0 + (uint32_t)(T / 16) * i) * kRowA + aunit * 2u]) = pv;
      }
#pragma unroll
      for (int i = 0; i < kBUnits; ++i)
        *reinterpret_cast<uint4*>(&s_b[buf][(brow0 + (uint32_t)(T / 4) * i) * kRowB + bunit]) = d.b[i];
      if (tid < 256) {
        const uint32_t c0 = stage * kStage, c1 = stage * kStage + 64u;
        s_s[buf][tid][0] = scale_from_bits<ST>(scale_bits<ST>(ssrc, (c0 < k ? c0 : 0u) >> group_shift));
        s_s[buf][tid][1] = scale_from_bits<ST>(scale_bits<ST>(ssrc, (c1 < k ? c1 : 0u) >> group_shift));
      }
    };

    float16_t acc[MT][WN];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < WN; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.f;

    Staged staged;
    load_stage(s0, staged);
    park_stage(s0, 0, staged);
    __syncthreads();

    auto run_stage = [&](uint32_t stage, int buf) {
      load_stage(stage + 1, staged);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint4 braw[WN];
        _Float16 ws[WN];
#pragma unroll
        for (int nt = 0; nt < WN; ++nt) {
          braw[nt] = *reinterpret_cast<const uint4*>(&s_b[buf][b_base + nt * 32 * kRowB + 32 * c]);
          ws[nt] = s_s[buf][wn * 64 + nt * 32 + frag_row][c];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          half8_t a[MT];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            a[mt] = *reinterpret_cast<const half8_t*>(
                &s_a[buf][a_base + mt * 32 * kRowA + 128 * c + 16 * j]);
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) {
            const uint32_t word = j == 0 ? braw[nt].x : j == 1 ? braw[nt].y : j == 2 ? braw[nt].z
                                                                                    : braw[nt].w;
            const half8_t b = __builtin_bit_cast(half8_t, dequant_word(word, ws[nt]));
            // the wave that feeds the matrix pipe goes first; the other one dequantises meanwhile
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt], b, acc[mt][nt], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
          }
        }
      }
      park_stage(stage + 1, buf ^ 1, staged);
      __syncthreads();
    };
    for (uint32_t stage = s0; stage < s1; stage += 2) {
      run_stage(stage, 0);
      if (stage + 1 < s1) run_stage(stage + 1, 1);
    }

    auto store_block = [&](int mt, int nt, const float16_t& total) {
      const uint32_t col = n0 + wn * 64 + nt * 32 + frag_row;
      const float b = (bias && col < n) ? bias_f32<XT>(bias, col) : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm * 32 * MT + mt * 32 + 8 * (r / 4) + 4 * frag_h + (r % 4);
        if (row < m && col < n) store_out<XT>(out, (size_t)row * n + col, total[r] + b);
      }
    };

    if (s0 == 0 && s1 == spt) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < WN; ++nt) store_block(mt, nt, acc[mt][nt]);
    } else {
      // Slot of workgroup u's partial of this tile: its second slot when its range began at or
      // before the tile's first unit, its first slot otherwise (a range holds at most one
      // partial of either kind).  16-byte piece c of thread t sits at [c * threads + t].
      const uint32_t tile_begin = tile * spt;
      auto slot_of = [&](uint32_t u) {
        return 2u * u + (deal_begin(deal, u) <= tile_begin ? 1u : 0u);
      };
      uint32_t* ticket = deal.tickets + (size_t)tile * kTicketStride;
      const uint32_t first = deal_owner(deal, tile_begin), last = deal_owner(deal, tile_begin + spt - 1u);
      // Every other partial already there (the usual case for the slice computed last: slices
      // that open a range finish early)?  Then this one need not be written at all.
      if (tid == 0)
        s_ticket = __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      bool merge = s_ticket == last - first;
      __syncthreads();  // s_ticket is written again below
      if (!merge) {
        float4_t* mine =
            reinterpret_cast<float4_t*>(deal.partials + (size_t)slot_of(v) * kPartialFloats);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < WN; ++nt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float4_t piece = {acc[mt][nt][4 * q], acc[mt][nt][4 * q + 1],
                                      acc[mt][nt][4 * q + 2], acc[mt][nt][4 * q + 3]};
              publish4(mine + (size_t)(((mt * WN + nt) * 4 + q) * T + tid), piece);
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial is in memory
        __syncthreads();
        if (tid == 0)
          s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        merge = s_ticket == last - first;  // arrived last after all
      }
      if (merge) {  // every other partial of the tile is complete
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float16_t total[WN];
          for (uint32_t u = first; u <= last; ++u) {
            float16_t part[WN];
#pragma unroll
            for (int nt = 0; nt < WN; ++nt) part[nt] = acc[mt][nt];
            if (u != v) {
              const float4_t* src =
                  reinterpret_cast<const float4_t*>(deal.partials + (size_t)slot_of(u) * kPartialFloats) +
                  (size_t)(mt * WN * 4 * T + tid);
              float4_t p[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) p[i] = observe4(src + (size_t)i * T);
              landed(p);
#pragma unroll
              for (int nt = 0; nt < WN; ++nt)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                  for (int i = 0; i < 4; ++i) part[nt][4 * q + i] = p[nt * 4 + q][i];
            }
#pragma unroll
            for (int nt = 0; nt < WN; ++nt) {
              if (u == first) {
                total[nt] = part[nt];
              } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) total[nt][r] += part[nt][r];
              }
            }
          }
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) store_block(mt, nt, total[nt]);
        }
        if (tid == 0)
          __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    left -= s1 - s0;
  }
}

// ------------------------------------------------ exact integer operands, 64 x 512 tiles
//
// The weights enter the matrix cores as the exact integers (u - 8) in fp16 and the group scale
// multiplies the f32 sum of a group afterwards — the arithmetic of the GEMV, on MFMA.  x is rounded to
// fp16 once (exact when it already is fp16): one MFMA a step.  (f32 x as hi + lo, and fp16 x where the
// ranges are long: gemm_i4_exact.hip, which also holds what was measured of both.)
// Tile 64 x 512, eight waves side by side (wave = 64 rows x 64 columns = 2 x 2 MFMA tiles), so
// every weight word is turned into integers exactly once per workgroup (in the 128 x 256 tile
// above the two waves of a column strip each do it).  Per MFMA step the wave holds the sums of
// the current scale group in `acc`; at a group's end total = fma(acc, scale[column], total)
// (the C layout keeps the column in lane % 32, so the scale is one value per lane and column
// tile).  Stages, LDS layout, the (tile, stage) deal over the CUs and the ordered merge of the
// partials are those of the kernel above.
// OT: of the bias and the result (f32 beside fp16 x: rows that were rounded before).
template <typename XT, typename OT, typename ST>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_i4_staged_kernel(const XT* __restrict__ x, const uint8_t* __restrict__ w,
                          const ST* __restrict__ scales, const OT* __restrict__ bias,
                          OT* __restrict__ out, uint32_t m, uint32_t n, uint32_t k,
                          uint32_t group_shift, uint32_t m_blocks, UnitDeal deal) {
  constexpr int MT = 2, WN = 2, T = 512;
  constexpr int BM = 64, BN = 512;
  constexpr int kStage = 128;
  constexpr int kRowA = kStage * 2 + 16;
  constexpr int kRowB = kStage / 2 + 16;
  constexpr int kAUnits = BM * (kStage / 8) / T;   // 2
  constexpr int kBUnits = BN * (kStage / 32) / T;  // 4
  constexpr bool kWhole = sizeof(ST) == 4 && sizeof(OT) == 4;  // the totals (see scales_whole)
  static_assert((size_t)BM * BN == kPartialFloats, "the partial slots hold one tile");
  __shared__ __align__(16) uint8_t s_a[2][BM * kRowA];
  __shared__ __align__(16) uint8_t s_b[2][BN * kRowB];
  __shared__ float s_s[2][BN][2];
  __shared__ uint32_t s_ticket;

  const int tid = threadIdx.x, lane = tid & 63, wn = tid >> 6;
  const int frag_row = lane & 31, frag_h = lane >> 5;
  const uint32_t groups = k >> group_shift;
  const bool half_stage_groups = group_shift == 6;  // 64 codes a group: two groups a stage
  const uint32_t spt = deal.stages_per_tile;
  const uint32_t arow0 = tid >> 4, aunit = (tid & 15u) * 8u;
  const uint32_t brow0 = tid >> 2, bunit = (tid & 3u) * 16u;
  const uint32_t a_base = (uint32_t)(frag_row * kRowA + 64 * frag_h);
  const uint32_t b_base = (uint32_t)((wn * 64 + frag_row) * kRowB + 16 * frag_h);

  uint32_t v = blockIdx.x;
  if ((gridDim.x & 7u) == 0) v = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const uint32_t my_begin = deal_begin(deal, v);
  uint32_t left = deal_units(deal, v);

  while (left > 0) {
    const uint32_t range_end = my_begin + left;
    const uint32_t tile = __builtin_amdgcn_readfirstlane((range_end - 1u) / spt);
    const uint32_t tile_first = tile * spt;
    const uint32_t s0 = my_begin > tile_first ? my_begin - tile_first : 0u;
    const uint32_t s1 = range_end - tile_first;
    const uint32_t nb = __builtin_amdgcn_readfirstlane(tile / m_blocks), mb = tile - nb * m_blocks;
    const uint32_t m0 = mb * BM, n0 = nb * BN;
    const ST* const s_tile = scales + (size_t)n0 * groups;
    const uint32_t s_row = min((uint32_t)tid, n - 1 - n0) * groups;
    // the tile's rows: one base each and 32-bit offsets (plan_staged bounds K)
    const uint8_t* const x_tile = reinterpret_cast<const uint8_t*>(x) + (size_t)m0 * k * sizeof(XT);
    const uint8_t* const w_tile = w + (size_t)n0 * (k >> 1);
    struct Staged {
      Acts8<XT> a[kAUnits];
      uint4 b[kBUnits];
    };
    auto load_stage = [&](uint32_t stage, Staged& d) {
      const uint32_t a_at = stage * kStage + aunit, b_at = stage * (kStage / 2) + bunit;
      // (opaque, so that the rows' offsets are formed here and hold no registers between stages)
      uint32_t a_last = m - 1 - m0, b_last = n - 1 - n0;
      asm volatile("" : "+s"(a_last), "+s"(b_last));
      const uint32_t a_off = a_at < k ? a_at : 0u, b_off = b_at < (k >> 1) ? b_at : 0u;
#pragma unroll
      for (int i = 0; i < kAUnits; ++i)
        d.a[i].load(reinterpret_cast<const XT*>(x_tile + (min(arow0 + 32u * i, a_last) * k + a_off) * (uint32_t)sizeof(XT)));
#pragma unroll
      for (int i = 0; i < kBUnits; ++i)
        d.b[i] = *reinterpret_cast<const uint4*>(w_tile + (min(brow0 + 128u * i, b_last) * (k >> 1) + b_off));
    };
    auto park_stage = [&](uint32_t stage, int buf, Staged& d) {
      const uint32_t keep = stage * kStage + aunit < k ? 0xFFFFFFFFu : 0u;
#pragma unroll
      for (int i = 0; i < kAUnits; ++i) {
        const uint32_t at = (arow0 + 32u * i) * kRowA + aunit * 2u;
        uint4 pv = d.a[i].paired();
        pv.x &= keep; pv.y &= keep; pv.z &= keep; pv.w &= keep;  // past K: zeros
        *reinterpret_cast<uint4*>(&s_a[buf][at]) = pv;
      }
#pragma unroll
      for (int i = 0; i < kBUnits; ++i)
        *reinterpret_cast<uint4*>(&s_b[buf][(brow0 + 128u * i) * kRowB + bunit]) = d.b[i];
      const uint32_t c0 = stage * kStage, c1 = stage * kStage + 64u;
      s_s[buf][tid][0] = load_scale_f32<ST>(s_tile, s_row + ((c0 < k ? c0 : 0u) >> group_shift));
      s_s[buf][tid][1] = load_scale_f32<ST>(s_tile, s_row + ((c1 < k ? c1 : 0u) >> group_shift));
    };

    float16_t total[MT][WN], acc[MT][WN];
    float16_t zero16;
#pragma unroll
    for (int r = 0; r < 16; ++r) zero16[r] = 0.f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < WN; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) total[mt][nt][r] = acc[mt][nt][r] = 0.f;

    Staged staged;
    load_stage(s0, staged);
    park_stage(s0, 0, staged);
    __syncthreads();

    auto run_stage = [&](uint32_t stage, int buf) {
      load_stage(stage + 1, staged);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint4 braw[WN];
        float ws[WN];
#pragma unroll
        for (int nt = 0; nt < WN; ++nt) {
          braw[nt] = *reinterpret_cast<const uint4*>(&s_b[buf][b_base + nt * 32 * kRowB + 32 * c]);
          ws[nt] = s_s[buf][wn * 64 + nt * 32 + frag_row][c];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          half8_t a[MT];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            a[mt] = *reinterpret_cast<const half8_t*>(&s_a[buf][a_base + mt * 32 * kRowA + 128 * c + 16 * j]);
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) {
            const uint32_t word = j == 0 ? braw[nt].x : j == 1 ? braw[nt].y : j == 2 ? braw[nt].z
                                                                                    : braw[nt].w;
            const half8_t b = ints_paired<true>(word);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
              // the first product of a scale group starts from zero (an inline constant of the
              // instruction: the sums are not cleared by VALU moves)
              const bool opens = j == 0 && (c == 0 || half_stage_groups);
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mt], b, opens ? zero16 : acc[mt][nt], 0, 0, 0);
            }
            __builtin_amdgcn_s_setprio(0);
          }
        }
        if (c == 1 || half_stage_groups) {  // the scale group ends here
          if constexpr (kWhole) {
            if (scales_whole(ws)) {
#pragma unroll
              for (int i = 0; i < MT * WN; ++i) acc[i / WN][i % WN] *= 1024.0f;
            }
          }
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < WN; ++nt)
#pragma unroll
              for (int r = 0; r < 16; ++r)
                total[mt][nt][r] = fmaf(acc[mt][nt][r], ws[nt], total[mt][nt][r]);
        }
      }
      park_stage(stage + 1, buf ^ 1, staged);
      __syncthreads();
    };
    for (uint32_t stage = s0; stage < s1; stage += 2) {
      run_stage(stage, 0);
      if (stage + 1 < s1) run_stage(stage + 1, 1);
    }

    auto store_block = [&](int mt, int nt, const float16_t& sum) {
      const uint32_t col = n0 + wn * 64 + nt * 32 + frag_row;
      const float b = (bias && col < n) ? bias_f32<OT>(bias, col) : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t local = mt * 32 + 8 * (r / 4) + 4 * frag_h + (r % 4);
        const uint32_t row = m0 + local;
        if (row < m && col < n) store_out<OT>(out, (size_t)row * n + col, (kWhole ? sum[r] : sum[r] * 1024.0f) + b);
      }
    };

    if (s0 == 0 && s1 == spt) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < WN; ++nt) store_block(mt, nt, total[mt][nt]);
    } else {
      const uint32_t tile_begin = tile * spt;
      auto slot_of = [&](uint32_t u) {
        return 2u * u + (deal_begin(deal, u) <= tile_begin ? 1u : 0u);
      };
      uint32_t* ticket = deal.tickets + (size_t)tile * kTicketStride;
      const uint32_t first = deal_owner(deal, tile_begin), last = deal_owner(deal, tile_begin + spt - 1u);
      if (tid == 0)
        s_ticket = __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      bool merge = s_ticket == last - first;
      __syncthreads();
      if (!merge) {
        float4_t* mine =
            reinterpret_cast<float4_t*>(deal.partials + (size_t)slot_of(v) * kPartialFloats);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < WN; ++nt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float4_t piece = {total[mt][nt][4 * q], total[mt][nt][4 * q + 1],
                                      total[mt][nt][4 * q + 2], total[mt][nt][4 * q + 3]};
              publish4(mine + (size_t)(((mt * WN + nt) * 4 + q) * T + tid), piece);
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
          s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        merge = s_ticket == last - first;
      }
      if (merge) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          float16_t sum[WN];
          for (uint32_t u = first; u <= last; ++u) {
            float16_t part[WN];
#pragma unroll
            for (int nt = 0; nt < WN; ++nt) part[nt] = total[mt][nt];
            if (u != v) {
              const float4_t* src =
                  reinterpret_cast<const float4_t*>(deal.partials + (size_t)slot_of(u) * kPartialFloats) +
                  (size_t)(mt * WN * 4 * T + tid);
              float4_t p[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) p[i] = observe4(src + (size_t)i * T);
              landed(p);
#pragma unroll
              for (int nt = 0; nt < WN; ++nt)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                  for (int i = 0; i < 4; ++i) part[nt][4 * q + i] = p[nt * 4 + q][i];
            }
#pragma unroll
            for (int nt = 0; nt < WN; ++nt) {
              if (u == first) {
                sum[nt] = part[nt];
              } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) sum[nt][r] += part[nt][r];
              }
            }
          }
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) store_block(mt, nt, sum[nt]);
        }
        if (tid == 0)
          __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();  // the LDS tiles are rewritten by the next tile of the range
    left -= s1 - s0;
  }
}

// The deal of the 64 x 512 tiles: one workgroup per CU, every workgroup at least two stages.
bool plan_staged(krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t group, bool half_x,
                     uint32_t& grid, UnitDeal& deal) {
  const uint64_t cus = (uint64_t)ctx->num_cus;
  const uint64_t tiles = (uint64_t)((m + 63) / 64) * ((n + 511) / 512);
  const uint32_t spt = (k + 127) / 128;
  const uint64_t units = tiles * spt;
  if (tiles > kTicketSlots || units > 0x7fffffffull || units < 2 * cus) return false;
  if (k > 1u << 24) return false;  // 32-bit offsets inside a tile's rows
  if (units < 12 * cus) {
    // Fewer than twelve stages a workgroup: the K-splitting tiles of gemm_i4_slices.hip, unless
    // their estimate is clearly above this form's, {fixed, a stage} in us, fitted over 16 to 21 shapes
    // (rms 6 to 8 %).  Over 100 shapes of 65 to 512 rows the choice is 1 % behind the better of the two
    // and 4 % at worst behind the tiles alone.  us there / here: fp16 406 x 24848 x 512 in groups of 64 61 / 27, 198 x 26342 x 768 35 / 24, 237 x
    // 7285 x 2688 in groups of 64 26 / 31; f32 rounded to fp16 399 x 26833 x 896 in groups of 64 115 /
    // 57, 169 x 8597 x 1664 19 / 33.
    struct Fit {
      float fixed, stage;
    };
    const bool wide_groups = group >= 128;
    const Fit f = half_x ? (wide_groups ? Fit{14.1f, 2.45f} : Fit{14.7f, 2.6f})
                         : (wide_groups ? Fit{19.8f, 2.7f} : Fit{20.6f, 3.1f});
    const float here = f.fixed + f.stage * ((float)units / (float)cus);
    if (here > 0.88f * slices_estimate_us(ctx, m, n, k, group, half_x, false)) return false;
  }
  // Up to six 32 x 32 tiles of output a CU stay with the tiles that split K inside a workgroup, which
  // need no scratch with fp16 operands (a side branch of a graph may hold them) and give a row the
  // same bits whatever M is.  fp16, us there / here: 128 x 12288 x 8192 41.9 / 52.2, 256 x 4096 x 12288
  // 39.8 / 48.2, 96 x 8192 x 16384 55.9 / 60.3, 192 x 8192 x 8192 48.8 / 47.7, but 384 x 4096 x 16384
  // 98 / 78.
  if ((uint64_t)((m + 31) / 32) * ((n + 31) / 32) <= 6 * cus) return false;
  if (tiles * 8 < cus) return false;  // a tile shared by more than eight workgroups
  if (!ctx->gemm_partials) return false;
  grid = (uint32_t)cus;
  deal.stages_per_tile = spt;
  deal.units_lo = (uint32_t)(units / cus);
  deal.extra = (uint32_t)(units % cus);
  deal.partials = ctx->gemm_partials;
  deal.tickets = ctx->tickets;
  return true;
}

// Workgroups, units and scratch of a dealt launch; false when the shape is not worth it.
bool plan_deal(krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t& grid, UnitDeal& deal) {
  const uint64_t cus = (uint64_t)ctx->num_cus;
  const uint64_t tiles = (uint64_t)((m + 127) / 128) * ((n + 255) / 256);
  const uint32_t spt = (k + 127) / 128;
  const uint64_t units = tiles * spt;
  // at least four stages to a workgroup: with less, a tile is the sum of so many short slices
  // that writing and merging the partials costs more than the idle CUs did (128 x 11264 x 2048:
  // 2.75 stages each, 36.8 us against 30.9 us for one workgroup per 128 x 64 tile)
  if (tiles > kTicketSlots || units > 0x7fffffffull || units < 4 * cus) return false;
  // whole rounds of tiles already use the chip well
  const uint64_t rounds = (tiles + cus - 1) / cus;
  if (tiles * 10 >= rounds * cus * 9) return false;
  // a tile shared by many workgroups costs more in partials than the idle CUs did
  if (tiles * 6 < cus) return false;
  if (!ctx->gemm_partials) return false;
  grid = (uint32_t)cus;
  deal.stages_per_tile = spt;
  deal.units_lo = (uint32_t)(units / cus);
  deal.extra = (uint32_t)(units % cus);
  deal.partials = ctx->gemm_partials;
  deal.tickets = ctx->tickets;
  return true;
}

template <typename XT, typename ST, int WM>
int32_t launch_dealt(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out,
                     uint32_t m, uint32_t n, uint32_t k, uint32_t group_shift, uint32_t grid,
                     const UnitDeal& deal) {
  KRM_TRY(needs_serial_scratch(ctx, "the unit-dealt GEMM"));
  gemm_i4_f16_dealt_kernel<XT, ST, WM><<<dim3(grid), dim3(WM * 256), 0, ctx->stream>>>(
      ptr<const XT>(x), ptr<const uint8_t>(w), ptr<const ST>(scales), ptr<const XT>(bias),
      ptr<XT>(out), m, n, k, group_shift, (m + 127) / 128, deal);
  return launched(ctx, "gemm_i4_f16_dealt_kernel");
}

template <typename XT, typename ST, int MT>
int32_t launch_packed(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias,
                      krm_buf out, uint32_t m, uint32_t n, uint32_t k, uint32_t group_shift) {
  const uint32_t m_blocks = (m + 64 * MT - 1) / (64 * MT), n_blocks = (n + 255) / 256;
  const uint64_t total = (uint64_t)((n_blocks + 7) / 8) * 8 * m_blocks;
  if (total > 0x7fffffffull) return fail(ctx, KRM_ERR_VALIDATION, "linear: grid too large");
  gemm_i4_f16_packed_kernel<XT, ST, MT><<<dim3((unsigned)total), dim3(512), 0, ctx->stream>>>(
      ptr<const XT>(x), ptr<const uint8_t>(w), ptr<const ST>(scales), ptr<const XT>(bias),
      ptr<XT>(out), m, n, k, group_shift, m_blocks, n_blocks);
  return launched(ctx, "gemm_i4_f16_packed_kernel");
}

template <typename XT, typename ST, int WM, int WN, int KC, int KS, int DEPTH, bool PIPE = false>
int32_t launch(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out,
               uint32_t m, uint32_t n, uint32_t k, uint32_t group_shift) {
  constexpr int BM = WM * 64, BN = WN * 64;
  const uint32_t m_blocks = (m + BM - 1) / BM, n_blocks = (n + BN - 1) / BN;
  uint64_t total;
  if (8 % m_blocks == 0) {
    total = (uint64_t)((n_blocks + 7) / 8) * 8 * m_blocks;
  } else {
    total = (uint64_t)m_blocks * n_blocks;
  }
  if (total > 0x7fffffffull) return fail(ctx, KRM_ERR_VALIDATION, "linear: grid too large");
  constexpr int kWordsPerThread = BN * (KC / 8) / (WM * WN * KS * 64);
  const uint32_t wide = (k % 32 == 0 && aligned(w, 16)) ? 1u : 0u;
  const bool fast = wide && kWordsPerThread >= 4 && k % KC == 0 &&
                    (((uint32_t)(kWordsPerThread * 8 - 1) >> group_shift) == 0);
  if (fast)
    gemm_i4_f16_kernel<XT, ST, WM, WN, KC, KS, DEPTH, PIPE, true>
        <<<dim3((unsigned)total), dim3(WM * WN * KS * 64), 0, ctx->stream>>>(
            ptr<const XT>(x), ptr<const uint32_t>(w), ptr<const ST>(scales), ptr<const XT>(bias),
            ptr<XT>(out), m, n, k, group_shift, m_blocks, n_blocks, wide);
  else
    gemm_i4_f16_kernel<XT, ST, WM, WN, KC, KS, DEPTH, PIPE, false>
        <<<dim3((unsigned)total), dim3(WM * WN * KS * 64), 0, ctx->stream>>>(
            ptr<const XT>(x), ptr<const uint32_t>(w), ptr<const ST>(scales), ptr<const XT>(bias),
            ptr<XT>(out), m, n, k, group_shift, m_blocks, n_blocks, wide);
  return launched(ctx, "gemm_i4_f16_kernel");
}

template <typename XT, typename ST>
int32_t pick_tile(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out,
                  uint32_t m, uint32_t n, uint32_t k, uint32_t group) {
  uint32_t group_shift = 0;
  while ((1u << group_shift) < group) ++group_shift;
  // 128 x 64 tiles (two waves, chunks of 64 codes, two chunks in flight) when they fill the
  // chip at least twice over.  Otherwise four wave groups split every 128-code chunk of K
  // between them on a 64 x 64 tile: four times the waves for the same outputs.
  // Enough 128 x 128 tiles for every CU: four waves a tile, chunks of 64 codes, pipelined with
  // four chunks in flight.  Fewer (a narrow output with a long K, or few rows): 128 x 64 tiles
  // whose two wave groups split every 128-code chunk of K, or 64 x 64 tiles with four groups.
  const uint64_t cus = (uint64_t)ctx->num_cus;
  // 128 x 256 tiles with the packed weights in LDS.  Dealt by (tile, stage) units over all CUs
  // when whole rounds of tiles would leave part of the chip idle (512 x 11008 x 4096: 69 us
  // against 77 us for one workgroup per tile; 512 x 4096 x 11008: 75 us against 93 us for the
  // K-splitting form below); one workgroup per tile when the tiles cover most of the chip; with
  // fewer tiles the forms below, which split K inside a workgroup.
  const uint64_t packed_tiles = (uint64_t)((m + 127) / 128) * ((n + 255) / 256);
  const bool packed_ok = m > 64 && group >= 64 && k % 8 == 0 && aligned(w, 16) && aligned(x, 16);
  if (packed_ok) {
    uint32_t grid = 0;
    UnitDeal deal{};
    if (plan_deal(ctx, m, n, k, grid, deal))
      return launch_dealt<XT, ST, 2>(ctx, x, w, scales, bias, out, m, n, k, group_shift, grid, deal);
  }
  if (packed_ok && packed_tiles * 5 >= cus * 3)
    return launch_packed<XT, ST, 2>(ctx, x, w, scales, bias, out, m, n, k, group_shift);
  const uint64_t tiles = (uint64_t)((m + 127) / 128) * ((n + 127) / 128);
  if (m > 64 && tiles >= cus)
    return launch<XT, ST, 2, 2, 64, 1, 4, true>(ctx, x, w, scales, bias, out, m, n, k, group_shift);
  // Few tiles and a K of several chunks: 64 x 64 tiles whose four wave groups split every
  // 128-code chunk, two LDS copies and two chunks in flight (measured on 128-row products:
  // N = 2048, K = 2048 21.5 us against 28.3 us for the 128 x 64 form below and 25.7 us for the
  // same tiles with one copy; N = 2048, K = 5632 37 us against 58 us).
  const uint64_t tiles_128x64 = (uint64_t)((m + 127) / 128) * ((n + 63) / 64);
  if (k >= 512 && (m <= 64 || tiles_128x64 * 2 < cus))
    return launch<XT, ST, 1, 1, 128, 4, 2, true>(ctx, x, w, scales, bias, out, m, n, k, group_shift);
  if (m > 64 && k >= 256)
    return launch<XT, ST, 2, 1, 128, 2, 2, true>(ctx, x, w, scales, bias, out, m, n, k, group_shift);
  return launch<XT, ST, 1, 1, 64, 1, 1>(ctx, x, w, scales, bias, out, m, n, k, group_shift);
}

template <typename XT, typename OT, typename ST>
int32_t launch_staged(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out,
                     uint32_t m, uint32_t n, uint32_t k, uint32_t group_shift, uint32_t grid,
                     const UnitDeal& deal) {
  KRM_TRY(needs_serial_scratch(ctx, "the unit-dealt GEMM"));
  gemm_i4_staged_kernel<XT, OT, ST><<<dim3(grid), dim3(512), 0, ctx->stream>>>(
      ptr<const XT>(x), ptr<const uint8_t>(w), ptr<const ST>(scales), ptr<const OT>(bias),
      ptr<OT>(out), m, n, k, group_shift, (m + 63) / 64, deal);
  return launched(ctx, "gemm_i4_staged_kernel");
}

}  // namespace

namespace krm {

// Whether f32 x of this shape, rounded to fp16, comes to the staged tiles (buffers aligned, main stream).
bool gemm_staged_takes_f32(krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t group) {
  uint32_t grid = 0;
  UnitDeal deal{};
  return group >= 64 && plan_staged(ctx, m, n, k, group, false, grid, deal);
}

// The exact-integer GEMM with x in fp16 for shapes whose (tile, stage) units cover the chip; sets
// *handled = false (and launches nothing) for every other shape.
int32_t linear_i4_gemm_staged(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias,
                             krm_buf out, uint32_t m, uint32_t n, uint32_t k, uint32_t group,
                             int32_t io_dtype, int32_t scale_dtype, int32_t compute,
                             bool* handled, int32_t x_dtype) {
  *handled = false;
  if (compute == KRM_COMPUTE_F32 && io_dtype == KRM_F32) return KRM_OK;
  if (group < 64 || k % 32 != 0 || !aligned(w, 16) || !aligned(x, 16)) return KRM_OK;
  uint32_t grid = 0;
  UnitDeal deal{};
  // (a side branch of a graph has no scratch: there the K-splitting tiles, which need none with fp16
  // operands, take these shapes too)
  if (ctx->stream != ctx->main_stream) return KRM_OK;
  if (!plan_staged(ctx, m, n, k, group, x_dtype == KRM_F16, grid, deal)) return KRM_OK;
  uint32_t group_shift = 0;
  while ((1u << group_shift) < group) ++group_shift;
  *handled = true;
#define KRM_STAGED(XT, OT, ST) \
  return launch_staged<XT, OT, ST>(ctx, x, w, scales, bias, out, m, n, k, group_shift, grid, deal)
  if (io_dtype == KRM_F16) {
    if (scale_dtype == KRM_F16) KRM_STAGED(__half, __half, __half);
    KRM_STAGED(__half, __half, float);
  }
  if (x_dtype == KRM_F16) {
    if (scale_dtype == KRM_F16) KRM_STAGED(__half, float, __half);
    KRM_STAGED(__half, float, float);
  }
  if (scale_dtype == KRM_F16) KRM_STAGED(float, float, __half);
  KRM_STAGED(float, float, float);
#undef KRM_STAGED
}

int32_t linear_i4_gemm_f16(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias,
                           krm_buf out, uint32_t m, uint32_t n, uint32_t k, uint32_t group,
                           int32_t io_dtype, int32_t scale_dtype) {
  if (io_dtype == KRM_F16) {
    if (scale_dtype == KRM_F16)
      return pick_tile<__half, __half>(ctx, x, w, scales, bias, out, m, n, k, group);
    return pick_tile<__half, float>(ctx, x, w, scales, bias, out, m, n, k, group);
  }
  if (scale_dtype == KRM_F16)
    return pick_tile<float, __half>(ctx, x, w, scales, bias, out, m, n, k, group);
  return pick_tile<float, float>(ctx, x, w, scales, bias, out, m, n, k, group);
}

}  // namespace krm
