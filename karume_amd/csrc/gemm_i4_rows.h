// What the exact-integer MFMA products share (gemm_i4_slices.hip, gemm_i4_exact.hip): packed codes to
// fp16 integers, loads from memory into LDS with counted waits, f32 x as two fp16 planes, and what
// happens to a finished pair of columns.
#pragma once

#include "i4_codes.h"
#include "lds_stream.h"

namespace krm {
namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));

// 8 codes of a word -> 8 fp16 integers in their own order (ints_paired: the order of activations stored
// as (x0,x4,x1,x5,x2,x6,x3,x7)).
// Natural order c0..c7, as (u - 8) / 1024 (the sum over K is multiplied by 1024 at the end): the
// even and the odd codes of the word are masked apart where they are and a byte of each becomes a pair
// of fp16 subnormals, u 2^-24 and 16 u 2^-24, which one packed fma scales and offsets exactly (ten
// ops a word; magic numbers in the mantissa took a byte copy and a mask a pair, twelve: 512 x 11008 x
// 4096, fp16 x, 57.8 us, 56.8 so).
__device__ inline half8_t ints_natural(uint32_t word) {
  const half2_t factor = {(_Float16)16384.0f, (_Float16)1024.0f};
  const half2_t offset = {(_Float16)-0.0078125f, (_Float16)-0.0078125f};
  const uint32_t even = word & 0x0F0F0F0Fu, odd = word & 0xF0F0F0F0u;
  half2_t q[4];
  const uint32_t pair[4] = {__builtin_amdgcn_perm(odd, even, 0x0c040c00u),
                            __builtin_amdgcn_perm(odd, even, 0x0c050c01u),
                            __builtin_amdgcn_perm(odd, even, 0x0c060c02u),
                            __builtin_amdgcn_perm(odd, even, 0x0c070c03u)};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    q[i] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, pair[i]), factor, offset);
  return half8_t{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
}

// ------------------------------------------------------------------- memory -> LDS, counted waits
//
// The loads below do not pass through registers and the compiler does not see them; the waits are
// counted by hand (vector memory operations of a wave complete in order).  Nothing else of the K
// loop loads from memory through the compiler.

// silu(gate) * up with the roundings of the decode row's epilogue
__device__ inline float silu_times(float gate, float up) {
  const float t = __builtin_amdgcn_exp2f(-fabsf(gate) * 1.4426950408889634f);
  const float r = __builtin_amdgcn_rcpf(1.0f + t);
  const float sig = gate < 0.f ? t * r : r;
  return __fmul_rn(__fmul_rn(gate, sig), up);
}

// Columns (col, col + 1) of output row `row`, summed: bias, then what the call asked for.
template <typename T>
__device__ inline void finish_pair(float v0, float v1, uint32_t row, uint32_t col, uint32_t m,
                                   uint32_t n, const T* __restrict__ bias, T* __restrict__ out,
                                   const RowsFusion& fuse) {
  const T* residual = static_cast<const T*>(fuse.residual);
  const bool two = col + 1 < n;
  if (bias) {
    v0 += to_f32<T>(bias[col]);
    if (two) v1 += to_f32<T>(bias[col + 1]);
  }
  if (fuse.mode == 1) {
    float value = silu_times(v0, v1);
    const size_t at = (size_t)row * (n >> 1) + (col >> 1);
    if (residual) value += to_f32<T>(residual[at]);
    out[at] = from_f32<T>(value);
  } else if (fuse.mode == 2) {
    // what a separate linear would have stored, then the rotation of krm_rope_half
    const float x0 = to_f32<T>(from_f32<T>(v0)), x1 = to_f32<T>(from_f32<T>(v1));
    const uint32_t half = fuse.depth >> 1, pair = col >> 1;
    const uint32_t rope_pairs = (fuse.heads + fuse.kv_heads) * half;
    if (pair < rope_pairs) {
      const uint32_t head = pair / half, j = pair - head * half;
      const int32_t pos = fuse.positions[row];
      float o0 = NAN, o1 = NAN;  // a position outside the table is never a valid rotation
      if (pos >= 0 && (uint32_t)pos < fuse.table_rows) {
        const size_t t = (size_t)pos * fuse.depth + j;
        o0 = __fadd_rn(__fmul_rn(x0, fuse.cos_table[t]), __fmul_rn(-x1, fuse.sin_table[t]));
        o1 = __fadd_rn(__fmul_rn(x1, fuse.cos_table[t + half]),
                       __fmul_rn(x0, fuse.sin_table[t + half]));
      }
      T* dst = head < fuse.heads
                   ? static_cast<T*>(fuse.q_out) + ((size_t)head * m + row) * fuse.depth
                   : static_cast<T*>(fuse.k_out) + ((size_t)(head - fuse.heads) * m + row) * fuse.depth;
      dst[j] = from_f32<T>(o0);
      dst[j + half] = from_f32<T>(o1);
    } else {
      const uint32_t e = (pair - rope_pairs) * 2u;  // the v section keeps its natural order
      const uint32_t plane = e / fuse.depth, d = e - plane * fuse.depth;
      T* dst = static_cast<T*>(fuse.v_out) + ((size_t)plane * m + row) * fuse.depth;
      dst[d] = from_f32<T>(x0);
      dst[d + 1] = from_f32<T>(x1);
    }
  } else {
    const size_t at = (size_t)row * n + col;
    if (residual) {
      v0 += to_f32<T>(residual[at]);
      if (two) v1 += to_f32<T>(residual[at + 1]);
    }
    out[at] = from_f32<T>(v0);
    if (two) out[at + 1] = from_f32<T>(v1);
  }
}

// Four elements next to each other, as wide as they are aligned (`quads_aligned` below), as they lie in
// memory (fp16: the first eight bytes).  They become numbers where they are used: a conversion waits for its
// load, and so for everything that was asked for in front of it.
template <typename T>
__device__ inline void load_quad(uint4& to, const T* p) {
  if constexpr (sizeof(T) == 4) {
    to = *reinterpret_cast<const uint4*>(p);
  } else {
    const uint2 raw = *reinterpret_cast<const uint2*>(p);
    to.x = raw.x; to.y = raw.y;
  }
}
template <typename T>
__device__ inline float4 quad_f32(const uint4& raw) {
  if constexpr (sizeof(T) == 4) {
    return make_float4(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z),
                       __uint_as_float(raw.w));
  } else {
    const half2_t a = __builtin_bit_cast(half2_t, raw.x), b = __builtin_bit_cast(half2_t, raw.y);
    return make_float4((float)a.x, (float)a.y, (float)b.x, (float)b.y);
  }
}
// Two elements at any element's alignment likewise.
template <typename T>
__device__ inline void load_pair(uint4& to, const T* p) {
  __builtin_memcpy(&to, p, 2 * sizeof(T));
}
template <typename T>
__device__ inline void store_pair(T* p, float v0, float v1) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float2*>(p) = make_float2(v0, v1);
  } else {
    *reinterpret_cast<uint32_t*>(p) =
        __builtin_bit_cast(uint32_t, half2_t{(_Float16)v0, (_Float16)v1});
  }
}
template <typename T>
__device__ inline void store_quad(T* p, float v0, float v1, float v2, float v3) {
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v0, v1, v2, v3);
  } else {
    *reinterpret_cast<uint2*>(p) =
        make_uint2(__builtin_bit_cast(uint32_t, half2_t{(_Float16)v0, (_Float16)v1}),
                   __builtin_bit_cast(uint32_t, half2_t{(_Float16)v2, (_Float16)v3}));
  }
}
// Columns col .. col + 3 (a multiple of 4, all below n) of a row at once: what the end of the
// product reads from memory, asked for while the sums are still on their way through LDS, and the
// same arithmetic as finish_pair behind them.
struct QuadAhead {
  uint4 bias, residual;   // (load_quad; a silu's residual: load_pair)
  float2 cos[2], sin[2];  // mode 2: of dims j, j + 1 and of j + D/2, j + 1 + D/2
};
template <typename T>
__device__ inline void fetch_quad(QuadAhead& q, uint32_t row, uint32_t col, uint32_t n, int32_t pos,
                                  const T* bias, const RowsFusion& fuse) {
  if (bias) load_quad<T>(q.bias, bias + col);
  const T* residual = static_cast<const T*>(fuse.residual);
  if (fuse.mode == 2) {
    const uint32_t half = fuse.depth >> 1, pair = col >> 1;
    if (pair < (fuse.heads + fuse.kv_heads) * half && pos >= 0 && (uint32_t)pos < fuse.table_rows) {
      const size_t t = (size_t)pos * fuse.depth + pair % half;
      q.cos[0] = *reinterpret_cast<const float2*>(fuse.cos_table + t);
      q.sin[0] = *reinterpret_cast<const float2*>(fuse.sin_table + t);
      q.cos[1] = *reinterpret_cast<const float2*>(fuse.cos_table + t + half);
      q.sin[1] = *reinterpret_cast<const float2*>(fuse.sin_table + t + half);
    }
  } else if (residual && fuse.mode == 0) {
    load_quad<T>(q.residual, residual + (size_t)row * n + col);
  } else if (residual) {
    load_pair<T>(q.residual, residual + (size_t)row * (n >> 1) + (col >> 1));
  }
}
template <typename T>
__device__ inline void finish_quad(float4 v, const QuadAhead& q, uint32_t row, uint32_t col,
                                   uint32_t m, uint32_t n, int32_t pos, bool bias, T* out,
                                   const RowsFusion& fuse) {
  if (bias) {
    const float4 b = quad_f32<T>(q.bias);
    v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
  }
  if (fuse.mode == 0) {
    if (fuse.residual) {
      const float4 r = quad_f32<T>(q.residual);
      v.x += r.x; v.y += r.y; v.z += r.z; v.w += r.w;
    }
    store_quad<T>(out + (size_t)row * n + col, v.x, v.y, v.z, v.w);
  } else if (fuse.mode == 1) {
    float a = silu_times(v.x, v.y), b = silu_times(v.z, v.w);
    if (fuse.residual) {
      const float4 r = quad_f32<T>(q.residual);
      a += r.x; b += r.y;
    }
    store_pair<T>(out + (size_t)row * (n >> 1) + (col >> 1), a, b);
  } else {
    // what a separate linear would have stored, then the rotation
    auto stored = [](float x) { return to_f32<T>(from_f32<T>(x)); };
    const float x[2][2] = {{stored(v.x), stored(v.y)}, {stored(v.z), stored(v.w)}};
    const uint32_t half = fuse.depth >> 1, pair = col >> 1;
    const uint32_t rope_pairs = (fuse.heads + fuse.kv_heads) * half;
    if (pair < rope_pairs) {
      const uint32_t head = pair / half, j = pair - head * half;
      float lo[2] = {NAN, NAN}, hi[2] = {NAN, NAN};  // outside the table: never a valid rotation
      if (pos >= 0 && (uint32_t)pos < fuse.table_rows) {
        const float c0[2] = {q.cos[0].x, q.cos[0].y}, s0[2] = {q.sin[0].x, q.sin[0].y};
        const float c1[2] = {q.cos[1].x, q.cos[1].y}, s1[2] = {q.sin[1].x, q.sin[1].y};
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          lo[i] = __fadd_rn(__fmul_rn(x[i][0], c0[i]), __fmul_rn(-x[i][1], s0[i]));
          hi[i] = __fadd_rn(__fmul_rn(x[i][1], c1[i]), __fmul_rn(x[i][0], s1[i]));
        }
      }
      T* dst = head < fuse.heads
                   ? static_cast<T*>(fuse.q_out) + ((size_t)head * m + row) * fuse.depth
                   : static_cast<T*>(fuse.k_out) + ((size_t)(head - fuse.heads) * m + row) * fuse.depth;
      store_pair<T>(dst + j, lo[0], lo[1]);
      store_pair<T>(dst + j + half, hi[0], hi[1]);
    } else {
      const uint32_t e = (pair - rope_pairs) * 2u;
      const uint32_t plane = e / fuse.depth, d = e - plane * fuse.depth;
      store_quad<T>(static_cast<T*>(fuse.v_out) + ((size_t)plane * m + row) * fuse.depth + d, x[0][0],
                    x[0][1], x[1][0], x[1][1]);
    }
  }
}
// Whether quads of columns may be read and written at once: n in whole quads, rows and buffers
// aligned to them (a rope table to the pairs it is read in).
inline bool quads_aligned(const void* bias, const void* out, uint32_t n, size_t eb,
                          const RowsFusion& fuse) {
  auto at = [](const void* p, size_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; };
  if (n % 4 != 0 || !at(bias, 4 * eb)) return false;
  if (fuse.mode == 2)
    return fuse.depth % 4 == 0 && at(fuse.cos_table, 8) && at(fuse.sin_table, 8) &&
           at(fuse.q_out, 2 * eb) && at(fuse.k_out, 2 * eb) && at(fuse.v_out, 4 * eb);
  return fuse.mode == 0 ? at(out, 4 * eb) && at(fuse.residual, 4 * eb) : at(out, 2 * eb);
}

template <typename T>
struct type_tag { using type = T; };

struct SliceTail {         // what the end of the kernel needs
  const void* bias;
  void* out;
  const float* row_scale;  // kXSplit
  uint32_t quads;          // quads_aligned
  RowsFusion fuse;
};

// ------------------------------------------------------------------------------- x = hi + lo
//
// Row r of the split form: for every 32 codes, 64 bytes of hi and 64 bytes of lo (one line), eight
// codes at a time in the order (x0,x4,x1,x5,x2,x6,x3,x7); scale[2r] = 2^e with max|x[r, :]| * 2^e in [2^13, 2^14) (no
// overflow, small entries keep a resolution of 2^-38 of the row's maximum), scale[2r + 1] = 2^-e.
// A row of zeros, or whose maximum is not finite, gets 1 / 1: what is not finite stays so.
// One trip over memory up to 16384 codes a row (kept in registers between the maximum and the
// split), two beyond.  A row takes `padded` codes in the planes, zeros past k.
template <uint32_t kThreads, uint32_t kHeld>
__global__ __launch_bounds__(kThreads) void split_rows_kernel(const float* __restrict__ x,
                                                         uint4* __restrict__ planes,
                                                         float* __restrict__ scale, uint32_t k,
                                                         uint32_t padded) {
  __shared__ uint32_t s_max[kThreads / kWave];
  const uint4* row = reinterpret_cast<const uint4*>(x + (size_t)blockIdx.x * k);
  const uint32_t pieces = k >> 3;
  uint4 a[kHeld], b[kHeld];
#pragma unroll
  for (uint32_t i = 0; i < kHeld; ++i) {
    const uint32_t p = threadIdx.x + kThreads * i;
    const uint32_t at = p < pieces ? p : 0u;
    a[i] = row[2 * at];
    b[i] = row[2 * at + 1];
  }
  auto larger = [](uint32_t top, const uint4& v) {
    return max(max(top, v.x & 0x7fffffffu),
               max(v.y & 0x7fffffffu, max(v.z & 0x7fffffffu, v.w & 0x7fffffffu)));
  };
  uint32_t top = 0;  // largest |x| as raw bits (monotonic for non-negative floats; NaN on top)
#pragma unroll
  for (uint32_t i = 0; i < kHeld; ++i) top = larger(larger(top, a[i]), b[i]);
  for (uint32_t p = threadIdx.x + kThreads * kHeld; p < pieces; p += kThreads)
    top = larger(larger(top, row[2 * p]), row[2 * p + 1]);
  for (int off = 32; off > 0; off >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, off, kWave));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = top;
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < kThreads / kWave; ++i) top = max(top, s_max[i]);
  const uint32_t biased = top >> 23;  // exponent of the maximum
  uint32_t up = 127u, down = 127u;    // 2^0
  if (top != 0 && biased != 255u) {
    // e = 13 - (biased - 127), kept inside the normal range of both 2^e and 2^-e
    int e = 13 - ((int)biased - 127);
    e = e > 126 ? 126 : (e < -126 ? -126 : e);
    up = (uint32_t)(127 + e);
    down = (uint32_t)(127 - e);
  }
  const float factor = __uint_as_float(up << 23);
  if (threadIdx.x == 0) {
    scale[2 * (size_t)blockIdx.x] = factor;
    scale[2 * (size_t)blockIdx.x + 1] = __uint_as_float(down << 23);
  }
  uint4* dst = planes + (size_t)blockIdx.x * (padded >> 2);
  auto split = [&](uint32_t p, const uint4& va, const uint4& vb) {
    const uint32_t raw[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    _Float16 h[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float xs = __uint_as_float(raw[i]) * factor;  // exact: a power of two
      h[i] = (_Float16)xs;                                // round to nearest even
      l[i] = (_Float16)(xs - (float)h[i]);                // the difference is exact in f32
    }
    auto pack = [](_Float16 p0, _Float16 p1) {
      const half2_t t = {p0, p1};
      return __builtin_bit_cast(uint32_t, t);
    };
    const uint32_t at = (p >> 2) * 8u + (p & 3u);
    dst[at] = make_uint4(pack(h[0], h[4]), pack(h[1], h[5]), pack(h[2], h[6]), pack(h[3], h[7]));
    dst[at + 4] =
        make_uint4(pack(l[0], l[4]), pack(l[1], l[5]), pack(l[2], l[6]), pack(l[3], l[7]));
  };
#pragma unroll
  for (uint32_t i = 0; i < kHeld; ++i) {
    const uint32_t p = threadIdx.x + kThreads * i;
    if (p < pieces) split(p, a[i], b[i]);
  }
  for (uint32_t p = threadIdx.x + kThreads * kHeld; p < pieces; p += kThreads)
    split(p, row[2 * p], row[2 * p + 1]);
  for (uint32_t p = pieces + threadIdx.x; p < padded >> 3; p += kThreads) {
    const uint32_t at = (p >> 2) * 8u + (p & 3u);
    dst[at] = dst[at + 4] = make_uint4(0u, 0u, 0u, 0u);
  }
}
// Threads and pieces a thread: as many as the row has (512 and four for every row, most of them spare copies of the first
// piece, took 0.4 us more: 67 x 673 x 1024 7.83 / 7.45 us, 128 x 2560 x 2048 11.4 / 11.0, 319 x 715 x 3840 18.0 / 17.3).
inline void launch_split_rows(krm_ctx* ctx, const float* x, uint4* planes, float* scale, uint32_t rows, uint32_t k,
                              uint32_t padded) {
  if (k <= 2048)
    split_rows_kernel<256, 1><<<dim3(rows), dim3(256), 0, ctx->stream>>>(x, planes, scale, k, padded);
  else if (k <= 4096)
    split_rows_kernel<512, 1><<<dim3(rows), dim3(512), 0, ctx->stream>>>(x, planes, scale, k, padded);
  else if (k <= 8192)
    split_rows_kernel<512, 2><<<dim3(rows), dim3(512), 0, ctx->stream>>>(x, planes, scale, k, padded);
  else
    split_rows_kernel<512, 4><<<dim3(rows), dim3(512), 0, ctx->stream>>>(x, planes, scale, k, padded);
}

}  // namespace
}  // namespace krm
