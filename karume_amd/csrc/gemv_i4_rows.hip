// int4 `linear` of 2 to 16 rows of x with the bits of each row alone: the additions of gemv_i4_kernel
// (linear_i4.hip), dealt in another way.
//
// A row's sum there is that of 64 lanes: lane l adds the segments l, l + 64, ... of 32 codes, each a chain of
// products in a fixed order times its scale, and the lanes' sums are added by a fixed tree.  What those
// bits leave open is which thread forms which segment.  There a wave meets 1 to 4 rows of W and reads all of x
// for them; here a lane has a row of W, a wave 64 of them (or 16, four segments' groups each), and x is the operand that the
// lanes share: a code is converted once for all rows of x, and no lane idles where K is no multiple of 2048.
//
// What bounds it: the vector ALU (a chain's products one by one, 4.8 clk for 64).  us in the one-row kernel / here: 16 f32 rows 16901 x 2304 170 / 45 (of which products
// 19), 8 rows 23296 x 1920 86 / 23, 13 rows 1150 x 10880 72 / 17, 5 rows 3820 x 2048 13.1 / 5.8; 12 fp16 rows 29384 x 4608
// in groups of 32 164 / 66, 9 rows 1173 x 2432 15.5 / 5.7; over 50 shapes 1.0 to 4.2 times, 2.3 in the mean.
#include "gemv_i4_rows_plan.h"
#include "i4_codes.h"
#include "lds_stream.h"

using namespace krm;

static_assert(kRowsWave == kWave, "the plan counts lanes");

namespace {

// SPAN quads of 64 / SPAN rows of W a stage, and R rows of x.
template <typename XT, int SPAN, int R>
struct Stage {
  static constexpr uint32_t kW = kWave * 64, kXRow = kQuad * kSegment * sizeof(XT), kX = R * SPAN * kXRow;
  static constexpr uint32_t kXLoads = (kX + 1023) / 1024, kBytes = kW + kXLoads * 1024;
};

// A chunk of 16 lanes x 16 bytes of x, the same in every 16 lanes: lane i of them holds elements 4 i .. 4 i + 3 (f32: two
// segments) or 8 i .. 8 i + 7 (fp16: four).  A lane's products take their element from there by a row broadcast, which
// costs nothing beside the product (v_fmac_f32 4.8 clk a wave with one, 4.7 with a scalar operand).  s_nop: a DPP
// operand written by the vector ALU needs two states between, a dot product's result three before another
// kind of instruction reads it.
template <typename XT>
struct Chains;

template <>
struct Chains<float> {
  static constexpr int kSegments = 2;
  typedef float Weights[kSegments][4][8];
  struct X { float v[4]; };
  __device__ static inline void weights(uint32_t word, float (&w)[8]) {
    // bytes of u - 8 in two's complement: 0x78 + u, top bit flipped
    const uint32_t low = ((word & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
    const uint32_t high = (((word >> 4) & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[2 * i] = (float)(int8_t)(low >> (8 * i));
      w[2 * i + 1] = (float)(int8_t)(high >> (8 * i));
    }
  }
  __device__ static inline X load(const void* p) {
    const float4 a = *static_cast<const float4*>(p);
    return X{{a.x, a.y, a.z, a.w}};
  }
  // (The first product of a chain is v_mul: an addition to +0 differs from it in the sign of zero alone, which the
  // addition to the lane's sum drops.)
  template <int J>
  __device__ static inline void word(float (&acc)[kSegments], const X& x, const Weights& w) {
#define KRM_PRODUCT(OP, ACC, X, W, LANE) OP "_dpp %" #ACC ", %" #X ", %" #W " row_newbcast:%" #LANE " row_mask:0xf bank_mask:0xf\n"
#define KRM_FMAC(ACC, X, W, LANE) KRM_PRODUCT("v_fmac_f32", ACC, X, W, LANE)
#define KRM_PAIR(X, W0, W4, V0, V4) KRM_FMAC(0, X, W0, 22) KRM_FMAC(1, X, V0, 24) KRM_FMAC(0, X, W4, 23) KRM_FMAC(1, X, V4, 25)
#define KRM_FIRST(X, W0, W4, V0, V4)                                                                    \
  KRM_PRODUCT("v_mul_f32", 0, X, W0, 22) KRM_PRODUCT("v_mul_f32", 1, X, V0, 24) KRM_FMAC(0, X, W4, 23) \
  KRM_FMAC(1, X, V4, 25)
#define KRM_OPERANDS                                                                                                  \
  "v"(x.v[0]), "v"(x.v[1]), "v"(x.v[2]), "v"(x.v[3]), "v"(w[0][J][0]), "v"(w[0][J][1]), "v"(w[0][J][2]),           \
      "v"(w[0][J][3]), "v"(w[0][J][4]), "v"(w[0][J][5]), "v"(w[0][J][6]), "v"(w[0][J][7]), "v"(w[1][J][0]),           \
      "v"(w[1][J][1]), "v"(w[1][J][2]), "v"(w[1][J][3]), "v"(w[1][J][4]), "v"(w[1][J][5]), "v"(w[1][J][6]),           \
      "v"(w[1][J][7]), "n"(2 * J), "n"(2 * J + 1), "n"(2 * J + 8), "n"(2 * J + 9)
    if constexpr (J == 0)
      asm("s_nop 1\n" KRM_FIRST(2, 6, 10, 14, 18) KRM_PAIR(3, 7, 11, 15, 19) KRM_PAIR(4, 8, 12, 16, 20)
              KRM_PAIR(5, 9, 13, 17, 21)
          : "=&v"(acc[0]), "=&v"(acc[1])
          : KRM_OPERANDS);
    else
      asm("s_nop 1\n" KRM_PAIR(2, 6, 10, 14, 18) KRM_PAIR(3, 7, 11, 15, 19) KRM_PAIR(4, 8, 12, 16, 20)
              KRM_PAIR(5, 9, 13, 17, 21)
          : "+v"(acc[0]), "+v"(acc[1])
          : KRM_OPERANDS);
#undef KRM_OPERANDS
#undef KRM_FIRST
#undef KRM_PAIR
#undef KRM_FMAC
#undef KRM_PRODUCT
  }
  __device__ static inline float finish(float acc) { return acc; }
};

template <>
struct Chains<__half> {
  static constexpr int kSegments = 4;
  typedef half2_t Weights[kSegments][4][4];
  struct X { half2_t v[4]; };  // pairs (i, i + 4)
  __device__ static inline void weights(uint32_t word, half2_t (&w)[4]) { codes_over_1024(word, w); }
  __device__ static inline X load(const void* p) {
    X x;
    pair_activations(*static_cast<const uint4*>(p), x.v);
    return x;
  }
  template <int J>
  __device__ static inline void word(float (&acc)[kSegments], const X& x, const Weights& w) {
    if constexpr (J == 0) acc[0] = acc[1] = acc[2] = acc[3] = 0.f;
#define KRM_DOT(ACC, X, W, LANE) "v_dot2c_f32_f16_dpp %" #ACC ", %" #X ", %" #W " row_newbcast:%" #LANE " row_mask:0xf bank_mask:0xf\n"
#define KRM_FOUR(X, W0, W1, W2, W3) KRM_DOT(0, X, W0, 24) KRM_DOT(1, X, W1, 25) KRM_DOT(2, X, W2, 26) KRM_DOT(3, X, W3, 27)
    asm("s_nop 1\n" KRM_FOUR(4, 8, 12, 16, 20) KRM_FOUR(5, 9, 13, 17, 21) KRM_FOUR(6, 10, 14, 18, 22)
            KRM_FOUR(7, 11, 15, 19, 23) "s_nop 2\n"
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
        : "v"(x.v[0]), "v"(x.v[1]), "v"(x.v[2]), "v"(x.v[3]), "v"(w[0][J][0]), "v"(w[0][J][1]), "v"(w[0][J][2]),
          "v"(w[0][J][3]), "v"(w[1][J][0]), "v"(w[1][J][1]), "v"(w[1][J][2]), "v"(w[1][J][3]), "v"(w[2][J][0]),
          "v"(w[2][J][1]), "v"(w[2][J][2]), "v"(w[2][J][3]), "v"(w[3][J][0]), "v"(w[3][J][1]), "v"(w[3][J][2]),
          "v"(w[3][J][3]), "n"(J), "n"(J + 4), "n"(J + 8), "n"(J + 12));
#undef KRM_FOUR
#undef KRM_DOT
  }
  __device__ static inline float finish(float acc) { return acc * 1024.0f; }  // exact
};

// A workgroup has 64 / SPAN rows of W and up to R of x; its waves share the sixteen quads of four neighbouring lanes
// of the one-row kernel: SPAN positions a wave at a time, `deal` (4, 2 or 1; 1 where SPAN is more) times.
// Sixteen lanes have one quad.  A wave walks its quads by stages of its own, the next one on its way to LDS (W, x and
// scales) while this one is used, without a barrier until the sums of the waves meet.
template <typename XT, typename ST, int SPAN, int R>
__global__ __launch_bounds__(kMaxUnits * 64) void gemv_i4_rows_kernel(
    const XT* __restrict__ x, const uint32_t* __restrict__ w, const ST* __restrict__ scales, const XT* __restrict__ bias,
    XT* __restrict__ out, uint32_t m, uint32_t n, uint32_t k, uint32_t group_shift, uint32_t row_blocks, uint32_t deal,
    uint32_t scale_area, uint32_t whole_scales) {
  using C = Chains<XT>;
  using S = Stage<XT, SPAN, R>;
  constexpr uint32_t kTile = kWave / SPAN, kPieces = 4 * SPAN;  // rows of W, 16-byte pieces of one a stage
  extern __shared__ __align__(1024) uint8_t s_stages[];
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The blocks of rows of one tile follow each other on one XCD: its L2 has the weights for all of them.
  const uint32_t slot = blockIdx.x >> 3;
  const uint32_t block = slot % row_blocks, n0 = ((slot / row_blocks) * 8 + (blockIdx.x & 7)) * kTile;
  if (n0 >= n) return;
  const uint32_t row0 = block * R, last_x = min((uint32_t)R, m - row0) - 1;  // rows past M are the last one
  const uint32_t segments = k / kSegment, groups = k >> group_shift;

  const uint32_t position0 = wave * deal * SPAN;
  uint8_t* const ring = s_stages + scale_area + wave * 2 * S::kBytes;
  auto lds_address = [](const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
  };
  const uint32_t ring_lds = lds_address(ring);

  const uint8_t* const w_tile = reinterpret_cast<const uint8_t*>(w) + (size_t)n0 * (k / 2);
  const ST* const s_tile = scales + (size_t)n0 * groups;
  const XT* const x_block = x + (size_t)row0 * k;
  const uint32_t last_row = min(kTile, n - n0) - 1;  // rows past N are the last one, and not stored
  const uint32_t own_row = lane % kTile, own_sub = lane / kTile;  // of W, of the SPAN quads
  // Piece p of row r is at slot p ^ f(r): sixteen lanes' 16-byte reads then meet different banks.
  auto fold = [](uint32_t row) { return (row / (4 / SPAN)) & (kPieces - 1); };
  constexpr uint32_t kLoadWRows = kWave / kPieces;
  uint32_t w_row[4], w_piece[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t row = kLoadWRows * i + lane / kPieces;
    w_row[i] = min(row, last_row) * (k / 2);
    w_piece[i] = (lane % kPieces) ^ fold(row);
  }
  const uint32_t own_scales = min(own_row, last_row) * groups;
  constexpr uint32_t kXRowLanes = S::kXRow / 16;  // lanes a quad of a row of x: 32 or 16
  constexpr uint32_t kLoadX = kWave / kXRowLanes;

  // segment of quad `sub` of the positions from `position` on
  auto segment_of = [](uint32_t step, uint32_t position, uint32_t sub) {
    return step * 64 + quad_at(position + sub) * kQuad;
  };
  auto request = [&](uint32_t position, uint32_t step, uint32_t buf) {
    const uint32_t lds = ring_lds + buf * S::kBytes;
    // segments past K: the last one, not used
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t at = min(segment_of(step, position, w_piece[i] / 4) + w_piece[i] % 4, segments - 1);
      stream_to_lds(lds + 1024u * i, w_row[i] + at * 16, w_tile);
    }
#pragma unroll
    for (uint32_t i = 0; i < S::kXLoads; ++i) {
      const uint32_t index = kLoadX * i + lane / kXRowLanes;
      const uint32_t at = segment_of(step, position, index % SPAN) * kSegment * (uint32_t)sizeof(XT) + lane % kXRowLanes * 16;
      stream_to_lds(lds + S::kW + 1024u * i,
                    min(index / SPAN, last_x) * k * (uint32_t)sizeof(XT) + min(at, k * (uint32_t)sizeof(XT) - 16), x_block);
    }
  };

  float hold[R], value[R];
#pragma unroll
  for (uint32_t r = 0; r < R; ++r) hold[r] = value[r] = 0.f;
  if (segment_of(0, position0, 0) < segments) request(position0, 0, 0);  // (the first quad of SPAN is the lowest)
  // The tile's scales stand together in memory and are brought to LDS once (where they fit: scale_area).  A load costs by
  // the lines it touches, 64 for a scale of each of 64 rows, up to four such loads a stage beside 96 lines of W and x:
  // 16 rows 16901 x 2304 in groups of 32 49.0 us so, 44.8 from LDS.
  if (scale_area) {
    const uint32_t count = (last_row + 1) * groups, whole = whole_scales ? count * (uint32_t)sizeof(ST) & ~15u : 0u;
    for (uint32_t at = wave * 1024; at < whole; at += blockDim.x * 16)  // (what lies past the last piece repeats it)
      stream_to_lds(lds_address(s_stages) + at, min(at + lane * 16, whole - 16), s_tile);
    wait_vm<0>();
    __syncthreads();  // (the repeated pieces)
    for (uint32_t i = whole / (uint32_t)sizeof(ST) + threadIdx.x; i < count; i += blockDim.x)
      reinterpret_cast<ST*>(s_stages)[i] = s_tile[i];
    __syncthreads();
  }
  uint32_t buf = 0;
  for (uint32_t t = 0; t < deal; ++t) {
    const uint32_t position = position0 + t * SPAN;
    float sums[R][kQuad];
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
#pragma unroll
      for (uint32_t j = 0; j < kQuad; ++j) sums[r][j] = 0.f;
    for (uint32_t step = 0; segment_of(step, position, 0) < segments; ++step) {
      const uint32_t own = segment_of(step, position, own_sub);
      wait_streamed_and_read();  // (the other half of the ring, which is filled next, was read a stage ago)
      if (segment_of(step + 1, position, 0) < segments) {
        request(position, step + 1, buf ^ 1u);
      } else {
        for (uint32_t u = t + 1; u < deal; ++u)  // the next quad that has a segment
          if (segment_of(0, position0 + u * SPAN, 0) < segments) {
            request(position0 + u * SPAN, 0, buf ^ 1u);
            break;
          }
      }
      const uint8_t* const stage = ring + buf * S::kBytes;
      float scale[kQuad];
#pragma unroll
      for (uint32_t j = 0; j < kQuad; ++j) {
        const uint32_t at = own_scales + (min(own + j, segments - 1) >> (group_shift - 5));
        scale[j] = to_f32<ST>(scale_area ? reinterpret_cast<const ST*>(s_stages)[at] : s_tile[at]);
      }
#pragma unroll
      for (uint32_t pass = 0; pass < kQuad / C::kSegments; ++pass) {
        typename C::Weights codes;
#pragma unroll
        for (uint32_t j = 0; j < C::kSegments; ++j) {
          const uint32_t piece = own_sub * 4 + pass * C::kSegments + j;
          const uint4 v = *reinterpret_cast<const uint4*>(stage + own_row * (16 * kPieces) + (piece ^ fold(own_row)) * 16);
          C::weights(v.x, codes[j][0]);
          C::weights(v.y, codes[j][1]);
          C::weights(v.z, codes[j][2]);
          C::weights(v.w, codes[j][3]);
        }
        const uint8_t* const x_pass = stage + S::kW + own_sub * S::kXRow + pass * 256 + (lane & 15) * 16;
        typename C::X ahead = C::load(x_pass);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r) {
          const typename C::X x_row = ahead;
          if (r + 1 < R) ahead = C::load(x_pass + (r + 1) * SPAN * S::kXRow);
          float acc[C::kSegments];
          C::template word<0>(acc, x_row, codes);
          C::template word<1>(acc, x_row, codes);
          C::template word<2>(acc, x_row, codes);
          C::template word<3>(acc, x_row, codes);
#pragma unroll
          for (uint32_t j = 0; j < C::kSegments; ++j) {
            const uint32_t piece = pass * C::kSegments + j;
            const uint32_t keep = own + piece < segments ? 0xFFFFFFFFu : 0u;
            sums[r][piece] += __uint_as_float(__float_as_uint(C::finish(acc[j]) * scale[piece]) & keep);
          }
        }
      }
      buf ^= 1u;
    }
    // the quad's sum, and the tree over a wave's quads
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
      const float quad_sum = (sums[r][0] + sums[r][1]) + (sums[r][2] + sums[r][3]);
      if (t & 1u) value[r] = t == 1 ? hold[r] + quad_sum : value[r] + (hold[r] + quad_sum);
      else hold[r] = quad_sum;
    }
  }

  // [wave][row][lane] in the wave's own ring, which nothing writes any more
  constexpr uint32_t kUnitFloats = 2 * S::kBytes / 4;
  const float* const s_sums = reinterpret_cast<const float*>(s_stages + scale_area);
  float* const mine = reinterpret_cast<float*>(ring);
#pragma unroll
  for (uint32_t r = 0; r < R; ++r)
    mine[r * kWave + lane] = deal == 1 ? hold[r] : value[r];
  __syncthreads();
  const uint32_t parts = (blockDim.x >> 6) * SPAN;
  for (uint32_t i = threadIdx.x; i < (last_x + 1) * kTile; i += blockDim.x) {
    const uint32_t r = i / kTile, c = i % kTile;
    if (n0 + c >= n) continue;
    float sixteen[4];  // sums of sixteen lanes of the one-row kernel each; a part past the last one is zero
    auto part = [&](uint32_t p) {
      return p < parts ? s_sums[p / SPAN * kUnitFloats + r * kWave + p % SPAN * kTile + c] : 0.f;
    };
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
      sixteen[j] = deal == 4   ? part(j)
                   : deal == 2 ? part(2 * j) + part(2 * j + 1)
                               : (part(4 * j) + part(4 * j + 1)) + (part(4 * j + 2) + part(4 * j + 3));
    const float total = (sixteen[0] + sixteen[1]) + (sixteen[2] + sixteen[3]);
    out[(size_t)(row0 + r) * n + n0 + c] = from_f32<XT>(total + (bias ? to_f32<XT>(bias[n0 + c]) : 0.f));
  }
}

template <typename XT, typename ST>
int32_t launch_rows(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out, uint32_t m, uint32_t n,
                    uint32_t k, uint32_t group) {
  uint32_t group_shift = 0;
  while ((1u << group_shift) < group) ++group_shift;
  const RowsPlan p = plan_rows(sizeof(XT), sizeof(ST), (uint32_t)ctx->num_cus, m, n, k, group_shift);
  const uint32_t tiles = p.blocks / p.row_blocks;
#define KRM_ROWS(SPAN, R)                                                                                               \
  if (p.span == SPAN && p.rows == R) {                                                                                \
    gemv_i4_rows_kernel<XT, ST, SPAN, R>                                                                              \
        <<<dim3((tiles + 7) / 8 * 8 * p.row_blocks), dim3(p.units * 64), p.lds, ctx->stream>>>(                       \
            ptr<const XT>(x), ptr<const uint32_t>(w), ptr<const ST>(scales), ptr<const XT>(bias), ptr<XT>(out), m, n, \
            k, group_shift, p.row_blocks, p.deal, p.scale_area, aligned(scales, 16) ? 1u : 0u);                       \
    return launched(ctx, "gemv_i4_rows_kernel");                                                                      \
  }
  KRM_ROWS(1, 2) KRM_ROWS(1, 3) KRM_ROWS(1, 4) KRM_ROWS(1, 5) KRM_ROWS(1, 6) KRM_ROWS(1, 8)
  KRM_ROWS(4, 1) KRM_ROWS(4, 2) KRM_ROWS(4, 3) KRM_ROWS(4, 4) KRM_ROWS(4, 5)
#undef KRM_ROWS
  return fail(ctx, KRM_ERR_VALIDATION, "rows: no form of %u x %u", p.span, p.rows);
}

}  // namespace

namespace krm {

int32_t linear_i4_gemv_rows(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias, krm_buf out, uint32_t m,
                            uint32_t n, uint32_t k, uint32_t group, int32_t io_dtype, int32_t scale_dtype, bool* handled) {
  const bool f32 = io_dtype == KRM_F32;
  *handled = false;
  if (!rows_dealt(f32, m, n, k, group) || !aligned(w, 16)) return KRM_OK;
  *handled = true;
  if (f32)
    return scale_dtype == KRM_F16 ? launch_rows<float, __half>(ctx, x, w, scales, bias, out, m, n, k, group)
                                  : launch_rows<float, float>(ctx, x, w, scales, bias, out, m, n, k, group);
  return scale_dtype == KRM_F16 ? launch_rows<__half, __half>(ctx, x, w, scales, bias, out, m, n, k, group)
                                : launch_rows<__half, float>(ctx, x, w, scales, bias, out, m, n, k, group);
}

}  // namespace krm
