// int4 `linear` for a chunk of rows on the gfx950 matrix cores: eight waves split K.
//
// out[m, n] = sum_k x[m,k] * dequant(w)[n,k] + bias[n]
// (packages/runtime/src/kernels/linear.ts:34-64, packages/runtime/src/kernels/gemm.ts:1187-1237).
// The weights enter the matrix cores as the exact integers (u - 8) in fp16, products are exact,
// sums are f32 (v_mfma_f32_32x32x16_f16) and the group scale multiplies the f32 sum of each scale
// group.  Four forms of x:
//   kX16     fp16 activations as they are;
//   kX32     f32 activations, each rounded to fp16 once where it is read from LDS;
//   kXSplit  f32 activations as x * 2^e = hi + lo (both fp16, e per row), written once per call
//            by split_rows_kernel: two matrix instructions a step, 22 bits of x;
//   kXThree  f32 activations with all their bits, groups of 16 and 32: x = t1 + t2 + t3, each the
//            next 8 bits as a bf16, taken where x is read from LDS: three matrix instructions a
//            step, no scratch, no pass ahead and no exponent that a row's entries would share.
//
// A workgroup owns a tile of 32 MT rows x 32 NT columns; its eight waves take an eighth of K each
// and run on their own: a wave streams its slice of x and of the packed weights from memory
// straight into its own LDS rings (global_load_lds, no registers, no parking instructions), so
// the K loop has no barrier, every LDS byte is read once and every weight word is turned into
// integers once per 32 MT rows.  The waves' sums meet in LDS and are added in wave order.  How K
// is cut depends on K and the group size alone, and every tile size adds in the same order: a
// row's bits depend neither on M nor on the tile picked for the shape.
//
// LDS rings: x in stages of 64 or 32 codes, weights in units of 64 to 256 codes; the 16-byte pieces
// of a row are permuted by the row number, so that the fragment reads of 32 consecutive rows spread
// over all banks.
//
// What bounds it: what the second-level cache delivers to a CU (tiles of 64 x 96: 2 * 64 + 96 / 2
// bytes a code), then the conversion of the weights on the vector ALUs (10 operations a word, 9 beside hi + lo planes).
// Measured on cold weights, fp16 x (f32 class in brackets), against the kernel that loaded through
// registers, one 32 x 32 or 32 x 64 tile a workgroup: 128 x 2560 x 2048 6.6 us, 9.6 before (11.0,
// 14.5); 128 x 2048 x 2048 5.4, 7.0 (10.1, 12.5); 128 x 11264 x 2048 15.1, 27.0 (22.6, 38.6); 128 x
// 2048 x 5632 10.6, 13.0 (19.0, 26.2).
//
// kXThree is bounded by the vector ALUs (11 operations a pair of x, 10 a word of weights, both at
// every step; tiles of up to four columns share x).  Groups of 32, against the GEMV over blocks of 16
// rows (in brackets: hi + lo planes, which lost the small entries of a row beside a large one): 77 x
// 3000 x 2080 12.9 us, 210 (13.8); 17 rows of it 10.1, 45.5 (10.2); 128 x 2048 x 2048 11.2, 156 (12.0);
// 32 x 4096 x 8192 29, - (25); 512 x 4096 x 4096 77, 1969 (81); 512 x 11008 x 4096 215, 5594 (214); in
// groups of 16 277, 2427 (332).  Error against 64 bits (2-norm,
// normal x): 77 x 3000 x 2080 in groups of 32 9.5e-8, the GEMV 1.24e-7; 40 x 1000 x 4096 in groups of
// 16 1.04e-7 and 1.05e-7; 300 x 512 x 11008 in groups of 32 1.21e-7 and 1.33e-7.
#include "gemm_i4_rows.h"

#include <type_traits>

using namespace krm;

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kX16 = 0, kXSplit = 1, kX32 = 2, kXThree = 3;
constexpr int kWaves = 8;

// The high halves of two f32 as a pair of bf16.
__device__ inline uint32_t high_pair(uint32_t even, uint32_t odd) {
  return __builtin_amdgcn_perm(odd, even, 0x07060302u);
}
// 8 codes of a word -> 8 bf16 (u - 8) / 16, exact, natural order (a 4-bit integer with its sign is
// what v_cvt_off_f32_i4 takes; the sum over K is multiplied by 16 at the end).
__device__ inline half8_t sixteenths(uint32_t word) {
  const uint32_t even = word ^ 0x88888888u, odd = even >> 4;
  uint32_t v[8];  // (a byte of a register is an operand; the compiler shifts most of them down first)
#define KRM_SIXTEENTH(TO, FROM, BYTE)                                                          \
  asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #BYTE  \
      : "=v"(TO) : "v"(FROM))
  KRM_SIXTEENTH(v[0], even, 0); KRM_SIXTEENTH(v[1], odd, 0);
  KRM_SIXTEENTH(v[2], even, 1); KRM_SIXTEENTH(v[3], odd, 1);
  KRM_SIXTEENTH(v[4], even, 2); KRM_SIXTEENTH(v[5], odd, 2);
  KRM_SIXTEENTH(v[6], even, 3); KRM_SIXTEENTH(v[7], odd, 3);
#undef KRM_SIXTEENTH
  return __builtin_bit_cast(half8_t, make_uint4(high_pair(v[0], v[1]), high_pair(v[2], v[3]),
                                                high_pair(v[4], v[5]), high_pair(v[6], v[7])));
}
// 8 f32 -> three times 8 bf16 whose sum they are, every part the leading 8 bits of what is left.
// (Cut off, not rounded: the first part of the largest f32 stays finite.)  An infinity is its own
// first part; the rest of it would be inf - inf.
__device__ inline void three_parts(const float (&x)[8], half8_t (&part)[3]) {
  uint32_t bits[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) bits[i] = __float_as_uint(x[i]);
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    part[p] = __builtin_bit_cast(
        half8_t, make_uint4(high_pair(bits[0], bits[1]), high_pair(bits[2], bits[3]),
                            high_pair(bits[4], bits[5]), high_pair(bits[6], bits[7])));
    if (p == 2) break;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bits[i] = __float_as_uint(__uint_as_float(bits[i]) - __uint_as_float(bits[i] & 0xffff0000u));
    if (p == 0) {
      float top = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) top = fmaxf(top, fabsf(x[i]));
      if (__any(top == INFINITY)) {
        asm volatile("");  // (a branch that is hardly ever taken, not selects in every step)
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (fabsf(x[i]) == INFINITY) bits[i] = 0u;
      }
    }
  }
}
template <int XKIND>
__device__ inline float16_t product(const half8_t& a, const half8_t& b, const float16_t& sum) {
  if constexpr (XKIND == kXThree)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), sum, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, sum, 0, 0, 0);
}

// ------------------------------------------------------------------------------------ the product
// STEPS: matrix steps (16 codes) of a scale group inside a flush block: 8 (blocks of 128 codes,
// groups of 128 and more), or 4, 2, 1 (blocks of 64 codes, groups of 64, 32, 16).
template <int XKIND, int MT, int NT, int STEPS>
struct SliceGeometry {
  static constexpr int kPlanes = XKIND == kXThree ? 3 : XKIND == kXSplit ? 2 : 1;
  // Two running totals, groups in turn, where x keeps its bits: a sum's rounding then acts on half as
  // much, and the error against 64 bits is not above that of the GEMV over blocks of 16 rows.
  static constexpr int kTotals = XKIND == kXThree ? 2 : 1;
  static constexpr int kArea = 20 * 1024;            // a wave's share of the LDS
  // An x stage holds whole 128-byte lines where the LDS has room: what the second-level cache
  // delivers counts lines and half lines alike (127 GB/s a CU in 128-byte segments, 80 in 64-byte,
  // 40 in 32-byte ones).  64 fp16 codes, 32 codes of hi and lo or of f32; the largest tiles take
  // stages of 32 fp16 codes.
  static constexpr int kStage = XKIND == kX16 && MT * NT <= (STEPS == 8 ? 4 : 2) ? 64 : 32;
  static constexpr int kRowBytes = kStage * (XKIND == kX16 ? 2 : 4);
  static constexpr int kXBytes = 32 * MT * kRowBytes;
  static constexpr int kXLoads = kXBytes / 1024;
  static constexpr int kScales = STEPS == 8 ? 1 : 4 / STEPS;  // of a column in a flush block
  static constexpr int kSLoads = STEPS == 8 ? 0 : (32 * NT * kScales + 63) / 64;  // a unit
  // codes of a weight unit: the most whose two copies leave room for two stages
  static constexpr int unit_bytes(int codes) { return NT * 16 * codes + kSLoads * 256; }
  static constexpr int kUnit =
      STEPS < 8 ? 64
                : (2 * unit_bytes(256) + 2 * kXBytes <= kArea
                       ? 256
                       : (2 * unit_bytes(128) + 2 * kXBytes <= kArea ? 128 : 64));
  static constexpr int kWBytes = unit_bytes(kUnit);
  static constexpr int kWLoads = NT * kUnit / 64;
  static constexpr int kStagesPerUnit = kUnit / kStage;
  // ring depths: at stage g, stages g .. g + DX - 1 are in LDS or on their way, and the units
  // they belong to
  static constexpr int units_of(int depth) { return (depth - 1 + kStagesPerUnit - 1) / kStagesPerUnit + 1; }
  static constexpr bool fits(int depth) { return depth * kXBytes + units_of(depth) * kWBytes <= kArea; }
  static constexpr int kDepthX = fits(4) ? 4 : fits(3) ? 3 : 2;
  static constexpr int kDepthW = units_of(kDepthX);
  static_assert(fits(kDepthX), "the rings fit a wave's area");
  // output columns (in tiles of 32) that are summed at once at the end
  static constexpr int kSumTiles = MT * NT * 4096 <= kArea ? NT : kArea / (MT * 4096);
};

// Bits of the kernel's `flags`: element types, and whether the end reads anything in quads (kFetches), rope
// positions among it (kRope).
constexpr uint32_t kScaleF16 = 1, kIoF16 = 2, kFetches = 4, kRope = 8;

// WHOLE: hi and lo beside f32 scales, totals of whole weights (see scales_whole; a branch beside each group's sums
// cost fp16 scales 2 to 5 %, this form has the conversion of twelve operations a word).
template <int XKIND, int MT, int NT, int STEPS, bool WHOLE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_i4_slices_kernel(
    // (the leading 14 dwords of the arguments arrive in scalar registers with the wave)
    const uint8_t* __restrict__ x,  // [m][k], but kXSplit: [m][k / 32][hi, lo][32] fp16
    const uint8_t* __restrict__ w, const uint8_t* __restrict__ scales, uint32_t row_begin,
    uint32_t row_end, uint32_t n, uint32_t k, uint32_t group_shift, uint32_t m_blocks, uint32_t tiles, uint32_t flags,
    uint32_t m, SliceTail tail) {
  using G = SliceGeometry<XKIND, MT, NT, STEPS>;
  constexpr int kPlanes = G::kPlanes, kStage = G::kStage, kRowBytes = G::kRowBytes;
  constexpr int kLanesPerRow = kRowBytes / 16, kRowsPerLoad = 64 / kLanesPerRow;
  constexpr int BM = 32 * MT, BN = 32 * NT;
  constexpr int kScales = G::kScales;
  constexpr int DX = G::kDepthX, DW = G::kDepthW;
  __shared__ __align__(1024) uint8_t s_area[kWaves][G::kArea];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frag_row = lane & 31, frag_h = lane >> 5;
  // blockIdx & 7 is the XCD: each XCD takes a contiguous range of tiles, the row tiles of a
  // column tile next to each other, so the weights of a column tile come from memory once
  const uint32_t per_xcd = (tiles + 7u) >> 3;
  const uint32_t tile = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles || (blockIdx.x >> 3) >= per_xcd) return;
  const uint32_t nb = tile / m_blocks, mb = tile - nb * m_blocks;
  const uint32_t m0 = row_begin + mb * BM, n0 = nb * BN;

  // K in flush blocks of 128 codes (64 below groups of 128), dealt to the waves in order.  A K
  // that ends half-way through a block of 64 codes is loaded as its last 64 and only the second
  // half of those is used.
  constexpr int kBlock = STEPS == 8 ? 128 : 64;
  const uint32_t blocks = (k + kBlock - 1u) / kBlock;
  const uint32_t b0 = (uint32_t)wave * blocks / kWaves, b1 = ((uint32_t)wave + 1u) * blocks / kWaves;
  const uint32_t k0 = b0 * kBlock, k1 = min(b1 * kBlock, k);
  const bool ends_early = STEPS < 4 && (k1 & 63u) != 0;  // this slice's last 64 codes are 32

  uint8_t* const area = s_area[wave];
  const uint32_t x_ring = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)area;
  const uint32_t w_ring = x_ring + DX * G::kXBytes;

  // offsets of this lane's pieces inside the tile: rows past M or N re-read the last row
  constexpr uint32_t kXSize = XKIND == kX16 ? 2 : 4;
  const uint32_t x_row_bytes = k * kXSize;
  uint32_t x_off[G::kXLoads];
#pragma unroll
  for (int i = 0; i < G::kXLoads; ++i) {
    const uint32_t row = kRowsPerLoad * i + lane / kLanesPerRow;
    const uint32_t turn = kRowBytes == 128 ? (row & 7u) : ((row >> 1) & 3u);
    const uint32_t piece = (lane % kLanesPerRow) ^ turn;
    x_off[i] = min(row, row_end - 1u - m0) * x_row_bytes + piece * 16u;
  }
  // weights: kUnit / 32 pieces of 16 bytes a row
  constexpr uint32_t kPieces = G::kUnit / 32, kWRows = 64 / kPieces;
  constexpr int kWRowLoads = 32 * NT / kWRows;
  static_assert(kWRowLoads == G::kWLoads, "a unit is whole loads");
  auto w_turn_of = [](uint32_t row) { return kPieces == 2 ? (row >> 2) & 1u : kPieces == 4 ? (row >> 1) & 3u : row & 7u; };
  uint32_t w_row[kWRowLoads];
#pragma unroll
  for (int i = 0; i < kWRowLoads; ++i)
    w_row[i] = min(kWRows * i + lane / kPieces, n - 1u - n0) * (k >> 1);
  const uint32_t w_piece = ((lane % kPieces) ^ w_turn_of(lane / kPieces)) * 16u;
  static_assert(kWRows % 8 == 0, "the turn of a row is the same in every load");
  // (the planes of the split form hold rows row_begin.. only)
  const uint8_t* const x_tile =
      x + (size_t)(XKIND == kXSplit ? m0 - row_begin : m0) * x_row_bytes;
  const uint8_t* const w_tile = w + (size_t)n0 * (k >> 1);

  // Group scales.  Blocks of 128 codes: one a column, requested into a register at the block's
  // start and used behind its last step.  Smaller groups: the scales of a unit travel with its
  // weights, entry e * 32 NT + column.
  const uint32_t groups = k >> group_shift;
  const bool scale_f16 = (flags & kScaleF16) != 0;
  const uint32_t scale_size = scale_f16 ? 2u : 4u;
  constexpr int kSOff = STEPS == 8 ? NT : G::kSLoads;
  uint32_t s_off[kSOff];
#pragma unroll
  for (int i = 0; i < kSOff; ++i) {
    const uint32_t entry = STEPS == 8 ? 32u * i + (uint32_t)frag_row
                                      : min(64u * i + (uint32_t)lane, 32u * NT * kScales - 1u);
    s_off[i] = (min(entry % (32u * NT), n - 1u - n0) * groups + entry / (32u * NT)) * scale_size;
  }
  const uint8_t* const s_tile = scales + (size_t)n0 * groups * scale_size;

  // Stage g of the slice (relative to its first): the weight unit, if it opens one, then x.
  constexpr int X = G::kXLoads, W = G::kWLoads + G::kSLoads, R = G::kStagesPerUnit;
  auto stage_code = [&](uint32_t g) {
    const uint32_t code = k0 + g * kStage;
    return STEPS < 4 ? min(code, k - kStage) : code;  // (a last half stage of 64: its last 64 codes)
  };
  auto request = [&](uint32_t g) {
    if (g % R == 0) {
      const uint32_t code = k0 + g * kStage;
      const uint32_t from = STEPS < 4 ? min(code, k - 64u) : code;  // (the last 64 codes likewise)
      const uint32_t dst = w_ring + (g / R % DW) * G::kWBytes;
      // a unit that reaches past the row's end re-reads its last piece, unused
      const uint32_t piece = G::kUnit > kBlock || STEPS == 8 ? min((from >> 1) + w_piece, (k >> 1) - 16u) : (from >> 1) + w_piece;
#pragma unroll
      for (int i = 0; i < kWRowLoads; ++i) stream_to_lds(dst + 1024u * i, w_row[i] + piece, w_tile);
      if constexpr (STEPS < 8) {
        const uint8_t* src = s_tile + (size_t)(from >> group_shift) * scale_size;
#pragma unroll
        for (int i = 0; i < G::kSLoads; ++i)
          stream_word_to_lds(dst + NT * 1024u + 256u * i, s_off[i], src, scale_f16);
      }
    }
    const uint8_t* src = x_tile + (size_t)stage_code(g) * kXSize;
    const uint32_t dst = x_ring + (g % DX) * G::kXBytes;
#pragma unroll
    for (int i = 0; i < X; ++i) stream_to_lds(dst + 1024u * i, x_off[i], src);
  };
  uint32_t scale_raw[NT];
  auto load_scales = [&](uint32_t first_code) {
    if constexpr (STEPS == 8) {
      const uint8_t* src = s_tile + (size_t)(first_code >> group_shift) * scale_size;
      if (scale_f16) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          asm volatile("global_load_ushort %0, %1, %2"
                       : "=v"(scale_raw[nt]) : "v"(s_off[nt]), "s"(src) : "memory");
      } else {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          asm volatile("global_load_dword %0, %1, %2"
                       : "=v"(scale_raw[nt]) : "v"(s_off[nt]), "s"(src) : "memory");
      }
    }
  };

  float16_t total[G::kTotals][MT][NT], acc[MT][NT];
  float16_t zero16;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero16[r] = 0.f;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      acc[mt][nt] = zero16;
#pragma unroll
      for (int i = 0; i < G::kTotals; ++i) total[i][mt][nt] = zero16;
    }

  // fragment addresses inside a stage / a unit.  Step j of 32 codes covers the 8-code pieces
  // 2 h + j (one 8-byte read of weights); groups of 16 need the two pieces of a step next to each
  // other: 2 j + h.
  const uint32_t x_turn = kRowBytes == 128 ? (frag_row & 7u) : ((frag_row >> 1) & 3u);
  const uint8_t* const x_frag = area + frag_row * kRowBytes;
  const uint8_t* const w_frag =
      area + DX * G::kXBytes + frag_row * (16 * kPieces) + (STEPS == 1 ? 4u : 8u) * frag_h;
  const uint32_t w_turn = w_turn_of(frag_row);

  auto flush = [&](uint32_t unit_slot, int e, int turn) {
    auto& to = total[turn % G::kTotals];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      uint32_t bits;
      if constexpr (STEPS == 8) {
        bits = scale_raw[nt];
      } else {
        bits = *reinterpret_cast<const uint32_t*>(area + DX * G::kXBytes + unit_slot * G::kWBytes + 1024 * NT +
                                                  4u * (e * 32 * NT + nt * 32 + frag_row));
      }
      const float s = scale_f16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)bits) : __uint_as_float(bits);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          to[mt][nt][r] = fmaf(acc[mt][nt][r], s, to[mt][nt][r]);
    }
  };
  // 32 codes: quarter `wq` of the weight unit in slot `unit_slot`, half `xq` of the stage in slot
  // `slot`; `opens`: the first step starts a scale group (its sums start from zero); `e`: the
  // unit's scale entry (half of 64 codes) for groups below 64, added to the totals of `turn`
  auto half = [&](uint32_t unit_slot, uint32_t wq, uint32_t slot, int xq, bool opens, int e,
                  int turn) {
    const uint8_t* xs = x_frag + slot * G::kXBytes;
    const uint8_t* ws = w_frag + unit_slot * G::kWBytes + ((wq ^ w_turn) * 16u);
    uint2 words[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint8_t* at = ws + nt * (512 * kPieces);
      if constexpr (STEPS == 1) {
        words[nt].x = *reinterpret_cast<const uint32_t*>(at);
        words[nt].y = *reinterpret_cast<const uint32_t*>(at + 8);
      } else {
        words[nt] = *reinterpret_cast<const uint2*>(at);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t piece = STEPS == 1 ? 2u * j + frag_h : 2u * frag_h + j;
      half8_t a[kPlanes][MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const uint8_t* row = xs + mt * (32 * kRowBytes);
        if constexpr (XKIND == kX32 || XKIND == kXThree) {
          const float4 lo = *reinterpret_cast<const float4*>(row + (((2u * piece) ^ x_turn) * 16u));
          const float4 hi = *reinterpret_cast<const float4*>(row + (((2u * piece + 1u) ^ x_turn) * 16u));
          if constexpr (XKIND == kXThree) {
            const float eight[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            half8_t part[3];
            three_parts(eight, part);
#pragma unroll
            for (int p = 0; p < 3; ++p) a[p][mt] = part[p];
          } else {
            a[0][mt] = half8_t{(_Float16)lo.x, (_Float16)lo.y, (_Float16)lo.z, (_Float16)lo.w,
                               (_Float16)hi.x, (_Float16)hi.y, (_Float16)hi.z, (_Float16)hi.w};
          }
        } else {
#pragma unroll
          for (int p = 0; p < kPlanes; ++p)
            a[p][mt] = *reinterpret_cast<const half8_t*>(
                row + (((4u * (kStage == 64 ? xq : p) + piece) ^ x_turn) * 16u));
        }
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const uint32_t word = j == 0 ? words[nt].x : words[nt].y;
        const half8_t b = XKIND == kXThree ? sixteenths(word)
                          : XKIND == kXSplit ? ints_paired<!WHOLE>(word) : ints_natural(word);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int p = 0; p < kPlanes; ++p) {
            const bool zero = p == 0 && (STEPS == 1 || (j == 0 && opens));
            acc[mt][nt] = product<XKIND>(a[p][mt], b, zero ? zero16 : acc[mt][nt]);
          }
      }
      if constexpr (STEPS == 1) flush(unit_slot, 2 * e + j, j);
    }
    if constexpr (STEPS == 2) flush(unit_slot, e, turn);
  };
  constexpr int kRegScales = STEPS == 8 ? NT : 0;  // loads of a block's scales

  // The end of the kernel, per thread: quads of columns p = thread + 512 i of the tile's rows.
  auto quad_at = [&](int p, int t0, int quads, uint32_t* row, uint32_t* col) {
    *row = m0 + (uint32_t)(p / quads);
    *col = n0 + 32u * t0 + 4u * (uint32_t)(p % quads);
    return p < BM * quads && *row < row_end && *col < n;
  };
  auto tiles_from = [](int t0) { return NT - t0 < G::kSumTiles ? NT - t0 : G::kSumTiles; };
  // Rope positions of those rows: the table rows that they name are a second trip behind this one.
  constexpr int kMostItems = (BM * 8 * G::kSumTiles + 511) / 512;
  int32_t pos[kMostItems];
  auto fetch_positions = [&](int t0) {
    const int quads = 8 * tiles_from(t0);
#pragma unroll
    for (int i = 0; i < kMostItems; ++i) {
      uint32_t row, col;
      pos[i] = -1;
      if (quad_at((int)threadIdx.x + 512 * i, t0, quads, &row, &col)) pos[i] = tail.fuse.positions[row];
    }
  };
  // (Decided by a word that arrives with the wave.  Read from `tail`, which does not, the decision stood in
  // front of the first stages; and fp16 that became f32 where it was asked for kept the K loop waiting for
  // every stage on its way.  64 to 256 rows, n and k of 256 to 2048, fp16, us with both / without, cold weights:
  // 64 x 256 x 256 in groups of 64 3.7 / 3.3, 64 x 1024 x 1024 4.84 / 4.40, 128 x 2048 x 1024 5.05 / 4.61; 104
  // products without rope take 0.85 to 0.98 of the time.)
  const bool fetches = (flags & kFetches) != 0, io_f16 = (flags & kIoF16) != 0;
  if ((flags & kRope) != 0) fetch_positions(0);
  QuadAhead ahead[kMostItems];
  float inv[kMostItems];
  auto fetch = [&](int t0) {
    const int quads = 8 * tiles_from(t0);
#pragma unroll
    for (int i = 0; i < kMostItems; ++i) {
      uint32_t row, col;
      if (quad_at((int)threadIdx.x + 512 * i, t0, quads, &row, &col)) {
        if constexpr (XKIND == kXSplit) inv[i] = tail.row_scale[2 * (size_t)row + 1];
        if (fetches) {
          if (io_f16) fetch_quad<__half>(ahead[i], row, col, n, pos[i], static_cast<const __half*>(tail.bias), tail.fuse);
          else fetch_quad<float>(ahead[i], row, col, n, pos[i], static_cast<const float*>(tail.bias), tail.fuse);
        }
      }
    }
  };
  // (larger tiles have no registers for it yet)
  constexpr bool kFetchFirst = MT * NT <= 2 && G::kTotals == 1;

  if (k0 < k1) {
    const uint32_t stages = (k1 - k0 + kStage - 1u) / kStage;
    constexpr int kStages = kBlock / kStage;  // of a flush block
    // At most the stages younger than g (and, `more`, other loads) are on their way.  (What the end of the
    // kernel fetches ahead is not counted, as its loads differ from wave to wave: the first waits then ask for
    // as many loads of a younger stage.)
    auto wait_for = [&](uint32_t g, auto more_tag) {
      constexpr int MORE = decltype(more_tag)::value;
      const uint32_t left = min((uint32_t)(DX - 1), stages - 1u - g);
      auto wait_n = [&](auto n_tag) {
        constexpr int N = decltype(n_tag)::value;
        if constexpr (R == 1) {
          wait_vm<N * (X + W) + MORE>();
        } else if constexpr (N == 0) {
          wait_vm<MORE>();
        } else if constexpr (N == R) {
          wait_vm<N * X + W + MORE>();
        } else {  // does one of the N younger stages open a unit?
          static_assert(N < R || (R == 2 && N == 3), "at most one or two units");
          constexpr int kBase = R == 2 && N == 3 ? 1 : 0;
          if ((g + N) / R - g / R > (uint32_t)kBase) wait_vm<N * X + (kBase + 1) * W + MORE>();
          else wait_vm<N * X + kBase * W + MORE>();
        }
      };
      if (DX >= 4 && left == 3u) wait_n(std::integral_constant<int, DX >= 4 ? 3 : 0>{});
      else if (DX >= 3 && left == 2u) wait_n(std::integral_constant<int, DX >= 3 ? 2 : 0>{});
      else if (left == 1u) wait_n(std::integral_constant<int, 1>{});
      else wait_n(std::integral_constant<int, 0>{});
    };
#pragma unroll
    for (int i = 0; i < DX - 1; ++i)
      if ((uint32_t)i < stages) request(i);
    if (kFetchFirst && (fetches || XKIND == kXSplit)) fetch(0);
    for (uint32_t b = b0; b < b1; ++b) {
      load_scales(b * kBlock);
#pragma unroll
      for (int i = 0; i < kStages; ++i) {
        const uint32_t g = (b - b0) * kStages + i;
        if (kStages == 1 || STEPS >= 4 || g < stages) {
          if (g + DX - 1 < stages) request(g + DX - 1);
          // stage g was requested before the block's scales while i < DX - 1
          if (i < DX - 1 && i < kStages - 1) wait_for(g, std::integral_constant<int, kRegScales>{});
          else wait_for(g, std::integral_constant<int, 0>{});
          const uint32_t unit_slot = g / R % DW, slot = g % DX, wq = (g % R) * (kStage / 32);
          if constexpr (kStage == 64) {
            const bool early = ends_early && g + 1 == stages;
            if (!early) half(unit_slot, wq, slot, 0, i == 0, 0, 0);
            half(unit_slot, wq + 1, slot, 1, STEPS <= 2, 1, 1);
          } else {
            const bool early = ends_early && g + 1 == stages;  // the last 64 codes: second half
            half(unit_slot, early ? 1u : wq, slot, 0, STEPS <= 2 || i == 0, early ? 1 : i % 2, i);
          }
          if constexpr (STEPS == 4) { if (i == kStages - 1) flush(unit_slot, 0, 0); }
          // the reads of a slot are over before it is filled again
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
      }
      if constexpr (STEPS == 8) {
        // requested before the block's last DX - 1 stages were
        if constexpr (kStages <= DX - 1) {
          const uint32_t g = (b - b0) * kStages + kStages - 1;
          if (g + DX - 1 < stages) wait_vm<kStages * X>(); else wait_vm<0>();
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) asm volatile("" : "+v"(scale_raw[nt])::"memory");
        flush(0, 0, 0);
      }
    }
  } else if (kFetchFirst && (fetches || XKIND == kXSplit)) {
    fetch(0);  // no codes, rows to finish all the same
  }
  wait_vm<0>();

  // The waves' sums, [row][column] in their own areas, kSumTiles column tiles at a time; every
  // thread adds four columns of a row in wave order and finishes them.  What the finish reads from
  // memory (bias, residual, rope table) is asked for in front of the sums: asked for behind them it
  // was one trip to memory more, with positions two.  Inside the launch, fp16 x, K of 2048 but the last: 128 x
  // 2560 with rope 7.3 us, 6.2 so; 128 x 2048 with residual 5.0, 4.6; 128 x 11264 with silu 13.1, 12.7;
  // 128 x 2048 x 5632 with residual 10.8, 9.8.
  constexpr int kCols = 32 * G::kSumTiles;
  auto finish_tiles = [&](auto type, auto t0_tag) {
    using T = typename decltype(type)::type;
    constexpr int t0 = decltype(t0_tag)::value;
    constexpr int kTiles = NT - t0 < G::kSumTiles ? NT - t0 : G::kSumTiles;
    constexpr int quads = 8 * kTiles, kItems = (BM * quads + 511) / 512;
    const T* const bias = static_cast<const T*>(tail.bias);
    T* const out = static_cast<T*>(tail.out);
    if (t0 > 0 && (flags & kRope) != 0) fetch_positions(t0);
    if ((!kFetchFirst || t0 > 0) && (fetches || XKIND == kXSplit)) fetch(t0);
    float* sums = reinterpret_cast<float*>(area);
    if (t0 > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sums[(mt * 32 + 8 * (r / 4) + 4 * frag_h + (r % 4)) * kCols + t * 32 + frag_row] =
              G::kTotals == 2 ? total[0][mt][t0 + t][r] + total[G::kTotals - 1][mt][t0 + t][r]
                              : total[0][mt][t0 + t][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int p = threadIdx.x + 512 * i;
      uint32_t row, col;
      if (quad_at(p, t0, quads, &row, &col)) {
        float4 part[kWaves];
#pragma unroll
        for (int wv = 0; wv < kWaves; ++wv)
          part[wv] = *reinterpret_cast<const float4*>(
              s_area[wv] + (size_t)((p / quads) * kCols + 4 * (p % quads)) * 4);
        auto add = [](float4& to, const float4& v) {
          to.x += v.x; to.y += v.y; to.z += v.z; to.w += v.w;
        };
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (XKIND == kXThree) {  // in pairs: three roundings of a whole sum, not seven
#pragma unroll
          for (int step = 1; step < kWaves; step *= 2)
#pragma unroll
            for (int wv = 0; wv < kWaves; wv += 2 * step) add(part[wv], part[wv + step]);
          v = part[0];
        } else {
#pragma unroll
          for (int wv = 0; wv < kWaves; ++wv) add(v, part[wv]);
        }
        if constexpr (XKIND == kXSplit) {  // exact: a power of two
          const float back = WHOLE ? inv[i] : inv[i] * 1024.0f;
          v.x *= back; v.y *= back; v.z *= back; v.w *= back;
        }
        if constexpr (XKIND != kXSplit) {  // the weights went in as sixteenths or 1024ths
          constexpr float kWhole = XKIND == kXThree ? 16.f : 1024.f;
          v.x *= kWhole; v.y *= kWhole; v.z *= kWhole; v.w *= kWhole;
        }
        if (tail.quads) {
          finish_quad<T>(v, ahead[i], row, col, m, n, pos[i], bias != nullptr, out, tail.fuse);
        } else {
          finish_pair<T>(v.x, v.y, row, col, m, n, bias, out, tail.fuse);
          if (col + 2 < n) finish_pair<T>(v.z, v.w, row, col + 2, m, n, bias, out, tail.fuse);
        }
      }
    }
  };
  auto finish = [&](auto type) {
    finish_tiles(type, std::integral_constant<int, 0>{});
    if constexpr (NT > G::kSumTiles) finish_tiles(type, std::integral_constant<int, G::kSumTiles>{});
  };
  static_assert(NT <= 2 * G::kSumTiles, "two passes over the areas hold every column tile");
  if (io_f16) finish(type_tag<__half>{}); else finish(type_tag<float>{});
}

struct SliceCall {
  const void *x, *w, *scales;
  uint32_t row_begin, row_end, m, n, k, group_shift, scale_f16, io_f16;
  SliceTail tail;
};

template <int XKIND, int MT, int NT, int STEPS>
int32_t launch_slices(krm_ctx* ctx, const SliceCall& c) {
  const uint32_t m_blocks = (c.row_end - c.row_begin + 32 * MT - 1) / (32 * MT);
  const uint32_t tiles = m_blocks * ((c.n + 32 * NT - 1) / (32 * NT));
  uint32_t flags = (c.scale_f16 ? kScaleF16 : 0u) | (c.io_f16 ? kIoF16 : 0u);
  if (c.tail.quads && (c.tail.fuse.mode == 2 || c.tail.bias || c.tail.fuse.residual)) flags |= kFetches;
  if ((flags & kFetches) && c.tail.fuse.mode == 2) flags |= kRope;
  auto kernel = gemm_i4_slices_kernel<XKIND, MT, NT, STEPS, false>;
  if constexpr (XKIND == kXSplit)
    if (!c.scale_f16) kernel = gemm_i4_slices_kernel<XKIND, MT, NT, STEPS, true>;
  kernel<<<dim3(((tiles + 7) / 8) * 8), dim3(512), 0, ctx->stream>>>(
          static_cast<const uint8_t*>(c.x), static_cast<const uint8_t*>(c.w),
          static_cast<const uint8_t*>(c.scales), c.row_begin, c.row_end, c.n, c.k, c.group_shift,
          m_blocks, tiles, flags, c.m, c.tail);
  return launched(ctx, "gemm_i4_slices_kernel");
}

// The tile of a shape.  One workgroup fills a CU (160 KB of LDS), so a launch takes
// ceil(tiles / CUs) rounds of a fixed part (latency, the sum over the waves, the epilogue) and a
// part in K (what the second-level cache delivers to a CU per code of its tile).  Both were
// measured for every tile (us, and us per 1024 codes, cold weights); the cheapest product wins.
struct TileCost {
  int mt, nt;
  float fixed, per_1024;
};
constexpr TileCost kCost16[] = {{1, 1, 0.8f, 1.5f}, {1, 2, 1.3f, 2.0f}, {1, 3, 1.7f, 2.5f},
                                {2, 1, 0.7f, 2.0f}, {2, 2, 2.4f, 2.6f}, {2, 3, 2.2f, 3.6f}};
constexpr TileCost kCostSplit[] = {{1, 1, 0.2f, 2.45f}, {1, 2, 0.4f, 2.9f}, {1, 3, 0.9f, 3.4f},
                                   {2, 1, 0.2f, 3.5f}, {2, 2, 1.0f, 4.5f}};
constexpr TileCost kCostThree[] = {{1, 1, 3.2f, 3.35f}, {1, 2, 4.8f, 4.5f}, {1, 3, 6.4f, 5.7f}, {1, 4, 8.5f, 6.85f}, {2, 1, 4.6f, 4.8f}};
constexpr TileCost kCost32[] = {{1, 1, 0.8f, 1.75f}, {1, 2, 1.3f, 2.3f}, {1, 3, 1.7f, 2.9f},
                                {2, 1, 0.7f, 2.75f}, {2, 2, 2.2f, 3.3f}};

// The cheapest tile of a shape, and its rounds over the CUs.
template <int XKIND, int STEPS>
TileCost cheapest_tile(const krm_ctx* ctx, uint64_t rows, uint32_t n, uint32_t k, uint64_t* rounds) {
  const TileCost* table = XKIND == kX16 ? kCost16 : XKIND == kXSplit ? kCostSplit
                          : XKIND == kXThree ? kCostThree : kCost32;
  const int count = XKIND == kX16 ? 6 : 5;
  const uint64_t cus = (uint64_t)ctx->num_cus;
  int best = 0;
  float best_cost = 0.f;
  for (int i = 0; i < count; ++i) {
    const TileCost& t = table[i];
    // (below groups of 128 codes the wide tiles' LDS goes to scales; groups of 16 take 32 x 32.  Three
    // parts of f32 x: wide tiles share the conversion, 32 x 128 in groups of 16 would spill)
    if ((STEPS < 8 && t.nt > 2 && XKIND != kXThree) || (STEPS < 8 && t.mt * t.nt > 2 && XKIND != kX16 && XKIND != kXThree) ||
        (STEPS == 1 && (XKIND == kXThree ? t.mt > 1 || t.nt > 3 : t.mt * t.nt > 1)))
      continue;
    const uint64_t tiles = ((rows + 32 * t.mt - 1) / (32 * t.mt)) * (((uint64_t)n + 32 * t.nt - 1) / (32 * t.nt));
    const uint64_t turns = (tiles + cus - 1) / cus;
    const float cost = (float)turns * (t.fixed + t.per_1024 * (float)k * (1.0f / 1024));
    if (i == 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
      *rounds = turns;
    }
  }
  return table[best];
}

template <int XKIND, int STEPS>
int32_t pick_tile(krm_ctx* ctx, const SliceCall& c) {
  uint64_t rounds = 0;
  const TileCost best = cheapest_tile<XKIND, STEPS>(ctx, c.row_end - c.row_begin, c.n, c.k, &rounds);
  const int tile = best.mt * 10 + best.nt;
  if constexpr (STEPS == 8 && XKIND == kX16) {
    if (tile == 23) return launch_slices<XKIND, 2, 3, STEPS>(ctx, c);
  }
  if constexpr (STEPS == 2 && XKIND == kXThree) {
    if (tile == 14) return launch_slices<XKIND, 1, 4, STEPS>(ctx, c);
  }
  if constexpr (STEPS == 8 || XKIND == kXThree) {
    if (tile == 13) return launch_slices<XKIND, 1, 3, STEPS>(ctx, c);
  }
  if constexpr (STEPS == 8 || (STEPS > 1 && XKIND == kX16)) {
    if (tile == 22) return launch_slices<XKIND, 2, 2, STEPS>(ctx, c);
  }
  if constexpr (STEPS > 1 || XKIND == kXThree) {
    if (tile == 12) return launch_slices<XKIND, 1, 2, STEPS>(ctx, c);
  }
  if constexpr (STEPS > 1) {
    if (tile == 21) return launch_slices<XKIND, 2, 1, STEPS>(ctx, c);
  }
  return launch_slices<XKIND, 1, 1, STEPS>(ctx, c);
}

template <int XKIND>
int32_t pick_steps(krm_ctx* ctx, const SliceCall& c) {
  if constexpr (XKIND != kXThree) {
    if (c.group_shift >= 7) return pick_tile<XKIND, 8>(ctx, c);
    if (c.group_shift == 6) return pick_tile<XKIND, 4>(ctx, c);
  }
  if constexpr (XKIND == kXSplit)
    return fail(ctx, KRM_ERR_VALIDATION, "linear: hi + lo planes need groups of 64 and more");
  else
    return c.group_shift == 5 ? pick_tile<XKIND, 2>(ctx, c) : pick_tile<XKIND, 1>(ctx, c);
}

}  // namespace

namespace krm {

// Microseconds of a call over more rounds than one, for the choice against the unit-dealt form of
// gemm_i4.hip (groups of 64 and more).  The costs above choose between tiles; a round's absolute time
// is {per call, more per round, factor of the part in K}, fitted over 17 to 33 shapes of 65 to 512
// rows each (rms 6 to 10 %).
float slices_estimate_us(const krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t group,
                         bool half_x, bool split) {
  struct Fit {
    float call, round, factor;
  };
  uint64_t rounds = 0;
  TileCost t;
  Fit f;
  if (group >= 128) {
    t = half_x ? cheapest_tile<kX16, 8>(ctx, m, n, k, &rounds)
        : split ? cheapest_tile<kXSplit, 8>(ctx, m, n, k, &rounds)
                : cheapest_tile<kX32, 8>(ctx, m, n, k, &rounds);
    f = half_x ? Fit{0.4f, 2.0f, 1.0f} : split ? Fit{5.1f, 2.0f, 0.93f} : Fit{0.5f, 1.25f, 1.15f};
  } else {
    t = half_x ? cheapest_tile<kX16, 4>(ctx, m, n, k, &rounds)
        : split ? cheapest_tile<kXSplit, 4>(ctx, m, n, k, &rounds)
                : cheapest_tile<kX32, 4>(ctx, m, n, k, &rounds);
    f = half_x ? Fit{1.2f, 0.7f, 1.26f} : split ? Fit{7.9f, 1.4f, 0.95f} : Fit{2.9f, 1.0f, 1.25f};
  }
  return f.call + (float)rounds * (t.fixed + f.round + f.factor * t.per_1024 * (float)k * (1.0f / 1024));
}

// Any shape with K a multiple of 32 (at least 64), any group size of the format and 16-byte
// aligned rows.  *handled = false (nothing launched) otherwise.
int32_t linear_i4_gemm_slices(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias,
                              krm_buf out, uint32_t m, uint32_t n, uint32_t k, uint32_t group,
                              int32_t io_dtype, int32_t scale_dtype, int32_t compute,
                              const RowsFusion& fuse, bool* handled, int32_t x_dtype) {
  *handled = false;
  const bool half_x = x_dtype == KRM_F16 && io_dtype == KRM_F32;  // fp16 x, f32 bias / out
  if (x_dtype != io_dtype && !(half_x && compute == KRM_COMPUTE_F16)) return KRM_OK;
  const bool split = compute == KRM_COMPUTE_F32 && io_dtype == KRM_F32;
  if (k % 32 != 0 || k < 64 || !aligned(w, 16) || !aligned(x, 16)) return KRM_OK;
  if ((uint64_t)m * k > 0xffffffffull || (uint64_t)n * (k >> 1) > 0xffffffffull) return KRM_OK;
  if ((uint64_t)((m + 31) / 32) * ((n + 31) / 32) > 0x7fffffffull) return KRM_OK;
  SliceCall c{};
  c.x = ptr<const void>(x);
  c.w = ptr<const void>(w);
  c.scales = ptr<const void>(scales);
  c.row_end = c.m = m;
  c.n = n;
  c.k = k;
  while ((1u << c.group_shift) < group) ++c.group_shift;
  c.scale_f16 = scale_dtype == KRM_F16;
  c.io_f16 = io_dtype == KRM_F16;
  c.tail.bias = ptr<const void>(bias);
  c.tail.out = ptr<void>(out);
  c.tail.fuse = fuse;
  c.tail.quads = quads_aligned(c.tail.bias, c.tail.out, n, dtype_bytes(io_dtype), fuse);
  if (!split) {
    *handled = true;
    return x_dtype == KRM_F16 ? pick_steps<kX16>(ctx, c) : pick_steps<kX32>(ctx, c);
  }
  if (group < 64) {
    *handled = true;
    return pick_steps<kXThree>(ctx, c);
  }
  // hi and lo of as many rows as the context's scratch holds at a time
  const uint64_t scratch = (uint64_t)2 * ctx->num_cus * kGemmPartialBytes, row_bytes = (uint64_t)k * 4;
  const uint64_t fit = scratch / row_bytes / 32 * 32;
  if (m > kMaxSplitRows || fit == 0) return KRM_OK;
  KRM_TRY(needs_serial_scratch(ctx, "the f32-class few-row GEMM"));
  *handled = true;
  c.tail.row_scale = ctx->row_scales;
  for (uint64_t first = 0; first < m; first += fit) {
    const uint32_t rows = (uint32_t)(m - first < fit ? m - first : fit);
    launch_split_rows(ctx, ptr<const float>(x) + first * k, reinterpret_cast<uint4*>(ctx->gemm_partials),
                      ctx->row_scales + 2 * first, rows, k, k);
    KRM_TRY(launched(ctx, "split_rows_kernel"));
    c.x = reinterpret_cast<const uint8_t*>(ctx->gemm_partials);
    c.row_begin = (uint32_t)first;
    c.row_end = (uint32_t)first + rows;
    KRM_TRY(pick_steps<kXSplit>(ctx, c));
  }
  return KRM_OK;
}

}  // namespace krm
