// int4 `linear` for products of many tiles on the gfx950 matrix cores: exact integer weights, the work
// dealt over one workgroup per CU.
//
// out[m, n] = sum_k x[m,k] * dequant(w)[n,k] + bias[n]
// (packages/runtime/src/kernels/linear.ts:34-64, packages/runtime/src/kernels/gemm.ts:1187-1237).
// The weights enter the matrix cores as the exact integers (u - 8) in fp16 and the group scale
// multiplies the f32 sum of a group afterwards — the arithmetic of the GEMV, on MFMA.  Two forms of x:
//   PLANES 1  fp16 x (f32 x that was rounded before: f32 bias and result): one MFMA a step;
//   PLANES 2  f32 x as x * 2^e = hi + lo, both fp16, |x * 2^e - (hi + lo)| <= 2^-23 |x * 2^e| (e per
//             row, chosen so that the row's largest magnitude lands in [2^13, 2^14): no overflow, and
//             small entries keep an absolute resolution of 2^-38 of the row's maximum), written once by
//             split_rows_kernel: two MFMAs a step, products exact, f32 sums — the class of the
//             reference's default f32 `linear`.
//
// Bound by its arithmetic: a stage of 128 codes and a 64 x 64 tile a wave is 64 (128 with hi and lo) MFMAs
// of 32 clk a SIMD pair of waves and about 550 vector instructions of 4.3 clk beside them (conversion of
// the integers, the scaled sums of the groups), of which only a part hides behind the MFMAs: a stage
// takes 3850 clk where the MFMAs alone take 2048.  What the layout is for is everything else:
//   - x and the weights go from memory to LDS directly (no registers, no second pass through them), in
//     lines of 128 bytes: a load costs about 2 clk a line that it touches, whatever it uses of it;
//   - scales come in blocks of two or four stages, neighbouring lanes taking neighbouring groups of a
//     column: one scale a lane from 64 columns cost 2048 clk a stage of a 4800-clk stage;
//   - hi and lo are written once, by a pass of their own, and not again by each of the n / 512 column
//     tiles, which took the K loop over the register file;
//   - the K loop is one basic block of eight steps, each step's products beside the reads and conversion
//     of the next step's operands, one barrier a stage.
// us, before (stages staged through registers, f32 x split in the loop; f32 512 x 4096 x 11008 in groups of 128: on
// the K-splitting tiles) / now, in replayed recordings over four weights, no bias, fp16 scales, groups of 128 and
// of 64: f32 512 x 11008 x 4096 119 / 96 and 126 / 100, 512 x 4096 x 11008 117 / 101 and 177 / 106, 348 x 8164 x 4608
// 88 / 69 and 96 / 73; fp16 512 x 11008 x 4096 72 / 65 and 77 / 66, 348 x 8164 x 4608 49 / 44 and 52 / 45.  (512 x
// 11008 x 4096 over one weight, fp16: 66 / 56.)  About 20 us of each are not the K loop: launch 7, first loads 3, the
// partials of shared tiles 8.
#include "gemm_i4_deal.h"
#include "gemm_i4_rows.h"

using namespace krm;

namespace {

constexpr int kStage = 128;  // codes of a stage

// N times 16 bytes a lane to LDS, 8 KB apart, unless `stage` lies past the range's end.
template <int N>
__device__ inline void stream_rows(uint32_t stage, uint32_t end, uint32_t lds, const uint32_t (&offset)[N],
                                   const void* base) {
#define KRM_ROWS_OPEN "s_cmp_lt_u32 %0, %1\n\ts_cbranch_scc0 .Lpast%=\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\t"
#define KRM_ROWS_NEXT "\n\ts_add_u32 m0, m0, 0x2000\n\ts_nop 0\n\t"
  static_assert(N == 2 || N == 4, "loads of a wave and stage");
  if constexpr (N == 2) {
    asm volatile(KRM_ROWS_OPEN "global_load_lds_dwordx4 %4, %3" KRM_ROWS_NEXT "global_load_lds_dwordx4 %5, %3\n"
                 ".Lpast%=:" ::"s"(stage), "s"(end), "s"(lds), "s"(base), "v"(offset[0]), "v"(offset[1])
                 : "memory", "scc");
  } else {
    asm volatile(KRM_ROWS_OPEN "global_load_lds_dwordx4 %4, %3" KRM_ROWS_NEXT
                 "global_load_lds_dwordx4 %5, %3" KRM_ROWS_NEXT "global_load_lds_dwordx4 %6, %3" KRM_ROWS_NEXT
                 "global_load_lds_dwordx4 %7, %3\n.Lpast%=:" ::"s"(stage), "s"(end), "s"(lds), "s"(base),
                 "v"(offset[0]), "v"(offset[1]), "v"(offset[2]), "v"(offset[3])
                 : "memory", "scc");
  }
#undef KRM_ROWS_OPEN
#undef KRM_ROWS_NEXT
}
// The loads of a stage have landed in every wave: at most N younger ones are on their way, none if
// `younger` lies past the range's end.
template <int N>
__device__ inline void stage_landed(uint32_t younger, uint32_t end) {
  asm volatile("s_cmp_lt_u32 %0, %1\n\ts_cbranch_scc1 .Lmore%=\n\ts_waitcnt vmcnt(0)\n.Lmore%=:\n\t"
               "s_waitcnt vmcnt(%2) lgkmcnt(0)\n\ts_barrier" ::"s"(younger), "s"(end), "n"(N)
               : "memory", "scc");
}

template <int PLANES, bool HALF, int WM_>
struct ExactGeometry {
  // Eight waves of 64 x 64 outputs: two rows of four (128 x 256) or one row of eight (64 x 512).  160 KB of
  // LDS hold three stages of fp16 x in groups of 128 or more and two of everything else.
  static constexpr int WM = WM_;
  static constexpr int BM = 64 * WM, BN = 512 / WM;
  static constexpr int kDepth = PLANES == 1 && !HALF ? 3 : 2;
  static constexpr int kXBytes = BM * kStage * 2 * PLANES, kXLoads = kXBytes / 8192;
  static constexpr int kWBytes = BN * kStage / 2, kWLoads = kWBytes / 8192;
  // Scales are asked for in blocks of stages, lane l of a load taking entry l % kEntries of column
  // l / kEntries: a load costs by the lines it touches, and one scale a lane touches 64 of them.  Every
  // stage's loads bring a part of the block behind its own (three blocks in LDS: one is read, one
  // waits, one is filled).  Four stages where the LDS allows: with two, hi and lo lost 8 %.
  static constexpr int kBlock = WM == 1 && (PLANES == 1 || HALF) ? 2 : 4;
  static constexpr int kEntries = kBlock * (HALF ? 2 : 1);
  static constexpr int kParts = BN * kEntries / 512, kSBytes = BN * kEntries * 4;
  static constexpr int kSLoads = (kParts + kBlock - 1) / kBlock;  // of a wave and stage
  static_assert(kBlock >= kDepth - 1, "a block of scales is read before its slot is filled again");
};

// HALF: groups of 64 codes, two a stage.
template <typename T, typename ST, int PLANES, bool HALF, int WM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_i4_exact_kernel(const uint8_t* __restrict__ x, const uint8_t* __restrict__ w,
                          const uint8_t* __restrict__ scales, uint32_t m, uint32_t n, uint32_t k,
                          uint32_t group_shift, uint32_t m_blocks, const T* __restrict__ bias,
                          T* __restrict__ out, UnitDeal deal, const float* __restrict__ row_scale) {
  using G = ExactGeometry<PLANES, HALF, WM>;
  constexpr int BM = G::BM, BN = G::BN, D = G::kDepth, X = G::kXLoads, W = G::kWLoads, S = G::kSLoads;
  // The totals (see scales_whole).  hi and lo have whole weights for it, twelve operations a word instead of nine:
  // 300 x 32000 x 2048 in groups of 64 102 -> 104 us (with the scales whole it spilled: 133).  f32 rows rounded before:
  // 512 x 11008 x 4096 in groups of 64 76 -> 86 (as much as in the tiles that round), in groups of 128 73 -> 74.
  constexpr bool kWhole = sizeof(ST) == 4 && sizeof(T) == 4, kWholeSums = kWhole && PLANES == 1;
  static_assert((size_t)BM * BN == kPartialFloats, "the partial slots hold one tile");
  __shared__ __align__(1024) uint8_t s_x[D * G::kXBytes];
  __shared__ __align__(1024) uint8_t s_w[D * G::kWBytes];
  __shared__ __align__(1024) uint8_t s_s[3 * G::kSBytes];
  __shared__ float s_inv[PLANES == 2 ? BM : 1];
  __shared__ uint32_t s_ticket;

  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wm = G::WM == 2 ? wave >> 2 : 0u, wn = G::WM == 2 ? wave & 3u : wave;
  const uint32_t frag_row = lane & 31u, frag_h = lane >> 5;
  const uint32_t groups = k >> group_shift, spt = deal.stages_per_tile;
  const uint32_t x_row_bytes = PLANES == 2 ? spt * (kStage * 4u) : k * 2u;  // (planes are padded)
  auto lds_address = [](const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
  };
  const uint32_t x_lds = lds_address(s_x) + wave * 1024u, w_lds = lds_address(s_w) + wave * 1024u;
  const uint32_t s_lds = lds_address(s_s) + wave * 256u;

  // Fragment addresses.  A stage of x in LDS: lines of 128 bytes (64 codes; or 32 codes, hi then lo),
  // [line][row][128]; of weights: [column][64].  The 16-byte pieces of a row are turned by the row
  // number so that the rows of a fragment spread over all banks.  Step (c, j) of a stage takes codes
  // 64 c + 32 h + 8 j .. of lane half h: word j of the 16 bytes that the lane reads of its weight row.
  const uint32_t x_turn = (frag_row >> 1) & 7u, w_turn = (frag_row >> 2) & 3u;
  uint32_t x_at[4], w_at[2];
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t piece = PLANES == 2 ? j : 4u * frag_h + j;
    x_at[j] = (PLANES == 2 ? frag_h * (BM * 128u) : 0u) + (wm * 64u + frag_row) * 128u + ((piece ^ x_turn) * 16u);
  }
#pragma unroll
  for (uint32_t c = 0; c < 2; ++c)
    w_at[c] = (wn * 64u + frag_row) * 64u + (((2u * c + frag_h) ^ w_turn) * 16u);
  const uint32_t s_at = (wn * 64u + frag_row) * (G::kEntries * 4u);

  // (workgroups are dealt to the eight XCDs in turn: neighbouring ranges lie on one)
  const uint32_t xcd = blockIdx.x & 7u;
  const uint32_t v = xcd * (gridDim.x >> 3) + min(xcd, gridDim.x & 7u) + (blockIdx.x >> 3);
  const uint32_t my_begin = deal_begin(deal, v);
  uint32_t left = deal_units(deal, v);

  // The tiles of the range are taken last to first: a range usually ends with the first stages of a
  // tile and begins with the last stages of the one before, so every workgroup walks K upwards from
  // (about) stage 0 and, at any moment, the chip reads few distinct K slices of x, which stay in the L2s.
  // What the loads of a tile need; rows past M or N re-read the last row.
  struct Tile {
    uint32_t tile, s0, s1, m0, n0;
    const uint8_t *x, *w, *s;
    uint32_t x_off[X], w_off[W], s_code;
  };
  const uint32_t w_piece = ((lane & 3u) ^ ((lane >> 4) & 3u)) * 16u;  // (row >> 2) & 3
  const uint32_t s_entry = wave * 64u + lane;                         // part q of a block: entries 512 q + ..
  auto locate = [&](uint32_t units_left) {
    Tile t;
    const uint32_t range_end = my_begin + units_left;
    t.tile = __builtin_amdgcn_readfirstlane((range_end - 1u) / spt);  // (the division runs on the vector ALUs)
    const uint32_t tile_first = t.tile * spt;
    t.s0 = __builtin_amdgcn_readfirstlane(my_begin > tile_first ? my_begin - tile_first : 0u);
    t.s1 = __builtin_amdgcn_readfirstlane(range_end - tile_first);
    const uint32_t nb = __builtin_amdgcn_readfirstlane(t.tile / m_blocks);
    t.m0 = (t.tile - nb * m_blocks) * BM;
    t.n0 = nb * BN;
    t.x = x + (size_t)t.m0 * x_row_bytes;
    t.w = w + (size_t)t.n0 * (k >> 1);
    t.s = scales + (size_t)t.n0 * groups * sizeof(ST);
#pragma unroll
    for (uint32_t i = 0; i < X; ++i) {  // load wave + 8 i: eight rows of a line
      const uint32_t load = wave + 8u * i, line = load / (BM / 8), row = load % (BM / 8) * 8u + lane / 8u;
      t.x_off[i] = min(row, m - 1u - t.m0) * x_row_bytes + line * 128u +
                   ((lane & 7u) ^ (((wave & 1u) * 4u + lane / 16u) & 7u)) * 16u;  // (row >> 1) & 7
    }
#pragma unroll
    for (uint32_t i = 0; i < W; ++i)  // sixteen columns a load
      t.w_off[i] = min((wave + 8u * i) * 16u + lane / 4u, n - 1u - t.n0) * (k >> 1);
    t.s_code = t.s0 * kStage + s_entry % G::kEntries * (HALF ? 64u : 128u);
    return t;
  };
  auto request_scales = [&](const Tile& t, uint32_t block, uint32_t slot, uint32_t part) {
    const uint32_t q = part % G::kParts;
    const uint32_t g = min((block * (G::kBlock * kStage) + t.s_code) >> group_shift, groups - 1u);
    const uint32_t col = min(s_entry / G::kEntries + q * (512u / G::kEntries), n - 1u - t.n0);
    stream_word_to_lds(s_lds + slot * G::kSBytes + q * 2048u, (col * groups + g) * (uint32_t)sizeof(ST), t.s,
                       sizeof(ST) == 2);
  };
  // A stage's loads, or none past the range's end: the branch is inside the instruction block, so that
  // the K loop stays one basic block and its products, reads and conversions are scheduled as one.
  auto request = [&](const Tile& t, uint32_t asked, uint32_t buf, uint32_t next_slot) {
    const uint32_t stage = __builtin_amdgcn_readfirstlane(min(asked, t.s1 - 1u));
    const uint32_t at = min(stage * (kStage / 2) + w_piece, (k >> 1) - 16u);
    const uint8_t* src = t.x + (size_t)stage * (kStage * 2u * PLANES);
    uint32_t w_from[W], x_from[X];
#pragma unroll
    for (int i = 0; i < W; ++i) w_from[i] = t.w_off[i] + at;
    // (fp16 x: the last stage of a K that ends half-way re-reads its first 64 codes, unused)
#pragma unroll
    for (int i = 0; i < X; ++i) {
      const bool past = PLANES == 1 && HALF && i >= X / 2 && stage * kStage + 64u >= k;
      x_from[i] = t.x_off[past ? i - X / 2 : i];
    }
    const uint32_t wanted = __builtin_amdgcn_readfirstlane(asked);
    stream_rows<W>(wanted, t.s1, w_lds + buf * G::kWBytes, w_from, t.w);
    stream_rows<X>(wanted, t.s1, x_lds + buf * G::kXBytes, x_from, src);
    const uint32_t since = asked - t.s0;
#pragma unroll
    for (int i = 0; i < S; ++i) request_scales(t, since / G::kBlock + 1u, next_slot, since % G::kBlock * S + i);
  };
  auto request_first = [&](const Tile& t) {
    request(t, t.s0, 0, 1);
#pragma unroll
    for (int q = 0; q < G::kParts; ++q) request_scales(t, 0, 0, q);
    __builtin_amdgcn_s_barrier();  // no wave's later stages queue in front of another's first
#pragma unroll
    for (uint32_t d = 1; d < D; ++d) request(t, t.s0 + d, d, 1u + d / G::kBlock);
  };

  {
    const Tile t = locate(left);
    request_first(t);
    if (t.s1 - t.s0 >= D) wait_vm<(D - 1) * (X + W + S)>(); else wait_vm<0>();
  }
  while (left > 0) {
    uint32_t tile, s0, s1, m0, n0;
    float16_t total[2][2];
    {
      const Tile t0 = locate(left);
      tile = t0.tile; s0 = t0.s0; s1 = t0.s1; m0 = t0.m0; n0 = t0.n0;
      float16_t acc[2][2], zero16;
#pragma unroll
      for (int r = 0; r < 16; ++r) zero16[r] = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) total[i >> 1][i & 1] = acc[i >> 1][i & 1] = zero16;
      float ws[2] = {0.f, 0.f};
      bool scales_past = false;
      half8_t a[2][PLANES][2], b[2][2];
      uint4 words[2];

      auto read_x = [&](int t, uint32_t base, half8_t (&to)[PLANES][2]) {
        const int c = t / 4, j = t % 4;
#pragma unroll
        for (int p = 0; p < PLANES; ++p)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) {
            const uint32_t at = (p == 1 ? x_at[j] ^ 64u : x_at[j]) + base;
            to[p][mt] = *reinterpret_cast<const half8_t*>(s_x + at + c * (BM * 128 * PLANES) + mt * 4096);
          }
      };
      auto read_words = [&](int c, uint32_t base, uint4 (&to)[2]) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) to[nt] = *reinterpret_cast<const uint4*>(s_w + w_at[c] + base + nt * 2048);
      };
      auto read_scales = [&](uint32_t since, uint32_t slot, int c) {
        const uint32_t entry = HALF ? 2u * (since % G::kBlock) + c : since % G::kBlock;
        const uint8_t* at = s_s + slot * G::kSBytes + s_at + 4u * entry;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const uint32_t bits = *reinterpret_cast<const uint32_t*>(at + nt * (32 * G::kEntries * 4));
          ws[nt] = sizeof(ST) == 2 ? (float)__builtin_bit_cast(_Float16, (uint16_t)bits) : __uint_as_float(bits);
        }
        if constexpr (kWholeSums) scales_past = scales_whole(ws);
      };
      auto convert = [&](int t, const uint4 (&from)[2], half8_t (&to)[2]) {
        const int j = t % 4;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          const uint32_t word = j == 0 ? from[nt].x : j == 1 ? from[nt].y : j == 2 ? from[nt].z : from[nt].w;
          to[nt] = PLANES == 2 ? ints_paired<!kWhole>(word) : ints_natural(word);
        }
      };
      // (inside a stage a branch for `whole_sums` cost registers and spilled: a multiplication there)
      auto flush = [&](int mt, int nt, bool inside) {
        const float factor = kWholeSums && inside && scales_past ? 1024.0f : 1.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          total[mt][nt][r] = fmaf(kWholeSums && inside ? acc[mt][nt][r] * factor : acc[mt][nt][r], ws[nt], total[mt][nt][r]);
      };
      // in front of the other flushes
      auto whole_sums = [&] {
        if constexpr (kWholeSums) {
          if (scales_past) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] *= 1024.0f;
          }
        }
      };
      // Step t of a stage whose operands are in registers; beside its products run the reads and the
      // conversion of the next step's operands (`next_x`, `next_words`: where they lie).
      auto products = [&](int t) {
        const int cur = t & 1;
        const bool opens = t == 0 || (HALF && t == 4);  // a group's sums start from zero
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt) {
            if (opens) flush(mt, nt, t == 4);
#pragma unroll
            for (int p = 0; p < PLANES; ++p)
              acc[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                  a[cur][p][mt], b[cur][nt], opens && p == 0 ? zero16 : acc[mt][nt], 0, 0, 0);
          }
      };

      // the first stage has landed in every wave (the others' loads of a later tile too)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      read_words(0, 0, words);
      read_x(0, 0, a[0]);
      convert(0, words, b[0]);

      uint32_t buf = 0, slot = 0, ask_slot = 1u + D / G::kBlock;  // of x and w; of the scales read, filled
      const uint32_t full = PLANES == 1 && HALF && s1 * kStage > k ? s1 - 1u : s1;
      for (uint32_t stage = s0; stage < full; ++stage) {
        const uint32_t x_base = buf * G::kXBytes, w_base = buf * G::kWBytes, since = stage - s0;
        const uint32_t free_buf = buf;
        buf = buf + 1 == D ? 0 : buf + 1;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const int next = (t & 1) ^ 1;
          if (t == 0) whole_sums();
          if (t == 7) {
            // the next stage has landed, in every wave, and this one has been read
            stage_landed<(D - 2) * (X + W + S)>(__builtin_amdgcn_readfirstlane(stage + D - 1), s1);
            request(t0, stage + D, free_buf, ask_slot);
            read_words(0, buf * G::kWBytes, words);
            read_x(0, buf * G::kXBytes, a[next]);
          } else {
            read_x(t + 1, x_base, a[next]);
          }
          products(t);
          if (t == 1) read_scales(since, slot, 0);
          if (HALF && t == 5) read_scales(since, slot, 1);
          convert(t + 1, words, b[next]);
          if (t == 2) read_words(1, w_base, words);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (since % G::kBlock == G::kBlock - 1u) slot = slot == 2u ? 0u : slot + 1u;
        if ((since + D) % G::kBlock == G::kBlock - 1u) ask_slot = ask_slot == 2u ? 0u : ask_slot + 1u;
      }
      if (full < s1) {  // the first 64 codes of the last stage
        const uint32_t x_base = buf * G::kXBytes;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (t == 0) whole_sums();
          if (t < 3) read_x(t + 1, x_base, a[(t & 1) ^ 1]);
          products(t);
          if (t == 1) read_scales(s1 - 1u - s0, slot, 0);
          if (t < 3) convert(t + 1, words, b[(t & 1) ^ 1]);
        }
      }
      wait_vm<0>();  // what was asked for past the end
      whole_sums();
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) flush(mt, nt, false);
    }
    __syncthreads();  // the LDS is free: the next tile's first stages come in beside what follows
    if (left > s1 - s0) request_first(locate(left - (s1 - s0)));

    // (the addresses below are formed here and not kept in registers across the loop above)
    uint32_t here = threadIdx.x;
    asm volatile("" : "+v"(here));
    const uint32_t o_row = (G::WM == 2 ? (here >> 8) * 64u : 0u) + ((here & 63u) >> 5) * 4u;
    const uint32_t o_col = n0 + (G::WM == 2 ? (here >> 6) & 3u : here >> 6) * 64u + (here & 31u);
    if constexpr (PLANES == 2) {
      if (here < BM) s_inv[here] = row_scale[2 * (size_t)min(m0 + here, m - 1u) + 1] * (kWhole ? 1.0f : 1024.0f);
      __syncthreads();
    }
    auto store_rows = [&](int mt, const float16_t (&sum)[2]) {
      const bool whole = m0 + BM <= m && n0 + BN <= n;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const uint32_t col = o_col + nt * 32u;
        const float add = bias && col < n ? to_f32<T>(bias[col]) : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const uint32_t local = o_row + mt * 32 + 8 * (r / 4) + (r % 4);
          float value = sum[nt][r];
          if (PLANES == 2 || !kWhole) value *= PLANES == 2 ? s_inv[local] : 1024.0f;  // exact: a power of two
          if (whole || (m0 + local < m && col < n))
            out[(size_t)(m0 + local) * n + col] = from_f32<T>(value + add);
        }
      }
    };
    if (s0 == 0 && s1 == spt) {
      store_rows(0, total[0]);
      store_rows(1, total[1]);
      // (64 stores behind the next tile's loads, fewer where the tile is cut off)
      if (m0 + BM <= m && n0 + BN <= n) wait_vm<63>(); else wait_vm<0>();
    } else {
      // Slot of workgroup u's partial of this tile: its second slot when its range began at or before
      // the tile's first unit, its first slot otherwise (a range holds at most one partial of either
      // kind).  16-byte piece c of thread t sits at [c * 512 + t].
      const uint32_t tile_begin = tile * spt;
      auto slot_of = [&](uint32_t u) { return 2u * u + (deal_begin(deal, u) <= tile_begin ? 1u : 0u); };
      uint32_t* ticket = deal.tickets + (size_t)tile * kTicketStride;
      const uint32_t first = deal_owner(deal, tile_begin), last = deal_owner(deal, tile_begin + spt - 1u);
      // Every other partial already there?  Then this one need not be written at all.
      if (here == 0)
        s_ticket = __hip_atomic_load(ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      bool merge = s_ticket == last - first;
      __syncthreads();  // s_ticket is written again below
      if (!merge) {
        float4_t* mine = reinterpret_cast<float4_t*>(deal.partials + (size_t)slot_of(v) * kPartialFloats) + here;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float16_t& t = total[i >> 3][(i >> 2) & 1];
          const int q = 4 * (i & 3);
          const float4_t piece = {t[q], t[q + 1], t[q + 2], t[q + 3]};
          publish4(mine + i * 512, piece);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this thread's partial is in memory
        __syncthreads();
        if (here == 0)
          s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        merge = s_ticket == last - first;  // arrived last after all
      } else {
        wait_vm<0>();
      }
      if (merge) {  // every other partial of the tile is complete; the sum is taken in K order
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          auto partial = [&](uint32_t u, float16_t (&part)[2]) {
            if (u == v) {
              part[0] = total[mt][0];
              part[1] = total[mt][1];
              return;
            }
            const float4_t* src = reinterpret_cast<const float4_t*>(
                deal.partials + (size_t)slot_of(u) * kPartialFloats) + mt * 8 * 512 + here;
            float4_t p[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = observe4(src + i * 512);
            landed(p);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
              for (int e = 0; e < 4; ++e) part[i >> 2][4 * (i & 3) + e] = p[i][e];
          };
          // (the first one outside the loop: a sum that its first turn set was kept over the tiles, in scratch)
          float16_t sum[2];
          partial(first, sum);
          for (uint32_t u = first + 1u; u <= last; ++u) {
            float16_t part[2];
            partial(u, part);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
              for (int r = 0; r < 16; ++r) sum[nt][r] += part[nt][r];
          }
          store_rows(mt, sum);
        }
        if (here == 0)
          __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    left -= s1 - s0;
  }
}

// Rows and columns of a tile: whichever pads M and N less; 128 x 256 where both pad alike (half
// the scales a stage: 512 x 11008 x 4096 67.8 us, 64 x 512 69.9; groups of 64 67.0, 70.5).  hi and lo: 64 x 512
// alone (128 rows of both planes do not fit the LDS twice).
uint32_t exact_rows(uint32_t m, uint32_t n, bool split) {
  const uint64_t tall = (uint64_t)((m + 127) / 128) * ((n + 255) / 256);
  const uint64_t wide = (uint64_t)((m + 63) / 64) * ((n + 511) / 512);
  return split || wide < tall ? 64u : 128u;
}

// Workgroups, units and scratch of a product; false when another form is the better one.
bool plan_exact(krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t group, bool split,
                uint32_t& grid, UnitDeal& deal) {
  const uint64_t cus = (uint64_t)ctx->num_cus;
  const uint32_t bm = exact_rows(m, n, split), bn = 32768u / bm;
  const uint64_t tiles = (uint64_t)((m + bm - 1) / bm) * ((n + bn - 1) / bn);
  const uint32_t spt = (k + 127) / 128;
  const uint64_t units = tiles * spt;
  if (tiles > kTicketSlots || units > 0x7fffffffull || units < 2 * cus) return false;
  // fp16 x: the tiles staged through registers (gemm_i4.hip) start and end sooner and are the better ones
  // while a workgroup has few stages or ends a tile every few stages.  Over 64 products of 65 to 512 rows, time
  // here / there: 1.03 to 1.11 at a K of up to 768 in groups of 128 (1.05 at most in groups of 64), 0.93 to 0.98
  // from nine stages a workgroup and a K of 1280 on, 0.90 for 348 x 8164 x 4608.  The f32 class gains at any
  // length (265 x 26247 x 512 0.67).
  if (!split && (spt < 10 || units < 9 * cus)) return false;
  if (units < 12 * cus) {
    // Fewer than twelve stages a workgroup: the K-splitting tiles of gemm_i4_slices.hip, unless
    // their estimate is clearly above this form's, {fixed, a stage} in us, fitted over 16 to 30 shapes each
    // (rms 5 to 8 %).  (f32 x in groups of 64 had {37.1, 3.35} while the sum of its partials lay in scratch: over 60
    // shapes 0.88 of that time, 1.01 at worst; 440 x 11375 x 1536 68 / 50, 306 x 9645 x 3840 96 / 66.)  Over 192
    // shapes of 65 to 512 rows the f32 class takes 0.95 of the time that it took with its hi and lo made in the
    // loop, 1.02 at worst.
    struct Fit {
      float fixed, stage;
    };
    const bool wide_groups = group >= 128;
    const Fit f = split ? (wide_groups ? Fit{25.3f, 3.33f} : Fit{27.0f, 3.54f})
                        : (wide_groups ? Fit{16.4f, 2.26f} : Fit{15.4f, 2.47f});
    const float here = f.fixed + f.stage * ((float)units / (float)cus);
    if (here > 0.92f * slices_estimate_us(ctx, m, n, k, group, !split, split)) return false;
  }
  // Up to six 32 x 32 tiles of output a CU stay with the tiles that split K inside a workgroup, which
  // need no scratch with fp16 operands (a side branch of a graph may hold them) and give a row the
  // same bits whatever M is.
  if ((uint64_t)((m + 31) / 32) * ((n + 31) / 32) <= 6 * cus) return false;
  if (tiles * 8 < cus) return false;  // a tile shared by more than eight workgroups
  if (!ctx->gemm_partials) return false;
  deal.stages_per_tile = spt;
  deal.partials = ctx->gemm_partials;
  deal.tickets = ctx->tickets;
  // Workgroups of a tile's own, as many as the CUs give each tile: some walk more stages than with all units
  // dealt evenly, but none ends two tiles, each end a partial written and some of them merged behind the last
  // workgroup's.  That is worth up to five stages of one workgroup a tile, which exchanges nothing, four and a half
  // of several; two that share a tile of hi and lo, whose stages take longest, gained nothing.  us dealt
  // evenly / so (more stages): fp16 512 x 4096 x 11008 61.8 / 58.6 (0.5), 113 x 14557 x 7168 47.9 / 44.5 (0), 333 x 6000 x
  // 4992 40.3 / 38.9 (2), 280 x 10758 x 6592 71.0 / 68.3 (3.7), 348 x 8164 x 4608 43.2 / 42.7 (4.5), 346 x 7484 x 5120 43.5 /
  // 46.3 (5.9), one a tile 228 x 25350 x 3072 51.1 / 47.5 (5.3), 512 x 11008 x 4096 55.7 / 58.6 (10.5); hi and lo 512 x
  // 4096 x 11008 102.8 / 99.8 (0.5), 131 x 14091 x 8320 98.8 / 93.2 (0.7), 275 x 6187 x 6784 72.5 / 71.8 (4.5), one a
  // tile 200 x 27000 x 2048 62.9 / 60.5 (2.8), two 286 x 12123 x 4352 74.9 / 76.5 (1.1).
  const uint32_t sharers = (uint32_t)(cus / tiles);
  if (sharers > 0) {
    const float more = (float)((spt + sharers - 1) / sharers) - (float)units / (float)cus;
    if (more <= (sharers == 1 ? 5.4f : sharers > 2 ? 4.7f : split ? 0.6f : 4.6f)) {
      grid = sharers * (uint32_t)tiles;
      deal.tile_groups = sharers;
      deal.units_lo = spt / sharers;
      deal.extra = spt % sharers;
      return true;
    }
  }
  grid = (uint32_t)cus;
  deal.tile_groups = 0;
  deal.units_lo = (uint32_t)(units / cus);
  deal.extra = (uint32_t)(units % cus);
  return true;
}

struct ExactCall {
  const uint8_t *x, *w, *scales;
  const void* bias;
  void* out;
  uint32_t m, n, k, group_shift;
  const float* row_scale;
};

template <typename T, typename ST, int PLANES, bool HALF, int WM>
int32_t launch_exact(krm_ctx* ctx, const ExactCall& c, uint32_t grid, const UnitDeal& deal) {
  gemm_i4_exact_kernel<T, ST, PLANES, HALF, WM><<<dim3(grid), dim3(512), 0, ctx->stream>>>(
      c.x, c.w, c.scales, c.m, c.n, c.k, c.group_shift, (c.m + 64 * WM - 1) / (64 * WM),
      static_cast<const T*>(c.bias), static_cast<T*>(c.out), deal, c.row_scale);
  return launched(ctx, "gemm_i4_exact_kernel");
}

// T: of the bias and the result (f32 beside fp16 x: rows that were rounded before).
template <typename T, typename ST, bool HALF>
int32_t pick_exact(krm_ctx* ctx, const ExactCall& c, bool split, uint32_t grid, const UnitDeal& deal) {
  if constexpr (sizeof(T) == 4)
    if (split) return launch_exact<T, ST, 2, HALF, 1>(ctx, c, grid, deal);
  return exact_rows(c.m, c.n, false) == 64 ? launch_exact<T, ST, 1, HALF, 1>(ctx, c, grid, deal)
                                           : launch_exact<T, ST, 1, HALF, 2>(ctx, c, grid, deal);
}

}  // namespace

namespace krm {

// Whether fp16 x of this shape comes here (buffers aligned, main stream).
bool gemm_exact_takes_half(krm_ctx* ctx, uint32_t m, uint32_t n, uint32_t k, uint32_t group) {
  uint32_t grid = 0;
  UnitDeal deal{};
  return group >= 64 && (uint64_t)k * 256 <= 0xffffffffull && plan_exact(ctx, m, n, k, group, false, grid, deal);
}

// The exact-integer GEMM of fp16 x and of the f32 class for shapes whose (tile, stage) units cover the
// chip; sets *handled = false (and launches nothing) for every other shape.
int32_t linear_i4_gemm_exact(krm_ctx* ctx, krm_buf x, krm_buf w, krm_buf scales, krm_buf bias,
                             krm_buf out, uint32_t m, uint32_t n, uint32_t k, uint32_t group,
                             int32_t io_dtype, int32_t scale_dtype, int32_t compute,
                             bool* handled, int32_t x_dtype) {
  *handled = false;
  const bool split = compute == KRM_COMPUTE_F32 && io_dtype == KRM_F32;
  if (!split && x_dtype != KRM_F16) return KRM_OK;
  if (group < 64 || !aligned(w, 16) || !aligned(x, 16)) return KRM_OK;
  // (a side branch of a graph has no scratch: there the K-splitting tiles, which need none with fp16
  // operands, take these shapes too; the f32 class is refused there)
  if (!split && ctx->stream != ctx->main_stream) return KRM_OK;
  if (split && (m > kMaxSplitRows || !ctx->row_scales)) return KRM_OK;
  // rows at a time: the planes of f32 x fit their scratch, offsets inside a tile fit 32 bits
  const uint64_t row_bytes = split ? (uint64_t)(k + 127) / 128 * 512 : (uint64_t)k * 2;
  if (row_bytes * 128 > 0xffffffffull || (uint64_t)(k >> 1) * 512 > 0xffffffffull) return KRM_OK;
  uint32_t rows = m;
  if (split) {
    const uint64_t fit = kPlaneBytes / row_bytes / 128 * 128;
    if (fit == 0) return KRM_OK;
    if (fit < rows) rows = (uint32_t)fit;
  }
  uint32_t grid = 0;
  UnitDeal deal{};
  if (!plan_exact(ctx, rows, n, k, group, split, grid, deal)) return KRM_OK;
  KRM_TRY(needs_serial_scratch(ctx, "the unit-dealt GEMM"));
  *handled = true;
  for (uint32_t r = 0; r < m; r += rows) {
    ExactCall c{};
    c.m = m - r < rows ? m - r : rows;
    if (c.m < rows && !plan_exact(ctx, c.m, n, k, group, split, grid, deal)) {
      // (what is left of the rows has too few units: the last rows once more, as a whole block)
      r = m - rows;
      c.m = rows;
      plan_exact(ctx, rows, n, k, group, split, grid, deal);
    }
    c.x = ptr<const uint8_t>(x) + (size_t)r * k * dtype_bytes(x_dtype);
    c.w = ptr<const uint8_t>(w);
    c.scales = ptr<const uint8_t>(scales);
    c.bias = ptr<const void>(bias);
    c.out = ptr<uint8_t>(out) + (size_t)r * n * dtype_bytes(io_dtype);
    c.n = n;
    c.k = k;
    while ((1u << c.group_shift) < group) ++c.group_shift;
    c.row_scale = ctx->row_scales;
    if (split) {
      launch_split_rows(ctx, reinterpret_cast<const float*>(c.x), static_cast<uint4*>(ctx->x_planes), ctx->row_scales,
                        c.m, k, deal.stages_per_tile * 128u);
      KRM_TRY(launched(ctx, "split_rows_kernel"));
      c.x = static_cast<const uint8_t*>(ctx->x_planes);
    }
    auto by_group = [&](auto io, auto scale) {
      using T = decltype(io);
      using ST = decltype(scale);
      return group == 64 ? pick_exact<T, ST, true>(ctx, c, split, grid, deal)
                         : pick_exact<T, ST, false>(ctx, c, split, grid, deal);
    };
    const bool half_scales = scale_dtype == KRM_F16;
    if (io_dtype == KRM_F16)
      KRM_TRY(half_scales ? by_group(__half{}, __half{}) : by_group(__half{}, float{}));
    else
      KRM_TRY(half_scales ? by_group(float{}, __half{}) : by_group(float{}, float{}));
  }
  return KRM_OK;
}

}  // namespace krm
