// How the products of gemv_i4_rows.hip are dealt: nothing of the device, so that a test can ask which form a shape takes.
#pragma once

#include <algorithm>
#include <cstdint>

namespace krm {
namespace {

constexpr uint32_t kRowsWave = 64;
constexpr uint32_t kSegment = 32;   // codes of a chain
constexpr uint32_t kQuad = 4;       // neighbouring segments a lane walks together
constexpr uint32_t kMaxUnits = 8;   // waves a workgroup

// Positions of the sixteen quads in the order in which the tree adds them: of four neighbours 0 and 3, 1 and 2, then both.
constexpr uint32_t quad_at(uint32_t position) {
  return (position & ~3u) | ((0x2130u >> (4 * (position & 3u))) & 3u);
}

constexpr uint32_t kLds = 160 * 1024;

// How a call is dealt: SPAN, R, `deal` and what follows from them.
struct RowsPlan {
  uint32_t span, rows, deal, units, scale_area, lds, blocks, row_blocks;
  float us;
};

// The vector ALU bounds a wave: I = 300 + 146 R instructions a stage for f32 x (64 R products in each of two passes, 240
// to convert the codes), 220 + 88 R for fp16.  A SIMD issues one in 7 clk for a lone wave, in 5.3 for two and 5.0 for
// more (products with a row broadcast alone: 7.1, 5.4, 4.9).  A CU's time is that of its longest wave or of all its
// waves, once for every time the grid fills the chip and once for the rest; a latency each.  Wide N wants many rows of x
// a wave, few rows of W (N below 4096) wants many workgroups, of 16 rows of W and few of x.  Over 106 shapes (2 to 16 rows,
// N 256 to 32000, K 512 to 11008) the form with the smallest estimate was 2 % slower than the fastest of the nine.
inline RowsPlan plan_rows(uint32_t x_size, uint32_t scale_size, uint32_t cus, uint32_t m, uint32_t n, uint32_t k,
                          uint32_t group_shift) {
  static constexpr uint32_t kForms[][3] = {{1, 8, 1}, {1, 8, 4}, {1, 4, 1}, {1, 4, 4}, {1, 2, 1},
                                           {4, 5, 1}, {4, 3, 1}, {4, 2, 1}, {4, 1, 1}};
  const uint32_t segments = k / kSegment, groups = k >> group_shift;
  auto steps = [&](uint32_t quad) { return quad * kQuad < segments ? (segments - quad * kQuad + 63) / 64 : 0u; };
  uint32_t last = 0;  // position of the tree's last quad that has a segment
  for (uint32_t position = 0; position < 16; ++position)
    if (steps(quad_at(position))) last = position;
  RowsPlan best{};
  for (const auto& form : kForms) {
    RowsPlan p{};
    p.span = form[0];
    p.row_blocks = (m + form[1] - 1) / form[1];
    p.rows = (m + p.row_blocks - 1) / p.row_blocks;
    if (p.rows == 7) p.rows = 8;
    if (p.span == 1 && p.rows == 1) continue;
    p.deal = form[2];
    while (last / (p.deal * p.span) + 1 > kMaxUnits) p.deal *= 2;
    p.units = last / (p.deal * p.span) + 1;
    const uint32_t tile = kRowsWave / p.span, tiles = (n + tile - 1) / tile;
    p.blocks = tiles * p.row_blocks;
    const uint64_t scale_bytes = (uint64_t)std::min(tile, n) * groups * scale_size;
    const uint32_t x_bytes = p.rows * p.span * kQuad * kSegment * x_size;
    const uint32_t stage = kRowsWave * 64 + (x_bytes + 1023) / 1024 * 1024, ring = p.units * 2 * stage;
    p.scale_area = ring + scale_bytes + 1023 > kLds ? 0u : (uint32_t)((scale_bytes + 1023) & ~(uint64_t)1023);
    p.lds = ring + p.scale_area;

    const float instructions = x_size == 4 ? 300.f + 146.f * p.rows : 220.f + 88.f * p.rows;
    uint32_t longest = 0, total = 0;  // stages of the first wave and of all
    for (uint32_t t = 0; t < p.deal; ++t) longest += steps(quad_at(t * p.span));
    for (uint32_t position = 0; position <= last; position += p.span) total += steps(quad_at(position));
    const uint32_t waves = p.rows <= 3 ? 20 : p.rows <= 5 ? 16 : 12;  // of a CU, by registers
    const uint32_t together = std::max(1u, std::min(kLds / p.lds, waves / p.units));
    auto clk = [&](uint32_t workgroups) {
      const float in_flight = workgroups * p.units * 0.25f, issue = in_flight <= 1 ? 7.f : in_flight <= 2 ? 5.3f : 5.f;
      return instructions * std::max(longest * 7.f, workgroups * total * 0.25f * issue) + 1200.f;
    };
    const uint32_t rest = p.blocks % (cus * together);
    const float alu = (p.blocks / (cus * together)) * clk(together) + (rest ? clk((rest + cus - 1) / cus) : 0.f);
    const float to_lds = (float)p.blocks * total * stage / (cus * 40.f);  // 40 bytes a clk a CU
    p.us = std::max(std::max(alu, to_lds) / 2300.f, (float)n * k / 1e7f + 0.3f);
    if (!best.rows || p.us < best.us) best = p;
  }
  return best;
}

// Which products are dealt.
// 2 rows: where the one-row kernel's form is the slower one.  us there / here: f32 1093 x 1920 5.4 / 4.1, 4806 x 1152
// 6.4 / 5.2, 7309 x 2560 8.4 / 7.7, 32000 x 4096 27.5 / 23.7, 1300 x 1024 4.2 / 3.9, but 1100 x 512 3.6 / 3.7, 701 x 576
// 3.0 / 3.8, 1945 x 3328 4.8 / 5.3, 4096 x 4096 6.42 / 6.44; fp16 548 x 8064 4.6 / 5.9, 6085 x 3840 6.9 / 7.2.  3 fp16 rows
// 422 x 2496 4.2 / 4.8, 2040 x 768 4.4 / 4.7, 1114 x 2016 4.9 / 4.5, 2453 x 544 5.1 / 4.7, 1977 x 3200 6.4 / 5.75, 3032
// x 704 4.4 / 4.0.  4 fp16 rows 388 x 2208 4.5 / 5.2, 700 x 5632 5.75 / 6.2, 1000 x 1024 3.94 / 4.3, 1455 x 640 4.37 /
// 4.69, 1932 x 512 4.44 / 4.30, 1740 x 1408 4.76 / 4.87, 1741 x 1600 4.92 / 4.74, 2152 x 640 5.4 / 5.0, 1955 x 3968 6.3 / 5.2.  3 f32
// rows and more, all faster here: 428 x 4480 6.7 / 6.1.
inline bool rows_dealt(bool f32, uint32_t m, uint32_t n, uint32_t k, uint32_t group) {
  if (m < 2 || m > 16 || k % kSegment || group < kSegment) return false;
  if (m == 2 && (!f32 || n < (k < 2048 ? 1024u : 6144u) || (uint64_t)n * k < 1250000)) return false;
  if (!f32 && m <= 4 && (n < 1024 || (n < 2048 && k > 512 && k <= 1536))) return false;
  return (uint64_t)kRowsWave * k <= 0x7fffffffull && n <= 0x7fffffffu / 16;  // offsets of 32 bits
}

}  // namespace
}  // namespace krm
