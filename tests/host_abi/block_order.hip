// The block order of the z-stencil passes by size: every logical block is
// launched once in each, and a convection step too small to gain from ranges
// of planes keeps the order of its temperature pass.
#include <cstdio>

#include "../../pour-over-coffee-lbm_amd/csrc/lbm_common.h"

using namespace pol;

static int failed = 0;
static void check(bool ok, const char* what, uint64_t cells) {
  if (!ok) {
    printf("%s: %llu cells\n", what, (unsigned long long)cells);
    failed = 1;
  }
}

// ordered_block of physical block b, restated
static uint32_t logical(const BlockOrder& o, uint32_t b) {
  if (o.order == ORDER_LINEAR) return b;
  if (o.order == ORDER_XCD_RANGES) return (b % NXCD) * o.per_xcd + b / NXCD;
  const uint32_t G = 1u << o.order, S = NXCD * G;
  return (b / S) * S + (b % NXCD) * G + (b / NXCD) % G;
}

int main() {
  for (uint64_t cells : {8ull, 255ull, 256ull, 257ull, 2047ull, 2048ull, 2049ull, 64ull * 64 * 64, 96ull * 96 * 96,
                         181ull * 97 * 53, 80ull * 80 * 80, 120ull * 121 * 122, 151ull * 150 * 149, 210ull * 211 * 212}) {
    for (uint64_t real : {4ull, 8ull}) {
      const uint64_t bytes = 20 * real * cells;
      const BlockOrder o = stencil_order(cells, bytes, CONVECTION_LINEAR_BYTES);
      check((o.order == ORDER_LINEAR) == (bytes < CONVECTION_LINEAR_BYTES), "linear below the limit only", cells);
      check(stencil_order(cells, bytes).order != ORDER_LINEAR, "without a limit never linear", cells);
      const uint32_t n = launch_blocks(o);
      uint64_t sum = 0, seen = 0;
      for (uint32_t b = 0; b < n; ++b) {
        const uint32_t l = logical(o, b);
        if (l >= o.nblk) continue;
        ++seen;
        sum += l;
      }
      check(seen == o.nblk && sum == (uint64_t)o.nblk * (o.nblk - 1) / 2, "every block once", cells);
    }
  }
  // the sizes that lost in ranges are linear, those that gained are not
  for (uint64_t n : {32, 48, 64, 80, 96}) check(stencil_order(n * n * n, 80 * n * n * n, CONVECTION_LINEAR_BYTES).order == ORDER_LINEAR, "FP32", n);
  for (uint64_t n : {32, 48, 64, 72}) check(stencil_order(n * n * n, 160 * n * n * n, CONVECTION_LINEAR_BYTES).order == ORDER_LINEAR, "FP64", n);
  for (uint64_t n : {104, 112, 128, 144}) check(stencil_order(n * n * n, 80 * n * n * n, CONVECTION_LINEAR_BYTES).order == ORDER_XCD_RANGES, "FP32", n);
  for (uint64_t n : {80, 96, 112}) check(stencil_order(n * n * n, 160 * n * n * n, CONVECTION_LINEAR_BYTES).order == ORDER_XCD_RANGES, "FP64", n);
  return failed;
}
