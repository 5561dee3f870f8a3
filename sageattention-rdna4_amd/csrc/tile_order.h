// The order in which a causal grid's query tiles start (host and device; no HIP dependency, so that
// a host program can check it to be a permutation).
//
// A causal tile's length grows with its row, so the order decides how long the card waits for the
// last tiles. Blocks are dispatched in the order of their number, block b to XCD b % 8. Each XCD
// takes whole planes (their K/V tiles are then read through one L2), P = BH / 8 of them, and
// starts their tiles longest first over all P planes at once; taking one plane after the other, as
// before, the last plane's longest tiles began when the others had nearly ended.
// Measured (main loop, us, before / after; fp16, head_dim 128 unless said): 32 heads of 3001 rows
// 88.1 / 67, 32 of 2048 62.9 / 44.7, 24 of 4096 154.5 / 90, 48 of 1024 35.7 / 26.5, 48 of 8771
// 718 / 700, head_dim 64, 32 of 4096 165.6 / 85. Calls of few rounds gain most, long ones little
// (48 of 16384 2146 / 2127).
#pragma once

#if defined(__HIPCC__)
#define SAGE_HD __host__ __device__ __forceinline__
#else
#define SAGE_HD inline
#endif

namespace sage {

constexpr int XCDS = 8, XCD_CUS = 32;   // MI355X: 256 CUs in 8 XCDs

struct CausalTile {
  int bh;     // plane
  int rank;   // 0: the plane's longest tile, num_qt - 1: its shortest
};

// Tile of block `block` of a grid of BH * num_qt blocks; span = BH * num_qt rounded down to a
// multiple of 8. `resident`: blocks of the kernel that a CU holds at once.
SAGE_HD CausalTile causal_tile(int block, int span, int num_qt, int resident) {
  const int per = (int)((unsigned)span / XCDS);   // blocks per XCD
  if (per <= XCD_CUS) {
    // A CU for each block: the order does not matter (and the divisions below are 0.3 us of a
    // 12 us call), so planes stay together.
    const unsigned u = (unsigned)block;
    const unsigned id = block < span ? (u % XCDS) * per + u / XCDS : u;
    const unsigned bh = id / (unsigned)num_qt;
    return {(int)bh, (int)(id - bh * num_qt)};
  }
  if (per % num_qt == 0 && block < span) {
    const int P = per / num_qt, x = block % XCDS;
    int i = block / XCDS;        // the XCD's i-th block
    // Blocks that start together: the first XCD_CUS of them, the longest, take a CU each, the next
    // XCD_CUS join them, and so on. Where two or three are resident, the second and third share of
    // them go to the CUs in an order that evens out the sums (in descending order the first CU
    // would get the longest of each: 32 heads of 3001 rows 73.9 us, so 67).
    const int k = i / XCD_CUS, c = i % XCD_CUS, h = c / 2;
    if (resident >= 3 && per >= 3 * XCD_CUS) {
      if (k == 1) i = XCD_CUS + ((c & 1) ? 15 - h : 31 - h);
      if (k == 2) i = 2 * XCD_CUS + ((c & 1) ? (h == 15 ? 31 : 30 - h) : 15 - h);
    } else if (resident >= 2 && per >= 2 * XCD_CUS && k == 1) {
      i = 2 * XCD_CUS + XCD_CUS - 1 - i;
    }
    // Longest first over G planes at a time: enough that the last group's tiles fill every slot
    // four times, no more, as all G planes' K/V are then in use at once. The first group takes
    // what is left over.
    const int want = (4 * XCD_CUS * resident + num_qt - 1) / num_qt;
    const int G = want < P ? want : P;
    const int first = (P - 1) % G + 1;
    int p0 = 0, g = first;
    if (i >= first * num_qt) {
      i -= first * num_qt;
      const int n = i / (G * num_qt);
      i -= n * (G * num_qt);
      p0 = first + n * G;
      g = G;
    }
    return {x * P + p0 + i % g, i / g};
  }
  if (per % num_qt != 0 && num_qt >= XCDS) {
    // Planes that do not share out evenly over the XCDs: longest first over all of them. The grid
    // has BH * num_qt blocks, fewer than num_qt beyond span.
    const int BH = (span + num_qt - 1) / num_qt;
    return {block % BH, block / BH};
  }
  return {block / num_qt, block % num_qt};
}

}  // namespace sage
