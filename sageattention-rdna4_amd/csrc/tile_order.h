// The order in which a causal grid's query tiles start (host and device; no HIP dependency, so that
// a host program can check it to be a permutation).
//
// A causal tile's length grows with its row, so the order decides how long the card waits for the
// last tiles. Blocks are dispatched in the order of their number, block b to XCD b % 8. Each XCD
// takes whole planes, P = BH / 8 of them (their K/V tiles are then read through one L2), and an
// eighth of the tiles of the BH % 8 planes left over, and starts them longest first, over as many
// of the P planes at once as fill its slots a few times; taking one plane after the other, the last
// plane's longest tiles would begin when the others had nearly ended.
// Measured (main loop, us, plane after plane / this; fp16, head_dim 128 unless said): 32 heads of
// 3001 rows 91.9 / 69.1, 24 of 4096 152 / 88, 48 of 1024 36.3 / 26.2, 48 of 8771 743 / 702. With
// planes left over (in between: all planes' tiles over all XCDs at once): 10 heads of 16384
// 703 / 511 / 499, 28 of 4096 153 / 111 / 102, 30 of 8192 479 / 415 / 386, 250 of 300
// 21.4 / 22.7 / 19.7, 250 of 8192 3691 / 3703 / 3196 (their K/V, 520 MB, no longer all in use at
// once), 3 of 32768 939 / 688 / 603; head_dim 64, 28 of 4096 162 / 83.5 / 74.3, 250 of 300
// 14.5 / 16.0 / 13.6.
#pragma once

#if defined(__HIPCC__)
#define SAGE_HD __host__ __device__ __forceinline__
#else
#define SAGE_HD inline
#endif

namespace sage {

constexpr int XCDS = 8, XCD_CUS = 32;   // MI355X: 256 CUs in 8 XCDs (a partition has fewer XCDs: the
                                        // eight shares then mix on them, each longest first)

struct CausalTile {
  int bh;     // plane
  int rank;   // 0: the plane's longest tile, num_qt - 1: its shortest
};

// Tile of block `block` of a grid of `blocks` blocks, num_qt tiles in each of its planes. `resident`:
// blocks of the kernel that a CU holds at once. (Given a number that is no multiple of num_qt, the
// planes are counted up from it; blocks past them take their tiles plane by plane.)
SAGE_HD CausalTile causal_tile(int block, int blocks, int num_qt, int resident) {
  const unsigned qt = (unsigned)num_qt, u = (unsigned)block;
  const unsigned x = u % XCDS;
  unsigned i = u / XCDS;                             // the XCD's i-th block
  const unsigned per = (unsigned)blocks / XCDS;      // blocks of an XCD, or one more
  if (__builtin_expect(per <= XCD_CUS, 1)) {
    // A CU for each block: the order does not matter, so planes stay together. (The branch that is
    // expected, so that these calls run straight on: instructions are fetched anew in a short one.)
    const unsigned id = u < per * XCDS ? x * per + i : u;
    const unsigned bh = id / qt;
    return {(int)bh, (int)(id - bh * qt)};
  }
  const unsigned BH = ((unsigned)blocks + qt - 1) / qt;
  if (u >= BH * qt) return {(int)(u / qt), (int)(u % qt)};
  // Each XCD takes P whole planes. The R planes that are left over are dealt out tile by tile,
  // longest first: tile t of them to XCD t % 8 (R = 1, 2 or 4: one of those planes per XCD).
  const unsigned P = BH / XCDS, R = BH % XCDS;
  // Blocks that start together: the first XCD_CUS of them, the longest, take a CU each, the next
  // XCD_CUS join them, and so on. Where two or three are resident, the second and third share of
  // them go to the CUs in an order that evens out the sums (in descending order the first CU
  // would get the longest of each: 32 heads of 3001 rows 73.9 us, so 67).
  const unsigned k = i / XCD_CUS, c = i % XCD_CUS, h = c / 2;
  if (resident >= 3 && per >= 3 * XCD_CUS) {
    if (k == 1) i = XCD_CUS + ((c & 1) ? 15 - h : 31 - h);
    if (k == 2) i = 2 * XCD_CUS + ((c & 1) ? (h == 15 ? 31 : 30 - h) : 15 - h);
  } else if (resident >= 2 && per >= 2 * XCD_CUS && k == 1) {
    i = 2 * XCD_CUS + XCD_CUS - 1 - i;
  }
  if (P == 0) {
    const unsigned t = XCDS * i + x, rank = t / R;
    return {(int)(t - rank * R), (int)rank};
  }
  // Longest first over G planes at a time: enough that the last group's tiles fill every slot four
  // times, no more, as all G planes' K/V are then in use at once. The first group has what is left
  // over of the P planes, and the XCD's tiles of the R planes.
  const unsigned slots = 4 * XCD_CUS * (unsigned)resident;
  unsigned G = P, first = P;
  if (P * qt > slots) {
    const unsigned want = (slots + qt - 1) / qt;
    G = want < P ? want : P;
    first = (P - 1) % G + 1;
  }
  // In the first group the tiles of rank r follow the `first` planes' tiles of each lower rank and
  // rest(r) tiles of the R planes (at most one of each rank, ahead of the others of that rank).
  auto rest = [&](unsigned r) { return (r * R + XCDS - 1 - x) / XCDS; };
  if (i < first * qt + rest(qt)) {
    unsigned r = XCDS * i / (XCDS * first + R);   // the rank, or one less
    if (i >= first * (r + 1) + rest(r + 1)) ++r;
    const unsigned before = rest(r), one = rest(r + 1) - before, at = i - first * r - before;
    if (at < one) return {(int)(XCDS * P + XCDS * before + x - r * R), (int)r};
    return {(int)(x * P + at - one), (int)r};
  }
  i -= first * qt + rest(qt);
  const unsigned n = i / (G * qt);
  i -= n * (G * qt);
  const unsigned rank = i / G;
  return {(int)(x * P + first + n * G + i - rank * G), (int)rank};
}

}  // namespace sage
