// The matrix-core skinny matmul from 9 activation rows on: the sums of skinny_mf.h (same K segments, same halves, same
// waves, same order, so the same bits), with full MFMA tiles and coalesced operand loads.
//
// skinny_mf.h carries the two halves of a segment's K slots in one 16 x 16 tile (8 weight rows x 8 activation rows x 2
// halves, half of the tile unused), and loads every operand in MFMA lane order (neighbouring lanes in different rows):
// right at one row, where the weights come from memory at the rate of the card. From about 9 rows the activations
// are what a workgroup takes in most, and a load whose neighbouring lanes touch different lines takes the address unit
// four times as long: 26 GB/s per CU, whatever the tile. Here:
//   - a wave takes weight rows in blocks of 16 and activation rows in blocks of 16, with one accumulator per half h:
//     half h's adds, for K slot (g, e), the products that skinny_mf.h's half h adds in the same slot of the same MFMA,
//     segment after segment, so D0 + D1 is its folded tile, bit for bit, with half the MFMAs and half the operands;
//   - a load reads 1 KiB of whole lines in lane order, and a pass through the wave's own LDS patch (16 rows x a segment,
//     swizzled, no barrier) turns it into the operands: lane (g = l / 16, i = l % 16) needs bytes 16 (2 g + h) of row i.
// 64 rows, one MI355X, before -> now: bf16 100352 x 2048 230 -> 101 us, 8192 x 2048 22.4 -> 12.7, 2048 x 8192 36.2 ->
// 16.1; int8 223 -> 78, 21.5 -> 10.3, 35.1 -> 13.7.
//
// Reference semantics: byteprof/optim/skinny.py:36-90, via skinny_mm (skinny.py:136-166).
#pragma once

#include <algorithm>

#include "byteprof_amd.h"
#include "skinny_mf.h"

namespace bp {

using MfWideFn = void (*)(const uint16_t*, const uint8_t*, const void*, int, uint16_t*, float*, int, int64_t, int64_t,
                          int);

// The kernel for activation blocks of 16 per workgroup (mb), weight blocks of 16 per wave (rp), waves sharing K (1, 2, 4,
// 8) and epilogue (0: y or partials, 1: the gate|up SiLU product), or null.
MfWideFn mf_wide_pick(int wkind, int mb, int rp, int waves, int epi);

// Most activation blocks of a workgroup at rp weight blocks: what stays in registers (int8's activation segments are
// twice as long).
constexpr int mf_wide_max_mb(int wkind, int rp) { return wkind == kBf16 ? 4 : rp == 4 ? 2 : 3; }

// The workgroup tile of a launch. A CU's time goes to the 16-row operand segments it takes in (weights: one per weight
// block, activations: one per activation block, two for int8, whose K segments are twice as long): the tile with the
// least of them per CU, ceil(workgroups / 256) x (rp + mb) or (rp + 2 mb), and of equals the one with fewer activation
// tiles (each reads the weights again). 64 weight rows only where no CU is left without a workgroup. Measured over
// (rp, mb) on one MI355X: bf16 2048 x 2048 at 64 rows (1, 2) 6.3 us, (1, 4) 8.2, (2, 4) 10.2, (4, 4) 16.1; 100352 x 2048
// at 64 rows (4, 4) 101 us, (2, 4) 113, (1, 4) 148, (4, 2) 154; int8 8192 x 2048 at 64 rows (4, 2) 10.3 us, (2, 2) 11.6,
// (1, 2) 14.9: the rule's choice is the fastest or within a few percent of it at every size timed.
struct MfWideTile {
  int rp, mb;
  int64_t wgs;  // grid.x
};
inline MfWideTile mf_wide_tile(int wkind, int64_t M, int64_t N, int split) {
  const int64_t blocks = (M + 15) / 16;
  MfWideTile best{0, 0, 0};
  int64_t best_cost = 0;
  for (int rp = 4; rp >= 1; rp /= 2)
    for (int64_t mb = std::min<int64_t>(blocks, mf_wide_max_mb(wkind, rp)); mb >= 1; --mb) {
      const int64_t mt = (blocks + mb - 1) / mb;
      const int64_t wt = (N + 16 * rp - 1) / (16 * rp);
      const int64_t tiles = wt * mt * split;
      if (rp == 4 && (tiles < 256 || blocks == 1)) continue;
      const int64_t cost = ((tiles + 255) / 256 * (rp + (wkind == kBf16 ? mb : 2 * mb))) * 8 + mt;
      if (best.rp == 0 || cost < best_cost) {
        best_cost = cost;
        best = MfWideTile{rp, static_cast<int>(mb), (wt + kXcds - 1) / kXcds * kXcds * mt};
      }
    }
  return best;
}

}  // namespace bp
