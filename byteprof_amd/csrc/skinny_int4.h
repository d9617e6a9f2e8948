// Operand helpers shared by the int4 group-128 kernels (skinny_int4.hip, skinny_int4_wide.hip).
#pragma once

#include "common.h"

namespace bp {

// The int4 matrix-core kernel of 1..64 activation rows (skinny_int4_wide.hip): activation blocks of 16 per workgroup (nb:
// 1, 2), tile rows, waves, scale dtype, epilogue (0: the product, 1: the gate|up SiLU product); or null.
using Int4WideFn = void (*)(const uint16_t*, const uint8_t*, const void*, const uint16_t*, uint16_t*, float*, int, int64_t,
                            int64_t, int);
Int4WideFn int4_wide_pick(int nb, int tile_rows, int waves, int scale_dt, int epi);

// Activation blocks per workgroup of a launch, or 0 where skinny_int4.hip's kernel runs it (the same bits). A few rows of
// few tiles are its: its waves have more groups in flight (one row of 2048 x 8192 in 128 tiles 6.6 us, wide 8.6; five
// rows 7.8 and 8.7, nine 9.0 and 8.8; but 2048 x 2048 five rows 4.3 and 4.0, and in 256 tiles 8192 x 2048 one row 5.3 and
// 4.8). Two blocks per workgroup read the codes once for 32 rows and take about 1.8 times one block's time: by the
// rounds of workgroups over 256 CUs (8192 x 2048 at 33 rows, three blocks: one 8.7 us, two 10.4; at 20 rows 7.4 and 6.7).
inline int int4_wide_nb(int64_t M, int64_t K, int64_t tiles) {
  const int64_t blocks = (M + 15) / 16;
  if (M <= 8 && tiles < 256 && (M <= 4 || K >= 4096)) return 0;
  if (blocks == 1) return 1;
  const int64_t one = (tiles * blocks + 255) / 256, two = (tiles * ((blocks + 1) / 2) + 255) / 256;
  return 10 * one <= 18 * two ? 1 : 2;
}

constexpr uint32_t kBf16Exp128 = 0x43434343u;  // 0x43 in every byte: bf16 0x43xx = 128 + xx
constexpr uint32_t kBf16OnePair = 0x3F803F80u; // two bf16 1.0

// Four codes (bytes of m, each below 128) as two bf16 pairs (128 + byte).
__device__ __forceinline__ void codes_to_bf16(uint32_t m, uint32_t& p01, uint32_t& p23) {
  // v_perm_b32 (S0 = m: bytes 4..7, S1 = 0x43434343: bytes 0..3): result bytes [m0, 0x43, m1, 0x43] / [m2, .., m3, ..]
  p01 = __builtin_amdgcn_perm(m, kBf16Exp128, 0x00050004u);
  p23 = __builtin_amdgcn_perm(m, kBf16Exp128, 0x00070006u);
}

__device__ __forceinline__ float half_bits_to_float(uint32_t h) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(h)));
}

using u32x2 = unsigned __attribute__((ext_vector_type(2)));

}  // namespace bp
