// Operand helpers shared by the int4 group-128 kernels (skinny_int4.hip, skinny_int4_wide.hip).
#pragma once

#include "common.h"

namespace bp {

// The int4 matrix-core kernel of any number of activation rows (skinny_int4_wide.hip): activation blocks of 16 per
// workgroup (nb: 1, 2), tile rows, waves, scale dtype, epilogue (0: the product, 1: the gate|up SiLU product); or null.
using Int4WideFn = void (*)(const uint16_t*, const uint8_t*, const void*, const uint16_t*, uint16_t*, float*, int, int64_t,
                            int64_t, int);
Int4WideFn int4_wide_pick(int nb, int tile_rows, int waves, int scale_dt, int epi);

// Activation blocks per workgroup of a launch, or 0 where skinny_int4.hip's kernel runs it (the same bits). A few rows of a
// long K in 16-row tiles are its: its waves have four groups in flight, the wide kernel's two. us on one MI355X, that
// kernel / the wide one, by the groups a wave walks (any number of tiles): 4 groups (2048 x 2048 in 128 tiles) one row 4.1
// / 4.3, two 4.3 / 4.3, four 4.7 / 4.4; 8 groups (4096 x 4096 in 256) one row 5.3 / 6.1, five 5.8 / 6.1, eight 6.7 / 6.1;
// 16 (2048 x 8192) one row 7.0 / 9.0, five 7.7 / 9.0, eight 9.3 / 9.0; 2 groups (4096 x 1024) 4.0 / 3.6. In tiles of 32
// and 64 rows the wide kernel is the faster at one row already (6144 x 4096 7.9 / 6.7, 64000 x 2048 19.3 / 18.0; 8192 x
// 8192 11.7 / 11.9). Two blocks per workgroup read the codes once for 32 rows and take about 1.8 times one block's time:
// by the rounds of workgroups over 256 CUs (8192 x 2048 at 33 rows, three blocks: one 8.7 us, two 10.4; at 20 rows 7.4
// and 6.7).
inline int int4_wide_nb(int64_t M, int64_t K, int64_t tiles, int tile_rows, int waves, int split) {
  const int64_t per_wave = K / 128 / (static_cast<int64_t>(waves) * split);
  if (tile_rows == 16 && ((M < 8 && per_wave >= 8) || (M <= 2 && per_wave >= 4))) return 0;
  const int64_t blocks = (M + 15) / 16;
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
