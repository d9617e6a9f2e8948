// The int4 matrix-core kernel for any number of activation rows in one launch: skinny_int4.hip's groups, waves and sums
// (an output is the same bits), with NB blocks of 16 activation rows as the MFMA's B columns, so a verify pass or a
// prompt of more than 16 rows streams the codes and decodes them once (or once per 32 rows).
//
// What bounds it is the activations: a group is 1 KiB of codes per 16 weight rows, and 4 KiB of activations per 16
// activation rows. They are loaded as whole 256-byte rows in lane order and turned into operands through the wave's own
// LDS patch (16 rows x 128 K, pieces swizzled by the row, no barrier): loaded in operand order, with neighbouring lanes
// in different rows, the address unit takes four times as long. us on one MI355X, before (launches of 16 rows by
// skinny_int4.hip) -> now: 64 rows of 2048 x 2048 25.3 -> 5.7, 8192 x 2048 31.5 -> 10.9, 2048 x 8192 50.1 -> 12.5, 100352 x
// 2048 120 -> 59; 16 rows 6.5 -> 4.2, 8.1 -> 5.3, 12.6 -> 8.9, 33.0 -> 26.3.
//
// Reference semantics: byteprof/optim/skinny.py:46-63 (MODE 3 kernel), through skinny_mm (skinny.py:136-166).

#include "byteprof_amd.h"
#include "skinny_int4.h"

namespace bp {
namespace {

template <int RB, int NB, int WAVES, int DEPTH, int SDT, int EPI>
__global__ __launch_bounds__(WAVES* kWave, 2) void skinny_int4_wide_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w, const void* __restrict__ scale,
    const uint16_t* __restrict__ zero, uint16_t* __restrict__ y, float* __restrict__ ws, int M_all, int64_t N,
    int64_t K, int split) {
  using floatx4 = float __attribute__((ext_vector_type(4)));
  using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
  constexpr int R = 16 * RB;
  constexpr bool f32 = SDT == BP_DT_F32;
  constexpr int SEB = f32 ? 4 : 2;
  constexpr int kScDw = R * SEB / 4, kRecDw = kScDw + R / 2;  // dwords of a record's scales / of the whole record
  constexpr int kRecLoads = (kRecDw + kWave - 1) / kWave;
  constexpr uint32_t kPast = 0x80000000u;  // beyond the activations' resource
  __shared__ __align__(16) union {
    float red[WAVES][R][16];
    uint8_t patch[WAVES][4096];
  } sh;
  __shared__ __attribute__((aligned(16))) uint32_t stage[WAVES][kRecLoads * kWave];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // uniform: the group loop is scalar
  const int i = lane & 15, kb = lane >> 4;
  // each XCD (workgroups go to the 8 in turn) takes one contiguous run of weight tiles, as skinny_int4.hip, and a tile's
  // activation tiles one after the other, so that its codes meet in that XCD's L2
  const int64_t T = (N + R - 1) / R;
  const uint32_t mtiles = (M_all + 16 * NB - 1) / (16 * NB);
  const uint32_t xcd = blockIdx.x % kXcds, at = blockIdx.x / kXcds;
  const int64_t run = T / kXcds + (xcd < T % kXcds ? 1 : 0);
  if (at / mtiles >= run) return;  // the grid covers the longest run on every XCD (the whole workgroup)
  const int64_t tb = xcd * (T / kXcds) + min(static_cast<int64_t>(xcd), T % kXcds) + at / mtiles;
  const int m0 = static_cast<int>(at % mtiles) * (16 * NB);  // the workgroup's activation rows
  const int M = min(M_all - m0, 16 * NB);
  const int64_t n0 = tb * R;
  const int64_t G = K / 128;
  const int s = blockIdx.y;
  const int64_t g_lo = split == 1 ? 0 : s * G / split;
  const int64_t g_hi = split == 1 ? G : (s + 1) * G / split;
  const int64_t first = g_lo + wave;
  const int cnt = first < g_hi ? static_cast<int>((g_hi - first + WAVES - 1) / WAVES) : 0;
  const uint8_t* tile = w + tb * G * R * 64 + i * 64 + kb * 16;
  // K < 2^24 and M <= 16 NB <= 32 (the workgroup's rows): 2 M K < 2^30; a row past M has an offset past the resource
  // (zeros, no memory request)
  static_assert(NB <= 2, "activation bytes below 2^31");
  const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(x + m0 * K, static_cast<int>(2 * M * K));
  uint32_t xoff[NB][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = 16 * b + 4 * u + kb;
      xoff[b][u] = m < M ? static_cast<uint32_t>(2 * m * K + 16 * i) : kPast;
    }
  // a group's record [R scales | R zeros (fp16)] of the tile's rows: dword 64 c + lane at rsrc[c] + g * rstride[c]
  // (lanes past it repeat its last dword; rows past N read row N - 2 of the group, never stored)
  const uint8_t* rsrc[kRecLoads];
  int64_t rstride[kRecLoads];
#pragma unroll
  for (int c = 0; c < kRecLoads; ++c) {
    const int p = min(c * kWave + lane, kRecDw - 1);
    if (p < kScDw) {
      const int64_t r0 = n0 + p * 4 / SEB;
      rsrc[c] = static_cast<const uint8_t*>(scale) + (r0 < N ? r0 : N - 4 / SEB) * SEB;
      rstride[c] = N * SEB;
    } else {
      const int64_t r0 = n0 + 2 * (p - kScDw);
      rsrc[c] = reinterpret_cast<const uint8_t*>(zero + (r0 < N ? r0 : N - 2));
      rstride[c] = N * 2;
    }
  }

  struct Slot {
    u32x4 wv[RB];
    u32x4 xv[NB][4];
    uint32_t rv[kRecLoads];
  };
  auto load = [&](Slot& sl, int j) {
    const int64_t g = first + static_cast<int64_t>(j) * WAVES;
#pragma unroll
    for (int h = 0; h < RB; ++h)
      sl.wv[h] = __builtin_nontemporal_load(as_global(reinterpret_cast<const u32x4*>(tile + (g * R + 16 * h) * 64)));
#pragma unroll
    for (int c = 0; c < kRecLoads; ++c)
      sl.rv[c] = *as_global(reinterpret_cast<const uint32_t*>(rsrc[c] + g * rstride[c]));
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        sl.xv[b][u] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[b][u] + static_cast<uint32_t>(256 * g), 0, 0));
  };

  float acc[RB][NB][4];
#pragma unroll
  for (int h = 0; h < RB; ++h)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[h][b][r] = 0.f;

  uint32_t* st = stage[wave];
  uint8_t* patch = sh.patch[wave];
  auto compute = [&](Slot& sl) {
    // the wave's LDS operations run in order: a write lands after the reads before it
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = 4 * u + kb;
        *reinterpret_cast<u32x4*>(patch + r * 256 + 16 * (i ^ r)) = sl.xv[b][u];
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int piece = 8 * (c / 2) + 2 * kb + c % 2;
        sl.xv[b][c] = *reinterpret_cast<const u32x4*>(patch + i * 256 + 16 * (piece ^ i));
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int c = 0; c < kRecLoads; ++c) st[c * kWave + lane] = sl.rv[c];
    __builtin_amdgcn_wave_barrier();
    const u32x4 ones = u32x4{kBf16OnePair, kBf16OnePair, kBf16OnePair, kBf16OnePair};
    floatx4 X[NB];  // the group's sum of each column's activations
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      X[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c)
        X[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones),
                                                       __builtin_bit_cast(bf16x8, sl.xv[b][c]), X[b], 0, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < RB; ++h) {
      const uint32_t d[4] = {sl.wv[h].x, sl.wv[h].y, sl.wv[h].z, sl.wv[h].w};
      u32x4 a[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int sh4 = c < 2 ? 0 : 4;
        uint32_t p0, p1, p2, p3;
        codes_to_bf16((d[2 * (c % 2)] >> sh4) & 0x0F0F0F0Fu, p0, p1);
        codes_to_bf16((d[2 * (c % 2) + 1] >> sh4) & 0x0F0F0F0Fu, p2, p3);
        a[c] = u32x4{p0, p1, p2, p3};
      }
      // the lane's four D rows 16 h + 4 kb + r of the group: their scales and zeros from the record
      const int rr = 16 * h + 4 * kb;
      const u32x2 zq = *reinterpret_cast<const u32x2*>(st + kScDw + rr / 2);
      uint32_t sw[4] = {0u, 0u, 0u, 0u};
      if constexpr (f32) {
        const u32x4 sq = *reinterpret_cast<const u32x4*>(st + rr);
        sw[0] = sq.x, sw[1] = sq.y, sw[2] = sq.z, sw[3] = sq.w;
      } else {
        const u32x2 sq = *reinterpret_cast<const u32x2*>(st + rr / 2);
        sw[0] = sq.x, sw[1] = sq.y;
      }
      const uint32_t zw[2] = {zq.x, zq.y};
      float sc[4], zf[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        zf[r] = half_bits_to_float(r % 2 == 0 ? zw[r / 2] & 0xffffu : zw[r / 2] >> 16);
        const uint32_t s16 = r % 2 == 0 ? sw[r / 2] & 0xffffu : sw[r / 2] >> 16;
        sc[r] = f32 ? __uint_as_float(sw[r])
                    : (SDT == BP_DT_BF16 ? bf16_bits_to_float(s16) : half_bits_to_float(s16));
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        floatx4 D = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c)
          D = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[c]),
                                                      __builtin_bit_cast(bf16x8, sl.xv[b][c]), D, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[h][b][r] += sc[r] * (D[r] - (128.f + zf[r]) * X[b][r]);
      }
    }
  };

  // whole rounds of DEPTH groups without a branch inside, then the last 1..DEPTH groups without loads
  if (cnt > 0) {
    Slot sl[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      load(sl[d], d < cnt ? d : cnt - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    int base = 0;
    if (cnt > DEPTH) {
      do {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
          compute(sl[d]);
          load(sl[d], base + d + DEPTH < cnt ? base + d + DEPTH : cnt - 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        base += DEPTH;
      } while (base + DEPTH < cnt);
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (base + d < cnt) compute(sl[d]);
  }

  // per activation block: the waves' sums in wave order
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    __syncthreads();  // the patches, or the block before, are done
#pragma unroll
    for (int h = 0; h < RB; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.red[wave][16 * h + 4 * kb + r][i] = acc[h][b][r];
    __syncthreads();
    const auto total = [&](int row, int c) {
      float t = sh.red[0][row][c];
#pragma unroll
      for (int v = 1; v < WAVES; ++v) t += sh.red[v][row][c];
      return t;
    };
    if constexpr (EPI == 0) {
      for (int e = threadIdx.x; e < R * 16; e += WAVES * kWave) {
        const int row = e % R, c = e / R, m = 16 * b + c;  // neighbouring threads on neighbouring outputs
        const int64_t n = n0 + row;
        if (m >= M || n >= N) continue;
        const float t = total(row, c);
        if (split == 1)
          y[static_cast<int64_t>(m0 + m) * N + n] = float_to_bf16_bits(t);
        else
          ws[(static_cast<int64_t>(s) * M_all + m0 + m) * N + n] = t;
      }
    } else {
      // the gate|up SiLU product of rows 2f, 2f + 1 (split 1), as skinny_int4.hip's epilogue
      for (int e = threadIdx.x; e < R * 8; e += WAVES * kWave) {
        const int row = 2 * (e % (R / 2)), c = e / (R / 2), m = 16 * b + c;
        const int64_t n = n0 + row;
        if (m >= M || n + 1 >= N) continue;
        const float gb = round_to_bf16(total(row, c));
        const float a = round_to_bf16(gb / (1.f + expf(-gb)));
        y[static_cast<int64_t>(m0 + m) * (N / 2) + n / 2] = float_to_bf16_bits(a * round_to_bf16(total(row + 1, c)));
      }
    }
  }
}

// Groups in flight per wave: 2 (with one, the compiler keeps the loads of the next group live across the decoding of this
// one and takes up to 80 more registers at 64 tile rows).
constexpr int kDepth = 2;

template <int RB, int NB, int SDT, int EPI>
Int4WideFn wide_waves(int waves) {
  switch (waves) {
    case 1: return &skinny_int4_wide_kernel<RB, NB, 1, kDepth, SDT, EPI>;
    case 2: return &skinny_int4_wide_kernel<RB, NB, 2, kDepth, SDT, EPI>;
    case 4: return &skinny_int4_wide_kernel<RB, NB, 4, kDepth, SDT, EPI>;
    case 8: return &skinny_int4_wide_kernel<RB, NB, 8, kDepth, SDT, EPI>;
    default: return nullptr;
  }
}

template <int NB, int SDT, int EPI>
Int4WideFn wide_tile(int tile_rows, int waves) {
  switch (tile_rows) {
    case 16: return wide_waves<1, NB, SDT, EPI>(waves);
    case 32: return wide_waves<2, NB, SDT, EPI>(waves);
    case 64: return wide_waves<4, NB, SDT, EPI>(waves);
    default: return nullptr;
  }
}

template <int SDT>
Int4WideFn wide_nb(int nb, int tile_rows, int waves, int epi) {
  if (nb == 1) return epi == 0 ? wide_tile<1, SDT, 0>(tile_rows, waves) : wide_tile<1, SDT, 1>(tile_rows, waves);
  if (nb == 2) return epi == 0 ? wide_tile<2, SDT, 0>(tile_rows, waves) : wide_tile<2, SDT, 1>(tile_rows, waves);
  return nullptr;
}

}  // namespace

Int4WideFn int4_wide_pick(int nb, int tile_rows, int waves, int scale_dt, int epi) {
  switch (scale_dt) {
    case BP_DT_BF16: return wide_nb<BP_DT_BF16>(nb, tile_rows, waves, epi);
    case BP_DT_F16: return wide_nb<BP_DT_F16>(nb, tile_rows, waves, epi);
    case BP_DT_F32: return wide_nb<BP_DT_F32>(nb, tile_rows, waves, epi);
    default: return nullptr;
  }
}

}  // namespace bp
