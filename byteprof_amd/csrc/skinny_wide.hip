// Kernels of the matrix-core skinny matmul from 9 activation rows on (skinny_wide.h). Launched by skinny_mf.hip.
//
// Reference semantics: byteprof/optim/skinny.py:36-90, via skinny_mm (skinny.py:136-166).

#include "skinny_wide.h"

#include <type_traits>

namespace bp {
namespace {

// Segments in flight per wave. More waves per SIMD hide more than more segments per wave: a second bf16 segment where
// the registers of two waves per SIMD hold it (one is 5 to 30% slower below 17 rows, three or four never faster), one
// int8 segment (two 3 to 10% slower, three or four up to 60%).
template <int KIND, int MB, int RP>
constexpr int wide_depth() {
  return KIND == kBf16 && RP * MB * 8 + 2 * 8 * (RP + MB) <= 216 ? 2 : 1;
}

template <int KIND, int MB, int RP, int WAVES, int EPI>
__global__ __launch_bounds__(WAVES* kWave, 2) void skinny_wide_kernel(const uint16_t* __restrict__ x,
                                                                      const uint8_t* __restrict__ w,
                                                                      const void* __restrict__ scale, int scale_dt,
                                                                      uint16_t* __restrict__ y, float* __restrict__ ws,
                                                                      int M_all, int64_t N, int64_t K, int split) {
  using G = MfGeom<KIND>;
  constexpr int P = G::kParts;
  constexpr int D = wide_depth<KIND, MB, RP>();
  constexpr int NT = WAVES * kWave;
  constexpr uint32_t kPast = 0x80000000u;  // beyond any resource
  union alignas(16) Shared {  // both are read and written in 16-byte pieces
    float red[WAVES][MB][kWave][4];
    uint8_t patch[WAVES][2][2048 * P];
  };
  static_assert(alignof(Shared) == 16 && sizeof(Shared::patch[0][0]) % 16 == 0, "16-byte LDS operations");
  __shared__ Shared sh;
  __shared__ __align__(16) float row_scale[KIND == kInt8 ? 16 * RP : 1];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // uniform: MFMAs ignore EXEC
  const MfLane ln(lane);
  // blockIdx.x: groups of 8 weight tiles, each with its mtiles activation tiles 8 workgroups apart, so that the
  // workgroups that read the same weights run on one XCD (workgroups go to the 8 XCDs in turn) and at about the same time
  const uint32_t mtiles = (M_all + 16 * MB - 1) / (16 * MB);
  const uint32_t grp = blockIdx.x / (kXcds * mtiles), in = blockIdx.x - grp * (kXcds * mtiles);
  const int64_t n0 = static_cast<int64_t>(grp * kXcds + in % kXcds) * (16 * RP);
  if (n0 >= N) return;  // the last group's missing tiles (the whole workgroup)
  const int sp = blockIdx.y;
  const int m0 = static_cast<int>(in / kXcds) * (16 * MB);
  const int M = std::min(M_all - m0, 16 * MB);
  uint16_t* yk = y;
  float* wsk = ws;
  asm volatile("" : "+s"(yk), "+s"(wsk));  // pinned: not loaded behind the weight stream
  const int q = threadIdx.x & 3;  // the thread's epilogue items: rows 4 q .. 4 q + 3 of every weight block
  // thread t's row scale (t < 16 RP), loaded ahead of the weights as raw halves, unconditionally (a conditional load is
  // waited for where the branches meet; without scales, split > 1, it reads x[0], unused)
  uint32_t sraw[2] = {0u, 0u};
  if constexpr (KIND == kInt8) {
    const bool have = split == 1 && scale != nullptr;
    const bool f32 = scale_dt == BP_DT_F32;
    const auto p = as_global(have ? static_cast<const uint16_t*>(scale) : x);
    const int64_t n = std::min<int64_t>(n0 + threadIdx.x % (16 * RP), N - 1);
    const int64_t e = !have ? 0 : f32 ? 2 * n : n;
    sraw[0] = p[e];
    sraw[1] = p[e + (have && f32 ? 1 : 0)];
  }
  const int64_t nseg_all = K / G::kSeg;
  const int64_t s_lo = split == 1 ? 0 : sp * nseg_all / split;
  const int64_t s_hi = split == 1 ? nseg_all : (sp + 1) * nseg_all / split;
  const int first = static_cast<int>(s_lo) + wave;
  const int nseg =
      __builtin_amdgcn_readfirstlane(first < s_hi ? (static_cast<int>(s_hi) - first + WAVES - 1) / WAVES : 0);

  // the workgroup's weight rows and the activation rows as buffer resources; rows past N or M and segments past the
  // wave's last have offsets past them (zeros, no memory request). K is a multiple of 64 below 2^24 (the launches'
  // kMaxVecK), so 64 rows x K x 2 bytes stay below 2^31.
  static_assert(RP <= 4 && MB <= 4, "operand sizes below 2^31 bytes");
  const int64_t rows = std::min<int64_t>(16 * RP, N - n0);
  const __amdgpu_buffer_rsrc_t wrs = buffer_rsrc(w + n0 * K * G::kEB, static_cast<int>(rows * K * G::kEB));
  const __amdgpu_buffer_rsrc_t xrs = buffer_rsrc(x + m0 * K, static_cast<int>(2 * M * K));
  constexpr int XL = 2 * P;           // loads of 1 KiB per activation block and segment
  constexpr int XR = 16 / XL;         // rows per load
  constexpr int XP = kWave / XR;      // 16-byte pieces of a row's segment
  uint32_t woff[RP][2], xoff[MB][XL];
#pragma unroll
  for (int rp = 0; rp < RP; ++rp)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = 16 * rp + 8 * u + (lane >> 3);
      woff[rp][u] = r < rows ? static_cast<uint32_t>(r * K * G::kEB + 16 * (lane & 7)) : kPast;
    }
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int u = 0; u < XL; ++u) {
      const int m = 16 * b + XR * u + lane / XP;
      xoff[b][u] = m < M ? static_cast<uint32_t>(2 * m * K + 16 * (lane % XP)) : kPast;
    }

  struct Slot {
    u32x4 w[RP][2];
    u32x4 x[MB][XL];
  };
  floatx4 acc[RP][MB][2];
#pragma unroll
  for (int rp = 0; rp < RP; ++rp)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[rp][b][0] = acc[rp][b][1] = floatx4{0.f, 0.f, 0.f, 0.f};

  // Every load is unconditional and every round computes D slots: a segment past the wave's last is loaded as zeros
  // (kPastSeg takes any row's offset past its resource) and adds exact zeros, so the waits count exactly.
  constexpr uint32_t kPastSeg = 0x7fffff00u;
  auto issue = [&](Slot& sl, int idx) {
    const uint32_t s = static_cast<uint32_t>(first + idx * WAVES);
    const uint32_t sw = idx < nseg ? s * 128u : kPastSeg;
    const uint32_t sx = idx < nseg ? s * (2u * G::kSeg) : kPastSeg;
#pragma unroll
    for (int rp = 0; rp < RP; ++rp)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        sl.w[rp][u] =
            __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrs, woff[rp][u] + sw, 0, 2 /* nt */));
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int u = 0; u < XL; ++u)
        sl.x[b][u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[b][u] + sx, 0, 0));
  };
  // The wave's own 16 rows x XP pieces through LDS: piece c of row r at slot c ^ r (16 pieces) or c ^ (r / 2) (8 pieces:
  // two rows per 256 bytes), so neither the row-wise writes nor the column-wise reads conflict.
  int par = 0;
  auto bounce = [&](auto& v, auto np) {
    constexpr int NP = decltype(np)::value;
    constexpr int NL = NP / 4;
    uint8_t* st = sh.patch[wave][par];
    par ^= 1;
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int r = (16 / NL) * u + lane / NP;
      const int key = NP == 16 ? r : r >> 1;
      *reinterpret_cast<u32x4*>(st + r * (16 * NP) + 16 * ((lane % NP) ^ key)) = v[u];
    }
    __builtin_amdgcn_wave_barrier();
    const int key = NP == 16 ? ln.i : ln.i >> 1;
#pragma unroll
    for (int u = 0; u < NL; ++u)
      v[u] = *reinterpret_cast<const u32x4*>(st + ln.i * (16 * NP) + 16 * ((NL * ln.g + u) ^ key));
    __builtin_amdgcn_wave_barrier();
  };
  auto compute = [&](Slot& sl) {
#pragma unroll
    for (int b = 0; b < MB; ++b) bounce(sl.x[b], std::integral_constant<int, XP>{});
#pragma unroll
    for (int rp = 0; rp < RP; ++rp) {
      bounce(sl.w[rp], std::integral_constant<int, 8>{});
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 a[P];
        if constexpr (KIND == kBf16) {
          a[0] = sl.w[rp][h];
        } else {
          a[0] = mf_i8x8(sl.w[rp][h].x, sl.w[rp][h].y);
          a[1] = mf_i8x8(sl.w[rp][h].z, sl.w[rp][h].w);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int p = 0; p < P; ++p) acc[rp][b][h] = mf_mfma(a[p], sl.x[b][h * P + p], acc[rp][b][h]);
      }
    }
  };

  // one block around the first loads and the rounds: with the loads ahead of a loop that may run no round the compiler
  // sinks them into the loop's preheader in an order of its own, and every round then waits for all of them
  if (nseg > 0) {
    Slot buf[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      issue(buf[d], d);
      __builtin_amdgcn_sched_barrier(0);
    }
    int base = 0;
    do {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(buf[d]);
        issue(buf[d], base + d + D);
        __builtin_amdgcn_sched_barrier(0);  // the slots in order: a slot's loads ahead of the next slot's arithmetic
      }
      base += D;
    } while (base < nseg);
  }

  if constexpr (KIND == kInt8) {
    if (threadIdx.x < 16 * RP)
      row_scale[threadIdx.x] =
          scale_dt == BP_DT_F32    ? __uint_as_float(sraw[0] | (sraw[1] << 16))
          : scale_dt == BP_DT_BF16 ? bf16_bits_to_float(sraw[0])
                                   : static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(sraw[0])));
  }
  __syncthreads();  // the patches are done
  // per weight block: half 0 + half 1, then the waves in wave order; lane l holds rows 4 (l / 16) + t of column l % 16
    const bool vec4 = EPI == 0 && N % 4 == 0 && (reinterpret_cast<uintptr_t>(yk) & 7) == 0;
#pragma unroll
  for (int rp = 0; rp < RP; ++rp) {
    if (rp > 0) __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b)
      *reinterpret_cast<floatx4*>(&sh.red[wave][b][lane][0]) = acc[rp][b][0] + acc[rp][b][1];
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * MB; e += NT) {
      const int m = e >> 2;
      const int64_t n = n0 + 16 * rp + 4 * q;
      if (m >= M || n >= N) continue;
      const int l = 16 * q + (m & 15);
      floatx4 t = *reinterpret_cast<const floatx4*>(&sh.red[0][m >> 4][l][0]);
#pragma unroll
      for (int v = 1; v < WAVES; ++v) t += *reinterpret_cast<const floatx4*>(&sh.red[v][m >> 4][l][0]);
      if (EPI == 0 && split > 1) {
        float* dst = wsk + (static_cast<int64_t>(sp) * M_all + m0 + m) * N + n;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (n + u < N) dst[u] = t[u];
        continue;
      }
      if constexpr (KIND == kInt8) {
        t *= *reinterpret_cast<const floatx4*>(&row_scale[16 * rp + 4 * q]);
      }
      if constexpr (EPI == 0) {
        uint16_t* dst = yk + static_cast<int64_t>(m0 + m) * N + n;
        if (vec4) {  // n + 3 < N as N % 4 == 0
          const uint2 o{float_to_bf16_bits(t[0]) | (static_cast<uint32_t>(float_to_bf16_bits(t[1])) << 16),
                        float_to_bf16_bits(t[2]) | (static_cast<uint32_t>(float_to_bf16_bits(t[3])) << 16)};
          *reinterpret_cast<uint2*>(dst) = o;
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (n + u < N) dst[u] = float_to_bf16_bits(t[u]);
        }
      } else {
#pragma unroll
        for (int u = 0; u < 4; u += 2) {
          if (n + u + 1 >= N) continue;
          const float gb = round_to_bf16(t[u]);
          const float a = round_to_bf16(gb / (1.f + expf(-gb)));
          yk[static_cast<int64_t>(m0 + m) * (N / 2) + (n + u) / 2] = float_to_bf16_bits(a * round_to_bf16(t[u + 1]));
        }
      }
    }
  }
}

template <int KIND, int MB, int RP, int EPI>
MfWideFn wide_waves(int waves) {
  switch (waves) {
    case 1: return &skinny_wide_kernel<KIND, MB, RP, 1, EPI>;
    case 2: return &skinny_wide_kernel<KIND, MB, RP, 2, EPI>;
    case 4: return &skinny_wide_kernel<KIND, MB, RP, 4, EPI>;
    case 8: return &skinny_wide_kernel<KIND, MB, RP, 8, EPI>;
    default: return nullptr;
  }
}

template <int KIND, int MB, int EPI>
MfWideFn wide_rp(int rp, int waves) {
  switch (rp) {
    case 1: return wide_waves<KIND, MB, 1, EPI>(waves);
    case 2: return wide_waves<KIND, MB, 2, EPI>(waves);
    case 4:
      if constexpr (MB <= mf_wide_max_mb(KIND, 4)) return wide_waves<KIND, MB, 4, EPI>(waves);
      return nullptr;
    default: return nullptr;
  }
}

template <int KIND, int EPI>
MfWideFn wide_mb(int mb, int rp, int waves) {
  switch (mb) {
    case 1: return wide_rp<KIND, 1, EPI>(rp, waves);
    case 2: return wide_rp<KIND, 2, EPI>(rp, waves);
    case 3: return wide_rp<KIND, 3, EPI>(rp, waves);
    case 4:
      if constexpr (mf_wide_max_mb(KIND, 1) >= 4) return wide_rp<KIND, 4, EPI>(rp, waves);
      return nullptr;
    default: return nullptr;
  }
}

}  // namespace

MfWideFn mf_wide_pick(int wkind, int mb, int rp, int waves, int epi) {
  if (wkind == kBf16) return epi == 0 ? wide_mb<kBf16, 0>(mb, rp, waves) : wide_mb<kBf16, 1>(mb, rp, waves);
  if (wkind == kInt8) return epi == 0 ? wide_mb<kInt8, 0>(mb, rp, waves) : wide_mb<kInt8, 1>(mb, rp, waves);
  return nullptr;
}

}  // namespace bp
