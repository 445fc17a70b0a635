// k_small_h.hip -- the fused spectrometer kernel (k_small's contract) for
// N = 64 .. 1024 on both units: unpack -> 32-point DFTs on the matrix cores ->
// N/32-point DFTs on the vector units (dft_hybrid.h) -> detection ->
// integration in registers -> FFT-shifted output, FP32-level error.
//
// What bounds it: vector instructions.  Per 1024 two-pol int8 samples a
// wavefront issues about 750 of them (110 unpack, 512 stage 2, 128 Stokes
// detection) and 32 matrix instructions, which run beside the other
// wavefront's vector work (counted over a launch of 16 units a wavefront, with
// set-up, sums and write-out: 824); the radix 4, 16, 16 vector kernel issues 1383
// and exchanges every value through LDS twice.  64 channels x 256 MiB, Stokes,
// 1024 points: 192 + 15 us with its partial sums before, 123 + 7 now; 64 MiB of
// 256 points in dumps of 4: 78 before, 44 now; 128 points, power, 41 and 25.
//
// One wavefront transforms 1024 consecutive samples of a channel at a time
// (1024 / N spectra, all of one dump group) and loads the next 1024 before
// transforming the current ones.  Two ways to share out the groups:
//   SOLO   every wavefront integrates whole groups, one after another, and
//          stores each from registers (many short groups);
//   else   the workgroup's wavefronts share one chunk of a group and add
//          their sums through LDS in wavefront order (few groups, or long ones,
//          whose chains of FP32 additions would round more in one wavefront).
#include <type_traits>

#include "dft_hybrid.h"
#include "kernels.h"

namespace rsk {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <int N, int NBPS, int NP, int PMODE, bool SOLO, int WAVES>
__global__ __launch_bounds__(64 * WAVES, PMODE == 1 ? 3 : 2) void k_small_h(SmallArgs a) {
  constexpr int M = N / 32, S = 1024 / N;
  constexpr int Q = nq<PMODE>();
  constexpr int AC = M <= 16 ? M : 16;         // bins per lane while integrating
  constexpr int OC = M <= 16 ? M / 2 : 16;     // bins per lane on output
  using In = HybIn<NBPS, NP>;
  using W = typename In::word;
  constexpr int kStBytes = SOLO ? 0 : WAVES * Q * N * 4;
  constexpr int WB = (int)sizeof(W), PAD = 16 / WB;
  constexpr int kTile = 1024 + 16 * PAD;       // samples of a wavefront's tile
  constexpr int kLoopBytes = (int)sizeof(Dft32K) + WAVES * kTile * WB;
  constexpr int kLds = kStBytes > kLoopBytes ? kStBytes : kLoopBytes;
  __shared__ __attribute__((aligned(16))) unsigned char lds_raw[kLds];
  Dft32K &K = *reinterpret_cast<Dft32K *>(lds_raw);
  float *st = reinterpret_cast<float *>(lds_raw);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & 31, h = lane >> 5;

  // this wavefront's run of units (1024 samples each): first unit of the
  // channel, units per group, number and stride of its units
  unsigned c, g, chunk = 0, u0, nu, ustep;
  const unsigned upg = a.na_buf / S;
  if constexpr (SOLO) {
    const unsigned wi = blockIdx.x * WAVES + wv;
    c = wi / a.bpc;
    g = (wi - c * a.bpc) * a.gpw;
    u0 = g * upg;
    ustep = 1;
    nu = c < a.Nc && g < a.Ng ? min(a.gpw, a.Ng - g) * upg : 0;
    if (c >= a.Nc) c = 0;
  } else {
    c = blockIdx.x / (a.Ng * a.G);
    const unsigned rest = blockIdx.x - c * (a.Ng * a.G);
    g = rest / a.G;
    chunk = rest - g * a.G;
    const unsigned first = chunk * (a.chunk / S), cu = min(a.chunk / S, upg - first);
    u0 = g * upg + first + wv;
    ustep = WAVES;
    nu = (unsigned)wv < cu ? (cu - wv + WAVES - 1) / WAVES : 0;
  }

  dft32_consts(K, a.tw, 64 * WAVES, 0u);
  float2 tg[hyb_ntw(M)];
  hyb_tw<M>(tg, a.tw, lane);
  __syncthreads();

  int rs, ra;
  hyb_row<M>(col, rs, ra);
  // Samples go through a per-wavefront LDS tile: 16-byte loads of consecutive
  // lanes, whatever the rows need.  Sample p lies at p + PAD (p / 64), which
  // spreads the rows of short transforms over the banks; the sample of K
  // element e = (kb, i) is this lane's first one plus E = M (8 kb + i), and
  // the two remainders modulo 64 never carry, so E + PAD (E / 64) is a
  // constant offset.
  W *tile = reinterpret_cast<W *>(lds_raw + sizeof(Dft32K)) + wv * kTile;
  const int l0 = rs * N + ra + M * 4 * h;
  const W *tr = tile + l0 + PAD * (l0 >> 6);
  constexpr int VL = WB;                       // 16-byte loads per lane: 1024 WB / 16 / 64
  u32x4 *const twr = reinterpret_cast<u32x4 *>(tile + PAD * lane + PAD * ((PAD * lane) >> 6));
  constexpr int kRow4 = (64 * PAD + PAD * PAD) * WB / 16;   // uint4 between a lane's tile stores
  const u32x4 *src = reinterpret_cast<const u32x4 *>(a.in + (unsigned long long)c * a.chan_stride +
                                                     (unsigned long long)u0 * (1024 * WB)) + lane;
  float acc[AC][Q];
#pragma unroll
  for (int d = 0; d < AC; ++d)
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[d][q] = 0.0f;
  // the inverse transform is the forward one read at bin -k: the cross
  // term's sign is then the input-conjugation sign alone
  const bool inv = a.isign < 0.0f;
  const float gam = a.gam * a.isign;
  const float sc = a.scale * (In::SCALE * In::SCALE);

  // The unit's spectra of a bin are added up before they join the running sum (a
  // single spectrum's four sums are not: an eighth more instructions)
  auto sum_unit = [&](const float2 (&x0)[16], const float2 (&x1)[16]) {
#pragma unroll
    for (int d = 0; d < AC; ++d) {
      if constexpr (PMODE == 1) {              // one pol
        float t = fmaf(x0[d].y, x0[d].y, x0[d].x * x0[d].x);
#pragma unroll
        for (int r = d + AC; r < 16; r += AC) t += fmaf(x0[r].y, x0[r].y, x0[r].x * x0[r].x);
        acc[d][0] += t;
      } else if constexpr (AC == 16) {
        detect_raw_np<PMODE, NP>(acc[d], x0[d], x1[d]);
      } else {
        float t[Q] = {};
#pragma unroll
        for (int r = d; r < 16; r += AC) detect_raw_np<PMODE, NP>(t, x0[r], x1[r]);
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[d][q] += t[q];
      }
    }
  };
  u32x4 ahead[VL];                             // the next unit's samples
  if (nu) {
#pragma unroll
    for (int e = 0; e < VL; ++e) ahead[e] = src[64 * e];
  }
  unsigned ug = 0;                             // units into the group (SOLO)
  for (unsigned t = 0; t < nu; ++t) {
    // an opaque zero in the index keeps the DFT matrix (64 registers) in LDS
    int z;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    // the tile is this wavefront's own: its LDS operations complete in order,
    // so fences for the compiler are all the exchange needs
    team_sync<true>();
#pragma unroll
    for (int e = 0; e < VL; ++e) twr[kRow4 * e] = ahead[e];
    if (t + 1 < nu) {
      const u32x4 *nx = src + (unsigned long long)(t + 1) * ustep * (64 * WB);
#pragma unroll
      for (int e = 0; e < VL; ++e) ahead[e] = nx[64 * e];
    }
    team_sync<true>();
    // operands of pol p (compile-time after unrolling) from the tile
    auto operands = [&](HybFrag<In::PARTS> &f, auto pol) {
      constexpr int p = decltype(pol)::value;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int E = M * (8 * (e >> 2) + (e & 3));
        unsigned int hi, lo = 0;
        if constexpr (NBPS == 16 && NP == 2)
          HybIn<16, 1>::template pair<0>(reinterpret_cast<const unsigned int *>(tr + E + PAD * (E >> 6))[p],
                                         hi, lo);
        else In::template pair<p>(tr[E + PAD * (E >> 6)], hi, lo);
        frag_set(f, e, hi, lo);
      }
    };
    // one pol after the other: power detects each at once and keeps 4 (3)
    // wavefronts per SIMD; int16 operands of both pols together spill
    f16v zr[NP], zi[NP];
    float2 x[NP][16];
    auto one = [&](auto pol) {
      constexpr int p = decltype(pol)::value;
      HybFrag<In::PARTS> f[1];
      f16v r1[1], i1[1];
      operands(f[0], pol);
      dft32_mfma<1, In::PARTS>(f, K, lane + z, r1, i1);
      if constexpr (PMODE == 1) {
        hyb_stage2<M>(r1[0], i1[0], tg, x[0]);
        sum_unit(x[0], x[0]);
      } else {
        zr[p] = r1[0];
        zi[p] = i1[0];
      }
    };
    if constexpr (PMODE == 1 || NBPS == 16) {
      one(std::integral_constant<int, 0>());
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NP == 2) one(std::integral_constant<int, NP - 1>());
    } else {
      HybFrag<In::PARTS> f[NP];
      operands(f[0], std::integral_constant<int, 0>());
      operands(f[NP - 1], std::integral_constant<int, NP - 1>());
      dft32_mfma<NP, In::PARTS>(f, K, lane + z, zr, zi);
    }
    if constexpr (PMODE != 1) {
#pragma unroll
      for (int p = 0; p < NP; ++p) hyb_stage2<M>(zr[p], zi[p], tg, x[p]);
      sum_unit(x[0], x[NP - 1]);
    }

    if constexpr (SOLO) {
      if (++ug == upg) {
        ug = 0;
        float o[OC][Q];
#pragma unroll
        for (int d = 0; d < AC; ++d) detect_finish<PMODE>(acc[d], gam);
        if constexpr (M <= 16) {
          // both lane halves hold every bin: the lower lanes keep d < M / 2
#pragma unroll
          for (int d = 0; d < OC; ++d)
#pragma unroll
            for (int q = 0; q < Q; ++q) {
              float lo = acc[d][q], hi = acc[d + AC / 2][q];
              half_swap(lo, hi);
              o[d][q] = lo + hi;
            }
        } else {
#pragma unroll
          for (int d = 0; d < OC; ++d)
#pragma unroll
            for (int q = 0; q < Q; ++q) o[d][q] = acc[d][q];
        }
        float *ob = a.acc + ((unsigned long long)g * Q * a.Nc + c) * N;
#pragma unroll
        for (int d = 0; d < OC; ++d) {
          const int k = col + 32 * (M <= 16 ? d + h * OC : h + 2 * d);
          const int jo = ((inv ? N - k : k) + N / 2) & (N - 1);
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            float *po = ob + (unsigned long long)q * a.Nc * N + jo;
            float v = o[d][q] * sc;
            if (!a.first) v += *po;
            *po = v;
          }
        }
#pragma unroll
        for (int d = 0; d < AC; ++d)
#pragma unroll
          for (int q = 0; q < Q; ++q) acc[d][q] = 0.0f;
        ++g;
      }
    }
  }

  if constexpr (!SOLO) {
    __syncthreads();                           // the constants' LDS is reused
    float *sw = st + wv * (Q * N);
#pragma unroll
    for (int d = 0; d < AC; ++d) detect_finish<PMODE>(acc[d], gam);
#pragma unroll
    for (int d = 0; d < OC; ++d) {
      const int k = col + 32 * (M <= 16 ? d + h * OC : h + 2 * d);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        float v;
        if constexpr (M <= 16) {
          float lo = acc[d][q], hi = acc[d + AC / 2][q];
          half_swap(lo, hi);
          v = lo + hi;
        } else {
          v = acc[d][q];
        }
        sw[q * N + k] = v;
      }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < Q * N; idx += 64 * WAVES) {
      const int q = idx / N, jo = idx & (N - 1);
      const int kk = (jo + N / 2) & (N - 1);
      const int k = inv ? (N - kk) & (N - 1) : kk;
      float v = st[q * N + k];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v += st[(w * Q + q) * N + k];
      if (a.direct) {
        float *po = a.acc + (((unsigned long long)g * Q + q) * a.Nc + c) * N + jo;
        v *= sc;
        if (!a.first) v += *po;
        *po = v;
      } else {
        a.part[((((unsigned long long)c * a.Ng + g) * a.G + chunk) * Q + q) * N + jo] =
            v * (In::SCALE * In::SCALE);
      }
    }
  }
}

// int16 products that the planner never sends here (rsd_runtime.hip, vector_pays):
// 64 points; power of two pols at 256 points, and from 256 points on where
// wavefronts take whole groups.
template <int N, int NBPS, int NP, int PMODE, bool SOLO>
constexpr bool h_built() {
  return NBPS == 8 || !(N == 64 || (N >= 256 && PMODE == 1 && (SOLO || (N == 256 && NP == 2))));
}
template <int N, int NBPS, int NP, int PMODE>
static int go_h(const SmallArgs &a, unsigned nb, int solo, int waves, hipStream_t s) {
  const dim3 g(nb), t(64 * waves);
  if (solo) {
    if constexpr (h_built<N, NBPS, NP, PMODE, true>())
      hipLaunchKernelGGL((k_small_h<N, NBPS, NP, PMODE, true, 4>), g, t, 0, s, a);
    else return 2;
  } else if constexpr (!h_built<N, NBPS, NP, PMODE, false>()) {
    return 2;
  } else if (waves == 8) {
    hipLaunchKernelGGL((k_small_h<N, NBPS, NP, PMODE, false, 8>), g, t, 0, s, a);
  } else {
    hipLaunchKernelGGL((k_small_h<N, NBPS, NP, PMODE, false, 4>), g, t, 0, s, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <int N, int NBPS>
static int go_h_mode(int np, int pmode, const SmallArgs &a, unsigned nb, int solo, int waves, hipStream_t s) {
  if (np == 1) return go_h<N, NBPS, 1, 1>(a, nb, solo, waves, s);
  switch (pmode) {
    case 1: return go_h<N, NBPS, 2, 1>(a, nb, solo, waves, s);
    case 4: return go_h<N, NBPS, 2, 4>(a, nb, solo, waves, s);
    case -4: return go_h<N, NBPS, 2, -4>(a, nb, solo, waves, s);
  }
  return 2;
}

template <int NBPS>
static int go_h_n(int n, int np, int pmode, const SmallArgs &a, unsigned nb, int solo, int waves, hipStream_t s) {
  switch (n) {
    case 64: return go_h_mode<64, NBPS>(np, pmode, a, nb, solo, waves, s);
    case 128: return go_h_mode<128, NBPS>(np, pmode, a, nb, solo, waves, s);
    case 256: return go_h_mode<256, NBPS>(np, pmode, a, nb, solo, waves, s);
    case 512: return go_h_mode<512, NBPS>(np, pmode, a, nb, solo, waves, s);
    case 1024: return go_h_mode<1024, NBPS>(np, pmode, a, nb, solo, waves, s);
  }
  return 2;
}

int small_h_ok(int n, unsigned na_buf) {
  return n >= 64 && n <= 1024 && (n & (n - 1)) == 0 && na_buf % (1024u / (unsigned)n) == 0;
}

int launch_small_h(int n, int nbps, int np, int pmode, const SmallArgs &a, unsigned nblocks, int solo,
                   int waves, hipStream_t s) {
  if (!small_h_ok(n, a.na_buf) || nblocks == 0 || a.nt != (unsigned)n) return 2;
  if (waves != 4 && (waves != 8 || solo)) return 2;
  const unsigned S = 1024u / (unsigned)n;
  // SOLO walks whole groups straight into the integration buffer; otherwise
  // the chunks are whole units that cover the group, the last one perhaps fewer
  if (solo ? (!a.direct || a.G != 1 || a.gpw == 0 || a.bpc == 0 ||
              (unsigned long long)a.bpc * a.gpw < a.Ng ||
              (unsigned long long)nblocks * 4ull < (unsigned long long)a.bpc * a.Nc)
           : (a.chunk == 0 || a.chunk % S != 0 || (unsigned long long)a.chunk * a.G < a.na_buf ||
              (unsigned long long)a.chunk * (a.G - 1) >= a.na_buf ||
              nblocks != (unsigned long long)a.Nc * a.Ng * a.G))
    return 2;
  if (nbps == 8) return go_h_n<8>(n, np, pmode, a, nblocks, solo, waves, s);
  if (nbps == 16) return go_h_n<16>(n, np, pmode, a, nblocks, solo, waves, s);
  return 2;
}

}  // namespace rsk
