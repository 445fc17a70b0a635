// fft_device.h -- device-side building blocks for the gfx950 spectrometer
// kernels: radix-2/4/8/16 butterflies, an LDS-exchanged Stockham FFT executed
// by a "team" of threads, sample unpacking and polarisation detection.
//
// Conventions used by every kernel:
//  * All transforms are computed with the forward kernel exp(-2 pi i k m / N).
//    The inverse transform rawspec asks for (fft_dir <= 0) is obtained as
//    conj(FFT(conj(x))): the unpacker negates the imaginary input and the
//    detector negates the imaginary cross term (powers are unchanged).
//  * Samples are transformed as raw integers (after the SNORM clamp of the
//    most negative code); the 1/127^2 or 1/32767^2 normalisation of the
//    texture read (rawspec_gpu.cu:845-863) is applied once to the detected
//    sums.
//  * A team of T threads holds an N = T*E point transform; thread j owns
//    elements j + m*T (m < E) on entry and frequency bins j + m*T on exit.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace rsk {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

// Multiplies a by W_R^k = exp(-2 pi i k / R), R <= 16, k compile-time after
// unrolling.  Exact special cases for multiples of pi/4.
template <int R>
__device__ __forceinline__ float2 twc(float2 a, int k) {
  constexpr float R2 = 0.70710678118654752440f;   // cos(pi/4)
  constexpr float C8 = 0.92387953251128675613f;   // cos(pi/8)
  constexpr float S8 = 0.38268343236508977173f;   // sin(pi/8)
  const int e = (k * (16 / R)) & 15;              // angle in units of 2 pi / 16
  switch (e) {
    case 0: return a;
    case 4: return make_float2(a.y, -a.x);
    case 8: return make_float2(-a.x, -a.y);
    case 12: return make_float2(-a.y, a.x);
    case 2: return make_float2((a.x + a.y) * R2, (a.y - a.x) * R2);
    case 6: return make_float2((a.y - a.x) * R2, -(a.x + a.y) * R2);
    case 10: return make_float2((-a.x - a.y) * R2, (a.x - a.y) * R2);
    case 14: return make_float2((a.x - a.y) * R2, (a.x + a.y) * R2);
    default: {
      // general angle: exp(-i t) * (x + i y) = (x c + y s) + i (y c - x s)
      float c, s;
      switch (e) {
        case 1: c = C8; s = S8; break;
        case 3: c = S8; s = C8; break;
        case 5: c = -S8; s = C8; break;
        case 7: c = -C8; s = S8; break;
        case 9: c = -C8; s = -S8; break;
        case 11: c = -S8; s = -C8; break;
        case 13: c = S8; s = -C8; break;
        default: c = C8; s = -S8; break;   // 15
      }
      return make_float2(a.x * c + a.y * s, a.y * c - a.x * s);
    }
  }
}

// In-place forward DFT of R points held in registers (radix-2 recursion,
// fully unrolled).
template <int R>
struct Dft {
  __device__ __forceinline__ static void run(float2 (&a)[R]) {
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int k = 0; k < R / 2; ++k) { e[k] = a[2 * k]; o[k] = a[2 * k + 1]; }
    Dft<R / 2>::run(e);
    Dft<R / 2>::run(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      float2 t = twc<R>(o[k], k);
      a[k] = cadd(e[k], t);
      a[k + R / 2] = csub(e[k], t);
    }
  }
};
template <>
struct Dft<1> {
  __device__ __forceinline__ static void run(float2 (&)[1]) {}
};
template <>
struct Dft<2> {
  __device__ __forceinline__ static void run(float2 (&a)[2]) {
    float2 t = a[1];
    a[1] = csub(a[0], t);
    a[0] = cadd(a[0], t);
  }
};

// ---- butterflies with their twiddle absorbed --------------------------------
// A decimation-in-time butterfly E +- w O with w = g (1 + i t), held as (t =
// tan, g = cos), is six fused multiply-adds and needs no separate product with
// the twiddle (Linzer and Feig, "Implementation of efficient FFT algorithms on
// fused multiply-add architectures", 1993); with ROT the factor is -i w.
template <bool ROT>
__device__ __forceinline__ void bfly(const float2 e, const float2 o, const float2 tg, float2 &lo, float2 &hi) {
  const float u = fmaf(-tg.x, o.y, o.x), v = fmaf(tg.x, o.x, o.y);
  if constexpr (!ROT) {
    lo = make_float2(fmaf(tg.y, u, e.x), fmaf(tg.y, v, e.y));
    hi = make_float2(fmaf(-tg.y, u, e.x), fmaf(-tg.y, v, e.y));
  } else {
    lo = make_float2(fmaf(tg.y, v, e.x), fmaf(-tg.y, u, e.y));
    hi = make_float2(fmaf(-tg.y, v, e.x), fmaf(tg.y, u, e.y));
  }
}

// In-register decimation in time of M points in natural order whose inputs
// carry a twiddle w^a, w = W_(S M)^k: sub-transforms of size m meet with
// factors W_(S m)^(k + S q), q < m / 2, of which q and q + m/4 differ by -i.
// tg[dit_off(m) + q] holds the (tan, cos) of the distinct ones.
template <int M>
struct MDit {
  template <int NT>
  __device__ __forceinline__ static void run(float2 (&x)[M], const float2 (&tg)[NT]) {
    float2 e[M / 2], o[M / 2];
#pragma unroll
    for (int k = 0; k < M / 2; ++k) { e[k] = x[2 * k]; o[k] = x[2 * k + 1]; }
    MDit<M / 2>::run(e, tg);
    MDit<M / 2>::run(o, tg);
    constexpr int G = M >= 8 ? M / 4 : 1, OFF = dit_off(M);
#pragma unroll
    for (int k = 0; k < M / 2; ++k) {
      if (k < G) bfly<false>(e[k], o[k], tg[OFF + k], x[k], x[k + M / 2]);
      else bfly<true>(e[k], o[k], tg[OFF + k - G], x[k], x[k + M / 2]);
    }
  }
};
template <>
struct MDit<1> {
  template <int NT>
  __device__ __forceinline__ static void run(float2 (&)[1], const float2 (&)[NT]) {}
};
constexpr int dit_ntw(int M) { return dit_off(M) + (M >= 8 ? M / 4 : 1); }

// Elements per thread for a team transform of N points (compile-time
// tunables; 16 is the largest radix the butterflies implement).
#ifndef RSK_E_MID
#define RSK_E_MID 8
#endif
#ifndef RSK_E_BIG
#define RSK_E_BIG 16
#endif
constexpr int elems_for(int n) {
  return n <= 16 ? n : (n <= 128 ? RSK_E_MID : RSK_E_BIG);
}
// Elements per thread of the four-step passes' sub-transforms.
#ifndef RSK_E_FS
#define RSK_E_FS 16
#endif
constexpr int elems_fs(int n) { return n <= 128 ? 8 : RSK_E_FS; }

// LDS exchange layout: element `pos` of a team's transform lives at
// lds_pos<PS>(pos), one float2 of padding after every 2^PS elements, and the
// regions of consecutive teams lie lds_len + a pad apart.  The LDS serves 32
// lanes' 8 bytes a cycle from 64 banks of 4, so the pads are chosen for the
// lanes that access it together.  Where the teams of a workgroup are its
// fastest lane index (the four-step passes, TEAMS columns), PS = 4 and 32 /
// TEAMS float2 between teams keep nearly all accesses apart: by a model of the
// banks 0 to 64 conflict cycles a spectrum and wavefront for 256 to 4096 points
// and 32 for 128, against 64 to 1408 with PS = 5 and 8 between teams (counted on
// the device for 512 points: 455, half of pass B's LDS time); one team
// of 4096 points and the small kernels, whose teams are consecutive lanes, are
// best with PS = 5.
template <int PS>
__device__ __forceinline__ constexpr int lds_pos(int pos) { return pos + (pos >> PS); }
// Offset of element pos + d where the powers of two in pos and d are disjoint
// (no carry in the sum): lds_pos is then linear, and a compile-time d leaves one
// base plus a constant.
template <int PS>
__device__ __forceinline__ constexpr int lds_at(int base, int d) { return base + lds_pos<PS>(d); }
constexpr int lds_len(int n, int ps) { return n + (n >> ps); }
constexpr int kSmallPad = 5, kSmallTeamPad = 8;
constexpr int fs_pad(int teams) { return teams > 1 ? 4 : 5; }
// Distance in float2 between the regions of consecutive teams: of the small
// kernels, and of the four-step passes with `teams` columns per workgroup.
constexpr int small_stride(int n) { return lds_len(n, kSmallPad) + kSmallTeamPad; }
constexpr int fs_stride(int n, int teams) {
  return lds_len(n, fs_pad(teams)) + (teams > 1 ? (32 / teams > 0 ? 32 / teams : 1) : 0);
}
// Exchange reads as single 8-byte instructions: the compiler pairs reads that
// lie a multiple of 256 bytes apart, whose halves then meet in the same banks
// (512 points: 782 conflict cycles a spectrum instead of 455).
__device__ __forceinline__ unsigned long long lds_read(const void *p) {
  return *(const volatile __attribute__((address_space(3))) unsigned long long *)p;
}
__device__ __forceinline__ float2 lds_read2(const float2 *p) {
  return __builtin_bit_cast(float2, lds_read(p));
}

// Synchronises a team between the write and the read half of an LDS
// exchange.  A team whose threads are consecutive lanes of one wavefront
// (WAVE) needs no workgroup barrier: a wavefront's LDS instructions complete
// in issue order, so only the compiler must keep the accesses on their side
// of this point.  Otherwise every thread of the workgroup waits here.
template <bool WAVE>
__device__ __forceinline__ void team_sync() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// (tan, cos) table of a team transform of N points (N / 2 entries in LDS), laid
// out for its last stage, which joins sub-transforms of NSL points with radix RL:
// level m's factors W_(NSL m)^x contiguous in x, so that consecutive lanes read
// consecutive entries.  Earlier stages, with few distinct factors, read level 2
// (W_(2 NSL)^x, x < NSL) with a stride.
template <int N>
struct TgTab {
  static constexpr int RL = N <= 128 ? elems_for(N) : 16, NSL = N / RL;
  static_assert(RSK_E_MID == 8 && RSK_E_BIG == 16 && RSK_E_FS == 16, "every transform's last radix");
  static constexpr int off(int m) { return m <= 2 ? 0 : off(m / 2) + NSL * (m / 2 <= 4 ? 1 : m / 8); }
  static constexpr int LEN = N > RL ? off(RL) + NSL * (RL >= 8 ? RL / 4 : 1) : 1;
};
// The factors of a radix-R butterfly at position k of a stage that joins
// sub-transforms of NS points.
template <int N, int R, int NS>
__device__ __forceinline__ void stage_tg(float2 (&tg)[dit_ntw(R)], const float2 *__restrict__ tw, int k) {
  using TT = TgTab<N>;
#pragma unroll
  for (int m = 2; m <= R; m *= 2)
#pragma unroll
    for (int q = 0; q < (m >= 8 ? m / 4 : 1); ++q) {
      if constexpr (NS == TT::NSL) tg[dit_off(m) + q] = tw[TT::off(m) + k + NS * q];
      else tg[dit_off(m) + q] = tw[(k + NS * q) * (2 * TT::NSL / (NS * m))];
    }
}

// One Stockham stage of radix R on an N = T*E point team transform, for NP
// interleaved polarisations.  Butterfly b = j + u*T (u < E/R) reads elements
// b + r*N/R, which are the thread's own slots u + r*E/R; it writes element r
// to (b / NS)*NS*R + (b % NS) + r*NS.  The last stage (NS*R == N) writes back
// into the same register slots, so no exchange follows it.  tw: TgTab's table.
// With NS > 1 the butterflies absorb the
// stage's twiddles: a radix-16 stage takes 192 instructions per transform of
// 16, against 228 as 15 products and a plain butterfly, and reads 8 table
// entries instead of 15.  The other polarisation goes through the same LDS
// region afterwards.
template <int N, int E, int NP, int R, int NS, bool LAST, int PS, bool WAVE>
__device__ __forceinline__ void stage(float2 (&v)[NP][E], float2 *lds, int j,
                                      const float2 *__restrict__ tw) {
  constexpr int T = N / E;
  constexpr int NB = E / R;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int b = j + u * T;
      const int k = b & (NS - 1);
      float2 a[R];
#pragma unroll
      for (int r = 0; r < R; ++r) a[r] = v[p][u + r * NB];
      if constexpr (NS > 1) {
        float2 tg[dit_ntw(R)];
        stage_tg<N, R, NS>(tg, tw, k);
        MDit<R>::run(a, tg);
      } else {
        Dft<R>::run(a);
      }
      if constexpr (LAST) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[p][u + r * NB] = a[r];
      } else {
        // (b / NS, r, b % NS) are disjoint bit fields of the position
        const int base = lds_pos<PS>((b / NS) * NS * R + k);
#pragma unroll
        for (int r = 0; r < R; ++r) lds[lds_at<PS>(base, r * NS)] = a[r];
      }
    }
    if constexpr (!LAST) {
      team_sync<WAVE>();
      const float2 *rd = lds + lds_pos<PS>(j);
#pragma unroll
      for (int m = 0; m < E; ++m) v[p][m] = lds_read2(rd + lds_pos<PS>(m * T));
      team_sync<WAVE>();
    }
  }
}

template <int N, int E, int NP, int NS, int PS, bool WAVE>
struct Stages {
  __device__ __forceinline__ static void run(float2 (&v)[NP][E], float2 *lds, int j,
                                             const float2 *__restrict__ tw) {
    if constexpr (NS * E == N) {
      stage<N, E, NP, E, NS, true, PS, WAVE>(v, lds, j, tw);
    } else {
      stage<N, E, NP, E, NS, false, PS, WAVE>(v, lds, j, tw);
      Stages<N, E, NP, NS * E, PS, WAVE>::run(v, lds, j, tw);
    }
  }
};

// Forward FFT of N points (power of two, E | N, N <= 4096) for NP
// polarisations held by a team of N/E threads.  lds: lds_len(N, PS) float2
// private to the team.  tw: tw_setup's table.  WAVE: the team is
// N/E consecutive lanes of one wavefront (N/E divides 64), so its exchanges
// need no workgroup barrier; otherwise every thread of the workgroup must call
// it (barriers inside).
template <int N, int E, int NP, int PS, bool WAVE = false>
__device__ __forceinline__ void team_fft(float2 (&v)[NP][E], float2 *lds, int j,
                                         const float2 *__restrict__ tw) {
  static_assert(!WAVE || (64 % (N / E) == 0), "a wave-synchronised team must fit in a wavefront");
  if constexpr (N > 1) {
    constexpr int R0 = 1 << (ilog2(N) % ilog2(E));
    if constexpr (R0 > 1) {
      if constexpr (R0 == N) {
        stage<N, E, NP, R0, 1, true, PS, WAVE>(v, lds, j, tw);
      } else {
        stage<N, E, NP, R0, 1, false, PS, WAVE>(v, lds, j, tw);
        Stages<N, E, NP, R0, PS, WAVE>::run(v, lds, j, tw);
      }
    } else {
      Stages<N, E, NP, 1, PS, WAVE>::run(v, lds, j, tw);
    }
  }
}

// ---- int8 samples in FP16 ---------------------------------------------------
// int8 samples are exact FP16 values, and so are sums of up to 16 of them (at
// most 2032 < 2048): the first two levels of a transform, additions only, run
// on packed (re, im) pairs, one instruction per complex addition, and give
// the same values as in FP32.  Unpacking to pairs takes 7 instructions a two-pol
// sample instead of 14.
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// What turns an unpacked (1024 + 128 + re, 1024 + 128 + im) pair into (re, im sg).
struct I8Sign {
  h2v s, c;
  __device__ __forceinline__ explicit I8Sign(float isign) {
    const _Float16 g = isign < 0.0f ? (_Float16)-1.0f : (_Float16)1.0f;
    s = (h2v){(_Float16)1.0f, g};
    c = (h2v){(_Float16)-1152.0f, (_Float16)-1152.0f * g};
  }
};
// Sample word (bytes re, im of pol 0, then of pol 1) to the pair of pol P, with
// the SNORM clamp of -128: the bytes, offset by 128, under exponent byte 0x64
// are FP16 values 1024 + u.
template <int P>
__device__ __forceinline__ h2v i8_pair_sg(unsigned int w, const I8Sign &g) {
  const unsigned int sel = P == 0 ? 0x04010400u : 0x04030402u;
  h2v v = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, w ^ 0x80808080u, sel));
  // 1025 as an integer: positive FP16 values order as their bit patterns
  typedef unsigned short u2v __attribute__((ext_vector_type(2)));
  v = __builtin_bit_cast(h2v, __builtin_elementwise_max(__builtin_bit_cast(u2v, v), (u2v){0x6401, 0x6401}));
  return __builtin_elementwise_fma(v, g.s, g.c);
}
__device__ __forceinline__ float2 h2f(h2v a) { return make_float2((float)a[0], (float)a[1]); }

// Forward DFT of R = 2 or 4 pairs in place.
template <int R>
__device__ __forceinline__ void dft_h(h2v (&a)[R]) {
  if constexpr (R == 2) {
    const h2v t = a[1];
    a[1] = a[0] - t;
    a[0] = a[0] + t;
  } else {
    static_assert(R == 4, "additions only");
    const h2v e0 = a[0] + a[2], e1 = a[0] - a[2], o0 = a[1] + a[3], o1 = a[1] - a[3];
    const h2v r = (h2v){o1[1], -o1[0]};          // -i o1
    a[0] = e0 + o0;
    a[1] = e1 + r;
    a[2] = e0 - o0;
    a[3] = e1 - r;
  }
}
// Forward DFT of R >= 4 pairs to floats: sizes 2 and 4 in FP16, the rest in FP32.
template <int R>
struct DftH {
  __device__ __forceinline__ static void run(const h2v (&a)[R], float2 (&out)[R]) {
    if constexpr (R == 4) {
      h2v b[4] = {a[0], a[1], a[2], a[3]};
      dft_h<4>(b);
#pragma unroll
      for (int k = 0; k < 4; ++k) out[k] = h2f(b[k]);
    } else {
      h2v e[R / 2], o[R / 2];
      float2 fe[R / 2], fo[R / 2];
#pragma unroll
      for (int k = 0; k < R / 2; ++k) { e[k] = a[2 * k]; o[k] = a[2 * k + 1]; }
      DftH<R / 2>::run(e, fe);
      DftH<R / 2>::run(o, fo);
#pragma unroll
      for (int k = 0; k < R / 2; ++k) {
        const float2 t = twc<R>(fo[k], k);
        out[k] = cadd(fe[k], t);
        out[k + R / 2] = csub(fe[k], t);
      }
    }
  }
};

// Forward DFT of 8 pairs: even bins are sums of samples and stay in FP16 (exact,
// at most 1016), odd bins meet W8 = (1 - i) / sqrt 2 in one fused multiply-add
// per component.  30 instructions, against 56 and 16 conversions in FP32.
struct Bins8 {
  h2v even[4];          // bins 0, 2, 4, 6
  float2 odd[4];        // bins 1, 3, 5, 7
  __device__ __forceinline__ float2 bin(int k) const { return k & 1 ? odd[k >> 1] : h2f(even[k >> 1]); }
};
__device__ __forceinline__ Bins8 dft8_h(const h2v (&x)[8]) {
  constexpr float R2 = 0.70710678118654752440f;
  h2v e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
  dft_h<4>(e);
  dft_h<4>(o);
  Bins8 b;
  const h2v r2 = (h2v){o[2][1], -o[2][0]};                 // -i O2
  b.even[0] = e[0] + o[0];
  b.even[2] = e[0] - o[0];
  b.even[1] = e[2] + r2;
  b.even[3] = e[2] - r2;
  const h2v s1 = o[1] + (h2v){o[1][1], -o[1][0]};          // sqrt 2 W8 O1
  const h2v s3 = (h2v){o[3][1], -o[3][0]} - o[3];          // sqrt 2 W8^3 O3
  const float2 f1 = h2f(s1), f3 = h2f(s3), g1 = h2f(e[1]), g3 = h2f(e[3]);
  b.odd[0] = make_float2(fmaf(R2, f1.x, g1.x), fmaf(R2, f1.y, g1.y));
  b.odd[2] = make_float2(fmaf(-R2, f1.x, g1.x), fmaf(-R2, f1.y, g1.y));
  b.odd[1] = make_float2(fmaf(R2, f3.x, g3.x), fmaf(R2, f3.y, g3.y));
  b.odd[3] = make_float2(fmaf(-R2, f3.x, g3.x), fmaf(-R2, f3.y, g3.y));
  return b;
}

// Forward DFT of N <= 8 pairs held by one thread.
template <int N>
__device__ __forceinline__ void dft_pairs(const h2v (&x)[N], float2 (&out)[N]) {
  static_assert(N <= 8, "16 points: dft_bytes");
  if constexpr (N == 8) {
    const Bins8 b = dft8_h(x);
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = b.bin(k);
  } else if constexpr (N >= 4) {
    DftH<N>::run(x, out);
  } else {
    h2v t[N];
#pragma unroll
    for (int k = 0; k < N; ++k) t[k] = x[k];
    if constexpr (N == 2) dft_h<2>(t);
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = h2f(t[k]);
  }
}

// Forward DFT of the N samples of pol P that one thread holds, in FP32: bytes offset
// by 128 take one conversion each (and the SNORM clamp at 1); the offset cancels
// exactly in every difference of integers, so only bin 0 carries it.  16 points of
// two pols, 128 MiB in dumps of 128 and 1024 spectra of power: 27 and 28 us; as
// FP16 pairs, fewer but mostly longer and mixed-width instructions, 33 and 34.
template <int P, int N, class W>
__device__ __forceinline__ void dft_bytes(const W (&raw)[N], float2 (&out)[N], float isign) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const unsigned int t = (unsigned int)raw[k] ^ 0x80808080u;
    out[k] = make_float2(fmaxf((float)((t >> (16 * P)) & 0xffu), 1.0f),
                         isign * fmaxf((float)((t >> (16 * P + 8)) & 0xffu), 1.0f));
  }
  Dft<N>::run(out);
  out[0].x -= 128.0f * N;
  out[0].y -= isign * (128.0f * N);
}

// team_fft of int8 samples held as pairs.  A first stage of radix 2 or 4 stays
// in FP16 through its exchange, both pols at once in the space of one.
template <int N, int E, int NP, int PS, bool WAVE = false>
__device__ __forceinline__ void team_fft_h(const h2v (&in)[NP][E], float2 (&v)[NP][E], float2 *lds, int j,
                                           const float2 *__restrict__ tw) {
  static_assert(!WAVE || (64 % (N / E) == 0), "a wave-synchronised team must fit in a wavefront");
  constexpr int T = N / E;
  constexpr int R0 = 1 << (ilog2(N) % ilog2(E)), R = R0 > 1 ? R0 : E, NB = E / R;
  static_assert(R < N, "a later stage follows");
  if constexpr (R <= 4) {
    uint2 *l2 = reinterpret_cast<uint2 *>(lds);
    unsigned int *l1 = reinterpret_cast<unsigned int *>(lds);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int base = lds_pos<PS>((j + u * T) * R);
      h2v a[NP][R];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int r = 0; r < R; ++r) a[p][r] = in[p][u + r * NB];
        dft_h<R>(a[p]);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const unsigned int w0 = __builtin_bit_cast(unsigned int, a[0][r]);
        if constexpr (NP == 2) l2[lds_at<PS>(base, r)] = make_uint2(w0, __builtin_bit_cast(unsigned int, a[NP - 1][r]));
        else l1[lds_at<PS>(base, r)] = w0;
      }
    }
    team_sync<WAVE>();
    const int rd = lds_pos<PS>(j);
#pragma unroll
    for (int m = 0; m < E; ++m) {
      if constexpr (NP == 2) {
        const uint2 w = __builtin_bit_cast(uint2, lds_read(l2 + rd + lds_pos<PS>(m * T)));
        v[0][m] = h2f(__builtin_bit_cast(h2v, w.x));
        v[NP - 1][m] = h2f(__builtin_bit_cast(h2v, w.y));
      } else {
        v[0][m] = h2f(__builtin_bit_cast(h2v, l1[lds_at<PS>(rd, m * T)]));
      }
    }
    team_sync<WAVE>();
  } else {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        h2v a[R];
        float2 o[R];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = in[p][u + r * NB];
        DftH<R>::run(a, o);
#pragma unroll
        for (int r = 0; r < R; ++r) lds[lds_at<PS>(lds_pos<PS>((j + u * T) * R), r)] = o[r];
      }
      team_sync<WAVE>();
#pragma unroll
      for (int m = 0; m < E; ++m) v[p][m] = lds_read2(lds + lds_pos<PS>(j) + lds_pos<PS>(m * T));
      team_sync<WAVE>();
    }
  }
  Stages<N, E, NP, R, PS, WAVE>::run(v, lds, j, tw);
}

// The workgroup's copy of the table (kernels.h: kTgOff).
template <int N, int WG>
__device__ __forceinline__ const float2 *tw_setup(float2 *twl, const float2 *tw) {
  using TT = TgTab<N>;
  if constexpr (TT::LEN > 1) {
#pragma unroll
    for (int m = 2; m <= TT::RL; m *= 2) {
      const int len = TT::NSL * (m >= 8 ? m / 4 : 1);
      for (int x = threadIdx.x; x < len; x += WG) twl[TT::off(m) + x] = tw[kTgOff + x * (kTwN / (TT::NSL * m))];
    }
    __syncthreads();
  }
  return twl;
}

// ---- sample unpacking ----------------------------------------------------
// Raw sample of NP pols with NBPS-bit components -> NP complex floats
// (integer valued), most negative code clamped to -(2^(NBPS-1)-1) as the
// SNORM read does, imaginary part negated when inv != 0.
template <int NBPS, int NP>
struct Sample;

template <>
struct Sample<8, 2> {
  using word = uint32_t;
  __device__ __forceinline__ static void cvt(word w, float2 (&o)[2], float isign) {
    int a = (int)(int8_t)(w & 0xff), b = (int)(int8_t)((w >> 8) & 0xff);
    int c = (int)(int8_t)((w >> 16) & 0xff), d = (int)(int8_t)(w >> 24);
    a = max(a, -127); b = max(b, -127); c = max(c, -127); d = max(d, -127);
    o[0] = make_float2((float)a, isign * (float)b);
    o[1] = make_float2((float)c, isign * (float)d);
  }
};
template <>
struct Sample<8, 1> {
  using word = uint16_t;
  __device__ __forceinline__ static void cvt(word w, float2 (&o)[1], float isign) {
    int a = (int)(int8_t)(w & 0xff), b = (int)(int8_t)(w >> 8);
    a = max(a, -127); b = max(b, -127);
    o[0] = make_float2((float)a, isign * (float)b);
  }
};
template <>
struct Sample<16, 2> {
  using word = uint2;
  __device__ __forceinline__ static void cvt(word w, float2 (&o)[2], float isign) {
    int a = (int)(int16_t)(w.x & 0xffff), b = (int)(int16_t)(w.x >> 16);
    int c = (int)(int16_t)(w.y & 0xffff), d = (int)(int16_t)(w.y >> 16);
    a = max(a, -32767); b = max(b, -32767); c = max(c, -32767); d = max(d, -32767);
    o[0] = make_float2((float)a, isign * (float)b);
    o[1] = make_float2((float)c, isign * (float)d);
  }
};
template <>
struct Sample<16, 1> {
  using word = uint32_t;
  __device__ __forceinline__ static void cvt(word w, float2 (&o)[1], float isign) {
    int a = (int)(int16_t)(w & 0xffff), b = (int)(int16_t)(w >> 16);
    a = max(a, -32767); b = max(b, -32767);
    o[0] = make_float2((float)a, isign * (float)b);
  }
};

// ---- detection -------------------------------------------------------------
// PMODE 1: total power (sum over pols); 4: XX, YY, Re XY*, Im XY*;
// -4: I, Q, U, V.  gam = +-1 is the sign applied to the imaginary cross term
// (input_conjugated and the inverse-via-conjugation trick combined).
template <int PMODE>
constexpr int nq() { return PMODE == 1 ? 1 : 4; }

// Detection into raw sums, fused multiply-adds: PMODE 1 accumulates the total
// power, a spectrum's terms added up before they join the running sum (an
// addition more per bin, and one rounding at the sum's size instead of four: 2^17
// points, 32 spectra in one run, rms 1.9e-7 to 1.35e-7); 4 and -4 accumulate XX, YY, Re X0 X1* and Im X0 X1* (no sign
// applied), and detect_finish turns the sums into the product's components
// (-4: I = XX + YY, Q = XX - YY; both: the sign gam on the imaginary cross
// term).  The finishing step is linear, so it may be applied to any sum of
// raw sums.
template <int PMODE>
__device__ __forceinline__ void detect_raw(float (&acc)[nq<PMODE>()], float xr0, float xi0,
                                           float xr1, float xi1) {
  if constexpr (PMODE == 1) {
    acc[0] += fmaf(xi1, xi1, fmaf(xr1, xr1, fmaf(xi0, xi0, xr0 * xr0)));
  } else {
    acc[0] = fmaf(xi0, xi0, fmaf(xr0, xr0, acc[0]));
    acc[1] = fmaf(xi1, xi1, fmaf(xr1, xr1, acc[1]));
    acc[2] = fmaf(xi0, xi1, fmaf(xr0, xr1, acc[2]));
    acc[3] = fmaf(-xr0, xi1, fmaf(xi0, xr1, acc[3]));
  }
}
// The same for NP polarisations held as complex values (NP = 1: power).
template <int PMODE, int NP>
__device__ __forceinline__ void detect_raw_np(float (&acc)[nq<PMODE>()], const float2 &x0,
                                              const float2 &x1) {
  if constexpr (NP == 2) {
    detect_raw<PMODE>(acc, x0.x, x0.y, x1.x, x1.y);
  } else {
    static_assert(PMODE == 1, "one polarisation: total power only");
    acc[0] += fmaf(x0.y, x0.y, x0.x * x0.x);
  }
}
template <int PMODE>
__device__ __forceinline__ void detect_finish(float (&v)[nq<PMODE>()], float gam) {
  if constexpr (PMODE != 1) {
    if constexpr (PMODE == -4) {
      const float xx = v[0], yy = v[1];
      v[0] = xx + yy;
      v[1] = xx - yy;
    }
    v[3] *= gam;
  }
}

// Four-step intermediate Y: written once by pass A and read once by the
// vector pass B a whole launch later, when far more than the caches hold
// has passed through them.  Bit 0 of RSK_NT_Y marks pass B's loads of Y
// non-temporal (streaming: the lines do not displace cached data), bit 1
// pass A's stores; both measured faster.  The matrix-core pass B reads Y
// with plain loads: its waves share lines, which streaming loads would
// fetch again.
#ifndef RSK_NT_Y
#define RSK_NT_Y 3
#endif
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_y(float4 *p, float4 v) {
  if constexpr (RSK_NT_Y & 2) {
    const f32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x4 *>(p));
  } else {
    *p = v;
  }
}
__device__ __forceinline__ void store_y(float2 *p, float2 v) {
  if constexpr (RSK_NT_Y & 2) {
    const f32x2 t = {v.x, v.y};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x2 *>(p));
  } else {
    *p = v;
  }
}
__device__ __forceinline__ float4 load_y(const float4 *p) {
  if constexpr (RSK_NT_Y & 1) {
    const f32x4 t = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(p));
    return make_float4(t.x, t.y, t.z, t.w);
  } else {
    return *p;
  }
}
__device__ __forceinline__ float2 load_y(const float2 *p) {
  if constexpr (RSK_NT_Y & 1) {
    const f32x2 t = __builtin_nontemporal_load(reinterpret_cast<const f32x2 *>(p));
    return make_float2(t.x, t.y);
  } else {
    return *p;
  }
}

// 24-bit intermediate (engine level 1, two pols): each float of Y is rounded
// to nearest at mantissa bit 8 (ties away from zero) and its upper three
// bytes kept, so a two-pol complex value takes 12 bytes instead of 16 (every
// value keeps its own exponent; 16 significant bits).  Adding half a unit of
// the kept bits to the sign-magnitude pattern rounds the magnitude; a carry
// out of the mantissa steps the exponent, as rounding up to the next binade
// needs.  One add per value (ties to even took a bit extract and a
// three-operand add); packing and unpacking are byte permutes.
__device__ __forceinline__ unsigned int round24(float x) {
  return __float_as_uint(x) + 0x80u;   // the upper three bytes hold the rounded value
}
// One 12-byte access per value (global_{load,store}_dwordx3 at 4-byte
// alignment): lanes holding consecutive values then cover a contiguous run
// with each instruction.  Three dword accesses per value would leave 8-byte
// gaps in every instruction's footprint, and non-temporal partial sectors
// are written to HBM separately.
typedef unsigned int u32x3 __attribute__((ext_vector_type(3), aligned(4)));
__device__ __forceinline__ u32x3 pack_y24(float4 v) {
  const unsigned int b0 = round24(v.x), b1 = round24(v.y), b2 = round24(v.z), b3 = round24(v.w);
  u32x3 w;
  w.x = __builtin_amdgcn_perm(b1, b0, 0x05030201u);
  w.y = __builtin_amdgcn_perm(b2, b1, 0x06050302u);
  w.z = __builtin_amdgcn_perm(b3, b2, 0x07060503u);
  return w;
}
__device__ __forceinline__ void store_y24(unsigned int *p, float4 v) {
  __builtin_nontemporal_store(pack_y24(v), reinterpret_cast<u32x3 *>(p));
}
__device__ __forceinline__ float4 load_y24(const unsigned int *p) {
  const u32x3 w = __builtin_nontemporal_load(reinterpret_cast<const u32x3 *>(p));
  return make_float4(__uint_as_float(w.x << 8), __uint_as_float(__builtin_amdgcn_perm(w.y, w.x, 0x0504030cu)),
                     __uint_as_float(__builtin_amdgcn_perm(w.z, w.y, 0x0403020cu)),
                     __uint_as_float(w.z & 0xffffff00u));
}

// The running sum of an integration in its internal layout: each block is
// read and written once per pass-B launch by the one workgroup (or
// wavefront) that owns it, so RSK_NT_ACC = 1 streams it past the caches
// (measured: one-buffer calls 1% faster, batches unchanged).
#ifndef RSK_NT_ACC
#define RSK_NT_ACC 1
#endif
__device__ __forceinline__ float load_acc(const float *p) {
  if constexpr (RSK_NT_ACC) return __builtin_nontemporal_load(p);
  else return *p;
}
__device__ __forceinline__ void store_acc(float *p, float v) {
  if constexpr (RSK_NT_ACC) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// Bijective blockIdx -> logical tile map that hands each of the 8 XCDs a
// contiguous range of tiles (hardware dispatches workgroups round-robin over
// XCDs), so neighbouring tiles share one L2.
__device__ __forceinline__ unsigned xcd_remap(unsigned bid, unsigned nb) {
  const unsigned q = nb >> 3, r = nb & 7, x = bid & 7, i = bid >> 3;
  return x * q + min(x, r) + i;
}

}  // namespace rsk
