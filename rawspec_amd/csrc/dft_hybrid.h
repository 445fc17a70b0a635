// dft_hybrid.h -- N-point DFTs of integer samples, N = 32 M: the first 32
// points on the gfx950 matrix cores, the remaining M points on the vector
// units, one wavefront per 1024 samples, no LDS exchange and no barrier.
//
//   n = a + M b, k = c + 32 d  (b, c < 32; a, d < M)
//   stage 1   Z[a][c] = sum_b x[a + M b] W_32^(b c)           (matrix cores)
//   stage 2   X[c + 32 d] = sum_a Z[a][c] W_N^(a c) W_M^(a d)  (vector units)
//
// Stage 1 is a complex 32 x 32 x 32 product per 32 rows, issued as
// v_mfma_f32_32x32x16_f16 with (re, im) interleaved along K (mfma_dft.h has
// the lane layout).  Integer samples are exact FP16 operands: int8 as it is,
// int16 as x / 256 = hi + lo with an 8-bit integer hi and an 8-bit fraction
// lo.  The 32-point DFT matrix is a hi + lo pair of FP16 values (at most 2^-25
// off, as an FP32 twiddle near 1; rms 1.8e-8 against FP32's 1.5e-8) and products
// accumulate in FP32, small ones first.  Against 64 bits the whole transform is
// as exact as the FP32 radix-16 transform it replaces, or more (rms of detected
// power, int8: 1024 points 0.91 times, 512 0.86, 256 0.92, 128 0.98, 64 0.95 to
// 1.04; int16 0.93, 0.89, 0.95 and 1.02).
//
// The 32 rows of one product are rows of different spectra (or columns)
// when M < 32.  Row rho of the product ends in register r = 4 (rho / 8) +
// rho % 4 of lane half (rho / 4) % 2 (the C layout); rows are assigned so
// that one lane holds every a it needs:
//   M <= 16   a = r % M of transform r / M + half (16 / M): 32 / M transforms
//             per product, stage 2 entirely within the lane;
//   M = 32    a = rho: the lane half is bit 2 of a.  Stage 2 does the bits
//             4 and 3 of a in the lane, trades the lane bit for bit 0 of the
//             partial output index (v_permlane32_swap), and finishes bits 2,
//             1 and 0 in the lane.
// Stage 2 is a decimation-in-time DFT whose every butterfly absorbs the
// twiddle W_N^(a c): at sub-transform size m the factor is W_(32 m)^(c + 32 k),
// a lane constant held as (t = tan, g = cos), so that E +- w O costs six fused
// multiply-adds and no separate twiddle product (Linzer and Feig, "Implementation
// of efficient FFT algorithms on fused multiply-add architectures", 1993); k and
// k + m/4 share a factor up to -i.  15 instructions per complex value for M = 32
// against the 32.5 of a radix 4, 16, 16 transform of the whole length.
#pragma once

#include "fft_device.h"
#include "mfma_dft.h"

namespace rsk {

// B operands of the 32-point DFT matrix, [re/im output][K-block][hi/lo][lane],
// in LDS, shared by a workgroup's wavefronts.
struct Dft32K {
  h8v b[2][4][2][64];
};

// The constants come from a table the host computes in 64 bits (behind the
// W_4096 table, kernels.h): the operands, then stage 2's factors of every M.
// sgn = 0x80000000 negates the rows that meet imaginary parts: the transform
// of the conjugated samples.
__device__ __forceinline__ void dft32_consts(Dft32K &k, const float2 *tw4096, int wg, unsigned int sgn) {
  const uint4 *src = reinterpret_cast<const uint4 *>(tw4096 + kTwN);
  uint4 *dst = reinterpret_cast<uint4 *>(&k);
  for (int e = threadIdx.x; e < (int)(sizeof(Dft32K) / 16); e += wg) {
    const uint4 v = src[e];
    dst[e] = make_uint4(v.x ^ sgn, v.y ^ sgn, v.z ^ sgn, v.w ^ sgn);
  }
}

// ---- samples -> FP16 operands ----------------------------------------------
// One sample word to the (re, im) FP16 pair of each pol (HybIn::hi) and, for
// int16, the pair of fractions (lo).  The SNORM clamp of the most negative code
// is applied.
template <int NBPS, int NP>
struct HybIn;
template <int NP>
struct HybIn<8, NP> {
  static constexpr int PARTS = 1;
  static constexpr float SCALE = 1.0f;         // Z scale: samples as they are
  using word = typename Sample<8, NP>::word;
  template <int P>
  __device__ __forceinline__ static void pair(word w, unsigned int &hi, unsigned int &) {
    hi = i8_pair_f16<P>((unsigned int)w ^ 0x80808080u);
  }
};
template <int NP>
struct HybIn<16, NP> {
  static constexpr int PARTS = 2;
  static constexpr float SCALE = 256.0f;       // Z holds the transform of x / 256
  using word = typename Sample<16, NP>::word;
  typedef short s2v __attribute__((ext_vector_type(2)));
  template <int P>
  __device__ __forceinline__ static void pair(word w, unsigned int &hi, unsigned int &lo) {
    unsigned int v;
    if constexpr (NP == 2) v = P == 0 ? w.x : w.y;
    else v = w;
    v = __builtin_bit_cast(unsigned int, __builtin_elementwise_max(__builtin_bit_cast(s2v, v),
                                                                   (s2v){-32767, -32767}));
    // high bytes offset by 128 under exponent byte 0x64: 1024 + 128 + hi
    const h2v h = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, v ^ 0x80008000u, 0x04030401u)) -
                  (h2v){(_Float16)1152.0f, (_Float16)1152.0f};
    // low bytes under exponent byte 0x44: 4 + lo / 256
    const h2v l = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x44444444u, v, 0x04020400u)) -
                  (h2v){(_Float16)4.0f, (_Float16)4.0f};
    hi = __builtin_bit_cast(unsigned int, h);
    lo = __builtin_bit_cast(unsigned int, l);
  }
};

template <int PARTS>
struct HybFrag {
  h8v v[PARTS][4];       // A operands [hi / lo part][K-block]
};
template <int PARTS>
__device__ __forceinline__ void frag_set(HybFrag<PARTS> &f, int e, unsigned int hi, unsigned int lo) {
  const h2v a = __builtin_bit_cast(h2v, hi);
  f.v[0][e >> 2][2 * (e & 3)] = a[0];
  f.v[0][e >> 2][2 * (e & 3) + 1] = a[1];
  if constexpr (PARTS == 2) {
    const h2v b = __builtin_bit_cast(h2v, lo);
    f.v[PARTS - 1][e >> 2][2 * (e & 3)] = b[0];
    f.v[PARTS - 1][e >> 2][2 * (e & 3) + 1] = b[1];
  }
}

// Stage 1 of NP pols at once (the DFT matrix is read from LDS once for all;
// its high halves once per sample part): (zr, zi)[p] = A[p] x F32, small terms
// first: the matrix's low halves, then its high ones with the samples' low
// parts (int16), then with the high parts, so that four of the sum's steps round
// at full size and not eight.  lane: threadIdx.x % 64 plus an opaque zero where
// the reads must not be hoisted out of the caller's loop.
template <int NP, int PARTS>
__device__ __forceinline__ void dft32_mfma(const HybFrag<PARTS> (&f)[NP], const Dft32K &k, int lane,
                                           f16v (&zr)[NP], f16v (&zi)[NP]) {
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int r = 0; r < 16; ++r) { zr[p][r] = 0.0f; zi[p][r] = 0.0f; }
  // parts first .. last of the samples times one half of the matrix
  auto half = [&](int hl, int first, int last) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const h8v br = k.b[0][kb][hl][lane], bi = k.b[1][kb][hl][lane];
#pragma unroll
      for (int p = 0; p < NP; ++p) {
#pragma unroll
        for (int part = first; part >= last; --part) {
          zr[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[p].v[part][kb], br, zr[p], 0, 0, 0);
          zi[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[p].v[part][kb], bi, zi[p], 0, 0, 0);
        }
      }
    }
  };
  half(1, PARTS - 1, 0);
  if constexpr (PARTS == 2) {
    half(0, 1, 1);
    asm volatile("" : "+v"(lane));             // operands kept for the second part would spill
  }
  half(0, 0, 0);
}

// ---- stage 2 -----------------------------------------------------------------
// Lane constants of stage 2: (tan, cos) of W_(32 m)^(x).
template <int M>
__device__ __forceinline__ void hyb_tw(float2 (&tg)[hyb_ntw(M)], const float2 *tw4096, int lane) {
  constexpr int NT = hyb_ntw(M), OFF = kTwN + kHybOperands + hyb_tw_off(M);
#pragma unroll
  for (int k = 0; k < NT; ++k) tg[k] = tw4096[OFF + 64 * k + lane];
}

// Trades values between the lane halves: afterwards a holds (lower lanes' a,
// lower lanes' b) and b (upper lanes' a, upper lanes' b) in (lower, upper)
// lanes.  The second result passes through an empty asm (this compiler's
// optimiser otherwise merges the two results once they are bit-cast).
__device__ __forceinline__ void half_swap(float &a, float &b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                  __builtin_bit_cast(unsigned, b), false, false);
  unsigned int r0 = r[0], r1 = r[1];
  asm volatile("" : "+v"(r1));
  a = __builtin_bit_cast(float, r0);
  b = __builtin_bit_cast(float, r1);
}

// Stage 2 on one product's result.  M <= 16: x[s M + d] = bin c + 32 d of the
// lane's transform s.  M = 32: x[j] = bin c + 32 (h + 2 j).
template <int M>
__device__ __forceinline__ void hyb_stage2(const f16v &zr, const f16v &zi, const float2 (&tg)[hyb_ntw(M)],
                                           float2 (&x)[16]) {
  if constexpr (M <= 16) {
#pragma unroll
    for (int s = 0; s < 16 / M; ++s) {
      float2 v[M];
#pragma unroll
      for (int a = 0; a < M; ++a) v[a] = make_float2(zr[s * M + a], zi[s * M + a]);
      MDit<M>::run(v, tg);
#pragma unroll
      for (int a = 0; a < M; ++a) x[s * M + a] = v[a];
    }
  } else {
    // a = 8 q + 4 h + i: sizes 2 and 4 over q for each i
    float2 y[4][4];                      // [i][k]
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int q = 0; q < 4; ++q) y[i][q] = make_float2(zr[4 * q + i], zi[4 * q + i]);
      MDit<4>::run(y[i], tg);
      // size 8 across the lane halves: the lane keeps k = h + 2 kappa
      float2 w[4];                       // k = h + 2 j
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        float2 e = y[i][2 * kp], o = y[i][2 * kp + 1];
        half_swap(e.x, o.x);
        half_swap(e.y, o.y);
        if (kp == 0) bfly<false>(e, o, tg[2], w[0], w[2]);
        else bfly<true>(e, o, tg[2], w[1], w[3]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) y[i][j] = w[j];
    }
    // sizes 16 (i, i + 2) and 32 (i = 0, 1)
    float2 z[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j < 2) bfly<false>(y[i][j], y[i + 2][j], tg[3 + j], z[i][j], z[i][j + 4]);
        else bfly<true>(y[i][j], y[i + 2][j], tg[3 + j - 2], z[i][j], z[i][j + 4]);
      }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < 4) bfly<false>(z[0][j], z[1][j], tg[5 + j], x[j], x[j + 8]);
      else bfly<true>(z[0][j], z[1][j], tg[5 + j - 4], x[j], x[j + 8]);
    }
  }
}

// Row rho = lane % 32 of a product as (transform within the product, a).
template <int M>
__device__ __forceinline__ void hyb_row(int rho, int &s, int &a) {
  if constexpr (M <= 16) {
    const int r = 4 * (rho >> 3) + (rho & 3);
    a = r & (M - 1);
    s = r / M + ((rho >> 2) & 1) * (16 / M);
  } else {
    a = rho;
    s = 0;
  }
}

}  // namespace rsk
