// k_small_r.hip -- fused spectrometer kernel for lengths 2^a 3^b and 2^a 5^b.
//
// k_small's work (unpack, FFT, detect, integrate a chunk of spectra, write
// the FFT-shifted sums; the reference plans these lengths with cuFFT,
// rawspec_gpu.cu:1182-1195) for decimal lengths such as 1000 and 2000 and
// for 3 * 2^a, which Bluestein's identity computes as two transforms of at
// least twice the length.  A Stockham transform with mixed radices: E = 10,
// 20 or 24 elements per thread, every stage's radix a divisor of E, so a thread
// holds E / R whole butterflies of any stage and one kernel per E takes all
// lengths of its family.  The stages' list is an argument (r_plan).
//
// Bound by instruction issue and LDS exchanges, at 2 wavefronts per SIMD (E = 10:
// 3 or 4; E = 24 with four sums, whose sums and values are 192 registers: 1);
// both polarisations share an exchange, in 16-byte elements.  64 MiB of int8, 16
// channels, two polarisations, dumps of 16 spectra of 4 sums, against
// Bluestein's identity: 1000 points 378 -> 100 us, 2000 439 -> 123, 1536 437 ->
// 118, 384 383 -> 141, 250 324 -> 91, 100 385 -> 92; one polarisation, one sum:
// 1000 points 233 -> 77, 1536 306 -> 99.
#include "fft_device.h"
#include "kernels.h"

namespace rsk {

// In-place forward DFT of R points: powers of two, 3, 5, and by the prime
// factor map P * M with coprime P (3 or 5) and M (a power of two), which has
// no twiddles: input (M p + P m) mod R, output k with k = kp mod P, km mod M.
constexpr int odd_part(int r) { return r % 2 ? r : odd_part(r / 2); }
constexpr int crt(int P, int M, int kp, int km) {
  for (int k = 0; k < P * M; ++k)
    if (k % P == kp && k % M == km) return k;
  return 0;
}
template <int R>
__device__ __forceinline__ void r_dft(float2 (&a)[R]) {
  constexpr int P = odd_part(R), M = R / P;
  if constexpr (P == 1) {
    Dft<R>::run(a);
  } else if constexpr (R == 3) {
    constexpr float S = 0.86602540378443864676f;          // sin(2 pi / 3)
    const float2 t = cadd(a[1], a[2]), u = csub(a[1], a[2]);
    const float2 m = make_float2(fmaf(-0.5f, t.x, a[0].x), fmaf(-0.5f, t.y, a[0].y));
    a[0] = cadd(a[0], t);
    a[1] = make_float2(fmaf(S, u.y, m.x), fmaf(-S, u.x, m.y));
    a[2] = make_float2(fmaf(-S, u.y, m.x), fmaf(S, u.x, m.y));
  } else if constexpr (R == 5) {
    constexpr float C1 = 0.30901699437494742410f, C2 = -0.80901699437494742410f;
    constexpr float S1 = 0.95105651629515357212f, S2 = 0.58778525229247312917f;
    const float2 t1 = cadd(a[1], a[4]), t2 = cadd(a[2], a[3]);
    const float2 u1 = csub(a[1], a[4]), u2 = csub(a[2], a[3]);
    const float2 m1 = make_float2(fmaf(C2, t2.x, fmaf(C1, t1.x, a[0].x)), fmaf(C2, t2.y, fmaf(C1, t1.y, a[0].y)));
    const float2 m2 = make_float2(fmaf(C1, t2.x, fmaf(C2, t1.x, a[0].x)), fmaf(C1, t2.y, fmaf(C2, t1.y, a[0].y)));
    const float2 n1 = make_float2(fmaf(S2, u2.x, S1 * u1.x), fmaf(S2, u2.y, S1 * u1.y));
    const float2 n2 = make_float2(fmaf(-S1, u2.x, S2 * u1.x), fmaf(-S1, u2.y, S2 * u1.y));
    a[0] = make_float2(a[0].x + t1.x + t2.x, a[0].y + t1.y + t2.y);
    a[1] = make_float2(m1.x + n1.y, m1.y - n1.x);
    a[4] = make_float2(m1.x - n1.y, m1.y + n1.x);
    a[2] = make_float2(m2.x + n2.y, m2.y - n2.x);
    a[3] = make_float2(m2.x - n2.y, m2.y + n2.x);
  } else {
    float2 b[M][P];
#pragma unroll
    for (int m = 0; m < M; ++m) {
#pragma unroll
      for (int p = 0; p < P; ++p) b[m][p] = a[(M * p + P * m) % R];
      r_dft<P>(b[m]);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      float2 c[M];
#pragma unroll
      for (int m = 0; m < M; ++m) c[m] = b[m][p];
      Dft<M>::run(c);
#pragma unroll
      for (int m = 0; m < M; ++m) a[crt(P, M, p, m)] = c[m];
    }
  }
}

// An exchange element: one sample of every polarisation.
template <int NP> struct RElem { float2 p[NP]; };
template <> struct __attribute__((aligned(16))) RElem<2> { float2 p[2]; };

// One element of padding after every eight: first stages write with a stride
// of their radix, and 8, 20 or 24 elements apart lanes would meet in 2 to 4
// of the 16 (one polarisation: 32) that lie in different banks.
__host__ __device__ __forceinline__ constexpr unsigned r_pos(unsigned pos) { return pos + (pos >> 3); }

// A stage of radix R: butterfly b = j + u T (u < E / R) takes the thread's
// slots u + r E / R, elements b + r N / R, times W_(NS R)^(r (b mod NS)) = tw[r
// (b mod NS) N / (NS R)], and writes (b / NS) NS R + b mod NS + r NS.  b / NS as
// (b magic) >> 22, exact for b < 1024 and NS < 2048 (magic = ceil(2^22 / NS)).
template <int E, int NP, int R, bool FIRST, bool LAST>
__device__ __forceinline__ void r_stage(float2 (&v)[NP][E], RElem<NP> *lds, const float2 *tw, unsigned j,
                                        unsigned T, unsigned N, unsigned NS, unsigned magic) {
  constexpr int NB = E / R;
  const unsigned ts = N / (NS * R);
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const unsigned b = j + u * T;
    unsigned q = b, k = 0;
    if constexpr (!FIRST) {
      q = (b * magic) >> 22;
      k = b - q * NS;
    }
    // one polarisation at a time, its twiddles read through an opaque offset: all
    // twiddles of a butterfly held for both would spill
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float2 a[R];
#pragma unroll
      for (int r = 0; r < R; ++r) a[r] = v[p][u + r * NB];
      if constexpr (!FIRST) {
        unsigned kt = k * ts;
        if constexpr (R >= 10) asm volatile("" : "+v"(kt));
#pragma unroll
        for (int r = 1; r < R; ++r) a[r] = cmul(a[r], tw[kt * r]);
      }
      r_dft<R>(a);
#pragma unroll
      for (int r = 0; r < R; ++r) v[p][u + r * NB] = a[r];
      if constexpr (R >= 10) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!LAST) {
      const unsigned pos = q * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        RElem<NP> e;
#pragma unroll
        for (int p = 0; p < NP; ++p) e.p[p] = v[p][u + r * NB];
        lds[r_pos(pos + r * NS)] = e;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// The stage of radix R, a divisor of E, that is not the last.
template <int E, int NP, bool FIRST>
__device__ __forceinline__ void r_pick(unsigned R, float2 (&v)[NP][E], RElem<NP> *lds, const float2 *tw, unsigned j,
                                       unsigned T, unsigned N, unsigned NS, unsigned magic) {
  if (R == 2) {
    r_stage<E, NP, 2, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
  } else if (R == E / 2) {
    r_stage<E, NP, E / 2, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
  } else if (R == E) {
    r_stage<E, NP, E, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
  } else if constexpr (E % 4 == 0) {
    if (R == 4) {
      r_stage<E, NP, 4, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
    } else if (R == E / 4) {
      r_stage<E, NP, E / 4, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
    } else if constexpr (E == 24) {
      if (R == 8) r_stage<E, NP, 8, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
      else r_stage<E, NP, 3, FIRST, false>(v, lds, tw, j, T, N, NS, magic);
    }
  }
}

template <int E, int NBPS, int NP, int PMODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(E > 10 && PMODE != 1 ? 1 : 2)))
void k_small_r(SmallArgs a, RPlan rp) {
  constexpr int Q = nq<PMODE>();
  using S = Sample<NBPS, NP>;
  using W = typename S::word;
  using X = RElem<NP>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const unsigned N = a.nt, T = N / E, slots = rp.slots;
  const unsigned len = r_pos(N - 1) + 1;
  X *xl = reinterpret_cast<X *>(smem);                     // [slots][len], then the sums
  float2 *tw = reinterpret_cast<float2 *>(smem + (size_t)slots * len * sizeof(X));

  const unsigned c = blockIdx.x / a.bpc;
  const unsigned rest = blockIdx.x - c * a.bpc;
  const unsigned gb = rest / a.G;
  const unsigned chunk = rest - gb * a.G;
  const unsigned g0 = gb * a.gpw;
  const unsigned tid = threadIdx.x;
  // the last wavefront may not be full: its other threads repeat thread 0's work
  // (the same values to the same places) and write no sums
  const bool act = tid < slots * T;
  const unsigned slot = act ? tid / T : 0u;
  const unsigned j0 = act ? tid - slot * T : 0u;
  const unsigned gi = slot / a.spg, si = slot - gi * a.spg;
  const unsigned g = g0 + gi;
  const bool gvalid = g < a.Ng;
  for (unsigned n = tid; n < N; n += blockDim.x) tw[n] = a.chirp[n];
  __syncthreads();

  const W *src = reinterpret_cast<const W *>(a.in + (unsigned long long)c * a.chan_stride);
  const unsigned s0 = (gvalid ? g : 0u) * a.na_buf + chunk * a.chunk;
  X *lds = xl + slot * len;
  float acc[E][Q];
#pragma unroll
  for (int m = 0; m < E; ++m)
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[m][q] = 0.0f;

  const unsigned iters = (a.chunk + a.spg - 1) / a.spg;
  for (unsigned it = 0; it < iters; ++it) {
    // opaque: the spectra's and stages' addresses are formed anew rather than
    // kept in 2 E registers
    unsigned j = j0;
    asm volatile("" : "+v"(j));
    const unsigned sl = si + it * a.spg;
    const bool valid = gvalid && sl < a.chunk;
    const W *sp = src + (unsigned long long)(s0 + (valid ? sl : 0u)) * N + j;
    float2 v[NP][E];
    {
      W raw[E];
#pragma unroll
      for (int m = 0; m < E; ++m) raw[m] = sp[m * T];
#pragma unroll
      for (int m = 0; m < E; ++m) {
        float2 o[NP];
        S::cvt(raw[m], o, a.isign);
#pragma unroll
        for (int p = 0; p < NP; ++p) v[p][m] = o[p];
      }
    }
    // all stages but the last leave their values in LDS; the last, of radix E,
    // keeps bin j + m T in slot m
    unsigned NS = 1;
    for (unsigned st = 0; st + 1 < rp.n; ++st) {
      const unsigned R = rp.r[st], mg = rp.magic[st];
      if (st == 0) r_pick<E, NP, true>(R, v, lds, tw, j, T, N, NS, mg);
      else r_pick<E, NP, false>(R, v, lds, tw, j, T, N, NS, mg);
      asm volatile("" : "+v"(j));
      __syncthreads();
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const X e = lds[r_pos(j + m * T)];
#pragma unroll
        for (int p = 0; p < NP; ++p) v[p][m] = e.p[p];
      }
      __syncthreads();
      NS *= R;
    }
    asm volatile("" : "+v"(j));
    __builtin_amdgcn_sched_barrier(0);
    r_stage<E, NP, E, false, true>(v, lds, tw, j, T, N, NS, rp.magic[rp.n - 1]);
    if (valid) {
#pragma unroll
      for (int m = 0; m < E; ++m) detect_raw_np<PMODE, NP>(acc[m], v[0][m], v[NP - 1][m]);
    }
  }
#pragma unroll
  for (int m = 0; m < E; ++m) detect_finish<PMODE>(acc[m], a.gam);

  float *base = a.direct ? a.acc : a.part;
  const bool accum = a.direct && !a.first;
  const unsigned hs = N / 2;                               // bin k goes to (k + N / 2) mod N
  if (a.spg == 1) {
    const unsigned gg = g0 + slot;
    if (!act || gg >= a.Ng) return;
    float *bg = a.direct ? base + (((unsigned long long)gg * Q) * a.Nc + c) * N
                         : base + ((((unsigned long long)c * a.Ng + gg) * a.G + chunk) * Q) * N;
    const unsigned long long qstride = a.direct ? (unsigned long long)a.Nc * N : N;
    const float sc = a.direct ? a.scale : 1.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      float *bq = bg + q * qstride;
#pragma unroll
      for (int m = 0; m < E; ++m) {
        const unsigned k = j0 + m * T + hs, pos = k >= N ? k - N : k;
        float val = acc[m][q] * sc;
        if (accum) val += bq[pos];
        bq[pos] = val;
      }
    }
    return;
  }
  // groups of spg >= 2 slots, as k_small: the upper half parks its sums, the
  // lower half adds its own, the write-out adds the half slots in order
  float *red = reinterpret_cast<float *>(smem);
  const unsigned half = a.spg >> 1;
  if (act && si >= half) {
#pragma unroll
    for (int m = 0; m < E; ++m)
#pragma unroll
      for (int q = 0; q < Q; ++q) red[((gi * half + si - half) * Q + q) * N + j0 + m * T] = acc[m][q];
  }
  __syncthreads();
  if (act && si < half) {
#pragma unroll
    for (int m = 0; m < E; ++m)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        float *r = red + ((gi * half + si) * Q + q) * N + j0 + m * T;
        *r = acc[m][q] + *r;
      }
  }
  __syncthreads();
  const unsigned nout = a.gpw * Q * N;
  for (unsigned idx = tid; idx < nout; idx += blockDim.x) {
    const unsigned go = idx / (Q * N), r2 = idx - go * (Q * N), q = r2 / N, jo = r2 - q * N;
    const unsigned k = jo >= hs ? jo - hs : jo + N - hs;
    const unsigned gg = g0 + go;
    if (gg >= a.Ng) break;
    const float *rp0 = red + ((go * half) * Q + q) * N + k;
    float sum = rp0[0];
    for (unsigned s2 = 1; s2 < half; ++s2) sum += rp0[s2 * Q * N];
    if (a.direct) {
      float *o = base + (((unsigned long long)gg * Q + q) * a.Nc + c) * N + jo;
      const float val = sum * a.scale;
      *o = accum ? *o + val : val;
    } else {
      base[((((unsigned long long)c * a.Ng + gg) * a.G + chunk) * Q + q) * N + jo] = sum;
    }
  }
}

// LDS of one slot and of the twiddles
static unsigned r_slot_bytes(unsigned n, int np) { return (n + (n - 1) / 8) * 8u * (unsigned)np; }

// The stages of an n-point transform: E = 24 for 3 * 2^a * 3^b with 8 | n; for 5 *
// 2^a * 5^b 10, or 20 where 4 | n and it takes fewer stages, for four sums
// only where 10 does not make n (20 would hold 160 registers of values and sums: 1
// wavefront per SIMD) (1000 points as 10, 10,
// 10 with 100 threads 100 us, as 5, 10, 20 with 50 149; 2000 as 5, 20, 20); as few
// radices (divisors of E) as make n, ascending (a first stage of radix 3 or 5
// writes without bank conflicts).  Slots: as many spectra as 256 threads and 64
// KB of LDS hold, a power of two, at most 16.
bool r_plan(unsigned n, int np, int pmode, RPlan &rp) {
  if (n < kRMinN || n > 2048) return false;
  unsigned m = n;
  const unsigned P = n % 3 == 0 ? 3 : 5;
  while (m % 2 == 0) m /= 2;
  if (m == 1) return false;
  while (m % P == 0) m /= P;
  if (m != 1) return false;
  const unsigned dv24[] = {24, 12, 8, 6, 4, 3, 2, 0}, dv20[] = {20, 10, 5, 4, 2, 0}, dv10[] = {10, 5, 2, 0};
  const unsigned *dv[] = {P == 3 ? dv24 : dv10, P == 3 ? nullptr : dv20};
  rp.n = kRMaxStages + 1;
  for (int f = 0; f < 2 && dv[f]; ++f) {
    const unsigned E = dv[f][0];
    if (n % E || (f == 1 && pmode != 1 && rp.n <= kRMaxStages)) continue;
    // the last radix is E; fewest stages before it by depth-first search, larger
    // radices first
    unsigned best[kRMaxStages], nb = kRMaxStages, cur[kRMaxStages];
    auto search = [&](auto &&self, unsigned left, unsigned i, unsigned from) -> void {
      if (left == 1) {
        nb = i;
        for (unsigned k = 0; k < i; ++k) best[k] = cur[k];
        return;
      }
      for (unsigned k = from; dv[f][k] && i + 1 < nb; ++k)
        if (left % dv[f][k] == 0) {
          cur[i] = dv[f][k];
          self(self, left / dv[f][k], i + 1, k);
        }
    };
    search(search, n / E, 0, 0);
    if (nb == kRMaxStages || nb + 1 >= rp.n) continue;
    rp.e = E;
    rp.n = nb + 1;
    unsigned ns = 1;
    for (unsigned i = 0; i <= nb; ++i) {
      rp.r[i] = i < nb ? best[nb - 1 - i] : E;
      rp.magic[i] = ((1u << 22) + ns - 1) / ns;
      ns *= rp.r[i];
    }
  }
  if (rp.n > kRMaxStages) return false;
  const unsigned t = n / rp.e;
  rp.slots = 1;
  while (rp.slots < 16 && 2 * rp.slots * t <= 256 && 2 * rp.slots * r_slot_bytes(n, np) + 8 * n <= 65536) rp.slots *= 2;
  rp.threads = (rp.slots * t + 63) / 64 * 64;
  return true;
}

template <int E, int NBPS>
static int go_r(int np, int pmode, const SmallArgs &a, const RPlan &rp, unsigned nb, unsigned lds, hipStream_t s) {
  const dim3 g(nb), t(rp.threads);
  if (np == 1) hipLaunchKernelGGL((k_small_r<E, NBPS, 1, 1>), g, t, lds, s, a, rp);
  else if (pmode == 1) hipLaunchKernelGGL((k_small_r<E, NBPS, 2, 1>), g, t, lds, s, a, rp);
  else if (pmode == 4) hipLaunchKernelGGL((k_small_r<E, NBPS, 2, 4>), g, t, lds, s, a, rp);
  else if (pmode == -4) hipLaunchKernelGGL((k_small_r<E, NBPS, 2, -4>), g, t, lds, s, a, rp);
  else return 2;
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

int launch_small_r(int nbps, int np, int pmode, const SmallArgs &a, const RPlan &rp, unsigned nblocks,
                   hipStream_t s) {
  if (nblocks == 0) return 0;
  RPlan w;
  if (!r_plan(a.nt, np, pmode, w) || w.e != rp.e || w.slots != rp.slots || w.threads != rp.threads || w.n != rp.n ||
      a.spg * a.gpw != rp.slots || !a.chirp || (np != 1 && np != 2))
    return 2;
  const unsigned lds = rp.slots * r_slot_bytes(a.nt, np) + 8 * a.nt;
  if (nbps == 8)
    return rp.e == 24 ? go_r<24, 8>(np, pmode, a, rp, nblocks, lds, s)
         : rp.e == 20 ? go_r<20, 8>(np, pmode, a, rp, nblocks, lds, s) : go_r<10, 8>(np, pmode, a, rp, nblocks, lds, s);
  if (nbps == 16)
    return rp.e == 24 ? go_r<24, 16>(np, pmode, a, rp, nblocks, lds, s)
         : rp.e == 20 ? go_r<20, 16>(np, pmode, a, rp, nblocks, lds, s) : go_r<10, 16>(np, pmode, a, rp, nblocks, lds, s);
  return 2;
}

}  // namespace rsk
