// k_fs_a_h.hip -- four-step pass A (k_fs_a's contract) for N1 = 128 .. 512
// with the first 32 points of each sub-transform on the matrix cores
// (dft_hybrid.h).
//
// A wavefront takes a tile of V S adjacent n1 columns (V: columns in 16 bytes
// of a row, S = 1024 / N2): each lane loads 16 bytes of each of its 16 rows
// n2, so the V words of a load belong to V products of the matrix cores, and
// transforms the columns one product after the other; the next tile's loads
// go out before the last product.  No wavefront waits for another one: the
// vector kernel's workgroup synchronised twice per polarisation and stage.
// Lane (c, h) ends with Y[n1][k2 = c + 32 d], so 32 lanes write 32
// consecutive k2 of one n1: runs of tby values in Y's tiled layout.
//
// The four-step twiddle W_N^(n1 k2) = W_N^(n1 (c + 32 h)) W_N^(64 n1 j) (M = 32;
// W_N^(n1 c) W_N^(32 n1 d) below): a lane factor per column times a factor
// common to the column, which the wavefront's lanes compute side by side
// once per tile into a small LDS table.  Looked up per value it would put the
// 32 lanes n1 entries apart, up to a 32-way bank conflict.
#include <type_traits>
#include <utility>

#include "dft_hybrid.h"
#include "kernels.h"

namespace rsk {

// Bytes of a row per load: 16; 8 where the spare registers are short (short
// transforms of one pol or int16 spill otherwise; their tiles are wide all the
// same); narrow: one sample (4 bytes at least), for launches of few tiles,
// whose wavefronts would otherwise transform V products in turn on an empty
// device (8192 points of 1 MiB in one channel: 23 us, the vector kernel 21).
constexpr int fs_a_h_load(int n2, int nbps, int np, int narrow) {
  const int word = np * 2 * nbps / 8;
  return narrow ? (word < 4 ? 4 : word) : n2 <= 128 && (np == 1 || nbps == 16) ? 8 : 16;
}

template <int N2, int R1, int NBPS, int NP, bool Y24, bool NARROW>
__global__ __launch_bounds__(256, 2) void k_fs_a_h(FsArgs a) {
  static_assert(!Y24 || NP == 2, "24-bit intermediate: two pols");
  constexpr int M = N2 / 32, S = 1024 / N2, N1C = R1 * N2, L1 = ilog2(N1C);
  using In = HybIn<NBPS, NP>;
  using W = typename In::word;
  constexpr int LB = fs_a_h_load(N2, NBPS, NP, NARROW);
  typedef unsigned int uld __attribute__((ext_vector_type(LB / 4)));
  constexpr int V = LB / (int)sizeof(W);       // columns per load
  constexpr int CW = V * S;                    // columns of a wavefront's tile
  static_assert(N1C % CW == 0, "whole tiles");
  constexpr int SL = M <= 16 ? 16 / M : 1;     // columns a lane holds per product
  constexpr int DC = M <= 16 ? M : 16;         // values of each
  constexpr int KT = CW * DC;                  // column factors of a tile
  constexpr int TBY = N1C <= 256 ? 16 : 8;     // Y's k2 tile, fs_tile_b(N1C)
  __shared__ Dft32K K;
  __shared__ float2 twl[N2];                   // W_N2^h
  __shared__ float2 twr[N1C];                  // W_N^r, r < N1
  __shared__ float2 ctab[4][KT];               // [wavefront][column of the tile][d or j]
  for (int m = threadIdx.x; m < N2; m += 256) twl[m] = a.tw[m * (kTwN / N2)];
  for (int m = threadIdx.x; m < N1C; m += 256) twr[m] = a.twf[m];
  dft32_consts(K, a.tw, 256, a.isign < 0.0f ? 0x80000000u : 0u);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // item arithmetic stays scalar
  int col = lane & 31;
  const int h = lane >> 5;
  float2 tg[hyb_ntw(M)];
  hyb_tw<M>(tg, a.tw, lane);
  __syncthreads();

  const unsigned long long N = (unsigned long long)N1C * N2;
  constexpr unsigned tiles = N1C / CW;
  const unsigned nsp = a.Nss * a.ynb;          // spectra per channel in Y
  const unsigned items = tiles * a.Nss * a.nbat * a.nch;
  const unsigned stride = gridDim.x * 4;
  int rs, ra;
  hyb_row<M>(col, rs, ra);
  // in words of W: this lane's first row and column group
  unsigned o0 = (unsigned)(ra + M * 4 * h) * N1C + (unsigned)(rs * V);

  uld raw[16];
  auto load = [&](unsigned l) {
    const unsigned tile = l % tiles;
    const unsigned cs = l / tiles;
    const unsigned sp = cs % a.Nss;            // spectrum within its buffer
    const unsigned cb = cs / a.Nss;
    const unsigned b = cb % a.nbat;            // buffer within the batch
    const unsigned cl = cb / a.nbat;           // channel within the chunk
    const W *src = reinterpret_cast<const W *>(a.in[b] + (unsigned long long)(a.c0 + cl) * a.chan_stride) +
                   (unsigned long long)sp * N + tile * CW;
#pragma unroll
    for (int e = 0; e < 16; ++e)
      raw[e] = *reinterpret_cast<const uld *>(src + (o0 + (unsigned)(M * (8 * (e >> 2) + (e & 3))) * N1C));
  };
  // consecutive wavefronts take consecutive tiles, so lines that hold several
  // tiles' columns are shared in one CU's and one XCD's caches
  unsigned l = xcd_remap(blockIdx.x, gridDim.x) * 4 + wv;
  if (l >= items) return;
  load(l);
  for (;;) {
    // the lane's offsets pass through an empty asm per tile: kept live across
    // the loop, the addresses of 16 loads and 16 stores would spill
    asm volatile("" : "+v"(o0), "+v"(col));
    const unsigned ln = l + stride;
    const unsigned tile = l % tiles;
    const unsigned cs = l / tiles;
    const unsigned sp = cs % a.Nss;
    const unsigned cb = cs / a.Nss;
    const unsigned b = cb % a.nbat;
    const unsigned cl = cb / a.nbat;
    const unsigned long long spec = (unsigned long long)cl * nsp + (a.yb0 + b) * a.Nss + sp;
    // spectrum `spec` starts at N * NP float2 (24-bit: N * 12 bytes) into Y
    float2 *dst = Y24 ? reinterpret_cast<float2 *>(reinterpret_cast<unsigned int *>(a.work) + spec * N * 3)
                      : a.work + spec * N * NP;
    // column factors of the tile: entry cc DC + j = W_N^(n1 32 j) (64 j for M = 32)
    team_sync<true>();
#pragma unroll
    for (int q = lane; q < KT; q += 64) {
      const unsigned n1 = tile * CW + (unsigned)(q / DC);
      const unsigned e = n1 * (unsigned)((M == 32 ? 64 : 32) * (q % DC));   // < N
      ctab[wv][q] = cmul(twl[e >> L1], twr[e & (N1C - 1)]);
    }
    team_sync<true>();

    auto product = [&](auto jc) {
      constexpr int j = decltype(jc)::value;
      asm volatile("" : "+v"(col));            // as above, per product
      f16v zr[NP], zi[NP];
      float2 x[NP][16];
      // an opaque zero keeps the DFT matrix in LDS
      int z;
      asm volatile("v_mov_b32 %0, 0" : "=v"(z));
      auto pol = [&](auto pc) {
        constexpr int p = decltype(pc)::value;
        HybFrag<In::PARTS> f[1];
        f16v r1[1], i1[1];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          W w;
          if constexpr (sizeof(W) == 8) w = make_uint2(raw[e][2 * j], raw[e][2 * j + 1]);
          else if constexpr (sizeof(W) == 4) w = raw[e][j];
          else w = (W)(raw[e][j / 2] >> (16 * (j & 1)));
          unsigned int hi, lo = 0;
          In::template pair<p>(w, hi, lo);
          frag_set(f[0], e, hi, lo);
        }
        if constexpr (j == V - 1 && p == NP - 1) {
          if (ln < items) load(ln);
        }
        dft32_mfma<1, In::PARTS>(f, K, lane + z, r1, i1);
        zr[p] = r1[0];
        zi[p] = i1[0];
        __builtin_amdgcn_sched_barrier(0);     // one pol's operands live at a time
      };
      pol(std::integral_constant<int, 0>());
      if constexpr (NP == 2) pol(std::integral_constant<int, NP - 1>());
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        hyb_stage2<M>(zr[p], zi[p], tg, x[p]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int s = 0; s < SL; ++s) {
        // column of slot s of this lane's half
        const unsigned cc = (unsigned)((M <= 16 ? (s + h * SL) * V : 0) + j);
        const unsigned n1 = tile * CW + cc;
        const unsigned e1 = n1 * (unsigned)(M == 32 ? col + 32 * h : col);
        float2 wc = cmul(twl[e1 >> L1], twr[e1 & (N1C - 1)]);
        wc.x *= In::SCALE;
        wc.y *= In::SCALE;
        // (k2 / tby, n1, k2 % tby); 32 k2 further is 32 N1 values further
        const unsigned off = ((unsigned)(col / TBY) * N1C + n1) * TBY + (unsigned)(col % TBY) +
                             (M == 32 ? (unsigned)h * (32u * N1C) : 0u);
#pragma unroll
        for (int d = 0; d < DC; ++d) {
          if (d % 4 == 0) __builtin_amdgcn_sched_barrier(0);   // few factors and addresses live
          const float2 w = cmul(ctab[wv][cc * DC + d], wc);
          const unsigned at = off + (unsigned)((M == 32 ? 64 : 32) * d) * N1C;
          if constexpr (NP == 2) {
            const float2 y0 = cmul(x[0][s * DC + d], w), y1 = cmul(x[NP - 1][s * DC + d], w);
            const float4 yv = make_float4(y0.x, y0.y, y1.x, y1.y);
            if constexpr (Y24) {
              unsigned int *p = reinterpret_cast<unsigned int *>(dst) + 3u * at;
              // runs of 96 bytes (N1 = 512) end within lines, which the L2
              // must put together: streamed they took 324 us instead of 202
              if constexpr (TBY == 16) store_y24(p, yv);
              else *reinterpret_cast<u32x3 *>(p) = pack_y24(yv);
            } else {
              store_y(reinterpret_cast<float4 *>(dst) + at, yv);
            }
          } else {
            store_y(dst + at, cmul(x[0][s * DC + d], w));
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);       // one product's values live at a time
    };
    auto products = [&]<int... J>(std::integer_sequence<int, J...>) {
      (product(std::integral_constant<int, J>()), ...);
    };
    products(std::make_integer_sequence<int, V>());
    if (ln >= items) break;
    l = ln;
  }
}

template <int N2, int R1, int NBPS, bool NARROW>
static int go(int np, const FsArgs &a, unsigned nb, hipStream_t s) {
  const dim3 g(nb), t(256);
  // narrow only where its loads are (not int16 of two pols up to 128 points)
  constexpr bool nw2 = NARROW && fs_a_h_load(N2, NBPS, 2, 1) != fs_a_h_load(N2, NBPS, 2, 0);
  constexpr bool nw1 = NARROW && fs_a_h_load(N2, NBPS, 1, 1) != fs_a_h_load(N2, NBPS, 1, 0);
  if constexpr (N2 < 512) {
    if (np == 2 && a.y24) {
      hipLaunchKernelGGL((k_fs_a_h<N2, R1, NBPS, 2, true, nw2>), g, t, 0, s, a);
      return hipGetLastError() == hipSuccess ? 0 : 1;
    }
  }
  if (np == 2) hipLaunchKernelGGL((k_fs_a_h<N2, R1, NBPS, 2, false, nw2>), g, t, 0, s, a);
  else hipLaunchKernelGGL((k_fs_a_h<N2, R1, NBPS, 1, false, nw1>), g, t, 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <int NBPS, bool NARROW>
static int go_n(int np, const FsArgs &a, unsigned nb, hipStream_t s) {
  switch (a.N1 * 4096 + a.N2) {
    case 128 * 4096 + 64: return go<64, 2, NBPS, NARROW>(np, a, nb, s);
    case 128 * 4096 + 128: return go<128, 1, NBPS, NARROW>(np, a, nb, s);
    case 256 * 4096 + 128: return go<128, 2, NBPS, NARROW>(np, a, nb, s);
    case 256 * 4096 + 256: return go<256, 1, NBPS, NARROW>(np, a, nb, s);
    case 512 * 4096 + 256: return go<256, 2, NBPS, NARROW>(np, a, nb, s);
    case 512 * 4096 + 512: return go<512, 1, NBPS, NARROW>(np, a, nb, s);
  }
  return 2;
}

// Up to N1 = 512.  Beyond, a tile is 4 or 8 columns, rows are read in 16 or
// 32 bytes and Y is written in 64-byte pieces 64 KB apart, which memory takes
// at 3.5 TB/s: 2^20 points 346 us per 256 MiB against the vector kernel's 288,
// 2^19 438 against 342; wider tiles of Y let this kernel write at 5.8 TB/s, but
// pass B then reads pieces and loses more.  The 24-bit Y of 2^18 points comes in
// 96-byte pieces: 205 us per 128 MiB against 171.  Below, 128 MiB of 64
// channels: 2^16 points 203 -> 113 us (6 TB/s), 2^15 178 -> 111, 2^14 169 -> 110,
// 2^13 472 -> 111; one pol of 2^17 286 -> 162.
int fs_a_h_ok(int n1, int n2, int y24) {
  return n2 >= 64 && n1 >= 128 && n1 <= 512 && (n1 == n2 || n1 == 2 * n2) && !(y24 && n2 == 512);
}

int launch_fs_a_h(int nbps, int np, const FsArgs &a, hipStream_t s) {
  if (!fs_a_h_ok((int)a.N1, (int)a.N2, a.y24) || (a.y24 && np != 2) || a.tby != (a.N1 <= 256 ? 16u : 8u) || a.tby != (unsigned)fs_tile_b((int)a.N1) ||
      a.nbat == 0 || a.nbat > (unsigned)kMaxBatch || a.yb0 + a.nbat > a.ynb)
    return 2;
  const unsigned long long spectra = (unsigned long long)a.Nss * a.nbat * a.nch;
  unsigned cw = 0;                             // a tile's columns
  unsigned long long items = 0;
  int narrow = 0;
  for (; narrow < 2; ++narrow) {
    cw = (unsigned)(fs_a_h_load((int)a.N2, nbps, np, narrow) / (np * 2 * nbps / 8)) * (1024u / a.N2);
    if (a.N1 % cw) return 2;
    items = (unsigned long long)(a.N1 / cw) * spectra;
    // enough tiles for a wavefront per SIMD, or nothing narrower
    if (items >= a.grid_a / 2) break;
  }
  if (narrow == 2) narrow = 1;
  if (items == 0 || items > 0x7fffffffull) return 2;
  unsigned long long nb = (items + 3) / 4;
  if (a.grid_a && a.grid_a < nb) nb = a.grid_a;
  if (nbps == 8 && narrow) return go_n<8, true>(np, a, (unsigned)nb, s);
  if (nbps == 8) return go_n<8, false>(np, a, (unsigned)nb, s);
  if (nbps == 16 && narrow) return go_n<16, true>(np, a, (unsigned)nb, s);
  if (nbps == 16) return go_n<16, false>(np, a, (unsigned)nb, s);
  return 2;
}

}  // namespace rsk
