// int4 x bf16 GEMM for many activation rows (prompts): Y[M, N] = X[M, K] . dq[N, K]^T on the matrix
// cores, the weights dequantised straight into MFMA operands, never written back as bf16.
//
// A workgroup of KW ways of NW waves computes BN = 16 NW NB weight rows x BM = 16 MB activation rows,
// each way over its part of the K groups (the ways' sums meet in LDS, in way order). Wave w of a way
// owns weight rows [16 NB w, 16 NB (w + 1)) of the tile, so no weight is dequantised twice in a
// workgroup and the weights need no LDS; X is what a way's waves share: one 128-group of its BM rows
// at a time in LDS, double-buffered, the next group's X and weights in flight in registers
// meanwhile (one barrier per group). Weights are the MFMA's A operand, so a lane ends with four
// consecutive weight rows of one activation row: RoPE pairs and gate/up pairs (adjacent packed
// rows) meet in one lane.
//
// What bounds it: matrix-core time plus what does not hide under it. 2048 x 16384 x 2560 takes 228 us
// (753 TFLOP/s; 64 launches of the 32-row kernel took 1489). In timing builds of it the MFMAs and
// barriers alone took 158 us, the dequantisation alone about 100: a v_dot2_f32_bf16 of the dequantisation
// runs on the matrix pipe itself (measured: beside a wave that issues MFMAs it gets next to no
// slots, where a v_fma_f32 keeps its rate), and other vector instructions issue at 0.6 of their rate beside 16x16 MFMAs.
// Measured and not taken: the next group's dequantisation interleaved with the MFMAs by hand (258 us), 32x32x16
// MFMAs (250; they leave the vector ALUs free, but need twice the LDS reads per wave).
//
// The ways are for calls of few tiles, where a group's memory latency, not its work, is what a step
// costs: 32 rows x 16384 x 2560 (256 tiles) takes 20 steps of one way or 5 of four, 64 rows 19 and
// 13 us; 512 x 3584 x 2560 (448 tiles) 28 us with one way and 21 with two.
// Two groups requested ahead instead of one (WD, XD) gain 7-10% with one way on the tiled layout (2048 x
// 16384 x 2560 222 -> 206 us), and lose with more ways (the registers cost a workgroup per CU).
#pragma once
#include <type_traits>
#include "fl_common.h"

struct GemmArgs {
  const uint32_t* q;   // [N, K/8], row layout or (TILED) fl_tile_int4's
  const uint32_t* sz;  // [N, K/128]
  const uint16_t* x;   // [M, K] bf16
  int m, n, k;
  int nblk, mblk;      // tiles along N and M
  int splits, gps;     // K cut into `splits` parts of gps 128-groups
};

// Workgroups: the tiles of one (weight block, K part) along M run next to each other on one XCD
// (blockIdx % 8 picks the XCD), so a weight tile comes from HBM once, into one L2.
inline unsigned gemm_grid(const GemmArgs& a) {
  return 8u * (unsigned)((a.nblk * a.splits + 7) / 8) * (unsigned)a.mblk;
}

// Epi(n, m, v, split): v[i] = the (partial) sum of weight row n + i and activation row m; n is a
// multiple of 4, rows past N or M are not filtered out.
template <bool TILED, int NW, int KW, int NB, int MB, int WD, int XD, class Epi>
__global__ __launch_bounds__(64 * NW * KW, NW * KW > 8 ? 4 : 2) void k_gemm_rows(GemmArgs a, Epi epi) {
  constexpr int BN = 16 * NW * NB, BM = 16 * MB;
  constexpr int RP = 4 * NW, XI = BM / RP;  // X rows per pass of a way's threads, passes
  constexpr int RED = (KW - 1) * NW * 64 * NB * MB * 16;  // the ways' sums, in X's place at the end
  constexpr int XS = KW * 2 * BM * 256;
  __shared__ __align__(16) unsigned char smem[XS > RED ? XS : RED];
  const int lane = threadIdx.x & 63, r = lane & 15, c = lane >> 4;
  const int wv0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wave = wv0 % NW, way = wv0 / NW, tid = wave * 64 + lane;  // within the way
  unsigned char (*const xs)[BM * 256] = reinterpret_cast<unsigned char (*)[BM * 256]>(smem + way * (2 * BM * 256));
  const int j = (int)(blockIdx.x >> 3), u = (j / a.mblk) * 8 + (int)(blockIdx.x & 7);
  if (u >= a.nblk * a.splits) return;
  const int split = u % a.splits, G = a.k >> 7;
  const int m0 = (j % a.mblk) * BM, n0 = (u / a.splits) * BN + wave * (16 * NB);
  // this way's groups; every way passes the same number of barriers
  const int gs0 = split * a.gps, gs1 = min(G, gs0 + a.gps), per = (gs1 - gs0 + KW - 1) / KW;
  const int g0 = gs0 + way * per, g1 = min(gs1, g0 + per);
  // range-checked: rows past M or N read as zeros
  const auto xr = buf_rsrc(a.x, (uint32_t)a.m * (uint32_t)a.k * 2u);
  const auto wr = buf_rsrc(a.q, (uint32_t)a.n * (uint32_t)(a.k >> 1));
  const auto sr = buf_rsrc(a.sz, (uint32_t)a.n * (uint32_t)G * 4u);
  // X: thread -> rows (tid >> 4) + RP i, 16-byte unit tid & 15 of the group
  const uint32_t xoff = ((uint32_t)(m0 + (tid >> 4)) * (uint32_t)a.k + (uint32_t)(tid & 15) * 8u) * 2u;
  const uint32_t xstep = (uint32_t)a.k * (2u * RP);
  const uint32_t woff = TILED ? (uint32_t)(n0 >> 4) * (uint32_t)G * 1024u + (uint32_t)lane * 16u
                              : (uint32_t)(n0 + r) * (uint32_t)(a.k >> 1) + (uint32_t)c * 16u;
  const uint32_t wstep = TILED ? (uint32_t)G * 1024u : (uint32_t)a.k * 8u;  // 16 rows, bytes
  const uint32_t soff = (uint32_t)(n0 + r) * (uint32_t)G * 4u;
  // requested ahead: the weights of WD groups, X of XD (past the way's last group: no memory access)
  uint4 xv[XD][XI], wv[WD][NB];
  uint32_t sv[WD][NB];
  auto load_w = [&](int g, uint4 (&w)[NB], uint32_t (&s)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      w[b] = buf_ld128(wr, g < g1 ? woff + (uint32_t)b * wstep + (uint32_t)g * (TILED ? 1024u : 64u) : 0xFFFFFFF0u);
      s[b] = buf_ld32(sr, g < g1 ? soff + (uint32_t)b * (uint32_t)G * 64u + (uint32_t)g * 4u : 0xFFFFFFF0u);
    }
  };
  auto load_x = [&](int g, uint4 (&x)[XI]) {
#pragma unroll
    for (int i = 0; i < XI; ++i)
      x[i] = buf_ld128(xr, g < g1 ? xoff + (uint32_t)i * xstep + (uint32_t)g * 256u : 0xFFFFFFF0u);
  };
  // LDS: row of 16 slots of 16 bytes, slot s of row t at s ^ (t & 15) (16 lanes reading one slot
  // of 16 rows touch every bank once). Row layout: slot = the 16-byte unit. Tiled layout: the dot
  // of tiles 2tp, 2tp + 1 takes columns 32tp + 4c + 0..3 and + 16 (unit_mma_t), kept as slot 4tp + c.
  auto store = [&](int buf, const uint4 (&xv)[XI]) {
    const int t = tid >> 4, un = tid & 15;
    unsigned char* row = xs[buf] + t * 256;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int sw = (t + i * RP) & 15;
      if constexpr (TILED) {
        const int s0 = (un & 12) + 2 * (un & 1), half = (un >> 1) & 1;
        *reinterpret_cast<uint2*>(row + i * (RP * 256) + ((s0 ^ sw) * 16) + half * 8) = make_uint2(xv[i].x, xv[i].y);
        *reinterpret_cast<uint2*>(row + i * (RP * 256) + (((s0 + 1) ^ sw) * 16) + half * 8) = make_uint2(xv[i].z, xv[i].w);
      } else {
        *reinterpret_cast<uint4*>(row + i * (RP * 256) + ((un ^ sw) * 16)) = xv[i];
      }
    }
  };
  fl_f32x4 acc[NB][MB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[b][i] = fl_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const MxLane mx = mx_lane();
  load_x(g0, xv[0]);
#pragma unroll
  for (int i = 0; i < WD; ++i) load_w(g0 + i, wv[i], sv[i]);
  store(0, xv[0]);
#pragma unroll
  for (int i = 1; i < XD; ++i) load_x(g0 + i, xv[i]);
  // one group: its operands are in wv[s] and LDS buffer s & 1
  auto group = [&](auto stage, int g) {
    constexpr int s = decltype(stage)::value, buf = s & 1;
    uint4 wc[NB];
    uint32_t sc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      wc[b] = wv[s % WD][b];
      sc[b] = sv[s % WD][b];
    }
    lds_barrier();
    load_w(g + WD, wv[s % WD], sv[s % WD]);
    load_x(g + XD, xv[s % XD]);
    if (KW > 1 && g >= g1) return;  // fewer groups than the other ways: its barriers only
    const unsigned char* xrow = xs[buf] + r * 256;
    auto mma = [&](int slot, const uint4 (&w)[NB]) {
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const uint4 xf = *reinterpret_cast<const uint4*>(xrow + i * 4096 + ((slot ^ r) * 16));
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(fl_bf16x8, w[b]),
                                                              __builtin_bit_cast(fl_bf16x8, xf), acc[b][i], 0, 0, 0);
      }
    };
    if constexpr (TILED) {
      // unit_dq_t's two exact steps, tiles 2tp, 2tp + 1 of every block together
      fl_s16x4 bs[NB];
      fl_f32x4 c1[NB], c2[NB];
      const fl_s16x4 ai = mx_s4(0x3F803F80u & mx.mlo, 0x3F803F80u & mx.mhi);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t sb = sc[b] & 0xFFFFu, sp = sb | (sb << 16);
        bs[b] = mx_s4(sp & mx.mlo, sp & mx.mhi);
        const float c1v = -136.0f * bf2f(sb), zv = bf2f(sc[b] >> 16);
        c1[b] = fl_f32x4{c1v, c1v, c1v, c1v};
        c2[b] = fl_f32x4{zv, zv, zv, zv};
      }
#pragma unroll
      for (int tp = 0; tp < 4; ++tp) {
        fl_f32x4 d[NB][2];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const uint32_t v[4] = {wc[b].x, wc[b].y, wc[b].z, wc[b].w};
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int t = 2 * tp + e;
            const uint32_t lo = v[t >> 2] >> (4 * (t & 3)), hi = v[2 + (t >> 2)] >> (4 * (t & 3));
            d[b][e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(
                mx_s4((lo & mx.mask) | mx.magic, (hi & mx.mask) | mx.magic), bs[b], c1[b], 0, 0, 0);
          }
        }
        uint32_t p[NB][2][2];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            p[b][e][0] = pack_bf16x2(d[b][e][0], d[b][e][1]);
            p[b][e][1] = pack_bf16x2(d[b][e][2], d[b][e][3]);
          }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 2; ++e)
            d[b][e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ai, mx_s4(p[b][e][0], p[b][e][1]), c2[b], 0, 0, 0);
        uint4 w[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
          w[b] = make_uint4(pack_bf16x2(d[b][0][0], d[b][0][1]), pack_bf16x2(d[b][0][2], d[b][0][3]),
                            pack_bf16x2(d[b][1][0], d[b][1][1]), pack_bf16x2(d[b][1][2], d[b][1][3]));
        mma(4 * tp + c, w);
      }
    } else {
      uint32_t d[NB][4][4];
#pragma unroll
      for (int b = 0; b < NB; ++b) dq32(wc[b], dq_const(sc[b]), d[b]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint4 w[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) w[b] = make_uint4(d[b][0][e], d[b][1][e], d[b][2][e], d[b][3][e]);
        mma(4 * c + e, w);
      }
    }
    if (g + 1 < g1) store(buf ^ 1, xv[(s + 1) % XD]);
  };
  constexpr int UN = WD < 2 ? 2 : WD;  // the loop unrolled so that every buffer's index is fixed
  for (int g = g0; g < g0 + per; g += UN) {
    group(std::integral_constant<int, 0>{}, g);
    if (g + 1 < g0 + per) group(std::integral_constant<int, 1>{}, g + 1);
    if constexpr (UN > 2) {
      if (g + 2 < g0 + per) group(std::integral_constant<int, 2>{}, g + 2);
      if (g + 3 < g0 + per) group(std::integral_constant<int, 3>{}, g + 3);
    }
  }
  if constexpr (KW > 1) {  // the ways' sums, added in way order
    lds_barrier();
    fl_f32x4* red = reinterpret_cast<fl_f32x4*>(smem);
    if (way > 0) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < MB; ++i) red[((way - 1) * NB * MB + b * MB + i) * (NW * 64) + tid] = acc[b][i];
    }
    lds_barrier();
    if (way > 0) return;
#pragma unroll
    for (int k = 0; k < KW - 1; ++k)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[b][i] += red[(k * NB * MB + b * MB + i) * (NW * 64) + tid];
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < MB; ++i) epi(n0 + 16 * b + 4 * c, m0 + 16 * i + r, acc[b][i], split);
}
