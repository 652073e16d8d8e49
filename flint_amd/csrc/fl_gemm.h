// int4 x bf16 GEMM for many activation rows (prompts): Y[M, N] = X[M, K] . dq[N, K]^T on the matrix
// cores, the weights dequantised straight into MFMA operands, never written back as bf16.
//
// A workgroup of NW waves computes BN = 16 NW NB weight rows x BM = 16 MB activation rows. Wave w
// owns weight rows [16 NB w, 16 NB (w + 1)) of the tile, so no weight is dequantised twice in a
// workgroup and the weights need no LDS; X is what the waves share: one 128-group of its BM rows
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
#pragma once
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
template <bool TILED, int NW, int NB, int MB, class Epi>
__global__ __launch_bounds__(64 * NW, 2) void k_gemm_rows(GemmArgs a, Epi epi) {
  constexpr int BN = 16 * NW * NB, BM = 16 * MB;
  constexpr int RP = 4 * NW, XI = BM / RP;  // X rows per pass of the workgroup's threads, passes
  __shared__ __align__(16) unsigned char xs[2][BM * 256];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, c = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = (int)(blockIdx.x >> 3), u = (j / a.mblk) * 8 + (int)(blockIdx.x & 7);
  if (u >= a.nblk * a.splits) return;
  const int split = u % a.splits, G = a.k >> 7;
  const int m0 = (j % a.mblk) * BM, n0 = (u / a.splits) * BN + wave * (16 * NB);
  const int g0 = split * a.gps, g1 = min(G, g0 + a.gps);
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
  uint4 xv[XI], wv[NB];
  uint32_t sv[NB];
  auto load = [&](int g) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      wv[b] = buf_ld128(wr, woff + (uint32_t)b * wstep + (uint32_t)g * (TILED ? 1024u : 64u));
      sv[b] = buf_ld32(sr, soff + (uint32_t)b * (uint32_t)G * 64u + (uint32_t)g * 4u);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) xv[i] = buf_ld128(xr, xoff + (uint32_t)i * xstep + (uint32_t)g * 256u);
  };
  // LDS: row of 16 slots of 16 bytes, slot s of row t at s ^ (t & 15) (16 lanes reading one slot
  // of 16 rows touch every bank once). Row layout: slot = the 16-byte unit. Tiled layout: the dot
  // of tiles 2tp, 2tp + 1 takes columns 32tp + 4c + 0..3 and + 16 (unit_mma_t), kept as slot 4tp + c.
  auto store = [&](int buf) {
    const int t = tid >> 4, sw = t & 15, un = tid & 15;
    unsigned char* row = xs[buf] + t * 256;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
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
  load(g0);
  store(0);
  uint4 wc[NB];
  uint32_t sc[NB];
  for (int g = g0; g < g1; ++g) {
    const int buf = (g - g0) & 1;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      wc[b] = wv[b];
      sc[b] = sv[b];
    }
    lds_barrier();
    if (g + 1 < g1) load(g + 1);
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
    if (g + 1 < g1) store(buf ^ 1);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < MB; ++i) epi(n0 + 16 * b + 4 * c, m0 + 16 * i + r, acc[b][i], split);
}
