// int4 x bf16 GEMM for many activation rows (prompts): Y[M, N] = X[M, K] . dq[N, K]^T on the matrix
// cores, the weights dequantised straight into MFMA operands, never written back as bf16.
//
// A workgroup of KW ways of NW waves computes BN = 16 NW weight rows x BM = 16 MB activation rows,
// each way over its part of the K groups (the ways' sums meet in LDS, in way order). Wave w of a way
// owns weight rows [16 w, 16 (w + 1)) of the tile, so no weight is dequantised twice in a
// workgroup and the weights need no LDS; X is what a way's waves share: one 128-group of its BM rows
// at a time in LDS, double-buffered, the next group's X and weights in flight in registers
// meanwhile (one barrier per group). Weights are the MFMA's A operand, so a lane ends with four
// consecutive weight rows of one activation row: RoPE pairs and gate/up pairs (adjacent packed
// rows) meet in one lane.
//
// What bounds it: matrix-core time plus vector time, which hardly overlap here. 2048 x 16384 x 2560 in
// 128 x 128 tiles took 228 us (64 launches of the former 32-row kernel 1489); in timing builds the MFMAs
// and barriers alone took 158 us, the dequantisation alone about 100. A v_dot2_f32_bf16 of the dequantisation
// runs on the matrix pipe itself (measured: beside a wave that issues MFMAs it gets next to no slots, where a
// v_fma_f32 keeps its rate), and other vector instructions issue at 0.6 of their rate beside 16x16 MFMAs.
// Calls of many tiles take k_gemm_big below instead (210 us).
//
// The ways are for calls of few tiles, where a group's memory latency, not its work, is what a step
// costs: 32 rows x 16384 x 2560 (256 tiles) takes 20 steps of one way or 5 of four, 64 rows 19 and
// 13 us; 512 x 3584 x 2560 (448 tiles) 28 us with one way and 21 with two.
// Two groups requested ahead instead of one (WD, XD) gain 7-10% with one way on the tiled layout (2048 x
// 16384 x 2560 222 -> 206 us). They cost with more ways, though a CU holds as many workgroups then (LDS sets their
// number): prompts of 64 / 512 tokens, 12 layers, 835 / 1901 us with one group ahead, 931 / 1924 with two; row layout 333 x
// 2570 x 2560 17.5 and 21.3 (two of the weights alone 18.5), 5 x 2560 x 8192 13.6 and 14.8.
#pragma once
#include <algorithm>
#include <type_traits>
#include "fl_common.h"

struct GemmArgs {
  const uint32_t* q;   // [N, K/8], row layout or (TILED) fl_tile_int4's
  const uint32_t* sz;  // [N, K/128]
  const uint16_t* x;   // [M, K] bf16
  int m, n, k;
  int nblk, mblk;      // tiles along N and M
  int splits, gps;     // K cut into `splits` parts of gps 128-groups
  int mper;            // tiles along M of one block of the launch order

  // tiles of bn x bm; X blocks of about 3 MB
  void tile(int bn, int bm) {
    nblk = (n + bn - 1) / bn;
    mblk = (m + bm - 1) / bm;
    const long rows = std::max(1L, (3L << 20) / (2L * gps * FL_GROUP));
    mper = (int)std::max(1L, std::min<long>(mblk, rows / bm));
  }
};

// Workgroups: blockIdx % 8 picks the XCD. Along M the tiles are taken in blocks of `mper`, small
// enough that a block's X stays in an XCD's L2 (4 MB); within a block, the tiles of one (weight block, K
// part) run next to each other on one XCD, so a weight tile comes from HBM once per block, into one L2.
// The last units % 8 of these are dealt in eight equal runs of tiles instead: 333 x 2570 x 2560 (41 weight
// blocks of 6 tiles) otherwise gives one XCD 36 of 246 four-way workgroups for its 32 CUs and takes 27 us, not 16.
__host__ __device__ inline int gemm_run(int units, int mper) {  // tiles of an XCD in a block of mper along M
  return (units >> 3) * mper + (((units & 7) * mper + 7) >> 3);
}
inline unsigned gemm_grid(const GemmArgs& a) {
  const int u = a.nblk * a.splits;
  return 8u * (unsigned)(a.mblk / a.mper * gemm_run(u, a.mper) + gemm_run(u, a.mblk % a.mper));
}
__device__ __forceinline__ bool gemm_tile(const GemmArgs& a, int& u, int& mb) {
  const int units = a.nblk * a.splits, run = gemm_run(units, a.mper), xcd = (int)(blockIdx.x & 7);
  const int j = (int)(blockIdx.x >> 3), blk = j / run, jj = j - blk * run;
  const int mper = min(a.mper, a.mblk - blk * a.mper), whole = (units >> 3) * mper;
  if (jj < whole) {
    u = (jj / mper) * 8 + xcd;
    mb = blk * a.mper + jj % mper;
    return true;
  }
  const int share = ((units & 7) * mper + 7) >> 3, i = xcd * share + jj - whole;
  u = (units & ~7) + i / mper;
  mb = blk * a.mper + i % mper;
  return jj - whole < share && u < units;
}

// Epi(n, m, v, split): v[i] = the (partial) sum of weight row n + i and activation row m; n is a
// multiple of 4, rows past N or M are not filtered out.
template <bool TILED, int NW, int KW, int MB, int WD, int XD, class Epi>
__global__ __launch_bounds__(64 * NW * KW, NW * KW > 8 ? 4 : 2) void k_gemm_rows(GemmArgs a, Epi epi) {
  static_assert((WD == 1 || WD == 2) && (XD == 1 || XD == 2), "groups requested ahead");
  constexpr int BN = 16 * NW, BM = 16 * MB;
  constexpr int RP = 4 * NW, XI = BM / RP;  // X rows per pass of a way's threads, passes
  constexpr int RED = (KW - 1) * NW * 64 * MB * 16;  // the ways' sums, in X's place at the end
  constexpr int XS = KW * 2 * BM * 256;
  __shared__ __align__(16) unsigned char smem[XS > RED ? XS : RED];
  const int lane = threadIdx.x & 63, r = lane & 15, c = lane >> 4;
  const int wv0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wave = wv0 % NW, way = wv0 / NW, tid = wave * 64 + lane;  // within the way
  unsigned char (*const xs)[BM * 256] = reinterpret_cast<unsigned char (*)[BM * 256]>(smem + way * (2 * BM * 256));
  int u, mb;
  if (!gemm_tile(a, u, mb)) return;
  const int split = u % a.splits, G = a.k >> 7;
  const int m0 = mb * BM, n0 = (u / a.splits) * BN + wave * 16;
  // this way's groups; every way passes the same number of barriers
  const int gs0 = split * a.gps, gs1 = min(G, gs0 + a.gps), per = (gs1 - gs0 + KW - 1) / KW;
  const int g0 = gs0 + way * per, g1 = min(gs1, g0 + per);
  // range-checked: rows past M or N read as zeros (or, in a matrix that almost fills 4 GB, where their 32-bit
  // offset wraps, as its first rows: the epilogue drops them either way)
  const auto xr = buf_rsrc(a.x, (uint32_t)a.m * (uint32_t)a.k * 2u);
  const auto wr = buf_rsrc(a.q, (uint32_t)a.n * (uint32_t)(a.k >> 1));
  const auto sr = buf_rsrc(a.sz, (uint32_t)a.n * (uint32_t)G * 4u);
  // X: thread -> rows (tid >> 4) + RP i, 16-byte unit tid & 15 of the group
  const uint32_t xoff = ((uint32_t)(m0 + (tid >> 4)) * (uint32_t)a.k + (uint32_t)(tid & 15) * 8u) * 2u;
  const uint32_t xstep = (uint32_t)a.k * (2u * RP);
  const uint32_t woff = TILED ? (uint32_t)(n0 >> 4) * (uint32_t)G * 1024u + (uint32_t)lane * 16u
                              : (uint32_t)(n0 + r) * (uint32_t)(a.k >> 1) + (uint32_t)c * 16u;
  const uint32_t soff = (uint32_t)(n0 + r) * (uint32_t)G * 4u;
  // requested ahead: the weights of WD groups, X of XD (past the way's last group: no memory access)
  uint4 xv[XD][XI], wv[WD];
  uint32_t sv[WD];
  auto load_w = [&](int g, uint4& w, uint32_t& s) {
    w = buf_ld128(wr, g < g1 ? woff + (uint32_t)g * (TILED ? 1024u : 64u) : 0xFFFFFFF0u);
    s = buf_ld32(sr, g < g1 ? soff + (uint32_t)g * 4u : 0xFFFFFFF0u);
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
  fl_f32x4 acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = fl_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
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
    const uint4 wc = wv[s % WD];
    const uint32_t sc = sv[s % WD];
    lds_barrier();
    load_w(g + WD, wv[s % WD], sv[s % WD]);
    load_x(g + XD, xv[s % XD]);
    if (KW > 1 && g >= g1) return;  // fewer groups than the other ways: its barriers only
    const unsigned char* xrow = xs[buf] + r * 256;
    auto mma = [&](int slot, const uint4 w) {
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const uint4 xf = *reinterpret_cast<const uint4*>(xrow + i * 4096 + ((slot ^ r) * 16));
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(fl_bf16x8, w),
                                                         __builtin_bit_cast(fl_bf16x8, xf), acc[i], 0, 0, 0);
      }
    };
    if constexpr (TILED) {
      // unit_dq_t's two exact steps, tiles 2tp, 2tp + 1 together
      const fl_s16x4 ai = mx_s4(0x3F803F80u & mx.mlo, 0x3F803F80u & mx.mhi);
      const uint32_t sb = sc & 0xFFFFu, sp = sb | (sb << 16);
      const fl_s16x4 bs = mx_s4(sp & mx.mlo, sp & mx.mhi);
      const float c1v = -136.0f * bf2f(sb), zv = bf2f(sc >> 16);
      const fl_f32x4 c1 = {c1v, c1v, c1v, c1v}, c2 = {zv, zv, zv, zv};
      const uint32_t v[4] = {wc.x, wc.y, wc.z, wc.w};
#pragma unroll
      for (int tp = 0; tp < 4; ++tp) {
        fl_f32x4 d[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int t = 2 * tp + e;
          const uint32_t lo = v[t >> 2] >> (4 * (t & 3)), hi = v[2 + (t >> 2)] >> (4 * (t & 3));
          d[e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(mx_s4((lo & mx.mask) | mx.magic, (hi & mx.mask) | mx.magic),
                                                        bs, c1, 0, 0, 0);
        }
        uint32_t p[2][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          p[e][0] = pack_bf16x2(d[e][0], d[e][1]);
          p[e][1] = pack_bf16x2(d[e][2], d[e][3]);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) d[e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ai, mx_s4(p[e][0], p[e][1]), c2, 0, 0, 0);
        mma(4 * tp + c, make_uint4(pack_bf16x2(d[0][0], d[0][1]), pack_bf16x2(d[0][2], d[0][3]),
                                   pack_bf16x2(d[1][0], d[1][1]), pack_bf16x2(d[1][2], d[1][3])));
      }
    } else {
      uint32_t d[4][4];
      dq32(wc, dq_const(sc), d);
#pragma unroll
      for (int e = 0; e < 4; ++e) mma(4 * c + e, make_uint4(d[0][e], d[1][e], d[2][e], d[3][e]));
    }
    if (g + 1 < g1) store(buf ^ 1, xv[(s + 1) % XD]);
  };
  for (int g = g0; g < g0 + per; g += 2) {  // by two, so that every buffer's index is fixed
    group(std::integral_constant<int, 0>{}, g);
    if (g + 1 < g0 + per) group(std::integral_constant<int, 1>{}, g + 1);
  }
  if constexpr (KW > 1) {  // the ways' sums, added in way order
    lds_barrier();
    fl_f32x4* red = reinterpret_cast<fl_f32x4*>(smem);
    if (way > 0) {
#pragma unroll
      for (int i = 0; i < MB; ++i) red[((way - 1) * MB + i) * (NW * 64) + tid] = acc[i];
    }
    lds_barrier();
    if (way > 0) return;
#pragma unroll
    for (int k = 0; k < KW - 1; ++k)
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[i] += red[(k * MB + i) * (NW * 64) + tid];
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) epi(n0 + 4 * c, m0 + 16 * i + r, acc[i], split);
}

typedef float fl_f32x16 __attribute__((ext_vector_type(16)));

// The same product for calls of many tiles: BN = 32 NW weight rows x BM = 128 activation rows per
// workgroup, on 32x32x16 MFMAs. A wave dequantises the operand of the next MFMA step (32 rows x 16 k)
// between the MFMAs of the current one, and reads its X fragments a step ahead, in that order
// (sched_barrier): beside 32x32 MFMAs the vector ALUs keep 0.9 of their rate (0.6 beside 16x16 ones), and a
// step's own VALU work then hides under its MFMAs. Both layouts run the 4x4x4 MFMA form of the dequantisation
// (unit_dq_t's steps; v_dot2 would take matrix-pipe time): a lane needs one column of four rows per step. The
// tiled layout holds that; from the row layout a lane loads the word it needs of each of its four rows
// (4-byte loads) and pairs their halves, and takes columns 8 apart in a step, which X in LDS follows.
// 1024 x 16384 x 2560: tiled 101 us, row 108 (k_gemm_rows with 128 x 128 tiles: 115, 128); 512: 53, 56 (57, 67).
// 2048: row 210, 0.82 PFLOP/s, the matrix pipes busy for 0.48 of the cycles.
// What is left (timing builds of the tiled form at 1024, 118 us there): the MFMAs alone 63 us, which is 1.5
// PFLOP/s, the rate that this card holds on any product; without the dequantisation 82; without storing X to LDS 99.
template <bool TILED, int NW, class Epi>
__global__ __launch_bounds__(64 * NW, 2) void k_gemm_big(GemmArgs a, Epi epi) {
  constexpr int TB = 4;  // 32-row tiles of X
  constexpr int BN = 32 * NW, BM = 32 * TB, RP = 4 * NW, XI = BM / RP;
  __shared__ __align__(16) unsigned char xs[2][BM * 256];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, c = lane >> 4, r32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int u, mb;
  if (!gemm_tile(a, u, mb)) return;
  const int split = u % a.splits, G = a.k >> 7;
  const int m0 = mb * BM, n0 = (u / a.splits) * BN + wave * 32;
  const int g0 = split * a.gps, g1 = min(G, g0 + a.gps);
  const auto xr = buf_rsrc(a.x, (uint32_t)a.m * (uint32_t)a.k * 2u);
  const auto wr = buf_rsrc(a.q, (uint32_t)a.n * (uint32_t)(a.k >> 1));
  const auto sr = buf_rsrc(a.sz, (uint32_t)a.n * (uint32_t)G * 4u);
  const uint32_t xoff = ((uint32_t)(m0 + (tid >> 4)) * (uint32_t)a.k + (uint32_t)(tid & 15) * 8u) * 2u;
  const uint32_t xstep = (uint32_t)a.k * (2u * RP);
  const uint32_t kb = (uint32_t)(a.k >> 1);  // bytes of a weight row
  const uint32_t woff = TILED ? (uint32_t)((n0 >> 4) + (c & 1)) * (uint32_t)G * 1024u + (uint32_t)((c & 2) * 16 + r) * 16u
                              : (uint32_t)(n0 + 16 * (c & 1) + 4 * ((lane >> 2) & 3)) * kb + (uint32_t)(h * 8 + (lane & 3)) * 4u;
  const uint32_t soff = (uint32_t)(n0 + r32) * (uint32_t)G * 4u;
  uint4 xv[XI], wv[2];
  uint32_t sv;
  auto load_w = [&](int g) {
    const bool in = g < g1;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      if constexpr (TILED) {
        wv[l] = buf_ld128(wr, in ? woff + (uint32_t)l * 256u + (uint32_t)g * 1024u : 0xFFFFFFF0u);
      } else {
        uint32_t t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          t[e] = buf_ld32(wr, in ? woff + (uint32_t)e * kb + (uint32_t)l * 16u + (uint32_t)g * 64u : 0xFFFFFFF0u);
        wv[l] = make_uint4(t[0], t[1], t[2], t[3]);
      }
    }
    sv = buf_ld32(sr, in ? soff + (uint32_t)g * 4u : 0xFFFFFFF0u);
  };
  auto load_x = [&](int g) {
    const bool in = g < g1;
#pragma unroll
    for (int i = 0; i < XI; ++i) xv[i] = buf_ld128(xr, in ? xoff + (uint32_t)i * xstep + (uint32_t)g * 256u : 0xFFFFFFF0u);
  };
  const int st = tid >> 4, un = tid & 15;
  auto store_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      unsigned char* row = xs[buf] + (st + i * RP) * 256;
      const int sw = (st + i * RP) & 15;
      if constexpr (TILED) {
        const int s0 = (un & 12) + 2 * (un & 1), half = (un >> 1) & 1;
        *reinterpret_cast<uint2*>(row + ((s0 ^ sw) * 16) + half * 8) = make_uint2(xv[i].x, xv[i].y);
        *reinterpret_cast<uint2*>(row + (((s0 + 1) ^ sw) * 16) + half * 8) = make_uint2(xv[i].z, xv[i].w);
      } else {
        const uint32_t v4[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
#pragma unroll
        for (int p = 0; p < 4; ++p) *reinterpret_cast<uint32_t*>(row + ((((un & 12) + p) ^ sw) * 16) + (un & 3) * 4) = v4[p];
      }
    }
  };
  const MxLane mx = mx_lane();
  const fl_s16x4 ai = mx_s4(0x3F803F80u & mx.mlo, 0x3F803F80u & mx.mhi);
  uint32_t v[2][4];
  fl_s16x4 bs;
  fl_f32x4 c1, c2;
  auto take = [&]() {  // the group's words and constants from the prefetch registers
#pragma unroll
    for (int l = 0; l < 2; ++l) {
      const uint4 w = wv[l];
      if constexpr (TILED) {
        v[l][0] = w.x, v[l][1] = w.y, v[l][2] = w.z, v[l][3] = w.w;
      } else {
        v[l][0] = __builtin_amdgcn_perm(w.y, w.x, 0x05040100u);
        v[l][1] = __builtin_amdgcn_perm(w.y, w.x, 0x07060302u);
        v[l][2] = __builtin_amdgcn_perm(w.w, w.z, 0x05040100u);
        v[l][3] = __builtin_amdgcn_perm(w.w, w.z, 0x07060302u);
      }
    }
    const uint32_t sb = sv & 0xFFFFu, sp = sb | (sb << 16);
    bs = mx_s4(sp & mx.mlo, sp & mx.mhi);
    const float c1v = -136.0f * bf2f(sb), zv = bf2f(sv >> 16);
    c1 = fl_f32x4{c1v, c1v, c1v, c1v};
    c2 = fl_f32x4{zv, zv, zv, zv};
  };
  fl_f32x4 d[2];
  uint32_t p[2][2];
  auto dq1 = [&](int l, int tp) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int t = TILED ? 2 * tp + e : tp + 4 * e;
      const uint32_t lo = v[l][t >> 2] >> (4 * (t & 3)), hi = v[l][2 + (t >> 2)] >> (4 * (t & 3));
      d[e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(mx_s4((lo & mx.mask) | mx.magic, (hi & mx.mask) | mx.magic), bs, c1, 0, 0, 0);
    }
  };
  auto dq2 = [&]() {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      p[e][0] = pack_bf16x2(d[e][0], d[e][1]);
      p[e][1] = pack_bf16x2(d[e][2], d[e][3]);
    }
  };
  auto dq3 = [&]() {
#pragma unroll
    for (int e = 0; e < 2; ++e) d[e] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ai, mx_s4(p[e][0], p[e][1]), c2, 0, 0, 0);
  };
  auto dq4 = [&]() {
    return TILED ? make_uint4(pack_bf16x2(d[0][0], d[0][1]), pack_bf16x2(d[0][2], d[0][3]), pack_bf16x2(d[1][0], d[1][1]), pack_bf16x2(d[1][2], d[1][3]))
                 : make_uint4(pack_bf16x2(d[0][0], d[1][0]), pack_bf16x2(d[0][1], d[1][1]), pack_bf16x2(d[0][2], d[1][2]), pack_bf16x2(d[0][3], d[1][3]));
  };
  fl_f32x16 acc[TB];
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
  const unsigned char* xb = xs[0] + r32 * 256;
  auto rd = [&](int buf, int s, int i) {  // X fragment of step s = 4l + tp, token tile i
    const int l = s >> 2, tp = s & 3, slot = TILED ? 4 * tp + 2 * h + l : 4 * (2 * h + l) + tp;
    return *reinterpret_cast<const uint4*>(xb + buf * (BM * 256) + i * 8192 + ((slot ^ r) * 16));
  };
  uint4 wq, xf[TB];
  load_w(g0);
  load_x(g0);
  store_x(0);
  take();
  load_w(g0 + 1);
  dq1(0, 0); dq2(); dq3(); wq = dq4();
  lds_barrier();
#pragma unroll
  for (int i = 0; i < TB; ++i) xf[i] = rd(0, 0, i);
  for (int g = g0; g < g1; ++g) {
    const int buf = (g - g0) & 1;
    load_x(g + 1);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (s == 6) store_x(buf ^ 1);
      if (s == 7) {
        take();          // the next group's words
        load_w(g + 2);
        lds_barrier();   // its X is in LDS; every wave has read this group's
      }
      uint4 xn[TB], wn;
#pragma unroll
      for (int i = 0; i < TB; ++i) {
        __builtin_amdgcn_sched_barrier(0);
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fl_bf16x8, wq), __builtin_bit_cast(fl_bf16x8, xf[i]), acc[i], 0, 0, 0);
        xn[i] = s < 7 ? rd(buf, s + 1, i) : rd(buf ^ 1, 0, i);
        if (i == 0) dq1(s < 7 ? (s + 1) >> 2 : 0, (s + 1) & 3);
        if (i == 1) dq2();
        if (i == 2) dq3();
        if (i == 3) wn = dq4();
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TB; ++i) xf[i] = xn[i];
      wq = wn;
    }
  }
#pragma unroll
  for (int i = 0; i < TB; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      epi(n0 + 8 * e + 4 * h, m0 + 32 * i + r32, fl_f32x4{acc[i][4 * e], acc[i][4 * e + 1], acc[i][4 * e + 2], acc[i][4 * e + 3]}, split);
}
