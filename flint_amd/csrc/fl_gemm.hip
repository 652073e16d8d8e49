// The int4 linear for more than one row: fl_gemm_int4 (up to 32 rows: speculative verify) and
// fl_gemm_rows_int4 (any number: a prompt through one layer).
#include "fl_gemm.h"
#include <algorithm>

namespace {

// bf16 output [M, N], any N; vec: every row of four values is 8-byte aligned
struct EpiBf16 {
  uint16_t* y;
  int m, n;
  bool vec;
  __device__ __forceinline__ void operator()(int nn, int mm, fl_f32x4 v, int) const {
    if (mm >= m || nn >= n) return;
    uint16_t* o = y + (size_t)mm * n + nn;
    if (vec) {
      *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nn + i < n) o[i] = (uint16_t)f2bf(v[i]);
    }
  }
};

// fp32 partial sums [splits, M, Np], Np = N rounded up to 4
struct EpiPart {
  float* p;
  int m, np;
  __device__ __forceinline__ void operator()(int nn, int mm, fl_f32x4 v, int split) const {
    if (mm < m && nn < np) *reinterpret_cast<fl_f32x4*>(p + ((size_t)split * m + mm) * np + nn) = v;
  }
};

// y = bf16(the partial sums, added in order); one thread per four columns
__global__ __launch_bounds__(256) void k_sum_parts(const float* __restrict__ p, EpiBf16 out, int np, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, total = (size_t)out.m * (np >> 2);
  if (i >= total) return;
  const int mm = (int)(i / (np >> 2)), nn = 4 * (int)(i % (np >> 2));
  fl_f32x4 v = *reinterpret_cast<const fl_f32x4*>(p + (size_t)mm * np + nn);
  for (int s = 1; s < splits; ++s) v += *reinterpret_cast<const fl_f32x4*>(p + ((size_t)s * out.m + mm) * np + nn);
  out(nn, mm, v, 0);
}

// How a call of m rows runs (us, weights from HBM).
// Large tiles, 128 rows x 256 weight rows (k_gemm_big, one workgroup per CU): from 224 of them on, but not where a
// second round would be half empty or more (257 to 383) at up to 12 groups, which the smaller tiles outrun, nor for one
// or two groups, which do not pay for its start-up. 512 x 16384 x 2560 (256) 56, in 64 x 64 tiles 89; 576 x 16384
// (320) x 640 35 and 31, x 1280 54 and 52, x 2560 92 and 97; 768 x 16384 (384) x 640 37 and 38; 448 x 12288 x 256 15 and 14.
// Else 64 x 64 tiles; a CU holds one workgroup of four ways, two of two (LDS), five of one (registers):
// - few tiles (up to 256; beyond 32 groups not 129 to 200, which leave CUs idle): four ways, two where a part has fewer
//   than 8 groups, and K cut while all parts' tiles still run at once. 333 x 2570 x 2560 (246 tiles) 16, with two ways
//   17, one 25, one in 2 parts, whose sums cost a launch, 20; 100 x 3584 x 2560 (112) 13 in 2 parts, 15 uncut;
// - more, beyond 32 groups: one way, parts of at least 12 groups for about 1536 workgroups. 200 x 2560 x 8192 (160) 34 in
//   4 parts, 38 with four ways; 333 x 2900 x 8192 (276) 52, in 2 parts 57, with two ways 66; 600 x 3584 x 8192
//   (560) 93 in 2, 100 uncut; 97 x 12260 x 4224 (384, 33 groups) 40 in 2, 43 in 4;
// - more, up to 32 groups: two ways, one beyond 512 tiles of at most 16 groups. 333 x 2900 x 2560 (276) 23, with one
//   26; 2048 x 2560 x 2560 (1280) 56 and 58; 389 x 11621 x 640 (1274) 24 and 22.
struct Plan {
  bool big;
  int ways, splits, gps;
};
Plan plan_rows(int m, int n, int k) {
  const int G = k / FL_GROUP;
  Plan p{true, 1, 1, G};
  const int64_t big = (int64_t)((m + 127) / 128) * ((n + 255) / 256);
  if (big >= 224 && G > 2 && (big <= 256 || big >= 384 || G > 12)) return p;
  p.big = false;
  const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
  const bool few = tiles <= 256 && (G <= 32 || tiles <= 128 || tiles > 200);
  const int64_t s = few ? 256 / tiles : G > 32 ? 1536 / tiles : 1;
  const int parts = (int)std::max<int64_t>(1, std::min<int64_t>({4, s, G / (few ? 4 : 12)}));
  p.gps = (G + parts - 1) / parts;
  p.splits = (G + p.gps - 1) / p.gps;
  if (few) p.ways = p.gps >= 8 ? 4 : 2;
  else if (G <= 32 && (tiles <= 512 || G > 16)) p.ways = 2;
  return p;
}

template <int NW, int KW, int MB, class Epi>
void launch(GemmArgs a, Epi epi, hipStream_t s) {
  a.tile(16 * NW, 16 * MB);
  hipLaunchKernelGGL((k_gemm_rows<false, NW, KW, MB, 1, 1, Epi>), dim3(gemm_grid(a)), dim3(64 * NW * KW), 0, s, a, epi);
}
template <class Epi>
void launch_small(int ways, const GemmArgs& a, Epi epi, hipStream_t s) {
  if (ways == 4) launch<4, 4, 4>(a, epi, s);
  else if (ways == 2) launch<4, 2, 4>(a, epi, s);
  else launch<4, 1, 4>(a, epi, s);
}

// The former kernel of 2 to 32 rows, kept for few K groups: one workgroup of four waves per 16 weight rows,
// the groups round-robin over the waves, X fragments straight from global memory (rows past M or N read as zeros),
// one barrier for the waves' sums, added in wave order. It starts up faster (3.5 us where k_gemm_rows takes 4.9: 8 x 2560
// x 512), but waits for each group's loads in turn and reads X once per 16 weight rows.
constexpr int kGemmWaves = 4;

__global__ __launch_bounds__(64 * kGemmWaves) void k_gemm(const uint32_t* __restrict__ q,
                                                          const uint32_t* __restrict__ sz,
                                                          const uint16_t* __restrict__ x,
                                                          uint16_t* __restrict__ y, int m, int n,
                                                          int k) {
  __shared__ float part[kGemmWaves][2][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, c = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int rows = min(16, n - n0);
  const int groups = k >> 7;
  const bool two = m > 16;  // a second 16-row block of activations (tokens 16..31)
  const auto wr = buf_rsrc(q + (size_t)n0 * (k >> 3), (uint32_t)rows * (uint32_t)(k >> 1));
  const auto sr = buf_rsrc(sz + (size_t)n0 * groups, (uint32_t)rows * (uint32_t)groups * 4u);
  const auto xr = buf_rsrc(x, (uint32_t)m * (uint32_t)k * 2u);
  const uint32_t woff = (uint32_t)r * (uint32_t)(k >> 1) + (uint32_t)c * 16u;   // bytes
  const uint32_t xoff = (uint32_t)r * (uint32_t)k * 2u + (uint32_t)c * 64u;     // bytes
  const uint32_t xoff2 = xoff + 16u * (uint32_t)k * 2u;
  fl_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, acc2 = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int u = wave; u < groups; u += kGemmWaves) {
    const uint4 w = buf_ld128(wr, woff + (uint32_t)u * 64u);
    const uint32_t s = buf_ld32(sr, ((uint32_t)r * (uint32_t)groups + (uint32_t)u) * 4u);
    uint4 xa[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) xa[e] = buf_ld128(xr, xoff + (uint32_t)u * 256u + (uint32_t)e * 16u);
    uint32_t d[4][4];
    dq32(w, dq_const(s), d);
    mfma_chunk(d, xa, acc);
    if (two) {
#pragma unroll
      for (int e = 0; e < 4; ++e) xa[e] = buf_ld128(xr, xoff2 + (uint32_t)u * 256u + (uint32_t)e * 16u);
      mfma_chunk(d, xa, acc2);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    part[wave][0][(c * 4 + i) * 16 + r] = acc[i];
    part[wave][1][(c * 4 + i) * 16 + r] = acc2[i];
  }
  __syncthreads();
  for (int t = threadIdx.x; t < (two ? 512 : 256); t += 64 * kGemmWaves) {
    const int row = t >> 4, col = t & 15;  // activation row (token), weight row in the tile
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kGemmWaves; ++w) v += part[w][t >> 8][t & 255];
    if (row < m && col < rows) y[(size_t)row * n + n0 + col] = (uint16_t)f2bf(v);
  }
}

// k_gemm against k_gemm_rows at m rows, t16 blocks of 16 weight rows and G groups (us, weights from HBM, k_gemm
// first): up to 16 rows 2 x 2560 x 1024 5.0 / 5.5, x 1280 5.7 / 5.6, x 1536 6.3 / 5.7; beyond 768 blocks, where
// k_gemm_rows has fewer ways, 2 x 16384 x 2048 11.2 / 11.5, x 2560 13.3 / 13.3, x 3072 15.1 / 14.6; with more rows
// earlier, by the products in all: 16 x 16384 x 768 7.2 / 7.7, x 1024 9.0 / 8.3. More than 16 rows read X twice per
// weight: 17 x 2560 x 768 5.0 / 5.1, x 1024 5.4 / 5.4; 32 x 8192 x 512 5.5 / 5.8, 32 x 12288 x 512 6.8 / 6.2; one or
// two groups always: 32 x 49152 x 128 8.3 / 11.2.
bool few_groups(int m, int t16, int G) {
  const int64_t work = (int64_t)m * t16 * G;
  return m <= 16 ? G <= (t16 <= 768 ? 10 : 20) && (G == 1 || work < 131072) : G <= 2 || (G <= 6 && work <= 65536);
}

EpiBf16 out_bf16(uint16_t* y, int m, int n) {
  return EpiBf16{y, m, n, n % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0};
}

// rows of one launch: 32-bit byte offsets over X and the rows of a last tile past its end; over the weights up to the
// matrix's own end (the rows of a 256-row tile past it may wrap, within the matrix, and are dropped)
constexpr int ROWS_PER_LAUNCH = 8192;
bool rows_ok(int n, int k) {
  return k <= 65536 && ((int64_t)n + 128) * (k / 2) <= 0xFFFFFFFFll;
}

}  // namespace

extern "C" {

int fl_gemm_int4(const uint32_t* q, const uint32_t* sz, const uint16_t* x, uint16_t* y, int32_t m, int32_t n,
                 int32_t k, void* stream) {
  if (!q || !sz || !x || !y || n <= 0 || k <= 0 || (k % FL_GROUP) != 0) return FL_E_ARG;
  if (m < 1 || m > FL_MAX_VERIFY) return FL_E_M;
  if ((int64_t)n * (k / 2) > 0xFFFFFFFFll || (int64_t)m * k * 2 > 0xFFFFFFFFll) return FL_E_ARG;
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const GemmArgs a{q, sz, x, m, n, k, 0, 0, 1, k / FL_GROUP, 0};
  const EpiBf16 epi = out_bf16(y, m, n);
  // k_gemm_rows, up to 16 rows: sixteen ways over 16 weight rows while one workgroup per CU holds them all (256
  // blocks of 16), eight over 32 up to two blocks per CU, then four: over 16 weight rows while that gives a CU
  // three blocks where 32 would give it four (8 rows x 11200 x 5120, 700 blocks, 22.6 us and 24.5), over 32 beyond
  // (12800, 800 blocks, 26.5 and 25.0; X is read half as often). 5 x 2560 x 8192 sixteen ways 11, eight 12; 12 x 6000 x
  // 5120 (375) sixteen 17, eight over 32 rows 12; 12 x 10477 x 3456 (655) sixteen 18, eight 14, four 12.
  // 17 to 32 rows hold twice the X in LDS, so eight ways at most: 32 x 2560 x 8192 15; 6000 x 5120 (375) eight over 16
  // weight rows 19, over 32 14; beyond 512 blocks four over 32: 12000 x 8192 (750) eight 37 to 41, four 33; 16384 x
  // 2560 eight over 16 rows 24, over 32 16, four 13.
  const int t16 = (n + 15) / 16;
  if (few_groups(m, t16, k / FL_GROUP)) {
    hipLaunchKernelGGL(k_gemm, dim3(t16), dim3(64 * kGemmWaves), 0, s, q, sz, x, y, m, n, k);
  } else if (m <= 16) {
    if (t16 <= 256) launch<1, 16, 1>(a, epi, s);
    else if (t16 <= 512) launch<2, 8, 1>(a, epi, s);
    else if (t16 <= 768) launch<1, 4, 1>(a, epi, s);
    else launch<2, 4, 1>(a, epi, s);
  } else {
    if (t16 <= 256) launch<1, 8, 2>(a, epi, s);
    else if (t16 <= 512) launch<2, 8, 2>(a, epi, s);
    else launch<2, 4, 2>(a, epi, s);
  }
  return hipGetLastError() == hipSuccess ? FL_OK : FL_E_LAUNCH;
}

int fl_gemm_rows_workspace(int32_t m, int32_t n, int32_t k, int64_t* bytes) {
  if (!bytes || m < 1 || n < 1 || k < 1 || k % FL_GROUP || !rows_ok(n, k)) return FL_E_ARG;
  int64_t most = 0;  // the full launches, then the rest
  for (int r : {std::min(m, ROWS_PER_LAUNCH), m % ROWS_PER_LAUNCH}) {
    if (!r) continue;
    const Plan p = plan_rows(r, n, k);
    if (p.splits > 1) most = std::max(most, (int64_t)p.splits * r * ((n + 3) / 4 * 4) * 4);
  }
  *bytes = most;
  return FL_OK;
}

int fl_gemm_rows_int4(const uint32_t* q, const uint32_t* sz, const uint16_t* x, uint16_t* y, float* ws, int32_t m,
                      int32_t n, int32_t k, void* stream) {
  if (!q || !sz || !x || !y) return FL_E_ARG;
  int64_t need = 0;
  if (fl_gemm_rows_workspace(m, n, k, &need) != FL_OK || (need > 0 && !ws)) return FL_E_ARG;
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int np = (n + 3) / 4 * 4;
  for (int r0 = 0; r0 < m; r0 += ROWS_PER_LAUNCH) {
    const int rows = std::min(ROWS_PER_LAUNCH, m - r0);
    const Plan p = plan_rows(rows, n, k);
    const EpiBf16 epi = out_bf16(y + (size_t)r0 * n, rows, n);
    const GemmArgs a{q, sz, x + (size_t)r0 * k, rows, n, k, 0, 0, p.splits, p.gps, 0};
    if (p.big) {
      GemmArgs b = a;
      b.tile(256, 128);
      hipLaunchKernelGGL((k_gemm_big<false, 8, EpiBf16>), dim3(gemm_grid(b)), dim3(512), 0, s, b, epi);
    } else if (p.splits == 1) {
      launch_small(p.ways, a, epi, s);
    } else {
      launch_small(p.ways, a, EpiPart{ws, rows, np}, s);
      const size_t quads = (size_t)rows * (np / 4);
      hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, ws, epi, np, p.splits);
    }
  }
  return hipGetLastError() == hipSuccess ? FL_OK : FL_E_LAUNCH;
}

}  // extern "C"
