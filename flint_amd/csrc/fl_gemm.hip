// int4 linear over more rows than one fl_gemm_int4 launch takes (a prompt through one layer).
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
__global__ __launch_bounds__(256) void k_sum_parts(const float* __restrict__ p, uint16_t* __restrict__ y, int m,
                                                   int n, int np, int splits, bool vec) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, total = (size_t)m * (np >> 2);
  if (i >= total) return;
  const int mm = (int)(i / (np >> 2)), nn = 4 * (int)(i % (np >> 2));
  fl_f32x4 v = *reinterpret_cast<const fl_f32x4*>(p + (size_t)mm * np + nn);
  for (int s = 1; s < splits; ++s) v += *reinterpret_cast<const fl_f32x4*>(p + ((size_t)s * m + mm) * np + nn);
  EpiBf16{y, m, n, vec}(nn, mm, v, 0);
}

// How a call of m rows runs. 128 x 128 tiles where they fill the chip (256 CUs, two workgroups each):
// 512 / 2048 rows x 16384 x 2560 took 60 / 235 us, 64 x 64 tiles 75 / 290. Else 64 x 64 tiles, K cut
// until there are about 768 workgroups of at least four 128-groups: 64 x 2560 x 8192 took 49 us
// uncut, 16 us in 4 parts and 13 in 8; 336 x 2576 x 2560 (246 tiles) 24 uncut, 17 in 2 and 15 in 4;
// 512 x 3584 x 2560 (448 tiles) 25 uncut and 23 in 2, less than the second launch that adds the
// parts costs (3-4 us).
struct Plan {
  bool big;
  int splits, gps;
};
Plan plan_rows(int m, int n, int k) {
  const int G = k / FL_GROUP;
  Plan p{true, 1, G};
  if ((int64_t)((m + 127) / 128) * ((n + 127) / 128) >= 256) return p;
  p.big = false;
  const int64_t tiles = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
  int s = (int)std::min<int64_t>(8, std::max<int64_t>(1, 768 / tiles));
  s = std::max(1, std::min(s, G / 4));
  p.gps = (G + s - 1) / s;
  p.splits = (G + p.gps - 1) / p.gps;
  return p;
}

// rows of one launch: 32-bit byte offsets over X (and the rows of a last tile past its end)
constexpr int ROWS_PER_LAUNCH = 8192;
bool rows_ok(int n, int k) {
  return k <= 65536 && ((int64_t)n + 128) * (k / 2) <= 0xFFFFFFFFll;
}

}  // namespace

extern "C" {

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
    const int t = p.big ? 128 : 64;
    uint16_t* yr = y + (size_t)r0 * n;
    const bool vec = n % 4 == 0 && (reinterpret_cast<uintptr_t>(yr) & 7) == 0;
    GemmArgs a{q, sz, x + (size_t)r0 * k, rows, n, k, (n + t - 1) / t, (rows + t - 1) / t, p.splits, p.gps};
    if (p.big) {
      hipLaunchKernelGGL((k_gemm_rows<false, 4, 2, 8, EpiBf16>), dim3(gemm_grid(a)), dim3(256), 0, s, a,
                         EpiBf16{yr, rows, n, vec});
    } else if (p.splits == 1) {
      hipLaunchKernelGGL((k_gemm_rows<false, 4, 1, 4, EpiBf16>), dim3(gemm_grid(a)), dim3(256), 0, s, a,
                         EpiBf16{yr, rows, n, vec});
    } else {
      hipLaunchKernelGGL((k_gemm_rows<false, 4, 1, 4, EpiPart>), dim3(gemm_grid(a)), dim3(256), 0, s, a,
                         EpiPart{ws, rows, np});
      const size_t quads = (size_t)rows * (np / 4);
      hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, ws, yr, rows, n, np,
                         p.splits, vec);
    }
  }
  return hipGetLastError() == hipSuccess ? FL_OK : FL_E_LAUNCH;
}

}  // extern "C"
