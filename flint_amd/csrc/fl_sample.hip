// Temperature / top-k sampling of logit rows on the GPU (reference engine/generate.py:36-55).
//
// Each row is split over up to SP_C chunks, one workgroup each, in one plain launch; two per-row
// barriers (an arrival counter in the row's scratch, bounded waits) separate the steps that need
// the whole row. The reference's steps with its bf16 rounding
// points: x = bf16(l / max(T, 1e-5)); the top-k pivot is the k-th largest x, found by a two-pass
// radix select over the 16-bit ordered keys of the bf16 values (each chunk's 256-bin histogram
// of the high byte, summed over the row in a fixed order, then the low byte within the selected
// bin); x < pivot drops out; p = bf16(exp(x - max) / sum), the sum of the chunks' partial sums in a
// fixed tree; q = bf16(-log(u)) with u from Philox4x32-10 keyed by the caller's seed, or q
// given; the sample is the first index of the largest bf16(p / q), which is
// multinomial_sample_one_no_sync's argmax(probs / exponential noise): 64-bit atomicMax of
// (ratio, ~index) per row, read out by the row's last chunk to finish.
#include <algorithm>
#include <mutex>
#include <stdlib.h>
#include "fl_common.h"

namespace {

constexpr int SAMPLE_MAXV = 65536;            // vocab limit

// One row is a chain of latencies (launch, logits, two row barriers with a read of every chunk's
// counts behind each, the argmax), 16 rows read 32 KB of counts per chunk and pass. Chunks of 512
// threads: us per call, top 200 of 49152, 1 row and 16 rows: 64 chunks of 256 threads 15.5 / 25.2,
// 32 of 512 14.6 / 18.3, 16 of 1024 16.5 / 17.1. With the reductions and the bin scan on DPP instead of
// LDS exchanges 13.8 / 17.5 (16.8 / 56.0 with 64 chunks, three barriers and an L2 write-back per chunk).
constexpr int SP_NT = 512;                     // threads per chunk workgroup
constexpr int SP_C = 32;                       // chunks per row (at most)
constexpr int SP_PT = 4;                       // values per thread: chunk <= 2048, vocab <= 65536
constexpr int SP_NWAVE = SP_NT / FL_WAVE;

// per-row scratch of the cooperative sampler (device memory owned by the library)
struct SampleWs {
  int hist[SP_C][2][256];                      // per chunk: high-byte, low-byte key histograms
  float mx[SP_C], ps[SP_C];                    // per chunk: max x, partial sum of exp(x - max)
  unsigned long long best;                     // (ratio bits, ~index), atomicMax
  unsigned int arrived;                        // chunks done (the last one reads best out)
  unsigned int bar;                            // barrier arrivals of this launch (reset by the last chunk)
  unsigned int fail;                           // a chunk's barrier wait timed out (reset by the last chunk)
};

constexpr unsigned long long SAMPLE_WAIT_TICKS = 200000000ull;  // 2 s of the 100 MHz realtime clock

// scratch words written before a row barrier and read after it by other workgroups (possibly on
// other XCDs): device-coherent accesses
__device__ __forceinline__ void st_ws(unsigned* a, unsigned v) {
  __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_ws(float* a, unsigned v) { st_ws(reinterpret_cast<unsigned*>(a), v); }
__device__ __forceinline__ unsigned ld_ws(unsigned* a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Barrier of the C chunk workgroups of one row: every thread's scratch stores are acknowledged
// (s_waitcnt 0) before the workgroup's arrival is counted, and the workgroup leaves once the
// row's count reaches `target` (C per barrier so far). The launch is a plain one: its grid (at
// most 16 rows x 32 chunks of 512 threads) is checked on the host to fit the device at once, so
// every chunk is resident on an idle device; should one not be (other work holding its CU), the
// wait gives up after 2 s and the row's token is reported as -1 instead of hanging.
// Work that needs nothing of the other chunks stands between the two halves.
__device__ __forceinline__ void row_arrive(SampleWs* ws) {
  wait_mem();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_fetch_add(&ws->bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void row_wait(SampleWs* ws, unsigned target, bool* timed_out) {
  if (threadIdx.x == 0) {
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    while (ld_ws(&ws->bar) < target) {
      __builtin_amdgcn_s_sleep(1);
      if (__builtin_amdgcn_s_memrealtime() - t0 > SAMPLE_WAIT_TICKS) {
        *timed_out = true;
        break;
      }
    }
  }
  __syncthreads();
}

__device__ __forceinline__ float bf_of_key(uint32_t key) {  // bf_key's inverse
  return __uint_as_float(((key & 0x8000u) ? key ^ 0x8000u : ~key & 0xFFFFu) << 16);
}

// the largest 64-bit word of a wave, in every lane (the exchanges of wave_max on both halves)
template <typename F>
__device__ __forceinline__ unsigned long long umax_step(unsigned long long v, F lane) {
  const uint32_t hi = __float_as_uint(lane(__uint_as_float((uint32_t)(v >> 32))));
  const uint32_t lo = __float_as_uint(lane(__uint_as_float((uint32_t)v)));
  const unsigned long long w = ((unsigned long long)hi << 32) | lo;
  return w > v ? w : v;
}
__device__ __forceinline__ unsigned long long wave_umax(unsigned long long v) {
  v = umax_step(v, lane_xor1);
  v = umax_step(v, lane_xor2);
  v = umax_step(v, lane_half_mirror);
  v = umax_step(v, lane_mirror);
  v = umax_step(v, lane_xor16);
  return umax_step(v, lane_xor32);
}

__device__ __forceinline__ float wg_max(float v, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = red[0];
  for (int w = 1; w < SP_NWAVE; ++w) v = fmaxf(v, red[w]);
  return v;
}
__device__ __forceinline__ float wg_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = 0.0f;
  for (int w = 0; w < SP_NWAVE; ++w) v += red[w];
  return v;
}
__device__ __forceinline__ unsigned long long wg_umax(unsigned long long v, unsigned long long* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = wave_umax(v);
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = red[0];
  for (int w = 1; w < SP_NWAVE; ++w) v = red[w] > v ? red[w] : v;
  return v;
}

__global__ __launch_bounds__(SP_NT) void k_sample(const float* __restrict__ logits, int V, int C, int row0,
                                                  float tdiv, int top_k, uint32_t seed_lo,
                                                  uint32_t seed_hi, uint32_t off_lo, uint32_t off_hi,
                                                  const float* __restrict__ noise,
                                                  int32_t* __restrict__ tokens_out,
                                                  float* __restrict__ probs_out, SampleWs* __restrict__ wsa) {
  __shared__ int hist[256];
  __shared__ __align__(16) int part[SP_NWAVE][256];
  __shared__ int sel[2];
  __shared__ float red[SP_NWAVE];
  __shared__ unsigned long long ured[SP_NWAVE];
  __shared__ bool last, timed_out;
  const int tid = threadIdx.x, row = blockIdx.x / C, c = blockIdx.x % C;
  const int CH = (V + C - 1) / C, j0 = c * CH, j1 = min(V, j0 + CH);
  SampleWs* ws = wsa + row;
  unsigned nsync = 0;  // row barriers passed
  if (tid == 0) timed_out = false;
  // the row's argmax word and arrival count start at zero: cleared here, before the first row
  // barrier, which orders it before every chunk's use after the last one. The barrier counter
  // itself is zero at launch: the last chunk of the previous call on this scratch reset it.
  if (c == 0 && tid == 0) {
    __hip_atomic_store(&ws->best, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ws->arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const float* lg = logits + (size_t)row * V;
  float x[SP_PT], y[SP_PT], q[SP_PT];
  // x = bf16(bf16(logit) / max(T, 1e-5))  (generate.py:42); max over the chunk
  float mx = -INFINITY;
#pragma unroll
  for (int e = 0; e < SP_PT; ++e) {
    const int j = j0 + tid + e * SP_NT;
    x[e] = j < j1 ? rbf(rbf(lg[j]) / tdiv) : -INFINITY;
    mx = fmaxf(mx, x[e]);
  }
  mx = wg_max(mx, red);
  if (tid == 0) st_ws(&ws->mx[c], __float_as_uint(mx));
  // this chunk's counts over the 256 bins of a key byte, published; the row's counts, into hist
  auto publish = [&](int pass, uint32_t top) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < SP_PT; ++e) {
      const uint32_t key = bf_key(x[e]);
      const bool in = (j0 + tid + e * SP_NT < j1) & (pass == 0 || (key >> 8) == top);
      if (in) atomicAdd(&hist[pass == 0 ? (key >> 8) : (key & 0xFFu)], 1);
    }
    __syncthreads();
    if (tid < 256) st_ws(reinterpret_cast<unsigned*>(&ws->hist[c][pass][tid]), (unsigned)hist[tid]);
  };
  auto gather = [&](int pass) {
    // a wave's lanes take 4 bins each of every SP_NWAVE-th chunk (16-byte coherent loads, all issued
    // before any is used); the waves' sums meet in LDS
    const auto hr = buf_rsrc(&ws->hist[0][0][0], (uint32_t)sizeof(ws->hist));
    const int wave = tid >> 6;
    uint4 hv[SP_C / SP_NWAVE];
#pragma unroll
    for (int i = 0; i < SP_C / SP_NWAVE; ++i) {
      const int cc = wave + SP_NWAVE * i;
      hv[i] = buf_ld128_coh(hr, cc < C ? (uint32_t)(((cc * 2 + pass) * 256 + 4 * (tid & 63)) * 4) : 0xFFFFFFF0u);
    }
    uint4 acc = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int i = 0; i < SP_C / SP_NWAVE; ++i) {
      acc.x += hv[i].x;
      acc.y += hv[i].y;
      acc.z += hv[i].z;
      acc.w += hv[i].w;
    }
    *reinterpret_cast<uint4*>(&part[wave][4 * (tid & 63)]) = acc;
    __syncthreads();
    if (tid < 256) {
      int n = 0;
#pragma unroll
      for (int w = 0; w < SP_NWAVE; ++w) n += part[w][tid];
      hist[tid] = n;
    }
    __syncthreads();
  };
  // the row's max: chunk cc's value is loaded by thread cc (one round trip), then reduced
  auto row_max = [&] {
    const float v = tid < C ? __uint_as_float(ld_ws(reinterpret_cast<unsigned*>(&ws->mx[tid]))) : -INFINITY;
    return wg_max(v, red);
  };
  // the noise of the values that may be kept, drawn while the other chunks arrive
  auto draw_noise = [&] {
#pragma unroll
    for (int e = 0; e < SP_PT; ++e) {
      const int j = j0 + tid + e * SP_NT;
      q[e] = 1.0f;
      if (y[e] == 0.0f || j >= j1) continue;  // p is 0: never beats the kept maximum's ratio
      if (noise) {
        q[e] = rbf(noise[(size_t)row * V + j]);
      } else {
        const uint32_t r = philox_x0((uint32_t)j, (uint32_t)(row0 + row), off_lo, off_hi, seed_lo, seed_hi);
        const double u = ((double)(r >> 8) + 0.5) * (1.0 / 16777216.0);
        q[e] = rbf((float)(-log(u)));
      }
    }
  };
  // The sum of exp(x - max) over the kept x. With a top-k it needs no row barrier of its own: what
  // lies above the pivot's high byte is known after the first count, so its partial sums go out with
  // the second one, and inside that byte equal keys are equal values, so their counts give the sum
  // (top 200 of 49152: 16.8 us with the third barrier and the noise after it, 15.5 without).
  float s;
  if (top_k > 0 && top_k < V) {
    // top-k pivot (generate.py:44-47): keys >= the k-th largest key stay
    publish(0, 0);
    row_arrive(ws);
    row_wait(ws, (unsigned)C * ++nsync, &timed_out);
    const float gmx = row_max();
    gather(0);
    int above = 0;
    const uint32_t top = (uint32_t)select_bin(hist, top_k, &above, sel);
    const int k = top_k - above;
    s = 0.0f;
#pragma unroll
    for (int e = 0; e < SP_PT; ++e) {
      const uint32_t hi = bf_key(x[e]) >> 8;
      y[e] = hi < top || x[e] == -INFINITY ? 0.0f : expf(x[e] - gmx);
      s += hi > top ? y[e] : 0.0f;
    }
    s = wg_sum(s, red);
    if (tid == 0) st_ws(&ws->ps[c], __float_as_uint(s));
    publish(1, top);
    row_arrive(ws);
    draw_noise();
    row_wait(ws, (unsigned)C * ++nsync, &timed_out);
    s = tid < C ? __uint_as_float(ld_ws(reinterpret_cast<unsigned*>(&ws->ps[tid]))) : 0.0f;
    gather(1);
    const uint32_t pivot = (top << 8) | (uint32_t)select_bin(hist, k, &above, sel);
    if (tid < 256 && tid >= (int)(pivot & 0xFFu) && hist[tid] != 0) {
      const float v = bf_of_key((top << 8) | (uint32_t)tid);
      s += v == -INFINITY ? 0.0f : (float)hist[tid] * expf(v - gmx);
    }
#pragma unroll
    for (int e = 0; e < SP_PT; ++e) y[e] = bf_key(x[e]) < pivot ? 0.0f : y[e];
  } else {
    row_arrive(ws);
    row_wait(ws, (unsigned)C * ++nsync, &timed_out);
    const float gmx = row_max();
    s = 0.0f;
#pragma unroll
    for (int e = 0; e < SP_PT; ++e) {
      y[e] = x[e] == -INFINITY ? 0.0f : expf(x[e] - gmx);
      s += y[e];
    }
    s = wg_sum(s, red);
    if (tid == 0) st_ws(&ws->ps[c], __float_as_uint(s));
    row_arrive(ws);
    draw_noise();
    row_wait(ws, (unsigned)C * ++nsync, &timed_out);
    s = tid < C ? __uint_as_float(ld_ws(reinterpret_cast<unsigned*>(&ws->ps[tid]))) : 0.0f;
  }
  s = wg_sum(s, red);  // a fixed reduction tree: the same sum in every chunk
  // p = bf16(exp(x - max) / sum); argmax(bf16(p / q)), the first index among equal ratios
  unsigned long long best = 0ull;
#pragma unroll
  for (int e = 0; e < SP_PT; ++e) {
    const int j = j0 + tid + e * SP_NT;
    if (j < j1) {
      const float p = rbf(y[e] / s);
      if (probs_out) probs_out[(size_t)row * V + j] = p;
      if (p != 0.0f) {  // ratio 0 never beats the kept maximum's (p > 0)
        const float ratio = rbf(p / q[e]);
        const unsigned long long key =
            ((unsigned long long)__float_as_uint(ratio) << 32) | (0xFFFFFFFFu - (uint32_t)j);
        best = key > best ? key : best;
      }
    }
  }
  best = wg_umax(best, ured);
  if (tid == 0) {
    if (best) __hip_atomic_fetch_max(&ws->best, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (timed_out) __hip_atomic_store(&ws->fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wait_mem();  // both are performed before the arrival is counted
    const unsigned prev = __hip_atomic_fetch_add(&ws->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = prev == (unsigned)(C - 1);
  }
  __syncthreads();
  // every chunk's atomicMax and failure mark precede its arrival, and every chunk has left its
  // last barrier: the last one reads the row out and resets the scratch for the next call
  if (last && tid == 0) {
    const unsigned long long b =
        __hip_atomic_exchange(&ws->best, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool failed = __hip_atomic_exchange(&ws->fail, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    tokens_out[row] = failed ? -1 : (int32_t)(0xFFFFFFFFu - (uint32_t)(b & 0xFFFFFFFFull));
    __hip_atomic_store(&ws->bar, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&ws->arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

}  // namespace

namespace {

// Rows per launch, and rows of each scratch block: 16 rows of up to SP_C chunks.
constexpr int SAMPLE_ROWS = 16;

// Scratch of fl_sample_noalloc: a fixed block per device for SAMPLE_ROWS rows (1.1 MB), part of
// the code object, so no call allocates. Host code must not pass `scratch` itself to a kernel (it
// names a host-side stand-in): its device address comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) SampleWs scratch[SAMPLE_ROWS];

std::mutex g_scratch_mu;
SampleWs* g_scratch_ptr[64] = {};

// Workgroups of k_sample the device holds at once (occupancy x CUs), per device, looked up on the
// first call: a launch's grid must fit, since its row barriers wait for every chunk of a row.
std::mutex g_fit_mu;
int g_fit[64] = {};
int sample_capacity(int dev) {
  std::lock_guard<std::mutex> lk(g_fit_mu);
  if (!g_fit[dev]) {
    int cu = 0, occ = 0;
    if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(k_sample), SP_NT, 0) !=
            hipSuccess)
      return 0;
    g_fit[dev] = cu * occ;
  }
  return g_fit[dev];
}
bool sample_coop() {
  const char* e = getenv("FLINT_AMD_COOPERATIVE");
  return e && atoi(e) != 0;
}

int sample_launch(const float* logits, int32_t rows, int32_t vocab, float temperature, int32_t top_k,
                  uint64_t seed, uint64_t offset, const float* noise, int32_t* tokens_out,
                  float* probs_out, SampleWs* wsp, void* stream) {
  const float tdiv = temperature > 1e-5f ? temperature : 1e-5f;
  const int C = std::min(SP_C, std::max(1, (vocab + SP_NT - 1) / SP_NT));  // chunks of <= SP_PT * SP_NT
  if ((vocab + C - 1) / C > SP_PT * SP_NT) return FL_E_ARG;
  int v = vocab, ci = C, tk = top_k;
  uint32_t slo = (uint32_t)seed, shi = (uint32_t)(seed >> 32), olo = (uint32_t)offset, ohi = (uint32_t)(offset >> 32);
  float td = tdiv;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return FL_E_HIP;
  const int cap = sample_capacity(dev);
  const bool coop = sample_coop();
  for (int r0 = 0; r0 < rows; r0 += SAMPLE_ROWS) {  // SAMPLE_ROWS rows per launch (the scratch's rows)
    const int n = std::min(SAMPLE_ROWS, rows - r0);
    const float* lg = logits + (size_t)r0 * vocab;
    const float* nz = noise ? noise + (size_t)r0 * vocab : nullptr;
    int32_t* to = tokens_out + r0;
    float* po = probs_out ? probs_out + (size_t)r0 * vocab : nullptr;
    int rb = r0;
    void* args[] = {(void*)&lg, &v, &ci, &rb, &td, &tk, &slo, &shi, &olo, &ohi, (void*)&nz, &to, &po, &wsp};
    if (n * C > cap) return FL_E_LAUNCH;  // the row barriers need every chunk resident at once
    // a plain launch (FLINT_AMD_COOPERATIVE=1: a cooperative one, which also guarantees residency)
    const hipStream_t hs = reinterpret_cast<hipStream_t>(stream);
    const hipError_t e =
        coop ? hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_sample), dim3(n * C), dim3(SP_NT), args, 0, hs)
             : hipLaunchKernel(reinterpret_cast<const void*>(k_sample), dim3(n * C), dim3(SP_NT), args, 0, hs);
    if (e != hipSuccess) return FL_E_LAUNCH;
  }
  return FL_OK;
}

bool sample_args_ok(const float* logits, int32_t rows, int32_t vocab, float temperature, int32_t top_k,
                    int32_t* tokens_out) {
  return logits && tokens_out && rows >= 1 && vocab >= 1 && vocab <= SAMPLE_MAXV && top_k >= 0 &&
         temperature == temperature;  // not NaN
}

}  // namespace

extern "C" {

int fl_sample(const float* logits, int32_t rows, int32_t vocab, float temperature, int32_t top_k,
              uint64_t seed, uint64_t offset, const float* noise, int32_t* tokens_out,
              float* probs_out, void* stream) {
  if (!sample_args_ok(logits, rows, vocab, temperature, top_k, tokens_out)) return FL_E_ARG;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return FL_E_HIP;
  // per-device scratch, allocated on the first call on that device and kept until the process
  // ends; calls on one device must be stream-ordered
  static SampleWs* ws[64] = {};
  if (!ws[dev]) {
    SampleWs* w = nullptr;
    if (hipMalloc(&w, sizeof(SampleWs) * SAMPLE_ROWS) != hipSuccess) return FL_E_HIP;
    if (hipMemset(w, 0, sizeof(SampleWs) * SAMPLE_ROWS) != hipSuccess) return FL_E_HIP;
    ws[dev] = w;
  }
  return sample_launch(logits, rows, vocab, temperature, top_k, seed, offset, noise, tokens_out,
                       probs_out, ws[dev], stream);
}

int fl_sample_noalloc(const float* logits, int32_t rows, int32_t vocab, float temperature,
                      int32_t top_k, uint64_t seed, uint64_t offset, const float* noise,
                      int32_t* tokens_out, float* probs_out, void* stream) {
  if (!sample_args_ok(logits, rows, vocab, temperature, top_k, tokens_out)) return FL_E_ARG;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return FL_E_HIP;
  SampleWs* wsp;
  {
    // the device address of this device's copy of `scratch`, looked up once (with the device
    // current: each device holds its own copy at its own address)
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
      void* p = nullptr;
      if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FL_E_HIP;
      g_scratch_ptr[dev] = reinterpret_cast<SampleWs*>(p);
    }
    wsp = g_scratch_ptr[dev];
  }
  return sample_launch(logits, rows, vocab, temperature, top_k, seed, offset, noise, tokens_out,
                       probs_out, wsp, stream);
}

}  // extern "C"
