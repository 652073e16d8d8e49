// A prompt through the model in passes of up to PF_TOKENS tokens: ordinary kernels per layer instead
// of k_verify's persistent launch of at most 32 tokens, which reads and dequantises every weight
// once per 32 tokens. Same operations and bf16 rounding points (reference engine/model.py:134-242,
// engine/generate.py:57-60 prefill): per layer
//   RMSNorm -> QKV GEMM (RoPE and KV append in its epilogue) -> attention -> O GEMM ->
//   residual + RMSNorm -> gate/up GEMM (SwiGLU in its epilogue) -> down GEMM -> residual + RMSNorm,
// the O and down GEMMs cut along K into fp32 part sums that the residual kernel adds in order. After
// the last pass the LM head and argmax of the last token.
// At 512 tokens of flint-3b a layer takes 152 us (of which the GEMMs: QKV 22, O 18, gate/up 51, down 36;
// attention 11, the two norms 14), against 1336 in sixteen k_verify launches; 40 tokens take 64 us a
// layer (launches and latency) against 120, and up to 16 they take the one k_verify launch (16: 46 us a
// layer against 62; 24: 71 against 62, at 12000 cached keys 118 against 85).
#include "fl_gemm.h"
#include "fl_state.h"
#include <algorithm>
#include <string.h>

namespace {

constexpr int PF_TOKENS = 1024;  // tokens of a pass at most: 512 per pass cost 13.6 us a token, 1024 10.9
constexpr int PF_NT = 256;
constexpr int PF_SPLITS = 4;      // K parts of the O and down GEMMs at most
constexpr int PF_KEY_PARTS = 16;  // key parts of the attention at most
constexpr int PF_NORM_MAX = 3;    // 4-value chunks per thread of a row (D <= 3072)
constexpr int PF_LM_GRID = 512;   // LM-head workgroups

// ---- GEMM epilogues -----------------------------------------------------------------------------
// v[0..3]: packed rows n..n+3 of one token, i.e. two NEOX / gate-up pairs

// RoPE at pos + m, q rows out, K / V rows into the cache (engine/model.py:257-269, :88-98)
struct EpiQkv {
  uint16_t *q, *kc, *vc;  // q [T][NH * 64]; kc / vc of this layer [NKV][S][64]
  const uint32_t* rope;   // [rope_len][32] (cos, sin) pairs
  int m, nh, nkv, S, pos;
  __device__ __forceinline__ void operator()(int n, int mm, fl_f32x4 v, int) const {
    if (mm >= m || n >= (nh + 2 * nkv) * 64) return;
    const int hh = n >> 6, j = (n & 63) >> 1;  // pairs j, j + 1 (j even) of head hh
    float a0 = rbf(v[0]), b0 = rbf(v[1]), a1 = rbf(v[2]), b1 = rbf(v[3]);
    if (hh < nh + nkv) {
      const uint2 cs = *reinterpret_cast<const uint2*>(rope + (size_t)(pos + mm) * 32 + j);
      const float c0 = bflo(cs.x), s0 = bfhi(cs.x), c1 = bflo(cs.y), s1 = bfhi(cs.y);
      const float ta0 = a0 * c0 - b0 * s0, tb0 = b0 * c0 + a0 * s0;
      const float ta1 = a1 * c1 - b1 * s1, tb1 = b1 * c1 + a1 * s1;
      a0 = ta0, b0 = tb0, a1 = ta1, b1 = tb1;
    }
    uint16_t* d = hh < nh ? q + ((size_t)mm * nh + hh) * 64
                  : hh < nh + nkv ? kc + ((size_t)(hh - nh) * S + pos + mm) * 64
                                  : vc + ((size_t)(hh - nh - nkv) * S + pos + mm) * 64;
    *reinterpret_cast<uint32_t*>(d + j) = pack_bf16x2(a0, a1);
    *reinterpret_cast<uint32_t*>(d + j + 32) = pack_bf16x2(b0, b1);
  }
};

// act = bf16(bf16(silu(g)) * u)  (engine/model.py:227-228)
struct EpiSwiglu {
  uint16_t* act;  // [T][F]
  int m, f;
  __device__ __forceinline__ void operator()(int n, int mm, fl_f32x4 v, int) const {
    if (mm >= m || n >= 2 * f) return;
    const float o0 = rbf(silu_f(rbf(v[0]))) * rbf(v[1]), o1 = rbf(silu_f(rbf(v[2]))) * rbf(v[3]);
    *reinterpret_cast<uint32_t*>(act + (size_t)mm * f + (n >> 1)) = pack_bf16x2(o0, o1);
  }
};

struct EpiSum {  // fp32 part sums [splits][T][D]
  float* p;
  int m, d;
  __device__ __forceinline__ void operator()(int n, int mm, fl_f32x4 v, int split) const {
    if (mm < m && n < d) *reinterpret_cast<fl_f32x4*>(p + ((size_t)split * m + mm) * d + n) = v;
  }
};

// ---- embedding / residual + RMSNorm ---------------------------------------------------------------
// One workgroup per token: h = bf16(embed[token] * emb_mult) (splits = 0), or
// h += bf16(bf16(sum of the parts) * resid_mult); then xn = bf16(bf16(h * rsqrt(mean(h^2) + eps)) * w).
__global__ __launch_bounds__(PF_NT) void k_pf_norm(const float* __restrict__ part, int splits, int T, int D,
                                                   const int32_t* __restrict__ tokens, const uint16_t* __restrict__ embed,
                                                   int V, float mult, const uint16_t* __restrict__ w, float eps,
                                                   uint16_t* __restrict__ h, uint16_t* __restrict__ xn, int32_t* err) {
  __shared__ float red[PF_NT / FL_WAVE];
  const int tid = threadIdx.x, m = blockIdx.x, nq = D >> 2;
  int tok = 0;
  if (splits == 0) {
    tok = tokens[m];
    if (tok < 0 || tok >= V) {
      if (tid == 0) __hip_atomic_store(err, (int32_t)FL_E_ARG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      tok = 0;
    }
  }
  uint16_t* hr = h + (size_t)m * D;
  const uint16_t* src = splits == 0 ? embed + (size_t)tok * D : hr;
  float x[PF_NORM_MAX][4];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < PF_NORM_MAX; ++i) {
    const int c = tid + i * PF_NT;
    if (c >= nq) continue;
    const uint2 e = reinterpret_cast<const uint2*>(src)[c];
    const float in[4] = {bflo(e.x), bfhi(e.x), bflo(e.y), bfhi(e.y)};
    if (splits == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k) x[i][k] = rbf(in[k] * mult);
    } else {
      fl_f32x4 s = reinterpret_cast<const fl_f32x4*>(part + (size_t)m * D)[c];
      for (int p = 1; p < splits; ++p) s += reinterpret_cast<const fl_f32x4*>(part + ((size_t)p * T + m) * D)[c];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[i][k] = rbf(in[k] + rbf(rbf(s[k]) * mult));
    }
    reinterpret_cast<uint2*>(hr)[c] = make_uint2(pack_bf16x2(x[i][0], x[i][1]), pack_bf16x2(x[i][2], x[i][3]));
#pragma unroll
    for (int k = 0; k < 4; ++k) ss += x[i][k] * x[i][k];
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  ss = red[0];
#pragma unroll
  for (int k = 1; k < PF_NT / FL_WAVE; ++k) ss += red[k];
  const float r = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
  for (int i = 0; i < PF_NORM_MAX; ++i) {
    const int c = tid + i * PF_NT;
    if (c >= nq) continue;
    const uint2 g = reinterpret_cast<const uint2*>(w)[c];
    reinterpret_cast<uint2*>(xn + (size_t)m * D)[c] =
        make_uint2(pack_bf16x2(rbf(x[i][0] * r) * bflo(g.x), rbf(x[i][1] * r) * bfhi(g.x)),
                   pack_bf16x2(rbf(x[i][2] * r) * bflo(g.y), rbf(x[i][3] * r) * bfhi(g.y)));
  }
}

// ---- attention --------------------------------------------------------------------------------------
// The rows of a KV group are its (token, query head) pairs, token-major: row t * rep + j. A workgroup
// takes 128 / W rows of a group over one part of the keys [0, pos + its last token], in rounds of 64 W keys
// staged in LDS (K rows; V transposed), double-buffered, so a group's K / V rows are read once per
// workgroup. Its four waves are W ways of 4 / W: a way's waves take 32 rows each over the way's 64 keys of
// every round, and the ways' (max, sum, o) meet in LDS at the end. Two ways by default: a row's keys are a
// serial chain, and 512 tokens of flint-3b are only 320 workgroups of 64 rows (one way, 160 of 128: 16.8
// us, two 11.5); one way, which stages each key for twice the rows, where 128-row workgroups fill the
// chip and the keys are many (1024 tokens behind 4000 / 12000 keys: 403 / 672 us a layer, 418 / 716
// with two ways; behind none 274 and 267).
// Per 64 keys S^T = K Q^T on 32x32x16 MFMAs (lane = row, registers = keys), an online fp32 softmax per
// lane, and O^T += V^T P^T with P split into three bf16 terms (hi + mid + lo, each product exact, as
// k_verify's attention): the keys of a 16-key step are taken in the order that the score
// registers already hold them, so P needs no exchange between lanes. Bound by the vector ALUs
// (about 350 instructions per 64 keys and wave, 1.7x the MFMAs' cycles).
constexpr int PA_WGS = 512;   // workgroups that cutting the keys into parts may reach
constexpr int PA_VLD = 68;    // V^T row pitch of a way (bf16): 34 words spread a wave's 8-byte reads over all banks
struct PaArgs {
  const uint16_t *q, *kc, *vc;  // q [T][NH * 64], kc / vc of this layer
  uint16_t* out;                // [T][NH * 64]
  float* part;                  // with key parts: o [parts][NKV][rows][64], then (m, l) [parts][NKV][rows][2]
  int T, pos, S, nh, nkv, rep;
  int blocks, parts, kpp;       // row blocks per group; key parts, keys per part (multiple of 128)
  float sc;                     // attn_scale * log2 e
};

template <int W>
__global__ __launch_bounds__(256, 2) void k_pf_attn(PaArgs a) {
  constexpr int PA_ROWS = 128 / W, PA_KEYS = 64 * W, WR = 4 / W;  // rows, keys per round; waves of a way
  __shared__ __align__(16) unsigned char ks[2][PA_KEYS * 128];
  __shared__ __align__(16) uint16_t vt[2][W * 64 * PA_VLD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 31, hf = lane >> 5;
  const int sub = wave % WR, way = wave / WR;
  const int g = blockIdx.x % a.nkv, rest = blockIdx.x / a.nkv;
  const int part = rest % a.parts, blk = a.blocks - 1 - rest / a.parts;  // the longest rows first
  const int R = a.T * a.rep, row0 = blk * PA_ROWS;
  const int tlast = min(a.T - 1, (row0 + PA_ROWS - 1) / a.rep);
  const int kb0 = part * a.kpp, kend = min(a.pos + tlast + 1, kb0 + a.kpp);  // keys of this workgroup
  const int row = row0 + sub * 32 + r, rowc = min(row, R - 1);
  const int t = rowc / a.rep, head = g * a.rep + rowc % a.rep;
  const int lim = min(a.pos + t, kend - 1);  // the last key this row sees here
  const int wfirst = min(a.pos + min(row0 + sub * 32, R - 1) / a.rep, kend - 1);  // ... the wave's first row
  const int wlast = a.pos + min(row0 + sub * 32 + 31, R - 1) / a.rep;             // ... and its last
  const size_t cb = (size_t)g * a.S * 64;
  const auto kr = buf_rsrc(a.kc + cb, (uint32_t)(a.pos + a.T) * 128u);  // keys past the end read as zeros
  const auto vr = buf_rsrc(a.vc + cb, (uint32_t)(a.pos + a.T) * 128u);
  uint4 qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    qf[s] = *reinterpret_cast<const uint4*>(a.q + ((size_t)t * a.nh + head) * 64 + s * 16 + hf * 8);
  uint4 kv[2 * W], vv[2 * W];
  const int c8 = tid & 7, kp = tid >> 3;  // 16-byte chunk; K rows kp + 32 i; V rows 2 kp, 2 kp + 1 of every way
  auto load = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) {
      kv[i] = buf_ld128(kr, (uint32_t)(kb + kp + 32 * i) * 128u + (uint32_t)c8 * 16u);
      vv[i] = buf_ld128(vr, (uint32_t)(kb + 64 * (i >> 1) + 2 * kp + (i & 1)) * 128u + (uint32_t)c8 * 16u);
    }
  };
  auto store = [&](int b) {
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) {
      const int key = kp + 32 * i;
      *reinterpret_cast<uint4*>(ks[b] + key * 128 + ((c8 ^ ((key >> 1) & 7)) * 16)) = kv[i];
    }
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const uint32_t x[4] = {vv[2 * w].x, vv[2 * w].y, vv[2 * w].z, vv[2 * w].w};
      const uint32_t y[4] = {vv[2 * w + 1].x, vv[2 * w + 1].y, vv[2 * w + 1].z, vv[2 * w + 1].w};
      uint16_t* v = &vt[b][w * 64 * PA_VLD];
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // the two keys of a dim side by side
        *reinterpret_cast<uint32_t*>(v + (c8 * 8 + 2 * e) * PA_VLD + 2 * kp) = __builtin_amdgcn_perm(y[e], x[e], 0x05040100u);
        *reinterpret_cast<uint32_t*>(v + (c8 * 8 + 2 * e + 1) * PA_VLD + 2 * kp) = __builtin_amdgcn_perm(y[e], x[e], 0x07060302u);
      }
    }
  };
  fl_f32x16 o[2];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
  float mrun = -INFINITY, lrun = 0.0f;
  if (kb0 < kend) {
    load(kb0);
    store(0);
  }
  for (int kr0 = kb0; kr0 < kend; kr0 += PA_KEYS) {
    const int b = ((kr0 - kb0) / PA_KEYS) & 1, kb = kr0 + 64 * way;  // this way's 64 keys
    const bool more = kr0 + PA_KEYS < kend;
    __syncthreads();
    if (more) load(kr0 + PA_KEYS);
    if (kb <= wlast && kb < kend) {  // wave-uniform: some row of the wave sees a key of these
      fl_f32x16 s[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kt][i] = 0.0f;
        const int key = 64 * way + kt * 32 + r;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const uint4 kf = *reinterpret_cast<const uint4*>(ks[b] + key * 128 + (((2 * st + hf) ^ ((key >> 1) & 7)) * 16));
          s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fl_bf16x8, kf),
                                                          __builtin_bit_cast(fl_bf16x8, qf[st]), s[kt], 0, 0, 0);
        }
      }
      // s[kt][i]: key kb + 32 kt + 8 (i / 4) + 4 hf + i % 4 of this lane's row
      float mx = -INFINITY;
      if (kb + 63 > wfirst) {  // keys past some row's last one
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = kb + 32 * kt + 8 * (i >> 2) + 4 * hf + (i & 3);
            s[kt][i] = key <= lim ? s[kt][i] * a.sc : -INFINITY;
            mx = fmaxf(mx, s[kt][i]);
          }
      } else {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            s[kt][i] = s[kt][i] * a.sc;
            mx = fmaxf(mx, s[kt][i]);
          }
      }
      mx = xor32_max(mx);
      const float mn = fmaxf(mrun, mx), mu = mn == -INFINITY ? 0.0f : mn;
      const float corr = __builtin_amdgcn_exp2f(mrun - mu);
      mrun = mn;
      float ps = 0.0f;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[kt][i] = __builtin_amdgcn_exp2f(s[kt][i] - mu);
          ps += s[kt][i];
        }
      lrun = lrun * corr + xor32_sum(ps);
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= corr;
#pragma unroll
      for (int st = 0; st < 4; ++st) {  // 16 keys: score registers 8 (st % 2) .. + 7 of tile half st / 2
        uint32_t ph[4], pm[4], pl[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = s[st >> 1][8 * (st & 1) + 2 * e], p1 = s[st >> 1][8 * (st & 1) + 2 * e + 1];
          ph[e] = pack_bf16x2(p0, p1);
          const float r0 = p0 - bflo(ph[e]), r1 = p1 - bfhi(ph[e]);
          pm[e] = pack_bf16x2(r0, r1);
          pl[e] = pack_bf16x2(r0 - bflo(pm[e]), r1 - bfhi(pm[e]));
        }
        const fl_bf16x8 bh = __builtin_bit_cast(fl_bf16x8, make_uint4(ph[0], ph[1], ph[2], ph[3]));
        const fl_bf16x8 bm = __builtin_bit_cast(fl_bf16x8, make_uint4(pm[0], pm[1], pm[2], pm[3]));
        const fl_bf16x8 bl = __builtin_bit_cast(fl_bf16x8, make_uint4(pl[0], pl[1], pl[2], pl[3]));
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const uint16_t* vp = &vt[b][way * 64 * PA_VLD + (d * 32 + r) * PA_VLD + 16 * st + 4 * hf];
          const uint2 v0 = *reinterpret_cast<const uint2*>(vp), v1 = *reinterpret_cast<const uint2*>(vp + 8);
          const fl_bf16x8 va = __builtin_bit_cast(fl_bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, bh, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, bm, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, bl, o[d], 0, 0, 0);
        }
      }
    }
    if (more) store(b ^ 1);
  }
  if constexpr (W == 2) {  // the second way's (max, sum, o) into the first's, through LDS (K's place)
    __syncthreads();
    float* mrg = reinterpret_cast<float*>(&ks[0][0]) + sub * (34 * 64) + lane;
    static_assert(W == 1 || WR * 34 * 64 * 4 <= sizeof(ks), "the ways' exchange fits K's place");
    if (way == 1) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) mrg[(d * 16 + i) * 64] = o[d][i];
      mrg[32 * 64] = mrun;
      mrg[33 * 64] = lrun;
    }
    __syncthreads();
    if (way == 1) return;
    const float m1 = mrg[32 * 64], mm = fmaxf(mrun, m1), mu = mm == -INFINITY ? 0.0f : mm;
    const float e0 = __builtin_amdgcn_exp2f(mrun - mu), e1 = __builtin_amdgcn_exp2f(m1 - mu);
    mrun = mm;
    lrun = lrun * e0 + mrg[33 * 64] * e1;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * e0 + mrg[(d * 16 + i) * 64] * e1;
  }
  if (row >= R) return;
  if (a.parts == 1) {
    uint16_t* d0 = a.out + ((size_t)t * a.nh + head) * 64 + 4 * hf;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<uint2*>(d0 + 32 * d + 8 * e) =
            make_uint2(pack_bf16x2(o[d][4 * e] / lrun, o[d][4 * e + 1] / lrun),
                       pack_bf16x2(o[d][4 * e + 2] / lrun, o[d][4 * e + 3] / lrun));
  } else {
    const size_t idx = ((size_t)part * a.nkv + g) * R + row;
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<fl_f32x4*>(a.part + idx * 64 + 32 * d + 8 * e + 4 * hf) =
            fl_f32x4{o[d][4 * e], o[d][4 * e + 1], o[d][4 * e + 2], o[d][4 * e + 3]};
    if (hf == 0) {
      float* ml = a.part + (size_t)a.parts * a.nkv * R * 64 + idx * 2;
      ml[0] = mrun;
      ml[1] = lrun;
    }
  }
}

// The key parts of a row merged in order: one wave per row, lane = dim
__global__ __launch_bounds__(256) void k_pf_attn_merge(PaArgs a) {
  const int R = a.T * a.rep, lane = threadIdx.x & 63;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= a.nkv * R) return;
  const int g = w / R, row = w % R;
  const float* ml = a.part + (size_t)a.parts * a.nkv * R * 64;
  float mm = -INFINITY;
  for (int p = 0; p < a.parts; ++p) mm = fmaxf(mm, ml[(((size_t)p * a.nkv + g) * R + row) * 2]);
  float L = 0.0f, O = 0.0f;
  for (int p = 0; p < a.parts; ++p) {
    const size_t idx = ((size_t)p * a.nkv + g) * R + row;
    const float pm = ml[idx * 2], e = pm == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(pm - mm);
    L += ml[idx * 2 + 1] * e;
    O += a.part[idx * 64 + lane] * e;
  }
  a.out[((size_t)(row / a.rep) * a.nh + g * a.rep + row % a.rep) * 64 + lane] = (uint16_t)f2bf(O / L);
}

// ---- LM head of one token, greedy argmax -------------------------------------------------------------
// x: the final-normed row. Waves take rows of the tied embedding, four at a time; logits = bf16(bf16(x .
// E^T) / logits_scaling) (engine/model.py:144); each workgroup's best (value, -index) key to best[].
__global__ __launch_bounds__(PF_NT) void k_pf_lmhead(const uint16_t* __restrict__ x, const uint16_t* __restrict__ embed,
                                                     int V, int D, float scaling, unsigned long long* __restrict__ best) {
  constexpr int C = 6, RB = 4;  // 16-byte chunks per lane of a row (D <= 3072); rows per step
  __shared__ unsigned long long red[PF_NT / FL_WAVE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = gridDim.x * (PF_NT / FL_WAVE), w = blockIdx.x * (PF_NT / FL_WAVE) + wave;
  const auto xr = buf_rsrc(x, (uint32_t)D * 2u);
  uint4 xv[C];
#pragma unroll
  for (int i = 0; i < C; ++i) xv[i] = buf_ld128(xr, (uint32_t)(lane + 64 * i) * 16u);  // zeros past D
  unsigned long long b = 0ull;
  for (int r0 = w * RB; r0 < V; r0 += nw * RB) {
    uint4 e[RB][C];
    const auto er = buf_rsrc(embed + (size_t)r0 * D, (uint32_t)min(RB, V - r0) * (uint32_t)D * 2u);
#pragma unroll
    for (int k = 0; k < RB; ++k)
#pragma unroll
      for (int i = 0; i < C; ++i)
        e[k][i] = buf_ld128(er, lane + 64 * i < (D >> 3) ? (uint32_t)k * (uint32_t)D * 2u + (uint32_t)(lane + 64 * i) * 16u : 0xFFFFFFF0u);
#pragma unroll
    for (int k = 0; k < RB; ++k) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < C; ++i) {
        s = dot2_bf16(e[k][i].x, xv[i].x, s);
        s = dot2_bf16(e[k][i].y, xv[i].y, s);
        s = dot2_bf16(e[k][i].z, xv[i].z, s);
        s = dot2_bf16(e[k][i].w, xv[i].w, s);
      }
      s = wave_sum(s);
      if (r0 + k < V) b = u64max(b, amax_key(rbf(rbf(s) / scaling), (uint32_t)(r0 + k)));
    }
  }
  if (lane == 0) red[wave] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 1; k < PF_NT / FL_WAVE; ++k) b = u64max(b, red[k]);
    best[blockIdx.x] = b;
  }
}

__global__ __launch_bounds__(64) void k_pf_argmax(const unsigned long long* __restrict__ best, int n,
                                                  int32_t* __restrict__ token_out) {
  unsigned long long b = 0ull;
  for (int i = threadIdx.x; i < n; i += 64) b = u64max(b, best[i]);
  b = wave_max_u64(b);
  if (threadIdx.x == 0) *token_out = (int32_t)amax_index(b);
}

// ---- host ---------------------------------------------------------------------------------------------
// Workspace of one pass of T tokens (16-byte aligned pieces)
struct PfWs {
  uint16_t *h, *xn, *q, *attn, *act;
  float* part;
  unsigned long long* best;
  size_t bytes;
};
PfWs pf_layout(const fl_model_desc& d, int T, uint8_t* base) {
  PfWs w{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    uint8_t* p = base + at;
    at += (bytes + 255) / 256 * 256;
    return p;
  };
  const size_t row = (size_t)T * d.dim * 2;
  w.h = (uint16_t*)take(row);
  w.xn = (uint16_t*)take(row);
  w.q = (uint16_t*)take(row);
  w.attn = (uint16_t*)take(row);
  w.act = (uint16_t*)take((size_t)T * d.inter * 2);
  // the GEMMs' part sums; the attention's key parts (o and (m, l) per row) take turns with them
  // (more than one part only while parts x blocks x groups <= PA_WGS workgroups of 64 rows)
  const size_t rows = std::min((size_t)PF_KEY_PARTS * T * d.n_head, (size_t)PA_WGS * 64);
  w.part = (float*)take(std::max((size_t)PF_SPLITS * T * d.dim * 4, rows * 66 * 4));
  w.best = (unsigned long long*)take(PF_LM_GRID * 8);
  w.bytes = at;
  return w;
}

template <int NW, int KW, int MB, class Epi>
void pf_launch(GemmArgs a, Epi epi, hipStream_t s) {
  a.tile(16 * NW, 16 * MB);
  constexpr int D = KW == 1 ? 2 : 1;  // groups requested ahead
  hipLaunchKernelGGL((k_gemm_rows<true, NW, KW, MB, D, D, Epi>), dim3(gemm_grid(a)), dim3(64 * NW * KW), 0, s, a, epi);
}

// One GEMM of a pass. PARTS: the epilogue keeps fp32 sums of K parts, which k_pf_norm adds;
// returns their number. Measured at flint-3b's sizes (us, weights from HBM):
// - tiles of 256 x 128 (k_gemm_big, one workgroup per CU) where they and the parts give at least 160
//   workgroups: gate/up at 512 / 1024 tokens (256 / 512 tiles) 53 / 101, 57 / 115 in tiles of 128 x 128; down at
//   512 (40 tiles) 39 in four parts, 42 in tiles of 64 x 64; O at 512 has too few groups for four parts of eight; not
//   where a second round would be half empty or more: gate/up at 576 / 768 tokens (320 / 384) cost 12 / 8 us a layer more
//   than in tiles of 128 x 128, at 896 (448) 8 less;
// - else tiles of 64 x 64, up to 256 of them four ways, up to 512 two: QKV at 64 / 512 tokens (56 / 448 tiles)
//   20 / 27 with one way, 14 / - with four, - / 24 with two; gate/up at 64 (256) 21 and 15; parts of about ten
//   groups, four at most, more while they give fewer than 160 workgroups: O at 512 (320 tiles) 19 in two parts,
//   at 64 tokens 8 in four; down at 64 tokens 11 in four with four ways, 16 with one;
// - tiles of 128 x 128 in between: QKV at 1024 (224 tiles) 39.
template <bool PARTS, class Epi>
int pf_gemm(const uint32_t* qt, const uint32_t* sz, const uint16_t* x, int T, int n, int k, Epi epi, hipStream_t s) {
  const int G = k / FL_GROUP;
  GemmArgs a{qt, sz, x, T, n, k, 0, 0, 1, G, 0};
  const int t64 = ((n + 63) / 64) * ((T + 63) / 64), t256 = ((n + 255) / 256) * ((T + 127) / 128);
  auto cut = [&](int want, int least) {  // K in `want` parts of at least `least` groups
    const int s = std::max(1, std::min({PF_SPLITS, want, G / least}));
    a.gps = (G + s - 1) / s;
    a.splits = (G + a.gps - 1) / a.gps;
  };
  if (PARTS) cut(256 / t256, 8);
  const int big = t256 * a.splits;
  if (big >= 160 && (big <= 256 || big > 384)) {
    a.tile(256, 128);
    hipLaunchKernelGGL((k_gemm_big<true, 8, Epi>), dim3(gemm_grid(a)), dim3(512), 0, s, a, epi);
    return a.splits;
  }
  if (PARTS) cut(std::max(G / 10, (160 + t64 - 1) / t64), 4);
  if constexpr (!PARTS) {
    if (((n + 127) / 128) * ((T + 127) / 128) >= 160) {
      pf_launch<8, 1, 8>(a, epi, s);
      return a.splits;
    }
  }
  const int wgs = t64 * a.splits;
  if (wgs <= 256 && a.gps >= 8) pf_launch<4, 4, 4>(a, epi, s);
  else if (wgs <= 512 && a.gps >= 8) pf_launch<4, 2, 4>(a, epi, s);
  else pf_launch<4, 1, 4>(a, epi, s);
  return a.splits;
}

void pf_attention(const fl_state* st, const PfWs& w, int l, int T, int pos, hipStream_t s) {
  const fl_model_desc& d = st->d;
  PaArgs a{};
  const size_t layer = (size_t)l * d.n_kv_head * st->max_seq * 64;
  a.q = w.q;
  a.kc = st->kc + layer;
  a.vc = st->vc + layer;
  a.out = w.attn;
  a.part = w.part;
  a.T = T;
  a.pos = pos;
  a.S = st->max_seq;
  a.nh = d.n_head;
  a.nkv = d.n_kv_head;
  a.rep = d.n_head / d.n_kv_head;
  const int b128 = (T * a.rep + 127) / 128;
  // one way for rows that fill the chip behind many keys: 1024 tokens cost 7 us less a layer with two
  // over no keys and 0.006 us more per key (12 us at 4000), so the two meet near 1100
  const bool one_way = b128 * a.nkv >= 256 && pos >= 2048;
  a.blocks = one_way ? b128 : (T * a.rep + 63) / 64;
  a.sc = d.attn_scale * 1.4426950408889634f;
  // key parts up to PA_WGS workgroups (two per CU), at least 256 keys each: 40 tokens behind
  // 12000 keys (32 workgroups uncut) 94 us a layer, of which 31 over no keys; at most four parts 157
  const int keys = pos + T;
  const int parts = one_way ? 1 : std::max(1, std::min({PF_KEY_PARTS, PA_WGS / (a.blocks * a.nkv), keys / 256}));
  a.kpp = ((keys + parts - 1) / parts + 127) / 128 * 128;
  a.parts = (keys + a.kpp - 1) / a.kpp;
  const dim3 grid(a.blocks * a.parts * a.nkv);
  if (one_way) hipLaunchKernelGGL(k_pf_attn<1>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_pf_attn<2>, grid, dim3(256), 0, s, a);
  if (a.parts > 1)
    hipLaunchKernelGGL(k_pf_attn_merge, dim3((a.nkv * T * a.rep + 3) / 4), dim3(256), 0, s, a);
}

void pf_pass(const fl_weights* w, fl_state* st, const PfWs& ws, const int32_t* tokens, int T, int pos, hipStream_t s) {
  const fl_model_desc& d = st->d;
  const int D = d.dim, F = d.inter, NQKV = (d.n_head + 2 * d.n_kv_head) * FL_HEAD_DIM, L = d.n_layer;
  auto mat = [&](const uint32_t* p, int l, int n, int k, int per) { return p + (size_t)l * n * (k / per); };
  hipLaunchKernelGGL(k_pf_norm, dim3(T), dim3(PF_NT), 0, s, ws.part, 0, T, D, tokens, w->embed, d.vocab, d.emb_mult,
                     w->attn_norm, d.norm_eps, ws.h, ws.xn, st->err);
  for (int l = 0; l < L; ++l) {
    const size_t layer = (size_t)l * d.n_kv_head * st->max_seq * 64;
    pf_gemm<false>(mat(w->wqkv_t, l, NQKV, D, 8), mat(w->wqkv_sz, l, NQKV, D, 128), ws.xn, T, NQKV, D,
                   EpiQkv{ws.q, st->kc + layer, st->vc + layer, reinterpret_cast<const uint32_t*>(w->rope), T, d.n_head,
                          d.n_kv_head, st->max_seq, pos}, s);
    pf_attention(st, ws, l, T, pos, s);
    int parts = pf_gemm<true>(mat(w->wo_t, l, D, D, 8), mat(w->wo_sz, l, D, D, 128), ws.attn, T, D, D,
                              EpiSum{ws.part, T, D}, s);
    hipLaunchKernelGGL(k_pf_norm, dim3(T), dim3(PF_NT), 0, s, ws.part, parts, T, D, tokens, w->embed, d.vocab,
                       d.resid_mult, w->ffn_norm + (size_t)l * D, d.norm_eps, ws.h, ws.xn, st->err);
    pf_gemm<false>(mat(w->wgu_t, l, 2 * F, D, 8), mat(w->wgu_sz, l, 2 * F, D, 128), ws.xn, T, 2 * F, D,
                   EpiSwiglu{ws.act, T, F}, s);
    parts = pf_gemm<true>(mat(w->wd_t, l, D, F, 8), mat(w->wd_sz, l, D, F, 128), ws.act, T, D, F,
                          EpiSum{ws.part, T, D}, s);
    const uint16_t* next = l + 1 < L ? w->attn_norm + (size_t)(l + 1) * D : w->final_norm;
    hipLaunchKernelGGL(k_pf_norm, dim3(T), dim3(PF_NT), 0, s, ws.part, parts, T, D, tokens, w->embed, d.vocab,
                       d.resid_mult, next, d.norm_eps, ws.h, ws.xn, st->err);
  }
}

}  // namespace

extern "C" {

int fl_prefill_workspace(fl_state* st, int32_t n, int64_t* bytes) {
  if (!st || n < 1 || !bytes) return FL_E_ARG;
  *bytes = (int64_t)pf_layout(st->d, std::min(n, PF_TOKENS), nullptr).bytes;
  return FL_OK;
}

int fl_prefill(const fl_weights* w, fl_state* st, const int32_t* tokens, int32_t n, int32_t pos, int32_t* token_out,
               void* workspace, void* stream) {
  if (!st || !tokens || !token_out || !workspace || n < 1 || !fl_weights_ok(w)) return FL_E_ARG;
  // what fl_verify needs too: the tiled weight copies, a model that its kernels take
  if (!w->wqkv_t || !w->wo_t || !w->wgu_t || !w->wd_t || !st->verify_ok) return FL_E_ARG;
  if (pos < 0 || pos > st->max_seq - n || pos > w->rope_len - n) return FL_E_POS;
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int most = std::min(n, PF_TOKENS);
  const PfWs ws = pf_layout(st->d, most, static_cast<uint8_t*>(workspace));
  int T = 0;
  for (int at = 0; at < n; at += T) {
    T = std::min(most, n - at);
    pf_pass(w, st, ws, tokens + at, T, pos + at, s);
  }
  hipLaunchKernelGGL(k_pf_lmhead, dim3(PF_LM_GRID), dim3(PF_NT), 0, s, ws.xn + (size_t)(T - 1) * st->d.dim, w->embed,
                     st->d.vocab, st->d.dim, st->d.logits_scaling, ws.best);
  hipLaunchKernelGGL(k_pf_argmax, dim3(1), dim3(64), 0, s, ws.best, PF_LM_GRID, token_out);
  return hipGetLastError() == hipSuccess ? FL_OK : FL_E_LAUNCH;
}

}  // extern "C"
