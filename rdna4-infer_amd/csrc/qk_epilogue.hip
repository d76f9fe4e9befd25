// Pre-attention epilogue of a full-attention layer, fused (gfx950).
//
// The reference runs six launches between the QKV projections and attention
// (graph.cuh:914-954 for one token, graph.cuh:1444-1462 for a chunk):
//   deinterleave_q_gate (gdn.cuh:367-384, 836-860)  [q|gate] per head -> q, gate
//   rms_norm(q, attn_q_norm), rms_norm(k, attn_k_norm)        (nn.cuh:24-63)
//   rope(q), rope(k)                                         (attn.cuh:30-63)
//   kv_write_batch: K and V rows quantized into the cache    (kv.h:386-501)
// Every step is row-local, so one wave owns one head row of one token from
// load to store: the row is read once from HBM, normalised and rotated in
// registers, and written once (q, optionally k) plus its cache bytes.
//
// Bit-identity with the unfused sequence:
//   - the sum of squares follows rms_norm_kernel's order exactly: "thread" t
//     (t < 256) chains fmaf over elements t, t+256, ..., and the 256 partials
//     meet in the tree p[t] += p[t + s], s = 128 .. 1. A lane holds elements
//     4*lane + i (+256), so strides 128..4 are xor shuffles 32..1 (IEEE
//     addition commutes, so lane t^s adds the same pair) and strides 2, 1 are
//     the in-lane (e0+e2)+(e1+e3);
//   - rsqrtf(sum / ncols + eps), then (x * scale) * w;
//   - RoPE through rope_cs / rope_lo / rope_hi, shared with rope_kernel;
//   - the quantizer is store_group4, shared with kv_store_row and the decode
//     append, with the same lane-to-block mapping.
#include <algorithm>
#include <type_traits>

#include "kv_quant.hpp"
#include "merge.hpp"

namespace rd4 {

namespace {

constexpr int kRmsThreads = 256;  // rms_norm_kernel's block (nn.cuh:22)
constexpr int kEpiWaves = 4;
constexpr int kEpiMaxHd = 512;
// CTAs of a launch that fill the CUs: 2048 tokens take 43.9 us in 4096 CTAs (two per
// token), 48.3 us in 2048 and 46.3 us in 16384; 512 tokens 14.2-14.4 us in all of these
constexpr int kEpiCtas = 4096;

// Standalone row RMSNorm with the reference's arithmetic, any ncols.
__global__ __launch_bounds__(kRmsThreads) void rms_norm_kernel(const float *__restrict__ x,
                                                               const float *__restrict__ w,
                                                               float *y, int64_t ncols, float eps) {
  __shared__ float part[kRmsThreads];
  const int tid = threadIdx.x;
  const float *xr = x + (int64_t)blockIdx.x * ncols;
  float *yr = y + (int64_t)blockIdx.x * ncols;
  float acc = 0.0f;
  int64_t i = tid;
  for (; i + 3 * kRmsThreads < ncols; i += 4 * kRmsThreads) {
    const float v0 = xr[i], v1 = xr[i + kRmsThreads], v2 = xr[i + 2 * kRmsThreads],
                v3 = xr[i + 3 * kRmsThreads];
    acc = fmaf(v0, v0, acc);
    acc = fmaf(v1, v1, acc);
    acc = fmaf(v2, v2, acc);
    acc = fmaf(v3, v3, acc);
  }
  for (; i < ncols; i += kRmsThreads) acc = fmaf(xr[i], xr[i], acc);
  part[tid] = acc;
  __syncthreads();
  if (tid < 128) part[tid] = __fadd_rn(part[tid], part[tid + 128]);
  __syncthreads();
  if (tid < 64) {
    float v = __fadd_rn(part[tid], part[tid + 64]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = __fadd_rn(v, xor_f(v, m));
    if (tid == 0) part[0] = v;
  }
  __syncthreads();
  const float scale = rsqrtf(__fadd_rn(__fdiv_rn(part[0], (float)ncols), eps));
  for (int64_t j = tid; j < ncols; j += kRmsThreads) {
    const float s = __fmul_rn(xr[j], scale);
    yr[j] = w ? __fmul_rn(s, w[j]) : s;
  }
}

struct EpiArgs {
  const float *qg, *k, *v, *qw, *kw;
  const int *pos;
  float *q_out, *gate_out, *k_out;
  uint8_t *kc, *vc;
  int64_t krb, vrb;
  float eps, freq_base;
  int n_rot, n_tok, n_head, n_head_kv, head_dim, kt, vt;
  int groups;  // CTAs per token
};

// x summed over the 64 lanes, in every lane, pairing lanes 32, 16, .., 1 apart in
// that order (the tree of __shfl_xor sums, bit for bit: addition commutes, and
// past the stride-8 step lanes 8 apart hold equal values, so a rotation by 4 meets
// the same partner value as an exchange 4 apart).
__device__ __forceinline__ float tree_sum64(float x) {
  float a = x, b = x;
  swap32(a, b);
  a = __fadd_rn(a, b);
  b = a;
  swap16(a, b);
  x = __fadd_rn(a, b);
  auto dpp = [](float v, auto ctrl) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, decltype(ctrl)::value, 0xF, 0xF, false));
  };
  x = __fadd_rn(x, dpp(x, std::integral_constant<int, 0x128>{}));  // row_ror:8
  x = __fadd_rn(x, dpp(x, std::integral_constant<int, 0x124>{}));  // row_ror:4
  x = __fadd_rn(x, dpp(x, std::integral_constant<int, 0x4E>{}));   // quad_perm 2,3,0,1
  return __fadd_rn(x, dpp(x, std::integral_constant<int, 0xB1>{}));  // quad_perm 1,0,3,2
}

__device__ __forceinline__ void store_typed(int t, const float x[4], int sub, uint8_t *row, int blk) {
  switch (t) {
    case F32: store_group4<F32>(x, sub, row, blk); break;
    case F16: store_group4<F16>(x, sub, row, blk); break;
    case Q8_0: store_group4<Q8_0>(x, sub, row, blk); break;
    case Q4_0: store_group4<Q4_0>(x, sub, row, blk); break;
    case Q5_0: store_group4<Q5_0>(x, sub, row, blk); break;
    default: store_group4<Q4_1>(x, sub, row, blk); break;
  }
}

// One CTA per (token, row group): the group's rows are dealt to the CTA's waves,
// one row at a time per wave, the next row's loads in flight while a row is
// worked on. Rows of a token: n_head q heads, then n_head_kv k heads, then
// n_head_kv v heads.
// What bounds it: a chunk streams its projections once (HBM); one token is
// latency. The RoPE angles (a powf, a cosf and a sinf each, the long part of the
// arithmetic) are formed once per CTA, one per thread, while the first rows are
// on their way, instead of four per lane in every row; the sum of squares meets
// by VALU lane exchanges instead of LDS round trips. 2048 tokens, 24 / 4 heads,
// q8_0 caches: 90 -> 44 us (5.1 TB/s); one token 6.1 -> 4.3 us.
template <int G>  // 256-element groups per row: 1 (head_dim <= 256) or 2
__global__ __launch_bounds__(64 * kEpiWaves) void qk_epilogue_kernel(EpiArgs a) {
  __shared__ float rows[kEpiWaves][kEpiMaxHd];
  __shared__ float2 cs[kEpiMaxHd / 2];  // (cos, sin) of the rotated pairs
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int per_tok = a.n_head + 2 * a.n_head_kv;
  const int tok = (int)blockIdx.x / a.groups, grp = (int)blockIdx.x - tok * a.groups;
  const int step = kEpiWaves * a.groups;
  const int HD = a.head_dim;
  const bool on = 4 * lane < (HD < 256 ? HD : 256);
  const int pos = a.pos[tok];

  // row r of the token: kind 0 q, 1 k, 2 v; h its head; hrow its row in that array
  auto kind_of = [&](int r) { return r < a.n_head ? 0 : (r < a.n_head + a.n_head_kv ? 1 : 2); };
  auto head_of = [&](int r) { return r < a.n_head ? r : (r < a.n_head + a.n_head_kv ? r - a.n_head : r - a.n_head - a.n_head_kv); };
  float4 nx[G], ng[G];  // the row to come: values, and the gate half of a q row
  auto load = [&](int r) {
    const int kind = kind_of(r);
    const int64_t hrow = (int64_t)tok * (kind == 0 ? a.n_head : a.n_head_kv) + head_of(r);
    const float *src = kind == 0 ? a.qg + hrow * 2 * HD : (kind == 1 ? a.k : a.v) + hrow * HD;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nx[g] = on ? *(const float4 *)(src + 256 * g + 4 * lane) : make_float4(0.f, 0.f, 0.f, 0.f);
      if (kind == 0 && a.gate_out && on) ng[g] = *(const float4 *)(src + HD + 256 * g + 4 * lane);
    }
  };
  int r = grp * kEpiWaves + wave;
  if (r < per_tok) load(r);
  const int half = a.n_rot >> 1;
  if ((int)threadIdx.x < half) {  // (half <= 256 = the CTA's threads)
    float c, s;
    rope_cs(pos, (int)threadIdx.x, a.n_rot, a.freq_base, &c, &s);
    cs[threadIdx.x] = make_float2(c, s);
  }
  __syncthreads();

  for (; r < per_tok; r += step) {
    const int kind = kind_of(r), h = head_of(r);
    const int64_t hrow = (int64_t)tok * (kind == 0 ? a.n_head : a.n_head_kv) + h;
    float x[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      x[g][0] = nx[g].x;
      x[g][1] = nx[g].y;
      x[g][2] = nx[g].z;
      x[g][3] = nx[g].w;
    }
    if (kind == 0 && a.gate_out && on) {
#pragma unroll
      for (int g = 0; g < G; ++g) *(float4 *)(a.gate_out + hrow * HD + 256 * g + 4 * lane) = ng[g];
    }
    if (r + step < per_tok) load(r + step);

    if (kind != 2) {
      float t[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        t[i] = fmaf(x[0][i], x[0][i], 0.0f);
        if constexpr (G == 2) t[i] = fmaf(x[1][i], x[1][i], t[i]);
        t[i] = tree_sum64(t[i]);
      }
      const float sum = __fadd_rn(__fadd_rn(t[0], t[2]), __fadd_rn(t[1], t[3]));
      const float scale = rsqrtf(__fadd_rn(__fdiv_rn(sum, (float)HD), a.eps));
      const float *w = kind == 0 ? a.qw : a.kw;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float s = __fmul_rn(x[g][i], scale);
          x[g][i] = (w && on) ? __fmul_rn(s, w[256 * g + 4 * lane + i]) : s;
        }

      if (a.n_rot > 0) {
        float *row = rows[wave];
        // the row is exchanged between the lanes of this wave only: its writes stay
        // behind the reads of the wave's previous row, its reads behind them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (on) {
#pragma unroll
          for (int g = 0; g < G; ++g)
            *(float4 *)(row + 256 * g + 4 * lane) = make_float4(x[g][0], x[g][1], x[g][2], x[g][3]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int d = 256 * g + 4 * lane + i;
            if (on && d < a.n_rot) {
              const int p = d < half ? d : d - half;
              const float2 c = cs[p];
              const float x0 = row[p], x1 = row[p + half];
              x[g][i] = d < half ? rope_lo(x0, x1, c.x, c.y) : rope_hi(x0, x1, c.x, c.y);
            }
          }
      }
    }

    if (kind == 0 || (kind == 1 && a.k_out)) {
      float *dst = (kind == 0 ? a.q_out : a.k_out) + hrow * HD;
      if (on) {
#pragma unroll
        for (int g = 0; g < G; ++g)
          *(float4 *)(dst + 256 * g + 4 * lane) = make_float4(x[g][0], x[g][1], x[g][2], x[g][3]);
      }
    }
    if (kind != 0 && on) {
      const int type = kind == 1 ? a.kt : a.vt;
      uint8_t *row = (kind == 1 ? a.kc : a.vc) +
                     ((int64_t)pos * a.n_head_kv + h) * (kind == 1 ? a.krb : a.vrb);
#pragma unroll
      for (int g = 0; g < G; ++g) store_typed(type, x[g], lane & 7, row, 8 * g + (lane >> 3));
    }
  }
}

}  // namespace

hipError_t rms_norm_launch(const float *x, const float *w, float *y, int64_t nrows, int64_t ncols,
                           float eps, hipStream_t st) {
  if (nrows <= 0 || ncols <= 0) return hipSuccess;
  hipLaunchKernelGGL(rms_norm_kernel, dim3((unsigned)nrows), dim3(kRmsThreads), 0, st, x, w, y,
                     ncols, eps);
  return hipGetLastError();
}

hipError_t qk_epilogue_launch(const float *qg, const float *k, const float *v, const float *qw,
                              const float *kw, float eps, int n_rot, float freq_base,
                              const int *pos, int n_tok, int n_head, int n_head_kv, int head_dim,
                              float *q_out, float *gate_out, float *k_out, uint8_t *kc,
                              uint8_t *vc, int kt, int vt, hipStream_t st) {
  EpiArgs a;
  a.qg = qg;
  a.k = k;
  a.v = v;
  a.qw = qw;
  a.kw = kw;
  a.pos = pos;
  a.q_out = q_out;
  a.gate_out = gate_out;
  a.k_out = k_out;
  a.kc = kc;
  a.vc = vc;
  a.krb = row_bytes(kt, head_dim);
  a.vrb = row_bytes(vt, head_dim);
  a.eps = eps;
  a.freq_base = freq_base;
  a.n_rot = n_rot;
  a.n_tok = n_tok;
  a.n_head = n_head;
  a.n_head_kv = n_head_kv;
  a.head_dim = head_dim;
  a.kt = kt;
  a.vt = vt;
  if (n_tok <= 0) return hipSuccess;
  // CTAs per token: one row per wave while the tokens alone leave CUs short of
  // waves, else fewer groups of more rows, whose angles are shared
  const int most = (n_head + 2 * n_head_kv + kEpiWaves - 1) / kEpiWaves;
  a.groups = std::max(1, std::min(most, (kEpiCtas + n_tok - 1) / n_tok));
  const dim3 grid((unsigned)((int64_t)n_tok * a.groups)), block(64 * kEpiWaves);
  if (head_dim > 256)
    hipLaunchKernelGGL(qk_epilogue_kernel<2>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(qk_epilogue_kernel<1>, grid, block, 0, st, a);
  return hipGetLastError();
}

}  // namespace rd4
