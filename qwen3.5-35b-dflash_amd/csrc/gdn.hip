// Gated-DeltaNet mixer kernels (the decoder layer's non-GEMM arithmetic around its int4
// projections), head dims 128, four conv taps, fp32 throughout.
//
// Reference arithmetic: model/qwen35_moe_dflash/fused/model.py:206-263 (norms, conv, gates, gated
// norm) and fused/ops.py:54-71 (the delta rule per token: S <- e^g S; u = beta (v - S^T k);
// S <- S + k u^T; o = S^T q).  With G_t the running sum of g inside a chunk of 16 tokens, the rule is
//   (I + A) U = diag(beta) (V - diag(e^G) K S0),   A_ts = beta_t e^{G_t - G_s} k_t.k_s  (s < t)
//   O = diag(e^G) Q S0 + P U,                        P_ts = e^{G_t - G_s} q_t.k_s         (s <= t)
//   S16 = e^{G_16} S0 + K~^T U,                      k~_s = e^{G_16 - G_s} k_s
// and the solve is linear in S0: U = U0 - W S0 with U0 = (I + A)^-1 diag(beta) V and
// W = (I + A)^-1 diag(beta e^G) K.  So everything but three products with the state is
// independent of the state, and only those run chunk after chunk:
//   gdn_chunk_kernel  one workgroup per (value head, chunk): conv + SiLU, Q/K normalisation, the
//                     gates, K K^T and Q K^T on the fp32 matrix cores, the triangular solve by
//                     forward substitution (one right-hand column per thread);
//   gdn_state_kernel  one workgroup per (value head, 16 state columns), its 128 x 16 state slice in
//                     registers for the whole block: per chunk U = U0 - W S, O = Q~ S + P U, S update.
#include "kernels.h"

namespace dflash {
namespace {

constexpr int kD = 128;          // head dims (Dk = Dv)
constexpr int kChunk = 16;       // tokens per chunk
constexpr int kTaps = 4;         // depthwise conv taps
constexpr int kRow = kD + 4;     // LDS row pitch of a 128-wide fp32 row

__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + expf(-x)); }

// ------------------------------------------------------------------ residual add + RMS norm
// One workgroup per row.  mid = hidden + mixed (when mixed is given), normed = mid * rsqrt(mean mid^2 + eps) * (w + 1),
// bf16, or fp32 (kF32: a model's final norm, one launch in place of seven).  Bound by latency at the block sizes of a decode or verify call (one row is 8 KB);
// one launch (T = 16: 3.2 us) in place of eight elementwise and reduction launches (25 us).
template <bool kF32>
__global__ __launch_bounds__(512) void add_norm_kernel(const float* hidden, const uint16_t* mixed, const float* w,
                                                       float eps, int H, float* mid, void* normed) {
  __shared__ float part[8];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  constexpr int kPer = kMaxNormWidth / 2048;  // float4 columns a thread holds
  float4 v[kPer];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = 4 * tid + 2048 * i;
    if (c < H) {
      v[i] = *reinterpret_cast<const float4*>(hidden + row * H + c);
      if (mixed) {
        const uint2 m = *reinterpret_cast<const uint2*>(mixed + row * H + c);
        v[i].x += __uint_as_float(m.x << 16);
        v[i].y += __uint_as_float(m.x & 0xFFFF0000u);
        v[i].z += __uint_as_float(m.y << 16);
        v[i].w += __uint_as_float(m.y & 0xFFFF0000u);
        *reinterpret_cast<float4*>(mid + row * H + c) = v[i];
      }
      sum += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
    }
  }
  sum = wave_sum(sum);
  if ((tid & 63) == 0) part[tid >> 6] = sum;
  __syncthreads();
  const float total = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
  const float inv = rsqrtf(total / H + eps);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = 4 * tid + 2048 * i;
    if (c < H) {
      const float4 g = *reinterpret_cast<const float4*>(w + c);
      const float4 y = make_float4(v[i].x * inv * (g.x + 1.0f), v[i].y * inv * (g.y + 1.0f), v[i].z * inv * (g.z + 1.0f),
                                   v[i].w * inv * (g.w + 1.0f));
      if constexpr (kF32) {
        *reinterpret_cast<float4*>(static_cast<float*>(normed) + row * H + c) = y;
      } else {
        ushort4 o;
        o.x = f32_to_bf16(y.x);
        o.y = f32_to_bf16(y.y);
        o.z = f32_to_bf16(y.z);
        o.w = f32_to_bf16(y.w);
        *reinterpret_cast<ushort4*>(static_cast<uint16_t*>(normed) + row * H + c) = o;
      }
    }
  }
}

// ------------------------------------------------------------------ chunk preparation
// Latency-bound at one chunk (32 workgroups): a wave per token, so conv, SiLU and the Q/K normalisation stay in
// registers; then the two 16 x 16 products on one wave each beside the decay table, then the solve on four waves, while
// the other waves write what does not depend on it.  T = 16, 32 heads: 10 us (17 us with four waves a
// workgroup, each doing every phase, the window written last); T = 600: 31 us.
__global__ __launch_bounds__(1024) void gdn_chunk_kernel(GdnParams p) {
  __shared__ __align__(16) float qs[kChunk * kRow], ks[kChunk * kRow], vs[kChunk * kRow];
  __shared__ __align__(16) uint16_t raw[3][kChunk + kTaps - 1][kD + 2];  // window columns t0 - 3 .. t0 + 15
  __shared__ __align__(16) float aa[kChunk][kChunk];
  __shared__ __align__(16) float gs[kChunk];
  __shared__ float beta[kChunk], fwd[kChunk], bwd[kChunk];
  const int rep = gridDim.y, h = blockIdx.x * rep + blockIdx.y;  // key head, value head of it
  const int chunk = blockIdx.z, t0 = chunk * kChunk;
  const int n = min(kChunk, p.T - t0);  // tokens of this chunk
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int kw = gridDim.x * kD, C = 2 * kw + p.Hv * kD;
  // this head's channels of the conv: its key head's q and k, its own v
  const int base[3] = {static_cast<int>(blockIdx.x) * kD, kw + static_cast<int>(blockIdx.x) * kD, 2 * kw + h * kD};

  // conv + SiLU of token t0 + wave: a lane two neighbouring channels of each segment (256 contiguous bytes of
  // one projection row per load), every load in flight before the first use
  uint32_t x[3][kTaps];
  uint4 taps[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const int c = base[s] + 2 * lane;
    taps[s] = *reinterpret_cast<const uint4*>(p.conv + static_cast<int64_t>(c) * kTaps);
#pragma unroll
    for (int i = 0; i < kTaps; ++i) {
      const int t = t0 + wave + i - (kTaps - 1);
      if (t < 0) {
        const uint16_t* r = p.hist + static_cast<int64_t>(c) * (kTaps - 1) + (kTaps - 1) + t;
        x[s][i] = r[0] | (static_cast<uint32_t>(r[kTaps - 1]) << 16);
      } else {
        x[s][i] = *reinterpret_cast<const uint32_t*>(p.proj + static_cast<int64_t>(min(t, p.T - 1)) * p.ldp + c);
      }
    }
  }
  // the token's gates, the same in every lane (tokens past the end: g = beta = 0)
  float g = 0.f, b = 0.f;
  if (wave < n) {
    const uint16_t* r = p.proj + static_cast<int64_t>(t0 + wave) * p.ldp + C + p.Hv * kD;
    const float a = bf16_to_f32(r[p.Hv + h]) + p.dt_bias[h];
    b = 1.0f / (1.0f + expf(-bf16_to_f32(r[h])));
    g = -expf(p.a_log[h]) * (a > 20.0f ? a : log1pf(expf(a)));
  }
  if (lane == 0) {
    gs[wave] = g;
    beta[wave] = b;
  }
  float2 y[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const uint32_t tw[4] = {taps[s].x, taps[s].y, taps[s].z, taps[s].w};  // two channels' taps, four bf16 each
    float y0 = 0.f, y1 = 0.f;
#pragma unroll
    for (int j = 0; j < kTaps; ++j) {
      y0 += __uint_as_float(x[s][j] << 16) * __uint_as_float(j & 1 ? tw[j >> 1] & 0xFFFF0000u : tw[j >> 1] << 16);
      y1 += __uint_as_float(x[s][j] & 0xFFFF0000u) *
            __uint_as_float(j & 1 ? tw[2 + (j >> 1)] & 0xFFFF0000u : tw[2 + (j >> 1)] << 16);
    }
    y[s] = wave < n ? make_float2(silu_f32(y0), silu_f32(y1)) : make_float2(0.f, 0.f);
#pragma unroll
    for (int i = 0; i < kTaps; ++i)
      if (i == kTaps - 1 || wave == 0) *reinterpret_cast<uint32_t*>(&raw[s][wave + i][2 * lane]) = x[s][i];
  }
  // Q/K normalisation (q also takes Dk^-1/2)
  const float iq = rsqrtf(wave_sum(y[0].x * y[0].x + y[0].y * y[0].y) + 1e-6f) * 0.08838834764831845f;
  const float ik = rsqrtf(wave_sum(y[1].x * y[1].x + y[1].y * y[1].y) + 1e-6f);
  *reinterpret_cast<float2*>(qs + wave * kRow + 2 * lane) = make_float2(y[0].x * iq, y[0].y * iq);
  *reinterpret_cast<float2*>(ks + wave * kRow + 2 * lane) = make_float2(y[1].x * ik, y[1].y * ik);
  *reinterpret_cast<float2*>(vs + wave * kRow + 2 * lane) = y[2];
  lds_barrier();

  const int64_t row = static_cast<int64_t>(h) * gridDim.z + chunk, off = row * kChunk * kD;
  if (wave < 3) {
    // K K^T (wave 0) and Q K^T (wave 1): lane l supplies row l & 15 of both operands, k = 16 m + 4 (l >> 4) + e
    const int lr = lane & 15, kq = lane >> 4;
    f32x4 d0{0.f, 0.f, 0.f, 0.f}, d1{0.f, 0.f, 0.f, 0.f};
    if (wave < 2) {
      const float* ra = (wave ? qs : ks) + lr * kRow + 4 * kq;
      const float* rb = ks + lr * kRow + 4 * kq;
#pragma unroll
      for (int m = 0; m < 8; m += 2) {
        const f32x4 a0 = *reinterpret_cast<const f32x4*>(ra + 16 * m), b0 = *reinterpret_cast<const f32x4*>(rb + 16 * m);
        const f32x4 a1 = *reinterpret_cast<const f32x4*>(ra + 16 * m + 16),
                    b1 = *reinterpret_cast<const f32x4*>(rb + 16 * m + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d0 = mfma16x16x4f32(a0[e], b0[e], d0);
          d1 = mfma16x16x4f32(a1[e], b1[e], d1);
        }
      }
      d0 += d1;
    }
    // the running log decay, summed left to right in 64 bits so that a decay e^{G_t - G_s} is as exact as its own
    // exponent (the sum's fp32 rounding would be |G| / 2^24 of it): of token lr, and of tokens 4 kq .. 4 kq + 3
    double sum = 0.0, gl = 0.0, gr[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      sum += static_cast<double>(gs[i]);
      if (i == lr) gl = sum;
      if (i >> 2 == kq) gr[i & 3] = sum;
    }
    if (wave == 2) {
      if (lane < kChunk) {
        fwd[lr] = expf(static_cast<float>(gl));
        bwd[lr] = expf(static_cast<float>(sum - gl));
        if (lr < n) p.cum[static_cast<int64_t>(h) * p.T + t0 + lr] = static_cast<float>(gl);
        if (lr == 0) p.decay[row] = expf(static_cast<float>(sum));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 4 * kq + e;
        const float v = (lr <= t ? expf(static_cast<float>(gr[e] - gl)) : 0.f) * d0[e];
        if (wave == 0) aa[t][lr] = lr < t ? beta[t] * v : 0.f;
        else p.pmat[(row * kChunk + t) * kChunk + lr] = v;
      }
    }
  } else if (wave >= 4) {
    // the conv window (history, then the block's raw columns), token-contiguous per channel, 32 lanes a channel; q and
    // k by the first value head of their key head, the history by the first chunk
    const int64_t wp = p.T + kTaps - 1;
    const int t = lane & 31;
    const bool in = t >= (chunk == 0 ? 0 : kTaps - 1) && t < n + kTaps - 1;
#pragma unroll
    for (int s = 0; s < 3; ++s)
      if (s == 2 || blockIdx.y == 0)
        for (int c = 2 * (wave - 4) + (lane >> 5); c < kD; c += 24)
          if (in) {
            p.window[(base[s] + c) * wp + t0 + t] = raw[s][t][c];
            // the window's last three columns are also the conv history after the whole block
            if (t0 + t >= p.T) p.tail[(base[s] + c) * (kTaps - 1) + t0 + t - p.T] = raw[s][t][c];
          }
  }
  lds_barrier();

  const int ch = tid & (kD - 1), part = tid >> 7;
  if (part < 2) {
    // forward substitution, one right-hand column per thread: U0 (threads 0-127), W (128-255)
    float z[kChunk];
    const float* r = part ? ks : vs;
#pragma unroll
    for (int t = 0; t < kChunk; ++t) {
      float acc0 = r[t * kRow + ch] * (part ? beta[t] * fwd[t] : beta[t]), acc1 = 0.f;
#pragma unroll
      for (int s = 0; s < t; ++s) {
        if (s & 1) acc1 -= aa[t][s] * z[s];
        else acc0 -= aa[t][s] * z[s];
      }
      z[t] = acc0 + acc1;
    }
    // W row by row, U0 column by column (16 tokens contiguous: a 16-byte load per lane of the state kernel)
    if (part) {
#pragma unroll
      for (int t = 0; t < kChunk; ++t) p.w[off + t * kD + ch] = z[t];
    } else {
      float* u0 = p.u0 + off + ch * kChunk;
#pragma unroll
      for (int t = 0; t < kChunk; t += 4)
        *reinterpret_cast<float4*>(u0 + t) = make_float4(z[t], z[t + 1], z[t + 2], z[t + 3]);
    }
  } else if (part < 4) {
    // Q~ = e^G Q row by row, eight tokens a thread
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = 8 * (part - 2) + i;
      p.qt[off + t * kD + ch] = qs[t * kRow + ch] * fwd[t];
    }
  } else if (part < 6) {
    // K~ = e^{G16 - G} K column by column
    float* kt = p.kt + off + ch * kChunk + 8 * (part - 4);
    float k[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) k[i] = ks[(8 * (part - 4) + i) * kRow + ch] * bwd[8 * (part - 4) + i];
    *reinterpret_cast<float4*>(kt) = make_float4(k[0], k[1], k[2], k[3]);
    *reinterpret_cast<float4*>(kt + 4) = make_float4(k[4], k[5], k[6], k[7]);
  } else {
    // the normalised keys the caller keeps
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = 8 * (part - 6) + i;
      if (t < n) p.keys[(static_cast<int64_t>(h) * p.T + t0 + t) * kD + ch] = ks[t * kRow + ch];
    }
  }
}

// ------------------------------------------------------------------ state recurrence
// Four waves share a 128 x 16 state slice, wave w rows 32 w .. 32 w + 31: register (m, e) of lane l is row
// 32 w + 16 m + 4 (l >> 4) + e, column l & 15, the result layout of the fp32 MFMA and, with the reduction taken in that
// order of rows, also its B operand, so the state never leaves registers between chunks.  A 16-column slice is the
// narrowest MFMA tile: 256 workgroups at 32 heads, one per CU.  T = 16: 5 us; T = 600 (38 chunks in series, 80 MB of
// states written): 48 us, against about 4000 us for the same chunks as batched library products.
__global__ __launch_bounds__(256) void gdn_state_kernel(GdnParams p) {
  __shared__ f32x4 part[2][2][4][64];  // [buffer][W S, Q~ S][wave][lane]
  const int h = blockIdx.x % p.Hv, slice = blockIdx.x / p.Hv;  // a head's slices share an XCD when Hv % 8 == 0
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, kq = lane >> 4;
  const int col = slice * 16 + lr;
  const int64_t head = static_cast<int64_t>(h) * kD * kD;
  f32x4 s[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int e = 0; e < 4; ++e) s[m][e] = p.state[head + (32 * wave + 16 * m + 4 * kq + e) * kD + col];

  struct Ops {
    f32x4 w[2], q[2], k[2], u0, pm;
    float decay;
  };
  auto load = [&](int c, Ops& o) {
    const int64_t row = static_cast<int64_t>(h) * p.chunks + c;
    const int64_t off = row * kChunk * kD;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int k0 = 32 * wave + 16 * m;
      o.w[m] = *reinterpret_cast<const f32x4*>(p.w + off + lr * kD + k0 + 4 * kq);
      o.q[m] = *reinterpret_cast<const f32x4*>(p.qt + off + lr * kD + k0 + 4 * kq);
      o.k[m] = *reinterpret_cast<const f32x4*>(p.kt + off + (k0 + lr) * kChunk + 4 * kq);
    }
    o.u0 = *reinterpret_cast<const f32x4*>(p.u0 + off + col * kChunk + 4 * kq);
    o.pm = *reinterpret_cast<const f32x4*>(p.pmat + row * kChunk * kChunk + lr * kChunk + 4 * kq);
    o.decay = p.decay[row];
  };
  // one chunk: `cur` holds its operands, `dst` receives those of the chunk after next (a chunk's own work is shorter
  // than a round trip to the last-level cache).  Three operand sets take turns in an unrolled loop: moving one set
  // to another would wait for its loads.
  const int last = p.chunks - 1;
  auto step = [&](int c, const Ops& cur, Ops& dst) {
    load(min(c + 2, last), dst);
    f32x4 ws{0.f, 0.f, 0.f, 0.f}, qs{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ws = mfma16x16x4f32(cur.w[m][e], s[m][e], ws);
        qs = mfma16x16x4f32(cur.q[m][e], s[m][e], qs);
      }
    part[c & 1][0][wave][lane] = ws;
    part[c & 1][1][wave][lane] = qs;
    lds_barrier();  // two buffers: a wave writes one again only past the next chunk's barrier
    ws = (part[c & 1][0][0][lane] + part[c & 1][0][1][lane]) + (part[c & 1][0][2][lane] + part[c & 1][0][3][lane]);
    const f32x4 u = cur.u0 - ws;  // rows t = 4 kq + e, column lr
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      s[m] *= cur.decay;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[m] = mfma16x16x4f32(cur.k[m][e], u[e], s[m]);
    }
    if (wave == (c & 3)) {  // one wave per chunk adds P U and writes the block's outputs
      qs = (part[c & 1][1][0][lane] + part[c & 1][1][1][lane]) + (part[c & 1][1][2][lane] + part[c & 1][1][3][lane]);
#pragma unroll
      for (int e = 0; e < 4; ++e) qs = mfma16x16x4f32(cur.pm[e], u[e], qs);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = c * kChunk + 4 * kq + e;
        if (t < p.T) {
          const int64_t o = (static_cast<int64_t>(h) * p.T + t) * kD + col;
          p.core[o] = qs[e];
          p.u[o] = u[e];
        }
      }
    }
    float* so = p.states + static_cast<int64_t>(c) * p.Hv * kD * kD + head;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) so[(32 * wave + 16 * m + 4 * kq + e) * kD + col] = s[m][e];
  };
  Ops o0, o1, o2;
  load(0, o0);
  load(min(1, last), o1);
#pragma unroll 1
  for (int c = 0;; c += 3) {
    step(c, o0, o2);
    if (c + 1 > last) break;
    step(c + 1, o1, o0);
    if (c + 2 > last) break;
    step(c + 2, o2, o1);
    if (c + 3 > last) break;
  }
}

// Per-head RMS norm of the core output, times the norm weight and SiLU(z), as the bf16 rows of out_proj:
// one wave per (token, value head), two columns a lane.
__global__ __launch_bounds__(256) void gdn_gate_kernel(GdnParams p) {
  const int idx = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (idx >= p.T * p.Hv) return;
  const int t = idx / p.Hv, h = idx - t * p.Hv;
  const float2 x = *reinterpret_cast<const float2*>(p.core + (static_cast<int64_t>(h) * p.T + t) * kD + 2 * lane);
  const uint32_t z = *reinterpret_cast<const uint32_t*>(p.proj + static_cast<int64_t>(t) * p.ldp +
                                                        (2 * p.Hk + p.Hv + h) * kD + 2 * lane);
  const float2 g = *reinterpret_cast<const float2*>(p.norm + 2 * lane);
  const float inv = rsqrtf(wave_sum(x.x * x.x + x.y * x.y) / kD + p.eps);
  ushort2 o;
  o.x = f32_to_bf16(x.x * inv * g.x * silu_f32(__uint_as_float(z << 16)));
  o.y = f32_to_bf16(x.y * inv * g.y * silu_f32(__uint_as_float(z & 0xFFFF0000u)));
  *reinterpret_cast<ushort2*>(p.gated + (static_cast<int64_t>(t) * p.Hv + h) * kD + 2 * lane) = o;
}

// State after the first j tokens of a chunk: e^{G_j} S0 + sum_{s < j} e^{G_j - G_s} k_s u_s^T, one workgroup per
// (head, 16 state rows), a thread one column of 8 of the rows; and, in the workgroups past those, the conv history at
// the accepted token: three columns of the window.  Every load is issued before the first use (one round trip).
__global__ __launch_bounds__(256) void gdn_commit_kernel(const float* state, const float* keys, const float* u,
                                                         const float* cum, int64_t row_stride, int64_t cum_stride,
                                                         int heads, int j, float* out, const uint16_t* window,
                                                         int64_t pitch, int first, int channels, uint16_t* hist) {
  const int tid = threadIdx.x;
  if (blockIdx.x >= static_cast<unsigned>(heads * (kD / 16))) {
    const int i = (blockIdx.x - heads * (kD / 16)) * 256 + tid;
    if (i < channels * (kTaps - 1)) hist[i] = window[i / (kTaps - 1) * pitch + first + i % (kTaps - 1)];
    return;
  }
  __shared__ float kd[kChunk][16];
  const int h = blockIdx.x / (kD / 16), rb = blockIdx.x % (kD / 16) * 16;
  const int r0 = tid >> 7 << 3, col = tid & 127;
  const float* ur = u + h * row_stride + col;
  const float last = cum[h * cum_stride + j - 1];
  const int64_t o = (static_cast<int64_t>(h) * kD + rb + r0) * kD + col;
  float acc[8], us[kChunk];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = state[o + i * kD];
#pragma unroll
  for (int s = 0; s < kChunk; ++s) us[s] = ur[min(s, j - 1) * kD];
  {
    const int s = min(tid >> 4, j - 1);
    const float k = keys[h * row_stride + s * kD + rb + (tid & 15)];
    kd[tid >> 4][tid & 15] = tid >> 4 < j ? k * expf(last - cum[h * cum_stride + s]) : 0.f;
  }
  __syncthreads();
  const float dec = expf(last);
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] *= dec;
#pragma unroll
  for (int s = 0; s < kChunk; ++s)
    if (s < j)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] += kd[s][r0 + i] * us[s];
#pragma unroll
  for (int i = 0; i < 8; ++i) out[o + i * kD] = acc[i];
}

}  // namespace

void launch_add_norm(const float* hidden, const uint16_t* mixed, const float* w, float eps, int T, int H, float* mid,
                     uint16_t* normed, hipStream_t stream) {
  hipLaunchKernelGGL(add_norm_kernel<false>, dim3(T), dim3(512), 0, stream, hidden, mixed, w, eps, H, mid, normed);
}

void launch_norm_f32(const float* hidden, const float* w, float eps, int T, int H, float* normed, hipStream_t stream) {
  constexpr int kRows = 1 << 22;  // a launch stays below 2^32 work-items
  for (int t = 0; t < T; t += kRows)
    hipLaunchKernelGGL(add_norm_kernel<true>, dim3(min(kRows, T - t)), dim3(512), 0, stream, hidden + static_cast<int64_t>(t) * H,
                       nullptr, w, eps, H, nullptr, normed + static_cast<int64_t>(t) * H);
}

void launch_gdn(const GdnParams& p, hipStream_t stream) {
  hipLaunchKernelGGL(gdn_chunk_kernel, dim3(p.Hk, p.Hv / p.Hk, p.chunks), dim3(1024), 0, stream, p);
  hipLaunchKernelGGL(gdn_state_kernel, dim3(p.Hv * (kD / 16)), dim3(256), 0, stream, p);
  hipLaunchKernelGGL(gdn_gate_kernel, dim3((p.T * p.Hv + 3) / 4), dim3(256), 0, stream, p);
}

void launch_gdn_commit(const float* state, const float* keys, const float* u, const float* cum, int64_t row_stride,
                       int64_t cum_stride, int heads, int j, float* out, const uint16_t* window, int64_t pitch, int first,
                       int channels, uint16_t* hist, hipStream_t stream) {
  const int blocks = heads * (kD / 16) + (channels * (kTaps - 1) + 255) / 256;
  hipLaunchKernelGGL(gdn_commit_kernel, dim3(blocks), dim3(256), 0, stream, state, keys, u, cum, row_stride, cum_stride,
                     heads, j, out, window, pitch, first, channels, hist);
}

}  // namespace dflash
