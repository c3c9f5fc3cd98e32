// Attention mixer kernels: the arithmetic of a full-attention layer around its int4 projections
// (model/qwen35_moe_dflash/fused/model.py:265-294): per-head Q/K norms, partial rotary, cache append, causal
// grouped-query attention in fp32 over a bf16 cache, output gate.
//
// The products run on the bf16 matrix cores without rounding an fp32 operand to 16 bits: a query or a probability
// is the sum of three bf16 parts (8 + 8 + 8 significant bits: exact), each part times a bf16 cache value is exact in
// fp32, and the three products accumulate in fp32.  Three 16x16x32 products cost a fifth of the fp32 matrix
// instructions for the same block.
//   attn_prep_kernel     one wave per (token, head): norm, rotary, query parts; K and V rows into the cache
//   attn_split_kernel    one workgroup per (16 query rows of a KV head, split of the keys); its four waves take 32 keys
//                        at a time each and merge their softmax states through LDS
//   attn_combine_kernel  splits merged, times sigmoid(gate), as the bf16 rows of the output projection
// Rows of a KV head are ordered token by token (row = token * group + head in group), so a causal row tile
// spans few tokens.
//
// Bound by latency at verify sizes (T = 16 behind 4001 keys, 16 heads over 2 KV heads of 256: 8.4 MB of cache, 1.7 us at
// the copy rate): prep 4.1, split 15.8 (19.0 with the row tiles of a split spread over the XCDs), combine 5.3 (9.8 with the
// splits read one after the other), in place of 60 library launches (250 us).  Against 64
// bits the attention output is 4e-7 to 7e-7 off (fp32 library products 4e-7 to 1.8e-6).
//
// NaN and infinities as in a softmax over the visible keys: a NaN score makes its row NaN, a score of -inf has weight 0.
#include <algorithm>

#include "kernels.h"

namespace dflash {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Two fp32 values as bf16 pairs hi + mid + lo, exact for finite values of normal size (each part takes
// the next eight significant bits; the remainders are exact in fp32).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return f32_to_bf16(a) | (static_cast<uint32_t>(f32_to_bf16(b)) << 16);
}
__device__ __forceinline__ void split3(float a, float b, uint32_t (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    part[i] = pack_bf16(a, b);
    a -= __uint_as_float(part[i] << 16);
    b -= __uint_as_float(part[i] & 0xFFFF0000u);
  }
}

// ------------------------------------------------------------------ norms, rotary, cache rows
// D / 64 neighbouring features a lane; feature i < half rotates with i + half, which lane + half * 64 / D holds.
template <int D>
__global__ __launch_bounds__(256) void attn_prep_kernel(AttnParams p) {
  constexpr int F = D / 64;
  const int idx = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int per = p.heads + 2 * p.kv;
  if (idx >= p.T * per) return;
  const int t = idx / per, j = idx - t * per;
  const bool is_q = j < p.heads, is_k = !is_q && j < p.heads + p.kv;
  const int head = is_q ? j : is_k ? j - p.heads : j - p.heads - p.kv;
  const uint16_t* src = p.proj + static_cast<int64_t>(t) * p.ldp +
                        (is_q ? head * 2 * D : 2 * p.heads * D + (is_k ? 0 : p.kv * D) + head * D) + lane * F;
  const int64_t cache = (static_cast<int64_t>(head) * p.capacity + p.position + t) * D + lane * F;
  uint16_t x[F];
#pragma unroll
  for (int i = 0; i < F; ++i) x[i] = src[i];
  if (!is_q && !is_k) {
#pragma unroll
    for (int i = 0; i < F; ++i) p.values[cache + i] = x[i];
    return;
  }
  const float* w = (is_q ? p.q_norm : p.k_norm) + lane * F;
  float v[F], sum = 0.f;
#pragma unroll
  for (int i = 0; i < F; ++i) {
    v[i] = bf16_to_f32(x[i]);
    sum += v[i] * v[i];
  }
  const float inv = rsqrtf(wave_sum(sum) / D + p.eps);
  const int half_lanes = p.rotary_half / F;
  const bool first = lane < half_lanes, rot = lane < 2 * half_lanes;
  const int partner = rot ? (first ? lane + half_lanes : lane - half_lanes) : lane;
#pragma unroll
  for (int i = 0; i < F; ++i) v[i] = v[i] * inv * (w[i] + 1.0f);
  float other[F];
#pragma unroll
  for (int i = 0; i < F; ++i) other[i] = __shfl(v[i], partner, 64);
  if (rot) {
    const float pos = static_cast<float>(p.position + t);
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const float angle = pos * p.inv_freq[(first ? lane : lane - half_lanes) * F + i];
      const float c = cosf(angle), s = sinf(angle);
      v[i] = v[i] * c + (first ? -other[i] : other[i]) * s;
    }
  }
  if (is_k) {
#pragma unroll
    for (int i = 0; i < F; ++i) p.keys[cache + i] = f32_to_bf16(v[i]);
    return;
  }
  const int group = p.heads / p.kv;
  const int64_t row = (static_cast<int64_t>(head / group) * p.T + t) * group + head % group;
  const int64_t plane = static_cast<int64_t>(p.heads) * p.T * D;
#pragma unroll
  for (int i = 0; i < F; i += 2) {
    uint32_t part[3];
    split3(v[i] * p.scale, v[i + 1] * p.scale, part);
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint32_t*>(p.q + q * plane + row * D + lane * F + i) = part[q];
  }
}

// ------------------------------------------------------------------ one split of the keys
// Scores transposed, S^T = K Q^T: lane l holds query row l & 15 and keys 4 (l >> 4) + e of each of two key tiles,
// which, with those eight keys as the reduction's octet l >> 4, is the B operand of O^T = V^T P^T as it stands.  The A
// operand then needs eight keys of one dim per lane: a lane loads D / 16 neighbouring dims of its eight keys
// (512-byte rows, dim 16 (l & 15) + c of tile c) and pairs halves in registers, so V needs no transpose.
template <int D>
__global__ __launch_bounds__(256, 1) void attn_split_kernel(AttnParams p) {
  constexpr int NC = D / 16, KS = D / 32, VL = NC / 8;  // dims a lane, 32-dim steps, 16-byte loads a V row
  constexpr int kPitch = D + 4;
  __shared__ __align__(16) float osum[4][16][kPitch];
  __shared__ float mx[4][16], ls[4][16];
  // splits fastest: with a multiple of eight of them (workgroups go round robin over the XCDs) a split's keys and values
  // pass through one XCD's L2 only, for all row tiles
  const int tile = blockIdx.x / p.splits, split = blockIdx.x - tile * p.splits, kvh = blockIdx.z;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane & 15, kq = lane >> 4;
  const int group = p.heads / p.kv, rows = p.T * group;
  const int r = min(tile * 16 + lr, rows - 1);                     // this lane's query row
  const int visible = p.position + r / group + 1;                  // keys it sees
  const int last = min(tile * 16 + 15, rows - 1) / group;          // last token of the tile
  const int n = p.position + last + 1;                             // keys any row of the tile sees
  const int k0 = split * p.split_keys, k1 = min(k0 + p.split_keys, n);
  const int64_t out_row = (static_cast<int64_t>(split) * p.kv + kvh) * rows + tile * 16;
  const int nrows = min(16, rows - tile * 16);
  if (k0 >= k1) {  // the whole split lies past the tile's last key
    if (tid < nrows) p.ml[out_row + tid] = make_float2(-__builtin_inff(), 0.f);
    return;
  }
  const int64_t base = static_cast<int64_t>(kvh) * p.capacity * D;
  const uint16_t* keys = p.keys + base;
  const uint16_t* vals = p.values + base;
  u32x4 q[3][KS];
  {
    const int64_t plane = static_cast<int64_t>(p.heads) * p.T * D;
    const uint16_t* qr = p.q + (static_cast<int64_t>(kvh) * rows + r) * D + 8 * kq;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int s = 0; s < KS; ++s) q[i][s] = *reinterpret_cast<const u32x4*>(qr + i * plane + 32 * s);
  }
  f32x4 o[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -__builtin_inff(), l = 0.f;

  for (int j0 = k0 + 32 * wave; j0 < k1; j0 += 128) {
    u32x4 kf[2][KS], vf[8][VL];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint16_t* kr = keys + static_cast<int64_t>(min(j0 + 16 * b + lr, n - 1)) * D + 8 * kq;
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[b][s] = *reinterpret_cast<const u32x4*>(kr + 32 * s);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = min(j0 + 16 * (i >> 2) + 4 * kq + (i & 3), n - 1);
#pragma unroll
      for (int h = 0; h < VL; ++h)
        vf[i][h] = *reinterpret_cast<const u32x4*>(vals + static_cast<int64_t>(key) * D + NC * lr + 8 * h);
    }
    float s8[8];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 acc[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          acc[i] = mfma16x16x32(__builtin_bit_cast(uint4, kf[b][s]), __builtin_bit_cast(uint4, q[i][s]), acc[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = j0 + 16 * b + 4 * kq + e;
        // with an infinity in the key the leading part alone has the score (an infinity times a part of 0 or of the other
        // sign would make it NaN)
        const float score = __builtin_fabsf(acc[0][e]) < __builtin_inff() ? acc[0][e] + (acc[1][e] + acc[2][e]) : acc[0][e];
        s8[4 * b + e] = key < visible && key < k1 ? score : -__builtin_inff();
      }
    }
    float mc = fmaxf(fmaxf(fmaxf(s8[0], s8[1]), fmaxf(s8[2], s8[3])), fmaxf(fmaxf(s8[4], s8[5]), fmaxf(s8[6], s8[7])));
    mc = fmaxf(mc, __shfl_xor(mc, 16, 64));
    mc = fmaxf(mc, __shfl_xor(mc, 32, 64));
    const float mn = fmaxf(m, mc);
    // a row that has seen no key yet keeps weight 0 (its maximum is -inf, as is every score); a NaN score, which the
    // maximum skips, makes l and o NaN, and so they stay
    const float corr = mn == -__builtin_inff() ? 1.f : expf(m - mn);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      s8[i] = s8[i] == -__builtin_inff() ? 0.f : expf(s8[i] - mn);
      sum += s8[i];
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l = l * corr + sum;
    m = mn;
#pragma unroll
    for (int c = 0; c < NC; ++c) o[c] *= corr;
    u32x4 pf[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t part[3];
      split3(s8[2 * i], s8[2 * i + 1], part);
#pragma unroll
      for (int b = 0; b < 3; ++b) pf[b][i] = part[b];
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      u32x4 a;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[i] = __builtin_amdgcn_perm(vf[2 * i + 1][c >> 3][(c >> 1) & 3], vf[2 * i][c >> 3][(c >> 1) & 3],
                                     c & 1 ? 0x07060302u : 0x05040100u);
#pragma unroll
      for (int b = 2; b >= 0; --b)
        o[c] = mfma16x16x32(__builtin_bit_cast(uint4, a), __builtin_bit_cast(uint4, pf[b]), o[c]);
    }
  }
  // merge the four waves: each scales its sums to the workgroup's maximum (a wave without keys has sums of 0, not
  // only a maximum of -inf: with scores that are all NaN its sums are NaN and stay in)
  if (kq == 0) {
    mx[wave][lr] = m;
    ls[wave][lr] = l;
  }
  __syncthreads();
  const float M = fmaxf(fmaxf(mx[0][lr], mx[1][lr]), fmaxf(mx[2][lr], mx[3][lr]));
  const float f = m == -__builtin_inff() ? 0.f : expf(m - M);
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int c = 0; c < NC; c += 4)
      *reinterpret_cast<f32x4*>(&osum[wave][lr][NC * (4 * kq + e) + c]) =
          f32x4{o[c][e] * f, o[c + 1][e] * f, o[c + 2][e] * f, o[c + 3][e] * f};
  __syncthreads();
  for (int i = tid; i < nrows * (D / 4); i += 256) {
    const int row = i / (D / 4), c = i % (D / 4) * 4;
    f32x4 v = *reinterpret_cast<const f32x4*>(&osum[0][row][c]);
#pragma unroll
    for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&osum[w][row][c]);
    *reinterpret_cast<f32x4*>(p.part + (out_row + row) * D + c) = v;
  }
  if (tid < nrows) {
    const float mm = fmaxf(fmaxf(mx[0][tid], mx[1][tid]), fmaxf(mx[2][tid], mx[3][tid]));
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += mx[w][tid] == -__builtin_inff() ? ls[w][tid] * 0.f : ls[w][tid] * expf(mx[w][tid] - mm);
    p.ml[out_row + tid] = make_float2(mm, sum);
  }
}

// One workgroup per (token, head), one dim a thread.  Each wave reads every split's maximum and sum at once, a split a
// lane (one after the other they were most of this kernel's time), and the partial rows follow eight at a time.  Splits
// that hold no key of the row (sum 0, partial row maybe never written) are left out.
constexpr int kMaxSplits = 256;
template <int D>
__global__ __launch_bounds__(D) void attn_combine_kernel(AttnParams p) {
  __shared__ float fs[kMaxSplits];
  const int t = blockIdx.x / p.heads, head = blockIdx.x - t * p.heads, c = threadIdx.x, lane = threadIdx.x & 63;
  const int group = p.heads / p.kv, rows = p.T * group;
  const int64_t row = static_cast<int64_t>(head / group) * rows + t * group + head % group;
  const int64_t stride = static_cast<int64_t>(p.kv) * rows;
  const float gate = bf16_to_f32(p.proj[static_cast<int64_t>(t) * p.ldp + head * 2 * D + D + c]);
  constexpr int kPer = kMaxSplits / 64;
  float2 v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int s = lane + 64 * i;
    v[i] = s < p.splits ? p.ml[s * stride + row] : make_float2(-__builtin_inff(), 0.f);
  }
  float M = fmaxf(fmaxf(v[0].x, v[1].x), fmaxf(v[2].x, v[3].x));
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  float l = 0.f;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool used = v[i].y != 0.f;  // a NaN sum (NaN scores) is used and makes the row NaN
    const float f = used ? expf(v[i].x - M) : -1.f;
    if (used) l += v[i].y * f;
    if (threadIdx.x < 64) fs[lane + 64 * i] = f;
  }
  l = wave_sum(l);
  __syncthreads();
  float o = 0.f;
  for (int s0 = 0; s0 < p.splits; s0 += 8) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = p.part[(min(s0 + i, p.splits - 1) * stride + row) * D + c];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (s0 + i < p.splits && fs[s0 + i] >= 0.f) o += x[i] * fs[s0 + i];
  }
  p.out[(static_cast<int64_t>(t) * p.heads + head) * D + c] = f32_to_bf16(o / l / (1.0f + expf(-gate)));
}

}  // namespace

// Splits of the keys: enough workgroups for every CU at small blocks, at least 128 keys (32 a wave) each.  More splits
// only add partial rows (splits * rows * D * 4 bytes, written and read again).
int attn_splits(int rows, int kv, int keys, int cus) {
  const int tiles = kv * ((rows + 15) / 16);
  return std::max(1, std::min({(keys + 127) / 128, cus / tiles, kMaxSplits}));
}
int64_t attn_partial_rows(int rows, int kv, int cus) {
  // splits <= max(1, cus / tiles), and a tile holds 16 rows
  return std::max<int64_t>(static_cast<int64_t>(rows) * kv, static_cast<int64_t>(cus) * 16);
}

template <int D>
static void launch_attn(const AttnParams& p, hipStream_t stream) {
  const int rows = p.T * (p.heads / p.kv);
  hipLaunchKernelGGL(attn_prep_kernel<D>, dim3((p.T * (p.heads + 2 * p.kv) + 3) / 4), dim3(256), 0, stream, p);
  hipLaunchKernelGGL(attn_split_kernel<D>, dim3((rows + 15) / 16 * p.splits, 1, p.kv), dim3(256), 0, stream, p);
  hipLaunchKernelGGL(attn_combine_kernel<D>, dim3(p.T * p.heads), dim3(D), 0, stream, p);
}
void launch_attention(int head_dim, const AttnParams& p, hipStream_t stream) {
  if (head_dim == 256) launch_attn<256>(p, stream);
  else launch_attn<128>(p, stream);
}

}  // namespace dflash
