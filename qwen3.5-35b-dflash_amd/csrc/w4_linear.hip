// W4A16 linear for more rows than a verify block holds (a prompt, or a chunk of one): any packed matrix the
// library takes (K a multiple of 128, groups of 128 or 256, bf16 or fp32 scales, either layout).
//
// A prep launch writes the activations in MFMA fragment order (one kilobyte per 32 rows x 16 k) with -24 times each
// row's sum per 128-column k-block; the weights are dequantised to bf16 as 24 + q, exact (dequant24), and a k-block's
// sums start at the offset term.  Two forms:
//
//   w4_linear_tile_kernel   a workgroup of four waves takes 64 rows x 256 columns, a wave all rows x 64 columns, so a
//       weight is dequantised once per tile.  Activations reach LDS by direct-to-LDS loads, double buffered, one
//       barrier per k-block; weights go straight into registers a k-block ahead.  168 registers and 33 KB of LDS:
//       three workgroups share a CU, one computing while another waits at its barrier (against two: 2048 x 12288 x
//       8192 441 -> 352 us, 2048 x 12352 x 2048 118 -> 113 us each alone; 96-row tiles at two a CU 398 and 121 us).
//       The MFMAs accumulate into u, the running sum in units of the current group's scale: u is rescaled by
//       s_prev / s at each k-block in the FMA that adds the offset term, which saves a second accumulator set.
//       A wave that meets a scale which is no unit (zero, tiny, huge, not finite) takes its columns once more without.
//       Bound by power: in the k-loop a workgroup takes 1509 cycles a k-block where the matrix core needs 1024, at a clock
//       that falls from 2.4 to about 1.6 GHz.  2048 x 12352 x 2048 with the prep launch: 106 to 109 us among other calls,
//       0.95 to 0.98 PFLOP/s (bf16 library product of that size 102 us; the 16-column streaming kernel that served these
//       sizes before 267 us).  A zero scale in one column of every 64, so every wave twice: 269 us.
//   w4_linear_split_kernel  for outputs of few tiles: a workgroup takes 32 rows x 64 columns, its four waves every fourth
//       k-block each, operands straight into MFMA fragment registers, the four partial sums added in LDS in wave order.
//       Bound by the latency of its loads: 333 x 2048 x 4096 in 23.0 us with the prep launch (kernel trace: 17.8 + 6.2),
//       495 us on the per-wave kernel before.
//
// The line between them: tile when its tiles fill at least 5/8 of the CUs.  Measured, split / tile, us: 80 tiles 17.7 /
// 22.9 (300 x 4096 x 2048) and 33.1 / 50.5 (600 x 2048 x 4096, portable); 160 tiles 25.2 / 25.2 (600 x 4096 x 2048); 196
// tiles 26.1 / 24.1 (200 x 12352 x 2048); 256 tiles 34.1 / 26.7 (1024 x 4096 x 2048).
//
// Against 64 bits the fp32 sums are 1.0e-7 (split) and 2.1e-7 to 2.6e-7 (tile) off, relative (1.0e-6 to 2.8e-6
// with the 136 + q weights of the kernels before).
//
// Reference: OriginalQuantizedWeights.linear, fused/quantization.py:154-165; y = x (q s)^T.
#include "kernels.h"

namespace dflash {
namespace {

constexpr uint32_t kMinus24Pair = 0xC1C0C1C0u;  // bf16 pair (-24, -24)

// 8 signed nibbles -> 4 bf16 pairs (k0,k4) (k1,k5) (k2,k6) (k3,k7) holding 24 + q: the nibble with its sign bit
// flipped is q + 8, placed in mantissa bits 3..6 of 16.0
__device__ __forceinline__ uint32_t nibbles24(uint32_t w) {
  return __builtin_amdgcn_bitop3_b32(w, 0x00780078u, 0x41C041C0u, 0x6A);  // (w & mask) ^ bits
}
__device__ __forceinline__ uint4 dequant24(uint32_t w) {
  return make_uint4(nibbles24(w << 3), nibbles24(w >> 1), nibbles24(w >> 5), nibbles24(w >> 9));
}

// natural bf16 pairs (k0,k1)(k2,k3)(k4,k5)(k6,k7) -> (k0,k4)(k1,k5)(k2,k6)(k3,k7)
__device__ __forceinline__ uint4 octet_pairs(uint4 v) {
  return make_uint4(__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                    __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u));
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 zero16() { return f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}; }
// lane l supplies row (column) l & 31 and k-octet l >> 5 of each operand; register i of the result is row
// 8 (i / 4) + 4 (l >> 5) + i % 4, column l & 31.  A 32x32x16 product takes the matrix core as long per flop as a
// 16x16x32 one but half the issue slots: six VALU operations run beside each, against two beside a 16x16x32 one.
__device__ __forceinline__ f32x16 mfma32(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t word(const uint4& w, int j) { return j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w; }

// The workgroup's tile (row tile, column tile), or false past the last one.  The list runs in bands of kBand row
// tiles, rows fastest inside a band, and each XCD (workgroups go round robin over the eight) takes one contiguous range
// of it: the workgroups that run at a time under one L2 form a block of about 8 x 8 tiles, so each
// operand is read from memory once for eight of them.
constexpr int kBand = 8;
__device__ __forceinline__ bool find_tile(int rows, int cols, int& row, int& col) {
  const int total = rows * cols, per = (total + 7) >> 3;
  const int i = static_cast<int>(blockIdx.x) >> 3, t = (blockIdx.x & 7) * per + i;
  if (i >= per || t >= total) return false;
  const int band = t / (kBand * cols), first = band * kBand, height = min(kBand, rows - first);
  const int rest = t - first * cols;
  col = rest / height;
  row = first + rest - col * height;
  return true;
}

// ------------------------------------------------------------------ activations in fragment order
// Fragment s = 4 jj + o of a k-block (32 rows x 16 k): lane (h, r) holds octet o of row r's 32-column quarter 2 jj + h,
// the order in which a lane's 16 weight bytes hold theirs; rows past M are zero.  neg: -24 x each row's sum.  One wave
// per 32 rows and k-block.
__global__ __launch_bounds__(256) void w4_linear_prep_kernel(LinearParams p) {
  const int nkb = p.K >> 7, tiles = (p.M + 31) >> 5;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (idx >= static_cast<int64_t>(tiles) * nkb) return;
  const int t = static_cast<int>(idx / nkb), kb = static_cast<int>(idx - static_cast<int64_t>(t) * nkb);
  const int lane = lane_id(), r = lane & 31, h = lane >> 5;
  const int row = t * 32 + r;
  const uint4* src = reinterpret_cast<const uint4*>(p.x + static_cast<int64_t>(min(row, p.M - 1)) * p.K + kb * 128 + h * 32);
  uint4 v[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) v[s] = src[(s >> 2) * 8 + (s & 3)];
  uint4* dst = reinterpret_cast<uint4*>(p.xf) + idx * 512 + lane;
  const uint4 m24 = make_uint4(kMinus24Pair, kMinus24Pair, kMinus24Pair, kMinus24Pair);
  f32x16 neg = zero16();
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const uint4 o = row < p.M ? octet_pairs(v[s]) : make_uint4(0, 0, 0, 0);
    dst[s * 64] = o;
    neg = mfma32(o, m24, neg);
  }
  if (r == 0)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(p.neg + idx * 32 + 8 * g + 4 * h) = f32x4{neg[4 * g], neg[4 * g + 1], neg[4 * g + 2], neg[4 * g + 3]};
}

// This lane's operands of a wave's two 32-column weight fragments: 16 bytes per 32-column quarter pair (quarter
// 2 jj + h of row r) and the group scale of column r.  `first`: the matrix row the resources start at.
template <typename ScaleT>
struct Weights {
  buf_rsrc wrs, srs;
  uint32_t woff[2], soff[2], wkb, sg, jj;
  int gshift;
  __device__ __forceinline__ Weights(const LinearParams& p, int first, int rows, int c0, int c1) {
    const int lane = lane_id(), r = lane & 31, h = lane >> 5, ng = p.K / p.G;
    const uint32_t rb = static_cast<uint32_t>(p.K) >> 1;
    wrs = make_rsrc(p.w + static_cast<int64_t>(first) * rb, static_cast<uint32_t>(rows) * rb);
    srs = make_rsrc(static_cast<const char*>(p.s) + static_cast<int64_t>(first) * ng * sizeof(ScaleT),
                    static_cast<uint32_t>(rows * ng) * static_cast<uint32_t>(sizeof(ScaleT)));
    gshift = p.G == 256 ? 1 : 0;
    wkb = p.tiled ? 1024u : 64u;
    jj = p.tiled ? 512u : 32u;
    sg = (p.tiled ? 16u : 1u) * sizeof(ScaleT);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      const int r0 = f ? c1 : c0;
      woff[f] = p.tiled ? static_cast<uint32_t>(r0 + (r & 16)) * rb + h * 256u + (r & 15) * 16u
                        : static_cast<uint32_t>(r0 + r) * rb + h * 16u;
      soff[f] = (p.tiled ? static_cast<uint32_t>((r0 + (r & 16)) * ng + (r & 15)) : static_cast<uint32_t>((r0 + r) * ng)) *
                sizeof(ScaleT);
    }
  }
  __device__ __forceinline__ void load(int kb, uint4 (&w)[2][2], uint32_t (&s)[2]) const {
    const int wo = __builtin_amdgcn_readfirstlane(static_cast<int>(kb * wkb));
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int q = 0; q < 2; ++q) w[f][q] = buf_load16(wrs, woff[f], wo + q * jj);
    load_scales(kb, s);
  }
  __device__ __forceinline__ void load_scales(int kb, uint32_t (&s)[2]) const {
    const int so = __builtin_amdgcn_readfirstlane(static_cast<int>((kb >> gshift) * sg));
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      s[f] = sizeof(ScaleT) == 4 ? __builtin_amdgcn_raw_buffer_load_b32(srs, static_cast<int>(soff[f]), so, 0)
                                 : static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(srs, static_cast<int>(soff[f]), so, 0));
    }
  }
};

// ------------------------------------------------------------------ tiles
constexpr int kSub = 2;  // 32-row subtiles of a tile
// Scales a running sum may be in units of: the sum of a column whose scales lie in between stays finite in any of their
// units while its products' sum is below 2^95.
constexpr float kMinUnit = 0x1p-24f, kMaxUnit = 0x1p8f;

typedef __attribute__((address_space(3))) void* lds_ptr;
// 16 bytes a lane straight into LDS (lane l at dst + 16 l)
__device__ __forceinline__ void dma16(buf_rsrc r, void* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)dst, 16, static_cast<int>(voff), static_cast<int>(soff), 0, 0);
}

template <int N>
struct Int {
  static constexpr int value = N;
};

constexpr int kValuOps = 0x002, kMfmaOps = 0x008, kDsReads = 0x100;  // sched_group_barrier masks

template <typename ScaleT>
__global__ __launch_bounds__(256, 3) void w4_linear_tile_kernel(LinearParams p) {
  // a stage is an array of its own: the compiler makes reads of an array wait for the loads headed for it
  __shared__ uint4 a0[kSub * 512], a1[kSub * 512];
  __shared__ float n0[256], n1[256];
  const int N = p.N, nkb = p.K >> 7;
  const int tiles32 = (p.M + 31) >> 5, mt_count = (tiles32 + kSub - 1) / kSub, nt_count = (N + 255) >> 8;
  int mt, nt;
  if (!find_tile(mt_count, nt_count, mt, nt)) return;
  const int t0 = mt * kSub;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = lane_id(), r = lane & 31, h = lane >> 5;
  const int col0 = nt * 256 + wave * 64;

  // activations and offset terms of this tile's rows (subtiles past the end repeat the last one)
  const int live = min(kSub, tiles32 - t0);
  const buf_rsrc ars = make_rsrc(p.xf + static_cast<int64_t>(t0) * nkb * 4096, static_cast<uint32_t>(live * nkb) * 8192u);
  const buf_rsrc nrs = make_rsrc(p.neg + static_cast<int64_t>(t0) * nkb * 32, static_cast<uint32_t>(live * nkb) * 128u);
  const uint32_t noff = static_cast<uint32_t>(min((wave * 64 + lane) >> 5, live - 1) * nkb) * 128u + r * 4u;
  // weights and scales from this workgroup's first column on (fragments past N repeat the last one)
  const int base = nt * 256;
  const Weights<ScaleT> weights(p, base, min(256, N - base), min(col0, N - 32) - base, min(col0 + 32, N - 32) - base);

  f32x16 u[kSub][2];
  float s_cur[2], s_last[2], ratio[2];  // the group scale u is in units of, the one before, and their quotient
  bool odd = false;                     // some column of the wave has a scale that is no unit (in all lanes)
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    s_cur[f] = 0.f;
#pragma unroll
    for (int ms = 0; ms < kSub; ++ms) u[ms][f] = zero16();
  }
  uint4 wb[2][2][2];
  uint32_t sb[2][2];
  auto load = [&](int kb, auto stage) {  // past the last k-block it is loaded again, into a stage never read
    constexpr int S = decltype(stage)::value;
    kb = __builtin_amdgcn_readfirstlane(min(kb, nkb - 1));
#pragma unroll
    for (int ms = 0; ms < kSub; ++ms)
#pragma unroll
      for (int q = 0; q < 2; ++q)  // wave w: fragments w and w + 4 of every subtile
        dma16(ars, (S ? a1 : a0) + (ms * 8 + q * 4 + wave) * 64, lane * 16,
              (min(ms, live - 1) * nkb + kb) * 8192 + (q * 4 + wave) * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(nrs, (lds_ptr)((S ? n1 : n0) + wave * 64), 4, static_cast<int>(noff), kb * 128, 0, 0);
    weights.load(kb, wb[S], sb[S]);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto set_scale = [&](int kb, int f, uint32_t bits) {
    const float s = scale_value<ScaleT>(bits), mag = __builtin_fabsf(s);
    odd |= __builtin_amdgcn_ballot_w64(!(mag >= kMinUnit && mag <= kMaxUnit)) != 0;  // NaN too
    ratio[f] = weights.gshift && (kb & 1) ? 1.0f : s_cur[f] * __builtin_amdgcn_rcpf(s);  // the same group still
    s_last[f] = s_cur[f];
    s_cur[f] = s;
  };
  load(0, Int<0>{});
  uint4 a[kSub], b[2];  // fragments of the k-step about to run
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    b[f] = dequant24(wb[0][f][0].x);
    set_scale(0, f, sb[0][f]);
  }

  auto step = [&](int kb, auto stage) {
    constexpr int S = decltype(stage)::value;
    const uint4* ac = (S ? a1 : a0) + lane;
    const float* nc = (S ? n1 : n0) + 4 * h;
    // this k-block's loads are in, of every wave; all waves are done with the other stage
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load(kb + 1, Int<S ^ 1>{});
#pragma unroll
    for (int ms = 0; ms < kSub; ++ms) a[ms] = ac[ms * 512];
    // eight k-steps; while the MFMAs of one run, the next one's fragments are read and dequantised (in the last the next
    // k-block's first)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint4 bn[2];
#pragma unroll
      for (int f = 0; f < 2; ++f) bn[f] = dequant24(j < 7 ? word(wb[S][f][(j + 1) >> 2], (j + 1) & 3) : wb[S ^ 1][f][0].x);
#pragma unroll
      for (int ms = 0; ms < kSub; ++ms) {
        if (j == 0) {
          f32x4 start[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) start[g] = *reinterpret_cast<const f32x4*>(nc + ms * 32 + 8 * g);
#pragma unroll
          for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < 16; ++i) u[ms][f][i] = u[ms][f][i] * ratio[f] + start[i >> 2][i & 3];
        }
#pragma unroll
        for (int f = 0; f < 2; ++f) u[ms][f] = mfma32(a[ms], b[f], u[ms][f]);
        if (j < 7) a[ms] = ac[ms * 512 + (j + 1) * 64];
      }
      if (j == 7)
#pragma unroll
        for (int f = 0; f < 2; ++f) set_scale(kb + 1, f, sb[S ^ 1][f]);
      if (j == 0) {
        __builtin_amdgcn_sched_group_barrier(kDsReads, kSub + 4, 0);
        __builtin_amdgcn_sched_group_barrier(kValuOps, 16, 0);
#pragma unroll
        for (int i = 0; i < 2 * kSub; ++i) {
          __builtin_amdgcn_sched_group_barrier(kMfmaOps, 1, 0);
          if (i & 1) __builtin_amdgcn_sched_group_barrier(kDsReads, 1, 0);
          else __builtin_amdgcn_sched_group_barrier(kDsReads, 4, 0);
          __builtin_amdgcn_sched_group_barrier(kValuOps, 18, 0);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 2 * kSub; ++i) {
          __builtin_amdgcn_sched_group_barrier(kMfmaOps, 1, 0);
          if (j == 7) __builtin_amdgcn_sched_group_barrier(kValuOps, (36 + 2 * kSub - 1) / (2 * kSub), 0);
          else __builtin_amdgcn_sched_group_barrier(kValuOps, (16 + 2 * kSub - 1) / (2 * kSub), 0);
          if (j < 7 && (i & 1)) __builtin_amdgcn_sched_group_barrier(kDsReads, 1, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      b[0] = bn[0];
      b[1] = bn[1];
    }
  };
  for (int kb = 0; kb < nkb; kb += 2) {
    step(kb, Int<0>{});
    if (kb + 1 < nkb) step(kb + 1, Int<1>{});
  }

  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no load may land in LDS once the stages are reused

  if (odd) {
    // once more without units: every k-block's sums times its scale, operands straight from memory (u is free here, so
    // this costs the loop above no registers; a second accumulator there spilled 355 of them)
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      s_last[f] = 1.0f;
#pragma unroll
      for (int ms = 0; ms < kSub; ++ms) u[ms][f] = zero16();
    }
#pragma unroll 1
    for (int kb = 0; kb < nkb; ++kb) {
      uint4 w[2][2];
      uint32_t sc[2];
      weights.load(kb, w, sc);
#pragma unroll
      for (int ms = 0; ms < kSub; ++ms) {
        const int at = min(ms, live - 1) * nkb + kb;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          f32x16 acc;
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 start = __builtin_bit_cast(f32x4, buf_load16(nrs, h * 16, at * 128 + g * 32));
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * g + e] = start[e];
          }
#pragma unroll
          for (int j = 0; j < 8; ++j)
            acc = mfma32(buf_load16(ars, lane * 16, at * 8192 + j * 1024), dequant24(word(w[f][j >> 2], j & 3)), acc);
          u[ms][f] += scale_value<ScaleT>(sc[f]) * acc;
        }
      }
    }
  }

  // lane: rows 32 ms + 8 (i / 4) + 4 h + i % 4 of columns col0 + 32 f + r
  if (p.y_f32) {
    float* y = static_cast<float*>(p.y);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int ms = 0; ms < kSub; ++ms)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int row = (t0 + ms) * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
          if (row < p.M && col0 + f * 32 < N) y[static_cast<int64_t>(row) * N + col0 + f * 32 + r] = u[ms][f][i] * s_last[f];
        }
    return;
  }
  // bf16: through LDS (a wave's own 32 x 64 block at a time, rows 144 bytes apart), so that a store is 16 bytes of
  // a row and eight lanes write 128 contiguous bytes
  constexpr int kPitch = 72;
  __syncthreads();  // every wave is done with the stages
  uint16_t* out = reinterpret_cast<uint16_t*>(wave & 2 ? a1 : a0) + (wave & 1) * 32 * kPitch;
  const int c = col0 + (lane & 7) * 8;
#pragma unroll
  for (int ms = 0; ms < kSub; ++ms) {
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        out[(8 * (i >> 2) + 4 * h + (i & 3)) * kPitch + f * 32 + r] = f32_to_bf16(u[ms][f][i] * s_last[f]);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's block is in
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row = (t0 + ms) * 32 + q * 8 + (lane >> 3);
      const uint4 v = *reinterpret_cast<const uint4*>(out + (q * 8 + (lane >> 3)) * kPitch + (lane & 7) * 8);
      if (row < p.M && c < N) *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.y) + static_cast<int64_t>(row) * N + c) = v;
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // read before the next block is written
    __builtin_amdgcn_wave_barrier();
  }
}

// ------------------------------------------------------------------ k split over the waves
// kStaged (portable banks): a wave's weights of a k-block reach LDS by four direct-to-LDS loads of 16 whole 64-byte row
// pieces each, and lanes read their fragments from there; straight into registers each load would take 32 bytes of 32
// rows (333 x 2048 x 4096 27.6 -> 23.0 us, 600 x 2048 x 4096 39.3 -> 33.1).  Tiled banks lie in fragment order already.
template <typename ScaleT, bool kStaged>
__global__ __launch_bounds__(256, 2) void w4_linear_split_kernel(LinearParams p) {
  __shared__ f32x4 part[4][8][64];  // a wave's eight kilobytes are also its two weight stages, [64 rows][4 pieces] each
  const int N = p.N, nkb = p.K >> 7;
  const int mt_count = (p.M + 31) >> 5, nt_count = (N + 63) >> 6;
  int mt, nt;
  if (!find_tile(mt_count, nt_count, mt, nt)) return;
  const int col0 = nt * 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = lane_id(), r = lane & 31, h = lane >> 5;
  const int rows = min(32, p.M - mt * 32), cols = min(64, N - col0);
  const buf_rsrc xrs = make_rsrc(p.xf + static_cast<int64_t>(mt) * nkb * 4096, static_cast<uint32_t>(nkb) * 8192u);
  const buf_rsrc nrs = make_rsrc(p.neg + static_cast<int64_t>(mt) * nkb * 32, static_cast<uint32_t>(nkb) * 128u);
  const Weights<ScaleT> weights(p, col0, cols, 0, cols - 32);  // a fragment past N repeats the last one

  struct Block {
    uint4 w[2][2], x[8];
    uint32_t s[2];
    f32x4 neg[4];
  };
  // staged: load i takes rows 16 i .. 16 i + 15, lane l piece (l & 3) ^ (row / 2 & 3) of row 16 i + l / 4, so that the
  // lanes that read one piece of consecutive rows do not meet in a bank
  uint4* const own[2] = {reinterpret_cast<uint4*>(part[wave]), reinterpret_cast<uint4*>(part[wave] + 4)};
  uint32_t goff[4], loff[2][2];
  if constexpr (kStaged) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * i + (lane >> 2);  // columns past N repeat the last fragment's
      goff[i] = static_cast<uint32_t>(min(row, cols - 32 + (row & 31))) * (static_cast<uint32_t>(p.K) >> 1) +
                ((lane & 3) ^ (row >> 1 & 3)) * 16u;
    }
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int q = 0; q < 2; ++q) loff[f][q] = (f * 32 + r) * 4 + ((2 * q + h) ^ (r >> 1 & 3));
  }
  auto load = [&](int kb, Block& b, uint4* stage) {
    kb = __builtin_amdgcn_readfirstlane(kb);
    if constexpr (kStaged) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the block that lay there has been read
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < 4; ++i)
        dma16(weights.wrs, stage + i * 64, goff[i], kb * 64);
      weights.load_scales(kb, b.s);
    } else {
      weights.load(kb, b.w, b.s);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) b.x[j] = buf_load16(xrs, lane * 16, kb * 8192 + j * 1024);
#pragma unroll
    for (int g = 0; g < 4; ++g) b.neg[g] = __builtin_bit_cast(f32x4, buf_load16(nrs, h * 16, kb * 128 + g * 32));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);  // issued here, a k-block ahead of their use
  };
  f32x16 tot[2] = {zero16(), zero16()};
  auto compute = [&](Block& b, const uint4* stage) {
    if constexpr (kStaged) {
      // this block's loads are in once only the next one's (4 + 2 + 8 + 4) are pending; written out, since the compiler's
      // own wait for direct-to-LDS loads can be missing in a loop
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0F70 | (18 & 15) | (18 >> 4) << 14);  // vmcnt(18)
      asm volatile("" ::: "memory");
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int q = 0; q < 2; ++q) b.w[f][q] = stage[loff[f][q]];
    }
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = b.neg[i >> 2][i & 3];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = mfma32(b.x[j], dequant24(word(b.w[f][j >> 2], j & 3)), acc);
      tot[f] += scale_value<ScaleT>(b.s[f]) * acc;
    }
  };
  // wave w: k-blocks w, w + 4, ... (the four waves read neighbouring blocks of a weight row, whole cache lines of it in
  // the portable layout, at about the same time)
  Block b0, b1;
  load(min(wave, nkb - 1), b0, own[0]);  // past the last k-block it is loaded again: a load under a condition would make every use wait for all
#pragma unroll 1
  for (int kb = wave; kb < nkb; kb += 8) {
    load(min(kb + 4, nkb - 1), b1, own[1]);
    compute(b0, own[0]);
    if (kb + 4 >= nkb) break;
    load(min(kb + 8, nkb - 1), b0, own[0]);
    compute(b1, own[1]);
  }
  if constexpr (kStaged) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): part holds no stage any more
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      part[wave][f * 4 + g][lane] = f32x4{tot[f][4 * g], tot[f][4 * g + 1], tot[f][4 * g + 2], tot[f][4 * g + 3]};
  __syncthreads();
  // wave w adds rows 8 w + 4 h + e of both fragments over the waves, in wave order
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    if (f * 32 >= cols) break;
    const int g = f * 4 + wave;
    const f32x4 y = ((part[0][g][lane] + part[1][g][lane]) + part[2][g][lane]) + part[3][g][lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 8 * wave + 4 * h + e;
      if (row >= rows) continue;
      const int64_t o = static_cast<int64_t>(mt * 32 + row) * N + col0 + f * 32 + r;
      if (p.y_f32) static_cast<float*>(p.y)[o] = y[e];
      else static_cast<uint16_t*>(p.y)[o] = f32_to_bf16(y[e]);
    }
  }
}

static void launch_prep(const LinearParams& p, hipStream_t stream) {
  const int64_t waves = static_cast<int64_t>((p.M + 31) / 32) * (p.K / 128);
  hipLaunchKernelGGL(w4_linear_prep_kernel, dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), 0, stream, p);
}

}  // namespace

bool w4_linear_fits(int64_t M, int64_t N, int64_t K) {
  // 32-bit offsets inside a tile: 64 rows of 2 K bytes, 256 columns of K / 2
  return M >= 1 && N >= 32 && N % 32 == 0 && K >= 128 && K % 128 == 0 && K < (int64_t{1} << 25) &&
         ((M + 31) / 32) * ((N + 63) / 64) < (int64_t{1} << 30);
}

void launch_w4_linear(const LinearParams& p, int cus, hipStream_t stream) {
  launch_prep(p, stream);
  const int64_t tiles = static_cast<int64_t>((p.M + 32 * kSub - 1) / (32 * kSub)) * ((p.N + 255) / 256);
  if (8 * tiles >= 5 * cus) {
    const dim3 grid(static_cast<unsigned>((tiles + 7) / 8 * 8)), block(256);
    if (p.scale_f32) hipLaunchKernelGGL(w4_linear_tile_kernel<float>, grid, block, 0, stream, p);
    else hipLaunchKernelGGL(w4_linear_tile_kernel<uint16_t>, grid, block, 0, stream, p);
  } else {
    const int64_t parts = static_cast<int64_t>((p.M + 31) / 32) * ((p.N + 63) / 64);
    const dim3 grid(static_cast<unsigned>((parts + 7) / 8 * 8)), block(256);
    if (p.tiled) {
      if (p.scale_f32) hipLaunchKernelGGL((w4_linear_split_kernel<float, false>), grid, block, 0, stream, p);
      else hipLaunchKernelGGL((w4_linear_split_kernel<uint16_t, false>), grid, block, 0, stream, p);
    } else {
      if (p.scale_f32) hipLaunchKernelGGL((w4_linear_split_kernel<float, true>), grid, block, 0, stream, p);
      else hipLaunchKernelGGL((w4_linear_split_kernel<uint16_t, true>), grid, block, 0, stream, p);
    }
  }
}

}  // namespace dflash
