// The operations between a transformer layer's matrix products, one launch each, written for gfx950.
//
//  * norm_kernel      - RMSNorm and LayerNorm over the last dimension of bf16 rows, with what surrounds
//                       them folded in: the residual add (plain or gated) that makes the row, and the
//                       affine or AdaLN scale and shift that follow. A row is read once and stays in
//                       registers between its statistics and its output.
//  * rope_cache_kernel - rotary embedding of a step's queries and keys, with the keys and values written
//                       to their place in the KV cache.
//  * silu_mul_kernel  - silu(gate) * up.
//
// All ask for some LDS (kLdsToken), which keeps their workgroups off the CUs that a streamed pass's copy holds.
// Traced beside that copy, us (median) without and with it: silu_mul of 64 x 5504 12.2 and 3.8, of 128 x 28672
// 18.8 and 8.5; the rotary kernel for 64 tokens of 32 heads 12.1 and 5.3; the combine of 64 heads (attention)
// 26.3 and 6.3.
//
// All are bound by the bytes they read and write (for a decode token by the launch itself). Arithmetic is
// fp32; values round to bf16 where they are stored. As separate elementwise operations an RMSNorm is six
// launches that move each value 12 times (17 us for 8 rows of 8192 and 55 us for 512 rows), the rotary
// embedding and cache write sixteen.
#include <algorithm>

#include "ftx_internal.h"

namespace ftx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;
constexpr int kVec = 8;      // bf16 values per 16-byte access
constexpr int kNormVecs = 4; // vectors of a row a lane holds

struct Vec8 {
  float v[kVec];
};

__device__ __forceinline__ Vec8 unpack(u32x4 p) {
  Vec8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r.v[2 * i] = __uint_as_float(p[i] << 16);
    r.v[2 * i + 1] = __uint_as_float(p[i] & 0xffff0000u);
  }
  return r;
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

__device__ __forceinline__ u32x4 pack(const Vec8 &r) {
  return u32x4{pack2(r.v[0], r.v[1]), pack2(r.v[2], r.v[3]), pack2(r.v[4], r.v[5]), pack2(r.v[6], r.v[7])};
}

__device__ __forceinline__ Vec8 load8(const uint16_t *p) { return unpack(*reinterpret_cast<const u32x4 *>(p)); }
__device__ __forceinline__ void store8(uint16_t *p, const Vec8 &r) { *reinterpret_cast<u32x4 *>(p) = pack(r); }

// Sum of v over the WAVES wavefronts of one row, in every lane. `slots` holds WAVES floats per row of the
// workgroup; the leading barrier lets a second sum reuse them.
template <int WAVES>
__device__ __forceinline__ float row_sum(float v, float *slots) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  if (WAVES == 1) return v;
  const int wave = threadIdx.x / kWave;
  __syncthreads();
  if (threadIdx.x % kWave == 0) slots[wave] = v;
  __syncthreads();
  v = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) v += slots[w];
  return v;
}

// One row per WAVES wavefronts (a row of up to WAVES * 2048 values); workgroups of one row, or of four
// rows with a wavefront each.
template <int WAVES, int RESIDUAL, int NORM>
__global__ __launch_bounds__(WAVES == 1 ? 256 : WAVES * kWave) void norm_kernel(NormLaunch p) {
  __shared__ float slots[WAVES];
  const int64_t row = WAVES == 1 ? static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / kWave : blockIdx.x;
  if (row >= p.rows) return;
  const int lane = WAVES == 1 ? threadIdx.x % kWave : threadIdx.x;
  constexpr int kStep = WAVES * kWave * kVec;
  const int dim = p.dim;
  const uint16_t *x = p.x + row * dim;
  // AdaLN terms: the modulation row plus the row's batch element of the timestep embedding
  const uint16_t *e = p.e ? p.e + row / p.rows_per_batch * 6 * dim : nullptr;
  auto term = [&](int index, int at) {
    const Vec8 a = load8(p.mod + static_cast<int64_t>(index) * dim + at);
    const Vec8 b = load8(e + static_cast<int64_t>(index) * dim + at);
    Vec8 r;
#pragma unroll
    for (int i = 0; i < kVec; ++i) r.v[i] = a.v[i] + b.v[i];
    return r;
  };

  Vec8 v[kNormVecs];
#pragma unroll
  for (int q = 0; q < kNormVecs; ++q) {
    const int at = q * kStep + lane * kVec;
    if (at < dim) {
      v[q] = load8(x + at);
      if (RESIDUAL != kNormNoResidual) {
        const Vec8 d = load8(p.delta + row * dim + at);
        if (RESIDUAL == kNormGatedResidual) {
          const Vec8 gate = term(p.gate, at);
#pragma unroll
          for (int i = 0; i < kVec; ++i) v[q].v[i] = fmaf(d.v[i], gate.v[i], v[q].v[i]);
        } else {
#pragma unroll
          for (int i = 0; i < kVec; ++i) v[q].v[i] += d.v[i];
        }
        const u32x4 sum = pack(v[q]);
        *reinterpret_cast<u32x4 *>(p.x_out + row * dim + at) = sum;
        v[q] = unpack(sum);  // the norm reads the row as it is stored
      }
    } else {
#pragma unroll
      for (int i = 0; i < kVec; ++i) v[q].v[i] = 0.f;
    }
  }
  if (NORM == kNormNone) return;

  const float inv_dim = 1.0f / static_cast<float>(dim);
  float mean = 0.f;
  if (NORM != kNormRms) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < kNormVecs; ++q)
#pragma unroll
      for (int i = 0; i < kVec; ++i) s += v[q].v[i];
    mean = row_sum<WAVES>(s, slots) * inv_dim;
  }
  float ss = 0.f;
#pragma unroll
  for (int q = 0; q < kNormVecs; ++q)
    if (q * kStep + lane * kVec < dim)
#pragma unroll
      for (int i = 0; i < kVec; ++i) {
        const float c = v[q].v[i] - mean;
        ss = fmaf(c, c, ss);
      }
  const float rstd = rsqrtf(row_sum<WAVES>(ss, slots) * inv_dim + p.eps);

  uint16_t *y = p.y + row * dim;
#pragma unroll
  for (int q = 0; q < kNormVecs; ++q) {
    const int at = q * kStep + lane * kVec;
    if (at >= dim) continue;
    Vec8 out;
    if (NORM == kNormRms) {
      const Vec8 w = load8(p.w + at);
#pragma unroll
      for (int i = 0; i < kVec; ++i) out.v[i] = v[q].v[i] * rstd * w.v[i];
    } else {
      const Vec8 scale = NORM == kNormAffine ? load8(p.w + at) : term(p.scale, at);
      const Vec8 shift = NORM == kNormAffine ? load8(p.b + at) : term(p.shift, at);
#pragma unroll
      for (int i = 0; i < kVec; ++i)
        out.v[i] = fmaf((v[q].v[i] - mean) * rstd, NORM == kNormAffine ? scale.v[i] : 1.0f + scale.v[i], shift.v[i]);
    }
    store8(y + at, out);
  }
}

// A lane owns eight values of a head's first half and their partners in the second: out1 = x1 cos1 - x2 sin1,
// out2 = x2 cos2 + x1 sin2. Heads 0..heads-1 are queries, then kv_heads keys, then kv_heads values (copied).
__global__ __launch_bounds__(256) void rope_cache_kernel(RopeLaunch p) {
  const int half = p.d / 2;
  const int lanes = half / kVec;  // per head
  const int heads = p.heads + 2 * p.kv_heads;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t row_head = id / lanes;
  const int at = static_cast<int>(id % lanes) * kVec;
  const int64_t row = row_head / heads;  // batch * t + token
  int head = static_cast<int>(row_head % heads);
  if (row >= static_cast<int64_t>(p.batch) * p.t) return;
  const int64_t b = row / p.t;
  const int64_t pos = p.pos + row % p.t;
  const uint16_t *src;
  uint16_t *dst;
  if (head < p.heads) {
    src = p.q + (row * p.heads + head) * p.d;
    dst = p.q_out + (row * p.heads + head) * p.d;
  } else if ((head -= p.heads) < p.kv_heads) {
    src = p.k + (row * p.kv_heads + head) * p.d;
    dst = p.cache_k + b * p.k_stride[0] + pos * p.k_stride[1] + head * p.k_stride[2];
  } else {
    head -= p.kv_heads;
    src = p.v + (row * p.kv_heads + head) * p.d;
    dst = p.cache_v + b * p.v_stride[0] + pos * p.v_stride[1] + head * p.v_stride[2];
    const u32x4 lo = *reinterpret_cast<const u32x4 *>(src + at);
    const u32x4 hi = *reinterpret_cast<const u32x4 *>(src + half + at);
    *reinterpret_cast<u32x4 *>(dst + at) = lo;
    *reinterpret_cast<u32x4 *>(dst + half + at) = hi;
    return;
  }
  const Vec8 x1 = load8(src + at), x2 = load8(src + half + at);
  const float *cs = p.cos + pos * p.d + at, *sn = p.sin + pos * p.d + at;
  Vec8 o1, o2;
#pragma unroll
  for (int i = 0; i < kVec; ++i) {
    o1.v[i] = fmaf(x1.v[i], cs[i], -x2.v[i] * sn[i]);
    o2.v[i] = fmaf(x2.v[i], cs[half + i], x1.v[i] * sn[half + i]);
  }
  store8(dst + at, o1);
  store8(dst + half + at, o2);
}

// y = bf16(bf16(silu(g)) * u), rounded as the two operations on their own round.
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t *__restrict__ g, const uint16_t *__restrict__ u,
                                                       uint16_t *__restrict__ y, int64_t n) {
  const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * kVec;
  if (at >= n) return;
  const Vec8 a = load8(g + at), b = load8(u + at);
  Vec8 s;
#pragma unroll
  for (int i = 0; i < kVec; ++i) s.v[i] = a.v[i] / (1.0f + expf(-a.v[i]));
  s = unpack(pack(s));
#pragma unroll
  for (int i = 0; i < kVec; ++i) s.v[i] *= b.v[i];
  store8(y + at, s);
}

template <int WAVES, int RESIDUAL>
hipError_t launch_norm_residual(const NormLaunch &p, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(WAVES == 1 ? (p.rows + 3) / 4 : p.rows));
  const dim3 block(WAVES == 1 ? 256 : WAVES * kWave);
  constexpr unsigned lds = kLdsToken;  // a row within one wave, or without a norm, has none of its own
  switch (p.norm) {
    case kNormNone: hipLaunchKernelGGL((norm_kernel<WAVES, RESIDUAL, kNormNone>), grid, block, lds, stream, p); break;
    case kNormRms: hipLaunchKernelGGL((norm_kernel<WAVES, RESIDUAL, kNormRms>), grid, block, lds, stream, p); break;
    case kNormAffine:
      hipLaunchKernelGGL((norm_kernel<WAVES, RESIDUAL, kNormAffine>), grid, block, lds, stream, p);
      break;
    default: hipLaunchKernelGGL((norm_kernel<WAVES, RESIDUAL, kNormAdaln>), grid, block, lds, stream, p); break;
  }
  return hipGetLastError();
}

template <int WAVES>
hipError_t launch_norm_waves(const NormLaunch &p, hipStream_t stream) {
  switch (p.residual) {
    case kNormNoResidual: return launch_norm_residual<WAVES, kNormNoResidual>(p, stream);
    case kNormResidual: return launch_norm_residual<WAVES, kNormResidual>(p, stream);
    default: return launch_norm_residual<WAVES, kNormGatedResidual>(p, stream);
  }
}

}  // namespace

int64_t norm_max_rows(int64_t dim) {
  const int64_t threads = dim <= 2048 ? 64 : dim <= 8192 ? 256 : 1024;  // of a row: launch_norm
  return kMaxThreads / threads - 3;                                     // workgroups of four rows round up
}

// A row takes the fewest wavefronts whose registers hold it: one up to 2048 values (64 lanes x 4 vectors of
// 8), four up to 8192, sixteen up to 32768.
hipError_t launch_norm(const NormLaunch &p, hipStream_t stream) {
  constexpr int kPerWave = kWave * kVec * kNormVecs;
  static_assert(16 * kPerWave == kNormMaxDim, "the largest row the wavefronts of one workgroup hold");
  static_assert(kPerWave == 2048, "norm_max_rows counts the same wavefronts");
  if (p.dim <= kPerWave) return launch_norm_waves<1>(p, stream);
  if (p.dim <= 4 * kPerWave) return launch_norm_waves<4>(p, stream);
  return launch_norm_waves<16>(p, stream);
}

hipError_t launch_rope_cache(const RopeLaunch &p, hipStream_t stream) {
  const int64_t lanes = static_cast<int64_t>(p.batch) * p.t * (p.heads + 2 * p.kv_heads) * (p.d / 2 / kVec);
  hipLaunchKernelGGL(rope_cache_kernel, dim3(static_cast<unsigned>((lanes + 255) / 256)), dim3(256), kLdsToken,
                     stream, p);
  return hipGetLastError();
}

hipError_t launch_silu_mul(const uint16_t *g, const uint16_t *u, uint16_t *y, int64_t n, hipStream_t stream) {
  const int64_t per_block = 256 * kVec;
  hipLaunchKernelGGL(silu_mul_kernel, dim3(static_cast<unsigned>((n + per_block - 1) / per_block)), dim3(256),
                     kLdsToken, stream, g, u, y, n);
  return hipGetLastError();
}

}  // namespace ftx
