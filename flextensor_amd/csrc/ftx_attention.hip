// Attention over [batch, position, head, head_dim] tensors in bf16, written for gfx950.
//
//   o[b, t, h, :] = sum_s softmax_s(scale * q[b, t, h, :] . k[b, s, h / rep, :]) v[b, s, h / rep, :]
//
// with every stride but the last free, so queries, a KV cache and a transposed view are read where they
// lie: no head is repeated, nothing is transposed in memory and no score leaves the chip. Scores, the
// running maximum and the running sum are fp32; the probabilities enter the second product in bf16.
//
// Rows: the `rep` query heads that share a K/V head and the T query positions are one list of T * rep
// rows (row = position * rep + head in the group), so a group reads its keys once and one decode token of
// eight heads fills a quarter of a 32-row tile instead of one row of eight tiles. Causal attention
// compares positions, row / rep.
//
// One wavefront owns 32 rows; the NW wavefronts of a workgroup share K/V tiles of KT keys in an LDS ring.
// Per tile a wave computes S^T = K Q^T with v_mfma_f32_32x32x16_bf16: a lane then holds 16 of the 32 keys
// of ONE row, so the row's maximum and sum are register operations and one exchange between the wave's
// halves. O^T += V^T P^T takes the probabilities straight from those registers: lane group g = lane / 32
// holds keys 4g..4g+3 and 8+4g..8+4g+3 of every 16, and V^T is read with ds_read_b64_tr_b16 in that same
// key order (any order of k that both operands of an MFMA share gives the same sum).
//
// K and V go from memory into LDS by buffer loads (no register staging). Their descriptors end with the
// last key's row, so rows past it read as zero: a ragged end needs no clamped addresses, and a zero weight
// never meets a value from outside the tensor. Rows that overlap (TIGHT: a position stride below a row, 0 for
// expanded values) would lie inside the descriptor past the last key too, so V's loads of those rows are sent
// past its end by row number (in every kernel this cost 1 to 7%); K's need not, their scores are masked by
// position. Each load writes 1 KB, lane l at +16 l; the layout is chosen by which 16-byte chunk a lane fetches.
// Chunk c of row R lies at slot c ^ f(R), with f spreading the rows one read touches over all 64 banks: for K
// (16 bytes of 32 rows a read) f = R % 16 at 256-byte rows and (R / 2) % 8 at 128-byte rows; for V (four rows
// of 32 bytes a transposed read) 4 (R % 4) and 4 (R / 2 % 2).
//
// The maximum is only raised when a score exceeds it by more than 2^kSlack: the probabilities stay below
// 2^kSlack, keep their relative precision, and the accumulators are rescaled a few times per row instead
// of once per tile.
//
// Bound by the MFMA units at long sequences: 40 heads of 8190 x 8190 at d = 128 take 1.33 ms, 1.03 PFLOP/s
// of the 1.5-1.8 the units sustain; the library's flash attention took 4.7 ms (0.29 PFLOP/s). A decode
// token is bound by its keys and values: 8 x 64 / 8 heads over 1024 keys as one product on repeated,
// transposed copies of the cache took about 600 us.
//
// Block order: consecutive items (K/V head, then row tile, then split) run on one XCD, so the workgroups
// that read one head's keys share that XCD's L2.
#include <algorithm>
#include <cfloat>

#include "ftx_internal.h"

namespace ftx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr int kWave = 64;
constexpr int kRowsPerWave = 32;
constexpr float kSlack = 8.0f;

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// The larger (or the sum) of a value and its partner's in the other half of the wave.
__device__ __forceinline__ float half_max(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// 16 bytes per lane from base + offset into lds + 16 * lane; a lane whose offset is not below `bytes` writes
// zeros.
__device__ __forceinline__ void load_to_lds(const void *base, uint32_t bytes, uint32_t offset, uint8_t *lds) {
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00027000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void *)lds, 16, offset, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N < 64, "vmcnt holds six bits");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS reads are done
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int D, int NW, int KT, int STAGES, bool SPLIT, bool TIGHT = false>
__global__ __launch_bounds__(NW * kWave, NW == 8 ? 2 : 1) void attention_kernel(AttentionLaunch a) {
  constexpr int kRowBytes = 2 * D;
  constexpr int kRowChunks = D / 8;
  constexpr int kTileBytes = KT * kRowBytes;              // K or V of one tile
  constexpr int kStage = 2 * kTileBytes;
  constexpr int kLoads = kTileBytes / 1024;               // 1 KB loads per K or V tile
  constexpr int kPerWave = kLoads / NW;
  static_assert(kLoads % NW == 0, "every wave issues the same number of loads");
  constexpr int kRowsPerLoad = 1024 / kRowBytes;
  constexpr int kSub = KT / 32;                           // 32-key blocks per tile
  constexpr int kQSteps = D / 16;
  constexpr int kDTiles = D / 32;
  __shared__ __align__(1024) uint8_t lds[STAGES * kStage];

  const int64_t per_xcd = (a.items + a.xcds - 1) / a.xcds;
  const int64_t item = static_cast<int64_t>(blockIdx.x % a.xcds) * per_xcd + blockIdx.x / a.xcds;
  if (blockIdx.x / a.xcds >= per_xcd || item >= a.items) return;
  const int sp = SPLIT ? static_cast<int>(item % a.splits) : 0;
  const int64_t tile_item = SPLIT ? item / a.splits : item;
  const int qt = a.row_tiles - 1 - static_cast<int>(tile_item % a.row_tiles);  // causal: the longest first
  const int64_t bkv = tile_item / a.row_tiles;
  const int64_t b = bkv / a.kv_heads;
  const int kvh = static_cast<int>(bkv % a.kv_heads);

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane & 31;
  const int g = lane >> 5;
  const int row0 = (qt * NW + wave) * kRowsPerWave;
  const int row = min(row0 + r, a.rows - 1);
  const int token = row / a.rep;
  const int head = kvh * a.rep + (row - token * a.rep);

  // Keys this workgroup, this wave and this lane's row can see.
  const int last_row = min((qt + 1) * NW * kRowsPerWave, a.rows) - 1;
  const int wg_end = a.causal ? min(a.s, a.pos + last_row / a.rep + 1) : a.s;
  const int wave_last = min(row0 + kRowsPerWave, a.rows) - 1;
  const bool active = row0 < a.rows;
  const int wave_end = a.causal ? min(a.s, a.pos + wave_last / a.rep + 1) : a.s;
  const int wave_free = a.causal ? min(a.s, a.pos + row0 / a.rep + 1) : a.s;  // every row sees keys below this
  const int limit = a.causal ? min(a.s, a.pos + token + 1) : a.s;
  const int first = SPLIT ? sp * a.split_tiles : 0;
  int n_tiles = (wg_end + KT - 1) / KT;
  if (SPLIT) n_tiles = min(n_tiles, first + a.split_tiles);

  const uint16_t *kb = a.k + b * a.k_stride[0] + kvh * a.k_stride[2];
  const uint16_t *vb = a.v + b * a.v_stride[0] + kvh * a.v_stride[2];
  const uint32_t k_ss = static_cast<uint32_t>(a.k_stride[1]) * 2, v_ss = static_cast<uint32_t>(a.v_stride[1]) * 2;
  const uint32_t k_bytes = static_cast<uint32_t>(a.s - 1) * k_ss + kRowBytes;
  const uint32_t v_bytes = static_cast<uint32_t>(a.s - 1) * v_ss + kRowBytes;
  uint32_t koff[kPerWave], voff[kPerWave];
#pragma unroll
  for (int i = 0; i < kPerWave; ++i) {
    const int R = (wave * kPerWave + i) * kRowsPerLoad + lane / kRowChunks;
    const int c = lane % kRowChunks;
    const int kc = c ^ (D == 128 ? (R & 15) : ((R >> 1) & 7));
    const int vc = c ^ (D == 128 ? ((R & 3) << 2) : (((R >> 1) & 1) << 2));
    koff[i] = static_cast<uint32_t>(R) * k_ss + kc * 16;
    voff[i] = static_cast<uint32_t>(R) * v_ss + vc * 16;
  }
  auto issue = [&](int t) {
    uint8_t *base = lds + (t % STAGES) * kStage + wave * kPerWave * 1024;
    const uint32_t kt = static_cast<uint32_t>(t) * KT * k_ss, vt = static_cast<uint32_t>(t) * KT * v_ss;
#pragma unroll
    for (int i = 0; i < kPerWave; ++i)
      load_to_lds(kb, k_bytes, koff[i] + kt, base + i * 1024);
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      uint32_t offset = voff[i] + vt;
      if constexpr (TIGHT)
        if ((wave * kPerWave + i) * kRowsPerLoad + lane / kRowChunks >= a.s - t * KT) offset = v_bytes;
      load_to_lds(vb, v_bytes, offset, base + kTileBytes + i * 1024);
    }
  };

  // Queries: lane (r, g) holds elements 16 ks + 8 g .. + 7 of its row for every step ks.
  bf16x8 qf[kQSteps];
  {
    const uint16_t *qp = a.q + b * a.q_stride[0] + token * a.q_stride[1] + head * a.q_stride[2] + 8 * g;
#pragma unroll
    for (int ks = 0; ks < kQSteps; ++ks)
      qf[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(qp + 16 * ks));
  }
  // the queries are in registers before the ring's loads are counted
  asm volatile("" ::: "memory");
  wait_vmcnt<0>();
#pragma unroll
  for (int st = 0; st < STAGES - 1; ++st)
    if (first + st < n_tiles) issue(first + st);

  const int ka = r * kRowBytes + ((g ^ (D == 128 ? (r & 15) : ((r >> 1) & 7))) << 4);
  const int i16 = lane & 15;
  const int va = (4 * g + (i16 >> 2)) * kRowBytes +
                 (((((lane >> 4) & 1) * 2 + ((i16 & 3) >> 1)) ^ (D == 128 ? (i16 >> 2) << 2 : (i16 >> 3) << 2)) << 4) +
                 (i16 & 1) * 8;

  f32x16 o[kDTiles];
#pragma unroll
  for (int d = 0; d < kDTiles; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  // The row's reference maximum, in units of log2. It starts at the lowest finite value: while no key of the row
  // counts (every score so far is -inf, or a split holds no key that the row sees) -inf less it is -inf, a weight
  // of zero, where -inf less -inf is NaN. Selecting that case in the loop took 12 heads of 2000 x 2000 from 60.2
  // to 65.0 us.
  float m = -FLT_MAX;
  float l = 0.f;        // this lane's part of the row's sum

  for (int t = first; t < n_tiles; ++t) {
    if (t + STAGES - 2 < n_tiles)
      wait_vmcnt<(STAGES - 2) * 2 * kPerWave>();
    else
      wait_vmcnt<0>();
    ring_barrier();
    if (!active || t * KT >= wave_end) {
      if (t + STAGES - 1 < n_tiles) issue(t + STAGES - 1);
      continue;
    }
    const uint8_t *kt = lds + (t % STAGES) * kStage;
    const uint8_t *vt = kt + kTileBytes;

    f32x16 s[kSub];
#pragma unroll
    for (int j = 0; j < kSub; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[j][e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < kQSteps; ++ks)
#pragma unroll
      for (int j = 0; j < kSub; ++j) {
        const u32x4 kv = *reinterpret_cast<const u32x4 *>(kt + j * 32 * kRowBytes + (ka ^ (ks * 32)));
        s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kv), qf[ks], s[j], 0, 0, 0);
      }
    if ((t + 1) * KT > wave_free) {
#pragma unroll
      for (int j = 0; j < kSub; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (t * KT + j * 32 + 8 * (e >> 2) + 4 * g + (e & 3) >= limit) s[j][e] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int j = 0; j < kSub; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[j][e]);
    mx = half_max(mx) * a.scale_log2;
    if (__any(mx > m + kSlack)) {
      const float m_new = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < kDTiles; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[d][e] *= alpha;
    }
    bf16x8 p[2 * kSub];  // 16 keys each, in the order the V reads share
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < kSub; ++j) {
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 16; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[j][e], a.scale_log2, -m));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[j][e + 1], a.scale_log2, -m));
        sum += p0 + p1;
        w[e / 2] = pack_bf16(p0, p1);
      }
      p[2 * j] = __builtin_bit_cast(bf16x8, (u32x4){w[0], w[1], w[2], w[3]});
      p[2 * j + 1] = __builtin_bit_cast(bf16x8, (u32x4){w[4], w[5], w[6], w[7]});
    }
    l += sum;
#pragma unroll
    for (int f = 0; f < 2 * kSub; ++f)
#pragma unroll
      for (int d = 0; d < kDTiles; ++d) {
        const uint8_t *vp = vt + f * 16 * kRowBytes + (va ^ (d * 64));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vp));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(vp + 8 * kRowBytes));
        const bf16x8 vf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, p[f], o[d], 0, 0, 0);
      }
    // The buffer of tile t - 1 is free since the barrier. The compiler waits for every load to LDS ahead of
    // the transposed reads, so the next tile's loads go out after them and have the next scores to arrive in.
    if (t + STAGES - 1 < n_tiles) issue(t + STAGES - 1);
  }

  if (row0 + r >= a.rows) return;
  l = half_sum(l);
  if (SPLIT) {  // [split][batch * kv head][row][D] values, then [split][batch * kv head][row] maxima and sums
    const int64_t bkvs = static_cast<int64_t>(a.batch) * a.kv_heads;
    const int64_t at = (sp * bkvs + bkv) * a.rows + row;
    float *po = a.part + at * D;
    float *pm = a.part + a.splits * bkvs * a.rows * D;
#pragma unroll
    for (int d = 0; d < kDTiles; ++d)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4 *>(po + d * 32 + q * 8 + 4 * g) =
            (f32x4){o[d][4 * q], o[d][4 * q + 1], o[d][4 * q + 2], o[d][4 * q + 3]};
    if (g == 0) {
      pm[at] = m;
      pm[a.splits * bkvs * a.rows + at] = l;
    }
    return;
  }
  const float inv = 1.0f / l;
  uint16_t *op = a.o + b * a.o_stride[0] + token * a.o_stride[1] + head * a.o_stride[2] + 4 * g;
#pragma unroll
  for (int d = 0; d < kDTiles; ++d)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<u32x2 *>(op + d * 32 + q * 8) =
          (u32x2){pack_bf16(o[d][4 * q] * inv, o[d][4 * q + 1] * inv),
                  pack_bf16(o[d][4 * q + 2] * inv, o[d][4 * q + 3] * inv)};
}

// o = sum_i 2^(m_i - M) o_i / sum_i 2^(m_i - M) l_i over the splits, M the largest m_i; D / 4 lanes a row.
// A split that saw no key of a row has m = -FLT_MAX and l = 0.
template <int D>
__global__ __launch_bounds__(256) void attention_combine_kernel(AttentionLaunch a) {
  constexpr int kLanes = D / 4;
  const int64_t bkvs = static_cast<int64_t>(a.batch) * a.kv_heads;
  const int64_t n = bkvs * a.rows;
  const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / kLanes;
  const int c = threadIdx.x % kLanes;
  if (at >= n) return;
  const float *pm = a.part + a.splits * n * D;
  const float *pl = pm + a.splits * n;
  // Splits are read a batch at a time, the loads of a batch ahead of their use: one after the other their
  // latencies made this kernel as long as the attention of a decode token itself (5.9 us of 9 splits).
  constexpr int kBatch = 8;
  float mx = -FLT_MAX, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < a.splits; i0 += kBatch) {
    float m[kBatch], part_l[kBatch];
    f32x4 part[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {  // the last batch repeats its last split, with a weight of zero below
      const int64_t s = min(i0 + i, a.splits - 1) * n + at;
      m[i] = pm[s];
      part_l[i] = pl[s];
      part[i] = *reinterpret_cast<const f32x4 *>(a.part + s * D + 4 * c);
    }
    float m_new = mx;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) m_new = fmaxf(m_new, m[i]);
    const float alpha = __builtin_amdgcn_exp2f(mx - m_new);
    l *= alpha;
    acc *= alpha;
    mx = m_new;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (i0 + i >= a.splits) break;
      const float w = __builtin_amdgcn_exp2f(m[i] - m_new);
      l += w * part_l[i];
      acc += w * part[i];
    }
  }
  const float inv = 1.0f / l;
  const int64_t bkv = at / a.rows;
  const int row = static_cast<int>(at % a.rows);
  const int token = row / a.rep;
  const int head = static_cast<int>(bkv % a.kv_heads) * a.rep + (row - token * a.rep);
  uint16_t *op = a.o + bkv / a.kv_heads * a.o_stride[0] + token * a.o_stride[1] + head * a.o_stride[2] + 4 * c;
  *reinterpret_cast<u32x2 *>(op) =
      (u32x2){pack_bf16(acc[0] * inv, acc[1] * inv), pack_bf16(acc[2] * inv, acc[3] * inv)};
}

template <int D, int NW, int KT, int STAGES>
hipError_t launch_shape(const AttentionLaunch &p, hipStream_t stream) {
  const int64_t per_xcd = (p.items + p.xcds - 1) / p.xcds;
  const dim3 grid(static_cast<unsigned>(per_xcd * p.xcds));
  if constexpr (NW == 1) {  // only one-wave workgroups split the keys
    if (p.splits > 1) {
      hipLaunchKernelGGL((attention_kernel<D, NW, KT, STAGES, true>), grid, dim3(NW * kWave), 0, stream, p);
      hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
      const int64_t lanes = static_cast<int64_t>(p.batch) * p.kv_heads * p.rows * (D / 4);
      hipLaunchKernelGGL((attention_combine_kernel<D>), dim3(static_cast<unsigned>((lanes + 255) / 256)), dim3(256),
                         kLdsToken, stream, p);
      return hipGetLastError();
    }
    if (p.tight) {
      hipLaunchKernelGGL((attention_kernel<D, NW, KT, STAGES, false, true>), grid, dim3(NW * kWave), 0, stream, p);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((attention_kernel<D, NW, KT, STAGES, false>), grid, dim3(NW * kWave), 0, stream, p);
  return hipGetLastError();
}

template <int D>
hipError_t launch_dim(const AttentionLaunch &p, hipStream_t stream) {
  switch (p.waves) {
    case 1: return launch_shape<D, 1, 32, 3>(p, stream);
    case 2: return launch_shape<D, 2, 32, 3>(p, stream);
    case 4: return launch_shape<D, 4, 32, 3>(p, stream);
    default: return launch_shape<D, 8, 64, 3>(p, stream);
  }
}

}  // namespace

void plan_attention(AttentionLaunch *p, int cus, int xcds) {
  p->xcds = std::max(1, xcds);
  p->rep = p->heads / p->kv_heads;
  p->rows = p->t * p->rep;
  const int64_t heads = static_cast<int64_t>(p->batch) * p->kv_heads;
  // Rows per workgroup: as many as share a K/V tile well, as few as fill the chip. A CU's time is about its
  // workgroups, rounded up, times their rows; half the rows are taken where that makes it 1.4 times shorter.
  // 12 heads of 2000 x 2000 in workgroups of 128 rows (192 of them) 60.7 us, of 64 rows (384) 75.8, of 32 62.3;
  // 32 heads of 512 x 512, causal, of 64 rows (256) 19.2 us, of 128 19.8.
  const auto cost = [&](int waves) {
    const int64_t groups = heads * ((p->rows + kRowsPerWave * waves - 1) / (kRowsPerWave * waves));
    return (groups + cus - 1) / cus * waves;
  };
  // Overlapping values run unsplit one-wave workgroups, the only ones built for them.
  p->waves = p->tight ? 1 : 8;
  for (int w = 4; w >= 1 && !p->tight; w /= 2)
    if (p->rows <= kRowsPerWave * w || cost(p->waves) * 10 >= cost(w) * 14) p->waves = w;
  p->row_tiles = (p->rows + kRowsPerWave * p->waves - 1) / (kRowsPerWave * p->waves);
  const int kt = p->waves == 8 ? 64 : 32;
  const int tiles = (p->s + kt - 1) / kt;
  // One-wave workgroups (a decode token, a handful of rows): split the keys until two workgroups per CU have
  // work, with at least two tiles each. Up to four tiles the combine launch costs more than it saves: 16 heads
  // over 101 keys 6.7 us, split in two 7.9; over 528 keys of 32 heads 9 splits 10.0 us.
  const int64_t groups = heads * p->row_tiles;
  p->splits = 1;
  if (p->waves == 1 && groups < cus && tiles > 4 && !p->tight) {
    const int64_t want = std::min<int64_t>((2 * cus + groups - 1) / groups, (tiles + 1) / 2);
    p->split_tiles = static_cast<int>((tiles + want - 1) / want);
    p->splits = (tiles + p->split_tiles - 1) / p->split_tiles;
  }
  if (p->splits == 1) p->split_tiles = tiles;
  p->items = groups * p->splits;
  p->part_bytes = p->splits > 1 ? static_cast<size_t>(p->splits) * heads * p->rows * (p->d + 2) * sizeof(float) : 0;
}

hipError_t launch_attention(const AttentionLaunch &p, hipStream_t stream) {
  return p.d == 128 ? launch_dim<128>(p, stream) : launch_dim<64>(p, stream);
}

}  // namespace ftx
