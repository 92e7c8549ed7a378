// fp8-weight linear layer for decode-sized batches, written for gfx950.
//
//   y[m, n] = bf16( scale[n] * sum_k x[m, k] * w[n, k] )
//
// x is bf16 [M, K], w is float8 e4m3fn [N, K] (row-major, K contiguous),
// scale is one bf16 per output channel, y is bf16 [M, N]. A few rows run
// direct_linear_kernel (which takes bf16 weights too), up to 64 rows (decode)
// fp8_linear_kernel or 64-row tiles, more rows (prefill) the tiled
// fp8_prefill_kernel; the rules are at direct_linear_wins, mid_linear_wins and
// plan_fp8_linear.
//
// Decode multiplies a few activation rows by a large weight matrix, so the
// kernel is bound by reading the fp8 weights from HBM once (1 byte per
// weight). Each lane loads 16 weight bytes of one row, converts them to bf16
// in registers with v_cvt_scalef32_pk_bf16_fp8 (scale 1.0; every e4m3 value is
// exact in bf16) and feeds v_mfma_f32_16x16x32_bf16 with the weights as the A
// operand (16 output channels) and the activations as the B operand (16 batch
// columns). The activations stay bf16, so the products are exactly those of
// dequantizing the weights and running a bf16 GEMM; only the fp32
// accumulation order differs.
//
// Grouping: one launch can cover up to four weight matrices that share x and
// K (a layer's q/k/v projections, its gate/up projections). Their row groups
// are laid end to end in the grid, so the group pays one launch (and one
// reduce) instead of one per matrix.
//
// Work split: a workgroup of S wavefronts owns 16*S output channels (16 per
// wave) of one matrix and one K slice; the grid is row groups x K slices.
// Each workgroup stages its slice of x in LDS once, so L2 serves activations about 2M/(16 S)
// times the weight bytes. With one slice the kernel writes y directly;
// otherwise it writes fp32 partials [slice][M][N] and fp8_linear_reduce_kernel
// sums them in slice order, so results do not depend on timing. The split is
// a separate kernel: an in-kernel last-arriver reduction needs either
// agent-scope release/acquire (a whole-L2 writeback per workgroup) or
// device-coherent partials and counters, and the coherent form measured
// slower than two launches (218 against 172 us for a 70B layer's projections).
//
// MFMA 16x16x32 operand layout (gfx950): lane l supplies row/column l%16 and
// the eight k values 8*(l/16)..8*(l/16)+7 of the 32-wide k block; lane l
// receives D rows 4*(l/16)..4*(l/16)+3 of column l%16. Any permutation of k
// that A and B share gives the same sum, so here lane group g = l/16 holds the
// k values g*16..g*16+15 of a 64-byte piece: the first eight go to one MFMA,
// the last eight to a second one.
#include <algorithm>
#include <type_traits>

#include "ftx_internal.h"

namespace ftx {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// four floats at any 4-byte boundary: vector memory accesses need no more than dword alignment
typedef float f32x4_dword __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWave = 64;
constexpr int kPieceBytes = 16;              // fp8 bytes one lane loads per row and step
constexpr int kStepBytes = 4 * kPieceBytes;  // K bytes one step covers per row (4 lane groups)

__device__ __forceinline__ bf16x8 join8(bf16x2 a, bf16x2 b, bf16x2 c, bf16x2 d) {
  const bf16x4 lo = __builtin_shufflevector(a, b, 0, 1, 2, 3);
  const bf16x4 hi = __builtin_shufflevector(c, d, 0, 1, 2, 3);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// 16 e4m3fn bytes -> bf16 of bytes 0-7 (lo) and bytes 8-15 (hi), in byte order.
__device__ __forceinline__ void fp8x16_to_bf16(u32x4 w, bf16x8 &lo, bf16x8 &hi) {
  const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.0f, false);
  const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.0f, true);
  const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.0f, false);
  const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.0f, true);
  const bf16x2 p4 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2], 1.0f, false);
  const bf16x2 p5 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[2], 1.0f, true);
  const bf16x2 p6 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[3], 1.0f, false);
  const bf16x2 p7 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[3], 1.0f, true);
  lo = join8(p0, p1, p2, p3);
  hi = join8(p4, p5, p6, p7);
}

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// fp32 -> bf16 bits, round to nearest even; NaN stays NaN.
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return static_cast<uint16_t>((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

// Bytes of one weight row loaded per iteration: 16 lanes x 16 bytes, so one
// load instruction covers 4 rows x 256 contiguous bytes. Fewer, longer runs
// per instruction keep HBM near its streaming rate; the MFMA layout (16 rows
// per 16 lanes, 64 bytes each) is reached through a per-wave LDS tile.
constexpr int kIterK = 256;
constexpr int kRowsPerLoad = kWave * kPieceBytes / kIterK;   // 4
constexpr int kLoads = 16 / kRowsPerLoad;                     // 4 per 16 rows
constexpr int kSteps = kIterK / kStepBytes;                   // 4 MFMA steps per iteration
constexpr int kTileRow = kIterK + 16;                         // LDS bytes per staged row (+16: bank spread)
constexpr int kTileBytes = 16 * kTileRow;                     // per wave

// The weight matrices of one launch. Matrix s owns row groups
// [rg0[s], rg0[s+1]), its partial sums start at float offset part0[s]
// ([splits][M][n[s]]) and its outputs are reduced by blocks [rb0[s], rb0[s+1])
// of the reduce kernel.
struct SegTable {
  const uint8_t *w[kFp8MaxGroup];
  const uint16_t *scale[kFp8MaxGroup];
  uint16_t *y[kFp8MaxGroup];
  int n[kFp8MaxGroup];
  int rg0[kFp8MaxGroup + 1];
  int64_t part0[kFp8MaxGroup];
  int rb0[kFp8MaxGroup + 1];
  int count;
};

// Output tile of the prefill kernel (more than kFp8LinearMaxRows rows), below.
constexpr int kPTileM = 128;  // activation rows
constexpr int kPTileN = 128;  // output channels

// MB: 16-column batch blocks (M <= 16*MB). Workgroup b owns rows
// [rg*16*S, rg*16*S + 16*S) (S waves, 16 rows each), rg = b / splits, and
// the K slice [sp*Kc, min(K, (sp+1)*Kc)), sp = b % splits.
template <int MB>
__global__ __launch_bounds__(512) void fp8_linear_kernel(const uint8_t *__restrict__ x, SegTable seg,
                                                         float *__restrict__ part, int M, int K, int Kc, int splits) {
  extern __shared__ __align__(16) uint8_t lds[];  // [M][row_bytes] activations, then S weight tiles
  const int S = blockDim.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int rg_all = blockIdx.x / splits;
  const int sp = blockIdx.x % splits;
  int s = 0;  // the matrix this workgroup's row group belongs to (uniform per workgroup)
  while (s + 1 < seg.count && rg_all >= seg.rg0[s + 1]) ++s;
  const int rg = rg_all - seg.rg0[s];
  const int N = seg.n[s];
  const uint8_t *__restrict__ w = seg.w[s];
  const uint16_t *__restrict__ scale = seg.scale[s];
  uint16_t *__restrict__ y = seg.y[s];
  const int kb = sp * Kc;
  const int klen = min(K - kb, Kc);  // multiple of 16
  const int kpad = (klen + kIterK - 1) / kIterK * kIterK;
  const int row_bytes = kpad * 2 + 16;  // +16 spreads the 16 rows one MFMA operand load touches over all banks
  uint8_t *xs = lds;
  uint8_t *tile = lds + M * row_bytes + wave * kTileBytes;
  const int n0 = (rg * S + wave) * 16;

  // Load mapping: instruction j reads rows n0 + 4j + lane/16, bytes (lane%16)*16
  // of the iteration's 256-byte window. Rows past N read the last row.
  const int lrow = lane >> 4;
  const int lcol = (lane & 15) * kPieceBytes;
  const uint8_t *wr[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; ++j)
    wr[j] = w + static_cast<size_t>(min(n0 + j * kRowsPerLoad + lrow, N - 1)) * K + kb + lcol;

  // Two register stages: iterations it+1 and it+2 are in flight while it is
  // multiplied. A piece that starts at or past the slice end reads as zero
  // (the slice length is a multiple of 16).
  u32x4 va[kLoads], vb[kLoads];
  auto load = [&](u32x4(&v)[kLoads], int it) {
    const bool ok = it * kIterK + lcol < klen;
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      v[j] = ok ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wr[j] + it * kIterK))
                : u32x4{0u, 0u, 0u, 0u};
  };
  const int n_iter = kpad / kIterK;
  load(va, 0);
  if (n_iter > 1) load(vb, 1);

  // Stage x[0:M, kb:kb+kpad) in LDS (zero past the slice end) while the first
  // weight loads are in flight.
  const int vec_per_row = kpad / 8;
  for (int v = threadIdx.x; v < M * vec_per_row; v += blockDim.x) {
    const int m = v / vec_per_row;
    const int kk = (v - m * vec_per_row) * 8;
    u32x4 val = u32x4{0u, 0u, 0u, 0u};
    if (kk < klen) val = *reinterpret_cast<const u32x4 *>(x + (static_cast<size_t>(m) * K + kb + kk) * 2);
    *reinterpret_cast<u32x4 *>(xs + m * row_bytes + kk * 2) = val;
  }
  __syncthreads();

  const uint8_t *brow[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) brow[b] = xs + min(b * 16 + r, M - 1) * row_bytes;
  f32x4 acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One iteration: registers -> wave tile (row-contiguous), then MFMA
  // operands read back in the MFMA layout: lane (r, g) takes row r, bytes
  // s*64 + g*16 .. +15 of the window for step s.
  auto multiply = [&](const u32x4(&v)[kLoads], int it) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4 *>(tile + (j * kRowsPerLoad + lrow) * kTileRow + lcol) = v[j];
    // The tile is written and read back by different lanes of this wave:
    // order the LDS writes before the reads explicitly.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      const u32x4 a = *reinterpret_cast<const u32x4 *>(tile + r * kTileRow + st * kStepBytes + g * kPieceBytes);
      bf16x8 a_lo, a_hi;
      fp8x16_to_bf16(a, a_lo, a_hi);
      const int kk = it * kIterK + st * kStepBytes + g * kPieceBytes;
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        const u32x4 *bp = reinterpret_cast<const u32x4 *>(brow[b] + kk * 2);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_lo, as_bf16x8(bp[0]), acc[b], 0, 0, 0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_hi, as_bf16x8(bp[1]), acc[b], 0, 0, 0);
      }
    }
    // Every lane's reads of this tile come before the next iteration overwrites it.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  for (int it = 0; it < n_iter; it += 2) {
    multiply(va, it);
    if (it + 2 < n_iter) load(va, it + 2);
    if (it + 1 < n_iter) {
      multiply(vb, it + 1);
      if (it + 3 < n_iter) load(vb, it + 3);
    }
  }

  // Lane l holds rows n0 + 4*(l/16) + i, column b*16 + l%16.
  const int nb = n0 + 4 * g;
  if (part == nullptr) {  // one slice and no epilogue: the kernel writes y itself
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int m = b * 16 + r;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < N) {
          const float sc = __uint_as_float(static_cast<uint32_t>(scale[nb + i]) << 16);
          y[static_cast<size_t>(m) * N + nb + i] = f32_to_bf16_bits(acc[b][i] * sc);
        }
    }
    return;
  }
  float *__restrict__ pseg = part + seg.part0[s];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int m = b * 16 + r;
    if (m >= M) continue;
    float *dst = pseg + (static_cast<size_t>(sp) * M + m) * N + nb;
    if (nb + 3 < N) {
      *reinterpret_cast<f32x4_dword *>(dst) = acc[b];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nb + i < N) dst[i] = acc[b][i];
    }
  }
}

// y_s[i] = bf16(scale_s[i % n_s] * sum over slices of part_s[slice][i]),
// summed in slice order. Blocks [rb0[s], rb0[s+1]) reduce matrix s; each
// thread owns kReduceVec consecutive outputs and keeps up to kReduceBatch
// independent loads in flight.
//
// Epilogues fold the operation that consumes the output into the reduce, with
// the rounding of that operation run on its own in bf16 (each value rounded to
// bf16 where the separate operation would round it):
//   kFp8EpilogueSwiglu (two matrices of equal n, gate then up):
//     y_0[i] = bf16(bf16(silu(g)) * u), g = bf16(gate), u = bf16(up);
//   kFp8EpilogueResidual (one matrix): y_0[i] = bf16(residual[i] + bf16(...)).
constexpr int kReduceVec = 4;
constexpr int kReduceBatch = 8;
constexpr int kReduceThreads = 256;
// The reduce asks for kLdsToken bytes of LDS: in a streamed 70B decode, where it shared CUs with the ring copy,
// the SwiGLU reduce took 45 us (median) against 5 us alone, the q/k/v reduce 26 against 5.

// Sum over slices of kReduceVec consecutive partials starting at i0 (fewer at the end of MN).
__device__ __forceinline__ void sum_slices(const float *__restrict__ p, int64_t MN, int64_t i0, int splits,
                                           float (&acc)[kReduceVec]) {
#pragma unroll
  for (int e = 0; e < kReduceVec; ++e) acc[e] = 0.f;
  if (i0 + kReduceVec <= MN) {
    for (int p0 = 0; p0 < splits; p0 += kReduceBatch) {
      f32x4 v[kReduceBatch];
#pragma unroll
      for (int j = 0; j < kReduceBatch; ++j)
        v[j] = p0 + j < splits ? *reinterpret_cast<const f32x4_dword *>(p + (p0 + j) * MN + i0)
                               : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < kReduceBatch; ++j)
#pragma unroll
        for (int e = 0; e < kReduceVec; ++e) acc[e] += v[j][e];
    }
  } else {
    for (int q = 0; q < splits; ++q)
      for (int e = 0; e < kReduceVec; ++e)
        if (i0 + e < MN) acc[e] += p[q * MN + i0 + e];
  }
}

__global__ __launch_bounds__(kReduceThreads) void fp8_linear_reduce_kernel(const float *__restrict__ part,
                                                                           SegTable seg, int M, int splits,
                                                                           int epilogue,
                                                                           const uint16_t *__restrict__ residual) {
  int s = 0;
  while (s + 1 < seg.count && static_cast<int>(blockIdx.x) >= seg.rb0[s + 1]) ++s;
  const int N = seg.n[s];
  const int64_t MN = static_cast<int64_t>(M) * N;
  const int64_t i0 = (static_cast<int64_t>(blockIdx.x - seg.rb0[s]) * blockDim.x + threadIdx.x) * kReduceVec;
  if (i0 >= MN) return;
  const uint16_t *__restrict__ scale = seg.scale[s];
  uint16_t *__restrict__ y = seg.y[s];
  int col[kReduceVec];  // the channels of this thread's outputs (M N is at most 2^31)
  col[0] = static_cast<int>(static_cast<uint32_t>(i0) % static_cast<uint32_t>(N));
#pragma unroll
  for (int e = 1; e < kReduceVec; ++e) col[e] = col[e - 1] + 1 == N ? 0 : col[e - 1] + 1;
  float acc[kReduceVec];
  sum_slices(part + seg.part0[s], MN, i0, splits, acc);
  if (epilogue == kFp8EpilogueSwiglu) {  // s is 0: the gate; the up matrix is segment 1, same shape
    float up[kReduceVec];
    sum_slices(part + seg.part0[1], MN, i0, splits, up);
    const uint16_t *__restrict__ scale_up = seg.scale[1];
#pragma unroll
    for (int e = 0; e < kReduceVec; ++e) {
      const int64_t i = i0 + e;
      if (i < MN) {
        const float g = bf16_bits_to_f32(f32_to_bf16_bits(acc[e] * bf16_bits_to_f32(scale[col[e]])));
        const float u = bf16_bits_to_f32(f32_to_bf16_bits(up[e] * bf16_bits_to_f32(scale_up[col[e]])));
        const float act = bf16_bits_to_f32(f32_to_bf16_bits(g / (1.0f + expf(-g))));
        y[i] = f32_to_bf16_bits(act * u);
      }
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < kReduceVec; ++e) {
    const int64_t i = i0 + e;
    if (i < MN) {
      const uint16_t out = f32_to_bf16_bits(acc[e] * bf16_bits_to_f32(scale[col[e]]));
      y[i] = epilogue == kFp8EpilogueResidual
                 ? f32_to_bf16_bits(bf16_bits_to_f32(residual[i]) + bf16_bits_to_f32(out))
                 : out;
    }
  }
}

// ---- a few rows: one launch, no partial sums in memory ----------------------
//
// One workgroup of eight waves owns 16 output channels over the whole of K. The waves take turns along K
// (wave w the 256-byte windows w, w + 8, ... of every row), so the workgroup streams whole rows, and their
// sums meet in LDS in wave order at the end, where the epilogue is applied. Against the split-K kernel this
// saves the partial sums' trip through memory and the reduce launch that reads them (3.5 to 5 us a call).
// Under SwiGLU a workgroup owns the same 16 channels of gate and of up.
//
// Weights and the window of x that meets them go through per-wave LDS tiles, as the weights do in
// fp8_linear_kernel: loads cover whole rows and MFMA operands are read back in their layout. Weights are e4m3
// (with a scale per channel) or bf16 (without): a 256-byte window is 256 or 128 values of k, a 64-byte step
// two MFMAs or one. Two windows are in flight per wave and two workgroups fit a CU (one at 9 to 16 fp8 rows, whose
// tiles take 100 KB of LDS); 32 channels per workgroup read x half as often but need 140 registers, one workgroup
// per CU (28672 x 8192 fp8 in 57 against 41 us).
//
// The sum's order depends on K alone, not on the grouping or on M: a projection gives the same bits on its
// own and in a group that also runs this kernel (direct_linear_wins looks at an fp8 group's channels together).
//
// Bound by the weight bytes. Measured in a row on distinct weights, us: fp8 at 1 / 8 rows, before (split-K
// and reduce) and here: 1024 x 8192 7.7 / 8.6 and 6.6 / 8.2, 4096 x 4096 8.8 / 10.0 and 6.7 / 7.2,
// 28672 x 8192 44.0 / 48.5 and 41.5 / 45.6 (5.7 TB/s); bf16 at 1 row, the library's GEMM and here:
// 4096 x 4096 15.4 and 8.4, 11008 x 4096 26.8 and 19.2, 4096 x 11008 38.1 and 18.9, 8192 x 28672 87.6 and 75.0.
constexpr int kDirectWaves = 8;

// XL loads of 1 KB bring a window of x: 2 XL rows of 512 bytes (fp8) or 4 XL rows of 256 (bf16).
template <bool FP8, int XL, bool SWIGLU>
__global__ __launch_bounds__(kDirectWaves * kWave) void direct_linear_kernel(const uint8_t *__restrict__ x,
                                                                             SegTable seg, int M, int K,
                                                                             const uint16_t *__restrict__ residual) {
  constexpr int kWindowX = FP8 ? 2 * kIterK : kIterK;  // bytes of a row of x in one window
  constexpr int kXLanes = kWindowX / 16;               // lanes that load one row of it
  constexpr int kXRows = XL * kWave / kXLanes;
  constexpr int kXRow = kWindowX + 16;
  constexpr int kWaveBytes = kTileBytes + kXRows * kXRow;
  constexpr int kMatrices = SWIGLU ? 2 : 1;
  static_assert(kWaveBytes >= kMatrices * 256 * 4, "the waves' sums fit where the tiles were");
  __shared__ __align__(16) uint8_t lds[kDirectWaves * kWaveBytes];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  int s = 0;
  while (s + 1 < seg.count && static_cast<int>(blockIdx.x) >= seg.rg0[s + 1]) ++s;
  const int N = seg.n[s];
  const int n0 = (blockIdx.x - seg.rg0[s]) * 16;
  const int64_t row_bytes = FP8 ? K : 2 * static_cast<int64_t>(K);
  const int64_t x_bytes = 2 * static_cast<int64_t>(K);

  const int lrow = lane >> 4;
  const int lcol = (lane & 15) * kPieceBytes;
  int64_t row_at[kLoads];  // rows past N read the last row
#pragma unroll
  for (int j = 0; j < kLoads; ++j) row_at[j] = min(n0 + j * kRowsPerLoad + lrow, N - 1) * row_bytes + lcol;
  const int xrow = lane / kXLanes;
  const int xcol = lane % kXLanes * 16;
  const uint8_t *xp = x + xrow * x_bytes + xcol;
  const int windows = static_cast<int>((row_bytes + kIterK - 1) / kIterK);

  // Pieces that start at or past the end of the row read as zero (rows are whole pieces).
  auto load_w = [&](u32x4(&v)[kLoads], const uint8_t *w, int win) {
    const int64_t at = static_cast<int64_t>(win) * kIterK;
    const bool ok = at + lcol < row_bytes;
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      v[j] = ok ? __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(w + row_at[j] + at))
                : u32x4{0u, 0u, 0u, 0u};
  };
  auto load_x = [&](u32x4(&v)[XL], int win) {
    const int64_t at = static_cast<int64_t>(win) * kWindowX;
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int m = j * (kWave / kXLanes) + xrow;
      v[j] = m < M && at + xcol < x_bytes
                 ? *reinterpret_cast<const u32x4 *>(xp + j * (kWave / kXLanes) * x_bytes + at)
                 : u32x4{0u, 0u, 0u, 0u};
    }
  };
  uint8_t *tile = lds + wave * kWaveBytes;
  uint8_t *xt = tile + kTileBytes;
  // this lane's column of x: row r (columns past those loaded repeat the last one and are not stored)
  const uint8_t *xcolumn = xt + min(r, kXRows - 1) * kXRow + g * (FP8 ? 32 : 16);
  // Tiles are written and read back by different lanes of this wave: order each side's accesses explicitly.
  auto order = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  auto stage_x = [&](const u32x4(&v)[XL]) {
#pragma unroll
    for (int j = 0; j < XL; ++j)
      *reinterpret_cast<u32x4 *>(xt + (j * (kWave / kXLanes) + xrow) * kXRow + xcol) = v[j];
  };
  auto multiply = [&](const u32x4(&v)[kLoads], f32x4 &acc) {
#pragma unroll
    for (int j = 0; j < kLoads; ++j)
      *reinterpret_cast<u32x4 *>(tile + (j * kRowsPerLoad + lrow) * kTileRow + lcol) = v[j];
    order();
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      const u32x4 a = *reinterpret_cast<const u32x4 *>(tile + r * kTileRow + st * kStepBytes + g * kPieceBytes);
      const u32x4 *xv = reinterpret_cast<const u32x4 *>(xcolumn + st * (kWindowX / kSteps));
      if (FP8) {
        bf16x8 lo, hi;
        fp8x16_to_bf16(a, lo, hi);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, as_bf16x8(xv[0]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, as_bf16x8(xv[1]), acc, 0, 0, 0);
      } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(xv[0]), acc, 0, 0, 0);
      }
    }
    order();
  };

  f32x4 acc[kMatrices];
#pragma unroll
  for (int b = 0; b < kMatrices; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint8_t *w = seg.w[s];
  u32x4 wa[kLoads], wb[kLoads], xa[XL], xb[XL];
  if (SWIGLU) {  // a window of gate and the same one of up in flight; x serves both
    const uint8_t *up = seg.w[1];
    if (wave < windows) {
      load_w(wa, w, wave);
      load_x(xa, wave);
      load_w(wb, up, wave);
    }
    for (int win = wave; win < windows; win += kDirectWaves) {
      const bool more = win + kDirectWaves < windows;
      stage_x(xa);
      multiply(wa, acc[0]);
      if (more) {
        load_w(wa, w, win + kDirectWaves);
        load_x(xa, win + kDirectWaves);
      }
      multiply(wb, acc[kMatrices - 1]);
      if (more) load_w(wb, up, win + kDirectWaves);
    }
  } else {
    if (wave < windows) {
      load_w(wa, w, wave);
      load_x(xa, wave);
    }
    if (wave + kDirectWaves < windows) {
      load_w(wb, w, wave + kDirectWaves);
      load_x(xb, wave + kDirectWaves);
    }
    for (int win = wave; win < windows; win += 2 * kDirectWaves) {
      stage_x(xa);
      multiply(wa, acc[0]);
      if (win + 2 * kDirectWaves < windows) {
        load_w(wa, w, win + 2 * kDirectWaves);
        load_x(xa, win + 2 * kDirectWaves);
      }
      if (win + kDirectWaves < windows) {
        stage_x(xb);
        multiply(wb, acc[0]);
        if (win + 3 * kDirectWaves < windows) {
          load_w(wb, w, win + 3 * kDirectWaves);
          load_x(xb, win + 3 * kDirectWaves);
        }
      }
    }
  }

  // Lane l holds channels 4 (l / 16) .. + 3 of column l % 16 of each matrix.
  __syncthreads();  // the last tiles have been read
  float *sums = reinterpret_cast<float *>(lds);  // [wave][matrix][column][channel]
#pragma unroll
  for (int b = 0; b < kMatrices; ++b)
    *reinterpret_cast<f32x4 *>(sums + ((wave * kMatrices + b) * 16 + r) * 16 + 4 * g) = acc[b];
  __syncthreads();
  const int t = threadIdx.x;
  const int m = t / 16;
  const int n = n0 + t % 16;
  if (m >= M || n >= N) return;
  auto output = [&](int matrix, int at) {  // M <= 16, so t < 256
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < kDirectWaves; ++q) v += sums[q * kMatrices * 256 + at];
    return f32_to_bf16_bits(FP8 ? v * bf16_bits_to_f32(seg.scale[matrix][n]) : v);
  };
  const int64_t i = static_cast<int64_t>(m) * N + n;
  if (SWIGLU) {  // the epilogues round as fp8_linear_reduce_kernel's do
    const float gate = bf16_bits_to_f32(output(0, t));
    const float up = bf16_bits_to_f32(output(1, t + 256));
    const float act = bf16_bits_to_f32(f32_to_bf16_bits(gate / (1.0f + expf(-gate))));
    seg.y[0][i] = f32_to_bf16_bits(act * up);
    return;
  }
  const uint16_t out = output(s, t);
  seg.y[s][i] = residual ? f32_to_bf16_bits(bf16_bits_to_f32(residual[i]) + bf16_bits_to_f32(out)) : out;
}

SegTable seg_table(const Fp8LinearLaunch &p) {
  SegTable t{};
  t.count = p.group;
  const int64_t rows = p.prefill ? p.tile_n : 16 * static_cast<int64_t>(p.waves);  // of one workgroup
  int rg = 0, rb = 0;
  int64_t off = 0;
  for (int s = 0; s < p.group; ++s) {
    t.w[s] = static_cast<const uint8_t *>(p.w[s]);
    t.scale[s] = static_cast<const uint16_t *>(p.scale[s]);
    t.y[s] = static_cast<uint16_t *>(p.y[s]);
    t.n[s] = static_cast<int>(p.n[s]);
    t.rg0[s] = rg;
    t.part0[s] = off;
    t.rb0[s] = rb;
    rg += static_cast<int>((p.n[s] + rows - 1) / rows);
    off += static_cast<int64_t>(p.splits) * p.m * p.n[s];
    rb += static_cast<int>((p.m * p.n[s] + kReduceVec * kReduceThreads - 1) / (kReduceVec * kReduceThreads));
  }
  t.rg0[p.group] = rg;
  t.rb0[p.group] = rb;
  return t;
}

// ---- prefill: inputs of more than kFp8LinearMaxRows rows -------------------
//
// Many activation rows make the layer a compute-bound GEMM. This is a tiled
// MFMA GEMM that still reads the weights as fp8 and widens them in registers
// (no bf16 copy of the weights is ever written).
//
// Workgroup tile: 128 output channels x 128 activation rows, K in steps of 64.
// Each step's tiles go straight from global memory into an S-stage LDS ring
// with global_load_lds_dwordx4 (no register staging): the activation tile as
// 128 rows of 128 bytes, then the weight tile as 128 rows of 64 bytes. Each
// load instruction writes 1 KB of LDS, lane l at +16 l, so the layout is
// chosen by which global chunk each lane fetches:
//   activation row R, 16-byte chunk c (k = 8c..8c+7) at slot c ^ rot3(R & 7),
//     rot3(v) = (v & 3) << 1 | v >> 2 (a rotation of the row's low three bits),
//   weight row R,     16-byte chunk c (k = 16c..16c+15) at slot c ^ ((R >> 1) & 3).
// Both keep the MFMA operand reads below (ds_read_b128, 1 KB per wave) free
// of bank conflicts on gfx950: 6 LDS cycles per read, measured with the
// SQ_LDS_BANK_CONFLICT counter. The plain c ^ (R & 7) for the activations
// costs 8, two of them bank-conflict cycles.
//
// k permutation within a step (any one that both operands share gives the
// same sum): lane group g feeds k = 16g + 8kb + (0..7) to the kb-th of the
// step's two MFMAs, so one 16-byte weight read per lane covers both MFMAs.
//
// Two launch shapes of 128 x 128 tiles, chosen by the planner (measured on the 70B projection
// shapes at 512 rows):
//   * more tiles than CUs: 4 waves (2 x 2, 64 x 64 each), 2 stages (48 KB
//     LDS, three workgroups per CU);
//   * at most one tile per CU: 8 waves (2 x 4, 64 x 32 each), 4 stages
//     (96 KB, one workgroup per CU), so two waves share each SIMD; waves 0-3
//     issue the loads (all eight issuing them measured slower, by 5% to 50%
//     over runs).
// Both accumulate every output over the same MFMA sequence, so they give
// identical results.
//
// Rows past M or N read the last valid row (their products land in outputs
// that are never stored). A K that is not a multiple of 64 ends in a partial
// step: its loads past K are clamped into the row and both operands are
// zeroed for the lane groups past K.
//
// Block order: the hardware hands workgroup b to XCD b % xcds. An XCD walks up to kPBand m-tiles of one n-tile,
// then the same m-tiles of its next one, so weight tiles come from its L2 for the band's other m-tiles and the
// band's activations for its other n-tiles. us in bands and not: 4096 x 8192 of 4096 rows 231 and 298, 28672 x 528
// of 2048 rows 109.5 and 134.6, 2056 x 4112 of 4096 rows 96.2 and 112.8. Calls of up to 16 m-tiles and a short K
// whose tiles are resident nearly all at once walk whole columns: 8200 x 1024 of 1500 rows 37.2 and 35.3, 2056 x
// 1024 of 2048 rows 20.6 and 18.9 (28672 x 1024 of 1500 rows, 3.5 rounds: 109.8 and 119.7).
//
// Its n-tiles are every xcds-th one where tiles outnumber the CUs (4 waves: 577 x 23553 x 10224 368 us, in runs
// 388). Calls of at most one tile per CU and 64-row tiles give each XCD an equal run of tiles, since a CU that gets
// two of them doubles the time: of 17 n-tiles dealt in turn one XCD has 3 and the others 2 (887 rows x 2125 x 10064,
// 64-row tiles: 86.1 us dealt, 67.7 in runs). 8-wave calls whose uneven deal still fits one tile per CU are dealt:
// 129 rows x 11520 x 21456 187 us against 202, 1024 x 2056 x 528 11.2 against 11.7 (a whole number of n-tiles per
// XCD, 385 x 8192 x 8192: 67.9 dealt, 66.2 in runs).
//
// An XCD's spare workgroups come last: between its tiles they left CUs with none beside CUs with two (2048 rows x
// 2056 x 1024: 21.2 us, 18.7 with them last).
constexpr int kPTileK = 64;
constexpr int kPBand = 8;                            // m-tiles of a band

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ bf16x8 fp8x8_to_bf16(uint32_t w0, uint32_t w1) {
  const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false);
  const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true);
  const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false);
  const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true);
  return join8(p0, p1, p2, p3);
}

// Activation-tile swizzle: rotate a row's low three bits (see the layout above).
__device__ __forceinline__ int rot3(int v) { return ((v & 3) << 1) | ((v >> 2) & 1); }

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt left free).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N < 64, "vmcnt holds six bits");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}

// Workgroup barrier that also keeps the compiler from moving memory accesses
// across it; the LDS ring's ordering is carried by vmcnt waits and this.
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS reads are done
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// seg.rg0 holds each matrix's first n-tile (tiles of kPTileN output channels).
// SADDR: the activations and every weight matrix are under 2 GiB, so each load
// takes a scalar base (the matrix plus the step's K offset) and a per-lane
// 32-bit offset, and the loading wave's LDS address is scalar arithmetic: the
// per-step address work leaves the vector ALU (about 3% per layer, measured).
//
// Tiles are TM activation rows x TN channels. The smaller ones serve calls that leave the chip idle otherwise
// (plan_fp8_linear) and the batches between decode and prefill (mid_linear_wins); those also split K: workgroup sp
// of a tile takes the steps from sp * split_steps and writes fp32 sums for fp8_linear_reduce_kernel. At 64 x 128
// four waves of 32 channels x 64 rows, four stages of 16 KB, two workgroups per CU; bound by the weights' bytes
// (28672 x 8192 at 64 rows: 70.8 us, 3.3 TB/s). Five and eight stages, four steps at least per split and three
// workgroups per CU were within 5% or slower.
template <int TM, int TN, int WAVES, int S, bool SADDR, bool DEAL>
__global__ __launch_bounds__(WAVES * 64, TM == 128 && WAVES == 4 ? 3 : 2) void fp8_prefill_kernel(
    const uint8_t *__restrict__ x, SegTable seg, int M, int K, int m_tiles, int n_tiles, int xcds,
    int splits_or_band, int split_steps, float *__restrict__ part) {
  // 64-row tiles: how often K is split; dealt tiles: m-tiles of a band
  const int splits = splits_or_band, band = splits_or_band;
  static_assert(TM == 128 ? TN == 128 && (WAVES == 4 || WAVES == 8) : TM == 64 && WAVES == 4, "4 or 8 waves");
  constexpr int WN = TM == 64 && TN == 128 ? 4 : 2;       // waves side by side along the channels
  constexpr int IT = TN / WN / 16;                        // 16-channel weight tiles per wave
  constexpr int JT = TM / (WAVES / WN) / 16;              // 16-row activation tiles per wave
  constexpr int WROWS = 16 * JT;                   // activation rows per wave
  constexpr int kXStage = TM * kPTileK * 2;
  constexpr int kStage = kXStage + TN * kPTileK;
  constexpr int XL = TM / 32, WL = TN / 64;        // activation and weight loads per loading wave and step
  __shared__ __align__(1024) uint8_t lds[S * kStage];
  const int xcd = blockIdx.x % xcds;
  const int slot = blockIdx.x / xcds;
  // The block order described above; workgroups past an XCD's tiles come last.
  int mt, nt, sp = 0;
  if constexpr (DEAL) {
    if (WAVES == 8 || m_tiles <= band) {
      mt = slot % m_tiles;
      nt = slot / m_tiles * xcds + xcd;
    } else {
      const int n_own = (n_tiles - xcd + xcds - 1) / xcds;
      if (slot >= m_tiles * n_own) return;
      const int first = slot / (band * n_own) * band;
      const int at = slot - first * n_own;
      const int rows = min(band, m_tiles - first);
      mt = first + at % rows;
      nt = at / rows * xcds + xcd;
    }
    if (nt >= n_tiles) return;
  } else {
    const int items = m_tiles * n_tiles * (TM == 128 ? 1 : splits);
    const int per_xcd = (items + xcds - 1) / xcds;
    const int item = xcd * per_xcd + slot;
    if (slot >= per_xcd || item >= items) return;  // the last run may be shorter
    sp = TM == 128 ? 0 : item % splits;
    const int tile = TM == 128 ? item : item / splits;
    const int run = tile / (kPBand * n_tiles);
    const int at = tile - run * kPBand * n_tiles;
    const int rows = min(kPBand, m_tiles - run * kPBand);
    mt = run * kPBand + at % rows;
    nt = at / rows;
  }
  int s = 0;
  while (s + 1 < seg.count && nt >= seg.rg0[s + 1]) ++s;
  const int N = seg.n[s];
  const uint8_t *__restrict__ w = seg.w[s];
  const int n_base = (nt - seg.rg0[s]) * TN;
  const int m_base = mt * TM;

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int wn = wave % WN;
  const int wm = wave / WN;
  const bool loads = WAVES == 4 || wave < 4;
  const int lw = __builtin_amdgcn_readfirstlane(wave & 3);  // uniform: LDS destinations stay scalar

  // This lane's load sources: activation rows (lw*XL + t)*8 + lane/8, weight
  // rows (lw*WL + t)*16 + lane/4, at the chunk the swizzle assigns.
  const int xc = ((lane & 7) ^ rot3(lane >> 3)) * 8;        // k offset (elements) within a step
  const int wc = ((lane & 3) ^ ((lane >> 3) & 3)) * 16;     // k offset (bytes) within a step
  const uint8_t *xrow[4];  // XL of them
  const uint8_t *wrow[2];  // WL of them
  uint32_t xoff[4], woff[2];  // SADDR: byte offsets of this lane's chunk in step 0
#pragma unroll
  for (int t = 0; t < XL; ++t) {
    const int gm = min(m_base + (lw * XL + t) * 8 + (lane >> 3), M - 1);
    xrow[t] = x + static_cast<size_t>(gm) * K * 2;
    xoff[t] = static_cast<uint32_t>((static_cast<size_t>(gm) * K + xc) * 2);
  }
#pragma unroll
  for (int t = 0; t < WL; ++t) {
    const int gn = min(n_base + (lw * WL + t) * 16 + (lane >> 2), N - 1);
    wrow[t] = w + static_cast<size_t>(gn) * K;
    woff[t] = static_cast<uint32_t>(static_cast<size_t>(gn) * K + wc);
  }
  const int full = K / kPTileK;                 // whole steps
  const int tail = K % kPTileK;                 // k values of a final partial step, a multiple of 16
  const int first = TM == 128 ? 0 : sp * split_steps;
  const int steps = TM == 128 ? full + (tail ? 1 : 0) : min(full + (tail ? 1 : 0), first + split_steps);
  auto issue = [&](int st) {
    uint8_t *base = lds + (st % S) * kStage;
    if (SADDR && st < full) {  // whole step: scalar base, per-lane offsets fixed for the whole kernel
      const uint8_t *xb = x + static_cast<size_t>(st) * kPTileK * 2;
      const uint8_t *wb = w + static_cast<size_t>(st) * kPTileK;
#pragma unroll
      for (int t = 0; t < XL; ++t)
        __builtin_amdgcn_global_load_lds(xb + xoff[t], (lds_void *)(base + (lw * XL + t) * 1024), 16, 0, 0);
#pragma unroll
      for (int t = 0; t < WL; ++t)
        __builtin_amdgcn_global_load_lds(wb + woff[t], (lds_void *)(base + kXStage + (lw * WL + t) * 1024), 16, 0,
                                         0);
      return;
    }
    // the clamps only bind in a partial step (a whole step ends at K - 8 and K - 16)
    const int kx = min(st * kPTileK + xc, K - 8);
    const int kw = min(st * kPTileK + wc, K - 16);
    if (SADDR) {  // the same 32-bit offsets, moved by the clamped k
#pragma unroll
      for (int t = 0; t < XL; ++t)
        __builtin_amdgcn_global_load_lds(x + (xoff[t] + static_cast<uint32_t>(kx - xc) * 2),
                                         (lds_void *)(base + (lw * XL + t) * 1024), 16, 0, 0);
#pragma unroll
      for (int t = 0; t < WL; ++t)
        __builtin_amdgcn_global_load_lds(w + (woff[t] + static_cast<uint32_t>(kw - wc)),
                                         (lds_void *)(base + kXStage + (lw * WL + t) * 1024), 16, 0, 0);
      return;
    }
#pragma unroll
    for (int t = 0; t < XL; ++t)
      __builtin_amdgcn_global_load_lds(xrow[t] + static_cast<size_t>(kx) * 2,
                                       (lds_void *)(base + (lw * XL + t) * 1024), 16, 0, 0);
#pragma unroll
    for (int t = 0; t < WL; ++t)
      __builtin_amdgcn_global_load_lds(wrow[t] + kw, (lds_void *)(base + kXStage + (lw * WL + t) * 1024), 16, 0,
                                       0);
  };

  int aoff[IT], boff0[JT], boff1[JT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int R = wn * (16 * IT) + i * 16 + r;
    aoff[i] = kXStage + R * kPTileK + ((g ^ ((R >> 1) & 3)) << 4);
  }
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    const int R = wm * WROWS + j * 16 + r;
    boff0[j] = R * 128 + (((2 * g) ^ rot3(R & 7)) << 4);
    boff1[j] = R * 128 + (((2 * g + 1) ^ rot3(R & 7)) << 4);
  }

  f32x4 acc[IT][JT];
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // 16-row blocks of this wave that hold a row below M
  const int live = __builtin_amdgcn_readfirstlane(min(JT, max(0, (M - m_base - wm * WROWS + 15) / 16)));

  if (loads) {
#pragma unroll
    for (int st = 0; st < S - 1; ++st)
      if (first + st < steps) issue(first + st);
  }
  // One step: this wave's loads of step st are in LDS once at most the later
  // steps' loads are outstanding; the barrier then covers every loading wave,
  // and every wave has finished reading the buffer the next loads overwrite.
  // `partial` (the final step of a K that is not a multiple of 64) zeroes both
  // operands of the lane groups past K.
  auto step = [&](auto blocks, int st, bool partial) {
    if (loads) {
      if (st + S - 2 < steps)
        wait_vmcnt<(S - 2) * (XL + WL)>();
      else
        wait_vmcnt<0>();
    }
    ring_barrier();
    if (loads && st + S - 1 < steps) issue(st + S - 1);
    const uint8_t *sb = lds + (st % S) * kStage;
    constexpr int J = decltype(blocks)::value;
    if constexpr (J == 0) return;
    u32x4 A[IT], B0[J + 1], B1[J + 1];  // one spare: J may be 0
#pragma unroll
    for (int i = 0; i < IT; ++i) A[i] = *reinterpret_cast<const u32x4 *>(sb + aoff[i]);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      B0[j] = *reinterpret_cast<const u32x4 *>(sb + boff0[j]);
      B1[j] = *reinterpret_cast<const u32x4 *>(sb + boff1[j]);
    }
    if (partial && 16 * g >= tail) {
#pragma unroll
      for (int i = 0; i < IT; ++i) A[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < J; ++j) B0[j] = B1[j] = u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const bf16x8 a0 = fp8x8_to_bf16(A[i][0], A[i][1]);
      const bf16x8 a1 = fp8x8_to_bf16(A[i][2], A[i][3]);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, as_bf16x8(B0[j]), acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, as_bf16x8(B1[j]), acc[i][j], 0, 0, 0);
      }
    }
  };
  // The walk along K for J blocks of 16 rows: fewer than JT in the last tile of the rows, whose blocks past M
  // hold nothing. Each count has a loop of its own (a choice inside the loop costs 70 registers), and every
  // loop meets the same barriers.
  auto walk = [&](auto blocks) {
    for (int st = first; st < min(full, steps); ++st) step(blocks, st, false);
    if (tail && steps > full) step(blocks, full, true);
  };
  switch (live) {
    case 0: walk(std::integral_constant<int, 0>{}); break;
    case 1: walk(std::integral_constant<int, 1>{}); break;
    case 2: walk(std::integral_constant<int, JT < 2 ? JT : 2>{}); break;
    case 3: walk(std::integral_constant<int, JT < 3 ? JT : 3>{}); break;
    default: walk(std::integral_constant<int, JT>{}); break;
  }

  if (TM != 128 && part != nullptr) {
    float *__restrict__ pseg = part + seg.part0[s] + static_cast<size_t>(sp) * M * N;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int nb = n_base + wn * (16 * IT) + i * 16 + 4 * g;
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        const int m = wm * WROWS + j * 16 + r;
        if (m >= M) continue;
        float *dst = pseg + static_cast<size_t>(m) * N + nb;
        if (nb + 3 < N) {
          *reinterpret_cast<f32x4_dword *>(dst) = acc[i][j];
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nb + v < N) dst[v] = acc[i][j][v];
        }
      }
    }
    return;
  }
  const uint16_t *__restrict__ scale = seg.scale[s];
  uint16_t *__restrict__ y = seg.y[s];
  const bool vec = (N & 3) == 0;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int nb = n_base + wn * (16 * IT) + i * 16 + 4 * g;
    float sc[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) sc[v] = nb + v < N ? __uint_as_float(static_cast<uint32_t>(scale[nb + v]) << 16) : 0.f;
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const int m = m_base + wm * WROWS + j * 16 + r;
      if (m >= M) continue;
      uint16_t *dst = y + static_cast<size_t>(m) * N + nb;
      if (vec && nb + 3 < N) {
        const uint32_t lo = f32_to_bf16_bits(acc[i][j][0] * sc[0]) |
                            (static_cast<uint32_t>(f32_to_bf16_bits(acc[i][j][1] * sc[1])) << 16);
        const uint32_t hi = f32_to_bf16_bits(acc[i][j][2] * sc[2]) |
                            (static_cast<uint32_t>(f32_to_bf16_bits(acc[i][j][3] * sc[3])) << 16);
        *reinterpret_cast<u32x2 *>(dst) = u32x2{lo, hi};
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (nb + v < N) dst[v] = f32_to_bf16_bits(acc[i][j][v] * sc[v]);
      }
    }
  }
}

// ---- measurement: the sustained MFMA rate -------------------------------
//
// Each wave keeps 16 independent accumulators and cycles through 8 operand
// pairs of random bf16 values (finite, magnitude 0.5 to 4, from a hash of the
// lane), so the operands change from one MFMA to the next as in a GEMM; the
// MFMA pipe runs at a lower clock on changing data than on constant data.
// Writes nothing: sink is written only if the sum equals a fixed sentinel.
__device__ __forceinline__ uint32_t probe_hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

__global__ __launch_bounds__(256) void mfma_probe_kernel(float *sink, int iters) {
  const uint32_t id = blockIdx.x * 256u + threadIdx.x;
  u32x4 av[8], bv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t h = probe_hash(id * 64u + e * 8u + q);
      const uint32_t h2 = probe_hash(h);
      // two bf16 per dword: sign, exponent 126..129, 7 mantissa bits
      auto bf = [](uint32_t r) { return ((r & 1u) << 15) | ((126u + ((r >> 1) & 3u)) << 7) | ((r >> 3) & 0x7fu); };
      av[e][q] = bf(h) | (bf(h >> 10) << 16);
      bv[e][q] = bf(h2) | (bf(h2 >> 10) << 16);
    }
  }
  f32x4 acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(av[(i + h) & 7]), as_bf16x8(bv[(3 * i + h) & 7]),
                                                         acc[i], 0, 0, 0);
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) sum += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
  if (sum == 1234.5f) sink[0] = sum;
}

// The same probe on v_mfma_f32_32x32x16_bf16 (32768 flops each): 8
// independent accumulators per wave, 16 MFMAs per iteration, so an iteration
// has the flops of the 16 x 16 probe's. It reads half the operand registers
// per flop, and on changing data it sustains a higher rate.
__global__ __launch_bounds__(256) void mfma_probe_32x32_kernel(float *sink, int iters) {
  const uint32_t id = blockIdx.x * 256u + threadIdx.x;
  u32x4 av[8], bv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t h = probe_hash(id * 64u + e * 8u + q);
      const uint32_t h2 = probe_hash(h);
      auto bf = [](uint32_t r) { return ((r & 1u) << 15) | ((126u + ((r >> 1) & 3u)) << 7) | ((r >> 3) & 0x7fu); };
      av[e][q] = bf(h) | (bf(h >> 10) << 16);
      bv[e][q] = bf(h2) | (bf(h2 >> 10) << 16);
    }
  }
  f32x16 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(av[(i + h) & 7]), as_bf16x8(bv[(3 * i + h) & 7]),
                                                         acc[i], 0, 0, 0);
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) sum += acc[i][e];
  if (sum == 1234.5f) sink[0] = sum;
}

hipError_t launch_reduce(const Fp8LinearLaunch &p, const SegTable &seg, hipStream_t stream) {
  // the SwiGLU epilogue writes one output per gate/up pair: the gate's blocks only
  const int blocks = p.epilogue == kFp8EpilogueSwiglu ? seg.rb0[1] : seg.rb0[p.group];
  hipLaunchKernelGGL(fp8_linear_reduce_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kReduceThreads),
                     kLdsToken, stream, static_cast<const float *>(p.workspace), seg, static_cast<int>(p.m),
                     p.splits, p.epilogue, static_cast<const uint16_t *>(p.residual));
  return hipGetLastError();
}

template <int MB>
hipError_t launch_mb(const Fp8LinearLaunch &p, hipStream_t stream) {
  const SegTable seg = seg_table(p);
  const bool reduce = p.scratch_bytes > 0;  // split K, or an epilogue: partials, then the reduce kernel
  hipLaunchKernelGGL((fp8_linear_kernel<MB>), dim3(static_cast<unsigned>(p.grid)), dim3(p.waves * kWave),
                     p.lds_bytes, stream, static_cast<const uint8_t *>(p.x), seg,
                     reduce ? static_cast<float *>(p.workspace) : nullptr, static_cast<int>(p.m), static_cast<int>(p.k),
                     static_cast<int>(p.kc), p.splits);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || !reduce) return err;
  return launch_reduce(p, seg, stream);
}

}  // namespace

namespace {

// Whether 32-bit load offsets reach every byte of x and of each weight matrix (kept under 2^31, so they read
// the same whether the hardware widens the offset as signed or unsigned).
bool offsets_fit(const Fp8LinearLaunch &p) {
  bool fit = static_cast<uint64_t>(p.m) * p.k * 2 < (uint64_t(1) << 31);
  for (int s = 0; s < p.group; ++s) fit = fit && static_cast<uint64_t>(p.n[s]) * p.k < (uint64_t(1) << 31);
  return fit;
}

}  // namespace

Fp8LinearLaunch plan_fp8_linear(int64_t m, const int64_t *n, int group, int64_t k, int cus, int xcds, int waves,
                                int kc_override, int epilogue) {
  Fp8LinearLaunch p{};
  p.epilogue = epilogue;
  p.m = m;
  p.k = k;
  p.group = group;
  for (int s = 0; s < group; ++s) {
    p.n[s] = n[s];
    p.n_total += n[s];
  }
  if (m > kFp8LinearMaxRows) {
    // prefill: one workgroup per 128 x 128 output tile, whole K, no workspace
    p.prefill = true;
    p.splits = 1;
    p.kc = k;
    p.xcds = std::max(1, xcds);
    const int64_t m_tiles = (m + kPTileM - 1) / kPTileM;
    int64_t n_tiles = 0;
    for (int s = 0; s < group; ++s) n_tiles += (n[s] + kPTileN - 1) / kPTileN;
    p.m_tiles = m_tiles;
    p.row_groups = n_tiles;
    // at most one tile per CU: 8 waves (two per SIMD) and 4 LDS stages in one
    // workgroup; more tiles: 4 waves and 2 stages, three workgroups per CU
    p.waves = (waves == 4 || waves == 8) ? waves : (m_tiles * n_tiles <= cus ? 8 : 4);
    const int64_t dealt = m_tiles * ((n_tiles + p.xcds - 1) / p.xcds);  // the most tiles of an XCD
    p.deal = p.waves == 4 || (n_tiles % p.xcds && dealt <= cus / p.xcds);
    p.grid = p.xcds * (p.deal ? dealt : (m_tiles * n_tiles + p.xcds - 1) / p.xcds);
    // no bands where the tiles of a short K are all resident in a round and a half (three to a CU)
    p.band = m_tiles <= 2 * kPBand && k <= 2048 && dealt * 2 * p.xcds <= 9 * cus ? static_cast<int>(m_tiles) : kPBand;
    p.small = offsets_fit(p);
    p.tile_n = kPTileN;
    // Half of the chip or more would be idle: 64 x 128 tiles, and 64 x 64 while those leave half idle too. A
    // tile's time is its steps of K one after the other, so smaller tiles end sooner as well. us, 128 x 128
    // tiles, 64 x 128 and 64 x 64 at k = 8192: 100 rows x 8192 64.6, 58.3, 48.0; 512 x 1024 62.3, 54.8, 44.3;
    // 200 x 8192 67.2, 60.4, (58.3); with more tiles than that, 512 x 8192 (256 of 128 x 128) 73.2 and 75.8.
    // Eight stages instead of four: 49.2 against 48.0.
    if (!waves && m_tiles * n_tiles * 2 <= cus) {
      p.mid = true;
      p.waves = 4;
      p.kc = (k + kPTileK - 1) / kPTileK * kPTileK;
      p.m_tiles = (m + 63) / 64;
      p.tile_n = p.m_tiles * n_tiles * 2 <= cus ? 64 : 128;
      p.row_groups = 0;
      for (int s = 0; s < group; ++s) p.row_groups += (n[s] + p.tile_n - 1) / p.tile_n;
      p.deal = false;
      p.band = kPBand;
      p.grid = p.xcds * ((p.m_tiles * p.row_groups + p.xcds - 1) / p.xcds);
    }
    return p;
  }
  p.batch_blocks = static_cast<int>((m + 15) / 16);
  // LDS: m activation rows of (2*Kc + 16) bytes plus one weight tile per
  // wave, within kFp8LinearMaxLds (less a margin for the kernel's own flag).
  const int64_t budget = static_cast<int64_t>(kFp8LinearMaxLds) - 256;
  const int64_t kblocks = std::max<int64_t>(1, (k + kIterK - 1) / kIterK);
  p.waves = waves ? waves : 8;
  int64_t min_slice_blocks = 4;
  if (!waves && !kc_override && ((p.n_total + 127) / 128) * std::max<int64_t>(1, kblocks / 4) < 2 * cus) {
    // Narrow outputs (the 1024-channel k/v projections of a 70B layer) give
    // fewer than two workgroups per CU at 8 waves and 4-iteration slices;
    // 4 waves and 2-iteration slices give four times as many (7.1 against
    // 9.3 us for 1024 x 8192 at 8 rows, measured).
    p.waves = 4;
    min_slice_blocks = 2;
  }
  while (p.waves > 1 && m * (2 * kIterK + 16) + static_cast<int64_t>(p.waves) * kTileBytes > budget) --p.waves;
  const int64_t rows = 16 * static_cast<int64_t>(p.waves);
  int64_t row_groups = 0;
  for (int s = 0; s < group; ++s) row_groups += (n[s] + rows - 1) / rows;
  const int64_t tiles = static_cast<int64_t>(p.waves) * kTileBytes;
  const int64_t x_budget = budget - tiles;
  const int64_t lds_blocks = std::max<int64_t>(1, ((x_budget / m - 16) / 2) / kIterK);
  int64_t kc_blocks;
  if (kc_override) {
    kc_blocks = std::max<int64_t>(1, kc_override / kIterK);
  } else {
    // Aim for at least 4 workgroups per CU, with slices of at least
    // min_slice_blocks iterations.
    const int64_t want_splits = std::max<int64_t>(1, (4 * static_cast<int64_t>(cus) + row_groups - 1) / row_groups);
    kc_blocks = std::max<int64_t>(std::min<int64_t>(min_slice_blocks, kblocks),
                                  (kblocks + want_splits - 1) / want_splits);
  }
  kc_blocks = std::min(std::min(kc_blocks, kblocks), lds_blocks);
  p.splits = static_cast<int>((kblocks + kc_blocks - 1) / kc_blocks);
  p.kc = kc_blocks * kIterK;
  p.grid = row_groups * p.splits;
  p.row_groups = row_groups;
  p.lds_bytes = static_cast<size_t>(m) * (2 * p.kc + 16) + static_cast<size_t>(tiles);
  // partials when K is split, and always under an epilogue (the reduce kernel applies it)
  p.workspace_bytes = p.splits > 1 || epilogue != kFp8EpilogueNone
                          ? static_cast<size_t>(p.splits) * m * p.n_total * sizeof(float)
                          : 0;
  p.scratch_bytes = p.workspace_bytes;
  return p;
}

// Where the one-launch kernel is the faster one: both it and the plan of plan_fp8_linear measured at 1, 3, 4, 8, 9
// and 16 rows of K = 512 .. 28672 and 512 .. 131072 channels, plain and under SwiGLU (1580 calls, graph replays on
// distinct weights). Ratios below are its time by the other's; its line is crossed by 6% at most at 9 of them.
//
//  * Short K, many channels: a workgroup's 16 channels give its eight waves K / 2048 windows each (twice that under
//    SwiGLU, hence `depth`), so launching, filling and summing it is most of its time, once per 16 channels, while
//    wide plans of one K slice pay no reduce. At 8 rows 8192 x 512 0.70 and 10240 x 512 1.15; 22016 x 1024 0.91 and
//    45056 x 1024 1.07 (131072: 1.74); 28672 x 2048 1.00 and 45056 x 2048 1.10; 45056 x 4096 1.02 and 65536 x 4096
//    1.05 (1.15 at 4 rows); 65536 x 5120 and all longer ones below 1.02. One or two rows stage less of x: 65536 x
//    2048 1.00, 131072 x 2048 1.16.
//  * Long K, few channels: one workgroup walks the whole of K, on each of a few CUs. At 4 rows 1024 x 11008 0.89,
//    512 x 11008 1.05, 2048 x 16384 0.94, 1024 x 16384 1.07, 3072 x 28672 0.99, 2048 x 28672 1.25.
//  * 5 to 8 rows of a longer K: 8192 x 28672 at 8 rows in 48.1 us against 45.1.
//  * 9 to 16 rows take 100 KB of LDS, one workgroup per CU, and read as much of x as of the weights from L2: small
//    matrices only. At 9 rows 8192 x 4096 0.97 and 10240 x 4096 1.13, 12288 x 1024 0.92 and 14336 x 1024 1.10, under
//    SwiGLU 12288 x 512 0.97 and 14336 x 512 1.14; at 16 rows 2048 x 11008 0.91 and 1024 x 11008 1.09.
//
// bf16 weights are twice the bytes for the same x, and their only other kernel is the library's GEMM: faster for
// wide matrices of a short K only, which callers leave to it (hip.bf16_linear_eligible). us at 1 / 8 / 16 rows, here
// and the library: 4096 x 4096 8.4 / 8.5 / 9.4 and 15.4 / 15.6 / 15.5; 11008 x 4096 17.4 / 18.0 / 20.3 and 26.7 /
// 25.7 / 25.6; 32000 x 4096 (a head) 42.2 / 42.1 / 47.8 and 58.9 / 56.8 / 56.9; 128256 x 4096 157 / 156 / 179 and
// 182 / 184 / 186; 8192 x 28672 71.7 / 74.7 / 85.1 and 85.9 / 86.5 / 87.9; closest 1024 x 8192 at 16 rows, 12.0 and
// 12.1.
bool direct_linear_wins(int64_t m, int64_t n_total, int64_t k, int epilogue) {
  if (m > kDirectMaxRows || n_total > kDirectMaxChannels) return false;
  const int64_t matrices = epilogue == kFp8EpilogueSwiglu ? 2 : 1;  // of a workgroup
  const int64_t channels = n_total / matrices;                      // 16 of them to a workgroup
  if (m > 8)
    return n_total * k <= int64_t(48) << 20 &&
           channels <= (matrices == 2 || (k >= 1024 && k <= 2048) ? 12288 : 8192) && (k < 8192 || k <= 6 * channels);
  if (m > 4 && k > 16384) return false;
  if ((k > 8192 && k >= 16 * channels) || (k > 12288 && k > 10 * channels)) return false;
  const int64_t depth = matrices * k;
  if (depth >= 5120) return true;
  if (m <= 2 && k >= 1536) return channels <= 32 * std::max<int64_t>(k, 2048);
  return channels <= (depth < 1024 ? 8192 : 11 * depth + 17407);
}

// Where tiles of 64 rows beat the split-K decode kernel, whose workgroups hold all rows of x for their slice of
// K in LDS: from 33 rows that leaves slices of 256 to 512 values and as many partial sums as weights. us,
// decode kernel and tiles: 64 rows of 28672 x 8192 152 and 70.8, of 4096 x 4096 23.7 and 15.8, of 1024 x 8192
// 16.1 and 12.5, of 512 x 1024 8.3 and 9.3; 33 rows of 8192 x 8192 36.1 and 26.0; 24 rows of 11008 x 4096 25.5
// and 22.4, of 5003 x 4080 15.1 and 17.0.
bool mid_linear_wins(int64_t m, int64_t n_total, int64_t k) {
  return m > 16 && n_total * k >= (m <= 32 ? int64_t(1) << 25 : int64_t(1) << 23);
}

void plan_mid_linear(Fp8LinearLaunch *p, int cus, int xcds) {
  const int64_t steps = (p->k + kPTileK - 1) / kPTileK;
  int64_t n_tiles = 0;
  for (int s = 0; s < p->group; ++s) n_tiles += (p->n[s] + kPTileN - 1) / kPTileN;
  // two workgroups per CU (their LDS fits), at least eight steps each, and no more partial sums than the
  // split-K plan's, whose size callers are told to allocate
  int64_t splits = std::min<int64_t>((2 * cus + n_tiles - 1) / n_tiles, std::max<int64_t>(1, steps / 8));
  splits = std::max<int64_t>(1, std::min<int64_t>(splits, p->splits));
  const int64_t split_steps = std::max<int64_t>(1, (steps + splits - 1) / splits);
  p->prefill = p->mid = true;
  p->small = offsets_fit(*p);
  p->xcds = std::max(1, xcds);
  p->waves = 4;
  p->splits = static_cast<int>(std::max<int64_t>(1, (steps + split_steps - 1) / split_steps));
  p->kc = split_steps * kPTileK;
  p->tile_n = kPTileN;
  p->m_tiles = 1;
  p->band = 1;
  p->row_groups = n_tiles;
  p->grid = p->xcds * ((p->splits * n_tiles + p->xcds - 1) / p->xcds);
  p->scratch_bytes = p->splits > 1 || p->epilogue != kFp8EpilogueNone
                         ? static_cast<size_t>(p->splits) * p->m * p->n_total * sizeof(float)
                         : 0;
}

void plan_direct_linear(Fp8LinearLaunch *p) {
  p->direct = true;
  p->splits = 1;
  p->waves = 1;  // blocks of 16 channels per workgroup
  p->row_groups = 0;
  for (int s = 0; s < p->group; ++s) p->row_groups += (p->n[s] + 15) / 16;
  p->grid = p->row_groups;
  p->scratch_bytes = 0;
}

hipError_t launch_mfma_probe(int shape, int workgroups, int iters, float *sink, hipStream_t stream) {
  if (shape == kMfmaProbe32x32x16)
    hipLaunchKernelGGL(mfma_probe_32x32_kernel, dim3(static_cast<unsigned>(workgroups)), dim3(256), 0, stream, sink,
                       iters);
  else
    hipLaunchKernelGGL(mfma_probe_kernel, dim3(static_cast<unsigned>(workgroups)), dim3(256), 0, stream, sink,
                       iters);
  return hipGetLastError();
}

namespace {

template <bool FP8, int XL>
hipError_t launch_direct_rows(const Fp8LinearLaunch &p, hipStream_t stream) {
  const SegTable seg = seg_table(p);
  const auto *x = static_cast<const uint8_t *>(p.x);
  const auto *residual = p.epilogue == kFp8EpilogueResidual ? static_cast<const uint16_t *>(p.residual) : nullptr;
  const dim3 block(kDirectWaves * kWave);
  const int m = static_cast<int>(p.m), k = static_cast<int>(p.k);
  if (p.epilogue == kFp8EpilogueSwiglu)  // the grid covers the channels of one matrix
    hipLaunchKernelGGL((direct_linear_kernel<FP8, XL, true>), dim3(static_cast<unsigned>(seg.rg0[1])), block, 0, stream,
                       x, seg, m, k, residual);
  else
    hipLaunchKernelGGL((direct_linear_kernel<FP8, XL, false>), dim3(static_cast<unsigned>(seg.rg0[p.group])), block, 0,
                       stream, x, seg, m, k, residual);
  return hipGetLastError();
}

hipError_t launch_direct(const Fp8LinearLaunch &p, hipStream_t stream) {
  if (p.bf16) {
    if (p.m <= 4) return launch_direct_rows<false, 1>(p, stream);
    return p.m <= 8 ? launch_direct_rows<false, 2>(p, stream) : launch_direct_rows<false, 4>(p, stream);
  }
  if (p.m <= 2) return launch_direct_rows<true, 1>(p, stream);
  return p.m <= 8 ? launch_direct_rows<true, 4>(p, stream) : launch_direct_rows<true, 8>(p, stream);
}

template <int TM, int TN, int WAVES, int S, bool DEAL>
void launch_tiled(const Fp8LinearLaunch &p, const SegTable &seg, float *part, hipStream_t stream) {
  const auto *x = static_cast<const uint8_t *>(p.x);
  const int m = static_cast<int>(p.m), k = static_cast<int>(p.k), mt = static_cast<int>(p.m_tiles),
            nt = static_cast<int>(p.row_groups);
  const int split_steps = static_cast<int>(p.kc / kPTileK);
  const dim3 grid(static_cast<unsigned>(p.grid)), block(WAVES * kWave);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, stream, x, seg, m, k, mt, nt, p.xcds, DEAL ? p.band : p.splits,
                       split_steps, part);
  };
  p.small ? launch(fp8_prefill_kernel<TM, TN, WAVES, S, true, DEAL>)
          : launch(fp8_prefill_kernel<TM, TN, WAVES, S, false, DEAL>);
}

}  // namespace

hipError_t launch_fp8_linear(const Fp8LinearLaunch &p, hipStream_t stream) {
  if (p.direct) return launch_direct(p, stream);
  if (p.prefill) {
    const SegTable seg = seg_table(p);
    if (p.mid) {
      const bool reduce = p.scratch_bytes > 0;
      const auto tiles = p.tile_n == 64 ? launch_tiled<64, 64, 4, 4, false> : launch_tiled<64, 128, 4, 4, false>;
      tiles(p, seg, reduce ? static_cast<float *>(p.workspace) : nullptr, stream);
      const hipError_t err = hipGetLastError();
      return err != hipSuccess || !reduce ? err : launch_reduce(p, seg, stream);
    }
    if (p.waves == 4)
      launch_tiled<128, 128, 4, 2, true>(p, seg, nullptr, stream);
    else
      (p.deal ? launch_tiled<128, 128, 8, 4, true> : launch_tiled<128, 128, 8, 4, false>)(p, seg, nullptr, stream);
    return hipGetLastError();
  }
  switch (p.batch_blocks) {
    case 1: return launch_mb<1>(p, stream);
    case 2: return launch_mb<2>(p, stream);
    case 3: return launch_mb<3>(p, stream);
    default: return launch_mb<4>(p, stream);
  }
}

}  // namespace ftx
