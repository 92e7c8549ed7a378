// Internal declarations shared by the runtime (C ABI) and the kernel file.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <string>

#include "../../include/ftx.h"

namespace ftx {

// Thread-local error message behind ftx_last_error().
void set_error(const std::string &msg);
int fail(int code, const std::string &msg);
int hip_fail(hipError_t err, const char *what);

#define FTX_HIP(expr)                                   \
  do {                                                  \
    hipError_t ftx_err_ = (expr);                       \
    if (ftx_err_ != hipSuccess) return ::ftx::hip_fail(ftx_err_, #expr); \
  } while (0)

// Set once by ftx_shutdown. Entry points that start work or allocate refuse
// afterwards (FTX_REQUIRE_LIVE); releasing, waiting and querying still work.
bool is_shut_down();
#define FTX_REQUIRE_LIVE()                                                                        \
  do {                                                                                            \
    if (::ftx::is_shut_down())                                                                    \
      return ::ftx::fail(FTX_ERR_UNSUPPORTED, "the library has been shut down (ftx_shutdown)"); \
  } while (0)

// Threads one launch can hold: the runtime refuses grids of 2^32 and more.
constexpr int64_t kMaxThreads = (int64_t(1) << 32) - 1;

// Default bytes per wave tile of the scatter kernel: one round of 8 loads and
// 8 non-temporal stores of 16 bytes per lane (fastest of 8/16/32 KiB on the
// 2000-tensor set's 512 MiB chunks: 5.94 TB/s against 5.78 and 5.77).
constexpr size_t kScatterTileBytes = 8 * 1024;
// Default zero-copy grid: 64 workgroups keep the link at its peak (more
// workgroups only add outstanding PCIe reads).
constexpr int kZeroCopyDefaultGrid = 64;
// A zero-copy launch of at most this many workgroups takes each CU it runs on
// whole (its workgroups reserve the CU's LDS).
constexpr int kZeroCopyReserveMaxGrid = 16;
// LDS that kernels without LDS of their own ask for and never touch when they run between a layer's products:
// one allocation granule. A ring copy beside a streamed pass holds its CUs' whole LDS (a small zero-copy grid),
// so with any LDS request a workgroup stays off those CUs; one that shares a CU with the copy queues behind the
// copy's outstanding host reads.
constexpr unsigned kLdsToken = 512;
// Wave tiles handled by one workgroup (one tile per wavefront).
constexpr int kScatterWavesPerGroup = 4;
// Checksum block: 64 lanes x 8 bytes x 8 steps.
constexpr size_t kChecksumBlockBytes = 4096;

// Device-resident scatter plan.
struct ScatterPlanDev {
  const ftx_desc *descs;        // n_desc descriptors
  const uint64_t *tile_start;   // n_desc + 1 exclusive prefix of tiles per descriptor
  const uint32_t *group_desc0;  // n_groups: descriptor of each workgroup's first tile
  int n_desc;
  int64_t n_tiles;
  int64_t n_groups;
  uint64_t tile_bytes;
};

// One launch of the fp8-weight linear kernel (ftx_gemm.hip), as planned by
// plan_fp8_linear from the shapes, the CU count and optional overrides. A
// launch covers `group` weight matrices (segments) that share the input x and
// k: y_s = bf16(scale_s * x @ w_s^T) for each segment s.
constexpr int kFp8MaxGroup = 4;
// Epilogues the decode kernel's reduce can apply (FTX_FP8_EPILOGUE_* in ftx.h).
constexpr int kFp8EpilogueNone = FTX_FP8_EPILOGUE_NONE;
constexpr int kFp8EpilogueSwiglu = FTX_FP8_EPILOGUE_SWIGLU;
constexpr int kFp8EpilogueResidual = FTX_FP8_EPILOGUE_RESIDUAL;
struct Fp8LinearLaunch {
  const void *x;                       // bf16 [m, k]
  int group;                           // segments in this launch, 1..kFp8MaxGroup
  const void *w[kFp8MaxGroup];         // e4m3fn [n_s, k]
  const void *scale[kFp8MaxGroup];     // bf16 [n_s]
  void *y[kFp8MaxGroup];               // bf16 [m, n_s]
  int64_t n[kFp8MaxGroup];             // output rows of each segment
  int64_t n_total;                     // sum of n
  void *workspace;    // fp32 partial sums [splits, m, n_s] per segment, back to back, when splits > 1
  int64_t m, k;
  int batch_blocks;   // 16-column batch blocks, 1 to 4 (m <= 16 * batch_blocks)
  int waves;          // wavefronts per workgroup, 16 output rows each
  int splits;         // K slices, one workgroup each per row group
  int64_t kc;         // K values per slice (multiple of 256)
  int64_t row_groups; // groups of 16 * waves output rows, summed over segments
  int64_t grid;       // workgroups = row_groups * splits
  size_t lds_bytes;   // activation slice + one weight tile per wave
  size_t workspace_bytes; // what callers are told to allocate
  size_t scratch_bytes;   // what the launch touches: at most workspace_bytes
  int epilogue;         // kFp8Epilogue*: what the reduce kernel applies to the outputs
  const void *residual; // bf16 [m, n[0]] for kFp8EpilogueResidual
  bool prefill;       // more than kFp8LinearMaxRows rows: the tiled prefill kernel (no split, no workspace)
  int64_t m_tiles;    // prefill: tiles of 128 or 64 activation rows (row_groups then counts tiles of tile_n channels)
  int tile_n;         // prefill: channels of a tile
  int xcds;           // prefill: L2 domains the block order is arranged for
  int band;           // prefill of 4 waves: m-tiles an XCD walks before its next n-tile
  bool deal;          // prefill: n-tiles dealt to the XCDs in turn, or equal runs of tiles
  bool small;         // prefill: 32-bit load offsets reach every operand
  bool mid;           // prefill kernel with 64-row tiles; up to 64 rows K may be split over workgroups
  bool direct;        // the one-launch decode kernel: no workspace, a workgroup per 16 channels
  bool bf16;          // direct only: bf16 weights without scales
};
// The one-launch decode kernel: its most rows, whether it is the faster one for an fp8 call, and its plan.
constexpr int kDirectMaxRows = 16;
constexpr int64_t kDirectMaxChannels = (int64_t(1) << 27) - 128;  // 512 threads for 16 of them, within kMaxThreads
bool direct_linear_wins(int64_t m, int64_t n_total, int64_t k, int epilogue);
void plan_direct_linear(Fp8LinearLaunch *p);
// Tiles of 64 rows for the batches between decode and prefill: whether they are faster, and their plan.
bool mid_linear_wins(int64_t m, int64_t n_total, int64_t k);
void plan_mid_linear(Fp8LinearLaunch *p, int cus, int xcds);
constexpr int kFp8LinearMaxRows = 64;
constexpr size_t kFp8LinearMaxLds = 64 * 1024;
Fp8LinearLaunch plan_fp8_linear(int64_t m, const int64_t *n, int group, int64_t k, int cus, int xcds, int waves,
                                int kc, int epilogue);
hipError_t launch_fp8_linear(const Fp8LinearLaunch &p, hipStream_t stream);
// MFMA rate probe: `workgroups` x 4 waves, each iters x 32 v_mfma_f32_16x16x32_bf16.
constexpr int kMfmaProbe16x16x32 = 0;  // v_mfma_f32_16x16x32_bf16, the prefill kernel's instruction
constexpr int kMfmaProbe32x32x16 = 1;  // v_mfma_f32_32x32x16_bf16
hipError_t launch_mfma_probe(int shape, int workgroups, int iters, float *sink, hipStream_t stream);

// One attention call (ftx_attention.hip). Strides are in elements: [batch, position, head].
struct AttentionLaunch {
  const uint16_t *q, *k, *v;  // bf16
  uint16_t *o;                // bf16
  float *part;                // per-split values, maxima and sums (part_bytes), when splits > 1
  int64_t q_stride[3], k_stride[3], v_stride[3], o_stride[3];
  int batch, t, s, heads, kv_heads, d;
  int causal, pos;            // causal: query t sees the keys up to pos + t
  float scale_log2;           // the score scale times log2(e)
  // planned
  int rep, rows, waves, row_tiles, splits, split_tiles, xcds;
  int64_t items;
  size_t part_bytes;
  bool tight;                 // given: values overlap, a position stride below a row
};
// Fills the planned members from the shapes.
void plan_attention(AttentionLaunch *p, int cus, int xcds);
hipError_t launch_attention(const AttentionLaunch &p, hipStream_t stream);

// The operations between a layer's matrix products (ftx_layers.hip). dim is a multiple of 8.
constexpr int kNormMaxDim = 32768;
int64_t norm_max_rows(int64_t dim);  // of a launch within kMaxThreads
constexpr int kNormNone = FTX_NORM_NONE, kNormRms = FTX_NORM_RMS, kNormAffine = FTX_NORM_LAYER,
              kNormAdaln = FTX_NORM_ADALN;
constexpr int kNormNoResidual = 0, kNormResidual = 1, kNormGatedResidual = 2;
struct NormLaunch {
  const uint16_t *x;      // bf16 [rows, dim]
  const uint16_t *delta;  // bf16 [rows, dim]: added to x (times the gate when gated) before the norm
  uint16_t *x_out;        // bf16 [rows, dim]: the sum, when there is a delta
  uint16_t *y;            // bf16 [rows, dim]: the normalised rows (unless norm is kNormNone)
  const uint16_t *w, *b;  // bf16 [dim]: RMS weight, or LayerNorm weight and bias
  const uint16_t *mod;    // bf16 [6, dim]: AdaLN modulation
  const uint16_t *e;      // bf16 [rows / rows_per_batch, 6, dim]: timestep embedding, added to mod
  int64_t rows, rows_per_batch;
  int dim, norm, residual;
  int gate, scale, shift; // which of the six AdaLN terms
  float eps;
};
hipError_t launch_norm(const NormLaunch &p, hipStream_t stream);

struct RopeLaunch {
  const uint16_t *q, *k, *v;  // bf16 [batch, t, heads or kv_heads, d], contiguous
  uint16_t *q_out;            // like q
  uint16_t *cache_k, *cache_v;
  const float *cos, *sin;     // fp32 [positions, d]
  int64_t k_stride[3], v_stride[3];  // of the caches, in elements: batch, position, head
  int64_t pos;
  int batch, t, heads, kv_heads, d;  // d a multiple of 16
};
hipError_t launch_rope_cache(const RopeLaunch &p, hipStream_t stream);
constexpr int64_t kSiluMulMax = (int64_t(1) << 35) - 4096;  // a thread for 8 values, within kMaxThreads
hipError_t launch_silu_mul(const uint16_t *g, const uint16_t *u, uint16_t *y, int64_t n, hipStream_t stream);

// Staged copies from pageable host memory and the parallel host memcpy
// (ftx_staged.hip).
int staged_copy_h2d(void *dst, const void *src, size_t nbytes, hipStream_t stream);
int host_memcpy(void *dst, const void *src, size_t nbytes);
int set_staging_policy(size_t piece_bytes, int threads);
void get_staging_policy(size_t *piece_bytes, int *threads);
// Joins the host threads and frees every device's staging buffers and events
// (each device made current in turn). Returns the first failure, after trying all.
int staged_shutdown();

// Kernel launchers (ftx_kernels.hip). Each returns hipSuccess or the launch error.
// `reserve_lds` bytes of dynamic LDS per workgroup (0: none); see zero_copy_kernel.
hipError_t launch_zero_copy(void *dst, const void *src_dev, size_t nbytes, int grid, size_t reserve_lds,
                            hipStream_t stream);
// Lets zero_copy_kernel take `bytes` of dynamic LDS on the current device.
hipError_t allow_zero_copy_lds(size_t bytes);
hipError_t launch_scatter(const ScatterPlanDev &plan, const void *chunk, hipStream_t stream);
hipError_t launch_checksum(const void *dev, size_t nbytes, uint64_t *partials, int n_waves,
                           hipStream_t stream);
hipError_t launch_fill_u8(void *dev, uint8_t value, size_t nbytes, hipStream_t stream);
hipError_t launch_timestamp(uint64_t *slot, hipStream_t stream);
hipError_t launch_read_probe(const void *dev, size_t nbytes, uint32_t *sink, int grid, hipStream_t stream);

// Exponent-coded blocks (ftx_expcode.hip): the layout of one encoded block.
constexpr uint64_t kExpcodeHeaderBytes = 256;
constexpr uint64_t kExpcodeGroupWords = 1024;
// Default decode grid: workgroups of 8 waves, each lane with eight groups' loads in flight.
constexpr int kExpcodeDefaultGrid = 16;
struct ExpcodeInfo {
  uint64_t n;        // raw bytes
  uint64_t n_words;  // n / 2
  uint64_t groups;   // groups of kExpcodeGroupWords words
  uint64_t escapes;  // escaped words
  uint64_t off_b, off_s, off_x, total;  // section offsets and encoded size (plane A starts at the header's end)
  uint8_t table[16];                    // exponent of each code below 15
  uint8_t tail;                         // the odd last raw byte
};
// out == nullptr: only *out_bytes (the encoded size) is computed.
int expcode_encode(const void *raw, size_t nbytes, void *out, size_t out_capacity, size_t *out_bytes);
// Reads and checks the header of an encoded block of src_bytes bytes in host memory.
int expcode_parse(const void *src, size_t src_bytes, ExpcodeInfo *info);
// Decodes the block of raw size n at src_dev (a device-visible address, `capacity` bytes readable) into
// dst; the kernel reads the block's header when it runs. `reserve_lds` as for launch_zero_copy.
hipError_t launch_expcode_decode(void *dst, const void *src_dev, uint64_t capacity, uint64_t n, int grid,
                                 size_t reserve_lds, hipStream_t stream);
hipError_t allow_expcode_lds(size_t bytes);

// Dense exponent-coded blocks (version 2): 3-bit primary codes for the 7 most frequent exponents in three
// bit planes, a 4-bit secondary code per primary escape for the next 15, a list for the rest. Sections
// after the 256-byte header: plane A (1024 bytes a group), plane P (384 a group), S1 and S2 (G + 1 u32
// each, 16-byte aligned), Y (a nibble per primary escape, 16-byte aligned), X (a u32 per secondary escape).
constexpr uint64_t kDensePlaneBytes = 384;
struct DenseLayout {
  uint64_t n, n_words, groups, e1, e2;
  uint64_t off_p, off_s1, off_s2, off_y, off_x, total;
};
// The section offsets of a dense block of raw size n with e1 primary and e2 secondary escapes.
DenseLayout dense_layout(uint64_t n, uint64_t e1, uint64_t e2);
// out == nullptr: only *out_bytes (the encoded size) is computed.
int expcode_encode_dense(const void *raw, size_t nbytes, void *out, size_t out_capacity, size_t *out_bytes);
// Decodes the dense block of raw size n at src_dev (device memory, `capacity` bytes readable) into dst; the
// kernel reads the block's header when it runs and writes nothing for a header of another raw size.
hipError_t launch_expcode_dense_decode(void *dst, const void *src_dev, uint64_t capacity, uint64_t n, int grid,
                                       size_t reserve_lds, hipStream_t stream);
// Reads and checks the header of a dense block of src_bytes bytes in host memory.
int expcode_parse_dense(const void *src, size_t src_bytes, DenseLayout *layout);
// The dense decode from mapped host memory (over the link): `reserve_lds` as for launch_zero_copy.
hipError_t launch_expcode_dense_link_decode(void *dst, const void *src_dev, uint64_t capacity, uint64_t n, int grid,
                                            size_t reserve_lds, hipStream_t stream);

// Host-side helpers shared with the oracle's definition of the checksum.
inline uint64_t splitmix64(uint64_t x) {
  x += 0x9e3779b97f4a7c15ull;
  uint64_t z = x;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

}  // namespace ftx
