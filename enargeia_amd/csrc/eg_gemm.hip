// matmul_q4_prefill (matmul_q4_prefill.wgsl:77-162) on the matrix cores:
//   out[r*out_stride + col + out_offset] = sum_k x[r,k] * W[col,k] (+ bias[col])
//
// The prompt's projections are the dense contraction on the path. This file holds the host side:
// the checks, the choice of a tile for a shape (tile_for) and the launches. The kernel is
// gemm_kernel (eg_gemm_kernel.hpp), instantiated in eg_gemm_{bf16,f32,norm,pair,rope}.hip.
// Layouts it does not take (K not a multiple of 32 codes or the block size of 16, a block size that
// is not a power of two, unaligned streams) stage both operands element by element with the
// reference's indexing (element_kernel below).
#include <algorithm>

#include "eg_gemm_kernel.hpp"

namespace {

using namespace eg_gemm;

// ---- the element-by-element kernel ------------------------------------------------------------

constexpr int kTile = 64;   // M and N tile
constexpr int kBK = 64;     // K staged per iteration
constexpr int kPad = 8;     // bf16 elements of padding per LDS row
constexpr int kLds = kBK + kPad;

struct ElementArgs {
  const float* x;
  const uint32_t* packed;
  const float* scales;
  const uint32_t* zeros;
  const float* bias;
  const float* residual;
  float* out;
  float* partials;  // split-K: [splits][m][n] f32; NULL when grid.z == 1
  uint32_t m, n, k, block_size, blocks_per_row, k_per_split, out_stride, out_offset;
  int bits;
};

__device__ __forceinline__ uint16_t bf16_bits(float v) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)((u >> 16) | ((u & 0x7FFFFFu) ? 0x40u : 0u));
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// One 64 x 64 block of x and of W into LDS.
template <int ENC>
__device__ void stage_elements(const ElementArgs& a, uint32_t m0, uint32_t n0, uint32_t k0,
                               uint16_t (*As)[kLds], uint16_t (*Bs)[kLds]) {
  const uint32_t tid = threadIdx.x & 255u;
  const uint32_t per_word = 32u / (uint32_t)a.bits, mask = (1u << a.bits) - 1u;
#pragma unroll 4
  for (uint32_t e = tid; e < kTile * kBK; e += 256) {
    const uint32_t r = e / kBK, c = e % kBK;
    const uint32_t row = m0 + r, kk = k0 + c;
    const float v = (row < a.m && kk < a.k) ? a.x[(size_t)row * a.k + kk] : 0.f;
    As[r][c] = bf16_bits(v);
  }
#pragma unroll 4
  for (uint32_t e = tid; e < kTile * kBK; e += 256) {
    const uint32_t r = e / kBK, c = e % kBK;
    const uint32_t nrow = n0 + r, kk = k0 + c;
    float v = 0.f;
    if (nrow < a.n && kk < a.k) {
      const size_t flat = (size_t)nrow * a.k + kk;
      uint32_t code = (a.packed[flat / per_word] >> (a.bits * (flat % per_word))) & mask;
      const uint32_t blk = nrow * a.blocks_per_row + kk / a.block_size;
      int32_t z;
      if (ENC == EG_ENC_OFFSET_ZEROS) {
        z = (int32_t)((a.zeros[blk / per_word] >> (a.bits * (blk % per_word))) & mask);
      } else {
        code ^= 1u << (a.bits - 1);
        z = 1 << (a.bits - 1);
      }
      v = (float)((int32_t)code - z) * a.scales[blk];
    }
    Bs[r][c] = bf16_bits(v);
  }
}

// A workgroup owns a 64 x 64 output tile and a slice of K, KG groups of 4 waves the 64-deep blocks
// g, g + KG, ... of it (each wave 32 x 32 of the tile); the groups' sums meet in LDS and are added
// in group order.
template <int ENC, int KG>
__global__ __launch_bounds__(256 * KG) void element_kernel(ElementArgs a) {
#pragma clang fp contract(off)
  constexpr uint32_t kStageBytes = 2u * kTile * kLds * 2u;  // As + Bs of one group
  static_assert(kStageBytes >= kTile * kTile * 4u, "a group's buffers hold its 64 x 64 f32 sums");
  __shared__ __attribute__((aligned(16))) uint8_t lds[KG * kStageBytes];
  const uint32_t group = threadIdx.x >> 8;
  uint16_t(*As)[kLds] = reinterpret_cast<uint16_t(*)[kLds]>(lds + group * kStageBytes);
  uint16_t(*Bs)[kLds] = reinterpret_cast<uint16_t(*)[kLds]>(lds + group * kStageBytes + kTile * kLds * 2u);
  const uint32_t tid = threadIdx.x & 255u, wave = tid >> 6, lane = tid & 63u;
  const uint32_t m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
  const uint32_t wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const uint32_t kbeg = blockIdx.z * a.k_per_split, kend = min(a.k, kbeg + a.k_per_split);
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint32_t nblk = (kend - kbeg + kBK - 1) / kBK, iters = (nblk + KG - 1) / KG;
  for (uint32_t it = 0; it < iters; it++) {
    const uint32_t blk = group + KG * it;
    stage_elements<ENC>(a, m0, n0, kbeg + min(blk, nblk - 1) * kBK, As, Bs);
    __syncthreads();
    if (blk < nblk) {
#pragma unroll
      for (int ks = 0; ks < kBK / 32; ks++) {
        const uint32_t kofs = ks * 32 + 8 * (lane >> 4);
        bf16x8 af[2], bfr[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          af[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&As[wm + i * 16 + (lane & 15)][kofs]));
          bfr[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&Bs[wn + i * 16 + (lane & 15)][kofs]));
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // every group's sums into its own buffers (the last barrier ended the staging), then the groups
  // added in order by the thread that stores the element
  float* sums = reinterpret_cast<float*>(lds + group * kStageBytes);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        sums[(wm + i * 16 + 4 * (lane >> 4) + e) * kTile + wn + j * 16 + (lane & 15)] = acc[i][j][e];
  __syncthreads();
  for (uint32_t idx = threadIdx.x; idx < kTile * kTile; idx += 256u * KG) {
    const uint32_t r = idx / kTile, c = idx % kTile, row = m0 + r, col = n0 + c;
    if (row >= a.m || col >= a.n) continue;
    float v = reinterpret_cast<const float*>(lds)[idx];
#pragma unroll
    for (int g = 1; g < KG; g++) v += reinterpret_cast<const float*>(lds + g * kStageBytes)[idx];
    if (a.partials) {
      a.partials[((size_t)blockIdx.z * a.m + row) * a.n + col] = v;
    } else {
      const size_t o = (size_t)row * a.out_stride + col + a.out_offset;
      a.out[o] = v + (a.bias ? a.bias[col] : 0.f) + (a.residual ? a.residual[o] : 0.f);
    }
  }
}

// The split-K sum: splits added in index order, then the bias.
__global__ __launch_bounds__(256) void prefill_reduce_kernel(const float* __restrict__ partials,
                                                             const float* __restrict__ bias,
                                                             const float* __restrict__ residual, float* out, uint32_t m,
                                                             uint32_t n, uint32_t splits, uint32_t out_stride,
                                                             uint32_t out_offset) {
  const size_t total = (size_t)m * n;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    float acc = 0.f;
    for (uint32_t z = 0; z < splits; z++) acc += partials[(size_t)z * total + i];
    const uint32_t row = (uint32_t)(i / n), col = (uint32_t)(i % n);
    const size_t o = (size_t)row * out_stride + col + out_offset;
    out[o] = acc + (bias ? bias[col] : 0.f) + (residual ? residual[o] : 0.f);
  }
}

// ---- x as bf16 rows -----------------------------------------------------------------------------

// n f32 values (a multiple of 8) rounded to bf16, as the GEMM's own staging rounds them.
__global__ __launch_bounds__(256) void to_bf16_kernel(const float4* __restrict__ x, uint4* __restrict__ out, size_t n8) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += (size_t)gridDim.x * blockDim.x) {
    const float4 a = x[2 * i], b = x[2 * i + 1];
    out[i] = make_uint4(egd::pack_bf16(a.x, a.y), egd::pack_bf16(a.z, a.w), egd::pack_bf16(b.x, b.y), egd::pack_bf16(b.z, b.w));
  }
}

void to_bf16(eg_context* ctx, const float* x, size_t n, void* out) {
  const size_t n8 = n / 8;
  const uint32_t blocks = (uint32_t)std::min<size_t>((n8 + 255) / 256, (size_t)ctx->cu_count * 16);
  hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks), dim3(256), 0, ctx->stream, reinterpret_cast<const float4*>(x),
                     static_cast<uint4*>(out), n8);
}

// How many rows of k f32 values the context's buffer takes as bf16 at once, in whole tiles; 0: none, and
// the launch stages f32 rows. The buffer is used on the context's own stream alone and outside captures:
// every use is then ordered after the one before it, whatever other streams and replayed graphs do beside
// it.
uint32_t rows_at_once(const eg_context* ctx, uint32_t k, const Tile& t) {
  if (ctx->stream != ctx->own_stream || ctx->capturing) return 0;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return 0;
  const uint64_t rows = eg::kRowsBytes / ((uint64_t)k * 2);
  return (uint32_t)(rows / t.rows() * t.rows());
}

// ---- the choice of a tile -----------------------------------------------------------------------

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

uint64_t tile_count(const Tile& t, uint32_t m, uint64_t cols) {
  return ((cols + t.wn - 1) / t.wn) * ((m + t.rows() - 1) / t.rows());
}

// The tile of a launch over m rows and k. A sum's order is that of the chunks and K groups (BK, KG), so
// those are chosen for `cols` 64-column tiles - of one matrix, where a launch holds several of one shape:
// gate and up as a pair, in one launch and on their own give the same bits - and the rows and columns
// for the `launch_cols` tiles that the launch has.
//
// Up to K = 2048 the smallest tile that still covers the matrix in one workgroup per CU (a second round
// of these workgroups costs more than larger tiles), and the largest where none does: large tiles spread
// the dequantization over more rows, small ones fill the device and, with four groups of waves on alternate
// chunks of K, shorten the serial chain. The small ones take 64-deep chunks ("fine") up to K = 768 and where
// those leave fewer idle steps to the groups (K of 1025 to 1280); at 769 to 896, where both leave the
// same, where a launch or a pair of it takes 64 rows (64 x 4864 x 896 as a pair 10.2 us fine, 11.9 else; 70
// rows, 32 at a time, of the reference format 10.2 fine, 9.7 else). Measured on MI355X (us; f32 rows, int4
// sym; workgroups of 32x64 | 64x64 | 64x128 | 64x256):
//                     32x64 fine  32x64  64x64 fine  64x64  64x128  64x256  128x256
//     64 x 1024 x  320       5.1    5.3         6.7    7.3     7.9    10.6     13.5   (32)
//    128 x 4864 x  640       8.3    9.6         8.1    9.3     9.8    13.4     20.8   (304 | 152)
//    512 x  896 x  896       7.1    7.0         8.9    9.3    11.2    16.0     24.2   (224 | 112)
//    128 x 4864 x  896       9.7    9.9         9.1    9.4    11.3    16.1     23.9   (304 | 152)
//    128 x 4864 x 1152      10.8   12.2        10.1   11.2    12.8    18.5     27.1   (304 | 152)
//    384 x 1536 x 1536      15.4   13.4        11.8   11.2    16.5    22.2     35.9   (288 | 144)
//    256 x 4864 x  896      13.0   14.3        13.5   17.6    11.7    16.4     24.2   (608 | 304 | 152)
//    256 x 9728 x  896      19.1   21.8        19.3   25.8    17.1    17.1     25.0   (1216 | 608 | 304 | 152)
//   2048 x 1152 x  896, q|k|v (RoPE)
//                           23.5   24.7        23.6   26.6    23.5    22.0     29.7   (1152 | 576 | 288 | 160)
//    200 x 8960 x 1536      26.5   24.6        27.3   31.1    28.0    23.2     35.8   (980 | 560 | 280 | 140)
//    512 x 9728 x  896         -      -        29.5   42.7    25.7    26.1     27.8   (2432 | 1216 | 608 | 304)
//   2048 x 9728 x  896, gate|up (bf16 rows): 64x256 64, 128x256 58
//
// From K = 2048 on the grid may be split over K, at 2.3 us and the partial sums' traffic: 32 x 64 where
// three splits of it fill the CUs, or where it needs none and K is short enough; else larger tiles with more
// splits, which dequantize each weight for more rows (with no more than 32 rows none has more). Measured
// (splits in brackets; f32 rows, bf16 ones for 896 x 4864):
//                       32x64     64x64     64x128 long  64x128 deep  128x128   128x256
//    100 x 2048 x 2048  9.0 (2)   11.1 (4)  11.7 (4)     14.7 (4)     14.2 (8)  16.5 (8)
//    256 x 2048 x 2048  10.1      12.8      15.0 (4)     18.2 (2)     21.2 (4)  24.5 (6)
//     64 x 4096 x 4096  13.9 (2)  14.1 (4)  15.2 (4)     18.0 (4)     19.8 (8)  22.4 (8)
//     16 x 4096 x 11008 16.3 (4)  20.0 (4)  19.2 (8)     20.6 (8)     24.1 (8)  31.9 (8)
//    256 x  896 x 4864  14.9 (2)  13.8 (4)  16.6 (8)     16.5 (6)     19.8 (8)  22.8 (8)
//    100 x 1536 x 8960  22.1 (2)  20.2 (4)  18.8 (8)     22.1 (6)     25.3 (8)  33.0 (8)
//     64 x 4096 x 11008 26.3 (2)  23.9 (4)  22.2 (8)     23.8 (8)     26.7 (8)  35.0 (8)
//   1024 x  896 x 4864  31.2      24.6      26.5 (4)     25.8 (2)     25.5 (4)  30.3 (8)
//   2048 x  896 x 4864  60.1      48.7      41.8 (2)     35.7         36.6 (2)  39.8 (4)
//   1024 x 4096 x 4096  109       89.7      61.5         64.4         48.1      56.5 (2)
//   2048 x 4096 x 11008 -         420       276          300          221       207
//
// RoPE's epilogue (angles, rotation, f16 rows) grows with a tile's rows: 32 up to two workgroups per CU
// (q|k|v of 600 rows, fine: 11.6 us; 64 x 64, not fine: 13.3). Blocks of 16 codes need the 64-deep chunks.
Tile tile_for(const eg_context* ctx, uint32_t m, uint64_t cols, uint32_t k, uint32_t bs, uint64_t launch_cols,
              int epi) {
  if (ctx->gemm_tile[0]) {
    // (a lane's BK / 2 codes take two scales)
    const Tile t{ctx->gemm_tile[0], ctx->gemm_tile[1], ctx->gemm_tile[2], ctx->gemm_tile[3]};
    if (bs * 4 >= (uint32_t)t.bk && (epi == kStore || !t.store_only())) return t;
  }
  const uint64_t cus = (uint64_t)ctx->cu_count;
  auto count = [&](const Tile& t) { return tile_count(t, m, cols); };
  auto fits = [&](const Tile& t) { return count(t) <= cus; };
  // of two tiles of 32 and 64 rows: 32 where that is a workgroup per CU, 64 where that is one or the
  // workgroups are many in any case (two of the others fit on a CU)
  auto rows = [&](const Tile& low, const Tile& high) {
    const uint64_t n = tile_count(low, m, launch_cols);
    if (n <= cus || (epi == kRope && n <= 2 * cus)) return low;
    return tile_count(high, m, launch_cols) <= cus || n > 3 * cus ? high : low;
  };
  const uint64_t n = count(kTile32x64);
  if (bs < 32) return fits(kTile64x64Fine) ? rows(kTile32x64Fine, kTile64x64Fine) : kTile64x128;
  if (k < 2048) {
    const bool fine = k <= 768 || (k > 1024 && k <= 1280) ||
                      (k <= 896 && (n > cus || (n > cus / 2 && count(kTile64x64) <= cus / 2)));
    if (fits(kTile64x64) || (m <= 32 && n <= 2 * cus))
      return fine ? rows(kTile32x64Fine, kTile64x64Fine) : rows(kTile32x64, kTile64x64);
    if (fits(kTile64x128)) return kTile64x128;
    return fits(kTile64x256) ? kTile64x256 : kTile128x256;
  }
  if (n <= cus / 3 || (n <= cus && (m <= 32 || k <= (n <= cus / 2 ? 3584u : 4096u)))) return kTile32x64;
  if (n <= cus / 2 && k >= 8192) return kTile64x128Long;
  if (fits(kTile64x64)) return kTile64x64;
  if (fits(kTile64x128Deep)) return kTile64x128Deep;
  return fits(kTile128x128) ? kTile128x128 : kTile128x256;
}

// Ranges K is split into over the grid: where the tiles leave CUs idle over a long K, down to one
// chunk per group of waves. The partial sums cost a second launch.
uint64_t splits_for(const eg_context* ctx, const Tile& t, uint32_t m, uint64_t cols, uint32_t k) {
  if (ctx->gemm_tile[4]) return (uint64_t)ctx->gemm_tile[4];
  const uint64_t tiles = tile_count(t, m, cols), chunks = (k + t.bk - 1) / t.bk;
  if (k < 2048 || tiles >= (uint64_t)ctx->cu_count) return 1;
  return std::max<uint64_t>(1, std::min<uint64_t>(ctx->cu_count / tiles, chunks / t.kg));
}

// Runs launch(tile, x, xm, first, rows) over f32 rows of x (m rows of k): one launch of all of them,
// or - the largest tiles, which take bf16 rows - one per stretch of rows that the context's buffer
// holds. Where it holds none, the tile of the same chunks and K groups that stages f32 rows takes
// their place: slower, the same bits. Measured (MI355X): 2048 x 11008 x 4096 237 us with the rounding
// launch, 361 with 64 x 256 on f32 rows.
template <class F>
int over_f32_rows(eg_context* ctx, const Tile& t, const float* x, uint32_t m, uint32_t k, F launch) {
  if (!t.bf16_only()) return launch(t, x, (int)kXF32, 0u, m);
  const uint32_t at_once = rows_at_once(ctx, k, t);
  if (!at_once) return launch(t.f32_form(), x, (int)kXF32, 0u, m);
  for (uint32_t first = 0; first < m; first += at_once) {
    const uint32_t n = std::min(at_once, m - first);
    // behind the rows of the call before: written over those, whose lines the XCDs' L2s still hold, the
    // SwiGLU pair of 1024 x 4864 x 896 took 39.5 us for 38.3
    const size_t bytes = ((size_t)n * k * 2 + 255) / 256 * 256;
    if (ctx->rows_next + bytes > eg::kRowsBytes) ctx->rows_next = 0;
    void* const rows = ctx->rows + ctx->rows_next;
    ctx->rows_next += bytes;
    to_bf16(ctx, x + (size_t)first * k, (size_t)n * k, rows);
    const int st = launch(t, rows, (int)kXBf16, first, n);
    if (st != EG_OK) return st;
  }
  return EG_OK;
}

// The workgroup grid of a tile over m rows and `cols` 64-column tiles, and the order its tiles are
// dealt to the XCDs in: the one whose runs read fewer bytes into an L2 - column-major 1/8 of W and up to
// all of x, row-major 1/8 of x and up to all of W. (2048 x 896 x 4864, x 20 MB and W 2.4 MB: 44.7 us with
// column-major runs, 39.9 with row-major ones.)
void set_grid(const eg_context* ctx, Args& a, const Tile& t, uint64_t cols, int xm, int bits) {
  a.tiles_x = (uint32_t)((cols + t.wn - 1) / t.wn);
  a.tiles_y = (a.m + t.rows() - 1) / t.rows();
  const double run = (double)a.tiles_x * a.tiles_y / 8.0;
  const double x = (double)a.m * a.k * (xm == kXBf16 ? 2 : 4), w = (double)cols * kCols * a.k * bits / 8;
  const double column_major = x * std::min(1.0, run / a.tiles_y) + w / 8, row_major = x / 8 + w * std::min(1.0, run / a.tiles_x);
  a.xcd = !ctx->prefill_xcd ? 0u : column_major <= row_major ? 1u : 2u;
}

int launch_tile(eg_context* ctx, const char* op, KernelFn fn, const Args& a, const Tile& t, uint32_t splits) {
  if (!fn) return eg::fail(ctx, EG_ERR_INVALID, "%s: no kernel for tile %d,%d,%d,%d", op, t.bk, t.mf, t.wn, t.kg);
  hipLaunchKernelGGL(fn, dim3(a.tiles_x * a.tiles_y, splits), dim3(64 * t.wn * t.kg), 0, ctx->stream, a);
  return EG_OK;
}

// Whether a matrix's outputs take 16-byte stores.
bool vector_out(const Mat& w) {
  return w.n % 4 == 0 && w.out_stride % 4 == 0 && w.out_offset % 4 == 0 && aligned16(w.out);
}

}  // namespace

bool eg::prefill_tile_known(const int* tile) {
  for (const Tile& t : kTiles)
    if (t.bk == tile[0] && t.mf == tile[1] && t.wn == tile[2] && t.kg == tile[3]) return true;
  return false;
}

bool eg::prefill_chunked(uint32_t m, uint32_t n, uint32_t k, uint32_t bs, int bits, const void* x,
                         const uint32_t* packed) {
  return (bits == 4 || bits == 8) && k % 32 == 0 && bs % 16 == 0 && (bs & (bs - 1)) == 0 &&
         (uint64_t)m * k * 4 < kOutside && (uint64_t)n * k / 8 * bits < kOutside &&
         (reinterpret_cast<uintptr_t>(packed) & 7u) == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

int eg::prefill_gemm(eg_context* ctx, const float* x, const uint32_t* packed, const float* scales,
                     const uint32_t* zeros, const float* bias, const float* residual, float* out,
                     const eg_matmul_q4_dims* dims, int encoding, int bits, bool x_bf16) {
  const char* op = "matmul_q4_prefill";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (!dims || !x || !packed || !scales || !out) return eg::fail(ctx, EG_ERR_INVALID, "%s: NULL argument", op);
  if (bits != 4 && bits != 8) return eg::fail(ctx, EG_ERR_INVALID, "%s: bits must be 4 or 8, got %d", op, bits);
  if (encoding != EG_ENC_OFFSET_ZEROS && encoding != EG_ENC_SIGNED)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: unknown encoding %d", op, encoding);
  if (encoding == EG_ENC_OFFSET_ZEROS && !zeros)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: the offset encoding needs a zero-point stream", op);
  if (dims->use_bias && !bias) return eg::fail(ctx, EG_ERR_INVALID, "%s: useBias set but bias is NULL", op);
  const uint32_t m = dims->m, n = dims->n, k = dims->k, bs = dims->block_size;
  if (bs == 0 || k % bs != 0)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: reduction axis %u is not a multiple of %u", op, k, bs);
  if (dims->blocks_per_row != k / bs)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: blocksPerRow %u does not equal k / blockSize = %u", op,
                    dims->blocks_per_row, k / bs);
  if (m > 1 && dims->out_stride < n)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: outStride %u is less than n %u", op, dims->out_stride, n);
  if (((uint64_t)n * k) % (32 / bits) != 0)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: codes do not fill whole 32-bit words", op);
  if ((uint64_t)m * k >= (1ull << 40) || (uint64_t)n * dims->blocks_per_row >= (1ull << 32))
    return eg::fail(ctx, EG_ERR_RANGE, "%s: %u x %u x %u exceeds the index range", op, m, n, k);
  if (m == 0 || n == 0) return EG_OK;
  const uint32_t tiles_n = (n + kTile - 1) / kTile, tiles_m = (m + kTile - 1) / kTile;
  if (tiles_m > 65535) return eg::fail(ctx, EG_ERR_RANGE, "%s: m %u needs %u row tiles, over 65535", op, m, tiles_m);
  const bool chunked = eg::prefill_chunked(m, n, k, bs, bits, x, packed);
  if (x_bf16 && !chunked)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: bf16 rows of x need the chunked staging", op);
  // Split K only where the tile grid leaves most CUs idle over a long reduction: the partial sums
  // cost a second launch. They live in the context's workspace.
  Tile t{};
  uint64_t splits = 1;
  uint32_t step = kBK;
  int kg = 1;
  if (chunked) {
    t = tile_for(ctx, m, tiles_n, k, bs, tiles_n, kStore);
    splits = splits_for(ctx, t, m, tiles_n, k);
    step = t.bk;
  } else {
    // four groups of waves where the grid holds under a tile per CU, else one
    const uint64_t tiles = (uint64_t)tiles_n * tiles_m, blocks = (k + kBK - 1) / kBK;
    kg = tiles >= (uint64_t)ctx->cu_count ? 1 : 4;
    if (blocks >= 32 && kg == 4) splits = std::min<uint64_t>(ctx->cu_count / tiles, blocks / 8);
  }
  splits = std::min<uint64_t>(splits, std::max<uint64_t>(1, eg::kPartialsBytes / ((uint64_t)m * n * 4)));
  splits = std::max<uint64_t>(1, std::min<uint64_t>(splits, 65535));
  const uint32_t k_per_split = (uint32_t)((((uint64_t)k + splits - 1) / splits + step - 1) / step * step);
  splits = (k + k_per_split - 1) / k_per_split;
  float* const partials = splits > 1 ? reinterpret_cast<float*>(eg::partials(ctx)) : nullptr;
  const float* const use_bias = dims->use_bias ? bias : nullptr;
  // the splits' sum over `rows` rows from `first`
  auto reduce = [&](uint32_t first, uint32_t rows) {
    if (!partials) return;
    const size_t at = (size_t)first * dims->out_stride;
    const uint64_t total = (uint64_t)rows * n;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((total + 255) / 256, (uint64_t)ctx->cu_count * 8);
    hipLaunchKernelGGL(prefill_reduce_kernel, dim3(blocks), dim3(256), 0, ctx->stream, partials, use_bias,
                       residual ? residual + at : nullptr, out + at, rows, n, (uint32_t)splits, dims->out_stride,
                       dims->out_offset);
  };
  if (chunked) {
    auto launch = [&](const Tile& tile, const void* rows_x, int xm, uint32_t first, uint32_t rows) {
      const size_t at = (size_t)first * dims->out_stride;
      Args a{};
      a.x = rows_x;
      a.partials = partials;
      a.m = rows;
      a.k = k;
      a.block_shift = (uint32_t)__builtin_ctz(bs);
      a.blocks_per_row = dims->blocks_per_row;
      a.k_per_split = k_per_split;
      a.nmats = 1;
      a.mats[0] = Mat{packed, scales, encoding == EG_ENC_SIGNED ? nullptr : zeros, use_bias,
                      residual ? residual + at : nullptr, out + at, n, dims->out_stride, dims->out_offset, tiles_n};
      set_grid(ctx, a, tile, tiles_n, xm, bits);
      const KernelFn fn = xm == kXBf16 ? pick_store_bf16(encoding, bits, tile) : pick_store_f32(encoding, bits, tile);
      const int st = launch_tile(ctx, op, fn, a, tile, (uint32_t)splits);
      if (st == EG_OK) reduce(first, rows);
      return st;
    };
    const int st = x_bf16 ? launch(t, x, (int)kXBf16, 0u, m) : over_f32_rows(ctx, t, x, m, k, launch);
    if (st != EG_OK) return st;
  } else {
    const ElementArgs a{x, packed, scales, encoding == EG_ENC_SIGNED ? nullptr : zeros, use_bias, residual, out, partials,
                        m, n, k, bs, dims->blocks_per_row, k_per_split, dims->out_stride, dims->out_offset, bits};
    const dim3 grid(tiles_n, tiles_m, (uint32_t)splits), block(256 * kg);
    const auto fn = encoding == EG_ENC_SIGNED ? (kg == 4 ? element_kernel<EG_ENC_SIGNED, 4> : element_kernel<EG_ENC_SIGNED, 1>)
                                              : (kg == 4 ? element_kernel<EG_ENC_OFFSET_ZEROS, 4>
                                                         : element_kernel<EG_ENC_OFFSET_ZEROS, 1>);
    hipLaunchKernelGGL(fn, grid, block, 0, ctx->stream, a);
    reduce(0, m);
  }
  return eg::check_launch(ctx, op);
}

namespace {

// Whether matrices sharing x run in ONE launch: the chunked staging takes every one of them and
// no K split is wanted (K under 2048). Sets the total of their 64-column tiles, and the number the
// launch's tile is chosen for: matrices of one shape take the tile that one of them alone takes, so
// that gate and up as a pair, in one launch and on their own give the same bits; others their total.
bool one_launch(const float* x, uint32_t m, uint32_t k, uint32_t block_size, int encoding, int bits,
                const eg::PrefillMatrix* mats, uint32_t count, uint64_t* tiles_n, uint64_t* tile_cols) {
  bool ok = count >= 1 && count <= kMaxSegs && m > 0 && x && bits == 4 &&
            (encoding == EG_ENC_SIGNED || encoding == EG_ENC_OFFSET_ZEROS) && block_size >= 16 &&
            (block_size & (block_size - 1)) == 0 && k % block_size == 0 && k % 32 == 0 &&
            (k + kBK - 1) / kBK < 32 && (uint64_t)m * k * 4 < kOutside && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
  *tiles_n = 0;
  bool same = true;
  for (uint32_t i = 0; ok && i < count; i++) {
    const eg::PrefillMatrix& w = mats[i];
    ok = w.n > 0 && w.packed && w.scales && w.out && (encoding == EG_ENC_SIGNED || w.zeros) &&
         (m == 1 || w.out_stride >= w.n) && (uint64_t)w.n * k / 2 < kOutside &&
         (uint64_t)w.n * (k / block_size) < (1ull << 32) && (reinterpret_cast<uintptr_t>(w.packed) & 7u) == 0;
    *tiles_n += (w.n + kTile - 1) / kTile;
    if (w.n != mats[0].n) same = false;
  }
  *tile_cols = same && count ? *tiles_n / count : *tiles_n;
  return ok && *tiles_n <= 0x7FFFFFFFull && (m + kTile - 1) / kTile <= 65535;
}

// Whether a launch folds the rows' RMSNorm in: only under one 64 x 64 tile per CU (latency-bound),
// where the extra staging work (the weight multiply and the squares) is hidden; a launch that fills
// the device is bound by that work, and a separate rmsnorm_rows launch costs less. (The tiles of these
// launches, 64 x 64 at most, have the kernel; a forced one may not.)
bool fold_norm(const eg_context* ctx, const Tile& t, uint32_t m, uint64_t cols, const float* norm) {
  return norm && aligned16(norm) && cols * ((m + kTile - 1) / kTile) < (uint64_t)ctx->cu_count && t.folds_norm();
}

// The matrices (one_launch accepted them) as one launch over m rows of x, rows `first` on of the
// outputs; xm says how x is staged (kXNorm with norm and eps: the rows' RMSNorm folded in).
int launch_multi(eg_context* ctx, const void* x, uint32_t first, uint32_t m, uint32_t k, uint32_t block_size,
                 int encoding, const eg::PrefillMatrix* mats, uint32_t count, uint64_t cols, int xm, int epi,
                 const Tile& t, const float* norm, float eps, const eg::PrefillRope* rope = nullptr,
                 bool out_bf16 = false) {
  Args a{};
  a.x = x;
  a.m = m;
  a.k = k;
  a.block_shift = (uint32_t)__builtin_ctz(block_size);
  a.blocks_per_row = k / block_size;
  a.k_per_split = k;
  a.nmats = count;
  a.norm = norm;
  a.eps = eps;
  a.out_bf16 = out_bf16 ? 1u : 0u;
  if (rope) {
    a.rope = rope->table;
    a.q_rope = rope->q_rope + (size_t)first * rope->q_heads * kCols;
    a.k_cache = rope->k_cache;
    a.v_cache = rope->v_cache;
    a.rope_pos0 = rope->pos0 + first;
    a.q_heads = rope->q_heads;
    a.kv_heads = rope->kv_heads;
  }
  uint32_t end = 0;
  a.vec = 1;
  for (uint32_t i = 0; i < count; i++) {
    const eg::PrefillMatrix& w = mats[i];
    // (out_bf16: `out` holds 2-byte values)
    const size_t at = (size_t)first * w.out_stride;
    end = epi == kPair ? (uint32_t)cols : end + (w.n + kTile - 1) / kTile;
    a.mats[i] = Mat{w.packed, w.scales, encoding == EG_ENC_SIGNED ? nullptr : w.zeros, w.bias,
                    w.residual ? w.residual + at : nullptr,
                    out_bf16 ? reinterpret_cast<float*>(reinterpret_cast<uint16_t*>(w.out) + at) : w.out + at, w.n,
                    w.out_stride, w.out_offset, end};
    if (!vector_out(a.mats[i])) a.vec = 0;
  }
  set_grid(ctx, a, t, cols, xm, 4);
  KernelFn fn = nullptr;
  if (epi == kRope) fn = pick_rope(encoding, xm, t);
  else if (epi == kPair) fn = pick_pair(encoding, xm, t);
  else if (xm == kXNorm) fn = pick_store_norm(encoding, t);
  else fn = xm == kXBf16 ? pick_store_bf16(encoding, 4, t) : pick_store_f32(encoding, 4, t);
  const int st = launch_tile(ctx, "matmul_q4_prefill", fn, a, t, 1);
  return st != EG_OK ? st : eg::check_launch(ctx, "matmul_q4_prefill");
}

// Runs launch(tile, x, xm, first, rows) over the rows, RMS-normalised first where norm is given: folded
// into the launch where that pays (kXNorm), else by rmsnorm_rows into `normed` - as bf16 rows where the
// context stages them.
template <class F>
int over_rows(eg_context* ctx, const Tile& t, const float* x, uint32_t m, uint32_t k, uint64_t cols, const float* norm,
              float eps, float* normed, F launch) {
  if (fold_norm(ctx, t, m, cols, norm)) return launch(t, x, (int)kXNorm, 0u, m);
  if (norm) {
    if (!normed) return eg::fail(ctx, EG_ERR_INVALID, "matmul_q4_prefill: RMSNorm needs a buffer for the normed rows");
    const int st = eg::rmsnorm_rows(ctx, x, norm, m, k, eps, normed, ctx->prefill_xb16);
    if (st != EG_OK) return st;
    if (ctx->prefill_xb16) return launch(t, normed, (int)kXBf16, 0u, m);
    x = normed;
  }
  return over_f32_rows(ctx, t, x, m, k, launch);
}

}  // namespace

int eg::prefill_gemm_multi(eg_context* ctx, const float* x, uint32_t m, uint32_t k, uint32_t block_size,
                           int encoding, int bits, const PrefillMatrix* mats, uint32_t count, const float* norm,
                           float eps, float* normed) {
  const char* op = "matmul_q4_prefill";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (count > 0 && !mats) return eg::fail(ctx, EG_ERR_INVALID, "%s: NULL matrix list", op);
  uint64_t cols = 0, tile_cols = 0;
  // One launch where the chunked staging takes every matrix and no matrix would split K;
  // otherwise (and for anything the single path must reject with its own message) one each.
  if ((count >= 2 || norm) && one_launch(x, m, k, block_size, encoding, bits, mats, count, &cols, &tile_cols)) {
    return over_rows(ctx, tile_for(ctx, m, tile_cols, k, block_size, cols, kStore), x, m, k, cols, norm, eps, normed,
                     [&](const Tile& t, const void* rows_x, int xm, uint32_t first, uint32_t rows) {
                       return launch_multi(ctx, rows_x, first, rows, k, block_size, encoding, mats, count, cols, xm,
                                           kStore, t, norm, eps);
                     });
  }
  if (norm) {
    if (!normed) return eg::fail(ctx, EG_ERR_INVALID, "%s: RMSNorm needs a buffer for the normed rows", op);
    const int st = eg::rmsnorm_rows(ctx, x, norm, m, k, eps, normed, false);
    if (st != EG_OK) return st;
    x = normed;
  }
  for (uint32_t i = 0; i < count; i++) {
    const PrefillMatrix& w = mats[i];
    eg_matmul_q4_dims dm{};
    dm.m = m;
    dm.n = w.n;
    dm.k = k;
    dm.use_bias = w.bias != nullptr;
    dm.block_size = block_size;
    dm.blocks_per_row = block_size ? k / block_size : 0;
    dm.out_stride = w.out_stride;
    dm.out_offset = w.out_offset;
    const int st = eg::prefill_gemm(ctx, x, w.packed, w.scales, w.zeros, w.bias, w.residual, w.out, &dm, encoding, bits);
    if (st != EG_OK) return st;
  }
  return EG_OK;
}

int eg::prefill_qkv_rope(eg_context* ctx, const float* x, uint32_t m, uint32_t k, uint32_t block_size, int encoding,
                         int bits, const PrefillMatrix* mats, const float* norm, float eps, float* normed,
                         const PrefillRope& rope, bool* done) {
  *done = false;
  if (!ctx || !mats || !ctx->prefill_rope || m == 0) return EG_OK;
  uint64_t cols = 0, tile_cols = 0;
  if (!rope.table || !rope.q_rope || !rope.k_cache || !rope.v_cache || !aligned16(rope.q_rope) ||
      !aligned16(rope.k_cache) || !aligned16(rope.v_cache) || mats[0].n != rope.q_heads * kTile ||
      mats[1].n != rope.kv_heads * kTile || mats[2].n != rope.kv_heads * kTile ||
      !one_launch(x, m, k, block_size, encoding, bits, mats, 3, &cols, &tile_cols))
    return EG_OK;
  *done = true;
  return over_rows(ctx, tile_for(ctx, m, tile_cols, k, block_size, cols, kRope), x, m, k, cols, norm, eps, normed,
                   [&](const Tile& t, const void* rows_x, int xm, uint32_t first, uint32_t rows) {
                     return launch_multi(ctx, rows_x, first, rows, k, block_size, encoding, mats, 3, cols, xm, kRope, t,
                                         norm, eps, &rope);
                   });
}

int eg::prefill_gemm_swiglu(eg_context* ctx, const float* x, uint32_t m, uint32_t k, uint32_t block_size,
                            int encoding, int bits, const PrefillMatrix& gate, const PrefillMatrix& up, float* out,
                            float* scratch, const float* norm, float eps, float* normed, bool out_bf16) {
  const char* op = "matmul_q4_prefill";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (!out || !scratch || gate.n != up.n)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: SwiGLU pair needs matching gate and up and two outputs", op);
  const uint32_t n = gate.n;
  // the pair as ONE launch of paired tiles where the chunked staging takes both, K is short and there are no biases
  const PrefillMatrix pair[2] = {{gate.packed, gate.scales, gate.zeros, gate.bias, nullptr, out, n, n, 0},
                                 {up.packed, up.scales, up.zeros, up.bias, nullptr, out, n, n, 0}};
  uint64_t cols = 0, tile_cols = 0;
  if (n == 0 || m == 0 || !ctx->prefill_pair || gate.bias || up.bias ||
      !one_launch(x, m, k, block_size, encoding, bits, pair, 2, &cols, &tile_cols)) {
    // otherwise gate | up side by side in the scratch rows, then SiLU(gate) * up
    const PrefillMatrix gu[2] = {{gate.packed, gate.scales, gate.zeros, gate.bias, nullptr, scratch, n, 2 * n, 0},
                                 {up.packed, up.scales, up.zeros, up.bias, nullptr, scratch, n, 2 * n, n}};
    int st = eg::prefill_gemm_multi(ctx, x, m, k, block_size, encoding, bits, gu, 2, norm, eps, normed);
    if (st == EG_OK && m > 0 && n > 0) st = eg::silu_mul_rows(ctx, scratch, m, n, out, out_bf16);
    return st;
  }
  const uint64_t pairs = (n + 31) / 32;
  return over_rows(ctx, tile_for(ctx, m, tile_cols, k, block_size, pairs, kPair), x, m, k, pairs, norm, eps, normed,
                   [&](const Tile& t, const void* rows_x, int xm, uint32_t first, uint32_t rows) {
                     return launch_multi(ctx, rows_x, first, rows, k, block_size, encoding, pair, 2, pairs, xm, kPair, t,
                                         norm, eps, nullptr, out_bf16);
                   });
}

extern "C" int eg_matmul_q4_prefill_swiglu(eg_context* ctx, const float* x, const uint32_t* gate_packed,
                                           const float* gate_scales, const uint32_t* gate_zeros,
                                           const uint32_t* up_packed, const float* up_scales, const uint32_t* up_zeros,
                                           float* out, float* scratch, const eg_matmul_q4_dims* dims, int encoding,
                                           int bits) {
  const char* op = "matmul_q4_prefill_swiglu";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (!dims || !x || !gate_packed || !gate_scales || !up_packed || !up_scales || !out || !scratch)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: NULL argument", op);
  if (dims->use_bias || dims->out_offset != 0 || (dims->m > 1 && dims->out_stride != dims->n))
    return eg::fail(ctx, EG_ERR_INVALID, "%s: no bias, out_stride n and out_offset 0 are required", op);
  if (dims->block_size == 0 || dims->k % dims->block_size != 0 || dims->blocks_per_row != dims->k / dims->block_size)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: k %u, block size %u and blocks per row %u disagree", op, dims->k,
                    dims->block_size, dims->blocks_per_row);
  if (dims->n % 4 != 0 || (reinterpret_cast<uintptr_t>(scratch) & 15u) || (reinterpret_cast<uintptr_t>(out) & 15u))
    return eg::fail(ctx, EG_ERR_INVALID, "%s: n %u must be a multiple of 4 and out, scratch 16-byte aligned", op,
                    dims->n);
  const eg::PrefillMatrix gate{gate_packed, gate_scales, gate_zeros, nullptr, nullptr, out, dims->n, dims->n, 0};
  const eg::PrefillMatrix up{up_packed, up_scales, up_zeros, nullptr, nullptr, out, dims->n, dims->n, 0};
  return eg::prefill_gemm_swiglu(ctx, x, dims->m, dims->k, dims->block_size, encoding, bits, gate, up, out, scratch);
}

extern "C" int eg_matmul_q4_prefill(eg_context* ctx, const float* x, const uint32_t* packed, const float* scales,
                                    const uint32_t* zeros, const float* bias, float* out,
                                    const eg_matmul_q4_dims* dims, int encoding, int bits) {
  return eg::prefill_gemm(ctx, x, packed, scales, zeros, bias, nullptr, out, dims, encoding, bits);
}
