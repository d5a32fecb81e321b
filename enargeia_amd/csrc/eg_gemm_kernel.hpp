// The prefill GEMM's kernel template (host side and launch rules: eg_gemm.hip).
//
//   out[r][col] = sum_k x[r][k] * W[col][k],  W[col][k] = (code - zero) * scale[block]
//
// with both operands rounded to bf16 and f32 sums in v_mfma_f32_32x32x16_bf16.
//
// W never passes through LDS. A lane of the MFMA's operand layout holds 8 consecutive k of one row
// of W: exactly one 32-bit word of int4 codes (two of int8). So each lane reads its row's codes
// from memory as the MFMA wants them - BK / 2 consecutive codes per chunk of BK - and dequantizes
// them in registers. What the waves share is x, and only x is staged in LDS. Against staging both
// (64 x 64 tiles, W dequantized into LDS by every workgroup) that takes W's LDS writes and reads
// away, and a wave's tile of 32 MF rows x 64 columns spreads the dequantization (about 2.6 VALU
// operations per weight) over 32 MF rows of products.
//
// The k order. Chunk c covers k in [c BK, (c + 1) BK); lane group g = lane / 32 owns k = g BK / 2 +
// [0, BK / 2) of it, and step s multiplies the groups' 8 k at offset 8 s. x is read from LDS in
// the same order, so any order gives the whole sum; it follows from BK, KG and the K splits, which
// tile_for chooses by one matrix's shape: the same bits whatever a launch folds into its epilogue.
//
// The products are formed transposed (W rows as the MFMA's A operand, x rows as B): lane l then
// holds, for row m = l % 32 of x, runs of four consecutive columns of W - one 16-byte store each,
// with a SwiGLU pair's gate and up and a RoPE pair's halves in the same lane.
//
// KG groups of WN waves share a workgroup: group q takes the chunks q, q + KG, ... (its own x
// buffers), wave wn of a group the 64 columns 64 (tx WN + wn); the groups' sums meet in LDS and are
// added in group order.
#pragma once

#include "eg_internal.hpp"

namespace eg_gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any float's address
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// One matrix of a launch: its streams, outputs and the end of its range of 64-column tiles. A
// multi-matrix launch holds several that share x, M, K, the quant block size and the encoding;
// the usual launch holds one.
struct Mat {
  const uint32_t* packed;
  const float* scales;
  const uint32_t* zeros;
  const float* bias;
  const float* residual;  // nullable: out = acc + bias + residual[r * out_stride + col + out_offset]
  float* out;
  uint32_t n, out_stride, out_offset, tiles_end;
};
constexpr uint32_t kMaxSegs = 3;
constexpr uint32_t kCols = 64;             // columns per wave
constexpr uint32_t kOutside = 0x80000000u;  // an offset past every stream (streams < 2 GiB here)

struct Args {
  const void* x;    // bf16 rows (kXBf16) or f32
  float* partials;  // split-K: [splits][m][n] f32; NULL without a split
  uint32_t m, k, block_shift, blocks_per_row, k_per_split;
  uint32_t tiles_x, tiles_y;  // workgroup tiles
  uint32_t nmats;             // matrices in mats (> 1: no K split)
  uint32_t xcd;               // order in which tiles are dealt to the XCDs (see tile_of)
  uint32_t vec;               // kPair: out takes 16-byte (out_bf16: 8-byte) stores, n a multiple of 4
  const float* norm;          // kXNorm: x is RMS-normalised per row with these weights (no K split)
  float eps;
  // kRope launches (q | k | v, 64-column tiles = heads): q rows rotated and scaled by 1/8 into
  // q_rope [row][q heads][64], k rows rotated and v rows as they are into the f16 caches at
  // positions rope_pos0 + row ([pos][kv_heads][64]); rope = the cos/sin table [pos][32]
  const double2* rope;
  float* q_rope;
  uint16_t* k_cache;
  uint16_t* v_cache;
  uint32_t rope_pos0, q_heads, kv_heads;
  uint32_t out_bf16;  // kPair: SiLU(g) * u stored as bf16 (the next GEMM's x, bit for bit what its
                      // staging would round it to)
  Mat mats[kMaxSegs];
};

enum XMode { kXBf16 = 0, kXF32 = 1, kXNorm = 2 };
enum Epilogue { kStore = 0, kPair = 1, kRope = 2 };

// SiLU(g) * u with SiLU(g) = g / (1 + e^-g), silu_mul_rows' formula.
__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// Workgroup L's tile. Workgroups go to the 8 XCDs in turn (L on XCD L % 8), each with its own L2.
// With `xcd` each XCD takes a contiguous run of the tiles: in column-major order (1: it reads an
// eighth of the weights and up to all of x) or row-major (2: an eighth of x and up to all of the
// weights); otherwise the grid's own row-major order.
__device__ __forceinline__ void tile_of(const Args& a, uint32_t& tx, uint32_t& ty) {
  uint32_t id = blockIdx.x;
  if (a.xcd) {
    const uint32_t total = a.tiles_x * a.tiles_y, q = total / 8u, r = total % 8u, xcd = id % 8u;
    id = xcd * q + min(xcd, r) + id / 8u;
  }
  if (a.xcd == 1u) {
    tx = id / a.tiles_y;
    ty = id % a.tiles_y;
  } else {
    tx = id % a.tiles_x;
    ty = id / a.tiles_x;
  }
}

__device__ __forceinline__ half2v halves(uint32_t v) { return __builtin_bit_cast(half2v, v); }

// 8 codes of a block to 8 bf16 weights: RN_bf16((code - zero) * scale). A code masked into the low
// ten bits of an f16 1024.0 reads 1024 + code exactly (a high nibble, left in place, 1024 + 16 code);
// adding -(1024 + zero) leaves code - zero exactly; v_fma_mix_f32 multiplies that half by the f32
// scale (a high nibble's by scale / 16, exact) - one rounding, as (code - zero) * scale has - and
// v_cvt_pk_bf16_f32 rounds two at a time. Two's-complement codes are flipped to offset binary in
// the mask (one v_bitop3). zl, zh: -(1024 + zero) and -(1024 + 16 zero) in both halves.
template <int ENC>
__device__ __forceinline__ bf16x8 dequant4(uint32_t d, float s, uint32_t zl, uint32_t zh) {
  constexpr uint32_t lo = ENC == EG_ENC_SIGNED ? 0x64086408u : 0x64006400u;
  constexpr uint32_t hi = ENC == EG_ENC_SIGNED ? 0x64806480u : 0x64006400u;
  const uint32_t d8 = d >> 8;
  const float s16 = s * 0.0625f;
  const half2v a = halves((d & 0x000F000Fu) ^ lo) + halves(zl);   // elements 0 | 4
  const half2v b = halves((d & 0x00F000F0u) ^ hi) + halves(zh);   // 1 | 5
  const half2v c = halves((d8 & 0x000F000Fu) ^ lo) + halves(zl);  // 2 | 6
  const half2v e = halves((d8 & 0x00F000F0u) ^ hi) + halves(zh);  // 3 | 7
  const uint4 r = make_uint4(egd::pack_bf16(fmaf((float)a.x, s, 0.f), fmaf((float)b.x, s16, 0.f)),
                             egd::pack_bf16(fmaf((float)c.x, s, 0.f), fmaf((float)e.x, s16, 0.f)),
                             egd::pack_bf16(fmaf((float)a.y, s, 0.f), fmaf((float)b.y, s16, 0.f)),
                             egd::pack_bf16(fmaf((float)c.y, s, 0.f), fmaf((float)e.y, s16, 0.f)));
  return __builtin_bit_cast(bf16x8, r);
}

// The same for int8 codes: 1024 + code is exact up to 2047.
template <int ENC>
__device__ __forceinline__ bf16x8 dequant8(uint32_t d0, uint32_t d1, float s, uint32_t zl) {
  constexpr uint32_t flip = ENC == EG_ENC_SIGNED ? 0x64806480u : 0x64006400u;
  uint32_t r[4];
#pragma unroll
  for (int w = 0; w < 2; w++) {
    const uint32_t d = w ? d1 : d0;
    const half2v a = halves((d & 0x00FF00FFu) ^ flip) + halves(zl);         // elements 0 | 2
    const half2v b = halves(((d >> 8) & 0x00FF00FFu) ^ flip) + halves(zl);  // 1 | 3
    r[2 * w] = egd::pack_bf16(fmaf((float)a.x, s, 0.f), fmaf((float)b.x, s, 0.f));
    r[2 * w + 1] = egd::pack_bf16(fmaf((float)a.y, s, 0.f), fmaf((float)b.y, s, 0.f));
  }
  return __builtin_bit_cast(bf16x8, make_uint4(r[0], r[1], r[2], r[3]));
}

template <int ENC, int BITS, int BK, int MF, int WN, int KG, int XM, int EPI>
__global__ __launch_bounds__(64 * WN * KG, 2) void gemm_kernel(Args a) {
  // No contraction of separate operations into fused multiply-adds (the explicit fmaf calls stay):
  // every epilogue then rounds the row's norm scale and the bias addition on their own, so the
  // launches that fold different work into their epilogues give the same values.
#pragma clang fp contract(off)
  constexpr uint32_t TM = 32 * MF, kSlots = BK / 8, kSteps = BK / 16;
  constexpr uint32_t kRowBytes = BK * 2, kBuf = TM * kRowBytes;  // one x buffer of one group
  constexpr uint32_t kWords = BK / 2 * BITS / 32;                // code words per lane, row and chunk
  constexpr uint32_t kWave = 64 * TM * 4;                        // a wave's sums in bytes
  constexpr uint32_t kLds = 2 * KG * kBuf > (KG > 1 ? KG * WN * kWave : 0) ? 2 * KG * kBuf : KG * WN * kWave;
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLds];
  __shared__ float row_ss[XM == kXNorm ? KG : 1][TM];  // kXNorm: each group's sums of squares per row
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t group = wave / WN, wn = wave % WN, gtid = tid - group * (64u * WN);
  const uint32_t lr = lane & 31u, g = lane >> 5;
  uint32_t tx, ty;
  tile_of(a, tx, ty);
  const uint32_t m0 = ty * TM;

  // This wave's 64 columns: 64-column tile t of the launch's list (a tile past its end repeats the
  // last and stores nothing), as two fragments of 32 rows of W. kPair: rows 32 t .. of mats[0] (gate)
  // in fragment 0, the same rows of mats[1] (up) in 1.
  const uint32_t tiles = a.mats[EPI == kPair ? 0 : a.nmats - 1].tiles_end;
  const bool active = tx * WN + wn < tiles;
  const uint32_t t = min(tx * WN + wn, tiles - 1);
  uint32_t si = 0;
  if (EPI != kPair) {
#pragma unroll
    for (uint32_t i = 0; i + 1 < kMaxSegs; i++)
      if (i + 1 < a.nmats && t >= a.mats[i].tiles_end) si = i + 1;
  }
  const Mat& w0 = a.mats[si];
  const Mat& w1 = a.mats[EPI == kPair ? 1 : si];
  const uint32_t n0 = EPI == kPair ? 32u * t : (t - (w0.tiles_end - (w0.n + kCols - 1) / kCols)) * kCols;
  const uint32_t kbeg = blockIdx.y * a.k_per_split, kend = min(a.k, kbeg + a.k_per_split);
  const uint32_t nchunks = (kend - kbeg + BK - 1) / BK, iters = (nchunks + KG - 1) / KG;

  // ---- W: codes, scales and zero-point words per fragment, in flight one chunk ahead. A lane's BK /
  // 2 codes take two scales (a block is at least BK / 4 codes; of one block, the same scale twice).
  // Lanes past K (and fragments' rows past the matrix) read zeros: weights of zero.
  struct Weights {
    uint32_t q[2][kWords], zw[2][2];
    float s[2][2];
  };
  constexpr uint32_t kPer = 32 / BITS;  // zero-points per word
  const __amdgpu_buffer_rsrc_t wr[2] = {egd::buffer(w0.packed, w0.n * (a.k / 8u * BITS)),
                                        egd::buffer(w1.packed, w1.n * (a.k / 8u * BITS))};
  const __amdgpu_buffer_rsrc_t sr[2] = {egd::buffer(w0.scales, w0.n * a.blocks_per_row * 4u),
                                        egd::buffer(w1.scales, w1.n * a.blocks_per_row * 4u)};
  const __amdgpu_buffer_rsrc_t zr[2] = {
      egd::buffer(w0.zeros, ((w0.n * a.blocks_per_row + kPer - 1) / kPer) * 4u),
      egd::buffer(w1.zeros, ((w1.n * a.blocks_per_row + kPer - 1) / kPer) * 4u)};
  // Byte offsets of the lane's codes and scales in chunk 0 (kOutside past the rows) and its blocks
  // there; a chunk's own offsets are uniform (K is split at multiples of BK, a power of two like the
  // block), so they ride in the scalar offset of the loads.
  uint32_t woff[2], soff[2][2], wblk[2][2];
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const uint32_t row = n0 + (EPI == kPair ? 0u : 32u * f) + lr, out = row < w0.n ? 0u : kOutside;
    woff[f] = (row * (a.k / 8u * BITS) + g * (BK / 16 * BITS)) | out;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      wblk[f][h] = row * a.blocks_per_row + ((g * (BK / 2) + h * (BK / 4)) >> a.block_shift);
      soff[f][h] = (wblk[f][h] * 4u) | out;
    }
  }
  // load j of a chunk's weights: the code loads, two scales and two zero-point words per fragment.
  // past[h]: kOutside where the lane's half h of the chunk lies past K.
  constexpr uint32_t kCodeLoads = kWords / 4, kWLoads = 2 * (kCodeLoads + 2 + (ENC == EG_ENC_OFFSET_ZEROS ? 2 : 0));
  static_assert(kWords % 4 == 0, "whole 16-byte code loads");
  auto load_w = [&](uint32_t j, uint32_t k0, const uint32_t (&past)[2], Weights& w) {
    const uint32_t f = j & 1u, n = j >> 1, i = EPI == kPair ? f : 0u, b0 = k0 >> a.block_shift;
    if (n < kCodeLoads) {
      // (whole in K or whole past it: K is a multiple of 32)
      const egd::u32x4 v = egd::load_b128(wr[i], (woff[f] | past[n * (128 / BITS) / (BK / 4)]) + 16u * n, k0 / 8u * BITS);
      w.q[f][4 * n] = v.x;
      w.q[f][4 * n + 1] = v.y;
      w.q[f][4 * n + 2] = v.z;
      w.q[f][4 * n + 3] = v.w;
    } else {
      const uint32_t h = (n - kCodeLoads) & 1u;
      if (n < kCodeLoads + 2) w.s[f][h] = egd::load_f32(sr[i], soff[f][h] | past[h], b0 * 4u);
      else w.zw[f][h] = egd::load_b32(zr[i], ((wblk[f][h] + b0) / kPer * 4u) | (soff[f][h] & kOutside) | past[h]);
    }
  };

  // ---- x: rows m0 .. of a chunk into a buffer of this group, slot j (8 values) of row r at LDS slot
  // j ^ (r % slots), so that the rows an operand read touches fall on different banks. Rows past M
  // lie past the end of x and read as zeros, as slots past K do.
  uint8_t* const xbuf = lds + group * (2 * kBuf);
  const __amdgpu_buffer_rsrc_t xr = egd::buffer(a.x, a.m * a.k * (XM == kXBf16 ? 2u : 4u));
  // kXBf16: memory to LDS directly, 1 KiB (64 lanes x 16 bytes) per load
  constexpr uint32_t kRowsPer = 64 / kSlots, kDma = TM / (kRowsPer * WN);
  // otherwise through registers: 8 f32 values per slot, rounded (after the norm weights) on the way
  constexpr uint32_t kReg = XM == kXBf16 ? 1 : TM * kSlots / (64 * WN);
  constexpr uint32_t kXLoads = XM == kXBf16 ? kDma : 2 * kReg + (XM == kXNorm ? 2 : 0);
  egd::u32x4 xv[kReg][2], xg[2];
  float ss[XM == kXNorm ? kReg : 1] = {};
  const __amdgpu_buffer_rsrc_t gr = egd::buffer(XM == kXNorm ? a.norm : nullptr, XM == kXNorm ? a.k * 4u : 0u);
  // Load j covers rows j kStride + xrow. The slot swizzle of its row is the thread's own, x_swz, with
  // bits that depend on j alone flipped: the thread's column in it takes kSwz values.
  constexpr uint32_t kStride = XM == kXBf16 ? kRowsPer * WN : 64 * WN / kSlots;
  constexpr uint32_t kSwz = XM == kXBf16 && kStride < kSlots ? kSlots / kStride : 1;
  const uint32_t xrow = XM == kXBf16 ? wn * kRowsPer + lane / kSlots : gtid / kSlots;
  const uint32_t xcol = XM == kXBf16 ? (lane % kSlots) ^ (xrow & (kSlots - 1)) : gtid % kSlots;
  const uint32_t xbase = ((m0 + xrow) * a.k + kbeg) * (XM == kXBf16 ? 2u : 4u);
  struct XOffsets {
    uint32_t at[kSwz];  // kOutside where the column lies past K
  };
  auto x_offsets = [&](uint32_t k0, XOffsets& o) {
#pragma unroll
    for (uint32_t c = 0; c < kSwz; c++) {
      const uint32_t col = xcol ^ (c * kStride);
      o.at[c] = (xbase + (k0 - kbeg + 8u * col) * (XM == kXBf16 ? 2u : 4u)) | (k0 + 8u * col < kend ? 0u : kOutside);
    }
  };
  auto load_x = [&](uint32_t j, uint32_t k0, const XOffsets& o, uint32_t buf) {
    if (XM == kXBf16) {
      egd::load_to_lds(xr, xbuf + buf * kBuf + (j * WN + wn) * 1024u, o.at[j % kSwz] + j * kStride * a.k * 2u);
    } else if (j < 2 * kReg) {
      xv[j >> 1][j & 1u] = egd::load_b128(xr, o.at[0] + (j >> 1) * kStride * a.k * 4u + 16u * (j & 1u));
    } else {
      const uint32_t kk = k0 + 8u * xcol;
      xg[j & 1u] = egd::load_b128(gr, (kk * 4u + 16u * (j & 1u)) | (kk < kend ? 0u : kOutside));
    }
  };
  auto store_x = [&](uint32_t buf) {
    if (XM == kXBf16) return;
#pragma unroll
    for (uint32_t i = 0; i < kReg; i++) {
      const uint32_t r = (gtid + i * (64u * WN)) / kSlots, j = gtid % kSlots;
      uint32_t p[4];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float v[4] = {__uint_as_float(xv[i][h].x), __uint_as_float(xv[i][h].y), __uint_as_float(xv[i][h].z),
                      __uint_as_float(xv[i][h].w)};
        if (XM == kXNorm) {
          // x times its column's norm weight here, the row's 1 / rms in the epilogue
          const float gw[4] = {__uint_as_float(xg[h].x), __uint_as_float(xg[h].y), __uint_as_float(xg[h].z),
                               __uint_as_float(xg[h].w)};
#pragma unroll
          for (int e = 0; e < 4; e++) {
            ss[XM == kXNorm ? i : 0] = fmaf(v[e], v[e], ss[XM == kXNorm ? i : 0]);
            v[e] *= gw[e];
          }
        }
        p[2 * h] = egd::pack_bf16(v[0], v[1]);
        p[2 * h + 1] = egd::pack_bf16(v[2], v[3]);
      }
      *reinterpret_cast<uint4*>(xbuf + buf * kBuf + r * kRowBytes + 16u * (j ^ (r & (kSlots - 1)))) =
          make_uint4(p[0], p[1], p[2], p[3]);
    }
  };
  auto settle = [&]() {
    if (XM == kXBf16) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0: the memory-to-LDS loads have landed
    __syncthreads();
  };

  f32x16 acc[2][MF];
#pragma unroll
  for (int f = 0; f < 2; f++)
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[f][i][e] = 0.f;

  // One chunk's products from x buffer `buf` and weights w, with the loads of the group's next chunk (into the
  // other buffer and w_next) issued along the way. In 2 kSteps parts: part p multiplies the step's x
  // fragments by one column fragment's weights while the next part's weights are dequantized, and
  // the second part of a step frees its x fragments one by one for the next step's reads. The
  // scheduling barriers and groups hold the compiler to that interleaving: VALU work overlaps an
  // MFMA only inside its own wave's stream (a wave of MFMAs and a wave of VALU operations on one SIMD
  // take the sum of their times, measured), and loads issued in one burst stall the stream.
  auto past_of = [&](uint32_t k0, uint32_t (&past)[2]) {
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) past[h] = k0 + g * (BK / 2) + h * (BK / 4) < kend ? 0u : kOutside;
  };
  auto multiply = [&](uint32_t chunk, uint32_t buf, const Weights& w, Weights& w_next) {
    const uint32_t b0 = (kbeg + chunk * BK) >> a.block_shift, next = kbeg + (chunk + KG) * BK;
    uint32_t past[2];
    XOffsets xo;
    past_of(next, past);
    x_offsets(next, xo);
    uint32_t zl[2][2], zh[2][2];
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        if (ENC == EG_ENC_SIGNED) {
          zl[f][h] = BITS == 4 ? 0xE408E408u : 0xE480E480u;
          zh[f][h] = 0xE480E480u;
        } else {
          const uint32_t blk = wblk[f][h] + b0;
          const uint32_t z = (w.zw[f][h] >> (BITS * (blk % kPer))) & ((1u << BITS) - 1u);
          zl[f][h] = (0xE400u | z) * 0x10001u;
          zh[f][h] = (0xE400u | (z << 4)) * 0x10001u;
        }
      }
    const uint8_t* xb = xbuf + buf * kBuf + lr * kRowBytes;
    auto weight = [&](uint32_t s, int f) {
      const uint32_t h = s / (kSteps / 2);
      if constexpr (BITS == 4) return dequant4<ENC>(w.q[f][s], w.s[f][h], zl[f][h], zh[f][h]);
      else return dequant8<ENC>(w.q[f][2 * s], w.q[f][2 * s + 1], w.s[f][h], zl[f][h]);
    };
    auto rows = [&](uint32_t s, uint32_t i) {
      const uint32_t slot = 16u * ((g * kSteps + s) ^ (lr & (kSlots - 1)));
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(xb + i * (32 * kRowBytes) + slot));
    };
    constexpr uint32_t kParts = 2 * kSteps, kLoads = kXLoads + kWLoads, kShare = (kLoads + kParts - 1) / kParts;
    bf16x8 wf[2], xf[MF];
    wf[0] = weight(0, 0);
#pragma unroll
    for (uint32_t i = 0; i < MF; i++) xf[i] = rows(0, i);
#pragma unroll
    for (uint32_t p = 0; p < kParts; p++) {
      const uint32_t s = p / 2, f = p % 2;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (uint32_t j = p * kShare; j < (p + 1) * kShare; j++) {
        if (j < kXLoads) load_x(j, next, xo, buf ^ 1u);
        else if (j < kLoads) load_w(j - kXLoads, next, past, w_next);
      }
      if (p + 1 < kParts) wf[(p + 1) & 1u] = weight((p + 1) / 2, (p + 1) % 2);
#pragma unroll
      for (uint32_t i = 0; i < MF; i++) {
        acc[f][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[p & 1u], xf[i], acc[f][i], 0, 0, 0);
        if (f == 1 && s + 1 < kSteps) xf[i] = rows(s + 1, i);
      }
#pragma unroll
      for (uint32_t i = 0; i < MF; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (f == 1 && s + 1 < kSteps) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 28 / MF, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Two x buffers per group: a chunk's x and weights are in flight while the one before it is
  // multiplied. (Chunks past the last are all zeros.)
  Weights wa;
  {
    const uint32_t k0 = kbeg + group * BK;
    uint32_t past[2];
    XOffsets xo;
    past_of(k0, past);
    x_offsets(k0, xo);
#pragma unroll
    for (uint32_t j = 0; j < kXLoads; j++) load_x(j, k0, xo, 0);
#pragma unroll
    for (uint32_t j = 0; j < kWLoads; j++) load_w(j, k0, past, wa);
  }
  store_x(0);
  settle();
  for (uint32_t it = 0; it < iters; it++) {
    const uint32_t buf = it & 1u;
    Weights wb;
    multiply(group + KG * it, buf, wa, wb);
    // (not the last: it would wait for loads past K to convert their zeros; 1 x 64 x 256 4.4 -> 3.8 us)
    if (it + 1 < iters) store_x(buf ^ 1u);
    settle();
    wa = wb;
  }

  if (XM == kXNorm) {
    // the kSlots threads of a row hold its columns
#pragma unroll
    for (uint32_t i = 0; i < kReg; i++) {
      float v = ss[XM == kXNorm ? i : 0];
#pragma unroll
      for (uint32_t off = 1; off < kSlots; off <<= 1) v += __shfl_xor(v, off, 64);
      if (gtid % kSlots == 0) row_ss[XM == kXNorm ? group : 0][(gtid + i * (64u * WN)) / kSlots] = v;
    }
    __syncthreads();
  }

  // ---- epilogue: unit (i, p) = row fragment i with columns 8 p + 4 g .. +4 of both column fragments --
  // kRope: cos and sin of unit (i, p)'s four pairs and their biases, which the callers read ahead of the
  // sums (read where they are added, the biases took a round trip to memory per unit: q|k|v of 2048 rows,
  // its norm's launch included, 28.5 us for 23.2)
  struct Ahead {
    double2 cs[EPI == kRope ? 4 : 1];
    f32x4 bias[2];
  };
  auto read_ahead = [&](uint32_t i, uint32_t p, Ahead& c) {
    if (EPI != kRope) return;
    const float* b = w0.bias ? w0.bias + n0 + 8u * p + 4u * g : nullptr;
#pragma unroll
    for (int h = 0; h < 2; h++) c.bias[h] = b ? (f32x4)*reinterpret_cast<const f32x4u*>(b + 32 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
    if (si == 2) return;
    const uint32_t row = min(m0 + 32u * i + lr, a.m - 1);
#pragma unroll
    for (int e = 0; e < 4; e++) c.cs[EPI == kRope ? e : 0] = a.rope[(size_t)(a.rope_pos0 + row) * 32u + 8u * p + 4u * g + e];
  };
  // 1 / rms of row r of the tile, the groups' sums of squares added in group order
  auto inv_rms = [&](uint32_t r) {
    float sum = row_ss[0][r];
#pragma unroll
    for (int q = 1; q < (XM == kXNorm ? KG : 1); q++) sum += row_ss[q][r];
    return 1.0f / sqrtf(sum / (float)a.k + a.eps);
  };
  // One value of a row, and columns col .. +4 of it in one access wherever the rows start.
  auto store1 = [&](uint32_t row, uint32_t col, float v) {
    if (a.partials) {
      a.partials[((size_t)blockIdx.y * a.m + row) * w0.n + col] = v;
      return;
    }
    const size_t o = (size_t)row * w0.out_stride + col + w0.out_offset;
    w0.out[o] = v + (w0.bias ? w0.bias[col] : 0.f) + (w0.residual ? w0.residual[o] : 0.f);
  };
  // (their biases, the same for every row, are read once, ahead of the sums: read at each store they took
  // 256 x 4864 x 896 1.0 us)
  auto bias4 = [&](uint32_t col) {
    return !a.partials && w0.bias && active && col + 4 <= w0.n ? (f32x4)*reinterpret_cast<const f32x4u*>(w0.bias + col)
                                                               : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto store4 = [&](uint32_t row, uint32_t col, f32x4 v, f32x4 bias) {
    if (a.partials) {
      *reinterpret_cast<f32x4u*>(a.partials + ((size_t)blockIdx.y * a.m + row) * w0.n + col) = v;
      return;
    }
    const size_t o = (size_t)row * w0.out_stride + col + w0.out_offset;
    const f32x4 res = w0.residual ? (f32x4)*reinterpret_cast<const f32x4u*>(w0.residual + o) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = v[e] + bias[e] + res[e];
    *reinterpret_cast<f32x4u*>(w0.out + o) = v;
  };
  auto finish = [&](uint32_t i, uint32_t p, f32x4 lo, f32x4 hi, const Ahead& ahead) {
    const uint32_t r = 32u * i + lr, row = m0 + r;
    if (!active || row >= a.m) return;
    if (XM == kXNorm) {
      const float inv = inv_rms(r);
      lo *= inv;
      hi *= inv;
    }
    if (EPI == kPair) {
      const uint32_t col = n0 + 8u * p + 4u * g;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = silu_mul(lo[e] + 0.f, hi[e] + 0.f);  // (-0 to 0, as the stored sums)
      const size_t o = (size_t)row * w0.out_stride + col + w0.out_offset;
      if (a.vec) {
        if (col >= w0.n) return;
        if (a.out_bf16)
          *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(w0.out) + o) =
              make_uint2(egd::pack_bf16(v[0], v[1]), egd::pack_bf16(v[2], v[3]));
        else
          *reinterpret_cast<float4*>(w0.out + o) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (col + e >= w0.n) continue;
          if (a.out_bf16) reinterpret_cast<uint16_t*>(w0.out)[o + e] = (uint16_t)egd::pack_bf16(v[e], 0.f);
          else w0.out[o + e] = v[e];
        }
      }
      return;
    }
    if (EPI == kRope) {  // a tile is one head: elements e and e + 32 are in lo and hi
      const uint32_t hd = n0 / kCols, c = 8u * p + 4u * g;
      float x[4], y[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        x[e] = lo[e] + ahead.bias[0][e] + 0.f;
        y[e] = hi[e] + ahead.bias[1][e] + 0.f;
        if (si < 2) {
          const float2 rr = egd::rotate(x[e], y[e], ahead.cs[EPI == kRope ? e : 0]);
          x[e] = rr.x;
          y[e] = rr.y;
        }
      }
      if (si == 0) {
        float* dst = a.q_rope + ((size_t)row * a.q_heads + hd) * kCols + c;
        *reinterpret_cast<float4*>(dst) = make_float4(x[0] * 0.125f, x[1] * 0.125f, x[2] * 0.125f, x[3] * 0.125f);
        *reinterpret_cast<float4*>(dst + 32) = make_float4(y[0] * 0.125f, y[1] * 0.125f, y[2] * 0.125f, y[3] * 0.125f);
      } else {
        uint16_t* dst = (si == 1 ? a.k_cache : a.v_cache) + ((size_t)(a.rope_pos0 + row) * a.kv_heads + hd) * kCols + c;
        auto half4 = [](const float* v) {
          return make_uint2((uint32_t)egd::float_to_half(v[0]) | ((uint32_t)egd::float_to_half(v[1]) << 16),
                            (uint32_t)egd::float_to_half(v[2]) | ((uint32_t)egd::float_to_half(v[3]) << 16));
        };
        *reinterpret_cast<uint2*>(dst) = half4(x);
        *reinterpret_cast<uint2*>(dst + 32) = half4(y);
      }
      return;
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const uint32_t col = n0 + 8u * p + 32u * h + 4u * g;
      const f32x4 v = h ? hi : lo;
      if (col + 4 <= w0.n) {
        store4(row, col, v, ahead.bias[h]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (col + e < w0.n) store1(row, col + e, v[e]);
      }
    }
  };

  auto run = [](const f32x16& v, int p) { return f32x4{v[4 * p], v[4 * p + 1], v[4 * p + 2], v[4 * p + 3]}; };
  if constexpr (KG == 1) {
    f32x4 bias[EPI == kStore ? 4 : 1][2];
    if (EPI == kStore) {
#pragma unroll
      for (int p = 0; p < 4; p++)
#pragma unroll
        for (int h = 0; h < 2; h++) bias[EPI == kStore ? p : 0][h] = bias4(n0 + 8u * p + 32u * h + 4u * g);
    }
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
      for (int p = 0; p < 4; p++) {
        Ahead ahead;
        read_ahead(i, p, ahead);
        if (EPI == kStore) {
          ahead.bias[0] = bias[EPI == kStore ? p : 0][0];
          ahead.bias[1] = bias[EPI == kStore ? p : 0][1];
        }
        finish(i, p, run(acc[0][i], p), run(acc[1][i], p), ahead);
        __builtin_amdgcn_sched_barrier(0);  // one unit at a time: together they spill
      }
  } else if constexpr (EPI == kStore) {
    // Every wave's sums into LDS (the last barrier ended the staging), then rows of 64 columns shared out
    // over the groups: 16 lanes take the 16 runs of four columns of a row, 256 bytes in one store. Run
    // (f, p, g) of row lr is kept at slot lane ^ (4 f + p + 8 g) of its 64, which puts the 16 on different
    // banks. The run that n cuts comes after them, a value per lane: with its stores in every unrolled step
    // the launch took 1.2 to 2.5 us longer (749 x 1086 x 320 8.8 us, 749 x 1088 7.7), for instruction fetches.
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);
    auto at = [&](uint32_t q, uint32_t f, uint32_t u, uint32_t l) {
      return ((q * WN + wn) * (8u * MF) + f * (4 * MF) + u) * 64u + (l ^ (4u * f + (u & 3u) + 8u * (l >> 5)));
    };
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int u = 0; u < 4 * MF; u++) sums[at(group, f, u, lane)] = run(acc[f][u / 4], u % 4);
    const uint32_t c = lane & 15u, f = c >> 3, p = (c >> 1) & 3u;
    const f32x4 bias = bias4(n0 + 4u * c);
    __syncthreads();
    if (!active) return;
#pragma unroll
    for (uint32_t v = 0; v < 8u * MF / KG; v++) {
      const uint32_t r = (group + v * KG) * 4u + (lane >> 4), u = (r >> 5) * 4u + p, l = (r & 31u) + 32u * (c & 1u);
      f32x4 x = sums[at(0, f, u, l)];
#pragma unroll
      for (int q = 1; q < KG; q++) x += sums[at(q, f, u, l)];
      if (m0 + r >= a.m || n0 + 4u * c + 4u > w0.n) continue;
      if (XM == kXNorm) x *= inv_rms(r);
      store4(m0 + r, n0 + 4u * c, x, bias);
    }
    const uint32_t cut = w0.n & ~3u;  // the cut run's first column
    if (n0 + kCols <= cut || cut == w0.n) return;
    const uint32_t cc = cut - n0, r = (group * 64u + lane) % TM;
    if (m0 + r >= a.m) return;
    const uint32_t cf = cc >> 5, cu = (r >> 5) * 4u + ((cc >> 3) & 3u), cl = (r & 31u) + 32u * ((cc >> 2) & 1u);
#pragma unroll 1
    for (uint32_t e = (group * 64u + lane) / TM; e < (w0.n & 3u); e += KG * 64u / TM) {
      float x = sums[at(0, cf, cu, cl)][e];
#pragma unroll
      for (int q = 1; q < KG; q++) x += sums[at(q, cf, cu, cl)][e];
      if (XM == kXNorm) x *= inv_rms(r);
      store1(m0 + r, cut + e, x);
    }
  } else {
    // every wave's sums into LDS as its lanes hold them (the last barrier ended the staging), then
    // the units shared out over the groups
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);
    auto at = [&](uint32_t q, uint32_t f, uint32_t u) { return ((q * WN + wn) * (8u * MF) + f * (4 * MF) + u) * 64u + lane; };
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
      for (int u = 0; u < 4 * MF; u++) sums[at(group, f, u)] = run(acc[f][u / 4], u % 4);
    static_assert(4 * MF % KG == 0, "the groups share the units");
    Ahead ahead[4 * MF / KG];
#pragma unroll
    for (uint32_t v = 0; v < 4u * MF / KG; v++) read_ahead((group + v * KG) / 4, (group + v * KG) % 4, ahead[v]);
    __syncthreads();
#pragma unroll
    for (uint32_t v = 0; v < 4u * MF / KG; v++) {
      const uint32_t u = group + v * KG;
      f32x4 lo = sums[at(0, 0, u)], hi = sums[at(0, 1, u)];
#pragma unroll
      for (int q = 1; q < KG; q++) {
        lo += sums[at(q, 0, u)];
        hi += sums[at(q, 1, u)];
      }
      finish(u / 4, u % 4, lo, hi, ahead[v]);
    }
  }
}

using KernelFn = void (*)(Args);

// A launch's shape: BK, MF, WN and KG of the kernel.
struct Tile {
  int bk, mf, wn, kg;
  uint32_t rows() const { return 32u * mf; }
  // which kernels there are: the largest take bf16 rows of x only (f32 rows staged through registers do
  // not fit beside the sums), those for a long K store plain results, and the RMSNorm is folded into
  // launches of few tiles only, which take the small ones
  bool bf16_only() const { return mf * wn * kg >= 16; }
  bool store_only() const { return bk == 128 && wn == 2; }
  bool folds_norm() const { return wn == 1; }
  // the tile that takes a bf16_only one's f32 rows: its chunks and K groups, half its rows or columns
  Tile f32_form() const { return kg == 4 ? Tile{bk, mf, wn / 2, kg} : Tile{bk, mf / 2, wn, kg}; }
};

// The tiles: {BK, MF, WN, KG}. eg_gemm.hip's tile_for chooses among them.
constexpr Tile kTile32x64{128, 1, 1, 4}, kTile64x64{128, 2, 1, 4}, kTile64x128{64, 2, 2, 2}, kTile64x128Long{128, 2, 2, 2},
    kTile64x128Deep{128, 2, 2, 4}, kTile64x256{128, 2, 4, 1}, kTile128x128{128, 4, 2, 2}, kTile128x256{128, 4, 4, 1},
    kTile32x64Fine{64, 1, 1, 4}, kTile64x64Fine{64, 2, 1, 4};
constexpr Tile kTiles[] = {kTile32x64,  kTile64x64,   kTile64x128,  kTile64x128Long, kTile64x128Deep,
                           kTile64x256, kTile128x128, kTile128x256, kTile32x64Fine,  kTile64x64Fine};

template <int ENC, int BITS, int XM, int EPI>
KernelFn pick_tile(const Tile& t) {
#define EG_GEMM_CASE(B, M, W, G) \
  if (t.bk == B && t.mf == M && t.wn == W && t.kg == G) return gemm_kernel<ENC, BITS, B, M, W, G, XM, EPI>;
  EG_GEMM_CASE(128, 1, 1, 4)
  EG_GEMM_CASE(128, 2, 1, 4)
  EG_GEMM_CASE(64, 1, 1, 4)
  EG_GEMM_CASE(64, 2, 1, 4)
  if constexpr (XM != kXNorm) {
    EG_GEMM_CASE(64, 2, 2, 2)
    EG_GEMM_CASE(128, 2, 4, 1)
    if constexpr (EPI == kStore) {
      EG_GEMM_CASE(128, 2, 2, 2)
    }
  }
  if constexpr (XM == kXBf16) {
    if constexpr (EPI == kStore) {
      EG_GEMM_CASE(128, 2, 2, 4)
      EG_GEMM_CASE(128, 4, 2, 2)
    }
    EG_GEMM_CASE(128, 4, 4, 1)
  }
#undef EG_GEMM_CASE
  return nullptr;
}

// One translation unit per x mode and epilogue group, so they compile in parallel.
KernelFn pick_store_bf16(int encoding, int bits, const Tile& t);
KernelFn pick_store_f32(int encoding, int bits, const Tile& t);
KernelFn pick_store_norm(int encoding, const Tile& t);
KernelFn pick_pair(int encoding, int xm, const Tile& t);
KernelFn pick_rope(int encoding, int xm, const Tile& t);

}  // namespace eg_gemm
