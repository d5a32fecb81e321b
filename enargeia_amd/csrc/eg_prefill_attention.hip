// Chunked-prefill attention on the matrix cores: the reference's attn_scores -> softmax ->
// attn_apply over the KV cache (cache_variants.ts:81-145, graph.ts:435-459), with the RoPE and
// cache writes that precede them (rope.wgsl via graph.ts:411-430, k_pack / v_pack).
//
// A chunk of `queries` rows starting at absolute position `query_begin` attends causally over
// keys [0, query_begin + i] of the cache (query i; the reference's mask `j > i + queryBegin`).
//
// Two launches:
//   1. rope_append: RoPE on the chunk's q and k rows (double-precision angles, as the decode
//      path), q pre-scaled by 1/sqrt(D) into q_rope, k and v appended to the f16 caches at
//      positions [query_begin, query_begin + queries).
//   2. attention: flash attention, one workgroup per (64 queries, head), 16 queries per wave.
//      Key tiles of 64 are staged through LDS; S = Q K^T and
//      O += P V run on v_mfma_f32_16x16x32_f16 (f16 operands - the cache is f16 already, q and
//      the softmax weights are rounded to f16 - with f32 accumulation), the softmax is the
//      online (running max / sum) form in f32, masked scores are the reference's NEG_LARGE.
//      Only key tiles up to the workgroup's last query's causal limit are visited.
//      When those workgroups would leave most CUs idle over a long key range (a late chunk of a
//      long prompt: 4 x 14 workgroups walking up to 32 tiles at 2048 keys), the keys are split
//      over grid.z: each split writes its rows' unnormalised o and (max, sum) to the context's
//      workspace and 3. a combine launch merges the splits in split order.
//
// The f32 cache variant (eg_attention_prefill_f32; cache_variants.ts:21-40 generates the same
// kernels per cache dtype) appends exact f32 rows and runs the attention on the f32 matrix cores.
#include <algorithm>
#include <type_traits>

#include "eg_internal.hpp"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any float's address

constexpr int kD = 64;           // head_dim (the path's models)
constexpr int kQ = 64;           // queries per workgroup
constexpr int kK = 64;           // keys per tile
constexpr float kMasked = -1.0e30f;  // NEG_LARGE, cache_variants.ts

using egd::float_to_half;

// A value as the cache holds it: f16 bits or the f32 itself.
template <class CT>
__device__ __forceinline__ CT to_cache(float x) {
  if constexpr (std::is_same<CT, float>::value) return x;
  else return float_to_half(x);
}

// One workgroup per row. Bound by a chain of latencies: the row's read, the double-precision angles and
// the stores; so the pairs a thread takes first (all of a row of up to 16 heads of q and k) are read, and
// v is moved, before the angles are computed: the operator on 256 queries at 1792, 14 + 2 heads, went
// from 17.24 to 16.81 us over an f16 cache and from 35.41 to 34.97 over an f32 one.
template <class CT>
__global__ __launch_bounds__(256) void rope_append_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, float* __restrict__ q_rope,
                                                          CT* __restrict__ k_cache, CT* __restrict__ v_cache,
                                                          eg_attention_prefill_dims d) {
  constexpr uint32_t kThreads = 256, kAhead = 2;
  const uint32_t i = blockIdx.x;  // query row of the chunk
  const uint32_t pos = d.query_begin + i;
  const uint32_t tid = threadIdx.x;
  const uint32_t qn = d.heads * (kD / 2), kn = d.kv_heads * (kD / 2), vn = d.kv_heads * kD;
  const float* qr = q + (size_t)i * d.heads * kD;
  const float* kr = k + (size_t)i * d.kv_heads * kD;
  const float* vr = v + (size_t)i * vn;
  const auto pair_at = [&](uint32_t p) {
    const uint32_t pp = p < qn ? p : p - qn;
    const float* src = (p < qn ? qr : kr) + (size_t)(pp / (kD / 2)) * kD + pp % (kD / 2);
    return make_float2(src[0], src[kD / 2]);
  };
  float2 ahead[kAhead];
#pragma unroll
  for (uint32_t j = 0; j < kAhead; j++) {
    const uint32_t p = tid + j * kThreads;
    ahead[j] = p < qn + kn ? pair_at(p) : make_float2(0.f, 0.f);
  }
  CT* vdst = v_cache + (size_t)pos * vn;
  for (uint32_t p = tid; p < vn; p += kThreads) vdst[p] = to_cache<CT>(vr[p]);
  __shared__ double2 cs[kD / 2];
  if (tid < kD / 2) egd::rope_table<kD>(cs, tid, pos, d.theta);
  __syncthreads();
  const float scale = 1.0f / sqrtf((float)kD);  // a power of two: exact
  const auto put = [&](uint32_t p, float2 x) {
    const uint32_t pp = p < qn ? p : p - qn;
    const uint32_t head = pp / (kD / 2), e = pp % (kD / 2);
    const float2 r = egd::rotate(x.x, x.y, cs[e]);
    if (p < qn) {
      float* dst = q_rope + ((size_t)i * d.heads + head) * kD;
      dst[e] = r.x * scale;
      dst[e + kD / 2] = r.y * scale;
    } else {
      CT* dst = k_cache + ((size_t)pos * d.kv_heads + head) * kD;
      dst[e] = to_cache<CT>(r.x);
      dst[e + kD / 2] = to_cache<CT>(r.y);
    }
  };
#pragma unroll
  for (uint32_t j = 0; j < kAhead; j++)
    if (tid + j * kThreads < qn + kn) put(tid + j * kThreads, ahead[j]);
  for (uint32_t p = tid + kAhead * kThreads; p < qn + kn; p += kThreads) put(p, pair_at(p));
}

// Split partials: o [split][query][head][kD] (unnormalised), then m and l [split][query][head].
struct Splits {
  float* o;          // NULL: no split, out written directly
  uint32_t keys;     // keys per split (a multiple of kK)
  uint32_t count;    // splits (grid.z)
  uint32_t first;    // the launch's first query block (see over_blocks)
};

constexpr float kLog2e = 1.44269504088896340736f;

// Max over the 4 lanes that hold a query (lr, lr + 16, lr + 32, lr + 48), in the vector units.
__device__ __forceinline__ float max_of_query(float x) {
  const uint32_t a = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  const uint32_t b = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
  const auto t = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}

// Flash attention in the transposed form: S^T = K Q^T and O^T += V^T P^T, so that each lane holds
// ONE query's scores (the MFMA D layout puts a column in a lane) and P goes from the S^T
// accumulators straight into the B operand of the second product, with no LDS round trip: lane
// group g = lane / 16 holds keys 16 n + 4 g + e of S^T block n, and its 8 k-slots of the half h of
// the second product are those of blocks 2 h and 2 h + 1. The V^T operand is two transposed reads
// of 4 keys each from V as the cache has it.
//
// K and V rows go from memory to LDS directly (16-byte slots, 8 to a row; the next tile's while
// this one is multiplied). Row r's slot j is kept at j ^ ((r / 2) % 8) in K, which spreads the 16
// rows of an operand read over all banks, and at j ^ 2 ((r / 2) % 4) in V, which spreads the 4 rows
// a lane group's transposed read touches, and those of two groups: no conflicts. (Rows through
// registers, V transposed on the way into LDS: 62% of the LDS cycles were conflicts, and LDS was the
// busiest unit.) Bound by the softmax's vector instructions and, with few workgroups, their latency;
// 32 queries per wave, half the LDS reads, was slower at every size (2048 queries: 28 us for 25).
// MI355X, 14 heads, this kernel alone: 2048 queries 38.8 -> 24.3 us, 256 at 1792 13.0 -> 10.8.
constexpr uint32_t kTileBytes = kK * kD * 2;

// (5 waves per SIMD, what LDS holds.)
__global__ __launch_bounds__(256, 5) void attention_kernel(const float* __restrict__ q_rope,
                                                           const uint16_t* __restrict__ k_cache,
                                                           const uint16_t* __restrict__ v_cache,
                                                           float* __restrict__ out, eg_attention_prefill_dims d,
                                                           Splits sp, uint32_t out_bf16) {
  // [buffer][K or V][key][d]. (One array: between two the compiler has a read of K wait for the loads
  // into the other buffer.)
  __shared__ __attribute__((aligned(16))) uint8_t tiles[4 * kTileBytes];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lr = lane & 15u, lg = lane >> 4;  // MFMA lane coordinates
  const uint32_t h = blockIdx.x, kv = h / (d.heads / d.kv_heads);
  // the last query blocks (the longest causal walks) first, so they do not start last; heads vary
  // fastest, which deals every length of walk to each XCD
  const uint32_t q0 = (sp.first + gridDim.y - 1 - blockIdx.y) * kQ;
  const uint32_t query = q0 + wave * 16 + lr;  // this lane's query (its column of S^T and O^T)

  // Q^T fragments (B operand of S^T = K Q^T): query lr, d 32 ks + 8 lg .. +8.
  half8 qb[2];
  {
    const bool in = query < d.queries;
    const float4* src = reinterpret_cast<const float4*>(q_rope + ((size_t)(in ? query : 0) * d.heads + h) * kD + 8 * lg);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const float4 a = in ? src[8 * ks] : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 b = in ? src[8 * ks + 1] : make_float4(0.f, 0.f, 0.f, 0.f);
      qb[ks] = half8{(_Float16)a.x, (_Float16)a.y, (_Float16)a.z, (_Float16)a.w,
                     (_Float16)b.x, (_Float16)b.y, (_Float16)b.z, (_Float16)b.w};
    }
  }

  // O^T blocks (d 16 n .. +16) in the D layout: lane holds d 16 n + 4 lg + e of its query.
  f32x4 o[4];
#pragma unroll
  for (int n = 0; n < 4; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kMasked;  // the query's running max (the same in the 4 lanes holding it)
  float l = 0.f;      // this lane's share of the running sum (its 16 keys of each tile)

  const uint32_t last_query = min(q0 + (uint32_t)kQ, d.queries) - 1;
  uint32_t key_end = d.query_begin + last_query + 1;  // the keys any row of this group sees
  uint32_t key_begin = 0;
  if (sp.o) {  // this split's keys
    key_begin = blockIdx.z * sp.keys;
    key_end = min(key_end, key_begin + sp.keys);
  }
  const uint32_t ntiles = key_end > key_begin ? (key_end - key_begin + kK - 1) / kK : 0;
  const uint32_t limit = d.query_begin + query;  // the last key this query sees
  // a tile wholly at or below the wave's first query's limit (and inside the keys) needs no mask
  const uint32_t open_end = min(d.query_begin + q0 + wave * 16 + 1, key_end);

  // The caches are read through buffer resources that end at the workgroup's last key: rows past it
  // are zeros (a V row there must be finite - its weight is 0).
  const uint32_t pitch = d.kv_heads * kD * 2u;
  const auto kr = egd::buffer(k_cache, key_end * pitch), vr = egd::buffer(v_cache, key_end * pitch);
  const uint32_t trow = wave * 8 + (lane >> 3), slot = lane & 7u;  // this lane's row (and + 32) and LDS slot
  const uint32_t koff = trow * pitch + kv * kD * 2u + 16u * (slot ^ ((trow >> 1) & 7u));
  const uint32_t voff = trow * pitch + kv * kD * 2u + 16u * (slot ^ (trow & 6u));
  auto load_tile = [&](uint32_t j0, uint32_t buf) {
#pragma unroll
    for (uint32_t i = 0; i < 2; i++) {
      uint8_t* at = tiles + 2 * kTileBytes * buf + (4 * i + wave) * 1024u;
      egd::load_to_lds(kr, at, (j0 + 32 * i) * pitch + koff);
      egd::load_to_lds(vr, at + kTileBytes, (j0 + 32 * i) * pitch + voff);
    }
  };
  auto settle = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0: the memory-to-LDS loads have landed
    __syncthreads();
  };
  // LDS offsets of this lane's operand reads: K row lr, slots lg and lg + 4; V row 4 lg + lr / 4, d 4 (lr % 4).
  const uint32_t ksw = (lr >> 1) & 7u, vrow = 4 * lg + (lr >> 2);
  const uint32_t kat[2] = {lr * 128u + 16u * (lg ^ ksw), lr * 128u + 16u * ((lg + 4u) ^ ksw)};
  uint32_t vat[4];
#pragma unroll
  for (uint32_t n = 0; n < 4; n++)
    vat[n] = kTileBytes + vrow * 128u + 8u * (lr & 1u) + 16u * ((2 * n + ((lr >> 1) & 1u)) ^ (vrow & 6u));

  if (ntiles) load_tile(key_begin, 0);
  settle();
  for (uint32_t t = 0; t < ntiles; t++) {
    const uint32_t j0 = key_begin + t * kK, buf = t & 1u;
    const uint8_t* tile = tiles + 2 * kTileBytes * buf;
    // (the other buffer was last read before the barrier that ended the previous tile)
    if (t + 1 < ntiles) load_tile(j0 + kK, buf ^ 1u);

    f32x4 s[4];
#pragma unroll
    for (int n = 0; n < 4; n++) {
      s[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const half8 ka = *reinterpret_cast<const half8*>(tile + 2048u * n + kat[ks]);
        s[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qb[ks], s[n], 0, 0, 0);
      }
    }

    // Causal mask (tiles that cross a limit or the last key) and the online softmax: the lane's
    // 16 scores, then the max over the 4 lanes holding the query.
    if (j0 + kK > open_end) {
#pragma unroll
      for (int n = 0; n < 4; n++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t j = j0 + 16 * n + 4 * lg + e;
          if (!(j <= limit && j < key_end)) s[n][e] = kMasked;
        }
    }
    float mx = kMasked;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) mx = fmaxf(mx, s[n][e]);
    const float mnew = fmaxf(m, max_of_query(mx));
    const float alpha = __builtin_amdgcn_exp2f((m - mnew) * kLog2e);
    // a query with no visible key yet (a split wholly past its causal limit) keeps nothing: its
    // exponent offset is pushed past f32's range below zero
    const float ml = mnew == kMasked ? 3.0e38f : mnew * kLog2e;
    half8 pb[2];
    float sum = 0.f;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[n][e], kLog2e, -ml));
        sum += p;
        pb[n >> 1][4 * (n & 1) + e] = (_Float16)p;
      }
    l = l * alpha + sum;
    // the accumulators are rescaled only when some query of the wave found a larger max
    if (__builtin_amdgcn_ballot_w64(mnew > m) != 0) {
#pragma unroll
      for (int n = 0; n < 4; n++) o[n] *= alpha;
    }
    m = mnew;

    // O^T += V^T P^T over the two halves of the tile.
#pragma unroll
    for (int hh = 0; hh < 2; hh++)
#pragma unroll
      for (int n = 0; n < 4; n++) {
        const uint8_t* at = tile + vat[n] + 4096u * hh;
        const egd::s16x4 lo = egd::lds_read_transposed(at), hi = egd::lds_read_transposed(at + 2048u);
        const half8 va = __builtin_bit_cast(half8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pb[hh], o[n], 0, 0, 0);
      }
    settle();
  }

  // the query's sum over its 4 lanes
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (query >= d.queries) return;
  if (sp.o) {
    const size_t row = ((size_t)blockIdx.z * d.queries + query) * d.heads + h;
#pragma unroll
    for (int n = 0; n < 4; n++)
      *reinterpret_cast<float4*>(&sp.o[row * kD + 16 * n + 4 * lg]) = make_float4(o[n][0], o[n][1], o[n][2], o[n][3]);
    if (lg == 0) {
      float* mlp = sp.o + (size_t)sp.count * d.queries * d.heads * kD;
      mlp[row] = m;
      mlp[(size_t)sp.count * d.queries * d.heads + row] = l;
    }
    return;
  }
  const float inv = 1.0f / l;
  const size_t at = ((size_t)query * d.heads + h) * kD + 4 * lg;
#pragma unroll
  for (int n = 0; n < 4; n++) {
    const float4 v = make_float4(o[n][0] * inv, o[n][1] * inv, o[n][2] * inv, o[n][3] * inv);
    if (out_bf16) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + at + 16 * n) =
        make_uint2(egd::pack_bf16(v.x, v.y), egd::pack_bf16(v.z, v.w));
    else *reinterpret_cast<float4*>(out + at + 16 * n) = v;
  }
}

// ---- the f32 cache --------------------------------------------------------------------------
//
// The attention over f32 rows on the f32 matrix cores (v_mfma_f32_16x16x4_f32: f32 operands, products
// and sums), in attention_kernel's transposed form: S^T = K Q^T, O^T += V^T P^T, 16 queries per wave, 64
// per workgroup, key tiles of 64, the same online softmax and key splits. The operand layouts hold one
// k value per lane and step, and k is taken in the order that keeps every LDS read 16 bytes wide:
//   S^T block n (keys 16 n + lr): lane group g owns d = 16 g .. +16, four reads per key;
//   O^T: step (n, e) multiplies key 16 n + 4 g + e, which is where the S^T accumulators hold it, so P goes
//   from them straight into the operand; block nd's row lr is d = 4 lr + nd, one read per key for all four
//   blocks, and a lane's o[0..3][e] are the four consecutive d = 16 g + 4 e .. +4.
// K and V rows go from memory to LDS directly, the next tile's while this one is multiplied; K's 16-byte
// slots are swizzled by the row. Sums stay short for their error's sake: a score is two chains of 32 products,
// a tile's values are summed by themselves before they are added. A wave and tile take 128
// MFMAs of 32 cycles: 46% of the SIMDs' cycles (256 queries at 1792, 14 / 2 heads: two workgroups on three
// quarters of the CUs), vector instructions 24%, LDS conflicts (K's operand) 3%. Against a workgroup per query
// row with f32 FMAs the same call went from 208.8 to 35.1 us on MI355X (RoPE, append and combine included).
constexpr uint32_t kF32Group = 8;  // query heads per kv head that eg_attention_prefill_f32 takes (a limit of the
                                   // entry point, not of this kernel)
constexpr uint32_t kF32Tile = kK * kD * 4;  // bytes of a K (or V) tile

// SHORT: a tile that holds no more than 16 keys takes the products of those alone, for chunks that end
// within two tiles, whose time is one workgroup's (1 query at the start of the context, 8 heads: 9.7 -> 8.4 us;
// in the long walks the test and the second form cost 2%).
template <bool SHORT>
__global__ __launch_bounds__(256, 2) void attention_f32_kernel(const float* __restrict__ q_rope,
                                                            const float* __restrict__ k_cache,
                                                            const float* __restrict__ v_cache, float* __restrict__ out,
                                                            eg_attention_prefill_dims d, Splits sp) {
  __shared__ __attribute__((aligned(16))) uint8_t tiles[4 * kF32Tile];  // [buffer][K or V][key][d]
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lr = lane & 15u, lg = lane >> 4;
  const uint32_t h = blockIdx.x, kv = h / (d.heads / d.kv_heads);
  const uint32_t q0 = (sp.first + gridDim.y - 1 - blockIdx.y) * kQ;  // the longest causal walks first
  const uint32_t query = q0 + wave * 16 + lr;

  float qb[16];
  {
    const bool in = query < d.queries;
    const float4* src = reinterpret_cast<const float4*>(q_rope + ((size_t)(in ? query : 0) * d.heads + h) * kD + 16 * lg);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float4 v = in ? src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
      qb[4 * j] = v.x;
      qb[4 * j + 1] = v.y;
      qb[4 * j + 2] = v.z;
      qb[4 * j + 3] = v.w;
    }
  }
  f32x4 o[4];
#pragma unroll
  for (int n = 0; n < 4; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  const uint32_t last_query = min(q0 + (uint32_t)kQ, d.queries) - 1;
  uint32_t key_end = d.query_begin + last_query + 1, key_begin = 0;
  if (sp.o) {
    key_begin = blockIdx.z * sp.keys;
    key_end = min(key_end, key_begin + sp.keys);
  }
  const uint32_t ntiles = key_end > key_begin ? (key_end - key_begin + kK - 1) / kK : 0;
  const uint32_t limit = d.query_begin + query;
  const uint32_t open_end = min(d.query_begin + q0 + wave * 16 + 1, key_end);

  // A tile's rows, 4 per load of 1 KiB: row r's 16-byte slot j of K at LDS slot j ^ (r % 16), of V at j.
  // Rows past the last key repeat it (its scores are masked).
  const size_t pitch = (size_t)d.kv_heads * kD;
  auto load_tile = [&](uint32_t j0, uint32_t buf) {
    const auto kr = egd::buffer(k_cache + (size_t)j0 * pitch, min(key_end - j0, (uint32_t)kK) * d.kv_heads * (kD * 4u));
    const auto vr = egd::buffer(v_cache + (size_t)j0 * pitch, min(key_end - j0, (uint32_t)kK) * d.kv_heads * (kD * 4u));
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
      const uint32_t r = (4 * i + wave) * 4 + lg, row = min(r, key_end - j0 - 1);
      const uint32_t at = (row * d.kv_heads + kv) * (kD * 4u);
      uint8_t* to = tiles + 2 * kF32Tile * buf + (4 * i + wave) * 1024u;
      egd::load_to_lds(kr, to, at + 16u * (lr ^ (r & 15u)));
      egd::load_to_lds(vr, to + kF32Tile, at + 16u * lr);
    }
  };
  auto settle = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0: the memory-to-LDS loads have landed
    __syncthreads();
  };
  if (ntiles) load_tile(key_begin, 0);
  settle();
  for (uint32_t t = 0; t < ntiles; t++) {
    const uint32_t j0 = key_begin + t * kK, buf = t & 1u;
    const uint8_t *Ks = tiles + 2 * kF32Tile * buf, *Vs = Ks + kF32Tile;
    // (the other buffer was last read before the barrier that ended the previous tile)
    if (t + 1 < ntiles) load_tile(j0 + kK, buf ^ 1u);

    const bool few = SHORT && key_end - j0 <= 16u;
    f32x4 s[4], s1[4];
#pragma unroll
    for (int n = 0; n < 4; n++) s[n] = s1[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto scores = [&](auto blocks) {
      constexpr uint32_t N = decltype(blocks)::value;
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        f32x4 ka[N];
#pragma unroll
        for (uint32_t n = 0; n < N; n++)
          ka[n] = *reinterpret_cast<const f32x4*>(Ks + (16 * n + lr) * (kD * 4u) + 16u * ((4 * lg + j) ^ lr));
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
          for (uint32_t n = 0; n < N; n++) {
            f32x4& half = j < 2 ? s[n] : s1[n];
            half = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[n][c], qb[4 * j + c], half, 0, 0, 0);
          }
      }
    };
    if (few) scores(std::integral_constant<uint32_t, 1>());
    else scores(std::integral_constant<uint32_t, 4>());
#pragma unroll
    for (int n = 0; n < 4; n++) s[n] += s1[n];

    const bool masked = j0 + kK > open_end;
    if (masked) {
#pragma unroll
      for (int n = 0; n < 4; n++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t j = j0 + 16 * n + 4 * lg + e;
          if (!(j <= limit && j < key_end)) s[n][e] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) mx = fmaxf(mx, s[n][e]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mnew = fmaxf(m, mx);
    // (no visible key yet: nothing is kept, and no infinity is taken from another)
    const float base = mnew == -INFINITY ? 0.f : mnew;
    const float alpha = mnew == -INFINITY ? 1.f : expf(m - base);
    float sum = 0.f;
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float p = expf(s[n][e] - base);
        s[n][e] = p;
        sum += p;
      }
    l = fmaf(l, alpha, sum);
    m = mnew;

    // In a masked tile a key's weight of 0 must drop its value even where that is infinite or NaN (a
    // later row of the chunk): if any is, the tile's values are added one visible key at a time.
    f32x4 ot[4];
#pragma unroll
    for (int n = 0; n < 4; n++) ot[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    bool plain = true;
    if (masked) {
      bool finite = true;
#pragma unroll
      for (uint32_t n = 0; n < 16; n++) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(Vs + (4 * n + lg) * (kD * 4u) + 16u * lr);
#pragma unroll
        for (int c = 0; c < 4; c++) finite = finite && isfinite(v[c]);
      }
      plain = __builtin_amdgcn_ballot_w64(!finite) == 0;
    }
    auto values = [&](auto blocks) {
#pragma unroll
      for (uint32_t n = 0; n < decltype(blocks)::value; n++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const f32x4 va = *reinterpret_cast<const f32x4*>(Vs + (16 * n + 4 * lg + e) * (kD * 4u) + 16u * lr);
#pragma unroll
          for (int nd = 0; nd < 4; nd++) ot[nd] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[nd], s[n][e], ot[nd], 0, 0, 0);
        }
    };
    if (plain && few) {
      values(std::integral_constant<uint32_t, 1>());
    } else if (plain) {
      values(std::integral_constant<uint32_t, 4>());
    } else {
#pragma unroll
      for (uint32_t n = 0; n < 4; n++)
#pragma unroll
        for (uint32_t e = 0; e < 4; e++)
          for (uint32_t g = 0; g < 4; g++) {
            const uint32_t key = 16 * n + 4 * g + e;
            const float p = __shfl(s[n][e], lr + 16 * g, 64);
            if (j0 + key > limit || j0 + key >= key_end) continue;
#pragma unroll
            for (uint32_t c = 0; c < 4; c++) {
              const f32x4 v = *reinterpret_cast<const f32x4*>(Vs + key * (kD * 4u) + 16u * (4 * lg + c));
#pragma unroll
              for (int nd = 0; nd < 4; nd++) ot[nd][c] = fmaf(p, v[nd], ot[nd][c]);
            }
          }
    }
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
      for (int e = 0; e < 4; e++) o[n][e] = fmaf(o[n][e], alpha, ot[n][e]);
    settle();
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (query >= d.queries) return;
  if (sp.o) {
    const size_t row = ((size_t)blockIdx.z * d.queries + query) * d.heads + h;
#pragma unroll
    for (int e = 0; e < 4; e++)
      *reinterpret_cast<float4*>(&sp.o[row * kD + 16 * lg + 4 * e]) = make_float4(o[0][e], o[1][e], o[2][e], o[3][e]);
    if (lg == 0) {
      float* mlp = sp.o + (size_t)sp.count * d.queries * d.heads * kD;
      mlp[row] = m;
      mlp[(size_t)sp.count * d.queries * d.heads + row] = l;
    }
    return;
  }
  float* dst = out + ((size_t)query * d.heads + h) * kD + 16 * lg;
#pragma unroll
  for (int e = 0; e < 4; e++)
    *reinterpret_cast<f32x4u*>(dst + 4 * e) = f32x4u{o[0][e] / l, o[1][e] / l, o[2][e] / l, o[3][e] / l};
}

// The splits merged: out = sum_z o_z e^(m_z - M) / sum_z l_z e^(m_z - M), M = max_z m_z, splits
// in order (an empty split has l = 0 and is left out). One thread per 4 elements of a
// row. A row's splits past its causal limit are empty (z > zmax: the split's first key is past the
// row's last) and are not read. Up to kFastSplits splits, the statistics and values of the
// others are loaded at once (no chain of dependent round trips); more splits take the loop. Both
// add in split order: the same result.
constexpr uint32_t kFastSplits = 8;

__device__ __forceinline__ float4 merged(const float* __restrict__ part, const float* m, const float* l, size_t total,
                                         uint32_t rows, size_t row, size_t idx, uint32_t splits, uint32_t zmax) {
  float M = -INFINITY, L = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (splits <= kFastSplits) {
    float mz[kFastSplits], lz[kFastSplits];
    float4 vz[kFastSplits];
#pragma unroll
    for (uint32_t z = 0; z < kFastSplits; z++) {
      if (z <= zmax) {
        mz[z] = m[(size_t)z * rows + row];
        lz[z] = l[(size_t)z * rows + row];
        vz[z] = reinterpret_cast<const float4*>(part + (size_t)z * total)[idx];
      }
    }
#pragma unroll
    for (uint32_t z = 0; z < kFastSplits; z++)
      if (z <= zmax) M = fmaxf(M, mz[z]);
#pragma unroll
    for (uint32_t z = 0; z < kFastSplits; z++) {
      if (z <= zmax && lz[z] != 0.f) {  // (a NaN sum stays in)
        const float w = expf(mz[z] - M);
        L = fmaf(lz[z], w, L);
        acc.x = fmaf(vz[z].x, w, acc.x);
        acc.y = fmaf(vz[z].y, w, acc.y);
        acc.z = fmaf(vz[z].z, w, acc.z);
        acc.w = fmaf(vz[z].w, w, acc.w);
      }
    }
  } else {
    for (uint32_t z = 0; z <= zmax; z++) M = fmaxf(M, m[(size_t)z * rows + row]);
    for (uint32_t z = 0; z <= zmax; z++) {
      const float lzz = l[(size_t)z * rows + row];
      if (lzz == 0.f) continue;
      const float w = expf(m[(size_t)z * rows + row] - M);
      L = fmaf(lzz, w, L);
      const float4 v = reinterpret_cast<const float4*>(part + (size_t)z * total)[idx];
      acc.x = fmaf(v.x, w, acc.x);
      acc.y = fmaf(v.y, w, acc.y);
      acc.z = fmaf(v.z, w, acc.z);
      acc.w = fmaf(v.w, w, acc.w);
    }
  }
  return make_float4(acc.x / L, acc.y / L, acc.z / L, acc.w / L);
}

__global__ __launch_bounds__(256) void combine_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                      uint32_t rows, uint32_t splits, uint32_t out_bf16, uint32_t heads,
                                                      uint32_t query_begin, uint32_t split_keys) {
  const size_t total = (size_t)rows * kD;
  const float* m = part + (size_t)splits * total;
  const float* l = m + (size_t)splits * rows;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total / 4; idx += (size_t)gridDim.x * blockDim.x) {
    const size_t row = idx / (kD / 4);
    const uint32_t zmax = min(splits - 1, (query_begin + (uint32_t)(row / heads)) / split_keys);
    const float4 v = merged(part, m, l, total, rows, row, idx, splits, zmax);
    if (out_bf16) reinterpret_cast<uint2*>(out)[idx] = make_uint2(egd::pack_bf16(v.x, v.y), egd::pack_bf16(v.z, v.w));
    else *reinterpret_cast<f32x4u*>(out + 4 * idx) = f32x4u{v.x, v.y, v.z, v.w};
  }
}

}  // namespace

// The dims checks of eg_attention_prefill (pointers aside).
int eg::check_attention_prefill(eg_context* ctx, const char* op, const eg_attention_prefill_dims* dims) {
  const eg_attention_prefill_dims& d = *dims;
  if (d.head_dim != (uint32_t)kD)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: head_dim %u is not supported (64)", op, d.head_dim);
  if (d.kv_heads == 0 || d.heads == 0 || d.heads % d.kv_heads != 0)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: heads %u are not a multiple of kv_heads %u", op, d.heads, d.kv_heads);
  if (d.queries == 0) return EG_OK;
  if (d.keys != d.query_begin + d.queries)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: keys %u != query_begin %u + queries %u", op, d.keys, d.query_begin,
                    d.queries);
  if ((uint64_t)d.query_begin + d.queries > d.max_context)
    return eg::fail(ctx, EG_ERR_RANGE, "%s: positions up to %llu exceed the cache's %u", op,
                    (unsigned long long)d.query_begin + d.queries, d.max_context);
  if ((uint64_t)d.max_context * d.kv_heads * d.head_dim * 2 >= (1ull << 31))
    return eg::fail(ctx, EG_ERR_RANGE, "%s: a cache of %u positions x %u kv heads exceeds 2 GiB", op, d.max_context,
                    d.kv_heads);
  if (d.heads > 65535)
    return eg::fail(ctx, EG_ERR_RANGE, "%s: %u heads over the grid limit", op, d.heads);
  return EG_OK;
}

namespace {

// Keys split over a long key range, within the workspace: where the (query block, head) grid
// leaves most CUs idle, into splits of at least 4 key tiles, about per_cu workgroups per CU in all
// (2 over an f32 cache, whose time is the longest CU's MFMAs: 256 queries at 1792 take 4 us
// more at 1; f16 rows, bound by latency, take 19.3 us at 1 and 19.8 at 2);
// and so that no workgroup walks more than 8 tiles - the causal limit makes the last query
// blocks of a long chunk the longest, and with the split their keys spread over more
// workgroups while the early blocks' later splits are empty.
Splits splits_for(eg_context* ctx, const eg_attention_prefill_dims& d, uint32_t per_cu = 1) {
  const uint32_t blocks = (d.queries + kQ - 1) / kQ;
  const uint64_t grid = (uint64_t)blocks * d.heads;
  const uint32_t tiles = (d.keys + kK - 1) / kK;
  const uint32_t cap = ctx->attention_split_tiles;
  const uint64_t target = (uint64_t)ctx->cu_count * ctx->attention_split_fill * per_cu;
  uint32_t splits = 1;
  if (tiles >= 8) {
    if (grid < target) splits = (uint32_t)std::min<uint64_t>((target + grid - 1) / grid, tiles / 4);
    splits = std::max(splits, (tiles + cap - 1) / cap);
  }
  const uint64_t rows = (uint64_t)d.queries * d.heads;
  while (splits > 1 && (uint64_t)splits * rows * (kD + 2) * 4 > eg::kPartialsBytes) splits--;
  Splits sp{nullptr, 0, 1, 0};
  if (splits > 1) {
    sp.keys = ((tiles + splits - 1) / splits) * kK;
    sp.count = (d.keys + sp.keys - 1) / sp.keys;
    sp.o = reinterpret_cast<float*>(eg::partials(ctx));
  }
  return sp;
}

// Runs launch(grid, sp) over a chunk's query blocks: one launch, as a grid's y takes 65535, or several, the
// longest walks first.
template <class F>
void over_blocks(const eg_attention_prefill_dims& d, Splits sp, F launch) {
  constexpr uint32_t kMost = 65535;
  const uint32_t blocks = (d.queries - 1) / kQ + 1;
  for (uint32_t end = blocks; end > 0; end = sp.first) {
    sp.first = end > kMost ? end - kMost : 0;
    launch(dim3(d.heads, end - sp.first, sp.count), sp);
  }
}

}  // namespace

int eg::attention_prefill_run(eg_context* ctx, const float* q_rope, const uint16_t* k_cache, const uint16_t* v_cache,
                              float* out, const eg_attention_prefill_dims& d, bool out_bf16) {
  const char* op = "attention_prefill";
  if ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15u)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: the caches must be 16-byte aligned", op);
  if ((reinterpret_cast<uintptr_t>(q_rope) | reinterpret_cast<uintptr_t>(out)) & 15u)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: q_rope and out must be 16-byte aligned", op);
  if (d.queries == 0) return EG_OK;
  const uint64_t rows = (uint64_t)d.queries * d.heads;
  const Splits sp = splits_for(ctx, d);
  over_blocks(d, sp, [&](dim3 grid, const Splits& part) {
    hipLaunchKernelGGL(attention_kernel, grid, dim3(256), 0, ctx->stream, q_rope, k_cache, v_cache, out, d, part,
                       out_bf16 ? 1u : 0u);
  });
  if (sp.o) {
    const uint64_t total = rows * kD;
    const uint32_t cblocks = (uint32_t)std::min<uint64_t>((total / 4 + 255) / 256, (uint64_t)ctx->cu_count * 8);
    hipLaunchKernelGGL(combine_kernel, dim3(cblocks), dim3(256), 0, ctx->stream, sp.o, out, (uint32_t)rows, sp.count,
                       out_bf16 ? 1u : 0u, d.heads, d.query_begin, sp.keys);
  }
  return eg::check_launch(ctx, op);
}

extern "C" int eg_attention_prefill(eg_context* ctx, const float* q, const float* k, const float* v, uint16_t* k_cache,
                                    uint16_t* v_cache, float* q_rope, float* out,
                                    const eg_attention_prefill_dims* dims) {
  const char* op = "attention_prefill";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (!dims || !q || !k || !v || !k_cache || !v_cache || !q_rope || !out)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: NULL argument", op);
  int st = eg::check_attention_prefill(ctx, op, dims);
  if (st != EG_OK || dims->queries == 0) return st;
  if ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15u)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: the caches must be 16-byte aligned", op);
  if ((reinterpret_cast<uintptr_t>(q_rope) | reinterpret_cast<uintptr_t>(out)) & 15u)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: q_rope and out must be 16-byte aligned", op);
  const eg_attention_prefill_dims& d = *dims;
  hipLaunchKernelGGL(rope_append_kernel<uint16_t>, dim3(d.queries), dim3(256), 0, ctx->stream, q, k, v, q_rope,
                     k_cache, v_cache, d);
  return eg::attention_prefill_run(ctx, q_rope, k_cache, v_cache, out, d);
}

extern "C" int eg_attention_prefill_f32(eg_context* ctx, const float* q, const float* k, const float* v, float* k_cache,
                                        float* v_cache, float* q_rope, float* out,
                                        const eg_attention_prefill_dims* dims) {
  const char* op = "attention_prefill_f32";
  if (!ctx) return eg::fail(nullptr, EG_ERR_INVALID, "%s: ctx is NULL", op);
  if (!dims || !q || !k || !v || !k_cache || !v_cache || !q_rope || !out)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: NULL argument", op);
  int st = eg::check_attention_prefill(ctx, op, dims);
  if (st != EG_OK || dims->queries == 0) return st;
  const eg_attention_prefill_dims& d = *dims;
  if (d.heads / d.kv_heads > kF32Group)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: %u query heads per kv head (at most %u)", op, d.heads / d.kv_heads,
                    kF32Group);
  if ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
       reinterpret_cast<uintptr_t>(q_rope)) & 15u)
    return eg::fail(ctx, EG_ERR_INVALID, "%s: the caches and q_rope must be 16-byte aligned", op);
  hipLaunchKernelGGL(rope_append_kernel<float>, dim3(d.queries), dim3(256), 0, ctx->stream, q, k, v, q_rope, k_cache,
                     v_cache, d);
  const uint64_t rows = (uint64_t)d.queries * d.heads;
  const Splits sp = splits_for(ctx, d, 2);
  const auto kernel = d.keys <= 2u * kK ? attention_f32_kernel<true> : attention_f32_kernel<false>;
  over_blocks(d, sp, [&](dim3 grid, const Splits& part) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, ctx->stream, q_rope, k_cache, v_cache, out, d, part);
  });
  if (sp.o) {
    const uint32_t cblocks = (uint32_t)std::min<uint64_t>((rows * kD / 4 + 255) / 256, (uint64_t)ctx->cu_count * 8);
    hipLaunchKernelGGL(combine_kernel, dim3(cblocks), dim3(256), 0, ctx->stream, sp.o, out, (uint32_t)rows, sp.count, 0u,
                       d.heads, d.query_begin, sp.keys);
  }
  return eg::check_launch(ctx, op);
}
