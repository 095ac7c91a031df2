// Sparse attention over selected positions of the quantized pools, fused: the selected positions of each query row
// are resolved (position -> slot through req_to_token -> tier through the owner table), dequantized exactly as the
// reference's compact gather does (bf16(q * s * sm), patches/kv_tiers.py:446-538) and attended in one pass, with no
// bf16 scratch.  Two entry points share the kernel:
//   * kvt_sparse_decode (one query row per request): the reference's decode gathers the top-k positions into that
//     scratch and runs FlashAttention-2 over it (sglang/qwen4exp-serving-73a255206f.patch:1832-1882).  A block takes
//     64 selected columns of one (request, KV head) and writes an unnormalized partial; kvt_decode_combine merges
//     the column splits as it merges the dense decode's.
//   * kvt_sparse_prefill (one query row per chunk query): the reference's paged prefix-chunk attention
//     sparse_gqa_fwd_interface_paged (patches/kv_paged_prefix.py:141-365).  A block takes every selected column of
//     one (query, KV head): query j of a chunk of q_len queries over a context of kv_len attends the valid entries
//     (0 <= idx < kv_len) among the first min(topk, j + kv_len - q_len + 1) of its index row
//     (patches/kv_paged_prefix.py:199-229) and writes its normalized output (0/0 = NaN when nothing is attended).
//
// Inside a block, 4 wavefronts take 16-column tiles in turn.  Blocks with many columns (prefill rows, decode blocks
// of several tiles per wavefront) first resolve all of them into an LDS column table partitioned by tier, so every
// tile holds rows of one tier and padding columns cost nothing; a block of one tile per wavefront resolves its own
// tile.  A tile's K and V rows are dequantized into the wavefront's LDS rows as bf16, then QK^T and P.V run as bf16
// 16x16x32 matrix-core steps with fp32 accumulation:
//   S^T[row][head] = K[row][:] . Q[head][:]   (A = K tile, B = Q^T in registers; 8 steps over the 256 channels)
//   O[head][ch]   += P[head][row] V[row][ch]  (A = P straight from S^T's accumulator layout: bf16 high parts in one
//                                               half of the 32 k indices, bf16 remainders in the other; B = the 16 V
//                                               rows in both halves, by the transposing LDS read)
// with an online softmax across a wavefront's tiles.  The 16 accumulator rows hold up to 16 q heads per KV head
// (GQA 8 of the configurations, 12 of the served model).  The 4 wavefronts merge through LDS, 8 heads per pass.
// In decode, columns c of request b attend when c < the request's valid count (cu_k[b + 1] - cu_k[b]) and
// 0 <= indices[b][c] < seq_lens[b] - the columns the reference's gather writes and its attention reads when the
// valid positions come first (the indexer pads with -1 at the end).
//
// What bounds it: instruction issue, most of it the exact dequantization.  Counted per tile and wavefront over the paged
// prefix chunk, resolve and merge included: 546 vector instructions (24 of them products; 692 with smoothing products),
// 51 LDS accesses, 35 vector-memory and 30 scalar instructions, in 5,750 cycles of which 3,030 issue.  Two rows per wavefront instruction (8 channels a lane), no products with
// smoothing factors of 1, 32-deep products (the matrix pipe takes as long for a 16-deep one) and the next tile's loads
// in flight beside a tile's work took the paged prefix chunk (60,000 + 1,024 positions, top 2,051, 12 heads) from 237 to
// 169 us, the dense slot decode (4 x 65,536) from 70 to 55 us and the top-k decode (8 x 2,051, 12 layers) from 234 to
// 200 us, against one row per instruction, 16-deep products and loads waited for at the head of each tile.
//
// Kinds (the compact gather's codes): 0 INT8-G pool, 1 INT4-G32 pool, 2 tiered (INT8-G ring over INT4-G32 rows,
// owner test).

#include "kvt_common.h"

using namespace kvt;

namespace {

constexpr int kD = 256;
constexpr int kRows = 16;          // rows per MFMA tile
constexpr int kWaves = 4;          // wavefronts per block, one tile each
constexpr int kCols = kWaves * kRows;  // selected columns per block (one partial)
constexpr int kHeads = 16;         // q heads per KV head the tile holds (rows beyond the group are zero)
constexpr int kKPitch = kD + 8;    // bf16 per K row in LDS (the pad spreads a column of rows over the banks)

typedef short s4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4v lds_v4s;
typedef float f4 __attribute__((ext_vector_type(4)));

struct SparseArgs {
  const void* k;           // tiered / INT4: uint8 [rows, H, D/2]; INT8: int8 [rows, H, D]
  const void* v;
  const uint16_t* ks;      // scales of k / v: fp16 [rows, H, D/32] (INT4) or [rows, H, D/G8] (INT8)
  const uint16_t* vs;
  const int8_t* rk;        // tiered: INT8 ring [R, H, D], scales [R, H, D/G8], owner [R]
  const int8_t* rv;
  const uint16_t* rks;
  const uint16_t* rvs;
  const int32_t* owner;
  int64_t ring_mask;
  const uint16_t* sm_k;    // smoothing factors [H, D] fp16 (may be null: identity)
  const uint16_t* sm_v;
  const int32_t* req_to_token;
  int64_t req_stride;
  const void* req_indices;
  int req64;
  const int32_t* indices;  // [batch, idx_stride], the first topk columns used
  int64_t idx_stride;
  const int32_t* seq_lens;
  const void* cu_k;        // decode: the valid counts' prefix sum; null at the entry point: every column counts (the
  int cu64;                // launcher then points it at seq_lens, whose entry b is read for both bounds and not used)
  int all_columns;
  int topk;
  int H;
  int gs;
  int n_splits;
  int tiles;             // decode: 16-column tiles per wavefront (a block takes kCols x tiles columns)
  uint32_t rows8;        // rows of the INT8 tensors (ring R when tiered, the pool otherwise)
  uint32_t rows4;        // rows of the INT4 pool
  float scale;
  const uint16_t* q;       // bf16 query rows: row r, q head j at q + r sq_n + j sq_h
  int64_t sq_n, sq_h;
  int64_t si_m, si_g, si_n;  // indices of row r, KV head h, column c at indices + r si_m + h si_g + c si_n
  float* part_o;           // decode: [(b H + h) n_splits + split][gs][D]
  float* part_ml;          // decode: [(b H + h) n_splits + split][gs][2]
  int32_t* counters;       // decode, merged in the launch: [b H + h] arrivals (zero between calls); null: partials only
  float* mout_f32;         // decode, merged in the launch: out[b][h gs + j][D] fp32 or bf16, batch stride mout_b
  uint16_t* mout_bf16;
  int64_t mout_b;
  // prefill rows: chunk b holds rows cu_q[b] .. cu_q[b + 1] over a context of kv_lens[b] positions
  const void* cu_q;
  int cuq64;
  const int32_t* kv_lens;
  void* out;               // bf16 or fp32 (out_f32) rows: row r, q head j at out + r so_n + j so_h
  int out_f32;
  int64_t so_n, so_h;
};

// Entry i of an int32 or int64 index array (is64: exactly 0 or 1, as the launchers store it) without a branch on the
// width: both words are loaded unconditionally (an int32 entry reads its own word twice) and combined with integer
// arithmetic only.  Split in two (the loads, then the value) so that a caller can issue several entries' loads
// before it waits for any of them.
struct IdxWords {
  uint32_t lo, hi, wide;
};
KVT_DEV IdxWords idx_words(const void* p, int is64, int64_t i) {
  const uint32_t wide = (uint32_t)is64;
  const int32_t* w = reinterpret_cast<const int32_t*>(p) + (i << wide);
  return IdxWords{(uint32_t)w[0], (uint32_t)w[wide], wide};
}
KVT_DEV int64_t idx_value(const IdxWords& x) {
  const uint32_t mask = 0u - x.wide;   // all ones for int64 entries
  const uint32_t top = (x.hi & mask) | ((uint32_t)((int32_t)x.lo >> 31) & ~mask);
  return (int64_t)(((uint64_t)top << 32) | x.lo);
}

KVT_DEV f4 mfma_bf16(bf8 a, bf8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

KVT_DEV __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Eight channels of one row, dequantized: bf16((c * s) * sm) for code c, the row's fp16 scale s (bits sbits) and the
// channel's smoothing factor sm, as the gathers write them (finite scales; an infinite one gives NaN).  INT8 rows give
// 8 bytes of codes, INT4 rows 4 (byte j = channel 2 j in the low nibble, 2 j + 1 in the high one, stored as c + 8).  A
// code with offset o (c + o >= 0) goes into the mantissa of an fp16 magic value h = 1024 + (c + o) (v_perm_b32 for
// bytes, v_and_or_b32 for nibbles), in pairs of channels (0, 2), (1, 3), (4, 6), (5, 7); v_fma_mix_f32 converts h and s and computes
// h * s - (1024 + o) * s in one rounding, whose exact value c * s is representable (4 or 8 bits times the scale's
// 11), so the fp32 product equals the plain c * s; the caller then multiplies by the smoothing factor in fp32 and
// rounds each pair to nearest even with v_cvt_pk_bf16_f32.
KVT_DEV uint32_t and_or(uint32_t x, uint32_t m, uint32_t o) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(m), "v"(o));
  return r;
}
KVT_DEV float mix(uint32_t w, int half, _Float16 s, float c) {
  typedef _Float16 h2v __attribute__((ext_vector_type(2)));
  return fmaf((float)__builtin_bit_cast(h2v, w)[half], (float)s, c);
}
KVT_DEV void magic8(uint2 w, uint32_t m[4]) {
  const uint32_t u = w.x ^ 0x80808080u, v = w.y ^ 0x80808080u;
  m[0] = __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u);
  m[1] = __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u);
  m[2] = __builtin_amdgcn_perm(0x64646464u, v, 0x04020400u);
  m[3] = __builtin_amdgcn_perm(0x64646464u, v, 0x04030401u);
}
KVT_DEV void magic4(uint32_t w, uint32_t m[4]) {   // pairs (0, 4), (1, 5), (2, 6), (3, 7), one instruction less than magic8's
  m[0] = and_or(w, 0x000F000Fu, 0x64006400u);
  m[1] = and_or(w >> 4, 0x000F000Fu, 0x64006400u);
  m[2] = and_or(w >> 8, 0x000F000Fu, 0x64006400u);
  m[3] = and_or(w >> 12, 0x000F000Fu, 0x64006400u);
}
KVT_DEV void magic4_as8(uint32_t w, uint32_t m[4]) {   // in magic8's pairs
  const uint32_t a = __builtin_amdgcn_perm(0u, w, 0x0c010c00u);   // bytes 0, 1 in the low byte of each half
  const uint32_t b = __builtin_amdgcn_perm(0u, w, 0x0c030c02u);
  m[0] = and_or(a, 0x000F000Fu, 0x64006400u);
  m[1] = and_or(a >> 4, 0x000F000Fu, 0x64006400u);
  m[2] = and_or(b, 0x000F000Fu, 0x64006400u);
  m[3] = and_or(b >> 4, 0x000F000Fu, 0x64006400u);
}

// The 8 channels of magic words m (PAIRS4: magic4's pairs, else magic8's) as bf16; SM: times the smoothing factors (a
// product with 1 changes nothing, so identity factors take the body without it).  offset: 1024 + o (exact products: the
// scale's 11 bits times 1032 or 1152 fit fp32).
template <bool SM, bool PAIRS4>
KVT_DEV uint4 rows_bf16(const uint32_t m[4], uint32_t sbits, float offset, const uint4& sm) {
  const _Float16 s = __builtin_bit_cast(_Float16, (uint16_t)(sbits & 0xffffu));
  const float c = fmaf((float)s, -offset, 0.0f);   // (one v_fma_mix_f32)
  float x[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int lo = PAIRS4 ? j : 4 * (j >> 1) + (j & 1);
    x[lo] = mix(m[j], 0, s, c), x[lo + (PAIRS4 ? 4 : 2)] = mix(m[j], 1, s, c);
  }
  if constexpr (SM) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t w = i < 2 ? sm.x : i < 4 ? sm.y : i < 6 ? sm.z : sm.w;
      x[i] *= f16_bits_to_f32((uint16_t)(w >> (16 * (i & 1))));
    }
  }
  return uint4{bf16x2(x[0], x[1]), bf16x2(x[2], x[3]), bf16x2(x[4], x[5]), bf16x2(x[6], x[7])};
}

// The raw data of a tile: a wavefront takes two rows at once, lanes 0-31 row 2 i and lanes 32-63 row 2 i + 1, each
// lane 8 channels (8 (lane & 31) ..) -- half the loads and LDS stores of one row per wavefront, and no shuffling of
// half-used words.
constexpr int kPairs = kRows / 2;
struct Raw {
  uint2 w8[kPairs];      // INT8 codes
  uint32_t w4[kPairs];   // INT4 codes
  uint32_t s8[kPairs], s4[kPairs];
};

// A row of the pools as one word: row * H + head (below 2^24), bit 30 set for a ring (INT8) row of a mixed tile.
// kNoRow (not attended): every byte offset formed from it lies past the buffers (all below 2^31 bytes) without
// wrapping, so its loads return zeros.
constexpr uint32_t kNoRow = 0xffffffffu;
constexpr uint32_t kHotBit = 1u << 30;

// Buffer resources over whole tensors (byte offsets are 32-bit: the launcher checks the sizes).
struct PoolRsrc {
  __amdgpu_buffer_rsrc_t k8, v8, ks8, vs8, k4, v4, ks4, vs4;
};

// TIERS: the tile's rows are all INT8 (kRowsInt8), all INT4 (kRowsInt4) or each in its own tier (kRowsMixed: both
// tiers' loads are issued, the row's absent tier at an offset past its buffer, and the magic words selected).
enum { kRowsInt8 = 0, kRowsInt4 = 1, kRowsMixed = 2 };

// Issue the loads of K or V of a tile whose row words (of this lane's half: rows 2 i + (lane >> 5)) are e[i].
template <int G8, int TIERS>
KVT_DEV void issue_rows(__amdgpu_buffer_rsrc_t r8, __amdgpu_buffer_rsrc_t rs8, __amdgpu_buffer_rsrc_t r4,
                        __amdgpu_buffer_rsrc_t rs4, const uint32_t e[kPairs], int lane, Raw& R) {
  constexpr uint32_t kSh8 = kD / G8 * 2;   // scale bytes of an INT8 row
  const uint32_t g = (uint32_t)lane & 31u;
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    uint32_t e8 = e[i], e4 = e[i];
    if constexpr (TIERS == kRowsMixed) {
      const bool hot = (e[i] >> 30) == 1u;
      e8 = hot ? e[i] ^ kHotBit : kNoRow;
      e4 = hot ? kNoRow : e[i];
    }
    if constexpr (TIERS != kRowsInt4) {
      R.w8[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r8, (int)(e8 * 256u + 8u * g), 0, 0));
      R.s8[i] = __builtin_amdgcn_raw_buffer_load_b16(rs8, (int)(e8 * kSh8 + 2u * ((8u * g) / G8)), 0, 0);
    }
    if constexpr (TIERS != kRowsInt8) {
      R.w4[i] = __builtin_amdgcn_raw_buffer_load_b32(r4, (int)(e4 * 128u + 4u * g), 0, 0);
      R.s4[i] = __builtin_amdgcn_raw_buffer_load_b16(rs4, (int)(e4 * 16u + 2u * (g >> 2)), 0, 0);
    }
  }
}

// Dequantize the tile into the wavefront's LDS rows (row-major, 16 bytes per lane); sm_row: the head's 256 smoothing
// factors in LDS.
template <int TIERS, bool SM>
KVT_DEV void store_rows(const Raw& R, const uint32_t e[kPairs], uint16_t* kt, int lane, const uint16_t* sm_row) {
  uint4 sm{};
  if constexpr (SM) sm = *reinterpret_cast<const uint4*>(&sm_row[8 * (lane & 31)]);
  uint16_t* dst = &kt[(lane >> 5) * kKPitch + 8 * (lane & 31)];
#pragma unroll
  for (int i = 0; i < kPairs; ++i) {
    uint32_t m[4];
    uint32_t sb;
    float off;
    if constexpr (TIERS == kRowsInt8) {
      magic8(R.w8[i], m);
      sb = R.s8[i], off = 1152.0f;
    } else if constexpr (TIERS == kRowsInt4) {
      magic4(R.w4[i], m);
      sb = R.s4[i], off = 1032.0f;
    } else {
      uint32_t m8[4];
      magic8(R.w8[i], m8);
      magic4_as8(R.w4[i], m);
      const bool hot = (e[i] >> 30) == 1u;
#pragma unroll
      for (int j = 0; j < 4; ++j) m[j] = hot ? m8[j] : m[j];
      sb = hot ? R.s8[i] : R.s4[i];
      off = hot ? 1152.0f : 1032.0f;
    }
    *reinterpret_cast<uint4*>(dst + 2 * i * kKPitch) = rows_bf16<SM, TIERS == kRowsInt4>(m, sb, off, sm);
  }
}

// One resolved 16-column tile of a wavefront, whose raw rows are K and V, folded into its running softmax state (m, l
// per q head n16 of this lane, o): dequantize K into the wavefront's LDS rows, S^T = K Q^T, dequantize V into the same
// rows, online softmax, O += P V.  e: the row words of this lane's half; vm: bit r set when row r is attended
// (wave-uniform).  NEXT: K and V are loaded again, for the tile whose words are en, as soon as their registers are
// free, so that those loads travel beside this tile's work.
template <int G8, int TIERS, bool SM, bool NEXT>
KVT_DEV void attend_tile(const SparseArgs& A, const PoolRsrc& P, const bf8 qop[8], uint16_t* kt,
                         Raw& K, Raw& V, const uint32_t e[kPairs], uint32_t vm, const uint32_t en[kPairs], int lane,
                         const uint16_t* sm, float& m_run, float& l_run, f4 o[16]) {
  const int n16 = lane & 15, kq = lane >> 4;
  // K rows into this wavefront's LDS rows; a wavefront's LDS accesses complete in order, so these stores land after
  // the previous tile's V reads
  store_rows<TIERS, SM>(K, e, kt, lane, sm);
  if constexpr (NEXT) issue_rows<G8, TIERS>(P.k8, P.ks8, P.k4, P.ks4, en, lane, K);
  __builtin_amdgcn_sched_barrier(0);
  // S^T = K Q^T: lane l holds rows 4 (l >> 4) + i of q head l & 15
  f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint4 ka = *reinterpret_cast<const uint4*>(&kt[n16 * kKPitch + 32 * k + 8 * kq]);
    s = mfma_bf16(__builtin_bit_cast(bf8, ka), qop[k], s);
  }
  __builtin_amdgcn_sched_barrier(0);
  // from here to P the tile's chain runs at a raised wave priority: the V rows and the softmax issue ahead of the
  // other wavefronts' work on the SIMD, which keeps the products that wait for them fed (slot-pool decode and the
  // paged prefix-chunk attention ~6 % faster than without)
  __builtin_amdgcn_s_setprio(1);
  // V rows into the same LDS rows (the stores stay behind the K reads above, which may alias them)
  store_rows<TIERS, SM>(V, e, kt, lane, sm + kD);
  if constexpr (NEXT) issue_rows<G8, TIERS>(P.v8, P.vs8, P.v4, P.vs4, en, lane, V);
  // online softmax (log2 units): rows 4 kq + i of this lane's head, the other 12 rows in lanes n16 + 16 j
  constexpr float kLog2e = 1.4426950408889634f;
  const float cs = A.scale * kLog2e;
  float tv[4], mloc = -INFINITY;
  const uint32_t vq = vm >> (4 * kq);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    tv[i] = ((vq >> i) & 1u) != 0 ? s[i] * cs : -INFINITY;
    mloc = fmaxf(mloc, tv[i]);
  }
  const float m_new = fmaxf(m_run, max_xor16_32(mloc));
  const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
  float p[4], lsum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    // (the exponent in one rounding of the difference: the rounded score tv alone is off by up to 2^-24 |tv|)
    const float d = fmaf(s[i], cs, -m_new);
    p[i] = tv[i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(d);
    lsum += p[i];
  }
  l_run = l_run * alpha + sum_xor16_32(lsum);
  m_run = m_new;
  // o[n][i] is head 4 kq + i: its rescale factor lives in lane 4 kq + i; only when some head's max has grown
  if (__any(alpha != 1.0f)) {
    float ai[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ai[i] = __shfl(alpha, 4 * kq + i, 64);
#pragma unroll
    for (int n = 0; n < 16; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[n][i] *= ai[i];
  }
  // P as bf16 high part + bf16 remainder: P keeps ~16 significant bits, against 8 for a plain bf16 cast, so a peaked
  // softmax stays within the fp32 reference's tolerance.  Both go through one 32-deep product: this lane's 8 k indices
  // are the high parts of its 4 rows and their remainders, against the same 4 V rows twice (a 16x16x32 product takes
  // the matrix pipe as long as a 16x16x16 one).
  const uint32_t h01 = bf16x2(p[0], p[1]), h23 = bf16x2(p[2], p[3]);
  const uint32_t l01 = bf16x2(p[0] - __uint_as_float(h01 << 16), p[1] - __uint_as_float(h01 & 0xffff0000u));
  const uint32_t l23 = bf16x2(p[2] - __uint_as_float(h23 << 16), p[3] - __uint_as_float(h23 & 0xffff0000u));
  const bf8 pa = __builtin_bit_cast(bf8, uint4{h01, h23, l01, l23});
  __builtin_amdgcn_s_setprio(0);
  // O = P V.  B = V[rows 4 kq + k][channel 16 n + n16] by the transposing read: in each 16-lane group, lane L's
  // element k comes from element L & 3 of the 8 bytes lane 4 k + (L >> 2) addresses, so lane m addresses
  // V[4 kq + (m >> 2)][16 n + 4 (m & 3)]
  const uint32_t vbase = (uint32_t)(uintptr_t)&kt[(4 * kq + (n16 >> 2)) * kKPitch + 4 * (n16 & 3)];
#pragma unroll
  for (int n = 0; n < 16; ++n) {
    const uint2 v = __builtin_bit_cast(
        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(uintptr_t)(vbase + 32u * (uint32_t)n)));
    o[n] = mfma_bf16(pa, __builtin_bit_cast(bf8, uint4{v.x, v.y, v.x, v.y}), o[n]);
    if ((n & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // (at most 4 V operands held at once)
  }
}

template <int N>
struct Tiers {
  static constexpr int value = N;
};

// The tile of a one-tile decode block through the body for its rows' tiers: single-tier pools know them; in the
// tiered pool a tile whose 16 rows all sit in one tier (most of them: the ring holds a small share of the slots) takes
// that tier's body.  Lane r < 16 holds row r's word.
template <int KIND, int G8, bool SM>
KVT_DEV void attend_tile_any(const SparseArgs& A, const PoolRsrc& P, const bf8 qop[8], uint16_t* kt, uint32_t word,
                             int lane, const uint16_t* sm, float& m_run, float& l_run, f4 o[16]) {
  const uint32_t vm = (uint32_t)__builtin_amdgcn_ballot_w64(word != kNoRow) & 0xffffu;
  uint32_t e[kPairs];
#pragma unroll
  for (int i = 0; i < kPairs; ++i) e[i] = (uint32_t)__shfl((int)word, 2 * i + (lane >> 5), 64);
  auto one = [&](auto tiers) {
    constexpr int T = decltype(tiers)::value;
    Raw K, V;
    issue_rows<G8, T>(P.k8, P.ks8, P.k4, P.ks4, e, lane, K);
    issue_rows<G8, T>(P.v8, P.vs8, P.v4, P.vs4, e, lane, V);
    attend_tile<G8, T, SM, false>(A, P, qop, kt, K, V, e, vm, e, lane, sm, m_run, l_run, o);
  };
  if constexpr (KIND != 2) {
    one(Tiers<KIND == 0 ? kRowsInt8 : kRowsInt4>{});
  } else {
    const uint32_t hot = (uint32_t)__builtin_amdgcn_ballot_w64((word >> 30) == 1u) & 0xffffu;
    if (hot == 0) {
      one(Tiers<kRowsInt4>{});
    } else if (hot == vm) {
#pragma unroll
      for (int i = 0; i < kPairs; ++i) e[i] = e[i] == kNoRow ? kNoRow : e[i] ^ kHotBit;
      one(Tiers<kRowsInt8>{});
    } else {
      one(Tiers<kRowsMixed>{});
    }
  }
}

// Resolve a tile's columns, lane r < 16 column c0 + r, into its row word: position from the index row, slot from
// req_to_token, tier from the owner table (three dependent loads, independent of Q).
template <int KIND>
KVT_DEV uint32_t resolve_tile(const SparseArgs& A, int64_t c0, int64_t c_end, const int32_t* idx_row, int64_t L,
                              int64_t req, int h, int lane) {
  const int64_t col = c0 + (lane & 15);
  uint32_t word = kNoRow;
  if (lane < kRows && col < c_end) {
    const int64_t pos = idx_row[col * A.si_n];
    if (pos >= 0 && pos < L) {
      const int64_t slot = A.req_to_token[req * A.req_stride + pos];
      word = (uint32_t)(slot * A.H + h);
      if constexpr (KIND == 2) {
        const int64_t r = slot & A.ring_mask;
        if ((int64_t)A.owner[r] == slot) word = (uint32_t)(r * A.H + h) | kHotBit;
      }
    }
  }
  return word;
}

// LDS of a block: one tile buffer per wavefront (K rows until S is formed, then V rows), after the
// tiles the same space holds the merge of the 4 wavefronts; and the group's q heads, bf16 (zero beyond gs)
template <int CAP>
struct BlockLds {
  uint16_t kv[kWaves][kRows * kKPitch];
  uint16_t qs[kHeads * kKPitch];
  uint16_t sm[2 * kD];         // smoothing factors (fp16) of K, then V; read when they are not all 1
  uint32_t cols[CAP + 3 * kRows];   // the resolved columns' row words: ring rows first, INT4 rows from entry
                                    // CAP + 2 kRows down, each part padded with kNoRow to whole tiles; then one
                                    // tile of kNoRow
  int counts[2 * kWaves];
  int ones[kWaves];            // wavefront w's smoothing factors are all 1
  int last;                    // decode merged in the launch: this block counted last for its (request, KV head)
};
constexpr int kRowCols = 4096;   // prefill rows: selected columns resolved per pass
constexpr int kMultiCols = 1024; // decode blocks of several tiles per wavefront
// LDS per block, of 160 KB a CU: 3 one-tile blocks, 2 of the others (their registers allow no third)
static_assert(sizeof(BlockLds<1>) == 43512 && sizeof(BlockLds<kMultiCols>) == 47604 && sizeof(BlockLds<kRowCols>) == 59892,
              "LDS per block");

// The selected columns [k0, k1) (at most CAP) of a block's query row, resolved by all its threads
// together into the column table and partitioned by tier: ring (INT8) rows to cols[0 .. nh), INT4 rows from the end
// of the table down, both padded with kNoRow to whole tiles, unattended columns dropped (patches/kv_paged_prefix.py:199-229: position in
// [0, L)).  J columns per thread, so the position, slot and owner loads of many columns are in flight at once; a
// block scan of the per-thread counts places them, in an order fixed by the columns (thread, then j), so the result
// does not depend on timing.  Every tile of 16 table entries then sits in one tier.
template <int KIND, int CAP, int J>
KVT_DEV void resolve_rows(const SparseArgs& A, int64_t k0, int64_t k1, const int32_t* idx_row, int64_t L,
                          int64_t req, int h, BlockLds<CAP>& S, int& nh, int& nc) {
  constexpr int kThreads = 64 * kWaves;
  static_assert(J * kThreads >= CAP, "a pass covers the table");
  constexpr int kEnd = CAP + 2 * kRows - 1;   // nh + nc <= CAP: the parts and their padding never meet
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // (a later pass's column numbers are formed there, not held across the tile loops)
  const int lane = tid & 63, wave = tid >> 6;
  const int32_t* r2t = A.req_to_token + req * A.req_stride;
  int pos[J], slot[J], own[J];
  bool live[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int64_t c = k0 + tid + (int64_t)j * kThreads;
    pos[j] = c < k1 ? idx_row[c * A.si_n] : -1;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    live[j] = pos[j] >= 0 && (int64_t)pos[j] < L;
    slot[j] = live[j] ? r2t[pos[j]] : 0;
  }
#pragma unroll
  for (int j = 0; j < J; ++j) own[j] = (KIND == 2 && live[j]) ? A.owner[(int64_t)slot[j] & A.ring_mask] : -1;
  bool hot[J];
  int mh = 0, mc = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    hot[j] = KIND == 0 || (KIND == 2 && live[j] && own[j] == slot[j]);
    mh += (live[j] && hot[j]) ? 1 : 0;
    mc += (live[j] && !hot[j]) ? 1 : 0;
  }
  // inclusive scan over the wavefront, then the wavefronts' totals through LDS
  int sh = mh, sc = mc;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int th = __shfl_up(sh, d, 64), tc = __shfl_up(sc, d, 64);
    if (lane >= d) sh += th, sc += tc;
  }
  if (lane == 63) S.counts[wave] = sh, S.counts[kWaves + wave] = sc;
  __syncthreads();
  int oh = sh - mh, oc = sc - mc;
  nh = 0, nc = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const int a = S.counts[w], c = S.counts[kWaves + w];
    if (w < wave) oh += a, oc += c;
    nh += a, nc += c;
  }
  nh = __builtin_amdgcn_readfirstlane(nh), nc = __builtin_amdgcn_readfirstlane(nc);   // (the same in every lane)
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if (!live[j]) continue;
    const int64_t row = hot[j] && KIND == 2 ? ((int64_t)slot[j] & A.ring_mask) : (int64_t)slot[j];
    const uint32_t word = (uint32_t)(row * A.H + h);
    if (hot[j])
      S.cols[oh++] = word;
    else
      S.cols[kEnd - oc++] = word;
  }
  if (tid < kRows) {
    if (nh + tid < (nh + kRows - 1) / kRows * kRows) S.cols[nh + tid] = kNoRow;
    if (nc + tid < (nc + kRows - 1) / kRows * kRows) S.cols[kEnd - nc - tid] = kNoRow;
    S.cols[kEnd + 1 + tid] = kNoRow;
  }
}

// The row words of tile t < nt of a part of the table (HOT: from the front, INT4: from the end), for this lane's
// half; t >= nt: a tile of kNoRow words, whose loads cost no traffic.
template <bool HOT, int CAP>
KVT_DEV void table_tile(const BlockLds<CAP>& S, int t, int nt, int lane, uint32_t e[kPairs]) {
  const int i0 = 16 * t;
  const int lo = t >= nt ? CAP + 2 * kRows : HOT ? i0 : CAP + kRows - i0;   // the tile's lowest table entry
  // (ascending for either part: the order of rows within a tile is of no consequence, the padding's place is)
#pragma unroll
  for (int i = 0; i < kPairs; ++i) e[i] = S.cols[lo + 2 * i + (lane >> 5)];
}

// The attended rows of tile t of a part of n entries: its first n - 16 t words, the last ones in the INT4 part's
// descending order.
template <bool HOT>
KVT_DEV uint32_t table_mask(int t, int n) {
  const int rem = n - 16 * t;
  return rem >= kRows ? 0xffffu : HOT ? (1u << rem) - 1u : (0xffffu << (kRows - rem)) & 0xffffu;
}

// Device-scope stores and loads of the split partials: the partials cross XCDs (each has its own L2), so they are
// written through to the coherence point (read by the combine kernel, or by the block of this launch that merges
// them, which reads past its own L2: cache policy sc1 on the raw buffer accesses).
typedef unsigned int u4v __attribute__((vector_size(16)));   // the raw buffer builtins' 16- and 8-byte operands
typedef unsigned int u2v __attribute__((vector_size(8)));
typedef float f2 __attribute__((ext_vector_type(2)));
constexpr int kSc1 = 16;
KVT_DEV void wait_vm0() {   // s_waitcnt vmcnt(0), the other counters untouched
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}
// The partials of (request b, KV head h): n_splits x gs rows of D floats, then n_splits x gs (m, l) pairs.
KVT_DEV __amdgpu_buffer_rsrc_t part_o_rsrc(const SparseArgs& A, int64_t bh) {
  const int64_t rows = (int64_t)A.n_splits * A.gs;
  return rsrc(A.part_o + bh * rows * kD, (uint32_t)(rows * kD * 4));
}
KVT_DEV __amdgpu_buffer_rsrc_t part_ml_rsrc(const SparseArgs& A, int64_t bh) {
  const int64_t rows = (int64_t)A.n_splits * A.gs;
  return rsrc(A.part_ml + bh * rows * 2, (uint32_t)(rows * 8));
}

// The split merge inside the decode launch: after its partial's device-scope stores have completed, a block counts
// itself on its (request, KV head) counter; the block that counts last resets the counter for the next call and
// merges the n_splits partials in split order (so the result does not depend on which block is last), as
// kvt_decode_combine does for a separate launch: (m, num, den) <- (max(m, m_s), num e^(m - m') + o_s e^(m_s - m'),
// den e^(m - m') + l_s e^(m_s - m')), out = num / den (0 / 0 = NaN when no column was attended).  No block waits for
// another.  Thread t merges q head t / 16, dims 64 j + 4 (t % 16) .. + 3 (j = 0 .. 3), with the loads of 4 splits in flight
// at once: 16 threads read 256 contiguous bytes, so each line of a partial is asked for once past the L2 (16 dims per
// thread in a row asked for every line four times, which at 33 splits cost 461 us per 12 layers against 305; 8 splits in
// flight 315).
template <int CAP>
KVT_DEV void merge_last(const SparseArgs& A, BlockLds<CAP>& S, int b, int h) {
  wait_vm0();
  __syncthreads();   // every thread's partial stores have completed
  const int64_t bh = (int64_t)b * A.H + h;
  if (threadIdx.x == 0)
    S.last = __hip_atomic_fetch_add(&A.counters[bh], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == A.n_splits - 1;
  __syncthreads();
  if (!S.last) return;
  if (threadIdx.x == 0) __hip_atomic_store(&A.counters[bh], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  constexpr float kL2e = 1.4426950408889634f;
  constexpr int kB = 4;
  const int gs = A.gs, ns = A.n_splits;
  const int hq = (int)(threadIdx.x >> 4), c0 = 4 * (int)(threadIdx.x & 15);
  if (hq >= gs) return;
  const auto ro = part_o_rsrc(A, bh), rml = part_ml_rsrc(A, bh);
  float m = -INFINITY, den = 0.f, num[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) num[i] = 0.f;
  for (int s0 = 0; s0 < ns; s0 += kB) {
    f4 o[kB][4];
    f2 ml[kB];
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int s = s0 + k < ns ? s0 + k : s0;
      const int row = s * gs + hq;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o[k][j] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(ro, (row * kD + c0 + 64 * j) * 4, 0,
                                                                                kSc1));
      ml[k] = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(rml, row * 8, 0, kSc1));
    }
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      if (s0 + k >= ns) break;
      const float ms = ml[k][0], ls = ml[k][1];
      const float mn = fmaxf(m, ms);
      if (mn == -INFINITY) continue;   // both empty
      const float a = __builtin_amdgcn_exp2f((m - mn) * kL2e), c = __builtin_amdgcn_exp2f((ms - mn) * kL2e);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) num[4 * j + i] = num[4 * j + i] * a + o[k][j][i] * c;
      den = den * a + ls * c;
      m = mn;
    }
  }
  const int64_t off = (int64_t)b * A.mout_b + (int64_t)(h * gs + hq) * kD + c0;
  if (A.mout_f32 != nullptr) {
    float* dst = A.mout_f32 + off;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(dst + 64 * j) =
          float4{num[4 * j] / den, num[4 * j + 1] / den, num[4 * j + 2] / den, num[4 * j + 3] / den};
  } else {
    uint16_t* dst = A.mout_bf16 + off;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<uint2*>(dst + 64 * j) = uint2{bf16x2(num[4 * j] / den, num[4 * j + 1] / den),
                                                      bf16x2(num[4 * j + 2] / den, num[4 * j + 3] / den)};
  }
}

// XCD-aware work mapping.  The workgroups of a launch go to the 8 XCDs round robin by linear id, and each XCD has
// its own L2, so the block with linear id L takes the work item that shares lines with the items of ids L +- 8:
// * decode (grid n_splits x batch H): item i = b n_splits + split, in groups of 8 items whose H KV heads take ids
//   8 H g + 8 h + (i % 8) -- the blocks of one (request, split) run on one XCD side by side and share the lines of
//   the index, req_to_token and owner reads and of the rows' scales (both heads' scales sit in one 32-byte run);
// * prefill rows (grid max_q x batch H): XCD x takes the x-th eighth of the (query, KV head) items, consecutive
//   queries of one chunk, whose selections overlap.
// A tail of fewer than 8 items (decode) or ids (rows) keeps a plain order.
constexpr int kXcds = 8;
template <bool ROWS>
KVT_DEV void work_of_block(int H, int& wx, int& wy) {
  const uint32_t nx = gridDim.x, n = nx * gridDim.y, L = blockIdx.x + blockIdx.y * nx;
  if constexpr (ROWS) {
    const uint32_t m = n / kXcds * kXcds;
    const uint32_t w = L < m ? (L % kXcds) * (m / kXcds) + L / kXcds : L;
    wx = (int)(w % nx), wy = (int)(w / nx);
  } else {
    const uint32_t T = n / (uint32_t)H, full = T / kXcds * kXcds, gh = kXcds * (uint32_t)H;
    uint32_t i, hh;
    if (L < full * (uint32_t)H) {
      hh = (L % gh) / kXcds;
      i = L / gh * kXcds + L % kXcds;
    } else {
      const uint32_t t = T - full, r = L - full * (uint32_t)H;
      hh = r / t;
      i = full + r % t;
    }
    const uint32_t b = i / nx;
    wx = (int)(i - b * nx), wy = (int)(b * (uint32_t)H + hh);
  }
}

// The buffer resources of one tier (HOT: the INT8 tensors -- the ring when tiered --, else the INT4 pool), the
// other tier's left empty.  A block with a column table builds them just before that tier's tiles: the pointers
// pass through empty asm statements, so the compiler cannot hoist them to the kernel start and keep both tiers'
// 8 descriptors (32 scalar registers) live through the tile loops.
template <int KIND, int G8, bool HOT>
KVT_DEV PoolRsrc tier_rsrc(const SparseArgs& A, int H) {
  const void* pk = HOT && KIND == 2 ? (const void*)A.rk : A.k;
  const void* pv = HOT && KIND == 2 ? (const void*)A.rv : A.v;
  const void* pks = HOT && KIND == 2 ? (const void*)A.rks : (const void*)A.ks;
  const void* pvs = HOT && KIND == 2 ? (const void*)A.rvs : (const void*)A.vs;
  asm volatile("" : "+s"(pk), "+s"(pv), "+s"(pks), "+s"(pvs));
  PoolRsrc P{};
  if constexpr (HOT) {
    const uint32_t n8 = A.rows8 * (uint32_t)H * kD, s8 = A.rows8 * (uint32_t)H * (kD / G8) * 2;
    P.k8 = rsrc(pk, n8), P.v8 = rsrc(pv, n8), P.ks8 = rsrc(pks, s8), P.vs8 = rsrc(pvs, s8);
    P.k4 = P.v4 = P.ks4 = P.vs4 = rsrc(nullptr, 0u);
  } else {
    const uint32_t n4 = A.rows4 * (uint32_t)H * (kD / 2), s4 = A.rows4 * (uint32_t)H * (kD / kG4) * 2;
    P.k4 = rsrc(pk, n4), P.v4 = rsrc(pv, n4), P.ks4 = rsrc(pks, s4), P.vs4 = rsrc(pvs, s4);
    P.k8 = P.v8 = P.ks8 = P.vs8 = rsrc(nullptr, 0u);
  }
  return P;
}

template <bool B>
struct Flag {
  static constexpr bool value = B;
};

// ROWS: prefill rows (one query row per block) instead of decode splits; MULTI: a decode block of several tiles per
// wavefront; CAP > 1: the block resolves its columns into a column table of CAP entries partitioned by tier first.
template <int KIND, int G8, bool ROWS, bool MULTI, int CAP>
KVT_DEV void sparse_attn_block(const SparseArgs& A, BlockLds<CAP>& S) {
  auto& kv = S.kv;
  uint16_t* qs = S.qs;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = A.H, gs = A.gs;
  int wx, wy;   // the work item: split (decode) or query (rows), and request / chunk x H + KV head
  work_of_block<ROWS>(H, wx, wy);
  const int b = wy / H;
  const int h = wy - b * H;
  // The start-up loads go out in as few dependent rounds as the data allows: the request's index-array entries and
  // length together (no wait between them), with the decode's q rows and the smoothing factors into registers; then
  // the first tile's resolve chain (position, slot, owner).  The q rows reach LDS after the chain.
  const IdxWords wreq = idx_words(A.req_indices, A.req64, b);
  const IdxWords w0 = ROWS ? idx_words(A.cu_q, A.cuq64, b) : idx_words(A.cu_k, A.cu64, b);
  const IdxWords w1 = ROWS ? idx_words(A.cu_q, A.cuq64, b + 1) : idx_words(A.cu_k, A.cu64, b + 1 - A.all_columns);
  const int32_t len = ROWS ? A.kv_lens[b] : A.seq_lens[b];   // widened after the barrier (no wait before it)
  // the group's q heads (512 16-byte chunks, 2 per thread; heads beyond the group read head 0 and are zeroed)
  constexpr int kQChunks = kHeads * kD / 8 / (64 * kWaves);
  uint4 qv[kQChunks];
  auto load_q = [&](int64_t row) {
#pragma unroll
    for (int k = 0; k < kQChunks; ++k) {
      const int i = (int)threadIdx.x + 64 * kWaves * k;
      const int hq = i / (kD / 8), ch = i - hq * (kD / 8);
      const int hr = hq < gs ? hq : 0;
      const uint4 w = *reinterpret_cast<const uint4*>(A.q + row * A.sq_n + (int64_t)(h * gs + hr) * A.sq_h + 8 * ch);
      qv[k] = hq < gs ? w : uint4{0u, 0u, 0u, 0u};
    }
  };
  if constexpr (!ROWS) load_q(b);
  // the head's smoothing factors, 2 per thread: K's, then V's (an absent tensor: all 1).  The tensors need only 2-byte
  // alignment.
  typedef uint32_t u32_at2 __attribute__((aligned(2)));
  const uint16_t* smp = threadIdx.x < kD / 2 ? A.sm_k : A.sm_v;
  const uint32_t smw = smp != nullptr ? reinterpret_cast<const u32_at2*>(smp + h * kD)[threadIdx.x & (kD / 2 - 1)]
                                      : 0x3c003c00u;
  __builtin_amdgcn_sched_barrier(0);
  const int64_t req = idx_value(wreq), x0 = idx_value(w0), x1 = idx_value(w1), L = len;
  // the block's query row and column range
  int64_t qrow, c_begin, c_end;
  if constexpr (ROWS) {
    const int64_t j = wx;
    if (x0 + j >= x1) return;   // block-uniform: the chunk is shorter than the grid
    qrow = x0 + j;
    load_q(qrow);
    const int64_t visible = j + L - (x1 - x0) + 1;
    c_begin = 0;
    c_end = visible < (int64_t)A.topk ? (visible > 0 ? visible : 0) : (int64_t)A.topk;
  } else {
    qrow = b;
    const int64_t vcount = A.all_columns != 0 ? (int64_t)A.topk : x1 - x0;
    const int64_t span = (int64_t)kCols * (MULTI ? A.tiles : 1);
    c_begin = (int64_t)wx * span;
    const int64_t lim = vcount < (int64_t)A.topk ? vcount : (int64_t)A.topk;
    c_end = c_begin + span < lim ? c_begin + span : lim;
  }

  const int32_t* idx_row = A.indices + qrow * A.si_m + (int64_t)h * A.si_g;
  // every scalar the resolve chain needs, in registers here: the compiler would otherwise sink these loads (and the
  // kernel-argument reads) into the chain's branch, one wait each, behind the index load
  asm volatile("" ::"s"(idx_row), "s"(L), "s"(req), "s"(c_end), "s"(A.req_to_token), "s"(A.req_stride),
               "s"(A.owner), "s"(A.ring_mask), "s"(A.si_n));
  // the wavefront's first tile (prefill rows: the first pass of the column table)
  uint32_t word0 = kNoRow;
  const bool has_tile = c_begin + kRows * wave < c_end;
  int nh = 0, nc = 0;
  if constexpr (CAP > 1)
    resolve_rows<KIND, CAP, CAP / (64 * kWaves)>(A, c_begin, c_begin + CAP < c_end ? c_begin + CAP : c_end, idx_row,
                                                     L, req, h, S, nh, nc);
  else if (has_tile)
    word0 = resolve_tile<KIND>(A, c_begin + kRows * wave, c_end, idx_row, L, req, h, lane);
#pragma unroll
  for (int k = 0; k < kQChunks; ++k) {
    const int i = (int)threadIdx.x + 64 * kWaves * k;
    const int hq = i / (kD / 8), ch = i - hq * (kD / 8);
    *reinterpret_cast<uint4*>(&qs[hq * kKPitch + 8 * ch]) = qv[k];
  }
  PoolRsrc P;   // both tiers' descriptors, for the one-tile blocks (a column table's loops build one tier's each)
  if constexpr (CAP == 1) {
    const uint32_t n8 = A.rows8 * (uint32_t)H * kD, n4 = A.rows4 * (uint32_t)H * (kD / 2);
    const uint32_t s8 = A.rows8 * (uint32_t)H * (kD / G8) * 2, s4 = A.rows4 * (uint32_t)H * (kD / kG4) * 2;
    P.k8 = rsrc(KIND == 2 ? (const void*)A.rk : A.k, KIND == 1 ? 0u : n8);
    P.v8 = rsrc(KIND == 2 ? (const void*)A.rv : A.v, KIND == 1 ? 0u : n8);
    P.ks8 = rsrc(KIND == 2 ? A.rks : A.ks, KIND == 1 ? 0u : s8);
    P.vs8 = rsrc(KIND == 2 ? A.rvs : A.vs, KIND == 1 ? 0u : s8);
    P.k4 = rsrc(A.k, KIND == 0 ? 0u : n4);
    P.v4 = rsrc(A.v, KIND == 0 ? 0u : n4);
    P.ks4 = rsrc(A.ks, KIND == 0 ? 0u : s4);
    P.vs4 = rsrc(A.vs, KIND == 0 ? 0u : s4);
  }
  reinterpret_cast<uint32_t*>(S.sm)[threadIdx.x] = smw;
  const bool ones = __all(smw == 0x3c003c00u);
  if (lane == 0) S.ones[wave] = ones;
  __syncthreads();   // q staged
  // every factor of the head 1: the bodies without the products
  const bool identity = __builtin_amdgcn_readfirstlane(S.ones[0] & S.ones[1] & S.ones[2] & S.ones[3]) != 0;

  // the B operands of the score products: channels 32 k + 8 (lane >> 4) .. + 7 of q head lane & 15
  bf8 qop[8];
#pragma unroll
  for (int k = 0; k < 8; ++k)
    qop[k] = __builtin_bit_cast(bf8, *reinterpret_cast<const uint4*>(&qs[(lane & 15) * kKPitch + 32 * k + 8 * (lane >> 4)]));

  float m_run = -INFINITY, l_run = 0.f;   // of q head lane & 15
  f4 o[16];                               // O[head 4 (lane >> 4) + i][channel 16 n + (lane & 15)]
#pragma unroll
  for (int n = 0; n < 16; ++n) o[n] = f4{0.f, 0.f, 0.f, 0.f};
  if constexpr (CAP > 1) {
    // passes of the column table (the first resolved above): wavefront w takes tiles w, w + 4, ..., ring tiles first.
    // The choice by the smoothing factors stands outside the passes: inside, the two bodies' accumulators were held
    // in separate registers.
    auto passes = [&](auto smooth) {
      constexpr bool SM = decltype(smooth)::value;
      for (int64_t k0 = c_begin; k0 < c_end; k0 += CAP) {
        const int64_t k1 = k0 + CAP < c_end ? k0 + CAP : c_end;
        if (k0 > c_begin) {
          __syncthreads();   // the previous pass's entries are read
          resolve_rows<KIND, CAP, CAP / (64 * kWaves)>(A, k0, k1, idx_row, L, req, h, S, nh, nc);
          __syncthreads();
        }
        const int th = (nh + kRows - 1) / kRows, nt = th + (nc + kRows - 1) / kRows;
        int t = wave;
        // the tiles t, t + kWaves, .. < t_end of one tier (t0: its first tile, n: its entries)
        auto run = [&](const PoolRsrc& R, auto hot, int t0, int t_end, int n) {
          constexpr bool HOT = decltype(hot)::value;
          constexpr int T = HOT ? kRowsInt8 : kRowsInt4;
          if (t >= t_end) return;
          uint32_t e[kPairs];
          Raw K, V;
          table_tile<HOT>(S, t - t0, t_end - t0, lane, e);
          issue_rows<G8, T>(R.k8, R.ks8, R.k4, R.ks4, e, lane, K);
          issue_rows<G8, T>(R.v8, R.vs8, R.v4, R.vs4, e, lane, V);
          for (; t < t_end; t += kWaves) {
            table_tile<HOT>(S, t + kWaves - t0, t_end - t0, lane, e);
            attend_tile<G8, T, SM, true>(A, R, qop, kv[wave], K, V, e, table_mask<HOT>(t - t0, n), e, lane, S.sm, m_run,
                                         l_run, o);
          }
        };
        // the ring (INT8) tiles, then the INT4 ones, each tier's descriptors in turn
        if constexpr (KIND != 1) run(tier_rsrc<KIND, G8, true>(A, H), Flag<true>{}, 0, th, nh);
        if constexpr (KIND != 0) run(tier_rsrc<KIND, G8, false>(A, H), Flag<false>{}, th, nt, nc);
      }
    };
    if (identity)
      passes(Flag<false>{});
    else
      passes(Flag<true>{});
  } else if (has_tile) {   // at most one tile per wavefront (64 columns per block): no state is live across its loads
    if (identity)
      attend_tile_any<KIND, G8, false>(A, P, qop, kv[wave], word0, lane, S.sm, m_run, l_run, o);
    else
      attend_tile_any<KIND, G8, true>(A, P, qop, kv[wave], word0, lane, S.sm, m_run, l_run, o);
  }

  // merge the 4 wavefronts through LDS, 8 q heads per pass: wavefront w stores the O rows of the pass's heads and
  // (m, l) of every head; thread t then merges head t / 32 of the pass, channels 8 (t % 32) .. + 7, over the 4
  __syncthreads();   // every wavefront is done with its tile rows
  float* mo = reinterpret_cast<float*>(&kv[0][0]);   // [wave][8 heads][256]
  float* mml = mo + kWaves * 8 * kD;                  // [wave][16 heads][2]
  const int kq = lane >> 4, n16 = lane & 15;
  if (lane < gs) {
    mml[(wave * kHeads + lane) * 2] = m_run;
    mml[(wave * kHeads + lane) * 2 + 1] = l_run;
  }
  for (int hh = 0; hh < gs; hh += 8) {
    if (hh > 0) __syncthreads();   // the previous pass's reads are done
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int hq = 4 * kq + i - hh;
      if (hq >= 0 && hq < 8 && hq + hh < gs) {
#pragma unroll
        for (int n = 0; n < 16; ++n) mo[(wave * 8 + hq) * kD + 16 * n + n16] = o[n][i];
      }
    }
    __syncthreads();
    const int hq = hh + (threadIdx.x >> 5), c0 = 8 * (threadIdx.x & 31);
    if (hq < gs) {
      float mw[kWaves], M = -INFINITY;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        mw[w] = mml[(w * kHeads + hq) * 2];
        M = fmaxf(M, mw[w]);
      }
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, lt = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float a = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);
        lt += a * mml[(w * kHeads + hq) * 2 + 1];
        const float* src = &mo[(w * 8 + (hq - hh)) * kD + c0];
        const float4 o0 = *reinterpret_cast<const float4*>(src);
        const float4 o1 = *reinterpret_cast<const float4*>(src + 4);
        acc[0] += a * o0.x;
        acc[1] += a * o0.y;
        acc[2] += a * o0.z;
        acc[3] += a * o0.w;
        acc[4] += a * o1.x;
        acc[5] += a * o1.y;
        acc[6] += a * o1.z;
        acc[7] += a * o1.w;
      }
      if constexpr (ROWS) {
        // normalized output; nothing attended gives 0 / 0 = NaN (patches/kv_paged_prefix.py:259)
        const int64_t off = qrow * A.so_n + (int64_t)(h * gs + hq) * A.so_h + c0;
        if (A.out_f32) {
          float* dst = reinterpret_cast<float*>(A.out) + off;
          *reinterpret_cast<float4*>(dst) = float4{acc[0] / lt, acc[1] / lt, acc[2] / lt, acc[3] / lt};
          *reinterpret_cast<float4*>(dst + 4) = float4{acc[4] / lt, acc[5] / lt, acc[6] / lt, acc[7] / lt};
        } else {
          uint16_t* dst = reinterpret_cast<uint16_t*>(A.out) + off;
          *reinterpret_cast<uint4*>(dst) = uint4{bf16x2(acc[0] / lt, acc[1] / lt), bf16x2(acc[2] / lt, acc[3] / lt),
                                                 bf16x2(acc[4] / lt, acc[5] / lt), bf16x2(acc[6] / lt, acc[7] / lt)};
        }
      } else {
        // The partial, read after this launch by the combine kernel or inside it by the block that counts last, on
        // any XCD: device-scope stores (sc1), written through past this XCD's L2, so that no write-back of them is
        // left for the kernel's end (top-k decode 182.8 -> 180.4 us per step against plain stores)
        constexpr float kLn2 = 0.6931471805599453f;
        const float mnat = M == -INFINITY ? -INFINITY : M * kLn2;   // m of the block's partial in natural-log units
        const int row = wx * gs + hq;
        const auto ro = part_o_rsrc(A, (int64_t)b * H + h);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, f4{acc[0], acc[1], acc[2], acc[3]}), ro,
                                               (row * kD + c0) * 4, 0, kSc1);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, f4{acc[4], acc[5], acc[6], acc[7]}), ro,
                                               (row * kD + c0 + 4) * 4, 0, kSc1);
        if (c0 == 0)
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, f2{mnat, lt}),
                                                part_ml_rsrc(A, (int64_t)b * H + h), row * 8, 0, kSc1);
      }
    }
  }
  if constexpr (!ROWS) {
    if (A.counters != nullptr) merge_last(A, S, b, h);
  }
}

// decode: one tile per wavefront, 3 blocks per CU
template <int KIND, int G8>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(3))) sparse_decode_kernel(SparseArgs A) {
  __shared__ __align__(16) BlockLds<1> S;
  sparse_attn_block<KIND, G8, false, false, 1>(A, S);
}

// decode of long selections: the block's 64 A.tiles columns resolved into its column table, a wavefront looping over
// its tiles with the accumulators and the next tile's rows live; 2 blocks per CU (held to the 168 registers of 3, the
// next tile's loads and the operand reads no longer overlap: 74 us against 55 us)
template <int KIND, int G8>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2)))
sparse_decode_multi_kernel(SparseArgs A) {
  __shared__ __align__(16) BlockLds<kMultiCols> S;
  sparse_attn_block<KIND, G8, false, true, kMultiCols>(A, S);
}

// prefill rows: the query's selection resolved into the column table, a wavefront looping over its tiles with the
// accumulators live; 2 blocks per CU
template <int KIND, int G8>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) sparse_prefill_kernel(SparseArgs A) {
  __shared__ __align__(16) BlockLds<kRowCols> S;
  sparse_attn_block<KIND, G8, true, false, kRowCols>(A, S);
}

// Shared argument checks and pool resources of both entry points; returns KVT_OK or a status.
int pool_args(int kind, int64_t pool_rows, const void* ring_k, const void* owner, int64_t ring_mask, int H, int Hq,
              int D, int group8, int64_t* rows8, int64_t* rows4) {
  if (H <= 0 || Hq % H != 0 || Hq / H > kHeads || D != kD || kind < 0 || kind > 2) return KVT_EINVAL;
  if (kind == 2 && (owner == nullptr || ring_k == nullptr || ((ring_mask + 1) & ring_mask) != 0)) return KVT_EINVAL;
  if (pool_rows <= 0 || (kind != 1 && group8 != 64 && group8 != 256)) return KVT_EINVAL;
  // byte offsets are 32-bit and must stay below 2^31 (rows * H * D bytes of INT8 codes, / 2 for INT4)
  *rows8 = kind == 2 ? ring_mask + 1 : (kind == 0 ? pool_rows : 0);
  *rows4 = kind == 0 ? 0 : pool_rows;
  if (*rows8 * H * kD >= (1ll << 31) || *rows4 * H * (kD / 2) >= (1ll << 31)) return KVT_ERANGE;
  return KVT_OK;
}

template <bool ROWS>
int launch(int kind, int group8, dim3 grid, hipStream_t st, const SparseArgs& A) {
#define KVT_SD(KIND_, G_)                                                                                  \
  do {                                                                                                     \
    if constexpr (ROWS)                                                                                    \
      hipLaunchKernelGGL((sparse_prefill_kernel<KIND_, G_>), grid, dim3(64 * kWaves), 0, st, A);           \
    else if (A.tiles > 1)                                                                                  \
      hipLaunchKernelGGL((sparse_decode_multi_kernel<KIND_, G_>), grid, dim3(64 * kWaves), 0, st, A);      \
    else                                                                                                   \
      hipLaunchKernelGGL((sparse_decode_kernel<KIND_, G_>), grid, dim3(64 * kWaves), 0, st, A);            \
  } while (0)
  if (kind == 1) {
    KVT_SD(1, 64);
  } else if (group8 == 64) {
    if (kind == 2) {
      KVT_SD(2, 64);
    } else {
      KVT_SD(0, 64);
    }
  } else {
    if (kind == 2) {
      KVT_SD(2, 256);
    } else {
      KVT_SD(0, 256);
    }
  }
#undef KVT_SD
  KVT_CHECK_LAUNCH();
  return KVT_OK;
}

}  // namespace

extern "C" {

int kvt_sparse_decode(int kind, const void* q, int64_t q_stride_b, const void* k, const void* v, const void* k_scale,
                      const void* v_scale, int64_t pool_rows, const void* ring_k, const void* ring_v, const void* ring_ks,
                      const void* ring_vs, const void* owner, int64_t ring_mask, const void* sm_k, const void* sm_v,
                      const void* req_to_token, int64_t req_stride, const void* req_indices, int req_is_int64,
                      const void* indices, int64_t idx_stride, const void* seq_lens, const void* cu_k,
                      int cu_is_int64, int batch, int topk, int H, int Hq, int D, int group8, float scale,
                      int n_splits, void* part_o, void* part_ml, void* counters, void* out_f32, void* out_bf16,
                      int64_t out_stride_b, void* stream) {
  if (batch <= 0 || topk <= 0 || n_splits <= 0) return KVT_EINVAL;
  // one (request, KV head)'s partials are addressed with 32-bit offsets
  if ((int64_t)n_splits * (Hq / (H > 0 ? H : 1)) * D * 4 >= (1ll << 31)) return KVT_EINVAL;
  if (counters != nullptr && ((out_f32 == nullptr) == (out_bf16 == nullptr) || out_stride_b < (int64_t)Hq * D ||
                              ((uintptr_t)(out_f32 != nullptr ? out_f32 : out_bf16) & 15) != 0 ||
                              (out_stride_b & 7) != 0))
    return KVT_EINVAL;   // merged in the launch: 16-byte output pieces
  // n_splits blocks per (request, KV head) cover the topk columns with `tiles` 16-column tiles per wavefront
  const int tiles64 = (topk + kCols - 1) / kCols;
  const int tiles = (tiles64 + n_splits - 1) / n_splits;
  if ((q_stride_b & 7) != 0 || ((uintptr_t)q & 15) != 0) return KVT_EINVAL;
  int64_t rows8 = 0, rows4 = 0;
  const int st_ = pool_args(kind, pool_rows, ring_k, owner, ring_mask, H, Hq, D, group8, &rows8, &rows4);
  if (st_ != KVT_OK) return st_;
  SparseArgs A{};
  A.k = k, A.v = v, A.ks = (const uint16_t*)k_scale, A.vs = (const uint16_t*)v_scale;
  A.rk = (const int8_t*)ring_k, A.rv = (const int8_t*)ring_v, A.rks = (const uint16_t*)ring_ks;
  A.rvs = (const uint16_t*)ring_vs, A.owner = (const int32_t*)owner, A.ring_mask = ring_mask;
  A.sm_k = (const uint16_t*)sm_k, A.sm_v = (const uint16_t*)sm_v;
  A.req_to_token = (const int32_t*)req_to_token, A.req_stride = req_stride, A.req_indices = req_indices;
  A.req64 = req_is_int64 != 0, A.indices = (const int32_t*)indices, A.idx_stride = idx_stride;
  A.seq_lens = (const int32_t*)seq_lens, A.cu_k = cu_k != nullptr ? cu_k : seq_lens, A.cu64 = cu_k != nullptr && cu_is_int64 != 0;
  A.all_columns = cu_k == nullptr, A.topk = topk;
  A.H = H, A.gs = Hq / H, A.n_splits = n_splits, A.tiles = tiles, A.rows8 = (uint32_t)rows8;
  A.rows4 = (uint32_t)rows4, A.scale = scale, A.q = (const uint16_t*)q, A.sq_n = q_stride_b, A.sq_h = kD;
  A.si_m = idx_stride, A.si_g = 0, A.si_n = 1, A.part_o = (float*)part_o, A.part_ml = (float*)part_ml;
  A.counters = (int32_t*)counters, A.mout_f32 = (float*)out_f32, A.mout_bf16 = (uint16_t*)out_bf16;
  A.mout_b = out_stride_b;
  return launch<false>(kind, group8, dim3((unsigned)n_splits, (unsigned)(batch * H)), (hipStream_t)stream, A);
}

int kvt_sparse_prefill(int kind, const void* q, int64_t sq_n, int64_t sq_h, const void* cu_q, int cu_q_is_int64,
                       const void* kv_lens, int batch, int max_q, const void* indices, int64_t si_m, int64_t si_g,
                       int64_t si_n, int topk, const void* k, const void* v, const void* k_scale, const void* v_scale,
                       int64_t pool_rows, const void* ring_k, const void* ring_v, const void* ring_ks,
                       const void* ring_vs, const void* owner, int64_t ring_mask, const void* sm_k, const void* sm_v,
                       const void* req_to_token, int64_t req_stride, const void* req_indices, int req_is_int64, int H,
                       int Hq, int D, int group8, float scale, void* out, int out_f32, int64_t so_n, int64_t so_h,
                       void* stream) {
  if (batch < 0 || max_q < 0 || topk < 0) return KVT_EINVAL;
  // 16-byte q loads and output stores: row and head strides multiples of 8 elements (4 for fp32 output)
  if ((sq_n & 7) != 0 || (sq_h & 7) != 0 || ((uintptr_t)q & 15) != 0) return KVT_EINVAL;
  if (((uintptr_t)out & 15) != 0 || (so_n & (out_f32 ? 3 : 7)) != 0 || (so_h & (out_f32 ? 3 : 7)) != 0) return KVT_EINVAL;
  int64_t rows8 = 0, rows4 = 0;
  const int st_ = pool_args(kind, pool_rows, ring_k, owner, ring_mask, H, Hq, D, group8, &rows8, &rows4);
  if (st_ != KVT_OK) return st_;
  if (batch == 0 || max_q == 0) return KVT_OK;
  SparseArgs A{};
  A.k = k, A.v = v, A.ks = (const uint16_t*)k_scale, A.vs = (const uint16_t*)v_scale;
  A.rk = (const int8_t*)ring_k, A.rv = (const int8_t*)ring_v, A.rks = (const uint16_t*)ring_ks;
  A.rvs = (const uint16_t*)ring_vs, A.owner = (const int32_t*)owner, A.ring_mask = ring_mask;
  A.sm_k = (const uint16_t*)sm_k, A.sm_v = (const uint16_t*)sm_v;
  A.req_to_token = (const int32_t*)req_to_token, A.req_stride = req_stride, A.req_indices = req_indices;
  A.req64 = req_is_int64 != 0, A.indices = (const int32_t*)indices, A.topk = topk;
  A.H = H, A.gs = Hq / H, A.n_splits = 1, A.tiles = 1, A.rows8 = (uint32_t)rows8, A.rows4 = (uint32_t)rows4;
  A.scale = scale, A.q = (const uint16_t*)q, A.sq_n = sq_n, A.sq_h = sq_h;
  A.si_m = si_m, A.si_g = si_g, A.si_n = si_n;
  A.cu_q = cu_q, A.cuq64 = cu_q_is_int64 != 0, A.kv_lens = (const int32_t*)kv_lens;
  A.out = out, A.out_f32 = out_f32, A.so_n = so_n, A.so_h = so_h;
  return launch<true>(kind, group8, dim3((unsigned)max_q, (unsigned)(batch * H)), (hipStream_t)stream, A);
}

}  // extern "C"
