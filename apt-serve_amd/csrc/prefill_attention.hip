// Causal attention over freshly projected, packed (varlen) q/k/v for gfx950 — the prompt step.
//
// One 256-thread workgroup owns 128 (64) consecutive queries of one (sequence, head); each of its four
// wavefronts owns QT = 2 (1) tiles of 16 of them.  Keys/values are consumed 64 at a time through LDS.
//
// The score tile is computed transposed, S^T = K Q^T, with v_mfma_f32_16x16x32: in the result layout
// a lane owns ONE query (column lane%16) of each of its wavefront's query tiles and 4 of the 16 keys of
// every key tile, so the running max / sum of the online softmax are per-lane scalars plus two exchanges
// between the 16-lane rows.  The same registers, rounded to the operand dtype, are directly the B operand
// (k = keys) of O^T = V^T P^T, provided V^T comes in the key order the result layout produces: the lane
// of quad g takes keys 4g .. 4g+3 of two neighbouring key tiles.
// K and V tiles are copied global -> LDS (buffer_load ... lds) one tile ahead into a ring of two stages, row-major
// with their 16- and 32-byte pieces XOR-swizzled on the source side; V^T fragments are read with ds_read_b64_tr_b16,
// which hands the 16 lanes of a row a 4-key x 16-d block transposed.  No tile passes through registers, and one
// barrier a tile is enough.
// (The part lowers its clock under real operands, and 16x16x32 costs less energy per flop than 32x32x16:
// 4 x 2048 tokens of 40 x 128 f16 251 -> 243 us, and 243 -> 221 with the copies in place of staging registers.)
//
// PAGED variant (a prompt step that continues a cached prefix: chunked prompts, prefix caching): the queries are
// the step's new tokens, the keys and values the whole sequence so far — prefix and new tokens alike — read from
// the paged K/V cache through the sequence's block table; query i of a sequence with qlen new tokens and klen
// tokens in all attends to keys 0 .. i + (klen - qlen).  Everything after the address of a key row is shared.
#include "aps_common.h"
#include "mfma_common.h"

#include <math.h>

#include <algorithm>

namespace aps {
namespace {

constexpr int BKV = 64;   // keys per iteration
constexpr int kThreads = 256;
constexpr float kLog2e = 1.4426950408889634f;

struct PrefillArgs {
  const char* q; const char* k; const char* v; char* out;
  const int32_t* cu_seqlens;
  int64_t q_stride_b, k_stride_b, v_stride_b, out_stride_b;  // token row strides in bytes
  int num_heads;
  int64_t num_tokens;  // rows of q / k / v / out: sequence boundaries outside [0, num_tokens] are not followed
  float scale_log2;
  // PAGED: k / v are [blocks, block_size, heads, D] caches, k_stride_b / v_stride_b their token row strides
  const int32_t* cu_seqlens_k; const int32_t* block_tables;
  int64_t table_stride, table_width, block_stride_b, num_blocks;
  int block_size;
  int groups_shift;   // kPaged16: block_size = 16 << groups_shift
  // PAGED, key parts: a workgroup multiplies one of at most `parts` runs of key tiles of its queries, as many as runs of `part_tiles`
  // tiles take; with more than one of them fp32 sums, maxima and weights go to `partial` (one unit per workgroup: the O^T
  // registers as they lie, then max and sum per query) and prefill_combine_kernel adds them.
  int parts, part_tiles;
  float* partial;
};

// Key tiles of each part of a query tile that meets n key tiles (the last part may have fewer)
__device__ __forceinline__ int tiles_per_part(int n, int parts, int part_tiles) {
  const int p = min(parts, (n + part_tiles - 1) / part_tiles);
  return (n + p - 1) / p;
}
constexpr int kPartQueries = 64;   // queries per workgroup of a step in parts
template <int D>
__host__ __device__ constexpr int64_t unit_floats() { return kPartQueries * (D + 2); }
// Units of a query tile: tiles before it are counted as if each sequence began a new one behind the tokens in front of it
__device__ __forceinline__ int64_t first_unit(int s0, int seq, int q_tile, int heads, int head, int parts) {
  return ((int64_t)(s0 / kPartQueries + seq + q_tile) * heads + head) * parts;
}

// Two stages of a K and a V tile
template <int D>
constexpr int prefill_lds_bytes() { return 2 * 2 * BKV * D * 2; }

// Where the keys come from: packed rows; blocks of 16, 32, 64, ... tokens, so that 16 consecutive keys from a multiple
// of 16 on lie together in one block; the same key by key, for row pitches past 32 MiB and blocks of any other size.
enum KeySource { kPacked, kPaged16, kPackedAny, kPagedAny };

// PARTS: keys in several parts.  A variant of its own: in the one for all, steps of one part (6 sequences, 2048 tokens on 4200
// cached) ran 0.4 % longer.
template <bool BF16, int D, int SRC, int QT, bool PARTS>
// Two workgroups per CU (64 KiB of LDS each at head size 128) are two wavefronts per SIMD: the compiler may use the
// registers that leaves (202 at 128 queries a workgroup).  Head size 64 has the same bound, though its 32 KiB would leave room
// for more.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_attention_kernel(
    const PrefillArgs a) {
  constexpr int BQ = 64 * QT;         // queries per workgroup
  constexpr bool PAGED = SRC == kPaged16 || SRC == kPagedAny;
  constexpr int KS = D / 32;          // k-steps of the score product
  constexpr int KT = BKV / 16;        // key tiles of a score tile
  constexpr int DT = D / 16;          // 16-row tiles of O^T
  constexpr int KROW = D * 2;         // bytes per key row in LDS
  constexpr int KCH = KROW / 16;      // 16-byte chunks per key row
  constexpr int kTile = BKV * KROW, kStage = 2 * kTile;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  // K in LDS: 16-byte chunk c of key row r sits at slot c ^ k_swz(r), so that 16 consecutive rows read at one chunk (a
  // fragment) meet 16 different bank groups.  V: chunk c at slot c ^ v_swz(r), which moves 32-byte pieces: a transposing
  // read takes 32 bytes of each of 8 consecutive rows per pass, from 8 different bank groups.
  auto k_swz = [](int key) { return KCH == 16 ? key & 15 : (key >> 1) & 7; };
  auto v_swz = [](int key) { return KCH == 16 ? (key & 7) << 1 : ((key >> 1) & 3) << 1; };

  // Grid (head, sequence, query tile), the last query tiles first: under the causal mask a workgroup's work grows
  // with its tile's position, and workgroups start in grid order, so the long ones go first and the short ones
  // fill the end (list scheduling).
  const int seq = blockIdx.y, head = blockIdx.x;
  const int s0 = a.cu_seqlens[seq], s1 = a.cu_seqlens[seq + 1];
  if (s0 < 0 || s1 < s0 || s1 > a.num_tokens) return;  // boundaries come from device memory: never follow bad ones
  const int qlen = s1 - s0;          // queries of this sequence in this step
  int len = qlen;                    // keys: the same tokens, or (PAGED) everything cached so far
  if constexpr (PAGED) {
    len = a.cu_seqlens_k[seq + 1] - a.cu_seqlens_k[seq];
    if (len < qlen || (int64_t)(len + a.block_size - 1) / a.block_size > a.table_width) return;
  }
  const int off = len - qlen;        // query i sees keys 0 .. i + off
  int part = 0, q_tile = (int)(gridDim.z - 1 - blockIdx.z);
  if constexpr (PARTS) {
    part = (int)(blockIdx.z % (unsigned)a.parts);
    q_tile = (int)((gridDim.z - 1 - blockIdx.z) / (unsigned)a.parts);
  }
  const int q0 = q_tile * BQ;
  if (q0 >= qlen) return;
  const int kv_all = min(len, q0 + BQ + off);  // causal: keys beyond the tile's last query are never needed
  int kv_begin = 0, kv_end = kv_all;
  bool several = false;                        // this tile's keys are in more than one part
  if constexpr (PARTS) {
    const int n_tiles = (kv_all + BKV - 1) / BKV, per_part = tiles_per_part(n_tiles, a.parts, a.part_tiles);
    if (part >= (n_tiles + per_part - 1) / per_part) return;
    several = per_part < n_tiles;
    kv_begin = part * per_part * BKV;
    kv_end = min(kv_all, kv_begin + per_part * BKV);
  }
  const int tid = threadIdx.x & (kThreads - 1), wave = tid >> 6, lane = tid & 63;
  const int qcol = lane & 15, quad = lane >> 4;
  int my_q[QT];                                 // query index inside the sequence's new tokens (may be >= qlen)
#pragma unroll
  for (int u = 0; u < QT; ++u) my_q[u] = q0 + wave * (16 * QT) + 16 * u + qcol;

  // Q^T fragments: B operand, lane = (query, 8 consecutive d of each 32-wide k-step)
  u32x4 qf[QT][KS];
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    const char* qp = a.q + (int64_t)(s0 + min(my_q[u], qlen - 1)) * a.q_stride_b + (int64_t)head * D * 2;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[u][s] = *(const u32x4*)(qp + (32 * s + 8 * quad) * 2);
  }

  float4v o[QT][DT];
#pragma unroll
  for (int u = 0; u < QT; ++u)
#pragma unroll
    for (int t = 0; t < DT; ++t) o[u][t] = float4v{0.f, 0.f, 0.f, 0.f};
  float m_run[QT], l_run[QT];
#pragma unroll
  for (int u = 0; u < QT; ++u) { m_run[u] = -INFINITY; l_run[u] = 0.f; }

  // Copies.  A wave-wide copy moves RPC = 64 / KCH key rows; wavefront w makes copies w, w + 4, ... of K's and of V's, so
  // that a lane always moves the same row of a group of 16 keys (and has one swizzle), and the group is wave-uniform.
  // A lane keeps its offset inside a tile; the tile's (kPacked) or the group's (kPaged16) start is scalar work.  (Key by key,
  // every lane makes its addresses; the block numbers are loaded a tile ahead too.  Blocks of 48: 4 sequences, 200 tokens on 4000
  // cached, of 40 x 128 heads 57.6 -> 48.5 us against copies through the builtin, 8 sequences, 8000 on 8000 564 -> 533.)  (Every
  // lane multiplying out 64-bit offsets of twelve rows a tile, 130 quarter-rate multiplications with the divisions of a
  // block table, cost as much as the softmax: 274 against 251 us for 4 x 2048 tokens.)
  constexpr int RPC = 64 / KCH, PER = BKV / RPC / 4;   // key rows of a copy; copies per wavefront and operand
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int key0 = RPC * wave + lane / KCH;            // this lane's key in its wavefront's first copy; + 4 RPC each
  const int slot = lane % KCH;
  const char* k_base = a.k + (PAGED ? 0 : (int64_t)s0 * a.k_stride_b) + (int64_t)head * D * 2;
  const char* v_base = a.v + (PAGED ? 0 : (int64_t)s0 * a.v_stride_b) + (int64_t)head * D * 2;
  // (constant address space: scalar loads, which do not share a counter with the copies)
  const auto table = (const __attribute__((address_space(4))) int32_t*)(PAGED ? a.block_tables + (int64_t)seq * a.table_stride
                                                                              : a.cu_seqlens);
  auto block_start = [&](int blk) -> int64_t {   // a bad table: wrong numbers, no fault
    const int64_t b = blk < 0 ? 0 : (blk >= a.num_blocks ? a.num_blocks - 1 : (int64_t)blk);
    return b * a.block_stride_b;
  };
  // kPaged16: the blocks of the wavefront's groups of the next tile to be copied (past the sequence: its last group).
  // kPagedAny: those of the lane's keys, and their places in them (past the sequence: its last key).
  const int last_group = (len - 1) >> 4;
  auto group_of = [&](int kv0, int j) { return min((kv0 >> 4) + (KCH == 16 ? j : (wave_u >> 1) + 2 * j), last_group); };
  auto key_of = [&](int kv0, int j) { return min(kv0 + key0 + j * 4 * RPC, len - 1); };
  int blocks[PER], in_block[PER];
  auto load_blocks = [&](int kv0) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if constexpr (SRC == kPaged16) blocks[j] = table[group_of(kv0, j) >> a.groups_shift];
      if constexpr (SRC == kPagedAny) {
        const int bi = key_of(kv0, j) / a.block_size;
        blocks[j] = a.block_tables[(int64_t)seq * a.table_stride + bi];
        in_block[j] = key_of(kv0, j) - bi * a.block_size;
      }
    }
  };
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int row_in = SRC == kPaged16 ? key0 & 15 : key0;
  const uint32_t k_lane = (uint32_t)row_in * (uint32_t)a.k_stride_b + (slot ^ k_swz(key0)) * 16;
  const uint32_t v_lane = (uint32_t)row_in * (uint32_t)a.v_stride_b + (slot ^ v_swz(key0)) * 16;
  auto copy_tile = [&](int kv0, int stage) {
    const uint32_t dst = lds_base + stage * kStage + wave_u * 1024;   // copy i of an operand: bytes [1024 i, 1024 i + 1024)
    if constexpr (SRC == kPacked) {   // rows past the sequence read as zeros; the mask removes their scores
      const uint32_t last = (uint32_t)min(BKV - 1, len - kv0 - 1);
      const ScalarRsrc rk = scalar_rsrc(k_base, kv0 * a.k_stride_b, last * (uint32_t)a.k_stride_b, D * 2);
      const ScalarRsrc rv = scalar_rsrc(v_base, kv0 * a.v_stride_b, last * (uint32_t)a.v_stride_b, D * 2);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        copy_to_lds(dst + j * 4096, rk, k_lane, j * 4 * RPC * (uint32_t)a.k_stride_b);
        copy_to_lds(dst + kTile + j * 4096, rv, v_lane, j * 4 * RPC * (uint32_t)a.v_stride_b);
      }
    } else if constexpr (SRC == kPaged16) {
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int g = group_of(kv0, j);
        const int64_t start =
            block_start(blocks[j]) + (int64_t)((g & ((1 << a.groups_shift) - 1)) * 16) * a.k_stride_b;
        // what a block holds past its sequence may be anything, and a zero probability does not cancel a NaN: the buffer
        // ends with the sequence's last row and the others read as zeros
        const uint32_t last = (uint32_t)min(15, len - 1 - 16 * g) * (uint32_t)a.k_stride_b;
        copy_to_lds(dst + j * 4096, scalar_rsrc(k_base, start, last, D * 2), k_lane, 0);
        copy_to_lds(dst + kTile + j * 4096, scalar_rsrc(v_base, start, last, D * 2), v_lane, 0);
      }
      load_blocks(kv0 + BKV);
    } else {
      if constexpr (PAGED) {   // the block numbers have arrived before the first copy is counted
#pragma unroll
        for (int j = 0; j < PER; ++j) asm volatile("" : "+v"(blocks[j]));
      }
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        int64_t k_off, v_off;
        if constexpr (PAGED) {
          k_off = block_start(blocks[j]) + (int64_t)in_block[j] * a.k_stride_b;
          v_off = k_off;   // (both caches have the same strides)
        } else {
          k_off = (int64_t)key_of(kv0, j) * a.k_stride_b;
          v_off = (int64_t)key_of(kv0, j) * a.v_stride_b;
        }
        copy_lanes_to_lds(dst + j * 4096, k_base + k_off + (slot ^ k_swz(key0)) * 16);
        copy_lanes_to_lds(dst + kTile + j * 4096, v_base + v_off + (slot ^ v_swz(key0)) * 16);
      }
      load_blocks(kv0 + BKV);
    }
  };
  // V^T fragment (16 d of tile t, keys of this lane's quad in key tile kt): the lane gives the address of its share of the
  // 4 x 16 block, key i / 4 and d 4 (i % 4) for i = lane % 16, and receives d = i of the four keys
  const int v_key = 4 * quad + (qcol >> 2);
  const uint32_t v_frag = (uint32_t)(kTile + v_key * KROW + (qcol & 1) * 8);
  const int v_piece = (qcol & 3) >> 1;
  auto read_v = [&](int stage, int kt, int t) -> uint2 {
    typedef short short4v __attribute__((ext_vector_type(4)));
    const uint32_t at = v_frag + stage * kStage + kt * 16 * KROW + (((2 * t + v_piece) ^ v_swz(v_key)) << 4);
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                         (__attribute__((address_space(3))) short4v*)(lds + at)));
  };

  const int wave_q0 = q0 + wave * (16 * QT) + off;    // last key the first query of this wavefront sees
  load_blocks(kv_begin);
#pragma unroll
  for (int u = 0; u < QT; ++u)   // the queries have arrived before the first copy is counted
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[u][s]));
  copy_tile(kv_begin, 0);
  for (int kv0 = kv_begin, stage = 0; kv0 < kv_end; kv0 += BKV, stage ^= 1) {
    APS_WAIT_LGKM0();  // no fragment read of the previous tile is under way,
    APS_WAIT_VM(0);    // and this wavefront's copies of this tile have landed: past the barrier everyone's
    APS_BARRIER();
    if (kv0 + BKV < kv_end) copy_tile(kv0 + BKV, stage ^ 1);  // in flight while this tile is multiplied
    if (kv0 > wave_q0 + 16 * QT - 1) continue;                         // every key of the tile lies after this wavefront's queries
    const char* const k_lds = lds + stage * kStage;

    // ---- S^T = K Q^T: a K fragment serves both query tiles
    float4v st[QT][KT];
#pragma unroll
    for (int u = 0; u < QT; ++u)
#pragma unroll
      for (int t = 0; t < KT; ++t) st[u][t] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const int key = t * 16 + qcol, ch = 4 * s + quad;  // A operand row of this lane
        const u32x4 kf = *(const u32x4*)(k_lds + key * KROW + ((ch ^ k_swz(key)) * 16));
#pragma unroll
        for (int u = 0; u < QT; ++u) st[u][t] = mfma16<BF16>(kf, qf[u][s], st[u][t]);
      }
    // ---- online softmax for this lane's two queries (16 keys of each here, the others in lanes 16, 32, 48 apart)
    // Only a tile that reaches past the wavefront's first query or past the sequence needs the mask.
    // The maximum is taken on the raw scores (the scale is positive) and the scale goes into the exponent's
    // fused multiply-add: max, fma, exp2 and add per score, nothing else.
    const bool masked = kv0 + BKV - 1 > wave_q0 || kv0 + BKV > len;
    if (masked) {
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        const int last = min(my_q[u] + off, len - 1) - kv0 - 4 * quad;   // the last key of this lane's that is seen
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (16 * t + e > last) st[u][t][e] = -INFINITY;
      }
    }
    float mx[QT], m_use[QT], neg_m[QT];
    bool moved = false;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
      mx[u] = m_run[u];   // raw-score domain
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) mx[u] = fmaxf(mx[u], st[u][t][e]);
      // the other keys of this query: exchanges between the 16-lane rows of the wavefront, no LDS
      const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx[u]), __float_as_uint(mx[u]), false, false);
      mx[u] = fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1]));
      const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx[u]), __float_as_uint(mx[u]), false, false);
      mx[u] = fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
      m_use[u] = (mx[u] == -INFINITY) ? 0.f : mx[u];
      neg_m[u] = -m_use[u] * a.scale_log2;
      moved |= mx[u] != m_run[u];
    }
    // the running maximum rarely moves after the first tiles: rescale O only when some query of the wavefront
    // needs it (a wave-uniform branch)
    if (__builtin_amdgcn_ballot_w64(moved) != 0) {
#pragma unroll
      for (int u = 0; u < QT; ++u) {
        const float alpha = __builtin_amdgcn_exp2f((m_run[u] - m_use[u]) * a.scale_log2);
        l_run[u] *= alpha;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[u][t] *= alpha;
        m_run[u] = mx[u];
      }
    }
    // ---- O^T += V^T P^T : two k-steps of 32 keys; P^T fragment = the results of two neighbouring key tiles, a V^T
    // fragment serves both query tiles
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      u32x4 pf[QT];
#pragma unroll
      for (int u = 0; u < QT; ++u) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          float4v& p = st[u][2 * w + t];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            p[e] = __builtin_amdgcn_exp2f(fmaf(p[e], a.scale_log2, neg_m[u]));
            l_run[u] += p[e];   // (this lane's keys; the lanes of a query are added at the end)
          }
          pf[u][2 * t] = pack2<BF16>(p[0], p[1]);
          pf[u][2 * t + 1] = pack2<BF16>(p[2], p[3]);
        }
      }
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const uint2 v0 = read_v(stage, 2 * w, t), v1 = read_v(stage, 2 * w + 1, t);
        const u32x4 vf = {v0.x, v0.y, v1.x, v1.y};
#pragma unroll
        for (int u = 0; u < QT; ++u) o[u][t] = mfma16<BF16>(vf, pf[u], o[u][t]);
      }
    }
  }

  // ---- one of several key parts: sums as they are
  if (PARTS && several) {
    static_assert(!PARTS || BQ == kPartQueries, "units are laid out for one query tile a wavefront");
    float* const unit = a.partial + (first_unit(s0, seq, q_tile, a.num_heads, head, a.parts) + part) * unit_floats<D>();
    float* const ml = unit + BQ * D + wave * (16 * QT) + qcol;
#pragma unroll
    for (int u = 0; u < QT; ++u) {
#pragma unroll
      for (int t = 0; t < DT; ++t) ((float4v*)unit)[(u * DT + t) * kThreads + tid] = o[u][t];
      float l = l_run[u];
      l += __shfl_xor(l, 16);
      l += __shfl_xor(l, 32);
      if (quad == 0) { ml[16 * u] = m_run[u]; ml[BQ + 16 * u] = l; }
    }
    return;
  }
  // ---- normalise and store: lane owns queries my_q, rows d = 16 t + 4 quad + e
#pragma unroll
  for (int u = 0; u < QT; ++u) {
    float l = l_run[u];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (my_q[u] >= qlen) continue;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    char* op = a.out + (int64_t)(s0 + my_q[u]) * a.out_stride_b + (int64_t)head * D * 2 + quad * 8;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      uint2 w;
      w.x = pack2<BF16>(o[u][t][0] * inv, o[u][t][1] * inv);
      w.y = pack2<BF16>(o[u][t][2] * inv, o[u][t][3] * inv);
      *(uint2*)(op + t * 32) = w;
    }
  }
}

// out = sum of the key parts of a query tile, each weighted with exp2 of its maximum against the largest, over the sum of
// their weights: the same sums in fp32, rounded once.  Same grid (without the parts) and same lanes as the kernel above, so
// that units are written and read 1 KiB a wavefront.
template <bool BF16, int D>
__global__ __launch_bounds__(kThreads) void prefill_combine_kernel(const PrefillArgs a) {
  constexpr int BQ = kPartQueries, DT = D / 16;
  const int seq = blockIdx.y, head = blockIdx.x, q_tile = blockIdx.z, q0 = q_tile * BQ;
  const int s0 = a.cu_seqlens[seq], s1 = a.cu_seqlens[seq + 1];
  if (s0 < 0 || s1 < s0 || s1 > a.num_tokens) return;
  const int qlen = s1 - s0;
  const int len = a.cu_seqlens_k[seq + 1] - a.cu_seqlens_k[seq];
  if (len < qlen || (int64_t)(len + a.block_size - 1) / a.block_size > a.table_width || q0 >= qlen) return;
  const int n_tiles = (min(len, q0 + BQ + len - qlen) + BKV - 1) / BKV;
  const int per_part = tiles_per_part(n_tiles, a.parts, a.part_tiles), parts = (n_tiles + per_part - 1) / per_part;
  if (parts == 1) return;   // stored by its workgroup
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, qcol = lane & 15, quad = lane >> 4;
  const float* const units = a.partial + first_unit(s0, seq, q_tile, a.num_heads, head, a.parts) * unit_floats<D>();
  const int row = wave * 16 + qcol;
  float m = -INFINITY;
  for (int p = 0; p < parts; ++p) m = fmaxf(m, units[p * unit_floats<D>() + BQ * D + row]);
  const float m_use = m == -INFINITY ? 0.f : m;
  float4v o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = float4v{0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
  for (int p = 0; p < parts; ++p) {
    const float* const unit = units + p * unit_floats<D>();
    const float w = __builtin_amdgcn_exp2f((unit[BQ * D + row] - m_use) * a.scale_log2);
    l += w * unit[BQ * D + BQ + row];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const float4v v = ((const float4v*)unit)[t * kThreads + tid];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[t][e] = fmaf(w, v[e], o[t][e]);
    }
  }
  if (q0 + row >= qlen) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  char* op = a.out + (int64_t)(s0 + q0 + row) * a.out_stride_b + (int64_t)head * D * 2 + quad * 8;
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    uint2 w;
    w.x = pack2<BF16>(o[t][0] * inv, o[t][1] * inv);
    w.y = pack2<BF16>(o[t][2] * inv, o[t][3] * inv);
    *(uint2*)(op + t * 32) = w;
  }
}

}  // namespace
}  // namespace aps

using namespace aps;

namespace {
// Few workgroups: 64 queries each instead of 128.  A workgroup's time is its key tiles one after the other, 2.0 us each
// with 32 queries a wavefront and 1.5 with 16, so as long as the CUs are not full the shorter ones finish first (12
// heads, 2048 tokens: 34 -> 26 us; 40 heads, 361 tokens 11.1 -> 9.9, 4 x 50 on a prefix of 4000 61 -> 49); full CUs
// lose by reading every fragment for half the queries (40 heads, 1400 tokens 26 -> 28, 4 x 2048 243 -> 312).  The count
// looks at queries alone (16 chunks, 1000 new on 8000 cached tokens, 40 heads: 91 us, 89 with 64).
// (A longest sequence stated far beyond the tokens, within the grid's limit at 128 queries only, is taken at 128.)
int query_tiles(int64_t num_seqs, int64_t num_tokens, int64_t max_seqlen_q, int num_heads) {
  return num_heads * (num_tokens / 128 + num_seqs) <= 384 && max_seqlen_q <= 65535 * 64 ? 1 : 2;
}
// Key parts of a step on cached prefixes.  Few new tokens on a long prefix leave CUs idle while each workgroup walks its key
// tiles: the tiles are dealt over as many workgroups as 512 places (two a CU) take, the longest sequence's at least 8 tiles each;
// those of a shorter one, which tiles_per_part evens out, may hold 5 (9 tiles in parts of 8).  Writing and adding the parts
// takes about as long as five tiles (40 x 128 heads, 51 tokens, 16 tiles 25.5, in parts of 8 20.5), and the second launch 4 us of
// the host (12 x 64 heads, 26 tokens on 1000 cached 20, in two parts 23.5).
// Measured (us; 1 part, then as planned): 40 x 128 heads, 1 sequence, 64 tokens on 8000 cached 167, 49; 128 on 1900 49, 29.5; 4
// sequences, 64 on 4000 46, 30; 12 x 64 heads, 64 on 8000 100, 24; 8 sequences, 400 on 8000 36, 24; 4, 1000 on 4000 35, 27.
// Parts lose where workgroups are many already: beyond 512 places they stand in a second round, beyond 256 two share a CU.  How
// many there are without parts is known only from above (`groups`: each sequence may end with a partly filled tile, and none
// has more tiles than the longest), and that other sequences are shorter than the longest, which leaves places to its parts,
// is not known at all.  So the line lies where no batch measured loses, even lengths being the worst (1127 steps of 1 to 16
// sequences, 1 to 600 new tokens on up to 6000 cached, 12 to 64 heads: 433 in parts, 3 % to 4 times faster than in one; where
// only likely groups were counted, and no line drawn, 35 were 4 to 25 % slower).  Even lengths, us, at 128 wide, groups / key
// tiles: 96 / 16 26.8, 25.6; 144 / 16 27.4, 29.4; 120 / 20 32.3, 28.8; 160 / 20 34.3, 34.6; 160 / 24 37.6, 36.0; 216 / 24 37.4, 36.1;
// 240 / 24 39.1, 43.2; 240 / 64 110.9, 110.1; 280 / 18 36.7, 47.8.  64 wide: 256 / 24 25.8, 26.2; 256 / 32 31.9, 31.5; 320 / 24 29.4,
// 34.9.  Uneven ones would gain beyond it (40 x 128, 8 sequences, 64 on 8000 60, 45).  Full places lose in any case: 6 sequences,
// 2048 on 4200 99, in parts of 8 tiles 119; prompts without a prefix (1 x 1500 44, in two parts 52).
// (`likely` counts half a tile per sequence; more parts than it allows were not measured.)
struct KeyParts { int parts, part_tiles; int64_t bytes; };
KeyParts key_parts(int64_t num_seqs, int64_t num_tokens, int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads,
                   int head_size) {
  constexpr KeyParts kOne{1, INT32_MAX / 2, 0};
  if (64 * query_tiles(num_seqs, num_tokens, max_seqlen_q, num_heads) != kPartQueries) return kOne;
  const int64_t q_tiles = (max_seqlen_q + kPartQueries - 1) / kPartQueries, tiles = (max_seqlen_k + BKV - 1) / BKV;
  const int64_t most_tiles = num_tokens / kPartQueries + num_seqs;   // in all sequences
  const int64_t groups = std::min(most_tiles, num_seqs * q_tiles) * num_heads;
  const int64_t likely = (2 * num_tokens / kPartQueries + num_seqs) * num_heads / 2;
  const int64_t from = head_size == 64 ? (groups <= 192 ? 24 : 32)   // (beyond 256 groups there are no two parts)
                                       : groups <= 96 ? 16 : groups <= 128 ? 20 : groups <= 216 ? 24 : 64;
  const int64_t parts = std::min<int64_t>(512 / std::max<int64_t>({groups, likely, 1}), tiles / 8);
  if (parts < 2 || tiles < from || q_tiles * parts > 65535) return kOne;
  const int part_tiles = (int)std::min<int64_t>((tiles + parts - 1) / parts, INT32_MAX / 2);
  return KeyParts{(int)parts, part_tiles,
                  most_tiles * num_heads * parts * (head_size == 64 ? unit_floats<64>() : unit_floats<128>()) * 4};
}

int launch_prefill(PrefillArgs& a, bool paged, int64_t num_seqs, int64_t max_seqlen_q, int64_t max_seqlen_k, int num_heads,
                   int head_size, int dtype, void* workspace, int64_t workspace_bytes, aps_stream_t stream) {
  const int qt = query_tiles(num_seqs, a.num_tokens, max_seqlen_q, num_heads);
  const int64_t q_tiles = (max_seqlen_q + 64 * qt - 1) / (64 * qt);
  if (q_tiles > 65535 || num_seqs > 65535 || num_heads > 65535) return APS_ERR_UNSUPPORTED;
  a.parts = 1; a.part_tiles = INT32_MAX / 2;
  if (paged && workspace && max_seqlen_k > 0) {
    const KeyParts kp = key_parts(num_seqs, a.num_tokens, max_seqlen_q, max_seqlen_k, num_heads, head_size);
    if (workspace_bytes < kp.bytes || (addr(workspace) & 15)) return APS_ERR_WORKSPACE;
    a.parts = kp.parts; a.part_tiles = kp.part_tiles; a.partial = (float*)workspace;
  }
  const dim3 grid((unsigned)num_heads, (unsigned)num_seqs, (unsigned)(q_tiles * a.parts));
  hipStream_t s = (hipStream_t)stream;
  // 64 rows within 32-bit offsets; 16 << shift tokens a block and a row pitch that a 24-bit product takes
  int src = paged ? kPagedAny : kPackedAny;
  if (!paged && std::max(a.k_stride_b, a.v_stride_b) < (1 << 25)) src = kPacked;
  if (paged && a.block_size >= 16 && (a.block_size & (a.block_size - 1)) == 0 && a.v_stride_b < (1 << 24)) {
    src = kPaged16;
    a.groups_shift = __builtin_ctz((unsigned)a.block_size) - 4;
  }
#define APS_LAUNCH_PF_Q(B, D_, P, Q_)                                                                                 \
  do {                                                                                                                \
    constexpr bool kMayPart = (P == kPaged16 || P == kPagedAny) && 64 * Q_ == kPartQueries;                           \
    if (kMayPart && a.parts > 1)                                                                                      \
      APS_LAUNCH((prefill_attention_kernel<B, D_, P, Q_, kMayPart>), grid, dim3(kThreads), prefill_lds_bytes<D_>(), s, a); \
    else                                                                                                              \
      APS_LAUNCH((prefill_attention_kernel<B, D_, P, Q_, false>), grid, dim3(kThreads), prefill_lds_bytes<D_>(), s, a);   \
  } while (0)
#define APS_LAUNCH_PF(B, D_, P) do { if (qt == 2) APS_LAUNCH_PF_Q(B, D_, P, 2); else APS_LAUNCH_PF_Q(B, D_, P, 1); } while (0)
#define APS_LAUNCH_PF_D(B, P) do { if (head_size == 64) APS_LAUNCH_PF(B, 64, P); else APS_LAUNCH_PF(B, 128, P); } while (0)
#define APS_LAUNCH_PF_S(P) do { if (dtype == APS_F16) APS_LAUNCH_PF_D(false, P); else APS_LAUNCH_PF_D(true, P); } while (0)
  if (src == kPacked) APS_LAUNCH_PF_S(kPacked);
  else if (src == kPaged16) APS_LAUNCH_PF_S(kPaged16);
  else if (src == kPackedAny) APS_LAUNCH_PF_S(kPackedAny);
  else APS_LAUNCH_PF_S(kPagedAny);
#undef APS_LAUNCH_PF_S
#undef APS_LAUNCH_PF_D
#undef APS_LAUNCH_PF
#undef APS_LAUNCH_PF_Q
  const int st = launch_status();
  if (st != APS_OK || a.parts == 1) return st;
  const dim3 cgrid((unsigned)num_heads, (unsigned)num_seqs, (unsigned)q_tiles);
#define APS_LAUNCH_PC(B, D_) APS_LAUNCH((prefill_combine_kernel<B, D_>), cgrid, dim3(kThreads), 0, s, a)
#define APS_LAUNCH_PC_D(B) do { if (head_size == 64) APS_LAUNCH_PC(B, 64); else APS_LAUNCH_PC(B, 128); } while (0)
  if (dtype == APS_F16) APS_LAUNCH_PC_D(false); else APS_LAUNCH_PC_D(true);
#undef APS_LAUNCH_PC_D
#undef APS_LAUNCH_PC
  return launch_status();
}
}  // namespace

extern "C" {

int64_t aps_paged_prefill_attention_workspace_bytes(int64_t num_seqs, int64_t num_q_tokens, int64_t max_seqlen_q,
                                                    int64_t max_seqlen_k, int num_heads, int head_size) {
  if (num_seqs <= 0 || num_q_tokens <= 0 || max_seqlen_q <= 0 || max_seqlen_k <= 0 || num_heads <= 0 || num_heads > 65535 ||
      (head_size != 64 && head_size != 128))
    return 0;
  return key_parts(num_seqs, num_q_tokens, max_seqlen_q, max_seqlen_k, num_heads, head_size).bytes;
}

int aps_varlen_prefill_attention(void* out, const void* q, const void* k, const void* v, const int32_t* cu_seqlens,
                                 int64_t num_seqs, int64_t num_tokens, int64_t max_seqlen, int num_heads,
                                 int head_size, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t out_stride,
                                 float softmax_scale, int dtype, aps_stream_t stream) {
  if (num_seqs < 0 || num_tokens < 0 || max_seqlen < 0 || num_heads <= 0 || head_size <= 0) return APS_ERR_INVALID_ARG;
  // the running maximum is taken on raw scores and the scale folded into the exponent: a positive, finite scale only
  if (!(softmax_scale > 0.f) || softmax_scale > 3.0e38f) return APS_ERR_INVALID_ARG;
  if (num_seqs == 0 || num_tokens == 0 || max_seqlen == 0) return APS_OK;
  if (!out || !q || !k || !v || !cu_seqlens) return APS_ERR_INVALID_ARG;
  if (dtype != APS_F16 && dtype != APS_BF16) return APS_ERR_UNSUPPORTED;
  if (head_size != 64 && head_size != 128) return APS_ERR_UNSUPPORTED;
  const int64_t row = (int64_t)num_heads * head_size;
  if (q_stride < row || k_stride < row || v_stride < row || out_stride < row) return APS_ERR_INVALID_ARG;
  if (common_vec_bytes({addr(q), addr(k), addr(v), (uint64_t)q_stride * 2, (uint64_t)k_stride * 2,
                        (uint64_t)v_stride * 2}) != 16 ||
      common_vec_bytes({addr(out), (uint64_t)out_stride * 2}) < 8)
    return APS_ERR_UNSUPPORTED;
  PrefillArgs a{};
  a.q = (const char*)q; a.k = (const char*)k; a.v = (const char*)v; a.out = (char*)out;
  a.cu_seqlens = cu_seqlens;
  a.q_stride_b = q_stride * 2; a.k_stride_b = k_stride * 2; a.v_stride_b = v_stride * 2; a.out_stride_b = out_stride * 2;
  a.num_heads = num_heads;
  a.num_tokens = num_tokens;
  a.scale_log2 = softmax_scale * kLog2e;
  return launch_prefill(a, false, num_seqs, max_seqlen, max_seqlen, num_heads, head_size, dtype, nullptr, 0, stream);
}

int aps_paged_prefill_attention_split(void* out, const void* q, const void* k_cache, const void* v_cache,
                                const int32_t* block_tables, const int32_t* cu_seqlens_q,
                                const int32_t* cu_seqlens_k, int64_t num_seqs, int64_t num_q_tokens,
                                int64_t max_seqlen_q, int num_heads, int head_size, int block_size,
                                int64_t table_stride, int64_t table_width, int64_t q_stride, int64_t out_stride,
                                int64_t cache_block_stride, int64_t num_cache_blocks, float softmax_scale, int dtype,
                                int64_t max_seqlen_k, void* workspace, int64_t workspace_bytes, aps_stream_t stream) {
  if (num_seqs < 0 || num_q_tokens < 0 || max_seqlen_q < 0 || num_heads <= 0 || head_size <= 0 || block_size <= 0 ||
      table_width < 0 || num_cache_blocks < 0)
    return APS_ERR_INVALID_ARG;
  if (!(softmax_scale > 0.f) || softmax_scale > 3.0e38f) return APS_ERR_INVALID_ARG;
  if (num_seqs == 0 || num_q_tokens == 0 || max_seqlen_q == 0) return APS_OK;
  if (!out || !q || !k_cache || !v_cache || !block_tables || !cu_seqlens_q || !cu_seqlens_k || num_cache_blocks == 0)
    return APS_ERR_INVALID_ARG;
  if (dtype != APS_F16 && dtype != APS_BF16) return APS_ERR_UNSUPPORTED;
  if (head_size != 64 && head_size != 128) return APS_ERR_UNSUPPORTED;
  const int64_t row = (int64_t)num_heads * head_size;
  if (q_stride < row || out_stride < row || cache_block_stride < row * block_size || table_stride < table_width)
    return APS_ERR_INVALID_ARG;
  if (common_vec_bytes({addr(q), addr(k_cache), addr(v_cache), (uint64_t)q_stride * 2,
                        (uint64_t)cache_block_stride * 2}) != 16 ||
      common_vec_bytes({addr(out), (uint64_t)out_stride * 2}) < 8)
    return APS_ERR_UNSUPPORTED;
  PrefillArgs a{};
  a.q = (const char*)q; a.k = (const char*)k_cache; a.v = (const char*)v_cache; a.out = (char*)out;
  a.cu_seqlens = cu_seqlens_q; a.cu_seqlens_k = cu_seqlens_k; a.block_tables = block_tables;
  a.q_stride_b = q_stride * 2; a.k_stride_b = row * 2; a.v_stride_b = row * 2; a.out_stride_b = out_stride * 2;
  a.table_stride = table_stride; a.table_width = table_width;
  a.block_stride_b = cache_block_stride * 2; a.num_blocks = num_cache_blocks; a.block_size = block_size;
  a.num_heads = num_heads;
  a.num_tokens = num_q_tokens;
  a.scale_log2 = softmax_scale * kLog2e;
  return launch_prefill(a, true, num_seqs, max_seqlen_q, max_seqlen_k, num_heads, head_size, dtype, workspace, workspace_bytes,
                        stream);
}

int aps_paged_prefill_attention(void* out, const void* q, const void* k_cache, const void* v_cache,
                                const int32_t* block_tables, const int32_t* cu_seqlens_q,
                                const int32_t* cu_seqlens_k, int64_t num_seqs, int64_t num_q_tokens,
                                int64_t max_seqlen_q, int num_heads, int head_size, int block_size,
                                int64_t table_stride, int64_t table_width, int64_t q_stride, int64_t out_stride,
                                int64_t cache_block_stride, int64_t num_cache_blocks, float softmax_scale, int dtype,
                                aps_stream_t stream) {
  return aps_paged_prefill_attention_split(out, q, k_cache, v_cache, block_tables, cu_seqlens_q, cu_seqlens_k, num_seqs,
                                           num_q_tokens, max_seqlen_q, num_heads, head_size, block_size, table_stride,
                                           table_width, q_stride, out_stride, cache_block_stride, num_cache_blocks,
                                           softmax_scale, dtype, 0, nullptr, 0, stream);
}

}  // extern "C"
