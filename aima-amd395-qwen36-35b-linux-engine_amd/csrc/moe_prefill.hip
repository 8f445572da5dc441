// MoE block of the Qwen3.6-35B-A3B layer for a batch of T tokens (prefill).
//
// Replaces the reference's native MoE prefill (native/src/
// native_moe_prefill.hip.cpp: router GEMM + router_topk8_softmax_256_kernel
// :234-323, moe_align_block32_256_kernel :325-382, the two AOT vLLM
// fused_moe_kernel expert GEMMs with expert_silu_multiply_kernel :384-402
// between them, the shared-expert GEMMs and pointwise kernels :210-232,
// moe_sum8_kernel :404-430 and the residual add), with the arithmetic of
// the eager text four_layer_mini_engine.py:8479-8650 (router :7775-7789,
// routed experts :7791-7803, shared expert :8240-8300) -- the same formulas
// as the one-token qwen36_moe_decode:
//   after = bf16(inp + attn);  h2 = bf16(rmsnorm(after) * (w + 1))
//   logits = bf16(h2 @ router^T);  ids = top-8;  rw = bf16(softmax(top-8))
//   [gate | up] = bf16(h2 @ gate_up_e^T);  act = bf16(silu(gate) * up)
//   y_k = bf16(bf16(act @ down_e^T) * rw_k)
//   shared: same expert form with the shared weights, scaled by
//           bf16(sigmoid(bf16(h2 . shared_gate)))
//   out = bf16(after + bf16(bf16(sum_k y_k) + shared))
//
// Launches (T tokens, E experts; the shared expert is one more group of the
// expert GEMMs, with every token):
//  1. moe_pre_kernel       residual + RMSNorm, one wave per token.
//  2. moe_router_gemm      logits [T, E + 1] = h2 [router | shared_gate]^T;
//                          up to 8192 tokens in K slices whose fp32
//                          partials 3 sums.
//  3. moe_topk_kernel      top-8 + routing softmax + shared gate, a wave per token.
//  4. alignment            (token, rank) slots sorted by expert, each group
//                          padded to 32 rows and cut evenly into tiles of up
//                          to 64 (short prompts) or 256 rows: one workgroup
//                          up to 2048 tokens (moe_align_one), else per-chunk
//                          histograms, one scan workgroup and a per-chunk
//                          scatter.
//  5. gate/up              act [tile rows, 512] = silu(gate) * up per tile.
//  6. down                 y rows, scattered to their (token, rank) slot
//                          (5, 6: moe_stream.h up to 2048 tokens, moe_tile.h
//                          above).
//  7. moe_combine_kernel   per token: sum of the 8 weighted routed rows, + the
//                          shared row scaled by its gate, + after.
//
// Router GEMM: a workgroup computes 128 tokens against 256 router rows, K in
// steps of 32, with 8 waves of 64 x 64 on v_mfma_f32_32x32x16_bf16; 32-row
// blocks past the last token are neither computed nor fetched.  Both operands
// are K-contiguous in memory, so they are fetched straight into LDS
// (buffer_load ... lds, 16 bytes per lane, 1 KiB per instruction) with an XOR
// swizzle of the 16-byte chunks chosen by each lane's source address, which
// makes the ds_read_b128 operand reads bank-conflict-free.  A 3-stage ring,
// two workgroups per CU; the fetch is issued through inline asm (the
// compiler would otherwise wait for it before reading the current stage) and
// ordered by explicit vmcnt waits + barriers.
#include "moe_common.h"
#include "moe_stream.h"
#include "moe_tile.h"

#include <algorithm>
#include <mutex>

namespace q36 {
namespace {

constexpr int kPfPad = 32;                // group padding (rows)
// Router GEMM tile.
constexpr int kRtBM = 128, kRtBN = 256;   // tokens, router rows per workgroup
constexpr int kRtStages = 3;              // fetch ring depth
constexpr int kRtBK = 32;                 // K per stage
constexpr int kRtRowB = kRtBK * 2;        // bytes per row per stage
constexpr int kRtCpr = kRtRowB / 16;      // 16-byte chunks per row
constexpr int kRtRpi = 1024 / kRtRowB;    // rows per fetch instruction
constexpr int kRtRpw = 256 / kRtRowB;     // rows per 256-byte bank window
constexpr int kRtStage = (kRtBM + kRtBN) * kRtRowB;
constexpr int kRtLds = kRtStages * kRtStage;
constexpr int kRtWaves = 8;               // 2 x 4, each 64 tokens x 64 rows
constexpr int kRtInstr = kRtStage / 1024 / kRtWaves;   // fetch instructions per wave
// Swizzle: chunk c of stage row r sits at position c ^ key(r), key(r) =
// (r / kRtRpw) % kRtCpr, so the 16 rows one ds_read_b128 pass serves fall in
// 16 distinct 16-byte bank groups of the 256-byte bank window.
constexpr unsigned kPfMaxTokens = 262144;
constexpr unsigned kAlignChunk = 4096;    // expert ids per histogram / scatter workgroup (least)
constexpr unsigned kMaxAlignChunks = 256;
// Up to this many tokens the expert GEMMs are the streaming kernels of
// moe_stream.h (tiles of up to 64 rows) and the shared expert is one more
// group of them: MI355X, whole block, against 128-row tiles and a side stream
// at every length: T = 5 69 us against 110, 45 219 / 263, 300 309 / 350, 1000
// 337 / 411, 1400 372 / 452, 2048 462 / 477.  Longer prompts take the 256-row
// tiles of moe_tile.h (2100: 420 us against 476; one workgroup per CU and
// whole weights per tile pay from about 128 rows a group).
constexpr unsigned kStreamMaxTokens = 2048;

// Workspace layout for (T, E); every region 256-byte aligned.  The first
// three regions (expert ids, routing weights, router logits) are read back by
// the host's debug path at these fixed offsets.
struct PfLayout {
  size_t ids, rw, logits, sgw, meta, sorted, hist, after, h2, act, y, part, total;
  unsigned ld_logits, max_tiles, max_rows, n_chunks, chunk_ids, router_splits;
};

// K slices of the router GEMM: its T / 128 x 2 tiles leave most CUs idle
// at short prompts, each tile a chain of 64 K steps, so up to 8192 tokens
// the K range is cut into slices whose fp32 partials the top-8 kernel sums
// (MI355X, whole block: T = 1024 0.420 vs 0.431 ms with 4 slices, 8 and 16
// no better; T = 2048 0.473 vs 0.481 with 2; T = 8192 0.920 vs 0.925 with 2,
// 4 slices slower there).
unsigned router_splits(unsigned T) { return T <= 1024 ? 4u : T <= 8192 ? 2u : 1u; }

// 128-column blocks per down workgroup of the streaming path: one while the
// selected experts' items are few, then two to share the prologue (MI355X,
// whole block: T = 2 49 us with 1, 52 with 2, 63 with 4; 45 236 / 239 / 248;
// 128 285 / 281 / 308; 1000 343 / 342 / 354; 1400 380 / 373 / 381).
unsigned stream_down_subs(unsigned T) { return T <= 64 ? 1u : 2u; }

// The same, 256 columns each, for the long-prompt down workgroups (whole
// block: 4096 tokens 496 us with 1, 510 with 2; 8192 763 / 756).
unsigned tile_down_subs(unsigned T) { return T <= 6144 ? 1u : 2u; }

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

PfLayout pf_layout(unsigned T, unsigned E) {
  PfLayout L;
  L.ld_logits = (E + 1 + 7) & ~7u;
  const unsigned bm = T <= kStreamMaxTokens ? kStBM : kTlBM;
  L.max_tiles = (9u * T + bm - 1) / bm + E + 1;         // sum over groups of ceil(n / bm)
  L.max_rows = 9u * T + (kPfPad - 1) * (E + 1);         // sum of n rounded up to 32
  size_t o = 0;
  L.ids = o;     o = align256(o + (size_t)T * kMoeTopK * 4);
  L.rw = o;      o = align256(o + (size_t)T * kMoeTopK * 4);
  L.logits = o;  o = align256(o + (size_t)T * L.ld_logits * 2);
  L.sgw = o;     o = align256(o + (size_t)T * 4);
  L.meta = o;    o = align256(o + (size_t)(L.max_tiles + 1) * 16);
  L.sorted = o;  o = align256(o + (size_t)L.max_rows * 4);
  // at most kMaxAlignChunks chunks, each a multiple of 1024 ids
  L.n_chunks = std::min(kMaxAlignChunks, (kMoeTopK * T + kAlignChunk - 1) / kAlignChunk);
  L.chunk_ids = ((kMoeTopK * T + L.n_chunks - 1) / L.n_chunks + 1023) / 1024 * 1024;
  L.hist = o;    o = align256(o + (size_t)E * L.n_chunks * 4);
  L.after = o;   o = align256(o + (size_t)T * kMoeHidden * 2);
  L.h2 = o;      o = align256(o + (size_t)T * kMoeHidden * 2);
  L.act = o;     o = align256(o + (size_t)L.max_rows * kMoeInter * 2);
  L.y = o;       o = align256(o + (size_t)9 * T * kMoeHidden * 2);
  L.router_splits = router_splits(T);
  L.part = o;
  if (L.router_splits > 1) o = align256(o + (size_t)L.router_splits * T * L.ld_logits * 4);
  L.total = o;
  return L;
}

// ---- 1. residual + RMSNorm (arithmetic of moe_router_kernel) ---------------
__global__ __launch_bounds__(256) void moe_pre_kernel(
    const bf16* __restrict__ inp, const bf16* __restrict__ attn,
    const bf16* __restrict__ norm_w, bf16* __restrict__ after,
    bf16* __restrict__ h2, unsigned T) {
  const int lane = threadIdx.x & 63;
  const unsigned t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const size_t base = (size_t)t * kMoeHidden;
  float xa[4][8], ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16x8 a = *reinterpret_cast<const bf16x8*>(inp + base + 512 * j + 8 * lane);
    const bf16x8 b = *reinterpret_cast<const bf16x8*>(attn + base + 512 * j + 8 * lane);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      xa[j][e] = bf2f(f2bf(bf2f(a[e]) + bf2f(b[e])));
      ss = __builtin_fmaf(xa[j][e], xa[j][e], ss);
    }
  }
  ss = wave_sum(ss);
  const float inv = (float)(1.0 / sqrt((double)(ss / (float)kMoeHidden + kMoeEps)));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16x8 w = *reinterpret_cast<const bf16x8*>(norm_w + 512 * j + 8 * lane);
    bf16x8 oa, oh;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      oa[e] = f2bf(xa[j][e]);
      oh[e] = f2bf((xa[j][e] * inv) * (bf2f(w[e]) + 1.0f));
    }
    *reinterpret_cast<bf16x8*>(after + base + 512 * j + 8 * lane) = oa;
    *reinterpret_cast<bf16x8*>(h2 + base + 512 * j + 8 * lane) = oh;
  }
}

// ---- 3. top-8 + routing weights + shared gate, one wave per token ---------
// Token t's part by one wave; lane k < 8 returns the id of rank k.  With
// `splits` > 1 the router GEMM left fp32 partials of its K slices (part
// [splits][T][ld]): the wave sums them in slice order, rounds to bf16 and
// writes the logits row itself.
__device__ __forceinline__ int topk_token(
    unsigned t, bf16* __restrict__ logits, const float* __restrict__ part, unsigned splits,
    unsigned ld, unsigned E, unsigned T, int* __restrict__ ids_out, float* __restrict__ rw_out,
    float* __restrict__ sgw) {
  const int lane = threadIdx.x & 63;
  bf16* row = logits + (size_t)t * ld;
  int ids[kMoeTopK];
  float vals[kMoeTopK], rw[kMoeTopK];
  float sg_logit;
  if (splits > 1) {
    // lane l: columns l + 64i, i < 5 (E + 1 <= 257 columns: experts + shared gate)
    float acc[5];
    for (unsigned k = 0; k < splits; ++k) {
      const float* pr = part + ((size_t)k * T + t) * ld;
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        const unsigned e = lane + 64 * i;
        const float x = pr[e <= E ? e : 0u];
        acc[i] = k == 0 ? x : acc[i] + x;   // slice 0 as is (keeps a -0 sum)
      }
    }
    unsigned short raw[4];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const unsigned e = lane + 64 * i;
      const bf16 b = f2bf(acc[i]);
      if (e <= E) row[e] = b;
      if (i < 4) raw[i] = __builtin_bit_cast(unsigned short, b);
    }
    select_top8_bits(raw, E, ids, vals);
    // column E sits in lane E % 64, slot E / 64
    float v = acc[0];
#pragma unroll
    for (int i = 1; i < 5; ++i) v = (int)(E >> 6) == i ? acc[i] : v;
    sg_logit = bf2f(f2bf(__shfl(v, (int)(E & 63), 64)));
  } else {
    select_top8(row, E, ids, vals);
    sg_logit = bf2f(row[E]);
  }
  routing_weights(vals, rw);
  int id = ids[0];
  float w = rw[0];
#pragma unroll
  for (int k = 1; k < kMoeTopK; ++k) {
    id = lane == k ? ids[k] : id;
    w = lane == k ? rw[k] : w;
  }
  if (lane < kMoeTopK) {
    ids_out[(size_t)t * kMoeTopK + lane] = id;
    rw_out[(size_t)t * kMoeTopK + lane] = w;
  }
  if (lane == 0) sgw[t] = bf2f(f2bf(1.0f / (1.0f + expf(-sg_logit))));
  return id;
}

__global__ __launch_bounds__(256) void moe_topk_kernel(
    bf16* __restrict__ logits, const float* __restrict__ part, unsigned splits, unsigned ld,
    unsigned E, unsigned T, int* __restrict__ ids_out, float* __restrict__ rw_out,
    float* __restrict__ sgw) {
  const unsigned t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t < T) topk_token(t, logits, part, splits, ld, E, T, ids_out, rw_out, sgw);
}

// ---- 4. slots sorted by group, groups padded to 32 rows, tiles ------------
// sorted[p] = slot (t * 8 + k for routed rank k of token t) or -1 for
// padding; the shared expert is group E with slots 8T + t;
// group g occupies rows [row_off[g], row_off[g] + roundup32(n_g)).  meta
// (int4) [0] = {tiles}, [1 + i] = {group, first row, rows, tiles of the
// group} for tile i; a group's rows are dealt evenly to its tiles in whole
// blocks of 32: 300 rows make two 256-row tiles of 160 and 140, not 256 and 44
// (64-row tiles leave nothing to deal: full tiles and a rest).
// The 8T ids are cut into chunks of kAlignChunk: hist[g][chunk] counts, the
// scan turns them into each chunk's first row per group, the scatter places
// the chunk's slots.  Order inside a
// group is arbitrary: every GEMM row is computed independently, so it does
// not affect any value.

// 4a. per-chunk expert histogram.
__global__ __launch_bounds__(256) void moe_hist_kernel(const int* __restrict__ ids, unsigned T,
                                                       unsigned E, unsigned n_chunks,
                                                       unsigned chunk_ids,
                                                       int* __restrict__ hist) {
  __shared__ int cnt[kMoeMaxExperts];
  const unsigned tid = threadIdx.x, routed4 = kMoeTopK * T / 4;
  for (unsigned g = tid; g < E; g += blockDim.x) cnt[g] = 0;
  __syncthreads();
  const int4* ids4 = reinterpret_cast<const int4*>(ids);   // 8T ids: whole int4s
  const unsigned i0 = blockIdx.x * (chunk_ids / 4), i1 = min(i0 + chunk_ids / 4, routed4);
  for (unsigned b = i0; b < i1; b += 4 * 256) {
    int4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned i = b + tid + 256 * u;
      v[u] = i < i1 ? ids4[i] : int4{-1, -1, -1, -1};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (v[u].x >= 0) {
        atomicAdd(&cnt[v[u].x], 1);
        atomicAdd(&cnt[v[u].y], 1);
        atomicAdd(&cnt[v[u].z], 1);
        atomicAdd(&cnt[v[u].w], 1);
      }
    }
  }
  __syncthreads();
  for (unsigned g = tid; g < E; g += blockDim.x) hist[(size_t)g * n_chunks + blockIdx.x] = cnt[g];
}

// From the group counts cnt[0, G): exclusive offsets of the padded rows and
// of the tiles (one wave's scans; [G] = totals), the tile table meta and
// the padding rows of `sorted` (-1).  Called by every thread of the
// workgroup; ends with the offsets visible to all of them.
template <int kBM>
__device__ __forceinline__ void group_offsets(const int* cnt, unsigned G, unsigned tid,
                                              int* row_off, int* tile_off,
                                              int4* __restrict__ meta,
                                              int* __restrict__ sorted) {
  if (tid < 64) {   // one wave: exclusive scans of padded rows and tiles per group
    constexpr int kPer = (kMoeMaxExperts + 1 + 63) / 64;   // 5 groups per lane
    int rows[kPer], tiles[kPer], rsum = 0, tsum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const unsigned g = tid * kPer + j;
      const int c = g < G ? cnt[g] : 0;
      rows[j] = (c + kPfPad - 1) / kPfPad * kPfPad;
      tiles[j] = (c + kBM - 1) / kBM;
      rsum += rows[j];
      tsum += tiles[j];
    }
    int rincl = rsum, tincl = tsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int ru = __shfl_up(rincl, o, 64), tu = __shfl_up(tincl, o, 64);
      if ((int)tid >= o) {
        rincl += ru;
        tincl += tu;
      }
    }
    int roff = rincl - rsum, toff = tincl - tsum;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const unsigned g = tid * kPer + j;
      if (g <= G) {   // [G] = totals
        row_off[g] = roff;
        tile_off[g] = toff;
      }
      roff += rows[j];
      toff += tiles[j];
    }
    if (tid == 63) meta[0] = int4{tincl, 0, 0, 0};
  }
  __syncthreads();
  for (unsigned g = tid; g < G; g += blockDim.x) {
    const int c = cnt[g], r0 = row_off[g];
    const int nt = tile_off[g + 1] - tile_off[g];
    const int per = nt > 0 ? ((c + nt - 1) / nt + kPfPad - 1) / kPfPad * kPfPad : 0;
    for (int j = 0; j < nt; ++j)
      meta[1 + tile_off[g] + j] = int4{(int)g, r0 + per * j, max(0, min(per, c - per * j)), nt};
    for (int p = r0 + c; p < row_off[g + 1]; ++p) sorted[p] = -1;
  }
}

// 4b. one workgroup: group totals, row / tile offsets (one-wave scans), tile
// table, padding, shared-expert rows, and hist turned into each chunk's
// first row per group.
__global__ __launch_bounds__(1024) void moe_scan_kernel(unsigned T, unsigned E, unsigned n_chunks,
                                                        int* __restrict__ hist,
                                                        int4* __restrict__ meta,
                                                        int* __restrict__ sorted) {
  __shared__ int cnt[kMoeMaxExperts + 1];
  __shared__ int row_off[kMoeMaxExperts + 2];
  __shared__ int tile_off[kMoeMaxExperts + 2];
  const unsigned G = E + 1, tid = threadIdx.x;
  // totals: 4 threads per group, each summing a quarter of the chunks
  {
    const unsigned g = tid >> 2, part = tid & 3;
    int sum = 0;
    if (g < E)
      for (unsigned c = part; c < n_chunks; c += 4) sum += hist[(size_t)g * n_chunks + c];
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (g < E && part == 0) cnt[g] = sum;
    if (tid == 0) cnt[E] = (int)T;   // the shared expert: every token
  }
  __syncthreads();
  group_offsets<kTlBM>(cnt, G, tid, row_off, tile_off, meta, sorted);
  for (unsigned t = tid; t < T; t += blockDim.x) sorted[row_off[E] + t] = (int)(kMoeTopK * T + t);
  {   // chunk bases: one wave per group, exclusive prefix over the chunks
    const unsigned wave = tid >> 6, lane = tid & 63, waves = blockDim.x / 64;
    if (n_chunks <= 64) {   // every group's counts loaded up front (one round trip)
      constexpr int kGpw = (kMoeMaxExperts + 15) / 16;   // groups per wave (16 waves)
      int n[kGpw];
#pragma unroll
      for (int j = 0; j < kGpw; ++j) {
        const unsigned g = wave + waves * j;
        n[j] = (g < E && lane < n_chunks) ? hist[(size_t)g * n_chunks + lane] : 0;
      }
#pragma unroll
      for (int j = 0; j < kGpw; ++j) {
        const unsigned g = wave + waves * j;
        int incl = n[j];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int up = __shfl_up(incl, o, 64);
          if ((int)lane >= o) incl += up;
        }
        if (g < E && lane < n_chunks) hist[(size_t)g * n_chunks + lane] = row_off[g] + incl - n[j];
      }
    } else
    for (unsigned g = wave; g < E; g += waves) {
      int run = row_off[g];
      for (unsigned c0 = 0; c0 < n_chunks; c0 += 64) {
        const unsigned ch = c0 + lane;
        const int n = ch < n_chunks ? hist[(size_t)g * n_chunks + ch] : 0;
        int incl = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int up = __shfl_up(incl, o, 64);
          if ((int)lane >= o) incl += up;
        }
        if (ch < n_chunks) hist[(size_t)g * n_chunks + ch] = run + incl - n;
        run += __shfl(incl, 63, 64);
      }
    }
  }
}

// 4c. per-chunk scatter: slot i goes to its group's next row of this chunk.
__global__ __launch_bounds__(256) void moe_scatter_kernel(const int* __restrict__ ids, unsigned T,
                                                          unsigned E, unsigned n_chunks,
                                                          unsigned chunk_ids,
                                                          const int* __restrict__ base,
                                                          int* __restrict__ sorted) {
  __shared__ int pos[kMoeMaxExperts];
  const unsigned tid = threadIdx.x, routed4 = kMoeTopK * T / 4;
  for (unsigned g = tid; g < E; g += blockDim.x) pos[g] = base[(size_t)g * n_chunks + blockIdx.x];
  __syncthreads();
  const int4* ids4 = reinterpret_cast<const int4*>(ids);
  const unsigned i0 = blockIdx.x * (chunk_ids / 4), i1 = min(i0 + chunk_ids / 4, routed4);
  for (unsigned b = i0; b < i1; b += 4 * 256) {
    int4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned i = b + tid + 256 * u;
      v[u] = i < i1 ? ids4[i] : int4{-1, -1, -1, -1};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (v[u].x >= 0) {
        const int i = (int)(4 * (b + tid + 256 * u));
        sorted[atomicAdd(&pos[v[u].x], 1)] = i;
        sorted[atomicAdd(&pos[v[u].y], 1)] = i + 1;
        sorted[atomicAdd(&pos[v[u].z], 1)] = i + 2;
        sorted[atomicAdd(&pos[v[u].w], 1)] = i + 3;
      }
    }
  }
}

// 4'. short prompts (8T <= kAlignOneIds): histogram, offsets and scatter in
// one workgroup, the ids held in registers (16 per thread) -- one launch
// instead of 4a-4c, with tiles of 64 rows.
constexpr unsigned kAlignOneIds = 16384;
static_assert(kMoeTopK * kStreamMaxTokens <= kAlignOneIds, "streaming aligns in one workgroup");
__global__ __launch_bounds__(1024) void moe_align_one_kernel(const int* __restrict__ ids,
                                                             unsigned T, unsigned E,
                                                             int4* __restrict__ meta,
                                                             int* __restrict__ sorted) {
  __shared__ int cnt[kMoeMaxExperts + 1];
  __shared__ int row_off[kMoeMaxExperts + 2];
  __shared__ int tile_off[kMoeMaxExperts + 2];
  constexpr int kU = kAlignOneIds / 4 / 1024;
  const unsigned G = E + 1, tid = threadIdx.x, routed4 = kMoeTopK * T / 4;
  const int4* ids4 = reinterpret_cast<const int4*>(ids);
  int4 v[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const unsigned i = tid + 1024 * u;
    v[u] = i < routed4 ? ids4[i] : int4{-1, -1, -1, -1};
  }
  for (unsigned g = tid; g < G; g += blockDim.x) cnt[g] = g == E ? (int)T : 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (v[u].x >= 0) {
      atomicAdd(&cnt[v[u].x], 1);
      atomicAdd(&cnt[v[u].y], 1);
      atomicAdd(&cnt[v[u].z], 1);
      atomicAdd(&cnt[v[u].w], 1);
    }
  }
  __syncthreads();
  group_offsets<kStBM>(cnt, G, tid, row_off, tile_off, meta, sorted);
  __syncthreads();
  for (unsigned g = tid; g < G; g += blockDim.x) cnt[g] = row_off[g];   // next row per group
  for (unsigned t = tid; t < T; t += blockDim.x) sorted[row_off[E] + t] = (int)(kMoeTopK * T + t);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    if (v[u].x >= 0) {
      const int i = (int)(4 * (tid + 1024 * u));
      sorted[atomicAdd(&cnt[v[u].x], 1)] = i;
      sorted[atomicAdd(&cnt[v[u].y], 1)] = i + 1;
      sorted[atomicAdd(&cnt[v[u].z], 1)] = i + 2;
      sorted[atomicAdd(&cnt[v[u].w], 1)] = i + 3;
    }
  }
}

// 3 + 4 in one workgroup for up to kFewTokens tokens, a wave each: the ids go
// to the alignment through LDS (whole block, 2 .. 8 tokens: 1.4 us less; more
// tokens per wave cost more than the launch they save: 64 tokens 260 us
// against 249).
constexpr unsigned kFewTokens = 16;
__global__ __launch_bounds__(1024) void moe_topk_align_few_kernel(
    bf16* __restrict__ logits, const float* __restrict__ part, unsigned splits, unsigned ld,
    unsigned E, unsigned T, int* __restrict__ ids_out, float* __restrict__ rw_out,
    float* __restrict__ sgw, int4* __restrict__ meta, int* __restrict__ sorted) {
  __shared__ int cnt[kMoeMaxExperts + 1];
  __shared__ int row_off[kMoeMaxExperts + 2];
  __shared__ int tile_off[kMoeMaxExperts + 2];
  __shared__ int ids[kFewTokens * kMoeTopK];
  const unsigned G = E + 1, tid = threadIdx.x;
  for (unsigned g = tid; g < G; g += blockDim.x) cnt[g] = g == E ? (int)T : 0;
  __syncthreads();
  const unsigned t = tid >> 6;
  if (t < T) {
    const int id = topk_token(t, logits, part, splits, ld, E, T, ids_out, rw_out, sgw);
    if ((tid & 63) < (unsigned)kMoeTopK) {
      ids[t * kMoeTopK + (tid & 63)] = id;
      atomicAdd(&cnt[id], 1);
    }
  }
  __syncthreads();
  group_offsets<kStBM>(cnt, G, tid, row_off, tile_off, meta, sorted);
  __syncthreads();
  for (unsigned g = tid; g < G; g += blockDim.x) cnt[g] = row_off[g];   // next row per group
  if (tid < T) sorted[row_off[E] + tid] = (int)(kMoeTopK * T + tid);
  __syncthreads();
  if (tid < kMoeTopK * T) sorted[atomicAdd(&cnt[ids[tid]], 1)] = (int)tid;
}

// ---- 2. router GEMM -----------------------------------------------------------
struct RouterArgs {
  const bf16* a;            // h2 [T, 2048]
  const bf16* w;            // w_in: router and shared-gate rows first
  bf16* out;                // logits [T, ld]
  float* part;              // K slices: fp32 partials [slices][T][ld]
  unsigned T, E, ld;
};

unsigned router_blocks(unsigned E) { return (E + kRtBN) / kRtBN; }   // of its E + 1 rows

// The K loop for a wave computing NRB (0..2) row blocks of 32.  Every wave
// fetches and meets the barriers whatever its NRB.  Stage s of the ring
// holds K step s mod kRtStages; the fetch of step + kRtStages - 1 is issued
// once every wave has finished reading step - 1.
template <int NRB, int NSTEPS, typename Fetch>
__device__ __forceinline__ void router_k_loop(Fetch& fetch, const char* lds, int arow, int brow,
                                              const int (&koff)[kRtBK / 16], f32x16 (&acc)[2][2]) {
#pragma unroll
  for (int st = 0; st < kRtStages - 1; ++st) fetch(st);
  for (int step = 0; step < NSTEPS; ++step) {
    // this wave's fetches of `step` landed (later ones may stay in flight)
    if (step + kRtStages - 2 < NSTEPS)
      __builtin_amdgcn_s_waitcnt(stream_vmcnt((kRtStages - 2) * kRtInstr));
    else
      __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));
    __syncthreads();   // every wave's fetches landed; stage (step - 1) is free
    if (step + kRtStages - 1 < NSTEPS) fetch(step + kRtStages - 1);
    if constexpr (NRB > 0) {
      const char* st = lds + (step % kRtStages) * kRtStage;
#pragma unroll
      for (int s = 0; s < kRtBK / 16; ++s) {
        const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(st + brow * kRtRowB + koff[s]);
        const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(st + (brow + 32) * kRtRowB + koff[s]);
#pragma unroll
        for (int rb = 0; rb < NRB; ++rb) {
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(st + (arow + 32 * rb) * kRtRowB + koff[s]);
          acc[rb][0] = mfma32x32x16(a, b0, acc[rb][0]);
          acc[rb][1] = mfma32x32x16(a, b1, acc[rb][1]);
        }
      }
    }
  }
}

// Wave (wm = w % 2, wn = w / 2) computes tokens 64 wm .. + 63 against rows
// 64 wn .. + 63.  Fetch instruction i moves rows 16i .. 16i + 15 of the stage,
// token rows first; wave w issues instructions kRtInstr w + j.  Workgroup i
// covers K slice i % KS of tile i / KS, tiles dealt to the XCDs in
// contiguous ranges.
template <int KS>
__global__ __launch_bounds__(64 * kRtWaves, 2) void moe_router_gemm_kernel(RouterArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int nsteps = kMoeHidden / kRtBK / KS;
  static_assert(nsteps * kRtBK * KS == kMoeHidden, "K slices");
  const unsigned nb = (p.E + kRtBN) / kRtBN;
  const unsigned items = (p.T + kRtBM - 1) / kRtBM * nb * KS;
  const unsigned share = (items + 7) / 8;
  const unsigned xi = blockIdx.x >> 3;
  if (xi >= share) return;
  const unsigned item = (blockIdx.x & 7) * share + xi;
  if (item >= items) return;
  const unsigned ks = item % KS;
  const unsigned mt = item / KS / nb, nt = item / KS % nb;
  const int row0 = (int)(mt * kRtBM), rows = min(kRtBM, (int)p.T - row0);

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // Operand sources (buffer resources: out-of-range rows read as zero).
  const u32x4 ars = stream_rsrc(p.a, p.T * (unsigned)kMoeHidden * 2u);
  const u32x4 brs = stream_rsrc(p.w, (p.E + 1) * (unsigned)kMoeHidden * 2u);
  const int rin = lane / kRtCpr, cpos = lane % kRtCpr;   // row in the instruction, chunk
  unsigned f_off[kRtInstr];
  u32x4 f_rs[kRtInstr];
#pragma unroll
  for (int j = 0; j < kRtInstr; ++j) {
    const int srow = (wave * kRtInstr + j) * kRtRpi + rin;   // stage row this lane fills
    const bool is_a = srow < kRtBM;   // (uniform: an instruction's rows are of one operand)
    const unsigned off = !is_a ? (nt * kRtBN + srow - kRtBM) * (unsigned)kMoeHidden * 2u
                         : srow < rows ? (unsigned)(row0 + srow) * kMoeHidden * 2u : kStOob;
    f_off[j] = off + ((cpos ^ ((srow / kRtRpw) % kRtCpr)) * 16);
    const u32x4 r = is_a ? ars : brs;
#pragma unroll
    for (int c = 0; c < 4; ++c) f_rs[j][c] = __builtin_amdgcn_readfirstlane(r[c]);
  }
  const unsigned lds0 = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));
  auto fetch = [&](int step) {
    const unsigned sbase = lds0 + (step % kRtStages) * kRtStage;
    const unsigned kb = (ks * nsteps + (unsigned)step) * kRtRowB;
#pragma unroll
    for (int j = 0; j < kRtInstr; ++j)
      stream_fetch<false>(sbase + (wave * kRtInstr + j) * 1024, (int)(f_off[j] + kb), f_rs[j]);
  };

  const int wm = wave % 2, wn = wave / 2;
  const int li = lane & 31, kh = lane >> 5;
  const int arow = 64 * wm + li, brow = kRtBM + 64 * wn + li;
  int koff[kRtBK / 16];
#pragma unroll
  for (int s = 0; s < kRtBK / 16; ++s) koff[s] = (((2 * s + kh) ^ ((li / kRtRpw) % kRtCpr)) * 16);
  const int nrb = min(2, max(0, (rows - 64 * wm + 31) / 32));

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) acc[i][0] = acc[i][1] = f32x16{};
  if (nrb == 2) router_k_loop<2, nsteps>(fetch, lds, arow, brow, koff, acc);
  else if (nrb == 1) router_k_loop<1, nsteps>(fetch, lds, arow, brow, koff, acc);
  else router_k_loop<0, nsteps>(fetch, lds, arow, brow, koff, acc);

  // acc[rb][cb][i] = token 64 wm + 32 rb + 8(i/4) + 4kh + i%4, router row n + 32 cb
  const unsigned n = nt * kRtBN + 64 * wn + li;
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    if (rb >= nrb) break;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = 64 * wm + 32 * rb + 8 * (i >> 2) + 4 * kh + (i & 3);
      if (r >= rows) continue;
      if constexpr (KS > 1) {
        float* o = p.part + ((size_t)ks * p.T + row0 + r) * p.ld;
        if (n <= p.E) o[n] = acc[rb][0][i];
        if (n + 32 <= p.E) o[n + 32] = acc[rb][1][i];
      } else {
        bf16* o = p.out + (size_t)(row0 + r) * p.ld;
        if (n <= p.E) o[n] = f2bf(acc[rb][0][i]);
        if (n + 32 <= p.E) o[n + 32] = f2bf(acc[rb][1][i]);
      }
    }
  }
}

// The same in four K slices for short prompts: a workgroup takes 64 tokens,
// 32 router rows and one slice of 512 K, fetches all of it at once (96 KiB,
// one row per instruction) and multiplies it from LDS -- one round trip where
// the ring above makes one per 32 K.  Chunk c of row r sits at c ^ (r % 16).
// The products and their order are those of the ring's slices.  MI355X, whole
// block, against the ring: 2 tokens 46.6 us / 48.1, 45 225 / 229, 300 296 /
// 302, 600 317 / 318; from there on the ring's larger tiles win (1000: 339 /
// 335).
constexpr unsigned kRsMaxTokens = 512;
constexpr int kRsTokens = 64, kRsRows = 32, kRsRowB = kMoeHidden / 4 * 2;
constexpr int kRsLds = (kRsTokens + kRsRows) * kRsRowB;
__global__ __launch_bounds__(256) void moe_router_short_kernel(RouterArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const unsigned n0 = blockIdx.x * kRsRows, ks = blockIdx.y, row0 = blockIdx.z * kRsTokens;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  u32x4 ars = stream_rsrc(p.a, p.T * (unsigned)kMoeHidden * 2u);
  u32x4 brs = stream_rsrc(p.w, (p.E + 1) * (unsigned)kMoeHidden * 2u);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    ars[c] = __builtin_amdgcn_readfirstlane(ars[c]);
    brs[c] = __builtin_amdgcn_readfirstlane(brs[c]);
  }
  const unsigned lds0 = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));
  const int rows = min(kRsTokens, (int)(p.T - row0));
  // rows past the last token or router row read as zeros
  for (int r = wave; r < kRsTokens + kRsRows; r += 4) {
    const unsigned off = ks * kRsRowB + ((lane ^ (r & 15)) * 16);
    if (r >= kRsTokens)
      stream_fetch<false>(lds0 + r * kRsRowB, (int)((n0 + r - kRsTokens) * kMoeHidden * 2u + off), brs);
    else if (r < (rows + 31) / 32 * 32)
      stream_fetch<false>(lds0 + r * kRsRowB, (int)((row0 + r) * kMoeHidden * 2u + off), ars);
  }
  __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));
  __syncthreads();
  if (32 * wave >= rows) return;   // waves 0 and 1 own 32 tokens each
  const int li = lane & 31, kh = lane >> 5;
  const char* ap = lds + (32 * wave + li) * kRsRowB;
  const char* bp = lds + (kRsTokens + li) * kRsRowB;
  f32x16 acc = f32x16{};
#pragma unroll 8
  for (int s = 0; s < kRsRowB / 32; ++s) {
    const int at = ((2 * s + kh) ^ (li & 15)) * 16;
    acc = mfma32x32x16(*reinterpret_cast<const bf16x8*>(ap + at),
                       *reinterpret_cast<const bf16x8*>(bp + at), acc);
  }
  const unsigned n = n0 + li;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 32 * wave + 8 * (i >> 2) + 4 * kh + (i & 3);
    if (r < rows && n <= p.E) p.part[((size_t)ks * p.T + row0 + r) * p.ld + n] = acc[i];
  }
}

// ---- 7. per-token combine --------------------------------------------------
// kWeigh: the rows arrive unscaled (streaming path) and are scaled here, with
// the down epilogue's roundings.
// moe = bf16(sum over ranks 0..7 of y, fp32 in rank order); out = bf16(after +
// bf16(moe + shared)) -- the order of qwen36_moe_decode's combine.
template <bool kWeigh>
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const bf16* __restrict__ y, const float* __restrict__ rw, const bf16* __restrict__ after,
    const float* __restrict__ sgw, bf16* __restrict__ out, unsigned T) {
  const unsigned t = blockIdx.x;
  const int c = 8 * threadIdx.x;
  float moe[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 yk[kMoeTopK];
#pragma unroll
  for (int k = 0; k < kMoeTopK; ++k)
    yk[k] = *reinterpret_cast<const bf16x8*>(y + ((size_t)t * kMoeTopK + k) * kMoeHidden + c);
  const bf16x8 ys = *reinterpret_cast<const bf16x8*>(
      y + ((size_t)kMoeTopK * T + t) * kMoeHidden + c);
  const bf16x8 af = *reinterpret_cast<const bf16x8*>(after + (size_t)t * kMoeHidden + c);
  const float sg = sgw[t];
#pragma unroll
  for (int k = 0; k < kMoeTopK; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = bf2f(yk[k][e]);
      moe[e] += kWeigh ? bf2f(f2bf(v * rw[(size_t)t * kMoeTopK + k])) : v;
    }
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float shared = bf2f(f2bf(bf2f(ys[e]) * sg));   // the shared row scaled by its gate
    const float total = bf2f(f2bf(bf2f(f2bf(moe[e])) + shared));
    o[e] = f2bf(bf2f(af[e]) + total);
  }
  *reinterpret_cast<bf16x8*>(out + (size_t)t * kMoeHidden + c) = o;
}

}  // namespace
}  // namespace q36

using namespace q36;

// Workspace bytes of qwen36_moe_prefill for `tokens` tokens and `n_experts`
// experts (0 for invalid arguments).
Q36_EXPORT size_t qwen36_moe_prefill_workspace_bytes(unsigned tokens, unsigned n_experts) {
  if (tokens == 0 || tokens > kPfMaxTokens || n_experts < (unsigned)kMoeTopK ||
      n_experts > (unsigned)kMoeMaxExperts || (n_experts % 4) != 0)
    return 0;
  return pf_layout(tokens, n_experts).total;
}

// MoE block for T = `tokens` rows: out [T, 2048] = after + moe + shared with
// after = inp + attn_out (all bf16, row-major, 16-byte aligned).  Weights as
// in qwen36_moe_decode: w_in [E + 1 + 1024, 2048] = [router | shared_gate |
// shared gate_proj | shared up_proj], expert_gate_up [E, 1024, 2048],
// expert_down [E, 2048, 512], shared_down [2048, 512].  The workspace starts
// with the expert ids (int32 [T, 8]), the routing weights (fp32 [T, 8], bf16
// values) and the router logits (bf16 [T, ld], ld = (E + 8) & ~7, column E =
// the shared gate) at 256-byte-aligned offsets.
Q36_EXPORT int qwen36_moe_prefill(const void* inp, const void* attn_out, const void* post_norm_w,
                                  const void* w_in, const void* expert_gate_up,
                                  const void* expert_down, const void* shared_down,
                                  unsigned n_experts, unsigned tokens, void* out,
                                  void* workspace, size_t workspace_bytes, void* stream) {
  const size_t need = qwen36_moe_prefill_workspace_bytes(tokens, n_experts);
  if (need == 0 || inp == nullptr || attn_out == nullptr || post_norm_w == nullptr ||
      w_in == nullptr || expert_gate_up == nullptr || expert_down == nullptr ||
      shared_down == nullptr || out == nullptr || workspace == nullptr ||
      workspace_bytes < need || !aligned16(inp) || !aligned16(attn_out) ||
      !aligned16(post_norm_w) || !aligned16(w_in) || !aligned16(expert_gate_up) ||
      !aligned16(expert_down) || !aligned16(shared_down) || !aligned16(out) ||
      !aligned16(workspace))
    return Q36_EINVAL;
  const unsigned T = tokens, E = n_experts;
  static std::once_flag attr_once;   // 72 to 160 KiB of dynamic LDS per GEMM workgroup
  static hipError_t attr_status = hipSuccess;
  std::call_once(attr_once, [] {
    auto allow = [](const void* f, int bytes) {
      const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
      if (e != hipSuccess) attr_status = e;
    };
    allow(reinterpret_cast<const void*>(moe_router_gemm_kernel<1>), kRtLds);
    allow(reinterpret_cast<const void*>(moe_router_gemm_kernel<2>), kRtLds);
    allow(reinterpret_cast<const void*>(moe_router_gemm_kernel<4>), kRtLds);
    allow(reinterpret_cast<const void*>(moe_router_short_kernel), kRsLds);
    allow(reinterpret_cast<const void*>(moe_stream_kernel<false>), kStLds);
    allow(reinterpret_cast<const void*>(moe_stream_kernel<true>), kStLds);
    allow(reinterpret_cast<const void*>(moe_tile_kernel<false>), kTlLds);
    allow(reinterpret_cast<const void*>(moe_tile_kernel<true>), kTlLds);
  });
  if (attr_status != hipSuccess) return (int)attr_status;
  const PfLayout L = pf_layout(T, E);
  char* ws = static_cast<char*>(workspace);
  int* ids = reinterpret_cast<int*>(ws + L.ids);
  float* rw = reinterpret_cast<float*>(ws + L.rw);
  bf16* logits = reinterpret_cast<bf16*>(ws + L.logits);
  float* sgw = reinterpret_cast<float*>(ws + L.sgw);
  int4* meta = reinterpret_cast<int4*>(ws + L.meta);
  int* sorted = reinterpret_cast<int*>(ws + L.sorted);
  bf16* after = reinterpret_cast<bf16*>(ws + L.after);
  bf16* h2 = reinterpret_cast<bf16*>(ws + L.h2);
  bf16* act = reinterpret_cast<bf16*>(ws + L.act);
  bf16* y = reinterpret_cast<bf16*>(ws + L.y);
  const bf16* win = static_cast<const bf16*>(w_in);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned tok_blocks = (T + 3) / 4;

  hipLaunchKernelGGL(moe_pre_kernel, dim3(tok_blocks), dim3(256), 0, st,
                     static_cast<const bf16*>(inp), static_cast<const bf16*>(attn_out),
                     static_cast<const bf16*>(post_norm_w), after, h2, T);

  auto grid_for = [](unsigned max_items) { return dim3(8 * ((max_items + 7) / 8)); };
  const RouterArgs r{h2, win, logits, reinterpret_cast<float*>(ws + L.part), T, E, L.ld_logits};
  if (T <= kRsMaxTokens) {
    hipLaunchKernelGGL(moe_router_short_kernel,
                       dim3((E + kRsRows) / kRsRows, 4, (T + kRsTokens - 1) / kRsTokens), dim3(256),
                       kRsLds, st, r);
  } else {
    auto router = L.router_splits == 4   ? moe_router_gemm_kernel<4>
                  : L.router_splits == 2 ? moe_router_gemm_kernel<2>
                                         : moe_router_gemm_kernel<1>;
    hipLaunchKernelGGL(router, grid_for((T + kRtBM - 1) / kRtBM * router_blocks(E) * L.router_splits),
                       dim3(64 * kRtWaves), kRtLds, st, r);
  }
  if (T <= kFewTokens)
    hipLaunchKernelGGL(moe_topk_align_few_kernel, dim3(1), dim3(1024), 0, st, logits, r.part,
                       L.router_splits, L.ld_logits, E, T, ids, rw, sgw, meta, sorted);
  else
    hipLaunchKernelGGL(moe_topk_kernel, dim3(tok_blocks), dim3(256), 0, st, logits, r.part,
                       L.router_splits, L.ld_logits, E, T, ids, rw, sgw);

  StreamArgs a{h2, static_cast<const bf16*>(expert_gate_up), win + (size_t)(E + 1) * kMoeHidden,
               meta, sorted, rw, act, T, E, 1u};
  StreamArgs d{act, static_cast<const bf16*>(expert_down), static_cast<const bf16*>(shared_down),
               meta, sorted, rw, y, T, E, 1u};
  if (T <= kStreamMaxTokens) {
    if (T > kFewTokens)
      hipLaunchKernelGGL(moe_align_one_kernel, dim3(1), dim3(1024), 0, st, ids, T, E, meta, sorted);
    hipLaunchKernelGGL(moe_stream_kernel<false>, grid_for(L.max_tiles * kStGateUpBlocks), dim3(512),
                       kStLds, st, a);
    d.subs = stream_down_subs(T);
    hipLaunchKernelGGL(moe_stream_kernel<true>, grid_for(L.max_tiles * (kStDownBlocks / d.subs)),
                       dim3(512), kStLds, st, d);
    hipLaunchKernelGGL(moe_combine_kernel<true>, dim3(T), dim3(256), 0, st, y, rw, after, sgw,
                       static_cast<bf16*>(out), T);
  } else {
    int* hist = reinterpret_cast<int*>(ws + L.hist);
    hipLaunchKernelGGL(moe_hist_kernel, dim3(L.n_chunks), dim3(256), 0, st, ids, T, E,
                       L.n_chunks, L.chunk_ids, hist);
    hipLaunchKernelGGL(moe_scan_kernel, dim3(1), dim3(1024), 0, st, T, E, L.n_chunks, hist, meta,
                       sorted);
    hipLaunchKernelGGL(moe_scatter_kernel, dim3(L.n_chunks), dim3(256), 0, st, ids, T, E,
                       L.n_chunks, L.chunk_ids, hist, sorted);
    hipLaunchKernelGGL(moe_tile_kernel<false>, grid_for(L.max_tiles * kTlGateUpBlocks),
                       dim3(64 * kTlWaves), kTlLds, st, a);
    d.subs = tile_down_subs(T);
    hipLaunchKernelGGL(moe_tile_kernel<true>, grid_for(L.max_tiles * (kTlDownBlocks / d.subs)),
                       dim3(64 * kTlWaves), kTlLds, st, d);
    hipLaunchKernelGGL(moe_combine_kernel<false>, dim3(T), dim3(256), 0, st, y, rw, after, sgw,
                       static_cast<bf16*>(out), T);
  }
  return static_cast<int>(hipGetLastError());
}
