// Causal GQA flash-attention prefill (BF16 in, FP32 out) for gfx950.
//
// Drop-in for the reference's dlopen'd FMHA provider C ABI
// (benchmarks/shape-lab/native/src/qrt_ck_fmha_q8192_provider.cpp:134-325,
// consumed by native/src/native_full_prefill.hip.cpp:140-266):
//   Q [q_tokens, 16, 256] bf16 (token stride 4096), K/V [kv_tokens, 2, 256]
//   bf16 (token stride 512), out fp32 [q_tokens, 4096]; scale 1/sqrt(256);
//   query head h reads KV head h/8; top-left causal mask when
//   q_tokens == kv_tokens, bottom-right (query i sees keys
//   j <= i + kv_tokens - q_tokens) when kv_tokens > q_tokens.
//
// Kernel plan (MFMA-bound, 16384 flop per unmasked (q,k) pair):
//  * workgroup = 8 waves = 256 query rows = 32 tokens x the 8 query heads of
//    one KV head (row r: token r / 8, head r % 8 of the group); wave = 32
//    rows; one workgroup per CU (two waves per SIMD) shares each staged K/V
//    tile among 256 rows (measured 5-7% faster than two 4-wave workgroups per
//    CU, which stage every tile twice).  With the heads of the group in the
//    rows a tile spans 32 tokens instead of 256, so a short turn fills its
//    tiles (93 tokens: 3 tiles per KV head, all but 24 of 768 rows live, where
//    256-token tiles of 8 heads left 163 of every 256 rows dead) and only a
//    tile's last 32 keys are masked.  Short calls use 4-, 2- or 1-wave
//    workgroups (16, 8 or 4 tokens; see split_plan).
//  * per 32-key tile: K and V are staged in LDS (padded row-pair blocks, so
//    every LDS address is a per-lane base plus an immediate); S^T = K Q^T on
//    v_mfma_f32_32x32x16_bf16 (A = K from LDS, B = Q^T held in registers for
//    the whole kernel), online softmax per row
//    in fp32 (exp2 domain), O^T += V^T P^T (A = V^T read with
//    ds_read_b64_tr_b16, B = P^T taken straight from the S^T accumulator).
//  * LDS operand reads run 4 MFMAs ahead of their use (register rings whose
//    issue order is pinned by sched_group_barrier), so the dependent QK^T
//    chain and the PV MFMAs do not wait on LDS latency.
//  * K/V tiles are fetched straight into LDS (global_load_lds_dwordx4, no
//    register staging) into a double buffer (64 KiB), so the next tile's
//    HBM/L2 latency overlaps the current tile's MFMA work; the two waves
//    on each SIMD let one wave's softmax overlap the other's MFMAs.
//  * no per-tile row max: the reference max is the first tile's, raised
//    (with a rescale of O) only when a tile's probabilities would exceed
//    2^20, which the per-lane probability sum detects.
//  * blockIdx -> (KV head, query tile) is XCD-aware: the 8 XCDs
//    receive workgroups round-robin, so XCDs 0-3 serve KV head 0 and 4-7 KV
//    head 1 (their L2s then hold one head's K/V), and every XCD issues its
//    heaviest (latest) causal tiles first.
#include "common.h"

#include <algorithm>
#include <mutex>

namespace q36 {
namespace {

constexpr int kFmRowsPerWave = 32;
constexpr int kFmKv = 32;                             // keys per tile
constexpr int kRowBytes = kD * 2;                     // 512
constexpr int kTokBytes = kHkv * kD * 2;              // 1024: one cache row
// LDS tile layout: block b (0..15) holds key rows b and b+16 back to back
// (1 KiB, one direct-to-LDS instruction) followed by padding, so that every
// LDS address below is a per-lane base plus a compile-time offset and both
// access patterns are bank-conflict-free:
//  * K blocks are 1040 B apart: 16 rows at one 16-byte column fall in 16
//    distinct 16-byte bank groups (ds_read_b128 A operand);
//  * V blocks are 1088 B apart: 8 rows x 64 bytes (ds_read_b64_tr_b16) take
//    the minimum two passes.
constexpr int kKBlk = 1040, kVBlk = 1088;
constexpr int kKTile = 16 * kKBlk;                    // 16640
constexpr int kVTile = 16 * kVBlk;                    // 17408
constexpr int kFmStage = kKTile + kVTile;             // 34048
constexpr int kFmLds = 2 * kFmStage;                  // 68096: double buffer
// Gated kernels also prefetch the gate values of output rounds 0-1 (dims
// 0-127 of the head) of their 256 rows into LDS after the ring.
constexpr int kFmGateLds = 256 * 256;
constexpr int kFmLdsGated = kFmLds + kFmGateLds;      // 133632

typedef __attribute__((address_space(3))) void lds_void;

// Split-K partials (kSplit): workgroup (q tile, chunk, KV head) writes its
// unnormalised O rows and (m, l) for keys [chunk * chunk_keys, +chunk_keys).
struct SplitArgs {
  float* o;             // [tile][chunk][kv head][rows][256]
  float* ml;            // [tile][chunk][kv head][rows][2]
  unsigned chunk_keys;  // multiple of 32
  unsigned n_chunks;
  unsigned ranges;      // items dealt to the XCDs as contiguous ranges
};

// Gated output (kGate): out_bf16[row][h*256 + d] = gate_bf16(O, gate[row *
// gate_stride + h*512 + 256 + d]) -- the gate half of each head's 512-wide
// slice of the fused q projection -- in place of the fp32 attention rows.
struct GateArgs {
  const bf16* gate;
  unsigned gate_stride;   // elements between token rows of the q projection
  bf16* out;
};

// kSub = 2: two groups of kFmWaves waves share the tile's rows, each with an LDS
// ring of its own and half of the chunk's keys, and merge in LDS at the end, so
// the workgroup writes one partial of half as many rows as 2 kFmWaves waves of
// rows would, for the same keys per wave.
template <int kFmWaves, bool kSplit, bool kGate = false, int kSub = 1>
__global__ __launch_bounds__(64 * kFmWaves * kSub, kFmWaves * kSub == 8 ? 1 : 2) void fmha_prefill_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k,
    const bf16* __restrict__ v, float* __restrict__ out, unsigned q_tokens,
    unsigned kv_tokens, unsigned n_qtiles, SplitArgs sp, GateArgs ga) {
  static_assert(!(kSplit && kGate), "split partials are gated by the combine");
  static_assert(kSub == 1 || (kSub == 2 && kSplit), "the split form merges pairs");
  extern __shared__ __attribute__((aligned(1024))) char lds_all[];
  constexpr int kFmRows = kFmWaves * kFmRowsPerWave;
  constexpr unsigned kTok = kFmRows / kGroup;          // tokens per tile
  constexpr int kFmLoadsPerWave = 16 / kFmWaves;       // 16 row-pair blocks per tile

  // XCD-aware tile mapping (see header).  Split: the (chunk, tile) items of a
  // KV head, chunk by chunk and heaviest tile first, are dealt to its four
  // XCDs in turn, or as contiguous ranges so that the few tiles of a long
  // chunk read its keys through one L2 (see split_plan).
  const unsigned b = blockIdx.x, n = b >> 3, x4 = b & 3;
  const int kvh = (b >> 2) & 1;
  unsigned qtile, chunk = 0;
  if constexpr (kSplit) {
    const unsigned items = n_qtiles * sp.n_chunks, share = (items + 3) / 4;
    const unsigned i = sp.ranges ? x4 * share + n : 4 * n + x4;
    if (i >= items) return;
    chunk = i / n_qtiles;
    qtile = n_qtiles - 1 - i % n_qtiles;
  } else {
    if (4 * n + x4 >= n_qtiles) return;
    qtile = n_qtiles - 1 - (4 * n + x4);
  }
  const unsigned tok0 = qtile * kTok;

  const int tid = threadIdx.x;
  const int wave_wg = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wave = kSub == 1 ? wave_wg : wave_wg % kFmWaves;
  const int sub = kSub == 1 ? 0 : wave_wg / kFmWaves;
  char* lds = lds_all + sub * kFmLds;
  const int lj = lane & 31;     // MFMA column (query row within the wave)
  const int lg = lane >> 5;     // k-half
  const unsigned off = kv_tokens - q_tokens;   // bottom-right shift
  // this lane's query: token `tok`, query head `head`
  const unsigned row = wave * kFmRowsPerWave + lj;   // row of the tile
  const unsigned tok = tok0 + row / kGroup;
  const int head = kvh * kGroup + (int)(row % kGroup);
  const bool row_valid = tok < q_tokens;
  const unsigned row_lim = (row_valid ? tok : q_tokens - 1) + off;  // last key
  const unsigned wave_first = tok0 + wave * (kFmRowsPerWave / kGroup);   // first token
  const bool wave_live = wave_first < q_tokens;
  const unsigned wave_lim =
      min(wave_first + kFmRowsPerWave / kGroup - 1, q_tokens - 1) + off;
  const unsigned kv_end = min(kv_tokens, min(tok0 + kTok, q_tokens) + off);
  // key range of this workgroup: whole rows, or one chunk of them (kSub = 2: of
  // this half, which may be empty for the second)
  const unsigned kv_wg = kSplit ? chunk * sp.chunk_keys : 0u;
  if (kSplit && kv_wg >= kv_end) return;   // past the tile's last key
  const unsigned sub_keys = sp.chunk_keys / kSub;
  const unsigned kv_first = kv_wg + (kSub == 1 ? 0u : sub * sub_keys);
  const unsigned kv_stop = kSplit ? min(kv_end, kv_first + sub_keys) : kv_end;

  // Q^T operand: step s covers dims s*16 + 8*lg .. +8 of this lane's row.
  bf16x8 qf[16];
  {
    const bf16* qp = q + (size_t)tok * kQDim + head * kD + 8 * lg;
#pragma unroll
    for (int s = 0; s < 16; ++s)
      qf[s] = row_valid ? *reinterpret_cast<const bf16x8*>(qp + s * 16)
                        : bf16x8{};
  }

  f32x16 o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = f32x16{};
  float m = -INFINITY, l = 0.f;
  const float scale = 0.0625f * kLog2e;

  // Direct global->LDS fetch through buffer resources (base in SGPRs; rows at
  // or past kv_end are out of bounds and read as zeros).  Wave instruction j
  // fills block 2*wave + j: lanes 0-31 key row b, lanes 32-63 key row b+16.
  const int nrec = (int)(kv_end * (unsigned)kTokBytes);
  const __amdgpu_buffer_rsrc_t krs =
      __builtin_amdgcn_make_buffer_rsrc((void*)k, 0, nrec, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)v, 0, nrec, 0x00020000);
  const int fvoff = (kFmLoadsPerWave * wave + 16 * (lane >> 5)) * kTokBytes +
                    kvh * kRowBytes + (lane & 31) * 16;
  // gated: the gate values of output rounds 0-1 of this workgroup's rows
  // (row-major [256 rows][256 B]), fetched now so they are resident when the
  // epilogue starts; rows past the end read as zeros.
  if constexpr (kGate) {
    const unsigned toks_here = min(q_tokens - tok0, kTok);
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16*>(ga.gate) + (size_t)tok0 * ga.gate_stride, 0,
        (int)(toks_here * ga.gate_stride * 2), 0x00020000);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r0 = wave * kFmRowsPerWave + 4 * j, r = r0 + (lane >> 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          grs, (lds_void*)(lds + kFmLds + r0 * 256), 16,
          (int)((r / kGroup) * ga.gate_stride * 2 +
                ((kvh * kGroup + r % kGroup) * 2 * kD + kD) * 2 + (lane & 15) * 16), 0, 0, 0);
    }
  }
  auto fetch = [&](unsigned kv0, int stage) {
    char* ks = lds + stage * kFmStage;
    char* vs = ks + kKTile;
    const int soff = (int)(kv0 * (unsigned)kTokBytes);
#pragma unroll
    for (int j = 0; j < kFmLoadsPerWave; ++j) {
      const int blk = kFmLoadsPerWave * wave + j;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(krs, (lds_void*)(ks + blk * kKBlk), 16,
                                               fvoff + j * kTokBytes, soff, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (lds_void*)(vs + blk * kVBlk), 16,
                                               fvoff + j * kTokBytes, soff, 0, 0);
    }
  };

  // Per-lane LDS bases.  K A operand: key row lj, 16-byte chunk 2*st + lg.
  const int kbase = (lj & 15) * kKBlk + (lj >> 4) * kRowBytes + lg * 16;
  // V^T (transposed read): for step st and half h (keys +8), lane reads row
  // 16*st + 8*h + x, x = 4*lg + (lane%16)/4, 8 bytes at column
  // 32*((lane/16)&1) + 8*(lane%4) within the 64-byte block of dims dt.
  const int grp = lane >> 4, m16 = lane & 15;
  const int vx = 4 * lg + (m16 >> 2);
  const int vbase = vx * kVBlk + 32 * (grp & 1) + 8 * (m16 & 3);

  const unsigned t_first = kv_first / kFmKv;
  const unsigned n_tiles = (kv_stop + kFmKv - 1) / kFmKv;
  // both halves pass as many barriers as the first has tiles (it has the most)
  const unsigned t_end =
      kSub == 1 ? n_tiles : t_first + (min(kv_end - kv_wg, sub_keys) + kFmKv - 1) / kFmKv;
  if (kSub == 1 || t_first < n_tiles) fetch(kv_first, t_first & 1);
  for (unsigned t = t_first; t < t_end; ++t) {
    const unsigned kv0 = t * kFmKv;
    const int stage = t & 1;
    __builtin_amdgcn_s_waitcnt(0);   // this wave's fetches of tile t landed
    __syncthreads();                 // ... and every wave's; tile t-1 consumed
    if (t + 1 < n_tiles) fetch(kv0 + kFmKv, stage ^ 1);
    // no row of ours sees a key of the tile
    if (kv0 > wave_lim || !wave_live || (kSub > 1 && t >= n_tiles)) continue;
    const char* kp = lds + stage * kFmStage + kbase;
    const char* vp = lds + stage * kFmStage + kKTile + vbase;

    // S^T[key][row] for the 32-key tile.
    // K operands go through a 4-deep register ring: the read for step st + 4
    // is issued right after step st's MFMA (the sched_group_barrier sequence
    // pins that order; left alone, the scheduler keeps only 2 reads in flight
    // and each MFMA of the dependent chain waits a full LDS latency).
    bf16x8 kr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) kr[i] = *reinterpret_cast<const bf16x8*>(kp + i * 32);
    f32x16 s0 = f32x16{};
#pragma unroll
    for (int st = 0; st < 16; ++st) {
      s0 = mfma32x32x16(kr[st & 3], qf[st], s0);
      if (st + 4 < 16) kr[st & 3] = *reinterpret_cast<const bf16x8*>(kp + (st + 4) * 32);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    // Lane holds keys kv0 + 8*(r/4) + 4*lg + r%4 of its row.
    const bool diag = kv0 + kFmKv - 1 > wave_first + off || kv0 + kFmKv > kv_tokens;
    if (diag) {  // wave-uniform: only diagonal / ragged tiles pay for masking
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const unsigned key = kv0 + 8 * (r >> 2) + 4 * lg + (r & 3);
        s0[r] = (key <= row_lim && key < kv_tokens) ? s0[r] : -INFINITY;
      }
    }
    // Reference max, kept in the scaled log2 domain: m is the row max of the
    // first tile (key 0 is visible to every row) and is raised only when a
    // later tile's p = 2^(s*scale - m) would exceed 2^20.  Each lane's p sum
    // bounds its p values, so no per-tile max is taken on the common path;
    // p up to 2^20 is exact to bf16 rounding and O, l cannot overflow.  An
    // overflowed or non-finite sum also takes the rescale branch, which
    // recomputes P against the new max.
    auto row_max = [&]() {
      float mx = s0[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s0[r]);
      mx = wave_max_xor(mx, 32);
      return mx * scale;
    };
    if (t == t_first) {
      // a row whose keys all precede this chunk sees only masked scores in
      // its first tile (and in every later one): any finite m keeps p = 0
      m = row_max();
      if (kSplit && m == -INFINITY) m = 0.f;
    }
    float psum = 0.f;
    bf16x8 pb[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r], scale, -m));
      psum += p0;
      pb[r >> 3][r & 7] = f2bf(p0);
    }
    if (__any(!(psum <= 1048576.0f))) {
      const float mnew = fmaxf(m, row_max());
      const float alpha = __builtin_amdgcn_exp2f(m - mnew);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] *= alpha;
      m = mnew;
      psum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r], scale, -m));
        psum += p0;
        pb[r >> 3][r & 7] = f2bf(p0);
      }
    }
    l += psum;

    // O^T[d][row] += V^T[d][key] P^T[key][row]; step st reduction slots
    // (lg, e) <-> keys 16st + 4lg + e and +8 for e >= 4.
    // V^T operands: the same ring, 4 MFMAs (8 transposed reads) deep.
    i16x4 va[4][2];
    auto vread = [&](int i, int slot) {
      const char* p = vp + (i >> 3) * kRowBytes + (i & 7) * 64;
      va[slot][0] = lds_read_tr16(p);
      va[slot][1] = lds_read_tr16(p + 8 * kVBlk);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) vread(i, i);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      o[i & 7] = mfma32x32x16(cat_bf16x8(va[i & 3][0], va[i & 3][1]), pb[i >> 3], o[i & 7]);
      if (i + 4 < 16) vread(i + 4, i & 3);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 1);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4, 1);
  }
  l += __shfl_xor(l, 32, 64);
  if constexpr (kSub == 2) {
    // the second half's (m, l, O) to LDS, lane by lane, and merged by the first
    // (a half whose keys the row does not see has l = 0 and weighs nothing)
    __syncthreads();   // every wave is done with the K/V rings
    f32x4* xo = reinterpret_cast<f32x4*>(lds_all) + wave * 2048 + lane;
    float2* xml = reinterpret_cast<float2*>(lds_all + kFmWaves * 32768) + wave * 64 + lane;
    if (sub == 1) {
#pragma unroll
      for (int i = 0; i < 32; ++i)
        xo[i * 64] = f32x4{o[i >> 2][4 * (i & 3)], o[i >> 2][4 * (i & 3) + 1],
                           o[i >> 2][4 * (i & 3) + 2], o[i >> 2][4 * (i & 3) + 3]};
      *xml = float2{m, l};
    }
    __syncthreads();
    if (sub == 1) return;
    const float2 ml1 = *xml;
    const float m_all = fmaxf(l == 0.f ? -INFINITY : m, ml1.y == 0.f ? -INFINITY : ml1.x);
    const float w0 = l == 0.f ? 0.f : __builtin_amdgcn_exp2f(m - m_all);
    const float w1 = ml1.y == 0.f ? 0.f : __builtin_amdgcn_exp2f(ml1.x - m_all);
    m = m_all;
    l = l * w0 + ml1.y * w1;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const f32x4 x = xo[i * 64];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[i >> 2][4 * (i & 3) + e] = o[i >> 2][4 * (i & 3) + e] * w0 + x[e] * w1;
    }
  }
  if constexpr (kSplit) {
    if (!row_valid) return;
    const size_t item = ((size_t)qtile * sp.n_chunks + chunk) * kHkv + kvh;
    float* op = sp.o + (item * kFmRows + row) * kD + 4 * lg;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *reinterpret_cast<f32x4*>(op + dt * 32 + 8 * r4) =
            f32x4{o[dt][4 * r4], o[dt][4 * r4 + 1], o[dt][4 * r4 + 2], o[dt][4 * r4 + 3]};
    if (lg == 0) *reinterpret_cast<float2*>(sp.ml + (item * kFmRows + row) * 2) = float2{m, l};
    return;
  } else {
    // The output leaves through LDS in four rounds of 64 dims: each wave
    // stages its 32 rows x 64 dims (8 KiB, 16-byte chunks XOR-swizzled by
    // row so both the staging writes and the row reads are conflict-free)
    // and stores whole 256-byte row segments, instead of 32-byte pieces of
    // 32 rows per store instruction.
    const float inv = row_valid ? 1.0f / l : 0.f;
    // gated: rounds 0-1 take their gate values from the LDS prefetch; the
    // register loads of rounds 2-3 are issued now and land behind rounds 0-1
    // (rows past the end read the last row's and are not stored)
    bf16x4 gv[2][8];
    if constexpr (kGate) {
      __builtin_amdgcn_s_waitcnt(0);   // this wave's gate prefetch landed
#pragma unroll
      for (int rd = 0; rd < 2; ++rd)
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const unsigned r = it * 4 + (lane >> 4);
          const unsigned t = min(wave_first + r / kGroup, q_tokens - 1);
          gv[rd][it] = *reinterpret_cast<const bf16x4*>(
              ga.gate + (size_t)t * ga.gate_stride + (kvh * kGroup + r % kGroup) * 2 * kD + kD +
              (rd + 2) * 64 + (lane & 15) * 4);
        }
    }
    __syncthreads();   // every wave is done with the K/V ring
    char* stg = lds + wave * 8192;
#pragma unroll
    for (int rd = 0; rd < 4; ++rd) {
#pragma unroll
      for (int d2 = 0; d2 < 2; ++d2) {
        const int dt = 2 * rd + d2;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int ch = d2 * 8 + 2 * r4 + lg;   // dims 4 ch .. 4 ch + 3 of the round
          *reinterpret_cast<f32x4*>(stg + lj * 256 + ((ch ^ (lj & 15)) * 16)) =
              f32x4{o[dt][4 * r4] * inv, o[dt][4 * r4 + 1] * inv, o[dt][4 * r4 + 2] * inv,
                    o[dt][4 * r4 + 3] * inv};
        }
      }
      // this wave's staging writes land before its reads (and its reads
      // before the next round's writes): LDS serves one wave in order
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
      for (int it = 0; it < 8; ++it) {
        const int r = it * 4 + (lane >> 4), ch = lane & 15;
        const f32x4 v = *reinterpret_cast<const f32x4*>(stg + r * 256 + ((ch ^ (r & 15)) * 16));
        const unsigned t = wave_first + r / kGroup;
        const size_t orow = (size_t)t * kQDim + (kvh * kGroup + r % kGroup) * kD + rd * 64 + ch * 4;
        if constexpr (kGate) {
          if (t < q_tokens) {
            const bf16x4 g4 =
                rd < 2 ? *reinterpret_cast<const bf16x4*>(lds + kFmLds + (wave * kFmRowsPerWave + r) * 256 +
                                                          rd * 128 + ch * 8)
                       : gv[rd - 2][it];
            *reinterpret_cast<bf16x4*>(ga.out + orow) = gate4_bf16_fast(v, g4);
          }
        } else if (t < q_tokens) {
          // nontemporal: the output is not re-read here (459.0 vs 460.0 us at 8K)
          __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(out + orow));
        }
      }
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
    }
  }
}

// Split-K combine: kG groups of 32 threads (8 dims each) merge the live
// chunks' partials of one (token, head) row, group g chunks g, g + kG, ...:
// M = max m_c, L = sum l_c 2^(m_c - M), O = sum O_c 2^(m_c - M) / L (chunks
// where the row saw no key have l = 0 and weigh nothing; a NaN l, from a
// non-finite key or query, is kept and makes the row NaN, as without a split),
// then the groups through LDS, in group order.  block = 512 = 16 / kG rows of 32 kG threads.
// A group's (m, l) pairs, its first four chunks' O partials and the gate
// are requested together (indices clamped to the live range, so every load
// is unconditional and in bounds): one memory round trip for up to four
// chunks a group, so the launch picks kG for at most four.  The reads bound
// it: 42 chunks of 93 tokens, 62 MB, 12.9 us (with 8 groups of up to 16
// chunks the split and combine took 62 us, with 16 of 4 they take 59).
constexpr int kCombineMaxChunks = 128;   // split_plan's most
template <int kG, int kMaxC>   // kMaxC: chunks per group at most, a multiple of 4
__global__ __launch_bounds__(512) void fmha_split_combine_kernel(
    const float* __restrict__ po, const float* __restrict__ pml, float* __restrict__ out,
    unsigned q_tokens, unsigned kv_tokens, unsigned tile_toks, unsigned chunk_keys,
    unsigned n_chunks, GateArgs ga) {
  constexpr unsigned kRowsHere = 16 / kG;
  __shared__ __attribute__((aligned(16))) float part[kG > 1 ? 512 : 1][8];
  __shared__ float2 part_ml[16];
  const unsigned g = (threadIdx.x >> 5) % kG;
  const unsigned rid = blockIdx.x * kRowsHere + (threadIdx.x >> 5) / kG;   // token * 16 + head
  const unsigned tok = rid / kHq, head = rid % kHq, kvh = head / kGroup;
  const unsigned qtile = tok / tile_toks, rows = tile_toks * kGroup;
  const unsigned r = (tok - qtile * tile_toks) * kGroup + head % kGroup;   // row of the tile
  const int d0 = 8 * (threadIdx.x & 31);
  const unsigned off = kv_tokens - q_tokens;
  const unsigned kv_end = min(kv_tokens, min((qtile + 1) * tile_toks, q_tokens) + off);
  const unsigned live = (kv_end + chunk_keys - 1) / chunk_keys;   // 1 .. n_chunks
  auto row_of = [&](unsigned c) {
    return (((size_t)qtile * n_chunks + min(c, live - 1)) * kHkv + kvh) * rows + r;
  };
  float2 ml[kMaxC];
#pragma unroll
  for (int c = 0; c < kMaxC; ++c)
    ml[c] = *reinterpret_cast<const float2*>(pml + row_of(g + kG * c) * 2);
  f32x4 oa[4], ob[4];
  auto load_o = [&](int c0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4* src = reinterpret_cast<const f32x4*>(po + row_of(g + kG * (c0 + j)) * kD + d0);
      oa[j] = src[0];
      ob[j] = src[1];
    }
  };
  load_o(0);
  // gated: the gate row (any valid address otherwise; the value is unused)
  const bf16* gp = ga.out != nullptr
                       ? ga.gate + (size_t)tok * ga.gate_stride + head * 2 * kD + kD + d0
                       : reinterpret_cast<const bf16*>(po + row_of(0) * kD + d0);
  const bf16x8 gv = *reinterpret_cast<const bf16x8*>(gp);
  __builtin_amdgcn_sched_barrier(0);
  float M = -INFINITY;
#pragma unroll
  for (int c = 0; c < kMaxC; ++c)
    if (g + kG * c < live && ml[c].y != 0.f) M = fmaxf(M, ml[c].x);
  float L = 0.f, acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int c0 = 0; c0 < kMaxC; c0 += 4) {
    if (g + kG * c0 >= live) break;
    if (c0 > 0) load_o(c0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float2 m_l = ml[c0 + j];
      if (g + kG * (c0 + j) < live && m_l.y != 0.f) {
        const float w = __builtin_amdgcn_exp2f(m_l.x - M);
        L += w * m_l.y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[e] += w * oa[j][e];
          acc[4 + e] += w * ob[j][e];
        }
      }
    }
  }
  if constexpr (kG > 1) {
    f32x4* mine = reinterpret_cast<f32x4*>(part[threadIdx.x]);
    mine[0] = f32x4{acc[0], acc[1], acc[2], acc[3]};
    mine[1] = f32x4{acc[4], acc[5], acc[6], acc[7]};
    if ((threadIdx.x & 31) == 0) part_ml[threadIdx.x >> 5] = float2{M, L};
    __syncthreads();
    if (g != 0) return;
    float m_all = M;   // key 0's chunk is live: some group has L != 0
#pragma unroll
    for (int j = 1; j < kG; ++j) m_all = fmaxf(m_all, part_ml[(threadIdx.x >> 5) + j].x);
    const float w0 = L != 0.f ? __builtin_amdgcn_exp2f(M - m_all) : 0.f;
    L *= w0;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= w0;
#pragma unroll
    for (int j = 1; j < kG; ++j) {
      const float2 m_l = part_ml[(threadIdx.x >> 5) + j];
      const float w = m_l.y != 0.f ? __builtin_amdgcn_exp2f(m_l.x - m_all) : 0.f;
      L += w * m_l.y;
      const f32x4* src = reinterpret_cast<const f32x4*>(part[threadIdx.x + 32 * j]);
      const f32x4 a = src[0], b = src[1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[e] += w * a[e];
        acc[4 + e] += w * b[e];
      }
    }
  }
  const float inv = 1.0f / L;
  if (ga.out != nullptr) {   // gated bf16 rows (see GateArgs)
    const bf16x4 lo = gate4_bf16_fast(f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv},
                                      bf16x4{gv[0], gv[1], gv[2], gv[3]});
    const bf16x4 hi = gate4_bf16_fast(f32x4{acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv},
                                      bf16x4{gv[4], gv[5], gv[6], gv[7]});
    *reinterpret_cast<bf16x8*>(ga.out + (size_t)tok * kQDim + head * kD + d0) =
        bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return;
  }
  f32x4* dst = reinterpret_cast<f32x4*>(out + (size_t)tok * kQDim + head * kD + d0);
  dst[0] = f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
  dst[1] = f32x4{acc[4] * inv, acc[5] * inv, acc[6] * inv, acc[7] * inv};
}

// Split-K scratch: room for kSplitItems (tile, chunk, KV head) partials of 256
// rows.  The reference's provider ABI has no workspace argument, so the
// provider owns one scratch per device (allocated by qrt_ck_fmha_prepare,
// kept until the process ends: graphs captured with a split launch hold its
// address).  The first split launch on a device claims that scratch for its
// stream; split launches on that stream are ordered by it, and launches on
// any other stream run unsplit (same results, slower for short prompts), so
// concurrent streams never share partials.  qwen36_fmha_prefill takes a
// caller workspace instead and splits on any stream.
constexpr unsigned kSplitItems = 512;
constexpr size_t kSplitItemBytes = (size_t)256 * (kD + 2) * sizeof(float);
constexpr size_t kSplitScratchBytes = kSplitItems * kSplitItemBytes;
constexpr int kFmMaxDevices = 64;
std::mutex g_fm_mutex;
struct ProviderScratch {
  void* ptr = nullptr;
  bool claimed = false;
  hipStream_t owner = nullptr;
};
ProviderScratch g_fm_scratch[kFmMaxDevices];

// The provider scratch if `stream` may use it (claiming it on first use).
void* provider_scratch_for(hipStream_t stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kFmMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_fm_mutex);
  ProviderScratch& ps = g_fm_scratch[dev];
  if (ps.ptr == nullptr) return nullptr;
  if (!ps.claimed) {
    ps.claimed = true;
    ps.owner = stream;
  }
  return ps.owner == stream ? ps.ptr : nullptr;
}

std::once_flag g_fm_attr_once;
hipError_t g_fm_attr_status = hipSuccess;

// Split plan for short prompts: too few query tiles to fill the GPU, so each
// tile's key range is cut into n chunks (a multiple of 32 keys; a tile's
// chunks past its last key exit at once), and few rows take smaller tiles.
// Swept on MI355X over 1 .. 8192 tokens, prefixes of 0 .. 64000 and n = 1 ..
// 128 (graph-replayed, gated):
//  * rows over a prefix: every tile has about the same work, so n makes about
//    one workgroup per CU, of at least 96 keys each (93 rows over 24000: n =
//    32 .. 42 60 us, 16 73, 64 70; 8 over 65000: 33 us at 128, 41 at 64, 50 at
//    32).  8 waves, whose tiles read K/V least often, from tokens x keys =
//    1.4 M (256 over 8000: 54 us against 55; 64 over 64000: 86 against 98),
//    4 waves below (93 over 8000: 34 us against 38), 2 waves below 0.2 M
//    (2 / 4 waves: 32 over 4000 18.8 us / 23.9, 93 over 1000 18.0 / 22.0, over 1500
//    21.0 / 23.7, over 2050 23.5 / 22.7, 128 over 1000 20.5 / 24.1, over 1400 22.5 / 25.4,
//    200 over 700 21.4 / 25.1; 200 over 2000, 0.44 M, 28 / 26.8).  Three and more tiles of 2 waves make
//    at most 192 workgroups (93 over 1500, n = 5 .. 8 21.0 us, 10 22.8; 128 over 1000,
//    n = 4 20.1, 8 21.9; 64 over 2000, n = 10 19.6, 17 20.9; two tiles, 12 over 9000,
//    n = 64 18.5, 40 19.5).
//    Where 8 waves are chosen, pairs of 4-wave halves (kSub = 2) halve the
//    partials' traffic (62 MB written and read back at 93 over 24000) but read
//    each key twice as often, so they pay while a half has at most about 1250
//    keys of at most 32768 and where their tiles fill at least 115 of the 128
//    workgroups per head.  Pairs / 8 waves of rows:
//      pay: 93 over 15000 40.2 us / 46.3, over 24000 50.9 / 56.6; 128 over 20000
//        55.0 / 63.3; 500 over 2800 42.4 / 47.7; 150 over 30000 (1180 keys) 81.1 / 86.5
//      keys: 93 over 50000 94.7 / 90.7; 500 over 60000 (7600 keys) 458 / 393
//      workgroups: 800 over 8000 (100 of 128) 117 / 111
//    They are taken from 6 tiles on, which is no measured limit: 5 tiles (65 to
//    80 tokens) would gain too (65 over 18000 41.3 / 41.2, 70 over 20000 42.4 /
//    46.0, 75 over 24000 46.3 / 50.6, 80 over 28000 53.1 / 56.6), 4 are not measured.
//    The items go to the XCDs in ranges where 2 to 12 tiles share chunks of
//    at least 12000 keys in all (with / without, 93 over 24000 51.9 / 54.7, 150
//    over 30000 82.0 / 87.1, 64 over 16000 35.6 / 39.2, 32 over 30000 35.7 / 39.0,
//    64 over 64000 82.8 / 86.9; one tile: 16 over 8000 25.5 / 22.8; more tiles:
//    256 over 8000 52.1 / 51.2, 1000 over 4000 91 / 85; short: 93 over 2000 26.1 /
//    23.9).
//    Up to 3072 rows two chunks still win (2500 over 4000: 219 us against
//    299 unsplit; 3500: 339 against 325).  Where the later chunks of the first tiles
//    hold no key, three chunks may still be at most one workgroup per CU and take
//    the place of two (1400 over 1000 65.5 us against 74.1, 1500 over 1500 77.2 /
//    83.3, 1900 over 256 64.2 / 69.3; with more: 2048 over 256, 136, 79.5 / 74.1, 1900
//    over 1000, 150, 90.4 / 88.3; 1700 over 1000, 136, would gain, 75.8 / 80.4).
//  * square prompts: later tiles hold more chunks, 2 tiles (n + 1) / 2 in
//    all, again about one per CU: n = 4 up to 42 tiles, 3 up to 66, then 2
//    (2048 tokens: 63 us at n = 3, 68 at 2, 86 at 4; 3072: 105 us at 2, 120
//    at 4, 134 unsplit) up to 4096 (166 us against 181; 4500: 204 against
//    200).  8-token tiles up to 360 tokens (256: 16 us against 17), 16-token
//    tiles up to 960 (768: 29 us against 33; 1000: 37 against 36).
//  * few rows over few keys (48 tokens, 1024 keys): a wave's rows and, gated, its
//    256 gate values a row are a serial chain, so tiles of one wave (4 tokens)
//    and, over a prefix, chunks of 32 keys up to 8 rows and 64 above (gated, 1
//    wave / 2 waves and 96 keys / tiles of 256 rows of one head: 4 over 300 8.3 us /
//    10.2 / 8.9, 8 over 500 9.5 / 11.9 / 12.1, 24 over 256 9.8 / 12.5 / 12.8, 40 8.2 /
//    9.5 / 9.3, 48 over 500 12.8 / 13.6 / 17.0; only 2 to 12 rows over some 40 keys are
//    still behind the last, 7.8 / 9.1 / 7.2).  Up to 32 keys there is one chunk; the
//    plain form then runs unsplit (6 us), the gated one, whose rows would be gated
//    by a wave or two, still leaves them to the combine (split and combine /
//    unsplit / one head a workgroup: 1 token 7.0 / 7.3 / 7.2, 8 8.0 / 14.8 / 8.5, 16
//    8.1 / 15.8 / 10.5, 32 8.2 / 21.0 / 15.0).
struct SplitPlan {
  unsigned waves, sub, tiles, n_chunks, chunk_keys, ranges, items;   // items: (tile, chunk, KV head) partials
};
constexpr unsigned kFewRows = 48, kFewKeys = 1024;

unsigned tile_tokens(unsigned waves) { return waves * kFmRowsPerWave / kGroup; }

SplitPlan split_plan(unsigned q_tokens, unsigned kv_tokens) {
  SplitPlan p{};
  p.sub = 1u;
  p.n_chunks = 1u;
  p.chunk_keys = kv_tokens;
  const bool square = kv_tokens - q_tokens < 256u;
  if (q_tokens > (square ? 4096u : 3072u)) return p;
  const size_t work = (size_t)q_tokens * kv_tokens;
  const bool few = q_tokens <= kFewRows && kv_tokens <= kFewKeys;
  if (few)
    p.waves = 1u;
  else if (square)
    p.waves = q_tokens <= 360u ? 2u : q_tokens <= 960u ? 4u : 8u;
  else
    p.waves = work <= 200000u ? 2u : work <= 1400000u ? 4u : 8u;
  const unsigned pairs = (q_tokens + tile_tokens(4u) - 1) / tile_tokens(4u);
  if (!square && p.waves == 8u && pairs >= 6u && pairs <= 42u && 128u / pairs * pairs >= 115u &&
      kv_tokens <= 32768u && (size_t)pairs * kv_tokens <= 1250u * 256u) {
    p.waves = 4u;
    p.sub = 2u;
  }
  p.tiles = (q_tokens + tile_tokens(p.waves) - 1) / tile_tokens(p.waves);
  unsigned n;
  if (square) {
    n = p.tiles <= 42u ? 4u : p.tiles <= 66u ? 3u : 2u;
  } else {
    n = std::min((p.waves == 2u && p.tiles > 2u ? 96u : 128u) / p.tiles,
                 !few             ? kv_tokens / 96u
                 : q_tokens <= 8u ? (kv_tokens + 31u) / 32u
                                  : (kv_tokens + 63u) / 64u);
    n = std::max(2u, std::min(n, (unsigned)kCombineMaxChunks));
  }
  const unsigned quantum = kFmKv * p.sub;
  auto chunk_of = [&](unsigned chunks) {
    return ((kv_tokens + chunks - 1) / chunks + quantum - 1) / quantum * quantum;
  };
  if (!square && n == 2u) {
    unsigned live = 0;   // (tile, chunk) items of three chunks that hold a key
    for (unsigned i = 1; i <= p.tiles; ++i)
      live += (std::min(i * tile_tokens(p.waves), q_tokens) + kv_tokens - q_tokens + chunk_of(3u) - 1) /
              chunk_of(3u);
    if (live <= 128u) n = 3u;
  }
  const unsigned chunk = chunk_of(n);
  n = (kv_tokens + chunk - 1) / chunk;   // after rounding up
  if (n < 2u && !few) return p;
  p.n_chunks = n;
  p.chunk_keys = chunk;
  p.ranges = !square && p.tiles > 1u && p.tiles <= 12u && kv_tokens >= 12000u;
  p.items = p.tiles * n * kHkv;          // at most kSplitItems
  return p;
}

// One size serves every split of up to 2560 tokens, so a buffer that one of them
// sized is enough for the others, whatever their length and prefix (a shared buffer
// does not grow during a capture).  The most is 66 tiles of 32 tokens in 3 chunks
// for 2 KV heads: square prompts make at most 42 x 4, 66 x 3 or 80 x 2 (tile, chunk)
// pairs, rows over a prefix at most 128 or 80 x 2.  Longer prompts take at least as much.
constexpr size_t kSplitSharedBytes = 66 * 3 * kHkv * kSplitItemBytes;

size_t split_workspace_bytes(const SplitPlan& p) {
  const size_t exact = (size_t)p.items * (p.waves * p.sub * kFmRowsPerWave) * (kD + 2) * sizeof(float);
  return p.n_chunks > 1 ? std::max(kSplitSharedBytes, exact) : exact;   // (one chunk: at most 516 KB)
}

// Whether the call may run with this workspace, and whether it then splits.
// Without enough of it, calls of up to 2560 tokens are refused; longer ones (they
// do not need the split to fill the GPU) and those of one chunk run unsplit.
bool split_workspace_ok(unsigned q_tokens, unsigned kv_tokens, const void* workspace,
                        size_t workspace_bytes, bool* split) {
  const SplitPlan plan = split_plan(q_tokens, kv_tokens);
  const size_t need = split_workspace_bytes(plan);
  const bool enough = workspace != nullptr && workspace_bytes >= need;
  *split = need > 0 && enough;
  return need == 0 || enough || q_tokens > 2560u || plan.n_chunks < 2u;
}

bool valid_geometry(const void* q, const void* k, const void* v, const float* out,
                    unsigned q_tokens, unsigned kv_tokens) {
  return q != nullptr && k != nullptr && v != nullptr && out != nullptr && q_tokens != 0u &&
         q_tokens <= kMaxTokens && kv_tokens >= q_tokens && kv_tokens <= kMaxTokens;
}

// `scratch` null: run unsplit.  `ga.out` non-null: gated bf16 output (and
// `out` unused).
int launch_fmha(const void* q, const void* k, const void* v, float* out,
                unsigned q_tokens, unsigned kv_tokens, void* scratch, hipStream_t stream,
                const GateArgs& ga = GateArgs{nullptr, 0u, nullptr}) {
  std::call_once(g_fm_attr_once, [] {
    for (const void* f : {reinterpret_cast<const void*>(fmha_prefill_kernel<8, false>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<4, false>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<2, false>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<8, true>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<4, true>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<2, true>),
                          reinterpret_cast<const void*>(fmha_prefill_kernel<1, true>)}) {
      const hipError_t e =
          hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kFmLds);
      if (e != hipSuccess) g_fm_attr_status = e;
    }
    hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(fmha_prefill_kernel<4, true, false, 2>),
        hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kFmLds);
    if (e != hipSuccess) g_fm_attr_status = e;
    e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(fmha_prefill_kernel<8, false, true>),
        hipFuncAttributeMaxDynamicSharedMemorySize, kFmLdsGated);
    if (e != hipSuccess) g_fm_attr_status = e;
  });
  if (g_fm_attr_status != hipSuccess) return (int)g_fm_attr_status;
  const bf16* qb = static_cast<const bf16*>(q);
  const bf16* kb = static_cast<const bf16*>(k);
  const bf16* vb = static_cast<const bf16*>(v);
  const SplitPlan plan = split_plan(q_tokens, kv_tokens);
  const bool one_chunk = plan.items > 0 && plan.n_chunks == 1;
  if (scratch != nullptr && (plan.n_chunks > 1 || (one_chunk && ga.out != nullptr))) {
    SplitArgs sp;
    sp.o = static_cast<float*>(scratch);
    sp.ml = sp.o + (size_t)plan.items * (plan.waves * kFmRowsPerWave) * kD;   // after the O partials
    sp.chunk_keys = plan.chunk_keys;
    sp.n_chunks = plan.n_chunks;
    sp.ranges = plan.ranges;
    auto split = plan.sub == 2     ? fmha_prefill_kernel<4, true, false, 2>
                 : plan.waves == 8 ? fmha_prefill_kernel<8, true>
                 : plan.waves == 4 ? fmha_prefill_kernel<4, true>
                 : plan.waves == 2 ? fmha_prefill_kernel<2, true>
                                   : fmha_prefill_kernel<1, true>;
    hipLaunchKernelGGL(split, dim3(8 * ((plan.tiles * plan.n_chunks + 3) / 4)),
                       dim3(64 * plan.waves * plan.sub), kFmLds * plan.sub, stream, qb, kb, vb, out, q_tokens, kv_tokens,
                       plan.tiles, sp, ga);
    // groups of 32 threads per row: at most 4 chunks (one round trip) a group,
    // 8 past 64 chunks
    unsigned groups = 16;
    auto combine = fmha_split_combine_kernel<16, kCombineMaxChunks / 16>;
    if (plan.n_chunks <= 4) {
      groups = 1;
      combine = fmha_split_combine_kernel<1, 4>;
    } else if (plan.n_chunks <= 8) {
      groups = 2;
      combine = fmha_split_combine_kernel<2, 4>;
    } else if (plan.n_chunks <= 16) {
      groups = 4;
      combine = fmha_split_combine_kernel<4, 4>;
    } else if (plan.n_chunks <= 32) {
      groups = 8;
      combine = fmha_split_combine_kernel<8, 4>;
    } else if (plan.n_chunks <= 64) {
      combine = fmha_split_combine_kernel<16, 4>;
    }
    hipLaunchKernelGGL(combine, dim3(q_tokens * groups), dim3(512), 0, stream, sp.o, sp.ml,
                       out, q_tokens, kv_tokens, tile_tokens(plan.waves), plan.chunk_keys,
                       plan.n_chunks, ga);
    return static_cast<int>(hipGetLastError());
  }
  const SplitArgs none{nullptr, nullptr, 0u, 1u, 0u};
  auto tiles = [&](unsigned waves) { return (q_tokens + tile_tokens(waves) - 1) / tile_tokens(waves); };
  auto grid = [&](unsigned waves) { return dim3(8 * ((tiles(waves) + 3) / 4)); };
  if (ga.out != nullptr) {   // gated: 256-row workgroups at every length
    hipLaunchKernelGGL((fmha_prefill_kernel<8, false, true>), grid(8), dim3(512),
                       kFmLdsGated, stream, qb, kb, vb, out, q_tokens, kv_tokens, tiles(8), none, ga);
    return static_cast<int>(hipGetLastError());
  }
  // Rows per workgroup without a split: 256 (8 waves) when that gives at
  // least 256 workgroups or the rows extend a cached prefix (long rows); short
  // square prompts, and rows over one tile of keys (16 over 16: 5.8 us, 7.1 with 8
  // waves), use 128 or 64 rows so they still spread over the CUs.
  if (2 * tiles(8) >= 256u || (kv_tokens > q_tokens && !one_chunk)) {
    hipLaunchKernelGGL((fmha_prefill_kernel<8, false>), grid(8), dim3(512), kFmLds, stream,
                       qb, kb, vb, out, q_tokens, kv_tokens, tiles(8), none, ga);
  } else if (2 * tiles(4) >= 256u) {
    hipLaunchKernelGGL((fmha_prefill_kernel<4, false>), grid(4), dim3(256), kFmLds, stream,
                       qb, kb, vb, out, q_tokens, kv_tokens, tiles(4), none, ga);
  } else {
    hipLaunchKernelGGL((fmha_prefill_kernel<2, false>), grid(2), dim3(128), kFmLds, stream,
                       qb, kb, vb, out, q_tokens, kv_tokens, tiles(2), none, ga);
  }
  return static_cast<int>(hipGetLastError());
}

int provider_launch(const void* q, const void* k, const void* v, float* out,
                    unsigned q_tokens, unsigned kv_tokens, hipStream_t stream) {
  if (!valid_geometry(q, k, v, out, q_tokens, kv_tokens)) return Q36_EINVAL;
  void* scratch = split_plan(q_tokens, kv_tokens).n_chunks > 1 ? provider_scratch_for(stream)
                                                                : nullptr;
  return launch_fmha(q, k, v, out, q_tokens, kv_tokens, scratch, stream);
}

}  // namespace
}  // namespace q36

// ---- provider ABI ---------------------------------------------------------
// prepare allocates the split-K scratch on the current device (once, 132 MiB);
// it stays allocated until the process ends -- a graph captured with a split
// launch holds its address -- so release has nothing to free.

// Returns 0 for a valid token count, hipErrorInvalidValue otherwise (the
// reference's contract); if the scratch cannot be allocated (no device, out
// of memory) the provider simply stays without it and launches run unsplit.
Q36_EXPORT int qrt_ck_fmha_prepare(unsigned tokens) {
  if (tokens == 0u || tokens > q36::kMaxTokens) return Q36_EINVAL;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= q36::kFmMaxDevices) {
    (void)hipGetLastError();
    return Q36_OK;
  }
  std::lock_guard<std::mutex> lock(q36::g_fm_mutex);
  q36::ProviderScratch& ps = q36::g_fm_scratch[dev];
  if (ps.ptr == nullptr && hipMalloc(&ps.ptr, q36::kSplitScratchBytes) != hipSuccess) {
    ps.ptr = nullptr;
    (void)hipGetLastError();
  }
  return Q36_OK;
}

Q36_EXPORT int qrt_ck_fmha_bf16_launch(const void* q, const void* k,
                                       const void* v, float* out,
                                       unsigned tokens, void* stream) {
  return q36::provider_launch(q, k, v, out, tokens, tokens,
                              static_cast<hipStream_t>(stream));
}

Q36_EXPORT int qrt_ck_fmha_bf16_launch_ex(const void* q, const void* k,
                                          const void* v, float* out,
                                          unsigned query_tokens,
                                          unsigned kv_tokens, void* stream) {
  return q36::provider_launch(q, k, v, out, query_tokens, kv_tokens,
                              static_cast<hipStream_t>(stream));
}

Q36_EXPORT int qrt_ck_fmha_release(void) { return Q36_OK; }

// Legacy fixed-shape q8192 exports (qrt_ck_fmha_q8192_provider.cpp:214-300).
// The fp32-packed launch takes rows of [q (4096) | 4096 more q_proj features
// | k (512) | v (512)] fp32 (9216 per token, the q_proj + k_proj + v_proj
// outputs side by side), rounds q, k and v to bf16 into provider staging
// (q8192_prepare allocates it, 80 MiB per device; q8192_release frees it),
// and runs the square causal attention over the staged tensors.
namespace q36 {
namespace {
constexpr unsigned kQ8192 = 8192u;
constexpr unsigned kPackedRow = 2u * kQDim + 2u * kKvRow;   // 9216

// thread = 8 consecutive features of one token's q, k or v
__global__ __launch_bounds__(256) void fmha_pack_q8192_kernel(const float* __restrict__ packed,
                                                             bf16* __restrict__ qs,
                                                             bf16* __restrict__ ks,
                                                             bf16* __restrict__ vs) {
  constexpr unsigned kPerTok = (kQDim + 2u * kKvRow) / 8u;   // 640 octets per token
  const unsigned idx = blockIdx.x * 256u + threadIdx.x;
  if (idx >= kQ8192 * kPerTok) return;
  const unsigned tok = idx / kPerTok, o = idx % kPerTok;
  const float* src;
  bf16* dst;
  if (o < kQDim / 8u) {
    src = packed + (size_t)tok * kPackedRow + 8u * o;
    dst = qs + (size_t)tok * kQDim + 8u * o;
  } else if (o < (kQDim + kKvRow) / 8u) {
    const unsigned f = 8u * o - kQDim;
    src = packed + (size_t)tok * kPackedRow + 2u * kQDim + f;
    dst = ks + (size_t)tok * kKvRow + f;
  } else {
    const unsigned f = 8u * o - kQDim - kKvRow;
    src = packed + (size_t)tok * kPackedRow + 2u * kQDim + kKvRow + f;
    dst = vs + (size_t)tok * kKvRow + f;
  }
  const f32x4 a = reinterpret_cast<const f32x4*>(src)[0];
  const f32x4 b = reinterpret_cast<const f32x4*>(src)[1];
  // round to nearest even (NaN stays NaN), as the provider's packing does
  *reinterpret_cast<bf16x8*>(dst) = bf16x8{f2bf(a[0]), f2bf(a[1]), f2bf(a[2]), f2bf(a[3]),
                                           f2bf(b[0]), f2bf(b[1]), f2bf(b[2]), f2bf(b[3])};
}

struct Q8192Staging {
  bf16* q = nullptr;
  bf16* k = nullptr;
  bf16* v = nullptr;
};
Q8192Staging g_q8192[kFmMaxDevices];

// Allocates the current device's staging if absent (caller holds g_fm_mutex).
int q8192_prepare_locked(int dev) {
  Q8192Staging& st = g_q8192[dev];
  if (st.q != nullptr) return Q36_OK;
  const size_t qb = (size_t)kQ8192 * kQDim * 2, kvb = (size_t)kQ8192 * kKvRow * 2;
  void *q = nullptr, *k = nullptr, *v = nullptr;
  hipError_t e = hipMalloc(&q, qb);
  if (e == hipSuccess) e = hipMalloc(&k, kvb);
  if (e == hipSuccess) e = hipMalloc(&v, kvb);
  if (e != hipSuccess) {
    (void)hipFree(q);
    (void)hipFree(k);
    (void)hipFree(v);
    return static_cast<int>(e);
  }
  st.q = static_cast<bf16*>(q);
  st.k = static_cast<bf16*>(k);
  st.v = static_cast<bf16*>(v);
  return Q36_OK;
}

int current_device(int* dev) {
  if (hipGetDevice(dev) != hipSuccess || *dev < 0 || *dev >= kFmMaxDevices) {
    (void)hipGetLastError();
    return static_cast<int>(hipErrorInvalidDevice);
  }
  return Q36_OK;
}
}  // namespace
}  // namespace q36

Q36_EXPORT int qrt_ck_fmha_q8192_prepare(void) {
  int dev = 0;
  const int e = q36::current_device(&dev);
  if (e != Q36_OK) return e;
  std::lock_guard<std::mutex> lock(q36::g_fm_mutex);
  return q36::q8192_prepare_locked(dev);
}

Q36_EXPORT int qrt_ck_fmha_q8192_f32_launch(const float* packed_qkv, float* out, void* stream) {
  if (packed_qkv == nullptr || out == nullptr) return Q36_EINVAL;
  int dev = 0;
  int e = q36::current_device(&dev);
  if (e != Q36_OK) return e;
  q36::Q8192Staging st;
  {
    std::lock_guard<std::mutex> lock(q36::g_fm_mutex);
    e = q36::q8192_prepare_locked(dev);
    if (e != Q36_OK) return e;
    st = q36::g_q8192[dev];
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  constexpr unsigned kThreads = q36::kQ8192 * ((q36::kQDim + 2u * q36::kKvRow) / 8u);
  hipLaunchKernelGGL(q36::fmha_pack_q8192_kernel, dim3((kThreads + 255u) / 256u), dim3(256), 0,
                     s, packed_qkv, st.q, st.k, st.v);
  const hipError_t le = hipGetLastError();
  if (le != hipSuccess) return static_cast<int>(le);
  return q36::provider_launch(st.q, st.k, st.v, out, q36::kQ8192, q36::kQ8192, s);
}

Q36_EXPORT int qrt_ck_fmha_q8192_bf16_launch(const void* q, const void* k,
                                             const void* v, float* out,
                                             void* stream) {
  return q36::provider_launch(q, k, v, out, 8192u, 8192u,
                              static_cast<hipStream_t>(stream));
}

// Frees the fp32 path's staging (the caller has finished every launch that
// uses it, as with the reference's release).
Q36_EXPORT int qrt_ck_fmha_q8192_release(void) {
  int dev = 0;
  if (q36::current_device(&dev) != Q36_OK) return Q36_OK;
  std::lock_guard<std::mutex> lock(q36::g_fm_mutex);
  q36::Q8192Staging& st = q36::g_q8192[dev];
  (void)hipFree(st.q);
  (void)hipFree(st.k);
  (void)hipFree(st.v);
  st = q36::Q8192Staging{};
  return Q36_OK;
}

// ---- workspace form (no counterpart in the reference's provider ABI) -------
Q36_EXPORT size_t qwen36_fmha_prefill_workspace_bytes(unsigned query_tokens,
                                                      unsigned kv_tokens) {
  if (query_tokens == 0u || query_tokens > q36::kMaxTokens || kv_tokens < query_tokens ||
      kv_tokens > q36::kMaxTokens)
    return 0;
  return q36::split_workspace_bytes(q36::split_plan(query_tokens, kv_tokens));
}

Q36_EXPORT int qwen36_fmha_prefill(const void* q, const void* k, const void* v, float* out,
                                   unsigned query_tokens, unsigned kv_tokens, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  if (!q36::valid_geometry(q, k, v, out, query_tokens, kv_tokens)) return Q36_EINVAL;
  bool split = false;
  if (!q36::split_workspace_ok(query_tokens, kv_tokens, workspace, workspace_bytes, &split))
    return Q36_EINVAL;
  return q36::launch_fmha(q, k, v, out, query_tokens, kv_tokens, split ? workspace : nullptr,
                          static_cast<hipStream_t>(stream));
}

Q36_EXPORT int qwen36_fmha_prefill_gated(const void* q, const void* k, const void* v,
                                         const void* q_gate, unsigned q_gate_row_stride,
                                         void* out, unsigned query_tokens, unsigned kv_tokens,
                                         void* workspace, size_t workspace_bytes, void* stream) {
  // (out stands in for the fp32 pointer in the geometry check)
  if (!q36::valid_geometry(q, k, v, static_cast<const float*>(out), query_tokens, kv_tokens) ||
      q_gate == nullptr || q_gate_row_stride < 2u * q36::kQDim ||
      (reinterpret_cast<uintptr_t>(q_gate) & 7u) != 0 || (q_gate_row_stride & 7u) != 0 ||
      (reinterpret_cast<uintptr_t>(out) & 15u) != 0)
    return Q36_EINVAL;
  bool split = false;
  if (!q36::split_workspace_ok(query_tokens, kv_tokens, workspace, workspace_bytes, &split))
    return Q36_EINVAL;
  const q36::GateArgs ga{static_cast<const q36::bf16*>(q_gate), q_gate_row_stride,
                         static_cast<q36::bf16*>(out)};
  return q36::launch_fmha(q, k, v, nullptr, query_tokens, kv_tokens,
                          split ? workspace : nullptr, static_cast<hipStream_t>(stream), ga);
}
