// Grouped expert GEMMs of the MoE block for short prompts, where an expert
// has few rows and the call is a stream of expert weights.
//
// A workgroup computes one tile of up to 64 rows of one group against 128
// weight rows at a time, K in steps of 64, with 8 waves of one 32 x 32 block
// each (v_mfma_f32_32x32x16_bf16); gate/up workgroups own 64 act columns (gate
// and up rows of 16 columns side by side in each wave's 32 weight rows, so the
// SiLU is formed in registers), down workgroups `subs` blocks of 128 output
// columns, one continuous stream of steps.  Both operands go straight into LDS
// (buffer_load ... lds), a 3-stage ring of 24 KiB, two workgroups per CU:
// whole 128-byte lines of each weight row a step, two steps in flight.
//
// HBM-bound.  A copy of the fetch loop alone (no operand reads) streams 1 GiB
// of weights on MI355X at 6.1 TB/s as 64-byte pieces of 256 rows (the
// long-prompt GEMM's step), 6.3 as 128-byte pieces and 6.9 as 128-byte pieces
// with the nontemporal hint; a group of one tile, whose weights are read once,
// takes the hint, larger groups leave their weights to the L2 for the
// next tile (T = 1000, whole block: 343 us; no hints 371, hints everywhere
// 349).  At T = 1000 gate/up takes 184 us (1.07 GB, 5.8 TB/s; the 128-row
// kernel 214) and down 118 (130); the stores of down's rows are 22 us of it.
#pragma once
#include "moe_common.h"

namespace q36 {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kStBM = 64;                  // rows per tile (at most)
constexpr int kStBN = 128;                 // weight rows per block
constexpr int kStRowB = 128;               // bytes per row and step (64 K)
constexpr int kStStages = 3;
constexpr int kStStage = (kStBM + kStBN) * kStRowB;
constexpr int kStLds = kStStages * kStStage;      // 72 KiB
constexpr int kStIns = kStStage / 1024 / 8;       // fetch instructions per wave and step
constexpr int kStGateUpBlocks = kMoeInter / (kStBN / 2);
constexpr int kStDownBlocks = kMoeHidden / kStBN;

struct StreamArgs {
  const bf16* a;          // gate/up: h2 [T, 2048]; down: act [rows, 512]
  const bf16* w;          // expert_gate_up / expert_down
  const bf16* w_shared;   // group E: the shared expert's
  const int4* meta;       // [0].x tiles; [1 + i] = {group, first row, rows, tiles of the group}
  const int* sorted;      // slot of each row: t * 8 + k, or 8 T + t (shared)
  const float* rw;        // routing weight of each routed slot (long prompts' down)
  bf16* out;              // act [rows, 512] / y [9 T, 2048]
  unsigned T, E, subs;    // subs (down): 128-column blocks per workgroup
};

// Buffer resource over `bytes` bytes: reads past them give zeros.
__device__ __forceinline__ u32x4 stream_rsrc(const void* base, unsigned bytes) {
  const unsigned long long a = reinterpret_cast<unsigned long long>(base);
  return u32x4{(unsigned)a, (unsigned)(a >> 32), bytes, 0x00020000u};
}
constexpr unsigned kStOob = 0x80000000u;   // an offset past every buffer's range

// One 1 KiB fetch into LDS, with or without the nontemporal hint.  The
// leading s_nop covers a hazard the compiler cannot see through the
// inline assembly: the resource SGPRs (and m0) are written by VALU
// readfirstlane / SALU instructions right before, and a VMEM instruction
// reading an SGPR that a VALU wrote needs 5 wait states on gfx950 (issued
// earlier, it reads the old descriptor).
template <bool kNt>
__device__ __forceinline__ void stream_fetch(unsigned lds_addr, int voff, const u32x4& rsrc) {
  if constexpr (kNt)
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen nt lds"
                 :: "v"(voff), "s"(rsrc), "{m0}"(__builtin_amdgcn_readfirstlane(lds_addr))
                 : "memory");
  else
    asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                 :: "v"(voff), "s"(rsrc), "{m0}"(__builtin_amdgcn_readfirstlane(lds_addr))
                 : "memory");
}

// v of the lane beside (lane ^ 1), by DPP.
__device__ __forceinline__ float beside(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
}

// s_waitcnt immediate: at most n vector-memory operations outstanding.
constexpr int stream_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// One dword per lane, dropped where the offset is out of range.
__device__ __forceinline__ void stream_store(unsigned v, int voff, const u32x4& rsrc) {
  asm volatile("s_nop 4\n\tbuffer_store_dword %0, %1, %2, 0 offen" :: "v"(v), "v"(voff), "s"(rsrc) : "memory");
}

// Stage layout: 64 A rows then 128 weight rows of 128 bytes, the 16-byte
// chunk c of stage row r at position c ^ ((r / 2) % 8), so the 16 rows one
// ds_read_b128 pass serves fall in 16 distinct bank groups.
template <bool kDown>
__global__ __launch_bounds__(512, 4) void moe_stream_kernel(StreamArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int K = kDown ? kMoeInter : kMoeHidden;
  constexpr int kSteps = K * 2 / kStRowB;              // per block: 8 or 32
  const unsigned nb = kDown ? kStDownBlocks / p.subs : (unsigned)kStGateUpBlocks;
  const unsigned items = (unsigned)p.meta[0].x * nb;
  // items are dealt to the 8 XCDs in contiguous ranges: the blocks of a tile
  // and the tiles of a group share an L2
  const unsigned share = (items + 7) / 8, xi = blockIdx.x >> 3;
  const unsigned item = (blockIdx.x & 7) * share + xi;
  if (xi >= share || item >= items) return;
  const unsigned mt = item / nb, nt = item % nb;
  const int4 m = p.meta[1 + mt];
  const int group = m.x, row0 = m.y, rows = m.z;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const unsigned routed = kMoeTopK * p.T;

  u32x4 ars, brs, yrs;
  const bf16* wg = group < (int)p.E ? p.w + (size_t)group * (kDown ? 1 : 2) * kMoeInter * kMoeHidden
                                    : p.w_shared;
  brs = stream_rsrc(wg, (kDown ? 1u : 2u) * kMoeInter * kMoeHidden * 2u);
  yrs = stream_rsrc(p.out, kDown ? 9u * p.T * (unsigned)kMoeHidden * 2u : 0u);
  if constexpr (kDown)
    ars = stream_rsrc(p.a + (size_t)row0 * kMoeInter, (unsigned)rows * kMoeInter * 2u);
  else
    ars = stream_rsrc(p.a, p.T * (unsigned)kMoeHidden * 2u);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    ars[c] = __builtin_amdgcn_readfirstlane(ars[c]);
    brs[c] = __builtin_amdgcn_readfirstlane(brs[c]);
    yrs[c] = __builtin_amdgcn_readfirstlane(yrs[c]);
  }

  // Fetch plan: instruction i of a step fills stage rows 8i .. 8i + 7 (A
  // first), lane = row in the instruction x chunk position; a wave issues
  // instructions kStIns * wave + j.  Rows past the tile's end are fetched
  // out of range (nothing is read).
  const int rin = lane >> 3, cpos = lane & 7;
  unsigned f_off[kStIns];
#pragma unroll
  for (int j = 0; j < kStIns; ++j) {
    const int srow = 8 * (kStIns * wave + j) + rin;
    unsigned off;
    if (srow < kStBM) {
      if constexpr (kDown) {
        off = srow < rows ? (unsigned)srow * kMoeInter * 2u : kStOob;
      } else {
        const int slot = srow < rows ? p.sorted[row0 + srow] : -1;
        const unsigned t = (unsigned)slot < routed ? (unsigned)slot / kMoeTopK : (unsigned)slot - routed;
        off = slot < 0 ? kStOob : t * (unsigned)kMoeHidden * 2u;
      }
    } else {
      const int r = srow - kStBM;
      unsigned row;
      if constexpr (kDown)
        row = nt * p.subs * kStBN + r;
      else   // 16 gate rows, then the same 16 columns' up rows, per 32
        row = ((r & 16) ? kMoeInter : 0) + nt * (kStBN / 2) + 16 * (r >> 5) + (r & 15);
      off = row * (unsigned)K * 2u;
    }
    f_off[j] = off + ((cpos ^ ((srow / 2) % 8)) * 16);
  }
  const unsigned lds0 = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));
  const unsigned steps = kDown ? p.subs * kSteps : kSteps;
  const bool nt_hint = m.w == 1;
  unsigned f_step = 0, f_stage = 0;   // next step to fetch and its ring slot
  auto fetch = [&]() {
    // step s: K offset (s % kSteps) rows bytes, weight block s / kSteps
    const unsigned ka = (f_step % kSteps) * kStRowB;
    const unsigned kb = kDown ? ka + (f_step / kSteps) * (unsigned)(kStBN * K * 2) : ka;
    const unsigned base = lds0 + f_stage * kStStage;
#pragma unroll
    for (int j = 0; j < kStIns; ++j) {
      const int ins = kStIns * wave + j;   // wave-uniform: A or weight rows
      if (ins < kStBM / 8)
        stream_fetch<false>(base + ins * 1024, (int)(f_off[j] + ka), ars);
      else if (nt_hint)
        stream_fetch<true>(base + ins * 1024, (int)(f_off[j] + kb), brs);
      else
        stream_fetch<false>(base + ins * 1024, (int)(f_off[j] + kb), brs);
    }
    ++f_step;
    f_stage = f_stage + 1 == kStStages ? 0 : f_stage + 1;
  };

#pragma unroll
  for (int st = 0; st < kStStages - 1; ++st) fetch();

  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 31, kh = lane >> 5;
  const int arow = (32 * wm + li) * kStRowB, brow = (kStBM + 32 * wn + li) * kStRowB;
  int koff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) koff[s] = ((2 * s + kh) ^ ((li / 2) % 8)) * 16;
  const bool live = 32 * wm < rows;

  // Down: where this lane's rows go.  Lanes 2c and 2c + 1 exchange halves of
  // their accumulators, so each stores two adjacent columns of 8 rows
  // (dwords) instead of one of 16; row 2j + (lane & 1) of the 16 is this
  // lane's j-th.  Rows past the tile's end are stored out of range.
  constexpr int kStores = kDown ? 8 : 0;
  unsigned y_off[kDown ? 8 : 1];
  if constexpr (kDown) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = 2 * j + (li & 1);
      const int r = 32 * wm + 8 * (i >> 2) + 4 * kh + (i & 3);
      const int slot = r < rows ? p.sorted[row0 + r] : -1;
      y_off[j] = slot < 0 ? kStOob : (unsigned)slot * (kMoeHidden * 2u);
    }
  }

  f32x16 acc = f32x16{};
  unsigned stage = 0;
  for (unsigned step = 0; step < steps; ++step) {
    // this wave's fetches of `step` landed (the next step's may be in flight,
    // and so may the stores of a block that ended one or two steps ago: every
    // live wave issues exactly kStores of them)
    const unsigned ago = step % kSteps;
    if (step + 1 >= steps)
      __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));
    else if (kDown && live && step >= (unsigned)kSteps && ago < 2)
      __builtin_amdgcn_s_waitcnt(stream_vmcnt(kStIns + kStores));
    else
      __builtin_amdgcn_s_waitcnt(stream_vmcnt(kStIns));
    __syncthreads();   // every wave's fetches landed; the slot read last step is free
    if (step + kStStages - 1 < steps) fetch();
    const char* st = lds + stage * kStStage;
    stage = stage + 1 == kStStages ? 0 : stage + 1;
    if (live) {
      bf16x8 a[4], b[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        a[s] = *reinterpret_cast<const bf16x8*>(st + arow + koff[s]);
        b[s] = *reinterpret_cast<const bf16x8*>(st + brow + koff[s]);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = mfma32x32x16(a[s], b[s], acc);
    }
    if constexpr (kDown) {
      if ((step + 1) % kSteps == 0 && live) {   // one block of 128 columns done
        const unsigned c = (nt * p.subs + step / kSteps) * kStBN + 32 * wn + (li & 30);
        const bool odd = (li & 1) != 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float keep = odd ? acc[2 * j + 1] : acc[2 * j];
          const float got = beside(odd ? acc[2 * j] : acc[2 * j + 1]);
          const bf16x2 v = {f2bf(odd ? got : keep), f2bf(odd ? keep : got)};
          stream_store(__builtin_bit_cast(unsigned, v), (int)(y_off[j] + 2 * c), yrs);
        }
        acc = f32x16{};
      }
    }
  }
  if constexpr (!kDown) {
    if (!live) return;
    // lane li < 16 holds gate, li + 16 up of act column nt * 64 + 16 wn + li:
    // the low lanes finish rows of acc[0..7], the high lanes acc[8..15]
    const bool hi = (li & 16) != 0;
    const unsigned c = nt * (kStBN / 2) + 16 * wn + (li & 15);
    float g8[8], u8[8];
    bf16 a8[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float other = __shfl_xor(hi ? acc[i] : acc[i + 8], 16, 64);
      g8[i] = bf2f(f2bf(hi ? other : acc[i]));
      u8[i] = bf2f(f2bf(hi ? acc[i + 8] : other));
    }
    silu_mul8(g8, u8, a8);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int q = hi ? i + 8 : i;
      const int r = 32 * wm + 8 * (q >> 2) + 4 * kh + (q & 3);
      if (r < rows) p.out[(size_t)(row0 + r) * kMoeInter + c] = a8[i];
    }
  }
}

}  // namespace
}  // namespace q36
