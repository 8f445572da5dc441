// Grouped expert GEMMs of the MoE block for long prompts.
//
// A workgroup of 16 waves (four per SIMD, one workgroup per CU) computes one
// tile of up to 256 rows of one group against 256 weight rows (gate/up: 128
// gate rows and the same columns' up rows), K in steps of 64; wave (wm, wn)
// owns the 32-row blocks wm and wm + 4 and 64 of the weight rows on
// v_mfma_f32_32x32x16_bf16, so each SIMD holds every wm.  Down workgroups run
// `subs` blocks of 256 output columns as one continuous stream of steps.
// Both operands are fetched straight into LDS as whole 128-byte lines: the
// rows (L2 or Infinity Cache) into a ring of two 32 KiB slots, the weights,
// which come from HBM, into a ring of three, so two steps of weights are in
// flight -- all 160 KiB.
//
// Bound by the fill from L2 and HBM: at 8192 tokens gate/up moves 2.9 GB into
// LDS in 355 us (the 128-row kernel with 64-byte pieces 3.7 GB in 411, 256 rows
// with 64-byte pieces 390; without any fetch 205, without MFMAs 333), with
// 8 waves or two stages of both operands it took 380 to 460.  Touching the
// weights' lines three steps ahead was slower (+60 us: the L1's tag rate).
// Down took 341 us there; its epilogue was a third of it (two-byte stores of 64-byte
// pieces, slots and weights looked up per block) and now stages rows in the
// step's consumed slots and stores whole lines: 220 us.
#pragma once
#include "moe_stream.h"

#include <type_traits>

namespace q36 {
namespace {

constexpr int kTlBM = 256, kTlBN = 256;
constexpr int kTlSlot = kTlBM * kStRowB;            // 32 KiB
constexpr int kTlASlots = 2, kTlBSlots = 3;
constexpr int kTlLds = (kTlASlots + kTlBSlots) * kTlSlot;   // 160 KiB
constexpr int kTlWaves = 16;
constexpr int kTlGateUpBlocks = kMoeInter / (kTlBN / 2);
constexpr int kTlDownBlocks = kMoeHidden / kTlBN;

template <bool kDown>
__global__ __launch_bounds__(64 * kTlWaves, 4) void moe_tile_kernel(StreamArgs p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int K = kDown ? kMoeInter : kMoeHidden;
  constexpr int kSteps = K * 2 / kStRowB;              // per block: 8 or 32
  const unsigned nb = kDown ? kTlDownBlocks / p.subs : (unsigned)kTlGateUpBlocks;
  const unsigned items = (unsigned)p.meta[0].x * nb;
  const unsigned share = (items + 7) / 8, xi = blockIdx.x >> 3;   // contiguous per XCD
  const unsigned item = (blockIdx.x & 7) * share + xi;
  if (xi >= share || item >= items) return;
  const unsigned mt = item / nb, nt = item % nb;
  const int4 m = p.meta[1 + mt];
  const int group = m.x, row0 = m.y, rows = m.z;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const unsigned routed = kMoeTopK * p.T;

  u32x4 ars, brs;
  const bf16* wg = group < (int)p.E ? p.w + (size_t)group * (kDown ? 1 : 2) * kMoeInter * kMoeHidden
                                    : p.w_shared;
  brs = stream_rsrc(wg, (kDown ? 1u : 2u) * kMoeInter * kMoeHidden * 2u);
  if constexpr (kDown)
    ars = stream_rsrc(p.a + (size_t)row0 * kMoeInter, (unsigned)rows * kMoeInter * 2u);
  else
    ars = stream_rsrc(p.a, p.T * (unsigned)kMoeHidden * 2u);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    ars[c] = __builtin_amdgcn_readfirstlane(ars[c]);
    brs[c] = __builtin_amdgcn_readfirstlane(brs[c]);
  }

  // Fetch plan: instruction i of an operand fills its slot rows 8i .. 8i + 7,
  // lane = row x chunk position, chunk c of row r at c ^ ((r / 2) % 8); wave w
  // issues instructions 2w and 2w + 1 of both operands.  Rows past the tile's
  // end are fetched out of range.
  unsigned a_off[2], b_off[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (2 * wave + j) + (lane >> 3);
    const unsigned chunk = ((lane & 7) ^ ((r / 2) % 8)) * 16;
    unsigned off;
    if constexpr (kDown) {
      off = r < rows ? (unsigned)r * kMoeInter * 2u : kStOob;
    } else {
      const int slot = r < rows ? p.sorted[row0 + r] : -1;
      const unsigned t = (unsigned)slot < routed ? (unsigned)slot / kMoeTopK : (unsigned)slot - routed;
      off = slot < 0 ? kStOob : t * (unsigned)kMoeHidden * 2u;
    }
    a_off[j] = off + chunk;
    unsigned row;
    if constexpr (kDown)
      row = nt * p.subs * kTlBN + r;
    else
      row = (r < kTlBN / 2 ? 0 : kMoeInter - kTlBN / 2) + nt * (kTlBN / 2) + r;
    b_off[j] = row * (unsigned)K * 2u + chunk;
  }
  const unsigned lds0 = static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));
  const unsigned steps = kDown ? p.subs * kSteps : kSteps;
  const bool nt_hint = m.w == 1;
  auto fetch_a = [&](unsigned s) {
    const unsigned base = lds0 + (s % kTlASlots) * kTlSlot + wave * 2048;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      stream_fetch<false>(base + j * 1024, (int)(a_off[j] + (s % kSteps) * kStRowB), ars);
  };
  unsigned b_slot = 0;   // next weight slot to fill
  auto fetch_b = [&](unsigned s) {
    const unsigned base = lds0 + (kTlASlots + b_slot) * kTlSlot + wave * 2048;
    const unsigned kb = (s % kSteps) * kStRowB + (s / kSteps) * (unsigned)(kTlBN * K * 2);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (nt_hint) stream_fetch<true>(base + j * 1024, (int)(b_off[j] + kb), brs);
      else stream_fetch<false>(base + j * 1024, (int)(b_off[j] + kb), brs);
    }
    b_slot = b_slot + 1 == kTlBSlots ? 0 : b_slot + 1;
  };
  fetch_a(0);
  fetch_b(0);
  fetch_b(1);

  const int wm = wave >> 2, wn = wave & 3;
  const int li = lane & 31, kh = lane >> 5;
  const int blocks = (rows + 31) / 32;
  const int nrb = wm + 4 < blocks ? 2 : wm < blocks ? 1 : 0;   // this wave's row blocks
  const int arow = (32 * wm + li) * kStRowB;
  const int brow0 = (kDown ? 64 * wn : 32 * wn) * kStRowB + li * kStRowB;
  const int brow1 = brow0 + (kDown ? 32 : kTlBN / 2) * kStRowB;
  int koff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) koff[s] = ((2 * s + kh) ^ ((li / 2) % 8)) * 16;

  // Down: the slot and weight of this lane's row of each block, and how many
  // of the epilogue's stores (8 rows each) a finished block issues.
  int slots[2];
  float weights[2];
  int n_stores = 0;
  if constexpr (kDown) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int r = 32 * (wm + 4 * rb) + li;
      slots[rb] = r < rows ? p.sorted[row0 + r] : -1;
      weights[rb] = slots[rb] >= 0 && (unsigned)slots[rb] < routed ? p.rw[slots[rb]] : 1.0f;
      n_stores += min(4, max(0, (rows - 32 * (wm + 4 * rb) + 7) / 8));
    }
  }
  const bool odd = (li & 1) != 0;

  // The K loop for a wave of NRB (0 .. 2) row blocks; every wave fetches and
  // meets the barriers whatever its NRB.
  auto run = [&](auto nrb_c) {
    constexpr int NRB = decltype(nrb_c)::value;
    f32x16 acc[NRB > 0 ? NRB : 1][2];
    auto clear = [&]() {
#pragma unroll
      for (int i = 0; i < NRB; ++i) acc[i][0] = acc[i][1] = f32x16{};
    };
    clear();
    unsigned slot = 0;   // weight slot of `step`
    for (unsigned step = 0; step < steps; ++step) {
      // A(step), B(step) landed; B(step + 1) and, after a finished block, its
      // stores were issued later and may be in flight
      if (step + 1 >= steps) __builtin_amdgcn_s_waitcnt(stream_vmcnt(0));
      else if (kDown && NRB > 0 && step > 0 && step % kSteps == 0 && n_stores >= 8)
        __builtin_amdgcn_s_waitcnt(stream_vmcnt(2 + 8));
      else if (kDown && NRB > 0 && step > 0 && step % kSteps == 0 && n_stores >= 4)
        __builtin_amdgcn_s_waitcnt(stream_vmcnt(2 + 4));
      else __builtin_amdgcn_s_waitcnt(stream_vmcnt(2));
      __syncthreads();   // every wave's fetches of `step` landed; last step's slots are free
      if (step + 1 < steps) fetch_a(step + 1);
      if (step + kTlBSlots - 1 < steps) fetch_b(step + kTlBSlots - 1);
      if constexpr (NRB > 0) {
        const char* as = lds + (step % kTlASlots) * kTlSlot + arow;
        const char* bs = lds + (kTlASlots + slot) * kTlSlot;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bf16x8 b0 = *reinterpret_cast<const bf16x8*>(bs + brow0 + koff[s]);
          const bf16x8 b1 = *reinterpret_cast<const bf16x8*>(bs + brow1 + koff[s]);
#pragma unroll
          for (int rb = 0; rb < NRB; ++rb) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(as + 128 * rb * kStRowB + koff[s]);
            if constexpr (kDown) {   // lane = row, registers = columns
              acc[rb][0] = mfma32x32x16(b0, a, acc[rb][0]);
              acc[rb][1] = mfma32x32x16(b1, a, acc[rb][1]);
            } else {
              acc[rb][0] = mfma32x32x16(a, b0, acc[rb][0]);
              acc[rb][1] = mfma32x32x16(a, b1, acc[rb][1]);
            }
          }
        }
      }
      const unsigned used = slot;
      slot = slot + 1 == kTlBSlots ? 0 : slot + 1;
      if constexpr (kDown) {
        if ((step + 1) % kSteps == 0) {   // a block of 256 columns done
          // Once every wave has read the step's operands, its two slots are
          // free until the next step's barrier: each wave stages 32 rows x 64
          // columns (16-byte chunks XORed with the row) in 4 KiB of them and
          // stores whole 128-byte lines.
          lds_barrier();
          if constexpr (NRB > 0) {
            char* stg = lds + (wave < 8 ? (step % kTlASlots) : kTlASlots + used) * kTlSlot + (wave & 7) * 4096;
            const unsigned c = (nt * p.subs + step / kSteps) * kTlBN + 64 * wn + 8 * (lane & 7);
#pragma unroll
            for (int rb = 0; rb < NRB; ++rb) {
              const float w = weights[rb];
#pragma unroll
              for (int q = 0; q < 8; ++q) {   // columns 8q + 4kh .. + 3
                const f32x16& v = acc[rb][q >> 2];
                bf16x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = f2bf(bf2f(f2bf(v[4 * (q & 3) + e])) * w);
                *reinterpret_cast<bf16x4*>(stg + li * 128 + ((q ^ (li & 7)) * 16) + 8 * kh) = o;
              }
              __atomic_signal_fence(__ATOMIC_SEQ_CST);   // LDS serves a wave in order
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                const int r = 8 * k + (lane >> 3);
                const bf16x8 o = *reinterpret_cast<const bf16x8*>(stg + r * 128 + (((lane & 7) ^ (r & 7)) * 16));
                const int sl = __shfl(slots[rb], r, 64);
                if (sl >= 0) *reinterpret_cast<bf16x8*>(p.out + (size_t)sl * kMoeHidden + c) = o;
              }
              __atomic_signal_fence(__ATOMIC_SEQ_CST);
            }
            clear();
          }
        }
      }
    }
    if constexpr (!kDown && NRB > 0) {
      const unsigned c = nt * (kTlBN / 2) + 32 * wn + (li & 30);
      float g8[8], u8[8];
      bf16 a8[8];
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (j % 4 == 0) {   // acc rows 8h .. 8h + 7
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              g8[e] = bf2f(f2bf(acc[rb][0][2 * j + e]));
              u8[e] = bf2f(f2bf(acc[rb][1][2 * j + e]));
            }
            silu_mul8(g8, u8, a8);
          }
          const int i = 2 * j + (li & 1);
          const int r = 32 * (wm + 4 * rb) + 8 * (i >> 2) + 4 * kh + (i & 3);
          const float v0 = bf2f(a8[2 * (j % 4)]), v1 = bf2f(a8[2 * (j % 4) + 1]);
          const float keep = odd ? v1 : v0, got = beside(odd ? v0 : v1);
          const bf16x2 o = {f2bf(odd ? got : keep), f2bf(odd ? keep : got)};
          if (r < rows)
            *reinterpret_cast<bf16x2*>(p.out + (size_t)(row0 + r) * kMoeInter + c) = o;
        }
      }
    }
  };
  if (nrb == 2) run(std::integral_constant<int, 2>{});
  else if (nrb == 1) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 0>{});
}

}  // namespace
}  // namespace q36
