// Column kernel (dV, dK) of the flash-attention backward for d_qk = d_v = 128 and grids that fill the chip: 256 kv rows per
// block, 64 per wave, streaming 32-row tiles of Q and dO.
//
// The walk and the arithmetic are those of attn_bwd_chain's column kernel, which has 128 rows per block.  That one reads an LDS
// operand for every matrix instruction, and an LDS read and a vector instruction of one wave do not overlap (a read alone 21
// clocks, with two exponentials 51).  With two 32-row groups per wave an operand serves two matrix instructions, and the work
// between them -- P = exp2(S c2 - lse2) between those of dP, dS = P (dP - delta) and the packing between those of dV -- is about
// what one of them lasts.  The 512 registers of the SIMD's only wave hold both outputs (256 accumulation registers), the K and V
// fragments (128) and the tile's scores.
//
// A tile is one sequence of 32 steps (S, dP, dV, dK: 8 each; a step is one operand and two matrix instructions) with the reads
// PF steps ahead across all of them.  Reads, waits and matrix instructions are volatile assembly and stay in this order;
// the wait of each step is counted from the order of issue (reads_behind).
//
// Clocks per 32 streamed x 64 resident rows: 3350 (the matrix instructions: 2048), where the 128-row kernel takes 4219 for
// 64 x 32.  Whole backward, 128-row kernel and this: B4 H32 S2048 causal 555 -> 523 us, not causal 948 -> 886; B2 H32 S4096
// causal 984 -> 924; B16 H32 S512 255 -> 246.  What is left of a block besides its tiles is memory: all blocks of a round load (128 KB,
// 10000 clocks) and store (128 KB, 10000) at the same time, at 5 TB/s.
#pragma once
#include "bwd_chain.h"

namespace aat {

struct AttnBwdCol {
  static constexpr int D = 128, BX = 256, BY = 32, Nthreads = 256, NC = D / 8, KS = D / 16, DT = D / 32, WM = 64, NS = 3;
  static constexpr int PF = 3;                          // operand reads in flight; 2 and 4 measure the same
  using Dma = TileDma<BY, NC, Nthreads, Swz::Both, 0, true>;
  static constexpr int kYBytes = BY * D * 2, kStageBytes = 2 * kYBytes + 1024;   // Q, dO, and lse2 and delta of the rows
  static constexpr int kTileInstr = 2 * Dma::kIters + 1;                         // LDS-DMA instructions per thread per tile
  static constexpr int kOStride = D * 2 + 16;
  static constexpr int kMainBytes = NS * kStageBytes, kEpiBytes = BX * kOStride;
  static constexpr int kSmemBytes = kMainBytes > kEpiBytes ? kMainBytes : kEpiBytes;

  // LDS operations in issue order: PF operand reads up front; behind the matrix instructions of step i the read for step i + PF
  // and then the statistics that step i asks for.  Group g (rows 8g + 4h ..) of lse2 is used from step 8 + 2g on and that of
  // delta from step 16 + 2g on: each is issued just before the operand read that its step waits for.
  static constexpr int ops(int i) { return i < 2 * KS ? 1 : i < 4 * KS ? 2 : 0; }          // one b128, or two transposing b64
  static constexpr int group_of(int step, int first) {
    const int g = step + PF + 1 - first;
    return g >= 0 && g < 8 && g % 2 == 0 ? g / 2 : -1;
  }
  static constexpr int lse_group(int step) { return group_of(step, KS); }
  static constexpr int delta_group(int step) { return group_of(step, 2 * KS); }
  static constexpr int stats(int step) { return (lse_group(step) >= 0) + (delta_group(step) >= 0); }
  static constexpr int reads_behind(int i) {            // operations issued after the read of step i and before step i begins
    int n = i < PF ? 0 : stats(i - PF);
    for (int r = i + 1; r < PF; ++r) n += ops(r);
    for (int k = i < PF ? 0 : i - PF + 1; k < i; ++k) n += ops(k + PF) + stats(k);
    return n;
  }
};

// Transposing read at address base ^ x (lds_read_h8_async_xor).
AAT_DEV h4 lds_read_tr_h4_async_xor(uint32_t base, int x, int imm) {
  h4 v;
  uint32_t t;
  asm volatile("v_xor_b32 %1, %3, %2\n\tds_read_b64_tr_b16 %0, %1 offset:%4" : "=v"(v), "=&v"(t) : "v"(base), "n"(x), "i"(imm));
  return v;
}
// Matrix instructions that keep their place among the reads: scores in vector registers, outputs in accumulation registers.
AAT_DEV void mfma_score_first(f16v& c, h8 a, h8 b) { asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b)); }
AAT_DEV void mfma_score(f16v& c, h8 a, h8 b) { asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
AAT_DEV void mfma_output(f16v& c, h8 a, h8 b) { asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b)); }

// k, v [B*H, seq_k, 128]; q, dO [B*H, seq_q, 128]; lse2, delta [B*H, seq_q] from the row kernel, delta less than 4 GB behind
// lse2 (750 MB of either belong to 280 GB of operands).  Lengths are multiples of 32: the tiles divide seq_q, and 32-row groups that the last block of a
// head lacks load rows that exist and are not stored.
__global__ void __launch_bounds__(AttnBwdCol::Nthreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
attn_bwd_col(const half_t* __restrict__ k, const half_t* __restrict__ v, const half_t* __restrict__ q,
             const half_t* __restrict__ dO, const float* __restrict__ lse2, const float* __restrict__ delta,
             half_t* __restrict__ dv, half_t* __restrict__ dk, int seq_k, int seq_q, float c2, float out_scale, int causal) {
  using T = AttnBwdCol;
  constexpr int D = T::D, BX = T::BX, BY = T::BY, KS = T::KS, DT = T::DT, NC = T::NC, WM = T::WM, NS = T::NS, PF = T::PF;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 31, h = lane >> 5;
  const int Tx = (seq_k + BX - 1) / BX;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int bh = tile / Tx, xb = tile % Tx;
  if (causal) {                                   // longest blocks first
    const TileId t = causal_tile(blockIdx.x, gridDim.x, Tx, false);
    bh = t.bh;
    xb = t.blk;
  }
  const int x0 = xb * BX, w0 = x0 + wave * WM;    // first rows of the block and of the wave
  const int diag = seq_k - seq_q;                 // causal: score (q, kv) is kept when kv <= q + diag
  // The walk goes from the last tile down (blocks of a head share it in L2) to the first that sees row x0.  The first `plain` tiles
  // are seen by every row of the block.
  const int j_end = seq_q / BY;
  int j_begin = 0, j_full = 0;
  if (causal) {
    j_begin = x0 <= diag ? 0 : (x0 - diag) / BY;
    j_full = x0 + BX - 1 <= diag ? 0 : (x0 + BX - 1 - diag + BY - 1) / BY;
  }
  const int tiles = j_end > j_begin ? j_end - j_begin : 0, plain = j_end > j_full ? j_end - j_full : 0;

  const char* const qg = reinterpret_cast<const char*>(q + (size_t)bh * seq_q * D);
  const char* const dOg = reinterpret_cast<const char*>(dO + (size_t)bh * seq_q * D);
  const char* const statg = reinterpret_cast<const char*>(lse2 + (size_t)bh * seq_q);
  const uint32_t stat_off = 4 * n + (h ? (uint32_t)((const char*)delta - (const char*)lse2) : 0u);   // lanes 0..31 lse2, 32..63 delta
  T::Dma dma;
  dma.init(tid);
  const auto tile_of = [&](int step) { return j_end - 1 - step; };
  const auto issue = [&](int step, int st) {
    const int j = tile_of(step);
    char* const base = smem + st * T::kStageBytes;
    dma.issue(qg + (size_t)j * T::kYBytes, base, wave * 64);
    dma.issue(dOg + (size_t)j * T::kYBytes, base + T::kYBytes, wave * 64);
    // every wave copies the statistics (same bytes, same place): uniform instruction counts
    const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(AAT_AS3 char*)(base + 2 * T::kYBytes));
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 ::"s"(dst), "v"(stat_off), "s"(statg + (size_t)j * BY * 4) : "memory", "m0");
  };

  // resident operands: this lane's two rows of K and of V as MFMA B fragments
  const int groups = w0 >= seq_k ? 0 : (seq_k - w0) / 32 < 2 ? (seq_k - w0) / 32 : 2;    // the wave's 32-row groups that exist
  h8 kf[2][KS], vf[2][KS];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const size_t row = (size_t)bh * seq_k + (groups > 0 ? w0 : x0) + (rt < groups ? 32 * rt : 0) + n;
    load_q_frags<1, KS, D>(reinterpret_cast<h8(&)[1][KS]>(kf[rt]), k + row * D + 8 * h);
    load_q_frags<1, KS, D>(reinterpret_cast<h8(&)[1][KS]>(vf[rt]), v + row * D + 8 * h);
  }

  // LDS addresses inside stage 0 (attn_bwd_chain): k-step ks of a row-major fragment is at frag ^ 32 ks, d-tile dt of a transposing read
  // at tr_lo / tr_hi ^ 64 dt
  uint32_t frag, tr_lo, tr_hi;
  {
    int o1[KS];
    k_frag_offsets<KS, NC, Swz::Both>(o1, n, h);
    frag = lds_addr(smem + o1[0]);
    const int s16 = lane & 15, row = 4 * h + (s16 >> 2), col = 16 * ((lane >> 4) & 1) + 4 * (s16 & 3);
    tr_lo = lds_addr(smem + lds_chunk_off<NC, Swz::Both>(row, col >> 3) + (col & 7) * 2);
    tr_hi = lds_addr(smem + lds_chunk_off<NC, Swz::Both>(row + 8, col >> 3) + (col & 7) * 2);
  }
  const uint32_t stat = lds_addr(smem + 2 * T::kYBytes + 16 * h);

  f16v dvt[2][DT], dkt[2][DT];                    // dV^T and dK^T
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int i = 0; i < DT; ++i) dvt[rt][i] = dkt[rt][i] = zero16();
  if (tiles > 0) issue(0, 0);
  if (tiles > 1) issue(1, 1);

  const auto pin = [&]() {                        // outputs in accumulation registers, resident fragments in vector registers
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
#pragma unroll
      for (int i = 0; i < DT; ++i) asm volatile("" : "+a"(dvt[rt][i]), "+a"(dkt[rt][i]));
#pragma unroll
      for (int i = 0; i < KS; ++i) asm volatile("" : "+v"(kf[rt][i]), "+v"(vf[rt][i]));
    }
  };

  // One tile; register e of a score tile is streamed row 8 (e / 4) + 4h + e % 4.
  const auto walk = [&](auto masked_tag, uint32_t off, int jt) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const uint32_t fa = frag + off, zl = tr_lo + off, zh = tr_hi + off, sa = stat + off;
    const int lim = w0 + n - diag - jt * BY - 4 * h;         // masked: 32 rt + lim > the register's row
    f16v s[2], dp[2];                                        // S, then P, of the two row groups; dP, then dS
    h8 ef[2][2];                                             // P, then dS, as operand, per group of 16 streamed rows
    f4v lrow[4], drow[4];
    h8 ring[PF];
    h4 lo[PF], hi[PF];
    const auto read = [&](auto i_tag) {
      constexpr int i = decltype(i_tag)::value;
      if constexpr (i < 2 * KS) {
        constexpr int ks = i % KS, imm = i / KS * T::kYBytes;
        if constexpr (ks == 0) ring[i % PF] = lds_read_h8_async(fa, imm);
        else ring[i % PF] = lds_read_h8_async_xor(fa, ks << 5, imm);
      } else if constexpr (i < 4 * KS) {
        constexpr int dt = i % DT, imm = (i < 3 * KS ? T::kYBytes : 0) + i / DT % 2 * 16 * NC * 16;
        if constexpr (dt == 0) {
          lo[i % PF] = lds_read_tr_h4_async(zl, imm);
          hi[i % PF] = lds_read_tr_h4_async(zh, imm);
        } else {
          lo[i % PF] = lds_read_tr_h4_async_xor(zl, dt << 6, imm);
          hi[i % PF] = lds_read_tr_h4_async_xor(zh, dt << 6, imm);
        }
      }
    };
    // What runs behind matrix instruction rt of a step.  A score tile is read here two matrix instructions after its last one,
    // 16 passes where 12 wait states are asked for; a packed operand is used three or more matrix instructions on.
    const auto side = [&](auto step_tag, auto rt_tag) {
      constexpr int step = decltype(step_tag)::value, rt = decltype(rt_tag)::value, e0 = 2 * (step % KS);
      if constexpr (step >= KS && step < 2 * KS) {           // between those of dP
        if constexpr (step == KS) asm volatile("" : "+v"(s[rt]));
        if constexpr (step % 2 == 0 && rt == 0) asm volatile("" : "+v"(lrow[e0 / 4]));
#pragma unroll
        for (int e = e0; e < e0 + 2; ++e) {
          s[rt][e] = fast_exp2(s[rt][e] * c2 - lrow[e / 4][e % 4]);
          if (MASKED && 32 * rt + lim > 8 * (e / 4) + e % 4) s[rt][e] = 0.f;
        }
        if constexpr (step == 13) ef[rt][0] = pack8_rne(s[rt], 0);
      } else if constexpr (step >= 2 * KS && step < 3 * KS) {   // dV
        if constexpr (step == 2 * KS) {
          asm volatile("" : "+v"(dp[rt]));
          ef[rt][1] = pack8_rne(s[rt], 8);
        }
        if constexpr (step % 2 == 0 && rt == 0) asm volatile("" : "+v"(drow[e0 / 4]));
#pragma unroll
        for (int e = e0; e < e0 + 2; ++e) dp[rt][e] = s[rt][e] * (dp[rt][e] - drow[e / 4][e % 4]);
        if constexpr (step == 21) ef[rt][0] = pack8_rne(dp[rt], 0);
      } else if constexpr (step == 3 * KS) {                 // dK
        ef[rt][1] = pack8_rne(dp[rt], 8);
      }
    };
    static_for<PF>([&](auto i_tag) { read(i_tag); });
    sched_fence();
    static_for<4 * KS>([&](auto step_tag) {
      constexpr int step = decltype(step_tag)::value, ks = step % KS;
      h8 a;
      if constexpr (step < 2 * KS) {
        lds_wait_younger<T::reads_behind(step)>(ring[step % PF]);
        a = ring[step % PF];
      } else {
        lds_wait_younger<T::reads_behind(step)>(lo[step % PF], hi[step % PF]);
        a = cat_h4(lo[step % PF], hi[step % PF]);
      }
      static_for<2>([&](auto rt_tag) {
        constexpr int rt = decltype(rt_tag)::value;
        if constexpr (step == 0) mfma_score_first(s[rt], a, kf[rt][ks]);
        else if constexpr (step < KS) mfma_score(s[rt], a, kf[rt][ks]);
        else if constexpr (step == KS) mfma_score_first(dp[rt], a, vf[rt][ks]);
        else if constexpr (step < 2 * KS) mfma_score(dp[rt], a, vf[rt][ks]);
        else if constexpr (step < 3 * KS) mfma_output(dvt[rt][ks % DT], a, ef[rt][ks / DT]);
        else mfma_output(dkt[rt][ks % DT], a, ef[rt][ks / DT]);
        sched_fence();
        if constexpr (rt == 1) {                             // both have their operand: its registers are free
          read(std::integral_constant<int, step + PF>{});
          if constexpr (T::lse_group(step) >= 0) lrow[T::lse_group(step)] = lds_read_f4_async(sa, 32 * T::lse_group(step));
          if constexpr (T::delta_group(step) >= 0) drow[T::delta_group(step)] = lds_read_f4_async(sa, 128 + 32 * T::delta_group(step));
        }
        side(step_tag, rt_tag);
        sched_fence();
      });
    });
  };

  uint32_t off = 0;
  int st = 0;
  const auto tile_step = [&](int step, auto masked_tag) {
    pin();
    // tile `step` has landed (the next one may be in flight) and every wave is past the one before
    if (step + 1 < tiles) wait_vmcnt<T::kTileInstr>();
    else wait_vmcnt<0>();
    block_sync();
    if (step + 2 < tiles) issue(step + 2, (st + 2) % NS);
    const int jt = tile_of(step);
    // a wave none of whose rows is seen from the tile has nothing to add
    if (groups > 0 && (!decltype(masked_tag)::value || w0 <= jt * BY + BY - 1 + diag)) walk(masked_tag, off, jt);
    st = st + 1 == NS ? 0 : st + 1;
    off = st * T::kStageBytes;
  };
  int step = 0;
  for (; step < plain; ++step) tile_step(step, std::false_type{});
  for (; step < tiles; ++step) tile_step(step, std::true_type{});
  asm volatile("s_nop 15" ::: "memory");          // the last matrix instructions have written their outputs
  pin();

  // ---- epilogue: scale, round, transpose through wave-private LDS, 16-byte stores ---------------------
  block_sync();
  char* const ostage = smem + wave * WM * T::kOStride;
  const auto store = [&](auto& acc, half_t* out, float sc) {
    half_t* const og = out + ((size_t)bh * seq_k + w0) * D;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const h2 a = pack_rne(acc[rt][dt][4 * g] * sc, acc[rt][dt][4 * g + 1] * sc);
          const h2 b = pack_rne(acc[rt][dt][4 * g + 2] * sc, acc[rt][dt][4 * g + 3] * sc);
          h4 w;
          w[0] = a[0]; w[1] = a[1]; w[2] = b[0]; w[3] = b[1];
          *reinterpret_cast<h4*>(ostage + (rt * 32 + n) * T::kOStride + (32 * dt + 8 * g + 4 * h) * 2) = w;
        }
    wait_lgkm0();
#pragma unroll
    for (int t = 0; t < WM * NC / 64; ++t) {
      if (t * 64 / (32 * NC) >= groups) break;
      const int idx = t * 64 + lane, row = idx / NC, c = idx % NC;
      const u4v val = *reinterpret_cast<const u4v*>(ostage + row * T::kOStride + c * 16);
      *reinterpret_cast<u4v*>(reinterpret_cast<char*>(og) + (size_t)row * D * 2 + c * 16) = val;
    }
    wait_lgkm0();                                 // the staging rows are reused by the next output
  };
  store(dvt, dv, 1.0f);
  store(dkt, dk, out_scale);
}

}  // namespace aat
