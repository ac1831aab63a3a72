// RetNet backward, dK from a stored dS, for gfx950 (MI355X).
//
//     dK[kv][:] = sum_q dS[q][kv] Q[q][:]          dS = half(((dO V^T) / r) * M), B*H*S_q*S_kv fp16
//
// The chained-contraction passes (bwd_chain.h) evaluate dO V^T twice, once for dQ and once for dK: two thirds
// of either pass's matrix work.  When the caller grants a workspace of B*H*S_q*S_kv fp16 the row pass writes
// the dS tiles it forms anyway (its DS_OUT variant) and this kernel replaces the dK pass: it streams Q tiles
// and dS tiles and runs the second contraction only -- a third of the matrix work, no resident 512-wide
// fragment (128 registers), so two waves fit a SIMD.  The reference has neither (it accumulates dK in the
// registers of its single column-block kernel, csrc/kernels/retnet/bwd/bwd_colblock.h:556-576).
//
// dS lies in 64 x 64 blocks of 8 KB, [B*H][S_q/64][S_kv/64][64][64] (ds_block_offset): rows of a [S_q, S_kv]
// matrix are S_kv*2 bytes apart, a power of two at the usual lengths, so the tiles all blocks write (and read)
// at the same step of their walks would fall on the few memory channels that stride selects.  In blocks a tile
// is one contiguous piece.
//
// The row pass writes the tiles it walks and nothing else, so what lies outside its walk is garbage here:
// per query tile this kernel recomputes the kv range the writer covered (from the same mask mode, the same
// ranges and the writer's block and tile sizes) and takes dS as zero outside of it.
#pragma once
#include <type_traits>

#include "../../utils/block_parts.h"
#include "../../utils/cdna4.h"
#include "../../utils/mask_extents.h"
#include "../../utils/tile_ops.h"
#include "ds_layout.h"

namespace aat {

// What bounds it is the stream of dS: at B4 H8 S2048 d_qk 256 the causal walk takes 52 us for 142 MB of it, the dense one 90 for 268.
// Measured without effect on that: two to five tiles in flight (48 to 120 KB), tiles of 32 rows, half the LDS reads (64 kv rows per wave).
// Where LDS has no room for a second block beside one of four waves with two stages (d_qk 256, 96 KB), a block has eight waves and three
// stages: 56 -> 52 us causal, 98 -> 91 dense.
// Looking the writer's ranges up per tile, through loads that drained all copies in flight, cost the walks with ranges more: 86 -> 54.
//
// NWD waves share 32 kv rows, Kd / NWD columns of dK each.
// Kd: width of q/k rows; BX: kv rows per block; BY: query rows per streamed tile; NS: LDS stages, all but one of them on their way.
template <int Kd, int BX, int BY, int Nthreads, int NS>
struct RetBwdDk {
  static constexpr int NW = Nthreads / kWave, NWK = BX / 32, NWD = NW / NWK;
  static constexpr int DTW = Kd / 32 / NWD, KSTEPS = BY / 16;
  static constexpr int NCZ = Kd / 8, NCS = 8, NSUB = BX / 64;
  static_assert(NWD * NWK * kWave == Nthreads && DTW * NWD * 32 == Kd, "32 kv rows by whole 32-column tiles per wave");
  static_assert(BY == 64 && Kd % 64 == 0 && BX % 64 == 0, "a query tile is one row of dS blocks");
  static_assert(NS == 2 || NS == 3, "buffers");
  using ZDma = TileDma<BY, NCZ, Nthreads, Swz::Rows4>;   // Q tile
  static constexpr int kSIters = BY * NSUB * NCS / Nthreads, kSRows = Nthreads / NCS;   // dS tile: LDS-DMA instructions per thread, rows per instruction
  static_assert(kSIters * Nthreads == BY * NSUB * NCS, "whole 32-row pieces of dS blocks per instruction");
  static constexpr int kZBytes = BY * Kd * 2, kSBytes = BY * BX * 2;
  static constexpr int kStageBytes = kZBytes + kSBytes;
  static constexpr int kTileInstr = ZDma::kIters + kSIters;
  static_assert((NS - 2) * kTileInstr < 64, "copies in flight are counted by a 6-bit counter");
  static constexpr int kOStride = Kd * 2 + 16;
  static constexpr int kMainBytes = NS * kStageBytes;
  static constexpr int kEpiBytes = BX * kOStride;
  static constexpr int kSmemBytes = kMainBytes > kEpiBytes ? kMainBytes : kEpiBytes;
};

// q [B*H, seq_q, Kd], ds in 64 x 64 blocks (above), dk [B*H, seq_k, Kd], all fp16.
// causal / extents: the mask mode of the walk, as in ret_bwd_chain (extents = the scan's ranges or nullptr).
// seq_q is a multiple of wr_rows and seq_k of BX; GEN: both of 64, kv rows a last block does not have are computed from copies
// and not stored.
// wr_rows x wr_cols: resident rows and streamed-tile width of the row pass that wrote ds (wr_rows % BY == 0).
template <int Kd, int BX, int BY, int Nthreads, int NS, int WPE = 2, int GEN = 0>
__global__ void __launch_bounds__(Nthreads) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
ret_bwd_dk_from_ds(const half_t* __restrict__ q, const half_t* __restrict__ ds, half_t* __restrict__ dk, int H,
                   int seq_k, int seq_q, int causal, const int* __restrict__ extents, int wr_rows, int wr_cols, BlockParts in_parts = {}) {
  using T = RetBwdDk<Kd, BX, BY, Nthreads, NS>;
  constexpr int DTW = T::DTW, KSTEPS = T::KSTEPS, NCZ = T::NCZ, NCS = T::NCS;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % T::NWK, wd = wave / T::NWK;      // the wave's 32 kv rows and its share of the columns
  const int n = lane & 31, h = lane >> 5;

  const int Tx = GEN ? (seq_k + BX - 1) / BX : seq_k / BX;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  int bh = tile / Tx, xb = tile % Tx;
  PartId id{};
  if (causal || extents != nullptr) {             // longest blocks first: the first kv blocks
    id = causal_part(blockIdx.x, gridDim.x, Tx, false, in_parts);
    bh = id.bh;
    xb = id.blk;
  }
  const int x0 = xb * BX;
  const int cols = GEN && seq_k - x0 < BX ? seq_k - x0 : BX;   // kv rows of this block that exist, a multiple of 64
  const int diag = seq_k - seq_q;
  const int head = bh % H;
  int j_begin = 0, j_end = seq_q / BY;
  MaskExtents ext{};
  if (extents != nullptr) {
    ext = mask_extents_at(extents, H, seq_q, seq_k);
    int lo, hi;
    mask_col_range(ext, head, seq_q, seq_k, x0, cols, lo, hi);
    mask_tile_range(lo, hi, BY, j_end, j_begin, j_end);
  } else if (causal) {                            // q tiles that reach kv >= x0:  q >= x0 - diag
    const int first = x0 - diag;
    j_begin = first <= 0 ? 0 : first / BY;
    part_range(id, j_begin, j_end);
  }

  const char* zg = reinterpret_cast<const char*>(q + (size_t)bh * seq_q * Kd);
  const char* sg = reinterpret_cast<const char*>(ds + ds_block_offset(bh, 0, x0, seq_q, seq_k));
  const size_t s_pitch = (size_t)(seq_k >> 6) * 8192;    // from one row of blocks to the next
  typename T::ZDma zdma;
  zdma.init(tid);
  const int wave_base = wave * 64;
  // dS: LDS row r of the tile is row r % BY of block r / BY; a wave copies eight rows at a time
  const uint32_t s_lane = (uint32_t)(lane / NCS * 128 + swz<NCS, Swz::Rows4>(lane / NCS, lane % NCS) * 16);
  auto issue = [&](int jt, int st) {              // walked downwards from the end of the sequence, like the column passes of the chained kernel
    char* base = smem + st * T::kStageBytes;
    zdma.issue(zg + (size_t)jt * T::kZBytes, base, wave_base);
    const char* const rows = sg + (size_t)jt * s_pitch;
#pragma unroll
    for (int i = 0; i < T::kSIters; ++i) {
      const int r = i * T::kSRows + wave * (kWave / NCS), sub = r / BY;
      uint64_t src = (uint64_t)(uintptr_t)(rows + r % BY * 128 + (!GEN || sub * 64 < cols ? sub * 8192 : 0));   // a block that does not exist: copies of the first
      asm volatile("" : "+s"(src));
      __builtin_amdgcn_global_load_lds((const AAT_AS1 void*)(uintptr_t)(src + s_lane),
                                       (AAT_AS3 void*)(base + T::kZBytes + (i * Nthreads + wave_base) * 16), 16, 0, 2);
    }
  };

  // LDS addresses inside stage 0: Q^T fragments (A operand, d-tile dt) and this wave's dS columns (B operand);
  // both are transposing reads of rows 4h + (lane%16)/4 of a 16-row step, + 8 rows for the second half
  uint32_t zaddr[DTW], saddr;
  {
    const int s16 = lane & 15;
    const int row = 4 * h + (s16 >> 2), col = 16 * ((lane >> 4) & 1) + 4 * (s16 & 3);
#pragma unroll
    for (int dt = 0; dt < DTW; ++dt)
      zaddr[dt] = lds_addr(smem + lds_chunk_off<NCZ, Swz::Rows4>(row, 4 * (wd * DTW + dt) + (col >> 3)) + (col & 7) * 2);
    saddr = lds_addr(smem + T::kZBytes + lds_chunk_off<NCS, Swz::Rows4>((wk >> 1) * BY + row, 4 * (wk & 1) + (col >> 3)) + (col & 7) * 2);
  }
  constexpr int kZRow16 = 16 * NCZ * 16, kZRow8 = 8 * NCZ * 16, kSRow16 = 16 * NCS * 16, kSRow8 = 8 * NCS * 16;

  f16v acc[1][DTW];
#pragma unroll
  for (int dt = 0; dt < DTW; ++dt) acc[0][dt] = zero16();

  const int my_kv = x0 + wk * 32 + n;             // the kv position this lane owns
  // The kv range that the writer covered for the row block a query tile lies in.  Lane i holds that of row block 64 w + i, for the 64
  // the walk is in: looked up per tile, the ranges' loads drained every copy in flight.
  int window = -1, lane_lo = 0, lane_hi = seq_k;
  int wr = (j_end * BY - 1) / wr_rows;            // row block of the current tile
  const auto load_ranges = [&]() {
    window = wr >> 6;
    const int wx0 = (window * 64 + lane) * wr_rows;
    const int wrows = GEN && seq_q - wx0 < wr_rows ? seq_q - wx0 : wr_rows;
    lane_lo = 0;
    lane_hi = seq_k;
    if (wx0 < seq_q) {
      if (extents != nullptr) {
        int lo, hi, jb, je;
        mask_row_range(ext, head, seq_q, wx0, wrows, lo, hi);
        mask_tile_range(lo, hi, wr_cols, seq_k / wr_cols, jb, je);
        lane_lo = jb * wr_cols;
        lane_hi = je * wr_cols;
      } else if (causal) {
        const int last = wx0 + wrows - 1 + diag;
        const int lim = last < 0 ? 0 : last / wr_cols + 1;
        lane_hi = lim * wr_cols < seq_k ? lim * wr_cols : seq_k;
      }
    }
    asm volatile("" : "+v"(lane_lo), "+v"(lane_hi));      // waited for here
  };
  if (j_begin < j_end) load_ranges();

#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    if (j_end - 1 - i >= j_begin) issue(j_end - 1 - i, i);

  int st = 0;
  for (int jt = j_end - 1; jt >= j_begin; --jt) {
    if (jt - j_begin >= NS - 2) wait_vmcnt<(NS - 2) * T::kTileInstr>();
    else wait_vmcnt<0>();
    block_sync();
    if (jt - (NS - 1) >= j_begin) issue(jt - (NS - 1), st == 0 ? NS - 1 : st - 1);

    if (jt * BY < wr * wr_rows) --wr;
    if (wr >> 6 != window) load_ranges();
    const int wlo = __builtin_amdgcn_readlane(lane_lo, wr & 63), whi = __builtin_amdgcn_readlane(lane_hi, wr & 63);
    const bool mine_written = my_kv >= wlo && my_kv < whi;

    // The operand reads are issued as instructions with counted waits (tile_ops.h): in front of an LDS read it can see
    // the compiler waits for every LDS-DMA copy in flight.  All of the tile's B operands are read ahead of its A operands.
    const uint32_t off = st * T::kStageBytes, sa = saddr + off;
    uint32_t za[DTW];
#pragma unroll
    for (int dt = 0; dt < DTW; ++dt) za[dt] = zaddr[dt] + off;
    constexpr int S = KSTEPS * DTW, PF = S < 4 ? S : 4;
    h4 blo[KSTEPS], bhi[KSTEPS], lo[PF], hi[PF];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      blo[s] = lds_read_tr_h4_async(sa, s * kSRow16);
      bhi[s] = lds_read_tr_h4_async(sa, s * kSRow16 + kSRow8);
    }
#pragma unroll
    for (int i = 0; i < PF; ++i) {
      lo[i] = lds_read_tr_h4_async(za[i % DTW], i / DTW * kZRow16);
      hi[i] = lds_read_tr_h4_async(za[i % DTW], i / DTW * kZRow16 + kZRow8);
    }
    h8 bf;
    static_for<S>([&](auto i_tag) {
      constexpr int i = decltype(i_tag)::value, dt = i % DTW;
      // wait on the slot, take its value, refill it (a copy made before the wait could read a register whose load
      // has not landed); the B pairs are older: they have landed too
      lds_wait_younger<2 * ((i + PF - 1 < S) ? PF - 1 : S - 1 - i)>(lo[i % PF], hi[i % PF]);
      const h4 clo = lo[i % PF], chi = hi[i % PF];
      if constexpr (i + PF < S) {
        lo[i % PF] = lds_read_tr_h4_async(za[(i + PF) % DTW], (i + PF) / DTW * kZRow16);
        hi[i % PF] = lds_read_tr_h4_async(za[(i + PF) % DTW], (i + PF) / DTW * kZRow16 + kZRow8);
      }
      if constexpr (dt == 0) {
        constexpr int s = i / DTW;
        asm volatile("" : "+v"(blo[s]), "+v"(bhi[s]));
        bf = cat_h4(blo[s], bhi[s]);
#pragma unroll
        for (int e = 0; e < 8; ++e) bf[e] = mine_written ? bf[e] : (half_t)0.f;
      }
      acc[0][dt] = mfma_32x32x16(cat_h4(clo, chi), bf, acc[0][dt]);
    });
    st = st == NS - 1 ? 0 : st + 1;
  }

  wait_vmcnt<0>();
  block_sync();
  const auto finish = [&]() {                     // the waves' columns meet in LDS, rows leave whole
#pragma unroll
    for (int dt = 0; dt < DTW; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const h2 a = pack_rne(acc[0][dt][4 * g], acc[0][dt][4 * g + 1]), b = pack_rne(acc[0][dt][4 * g + 2], acc[0][dt][4 * g + 3]);
        h4 w;
        w[0] = a[0]; w[1] = a[1]; w[2] = b[0]; w[3] = b[1];
        *reinterpret_cast<h4*>(smem + (wk * 32 + n) * T::kOStride + (32 * (wd * DTW + dt) + 8 * g + 4 * h) * 2) = w;
      }
    __syncthreads();
    char* const out = reinterpret_cast<char*>(dk + ((size_t)bh * seq_k + x0) * Kd);
#pragma unroll 4
    for (int c = tid; c < (GEN ? cols : BX) * NCZ; c += Nthreads)
      *reinterpret_cast<u4v*>(out + (size_t)c * 16) = *reinterpret_cast<const u4v*>(smem + c / NCZ * T::kOStride + c % NCZ * 16);
  };
  if (id.parts > 1) {                             // to the end in here: joined again, the two paths' accumulators cost 68 bytes of scratch
    float none[1];
    if (combine_parts<0, Nthreads>(in_parts, id, acc, none, smem)) finish();
    return;
  }
  finish();
}

}  // namespace aat
