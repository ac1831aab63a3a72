// RetNet recurrent form  S_n = a_n * S_{n-1} + k_n^T v_n,  out_n = q_n S_n  (fp32, per-position decay a).
//
// Same result as reference csrc/kernels/retnet/recurrent/recurrent.h:133-463 (a CUB BlockScan over
// (decay, k*v) pairs, one scan per (key dim, value dim) pair, launched by retnet_recurrent_fwd :427-463),
// same tensors: q, k [B, H, kdim, L], v, out [B, H, vdim, L] (sequence contiguous), decay [H, L].
//
// The scan is evaluated chunk by chunk on the matrix cores instead of element by element on the
// vector ALU.  For a chunk of 32 positions, with State = S at the end of the previous chunk:
//   S^T[m][n]  = sum_kd K[kd][m] Q[kd][n]                          (keys m x queries n)
//   P[m][n]    = S^T[m][n] * prod_{m<j<=n} a_j  (0 for m > n)      exact running products, no logarithms
//   O^T[vd][n] = p_n * sum_kd State[kd][vd] Q[kd][n] + sum_m V[vd][m] P[m][n],   p_n = prod_{j<=n} a_j
//   State[kd][vd] = A * State[kd][vd] + sum_m K[kd][m] w_m V[vd][m],   w_m = prod_{j>m} a_j, A = prod_j a_j
// which is 5 flops per (position, kd, vd) -- what the element-wise recurrence itself costs -- but at the
// matrix cores' rate.  No logarithms or divisions: zero and negative decays behave as in the recurrence.
//
// One block owns one (batch, head) and a slice of DVS value dims; wave w owns value dims [32w, 32w+32) of
// the slice: its State tiles (KD x 32, fp32, in registers for the whole sequence) and its rows of O^T.
// Products of 32 x 32 tiles are fp32 matrix instructions (v_mfma_f32_32x32x2_f32) or, where that is the faster way, bf16 ones
// (v_mfma_f32_32x32x16_bf16) of the operands' parts (RecOp).  Lane l, half h = l/32, column j = l%32 of an fp32 one:
//   A (32 x 2): lane holds A[j][h];  B (2 x 32): lane holds B[h][j];  C (32 x 32): lane holds C[8g+4h+e][j].
// The contraction index of a step is free as long as A and B agree, so step (g, e) is given the index
// 8g+4h+e: then the C registers of one product ARE the A or B operand of the next (State feeds
// State^T*Q, P feeds V*P) and no value ever changes lanes.  The bf16 ones take 16 indices at a time in the same order.
// S^T is split over the waves along kd (each wave contracts KD/waves key dims), the partial tiles are
// summed through LDS; every other product is private to its wave.
#pragma once
#include "kernels/utils/cdna4.h"
#include "kernels/utils/tile_ops.h"

namespace aat {

AAT_DEV f16v mfma_32x32x2_f32(float a, float b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------------------------------
// LDS tile of ROWS x 32 floats (8 chunks of 16 bytes per row).  Row r sits at position pos(r) = r with
// bits 0 and 2 exchanged, chunk c of the row at position p in slot c ^ ((p >> 1) & 7).
//  * reads along the sequence (one dword per lane, lanes 0-31 one row, lanes 32-63 the row 4 below):
//    the two rows land on positions of different parity, i.e. on different halves of the 64 banks;
//  * reads across rows (one 16-byte chunk per lane, 16 consecutive rows per 256-byte LDS cycle): the
//    slot term is a bijection of the 16 positions onto the 16 slots.
AAT_DEV constexpr int rec_pos(int r) { return (r & ~5) | ((r & 1) << 2) | ((r >> 2) & 1); }
AAT_DEV constexpr int rec_slot(int p, int c) { return c ^ ((p >> 1) & 7); }
AAT_DEV constexpr int rec_off(int r, int col) {                       // byte offset of element (r, col)
  const int p = rec_pos(r);
  return p * 128 + rec_slot(p, col >> 2) * 16 + (col & 3) * 4;
}
constexpr bool rec_row_reads_conflict_free() {
  for (int r = 0; r < 32; ++r) {
    if (r & 4) continue;
    unsigned long long seen = 0;
    for (int l = 0; l < 64; ++l) {
      const int bank = (rec_off(r + 4 * (l >> 5), l & 31) >> 2) & 63;
      if (seen >> bank & 1ull) return false;
      seen |= 1ull << bank;
    }
  }
  return true;
}
constexpr bool rec_column_reads_conflict_free() {
  for (int r0 = 0; r0 < 32; r0 += 16)
    for (int c = 0; c < 8; ++c) {
      unsigned seen = 0;
      for (int i = 0; i < 16; ++i) {
        const int slot = (rec_off(r0 + i, 4 * c) >> 4) & 15;
        if (seen >> slot & 1u) return false;
        seen |= 1u << slot;
      }
    }
  return true;
}
static_assert(rec_row_reads_conflict_free() && rec_column_reads_conflict_free(),
              "both access patterns of the fp32 chunk tiles are free of LDS bank conflicts");

// ---------------------------------------------------------------------------------------------------
// Decay factors of one (head, chunk), computed once, by retnet_recurrent_factors or, beyond 128 key dims, by the first blocks of
// retnet_recurrent_pmat, and shared by every batch entry and value slice.
//
// State is kept as T = State / lambda with a per-head scalar lambda (the product of the decays since
// the last rescale), so that a chunk's decay does not have to be multiplied into the KD x DVS state:
//   O^T = (p_n lambda) (T^T Q) + V P,      T += K diag(w / lambda') V^T,   lambda' = A lambda.
// When |lambda'| leaves [2^-40, 2^40] (or is zero) the record says so: the kernel then multiplies T by
// `scale` = A lambda once and lambda restarts at 1.
//   [0, 4096)     D[g][lane][e]   = prod_{m<j<=n} a_j for m = 8g+4h+e, n = lane%32, h = lane/32 (0 for m > n); not written
//                                   by retnet_recurrent_pmat, which multiplies P by it, and not read after it
//   [4096, 4224)  W[h][g][e]      = w_m / lambda'      (w_m alone on a rescale)
//   [4224, 4352)  PNL[n]          = p_n lambda
//   [4352, 4360)  rescale flag (uint32), scale
constexpr int kRecFactorBytes = 5120;
constexpr int kRecFactorW = 4096, kRecFactorPnl = 4224, kRecFactorFlag = 4352;

// decay [H][L] -> factors [H][L/32][kRecFactorBytes], for part `part` of `parts` of head `head`'s sequence, by a block of
// WAVES waves with 8 bytes of dynamic LDS per chunk.  WITH_D: the D of the records too.  A head's chunks are shared out over the
// blocks of its row and the waves of a block.  Each block walks lambda from the first chunk to its own last one by itself (a product per thread and chunk, then one wave chains
// them); lambda is known before a record is written, so a record is written once.
//
// Bound by latency: a load, the walk (one dependent multiplication and comparison per chunk), a load and 32 products, a store.
template <int WAVES, bool WITH_D>
AAT_DEV void rec_factor_records(const float* __restrict__ decay, char* __restrict__ factors, int L, int head, int part, int parts) {
  extern __shared__ __align__(16) float fsm[];     // per chunk: A, then lambda before the chunk; and A lambda
  const int lane = threadIdx.x & 63, n = lane & 31, hi = lane >> 5, nchunk = L / 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per_block = (nchunk + parts - 1) / parts;
  const int first = part * per_block, last = min(nchunk, first + per_block);
  if (first >= last) return;
  const float* const dh = decay + (size_t)head * L;
  for (int c = threadIdx.x; c < last; c += WAVES * 64) {
    typedef f4v f4v_dword __attribute__((aligned(4)));                    // decay may start at any float
    const f4v_dword* p = reinterpret_cast<const f4v_dword*>(dh + (size_t)c * 32);
    f4v x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = p[i];
    float w = 1.f;
#pragma unroll
    for (int m = 31; m >= 0; --m) w *= x[m / 4][m % 4];
    fsm[2 * c] = w;                                                                    // A
  }
  __syncthreads();
  if (wave == 0) {
    float lam = 1.f;
    for (int base = 0; base < last; base += 64) {
      const float a = base + lane < last ? fsm[2 * (base + lane)] : 1.f;
      const int count = min(64, last - base);
      float before = 1.f, after = 1.f;
      for (int i = 0; i < count; ++i) {
        const float lam_new = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(a), i)) * lam;
        const float mag = __builtin_fabsf(lam_new);
        before = lane == i ? lam : before;
        after = lane == i ? lam_new : after;
        lam = mag >= 0x1p-40f && mag <= 0x1p40f ? lam_new : 1.f;
      }
      if (lane < count) {
        fsm[2 * (base + lane)] = before;
        fsm[2 * (base + lane) + 1] = after;
      }
    }
  }
  __syncthreads();
  for (int c = first + wave; c < last; c += WAVES) {
    const float* dg = dh + (size_t)c * 32;
    char* rec = factors + ((size_t)head * nchunk + c) * kRecFactorBytes;
    const float lam = fsm[2 * c], lam_new = fsm[2 * c + 1], mag = __builtin_fabsf(lam_new);
    const bool rescale = !(mag >= 0x1p-40f && mag <= 0x1p40f);
    const float inv = rescale ? 1.f : 1.f / lam_new;
    float dsel[16], wsel[16];
    float d = 0.f, w = 1.f;
#pragma unroll
    for (int m = 31; m >= 0; --m) {     // exact running products, from the diagonal down
      if (m < 31) { d *= dg[m + 1]; w *= dg[m + 1]; }
      d = (m == n) ? 1.f : d;
      const int idx = (m >> 3) * 4 + (m & 3);
      if (m & 4) { dsel[idx] = d; wsel[idx] = w; }
      else { dsel[idx] = hi ? dsel[idx] : d; wsel[idx] = hi ? wsel[idx] : w; }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f4v x = {dsel[4 * g], dsel[4 * g + 1], dsel[4 * g + 2], dsel[4 * g + 3]};
      if constexpr (WITH_D) *reinterpret_cast<f4v*>(rec + g * 1024 + lane * 16) = x;
      if (n == 0) {
        f4v y = {wsel[4 * g] * inv, wsel[4 * g + 1] * inv, wsel[4 * g + 2] * inv, wsel[4 * g + 3] * inv};
        *reinterpret_cast<f4v*>(rec + kRecFactorW + hi * 64 + g * 16) = y;
      }
    }
    if (hi == 0) *reinterpret_cast<float*>(rec + kRecFactorPnl + n * 4) = d * dg[0] * lam;    // p_n lambda
    if (lane == 0) {
      *reinterpret_cast<uint32_t*>(rec + kRecFactorFlag) = rescale ? 1u : 0u;
      *reinterpret_cast<float*>(rec + kRecFactorFlag + 4) = lam_new;
    }
  }
}

// Grid (H, parts of the sequence).
constexpr int kRecFactorThreads = 1024;
constexpr int kRecFactorWaves = kRecFactorThreads / 64;
__global__ __launch_bounds__(kRecFactorThreads) void retnet_recurrent_factors(const float* __restrict__ decay,
                                                                              char* __restrict__ factors, int L) {
  rec_factor_records<kRecFactorWaves, true>(decay, factors, L, blockIdx.x, blockIdx.y, gridDim.y);
}

// ---------------------------------------------------------------------------------------------------
// Operands of a contraction over 16 key dims or positions (one k-step): element j of half h stands for index 8(j/4)+4h+j%4
// of the step, the rows that registers 8s .. 8s+7 of a C tile hold, so the registers of one product are an operand of the next.
//
// FP32 = false, taken first: an fp32 value is the sum of three bf16 ones (hi, mid, lo: 8 significant bits each, rounded to
// nearest), and a product the sum of the six largest of their nine, on v_mfma_f32_32x32x16_bf16: 6 x 32 cycles for 16 indices
// where v_mfma_f32_32x32x2_f32 takes 8 x 64.  What is left out is below 2^-23 of a product and 2^-26 of it on average, less than
// the rounding of one fp32 addition.  A sum is rounded six times per k-step
// instead of eight, and results are no further from 64 bits than with fp32 products: relative 2-norm at B8 H32 L512 128/128
// 7.58e-7 -> 7.26e-7, most of it from the products of decays both have in common; with decays in [0.5, 1] 1.28e-7 -> 9.5e-8; the
// same with normal or positive values, magnitudes spread over 12 decades along the key dims, or products around 1e-24.
// bf16 ends where fp32 does upwards, but at 2^-133 downwards (conversion, v_dot2 and matrix instructions keep subnormals), so the parts of a
// value below 2^-110 would hold fewer than its 24 bits.  Therefore Q, K and V are multiplied by kRecUp = 2^16, with which every fp32 value
// there is has parts that are exact; sums carry the powers along (S^T, the State and P 2^32, outputs 2^48: the inputs of the products that
// follow have more room below than they need) and outputs are scaled back at the end.
// An infinity (or a value, or a sum, that the scale or bf16's rounding takes there: inputs from 2^112 on, outputs from 2^80, from 2^40
// where lambda is 2^-40) becomes a NaN in its parts: a block that finds a value in its output that
// is not finite runs once more from the start with FP32 = true, which scales nothing.
// FP32 = true: eight fp32 values and eight v_mfma_f32_32x32x2_f32.
template <bool FP32> struct RecOp {
  static constexpr int kParts = FP32 ? 2 : 3;
  u4v p[kParts];
};
typedef __bf16 rec_bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 rec_bf2 __attribute__((ext_vector_type(2)));
constexpr float kRecUp = 0x1p16f, kRecDown = 0x1p-48f;
template <bool FP32> AAT_DEV f4v rec_up(f4v x) { return FP32 ? x : x * kRecUp; }

// ALONE: where no matrix instruction is under way the remainder x - hi is one v_dot2_f32_bf16 (times -1 and 0, exact) instead of a
// shift or mask and a subtraction; it shares the matrix core's issue path and waits there for a matrix instruction to end.
template <bool FP32, bool ALONE = false> AAT_DEV RecOp<FP32> rec_op(f4v a, f4v b) {
  RecOp<FP32> o;
  if constexpr (FP32) {
    __builtin_memcpy(&o.p[0], &a, 16);
    __builtin_memcpy(&o.p[1], &b, 16);
  } else {
    // -1 in one half and 0 in the other; in scalar registers, for as constants the compiler writes both as the inline -1.0
    uint32_t minus1_lo = 0x0000bf80u, minus1_hi = 0xbf800000u;
    if constexpr (ALONE) asm("" : "+s"(minus1_lo), "+s"(minus1_hi));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x0 = i < 2 ? a[2 * i] : b[2 * i - 4], x1 = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const f2v x = {x0, x1};
        const rec_bf2 r = __builtin_convertvector(x, rec_bf2);
        uint32_t bits;
        __builtin_memcpy(&bits, &r, 4);
        o.p[t][i] = bits;
        if constexpr (ALONE) {
          if (t < 2) {
            x0 = __builtin_amdgcn_fdot2_f32_bf16(r, __builtin_bit_cast(rec_bf2, minus1_lo), x0, false);
            x1 = __builtin_amdgcn_fdot2_f32_bf16(r, __builtin_bit_cast(rec_bf2, minus1_hi), x1, false);
          }
        } else if (t < 2) {
          x0 -= __uint_as_float(bits << 16);
          x1 -= __uint_as_float(bits & 0xffff0000u);
        }
      }
    }
  }
  return o;
}
AAT_DEV f4v rec_quarter(const f16v& c, int v0) { return f4v{c[v0], c[v0 + 1], c[v0 + 2], c[v0 + 3]}; }
template <bool FP32> AAT_DEV RecOp<FP32> rec_op_of_c(const f16v& c, int s) {      // registers 8s .. 8s+7
  return rec_op<FP32>(rec_quarter(c, 8 * s), rec_quarter(c, 8 * s + 4));
}
// c += a b over the 16 indices of the step, the small partial products first.
template <bool FP32> AAT_DEV f16v rec_mma(const RecOp<FP32>& a, const RecOp<FP32>& b, f16v c) {
  if constexpr (FP32) {
#pragma unroll
    for (int j = 0; j < 8; ++j) c = mfma_32x32x2_f32(__uint_as_float(a.p[j >> 2][j & 3]), __uint_as_float(b.p[j >> 2][j & 3]), c);
  } else {
    constexpr int ai[6] = {2, 0, 1, 1, 0, 0}, bi[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      rec_bf8 x, y;
      __builtin_memcpy(&x, &a.p[ai[t]], 16);
      __builtin_memcpy(&y, &b.p[bi[t]], 16);
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    }
  }
  return c;
}
// Keeps an operand's making where it is written: the compiler moves it to its use otherwise, past a branch in between.
template <bool FP32> AAT_DEV void rec_pin(RecOp<FP32>& o) {
#pragma unroll
  for (int p = 0; p < RecOp<FP32>::kParts; ++p) asm volatile("" : "+v"(o.p[p]));
}
// Order of a region of the program: READS LDS reads, then each of a k-step's six matrix instructions with VALU vector instructions behind
// it, which issue while it runs.  Ends the region.
template <bool FP32, int READS, int VALU> AAT_DEV void rec_interleave() {
  if constexpr (!FP32) {
    if constexpr (READS > 0) __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, VALU, 0);
    }
  }
  sched_fence();
}
// The largest bit patterns seen, as signed and as unsigned numbers: beyond the infinities' once a value was not finite.
struct RecFinite {
  int32_t pos = 0;
  uint32_t neg = 0;
  AAT_DEV void see(const f16v& x) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t b = __float_as_uint(x[i]);
      pos = max(pos, (int32_t)b);
      neg = max(neg, b);
    }
  }
  AAT_DEV bool broken() const { return pos >= 0x7f800000 || neg >= 0xff800000u; }
};
// Whether any lane of the block says so; also a barrier in front of what the caller does with LDS next.
AAT_DEV bool rec_any_wave(char* smem, bool x) {
  const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  int* const flags = reinterpret_cast<int*>(smem);
  block_sync();
  flags[wave] = __ballot(x) != 0ull;
  block_sync();
  int any = 0;
  for (int i = 0; i < waves; ++i) any |= flags[i];
  block_sync();
  return __builtin_amdgcn_readfirstlane(any) != 0;
}

template <int KD, int DVS>
struct RetRecurrent {
  static constexpr int kChunk = 32;                       // positions per step
  static constexpr int kWaves = DVS / 32;
  static constexpr int kThreads = kWaves * 64 + 128;       // the matrix waves plus two that move the data
  static constexpr int kKB = KD / 32;                     // State tiles per wave
  static constexpr int kSteps = KD / 16;                  // k-steps over the key dims
  static constexpr int kUnits = kSteps / kWaves;          // of them, a wave's share of S^T and of the operands made for all waves
  static constexpr int kKTile = KD * 128, kVTile = DVS * 128;
  static constexpr int kQOff = kKTile, kVOff = 2 * kKTile, kFOff = 2 * kKTile + kVTile;
  static constexpr int kStage = kFOff + kRecFactorBytes;  // K, Q, V tiles and decay factors of one chunk
  static constexpr int kOpOff = 2 * kStage;               // operands of Q, then of K, made for all waves: 3 parts of 1 KB per unit
  static constexpr int kSmemBytes = kOpOff + 2 * kSteps * 3072;
  // Once the waves have taken a chunk over, their partial S^T tiles lie where K was (and Q: 64 key dims, four waves), and each wave's
  // output tile where its rows of V were.
  static_assert(kWaves * 4096 <= (KD == 64 && DVS == 128 ? 2 : 1) * kKTile, "partial tiles");
  static_assert(KD % 32 == 0 && DVS % 64 == 0 && DVS <= 256, "tile shape");
  static_assert(kSteps % kWaves == 0, "the waves share the k-steps evenly");
  static_assert(kSmemBytes <= 160 * 1024, "LDS");
  // Byte offset, from kOpOff, of part p of the operand of unit u (Q: k-step u over the key dims; K: k-step u%2 over the positions of State tile u/2).
  AAT_DEV static constexpr int op_at(bool of_q, int u, int p) { return ((of_q ? 0 : kSteps) + u) * 3072 + p * 1024; }
};

// q, k: [B*H][kdim][L]; v, out: [B*H][vdim][L]; factors: output of retnet_recurrent_factors.  Contracts
// the first KD key dims (the reference's block_kdim, reference recurrent.h:290,427).  Grid (vdim / DVS, B*H).
//
// Waves 0 .. DVS/32-1 do the arithmetic; the last two waves of the block only move data: they issue every LDS-DMA copy and store
// the previous chunk's output tiles from their LDS staging area.  An LDS-DMA or store instruction holds its wave for 16 to 50
// cycles, which a matrix wave would spend with the matrix core idle.
//
// A chunk has two phases.  In the first a wave reads its share of K and Q, makes their operands (44 vector instructions for eight
// values, so once per block and not once per wave) and leaves them in LDS; behind a barrier every wave reads all of them.  The
// second is a sequence of k-steps: six matrix instructions, with the vector instructions that make a later k-step's operand of
// T, V or P between them (7 fit behind one) and the LDS reads of the next k-step.
//
// Bound by the board's power: some 8000 cycles a chunk (120 matrix instructions = 3840, 1100 vector instructions and 450 KB through LDS)
// run at 2.35 GHz without the memory stream and at 1.8 GHz with it; the stream by itself takes 270 us of the 328 at B8 H32 L2048
// 128/128.  Whole calls on inputs that change, fp32 products and one data wave before, this kernel now: B8 H32 L2048 128/128 368 -> 328 us
// (L512 96 -> 87), 64/128 234 -> 222, 64/64 209 -> 184; 170 of the vector instructions and 14 of the 328 us go into the scale and into decay
// factors that stay with V.  Tried and not kept: two
// chunks' copies under way at all times, at the price of factors read from memory and a fourth barrier, 331 us; non-temporal copies or
// stores +-3 %.
template <bool FP32, int KD, int DVS>
AAT_DEV bool rec_scan(char* smem, const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                      const char* __restrict__ factors, float* __restrict__ out, int heads, int kdim, int vdim, int L) {
  using T = RetRecurrent<KD, DVS>;
  using Op = RecOp<FP32>;

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.y, h = bh % heads;
  const int nchunk = L / T::kChunk;
  const char* fg = factors + (size_t)h * nchunk * kRecFactorBytes;
  const int pitch = L * 4;
  // Output: a wave's O^T tile goes through LDS so that it leaves as four 16-byte-per-lane stores (8 rows
  // x 128 bytes each) instead of sixteen 4-byte ones.  Row r of the tile sits at position r ^ ((r>>2)&1):
  // the two rows a write covers (r, r+4) and the two rows a 16-lane read phase covers (2m, 2m+1) then
  // fall on different halves of the banks.
  const int orl = lane >> 3, occ = lane & 7;

  if (wave >= T::kWaves) {
    // ================================ data waves ================================================
    // LDS-DMA of a tile of 128-byte rows: instruction i covers positions 8i .. 8i+7, lane l position
    // 8i + l/8, chunk slot l%8.  The source row is rec_pos(position), the source chunk the slot XOR the
    // position's slot term (whose high bit is the parity of i).  Every address below is a scalar base that
    // moves with the chunk plus a per-lane 32-bit offset computed here once.
    const char* qg = reinterpret_cast<const char*>(q + (size_t)bh * kdim * L);
    const char* kg = reinterpret_cast<const char*>(k + (size_t)bh * kdim * L);
    const char* vg = reinterpret_cast<const char*>(v + ((size_t)bh * vdim + (size_t)blockIdx.x * DVS) * L);
    constexpr int kTileOps = (KD > DVS ? KD : DVS) / 8;
    uint32_t toff[kTileOps];
#pragma unroll
    for (int i = 0; i < kTileOps; ++i)
      toff[i] = (uint32_t)((8 * i + rec_pos(orl)) * pitch + (occ ^ (((i & 1) << 2) | (orl >> 1))) * 16);
    auto dma_one = [&](const char* g_uniform, uint32_t lane_off, char* lds) {   // written out: scalar base + lane offset form
      const uint64_t base = (uint64_t)(uintptr_t)g_uniform;
      const uint32_t dst = (uint32_t)(uintptr_t)(AAT_AS3 char*)lds;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :: "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
    };
    auto dma_k = [&](int c, int stage) {
#pragma unroll
      for (int i = 0; i < KD / 8; ++i) dma_one(kg + (size_t)c * T::kChunk * 4, toff[i], smem + stage * T::kStage + i * 1024);
    };
    auto dma_q = [&](int c, int stage) {
#pragma unroll
      for (int i = 0; i < KD / 8; ++i) dma_one(qg + (size_t)c * T::kChunk * 4, toff[i], smem + stage * T::kStage + T::kQOff + i * 1024);
    };
    auto dma_vf = [&](int c, int stage) {
      char* const s = smem + stage * T::kStage;
#pragma unroll
      for (int i = 0; i < DVS / 8; ++i) dma_one(vg + (size_t)c * T::kChunk * 4, toff[i], s + T::kVOff + i * 1024);
#pragma unroll
      for (int i = 0; i < kRecFactorBytes / 1024; ++i)
        dma_one(fg + (size_t)c * kRecFactorBytes + i * 1024, lane * 16, s + T::kFOff + i * 1024);
    };
    // output tiles of chunk c: one per matrix wave, four 8-row groups each; all reads first, one wait, then
    // the stores back to back, each a scalar base plus one of 16 precomputed lane offsets
    uint32_t ooff[T::kWaves][4];
#pragma unroll
    for (int w = 0; w < T::kWaves; ++w)
#pragma unroll
      for (int i = 0; i < 4; ++i) ooff[w][i] = (uint32_t)(((32 * w + 8 * i + orl) * L + occ * 4) * 4);
    const char* const oread = smem + T::kVOff + (orl ^ ((orl >> 2) & 1)) * 128 + occ * 16;
    float* const og = out + ((size_t)bh * vdim + (size_t)blockIdx.x * DVS) * L;
    const auto store_tiles = [&](const f4v (&x)[T::kWaves][4], int c) {
      wait_lgkm0();
      const uint64_t base = (uint64_t)(uintptr_t)(og + (size_t)c * T::kChunk);
#pragma unroll
      for (int w = 0; w < T::kWaves; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("global_store_dwordx4 %0, %1, %2" :: "v"(ooff[w][i]), "v"(x[w][i]), "s"(base) : "memory");
    };
    // The first requests K and Q, the second V and the factors and stores the output.  Q's place is free from a chunk's second
    // barrier on, the others' when the chunk is done.  Memory operations of a wave complete in order.
    constexpr bool kQEarly = T::kWaves * 4096 <= T::kKTile;
    constexpr int kKOps = KD / 8, kVfOps = DVS / 8 + kRecFactorBytes / 1024;
    if (wave == T::kWaves) {
      dma_k(0, 0);
      dma_q(0, 0);
      if (kQEarly && nchunk > 1) {
        dma_q(1, 1);
        wait_vmcnt<kKOps>();
      } else {
        wait_vmcnt<0>();
      }
      for (int c = 0; c < nchunk; ++c) {
        block_sync();                                      // chunk c is in LDS; the matrix waves are done with chunk c-1
        if (c + 1 < nchunk) {
          dma_k(c + 1, (c + 1) & 1);
          if (!kQEarly) dma_q(c + 1, (c + 1) & 1);
        }
        block_sync();                                      // they have taken chunk c over
        if (kQEarly && c + 2 < nchunk) dma_q(c + 2, c & 1);
        block_sync();                                      // (their partial S^T are in LDS)
        if (kQEarly && c + 2 < nchunk) wait_vmcnt<kKOps>();
        else wait_vmcnt<0>();                              // the next chunk has landed
      }
      block_sync();
    } else {
      f4v x[T::kWaves][4];
      const auto read_tiles = [&](int c) {
#pragma unroll
        for (int w = 0; w < T::kWaves; ++w)
#pragma unroll
          for (int i = 0; i < 4; ++i) x[w][i] = *reinterpret_cast<const f4v*>(oread + (c & 1) * T::kStage + w * 4096 + i * 1024);
        wait_lgkm0();
      };
      dma_vf(0, 0);
      wait_vmcnt<0>();
      for (int c = 0; c < nchunk; ++c) {
        block_sync();
        if (c > 0) read_tiles(c - 1);
        if (c + 1 < nchunk) dma_vf(c + 1, (c + 1) & 1);
        block_sync();
        if (c > 0) store_tiles(x, c - 1);
        block_sync();
        if (c > 0) wait_vmcnt<4 * T::kWaves>();            // the next chunk has landed; the stores may still be under way
        else wait_vmcnt<0>();
      }
      block_sync();                                        // the last chunk's tiles are staged
      read_tiles(nchunk - 1);
      store_tiles(x, nchunk - 1);
      wait_vmcnt<0>();
    }
    return false;
  }

  // ================================ matrix waves ================================================
  const int ow_even = T::kVOff + wave * 4096 + n * 4 + 5 * hi * 128;        // write offset for e even: position 4h + h
  const int ow_odd = T::kVOff + wave * 4096 + n * 4 + (3 * hi + 1) * 128;   // e odd: position 4h + (1 - h)

  // Per-lane LDS offsets inside a stage.
  //  row read (row 8G+4h+e, column n): the slot term of the row is the compile-time constant
  //  sw(G, e) = 4(G&1) + 2(e&1) + (e>>1), folded into the lane part by XOR; the row goes into the offset.
  //  column read (16-byte chunk 2g+h of row n of a 32-row block): position and slot term are per lane.
  const uint32_t row_lane = hi * 128 + (n >> 2) * 16 + (n & 3) * 4;
  const int cp = rec_pos(n);
  uint32_t colb[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) colb[g] = cp * 128 + rec_slot(cp, 2 * g + hi) * 16;
  const uint32_t lane16 = lane * 16;
  // LDS offsets beyond 64 KB do not fit the instructions' offset field: one register for all the operands and partial tiles
  uint32_t op0 = T::kOpOff + lane16;
  asm volatile("" : "+v"(op0));
  char* const ops = smem + op0;
  char* const ops_own = ops + wave * T::kUnits * 3072;

  f16v st[T::kKB];
#pragma unroll
  for (int i = 0; i < T::kKB; ++i) st[i] = zero16();
  RecFinite finite;

  for (int c = 0; c < nchunk; ++c) {
    char* const sm = smem + (c & 1) * T::kStage;
    block_sync();      // chunk c is in LDS (the data waves waited for it); every wave is done with chunk c-1

    // ---- this wave's share of the operands of Q and of K
    Op qown[T::kUnits], kop[T::kUnits];
    f4v kx[T::kUnits][2], vx[4];
    {
      f4v qx[T::kUnits][2], kc[T::kUnits][2];
#pragma unroll
      for (int s = 0; s < T::kUnits; ++s) {
        const int u = wave * T::kUnits + s;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          // row 16u + 8(j/4) + 4h + j%4
          const int p0 = 8 * (j >> 2) + 4 * (j & 1) + (j & 2), sw = (p0 >> 1) & 7;
          const uint32_t at = u * 2048 + p0 * 128 + (row_lane ^ (sw << 4));
          qx[s][j >> 2][j & 3] = *reinterpret_cast<const float*>(sm + T::kQOff + at);
          kx[s][j >> 2][j & 3] = *reinterpret_cast<const float*>(sm + at);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
          kc[s][i] = *reinterpret_cast<const f4v*>(sm + (u >> 1) * 4096 + cp * 128 + (rec_slot(cp, hi) ^ (4 * (u & 1) + 2 * i)) * 16);
      }
      Op kown[T::kUnits];
#pragma unroll
      for (int s = 0; s < T::kUnits; ++s) {
        qown[s] = rec_op<FP32, true>(rec_up<FP32>(qx[s][0]), rec_up<FP32>(qx[s][1]));
        kown[s] = rec_op<FP32, true>(rec_up<FP32>(kc[s][0]), rec_up<FP32>(kc[s][1]));
      }
#pragma unroll
      for (int s = 0; s < T::kUnits; ++s)
#pragma unroll
        for (int p = 0; p < Op::kParts; ++p) {
          *reinterpret_cast<u4v*>(ops_own + T::op_at(true, s, p)) = qown[s].p[p];
          *reinterpret_cast<u4v*>(ops_own + T::op_at(false, s, p)) = kown[s].p[p];
        }
#pragma unroll
      for (int g = 0; g < 4; ++g) vx[g] = rec_up<FP32>(*reinterpret_cast<const f4v*>(sm + T::kVOff + wave * 4096 + colb[g]));
      kop[0] = rec_op<FP32, true>(rec_up<FP32>(kx[0][0]), rec_up<FP32>(kx[0][1]));
    }
    block_sync();
    const auto read_op = [&](bool of_q, int u) {
      Op o;
#pragma unroll
      for (int p = 0; p < Op::kParts; ++p) o.p[p] = *reinterpret_cast<const u4v*>(ops + T::op_at(of_q, u, p));
      return o;
    };

    // From here to the end of the chunk: a region per k-step, its six matrix instructions with the vector instructions that make a
    // later region's operand between them, and the LDS reads of the next region.
    // ---- the wave's partial S^T
    f16v sp = zero16(), oacc = zero16();
    Op top, qop = read_op(true, 0);
    sched_fence();
    static_for<T::kUnits>([&](auto it) {
      constexpr int s = decltype(it)::value;
      if constexpr (s + 1 < T::kUnits) kop[s + 1] = rec_op<FP32>(rec_up<FP32>(kx[s + 1][0]), rec_up<FP32>(kx[s + 1][1]));
      else top = rec_op_of_c<FP32>(st[0], 0);
      sp = rec_mma<FP32>(kop[s], qown[s], sp);
      rec_interleave<FP32, 0, 8>();
    });

    // ---- T^T Q
    // w / lambda' goes with V as in the kernels below, before V is taken apart, at the price of two more operands a chunk: with K, whose
    // operands are made once, a factor of 2^-36 takes a K of 1e-28 out of fp32 where V has the room for it (B8 H32 L2048 128/128 315 -> 321 us).
    f4v wx[2];
    const auto read_w = [&](int s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) wx[i] = *reinterpret_cast<const f4v*>(sm + T::kFOff + kRecFactorW + hi * 64 + (2 * s + i) * 16);
    };
    Op vop[2], uop[2], pop[2];                             // V for V P, V w / lambda' for the State
    static_for<T::kSteps>([&](auto it) {
      constexpr int ks = decltype(it)::value;
      Op tnext, qnext;
      if constexpr (ks + 1 < T::kSteps) {
        qnext = read_op(true, ks + 1);
        if constexpr (ks + 2 == T::kSteps) read_w(0);
        tnext = rec_op_of_c<FP32>(st[(ks + 1) >> 1], (ks + 1) & 1);
        rec_pin(tnext);
      } else {
        uop[0] = rec_op<FP32>(vx[0] * wx[0], vx[1] * wx[1]);
        rec_pin(uop[0]);
        read_w(1);
      }
      oacc = rec_mma<FP32>(top, qop, oacc);
      rec_interleave<FP32, ks + 2 < T::kSteps ? 3 : ks + 1 < T::kSteps ? 5 : 2, 8>();
      if constexpr (ks == 1) {
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<f4v*>(sm + wave * 4096 + g * 1024 + lane16) = rec_quarter(sp, 4 * g);
        sched_fence();
      }
      top = tnext;
      qop = qnext;
    });
    f4v dd[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) dd[g] = *reinterpret_cast<const f4v*>(sm + T::kFOff + g * 1024 + lane16);
    const float pnl = *reinterpret_cast<const float*>(sm + T::kFOff + kRecFactorPnl + n * 4);
    Op wop = read_op(false, 0);
    const f4v flag = *reinterpret_cast<const f4v*>(sm + T::kFOff + kRecFactorFlag);
    if (__builtin_amdgcn_readfirstlane(__float_as_uint(flag[0])) != 0u) {   // lambda left its range: fold it into T
#pragma unroll
      for (int kb = 0; kb < T::kKB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kb][i] *= flag[1];
    }

    // ---- T += K diag(w / lambda') V^T, the positions 0-15 of every State tile first; meanwhile P, and
    // O^T = (p_n lambda) T^T Q + V P ahead of the last k-step, so that it has left the matrix core when it is stored
    f4v part[2][T::kWaves - 1];
    const auto read_partials = [&](int g0) {
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int t = 0; t < T::kWaves - 1; ++t) {
          const int w = wave + 1 + t < T::kWaves ? wave + 1 + t : wave + 1 + t - T::kWaves;
          part[g][t] = *reinterpret_cast<const f4v*>(sm + w * 4096 + (g0 + g) * 1024 + lane16);
        }
    };
    const auto add_partials = [&](int g0) {                // P of two row groups: the waves' partial sums times D
#pragma unroll
      for (int g = g0; g < g0 + 2; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int t = 0; t < T::kWaves - 1; ++t) sp[4 * g + e] += part[g - g0][t][e];
          sp[4 * g + e] *= dd[g][e];
        }
    };
    sched_fence();
    static_for<T::kSteps>([&](auto it) {
      constexpr int i = decltype(it)::value, kb = i % T::kKB, s = i / T::kKB;
      Op wnext;
      if constexpr (i + 1 < T::kSteps) wnext = read_op(false, 2 * ((i + 1) % T::kKB) + (i + 1) / T::kKB);
      constexpr auto at = [](int x) { return x * T::kSteps / 8; };
      if constexpr (i == at(0)) uop[1] = rec_op<FP32>(vx[2] * wx[0], vx[3] * wx[1]);
      if constexpr (i == at(1)) vop[0] = rec_op<FP32>(vx[0], vx[1]);
      if constexpr (i == at(2)) {
        add_partials(0);
        read_partials(2);
      }
      if constexpr (i == at(3)) pop[0] = rec_op_of_c<FP32>(sp, 0);
      if constexpr (i == at(4)) add_partials(2);
      if constexpr (i == at(5)) pop[1] = rec_op_of_c<FP32>(sp, 1);
      if constexpr (i == at(6)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[r] *= pnl;
        vop[1] = rec_op<FP32>(vx[2], vx[3]);
      }
      if constexpr (i == T::kSteps - 1) {
#pragma unroll
        for (int r = 0; r < 2; ++r) oacc = rec_mma<FP32>(vop[r], pop[r], oacc);
        sched_fence();
      }
      st[kb] = rec_mma<FP32>(wop, uop[s], st[kb]);
      rec_interleave<FP32, 3, 8>();
      if constexpr (i == at(0)) {
        block_sync();                                      // the partial S^T are in LDS
        read_partials(0);
      }
      wop = wnext;
    });
    finite.see(oacc);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<float*>(sm + (e & 1 ? ow_odd : ow_even) + (8 * g + (e & 2)) * 128) = FP32 ? oacc[4 * g + e] : oacc[4 * g + e] * kRecDown;
  }
  block_sync();               // the last chunk's output tiles are staged: the data wave stores them
  return finite.broken();
}

template <int KD, int DVS>
__global__ __launch_bounds__(DVS * 2 + 128) __attribute__((amdgpu_waves_per_eu(2, 2))) void retnet_recurrent_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const char* __restrict__ factors, float* __restrict__ out, int heads, int kdim, int vdim, int L) {
  extern __shared__ __align__(16) char smem[];
  const bool broken = rec_scan<false, KD, DVS>(smem, q, k, v, factors, out, heads, kdim, vdim, L);
  if (rec_any_wave(smem, broken)) rec_scan<true, KD, DVS>(smem, q, k, v, factors, out, heads, kdim, vdim, L);
}

// ---------------------------------------------------------------------------------------------------
// P of every (batch, head, chunk) for the kernels below, as C registers: [B*H][L/32][g][lane][e], 4 KB per chunk.  One block
// per chunk; its waves split the key dims, read q and k straight from memory (rows of 128 bytes, each used once) and wave w adds
// up row group w and multiplies it by D.  Bound by the read of q and k.
// OPS: also the operands of Q and K for retnet_recurrent_stream_kernel, [B*H][L/32][KD/16 of Q, KD/16 of K][part][lane][16 B];
// bound by their 12 bytes per key dim and position (B2 H8 L1056, 256 key dims: 8.8 us without them, 17 with).
//
// The first heads * parts blocks of the launch make the records of the decay factors instead, 8 bytes of dynamic LDS per chunk
// (the kernel below waits for both anyway): D, which P needs, depends on its own chunk only, and every wave forms its 8 rows
// while its loads are under way, in the order of the records.  B2 H8 L1056 256/512: 94.4 us a call with a launch of its own for the
// records (5.6 us and the gap behind it), 88.6 like this.  So also in long sequences, where the room of the records' walk in every
// block's LDS (48 KB with the static part at 131072 positions) takes places from the P blocks: B1 H8 L65536 256/128 5110 and 4988,
// B1 H8 L131072 256/64 10210 and 9948, B1 H2 L131072 192/64 9938 and 9871.
template <int KD, bool OPS>
__global__ __launch_bounds__(256) void retnet_recurrent_pmat(const float* __restrict__ q, const float* __restrict__ k,
                                                             const float* __restrict__ decay, char* __restrict__ factors,
                                                             char* __restrict__ pmat, char* __restrict__ ops, int heads, int parts, int kdim, int L) {
  __shared__ __align__(16) f4v part[4][4][64];
  const int records = heads * parts;
  if ((int)blockIdx.x < records) {
    rec_factor_records<4, false>(decay, factors, L, blockIdx.x / parts, blockIdx.x % parts, parts);
    return;
  }
  const int lane = threadIdx.x & 63, n = lane & 31, hi = lane >> 5, nchunk = L / 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_remap(blockIdx.x - records, gridDim.x - records), bh = tile / nchunk, c = tile % nchunk;
  constexpr int kUnits = KD / 64;                     // k-steps of 16 key dims of one wave
  const size_t at = ((size_t)bh * kdim + 16 * kUnits * wave + 4 * hi) * L + (size_t)c * 32 + n;
  f4v kx[kUnits][2], qx[kUnits][2];                   // rows 16u + 8(j/4) + 4h + j%4 of column n
#pragma unroll
  for (int s = 0; s < kUnits; ++s)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t row = at + (size_t)(16 * s + 8 * (j >> 2) + (j & 3)) * L;
      kx[s][j >> 2][j & 3] = k[row];
      qx[s][j >> 2][j & 3] = q[row];
    }
  // OPS: K once more, row n of State tiles wave and wave + 4: positions 8g + 4h .. + 3
  typedef f4v f4v_dword __attribute__((aligned(4)));  // q, k, v may start at any float
  constexpr int kTiles = KD / 32, kMine = (kTiles + 3) / 4;
  f4v kr[kMine][4];
  if constexpr (OPS) {
#pragma unroll
    for (int t = 0; t < kMine; ++t) {
      const int kb = wave + 4 * t < kTiles ? wave + 4 * t : wave % kTiles;
      const float* const row = k + ((size_t)bh * kdim + 32 * kb + n) * L + (size_t)c * 32 + 4 * hi;
#pragma unroll
      for (int g = 0; g < 4; ++g) kr[t][g] = *reinterpret_cast<const f4v_dword*>(row + 8 * g);
    }
  }
  sched_fence();                                      // all loads in flight before the first product
  const float* const dg = decay + (size_t)(bh % heads) * L + (size_t)c * 32;
  f4v dsel = {0.f, 0.f, 0.f, 0.f};                    // D of rows 8 wave + 4 hi + e
  float d = 0.f;
#pragma unroll
  for (int g = 3; g >= 0; --g) {
    f4v rows[2];
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      const int m = 8 * g + i;
      if (m < 31) d *= dg[m + 1];
      d = (m == n) ? 1.f : d;
      rows[i >> 2][i & 3] = d;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) dsel[e] = g == wave ? (hi ? rows[1][e] : rows[0][e]) : dsel[e];
  }
  f16v sp = zero16();
#pragma unroll
  for (int s = 0; s < kUnits; ++s) sp = rec_mma<true>(rec_op<true>(kx[s][0], kx[s][1]), rec_op<true>(qx[s][0], qx[s][1]), sp);
#pragma unroll
  for (int g = 0; g < 4; ++g) part[wave][g][lane] = rec_quarter(sp, 4 * g);
  if constexpr (OPS) {
    char* const mine = ops + ((size_t)bh * nchunk + c) * (2 * KD / 16) * 3072 + lane * 16;
#pragma unroll
    for (int s = 0; s < kUnits; ++s) {
      const RecOp<false> o = rec_op<false>(rec_up<false>(qx[s][0]), rec_up<false>(qx[s][1]));
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u4v*>(mine + (wave * kUnits + s) * 3072 + p * 1024) = o.p[p];
    }
#pragma unroll
    for (int t = 0; t < kMine; ++t)
      if (wave + 4 * t < kTiles) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const RecOp<false> o = rec_op<false>(rec_up<false>(kr[t][2 * s]), rec_up<false>(kr[t][2 * s + 1]));
#pragma unroll
          for (int p = 0; p < 3; ++p) *reinterpret_cast<u4v*>(mine + (KD / 16 + 2 * (wave + 4 * t) + s) * 3072 + p * 1024) = o.p[p];
        }
      }
  }
  __syncthreads();
  f4v x = part[0][wave][lane];
#pragma unroll
  for (int t = 1; t < 4; ++t) x += part[t][wave][lane];
  x *= dsel;
  *reinterpret_cast<f4v*>(pmat + ((size_t)bh * nchunk + c) * 4096 + wave * 1024 + lane * 16) = x;
}

// ---------------------------------------------------------------------------------------------------
// The same scan for problems whose 64- or 128-wide value slices leave compute units without a block, and for
// more key dims than those blocks hold: a block owns 32 value dims, and its waves split the key dims between
// them instead of the value dims.  Wave w holds State[KD/WK key dims][32]; its key dims contribute partial
// sums of S^T and of O^T, which are exchanged through LDS: every wave adds up 8 of the 32 rows of either
// (row group g of the C layout goes to wave g % WK), contracts its 8 positions of P with V, and stores its 8
// rows of the output.  Q is read once per wave and feeds both contractions.
//
// Bound by its fp32 matrix instructions, 64 cycles each: parts made by every wave for itself were slower (B2 H8 L1056 256/512 94 us
// against 87, made ahead see below).  A slice of 32 repeats S^T in every block, so a chunk has
// (3 KD + 32) / (2 KD + 32 + KD / 4) of the products of a 128-wide slice, 1.27 times (KD 64) and 1.30 (KD 128), against four times the
// blocks.  B4 H8 L2048 128/256, 256 blocks: 353 -> 145 us a call (the kernel above with fp32 products).
// All key dims are contracted in one pass, so nothing is written twice and added.  K, Q, V and the factors are
// double-buffered; S^T partials reuse the wave's own rows of the consumed Q tile.  The products D of the
// decays, 4 KB per chunk of which a wave needs the rows of its group, skip LDS, which at KD 256 has no room for them.
//
// PRE, taken beyond 128 key dims: P itself comes from global memory in the same layout, made once per (batch, head) by
// retnet_recurrent_pmat above, 4 KB per (batch, head, chunk).  That is a third of the matrix instructions of a wave (32 of 100 at KD
// 256: 68 x 64 cycles, 2.0 of 2.5 us a chunk) and the exchange of S^T, for one more read of q and k.  Whole calls, passes over 128 key
// dims -> one pass without PRE -> with it: B2 H8 L1056 256/512 376 -> 119 -> 94 us; B4 H16 L2048 192/256: 609 -> 466 -> 371.
template <int KD, int WK>
struct RetRecurrentSplit {
  static constexpr int kChunk = 32;
  static constexpr int kThreads = WK * 64 + 64;
  static constexpr int kRows = KD / WK;                    // key dims of one wave
  static constexpr int kKB = kRows / 32;                   // its State tiles
  static constexpr int kOwn = (4 + WK - 1) / WK;           // row groups of a C tile it adds up (the last may not exist)
  static constexpr int kQOff = KD * 128, kVOff = 2 * KD * 128, kFOff = kVOff + 4096;
  static constexpr int kFBytes = kRecFactorBytes - kRecFactorW;
  static constexpr int kStage = kFOff + kFBytes;
  static constexpr int kOutOff = 2 * kStage;               // per wave: its partial O^T tile
  static constexpr int kSmemBytes = kOutOff + WK * 4096;
  static_assert(KD % (32 * WK) == 0 && WK >= 2 && WK <= 4, "key dims per wave are whole State tiles");
  static_assert(kQOff + KD * 128 <= 65536, "row offsets go into the 16-bit offset field of the LDS reads");
  static_assert(kSmemBytes <= 160 * 1024, "LDS");
};

// LDS reads and stores issued by hand so that their waits can be counted: the compiler answers every
// dependency on an LDS load with lgkmcnt(0) while an LDS-DMA copy is in flight, and here one is in
// flight all the time.  LDS operations retire in order, so "at most N younger ones outstanding" is enough.
AAT_DEV float lds_read_f1_async(uint32_t base, int imm) {
  float v;
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(base), "i"(imm));
  return v;
}
template <int N, class V> AAT_DEV void lds_wait_younger_f(V& v) {
  static_assert(N >= 0 && N < 16, "lgkmcnt is a 4-bit counter");
  asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(N));
}

// Grid: B * H * vdim / 32 blocks, the slices of one (batch, head) on one XCD (they read the same q and k).
template <int KD, int WK, bool PRE>
__global__ __launch_bounds__(WK * 64 + 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void retnet_recurrent_split_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const char* __restrict__ factors, const char* __restrict__ pmat, float* __restrict__ out, int heads, int kdim, int vdim, int L) {
  using T = RetRecurrentSplit<KD, WK>;

  extern __shared__ __align__(16) char smem[];

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = xcd_remap(blockIdx.x, gridDim.x), slices = vdim / 32;
  const int bh = tile / slices, vd0 = (tile % slices) * 32, h = bh % heads;
  const int nchunk = L / T::kChunk;
  const char* fg = factors + (size_t)h * nchunk * kRecFactorBytes;

  if (wave == WK) {
    // Every address is a scalar base that moves with the chunk plus a per-lane 32-bit offset computed here once: the loop of this wave
    // must not contain a single vector instruction -- one has to find a gap between the fp32 MFMAs of the matrix wave that shares
    // the SIMD, and a copy that waits for one took 175 cycles to issue.
    const char* qg = reinterpret_cast<const char*>(q + (size_t)bh * kdim * L);
    const char* kg = reinterpret_cast<const char*>(k + (size_t)bh * kdim * L);
    const char* vg = reinterpret_cast<const char*>(v + ((size_t)bh * vdim + vd0) * L);
    const int orl = lane >> 3, occ = lane & 7, pitch = L * 4;
    uint32_t toff[KD / 8];
#pragma unroll
    for (int i = 0; i < KD / 8; ++i)
      toff[i] = (uint32_t)((8 * i + rec_pos(orl)) * pitch + (occ ^ (((i & 1) << 2) | (orl >> 1))) * 16);
    const uint32_t lane16off = lane * 16;
    auto dma_one = [&](const char* g_uniform, uint32_t lane_off, char* lds) {
      const uint64_t base = (uint64_t)(uintptr_t)g_uniform;
      const uint32_t dst = (uint32_t)(uintptr_t)(AAT_AS3 char*)lds;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :: "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
    };
    auto dma = [&](int c, int stage) {
      char* s = smem + stage * T::kStage;
      const size_t col = (size_t)c * T::kChunk * 4;
#pragma unroll
      for (int i = 0; i < KD / 8; ++i) dma_one(kg + col, toff[i], s + i * 1024);
#pragma unroll
      for (int i = 0; i < KD / 8; ++i) dma_one(qg + col, toff[i], s + T::kQOff + i * 1024);
#pragma unroll
      for (int i = 0; i < 4; ++i) dma_one(vg + col, toff[i], s + T::kVOff + i * 1024);
      dma_one(fg + (size_t)c * kRecFactorBytes + kRecFactorW, lane16off, s + T::kFOff);
    };
    dma(0, 0);
    wait_vmcnt<0>();
    for (int c = 0; c < nchunk; ++c) {
      asm volatile("s_barrier" ::: "memory");          // chunk c is in LDS; the matrix waves are done with chunk c-1
      if (c + 1 < nchunk) dma(c + 1, (c + 1) & 1);
      asm volatile("s_barrier" ::: "memory");          // (the matrix waves' barrier in front of the S^T sum)
      wait_vmcnt<0>();
    }
    asm volatile("s_barrier" ::: "memory");
    return;
  }

  const uint32_t lds0 = lds_addr(smem);
  const uint32_t row_lane = hi * 128 + (n >> 2) * 16 + (n & 3) * 4;
  const int cp = rec_pos(n);
  int own[T::kOwn];                                     // this wave's row groups; a missing one reads like its first
#pragma unroll
  for (int s = 0; s < T::kOwn; ++s) own[s] = wave + s * WK < 4 ? wave + s * WK : wave;
  const bool has_last = wave + (T::kOwn - 1) * WK < 4;

  constexpr int kNumBases = 8 + 4 + 4 + 2 * T::kOwn + 4;
  uint32_t bases[kNumBases];                            // LDS addresses that move to the other stage after every chunk
  uint32_t* const rowk = bases;                         // [8]  this wave's key dims along the sequence
  uint32_t* const colk = bases + 8;                     // [4]  K columns
  uint32_t* const colv = bases + 12;                    // [4]  V columns
  uint32_t* const vown = bases + 16;                    // [kOwn]  V columns of the wave's own positions
  uint32_t* const sown = vown + T::kOwn;                // [kOwn]  S^T partials of the own row groups
  uint32_t& wbase = sown[T::kOwn];
  uint32_t& pbase = sown[T::kOwn + 1];
  uint32_t& fbase = sown[T::kOwn + 2];
  uint32_t& smine = sown[T::kOwn + 3];                  // this wave's S^T partial
#pragma unroll
  for (int sw = 0; sw < 8; ++sw) rowk[sw] = lds0 + wave * T::kRows * 128 + (row_lane ^ (sw << 4));
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const uint32_t col = cp * 128 + rec_slot(cp, 2 * g + hi) * 16;
    colk[g] = lds0 + wave * T::kRows * 128 + col;
    colv[g] = lds0 + T::kVOff + col;
  }
#pragma unroll
  for (int s = 0; s < T::kOwn; ++s) {
    vown[s] = lds0 + T::kVOff + cp * 128 + rec_slot(cp, 2 * own[s] + hi) * 16;
    sown[s] = lds0 + own[s] * 1024 + lane * 16;
  }
  wbase = lds0 + T::kFOff + hi * 64;
  pbase = lds0 + T::kFOff + (kRecFactorPnl - kRecFactorW) + n * 4;
  fbase = lds0 + T::kFOff + (kRecFactorFlag - kRecFactorW);
  smine = lds0 + T::kQOff + wave * T::kRows * 128 + lane * 16;
  const uint32_t omine = lds0 + T::kOutOff + wave * 4096 + lane * 16;
  uint32_t oown[T::kOwn];
  float* orow[T::kOwn];
  const char* dptr[T::kOwn];
#pragma unroll
  for (int s = 0; s < T::kOwn; ++s) {
    oown[s] = lds0 + T::kOutOff + own[s] * 1024 + lane * 16;
    orow[s] = out + ((size_t)bh * vdim + vd0 + 8 * own[s] + 4 * hi) * L + n;
    dptr[s] = (PRE ? pmat + (size_t)bh * nchunk * 4096 : fg) + own[s] * 1024 + lane * 16;
  }
  auto lds_write_f4 = [&](uint32_t a, int imm_g, f4v x) {
    *reinterpret_cast<f4v*>(smem + (a - lds0) + imm_g * 1024) = x;
  };

  f16v st[T::kKB];
#pragma unroll
  for (int i = 0; i < T::kKB; ++i) st[i] = zero16();

  // One stream of LDS reads per chunk: rows of K and Q, the previous chunk's O^T
  // partials, flag, V, w, the K columns of one half of the State update, the S^T partials, p_n, the other half.
  constexpr int kPF = 6, kRing = kPF + 1, kOwn = T::kOwn;
  constexpr int nS1 = PRE ? T::kRows / 2 : T::kRows, nUpd = 4 * T::kKB, nHalf = nUpd / 2;
  constexpr int jO = nS1, jFlag = jO + kOwn * WK, jV = jFlag + 1, jW = jV + 4, jVo = jW + 4, jK1 = jVo + kOwn;
  constexpr int jRed = jK1 + nHalf, jPnl = jRed + (PRE ? 0 : kOwn * WK), jK2 = jPnl + 1, nElem = jK2 + nUpd - nHalf;
  static_assert(jRed - jO - kPF > kPF, "reads issued after the S^T stores have returned before the barrier that publishes them");

  auto chunk = [&](auto stage_tag, int c) {
    constexpr int S = decltype(stage_tag)::value;
    float fr[kRing];
    f4v vr[kRing];
    f16v sp = zero16(), oacc = zero16();
    f4v wv[4], vo[kOwn], pm[kOwn], dd[kOwn], ov[kOwn];
    float ka = 0.f;

    auto issue = [&](auto jt) {
      constexpr int j = decltype(jt)::value, slot = j % kRing;
      if constexpr (j < nS1) {
        constexpr int i = PRE ? j : j / 2, gg = i / 4, e = i % 4, p0 = 8 * gg + 4 * (e & 1) + (e & 2), sw = (p0 >> 1) & 7;
        fr[slot] = lds_read_f1_async(rowk[sw], (PRE || j % 2 ? T::kQOff : 0) + p0 * 128);
      } else if constexpr (j < jFlag) {
        vr[slot] = lds_read_f4_async(oown[(j - jO) / WK], (j - jO) % WK * 4096);
      } else if constexpr (j == jFlag) {
        vr[slot] = lds_read_f4_async(fbase, 0);
      } else if constexpr (j < jW) {
        vr[slot] = lds_read_f4_async(colv[j - jV], 0);
      } else if constexpr (j < jVo) {
        vr[slot] = lds_read_f4_async(wbase, (j - jW) * 16);
      } else if constexpr (j < jK1) {
        vr[slot] = lds_read_f4_async(vown[j - jVo], 0);
      } else if constexpr (j < jRed) {
        vr[slot] = lds_read_f4_async(colk[(j - jK1) % 4], (j - jK1) / 4 * 4096);
      } else if constexpr (j < jPnl) {
        vr[slot] = lds_read_f4_async(sown[(j - jRed) / WK], T::kQOff + (j - jRed) % WK * T::kRows * 128);
      } else if constexpr (j == jPnl) {
        fr[slot] = lds_read_f1_async(pbase, 0);
      } else {
        constexpr int u = nHalf + j - jK2;
        vr[slot] = lds_read_f4_async(colk[u % 4], u / 4 * 4096);
      }
    };

    auto consume = [&](auto jt) {
      constexpr int j = decltype(jt)::value, slot = j % kRing, younger = (nElem - 1 - j < kPF) ? nElem - 1 - j : kPF;
      if constexpr (j < nS1) {
        lds_wait_younger_f<younger>(fr[slot]);
        if constexpr (PRE) oacc = mfma_32x32x2_f32(st[j / 16][j % 16], fr[slot], oacc);
        else if constexpr (j % 2 == 0) ka = fr[slot];
        else {
          constexpr int i = j / 2;
          sp = mfma_32x32x2_f32(ka, fr[slot], sp);
          oacc = mfma_32x32x2_f32(st[i / 16][i % 16], fr[slot], oacc);
        }
        if constexpr (!PRE && j == nS1 - 1) {          // every row of Q has been read: its place takes the partial tile
#pragma unroll
          for (int g = 0; g < 4; ++g) lds_write_f4(smine, g, f4v{sp[4 * g], sp[4 * g + 1], sp[4 * g + 2], sp[4 * g + 3]});
          asm volatile("" ::: "memory");
        }
      } else if constexpr (j < jFlag) {
        constexpr int s = (j - jO) / WK, t = (j - jO) % WK;
        lds_wait_younger_f<younger>(vr[slot]);
        ov[s] = t == 0 ? vr[slot] : ov[s] + vr[slot];
        if constexpr (t == WK - 1) {
          if (c > 0 && (s + 1 < kOwn || has_last)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) orow[s][(size_t)e * L + (size_t)(c - 1) * T::kChunk] = ov[s][e];
          }
        }
      } else if constexpr (j == jFlag) {
        lds_wait_younger_f<younger>(vr[slot]);
        if (__builtin_amdgcn_readfirstlane(__float_as_uint(vr[slot][0])) != 0u) {   // lambda left its range: fold it into T
          const float sc = vr[slot][1];
#pragma unroll
          for (int kb = 0; kb < T::kKB; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) st[kb][i] *= sc;
        }
      } else if constexpr (j < jW) {
        lds_wait_younger_f<younger>(vr[slot]);
        wv[j - jV] = vr[slot];
      } else if constexpr (j < jVo) {
        lds_wait_younger_f<younger>(vr[slot]);
        wv[j - jW] *= vr[slot];
      } else if constexpr (j < jK1) {
        lds_wait_younger_f<younger>(vr[slot]);
        vo[j - jVo] = vr[slot];
      } else if constexpr (j < jRed) {
        constexpr int u = j - jK1;
        lds_wait_younger_f<younger>(vr[slot]);
#pragma unroll
        for (int e = 0; e < 4; ++e) st[u / 4] = mfma_32x32x2_f32(vr[slot][e], wv[u % 4][e], st[u / 4]);
      } else if constexpr (j < jPnl) {
        constexpr int s = (j - jRed) / WK, t = (j - jRed) % WK;
        lds_wait_younger_f<younger>(vr[slot]);
        pm[s] = t == 0 ? vr[slot] : pm[s] + vr[slot];
        if constexpr (t == WK - 1) pm[s] *= dd[s];
      } else if constexpr (j == jPnl) {
        lds_wait_younger_f<younger>(fr[slot]);
        // O^T = (p_n lambda) T^T Q + V P, over this wave's key dims and positions
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[i] *= fr[slot];
#pragma unroll
        for (int s = 0; s < kOwn; ++s)
          if (s + 1 < kOwn || has_last) {
#pragma unroll
            for (int e = 0; e < 4; ++e) oacc = mfma_32x32x2_f32(vo[s][e], PRE ? dd[s][e] : pm[s][e], oacc);
          }
      } else {
        constexpr int u = nHalf + j - jK2;
        lds_wait_younger_f<younger>(vr[slot]);
#pragma unroll
        for (int e = 0; e < 4; ++e) st[u / 4] = mfma_32x32x2_f32(vr[slot][e], wv[u % 4][e], st[u / 4]);
        if constexpr (j == nElem - 1) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            lds_write_f4(omine, g, f4v{oacc[4 * g], oacc[4 * g + 1], oacc[4 * g + 2], oacc[4 * g + 3]});
        }
      }
    };

    block_sync();        // chunk c is in LDS, chunk c-1's O^T partials are; every wave is done with chunk c-1
#pragma unroll
    for (int s = 0; s < kOwn; ++s) dd[s] = *reinterpret_cast<const f4v*>(dptr[s] + (size_t)c * (PRE ? 4096 : kRecFactorBytes));
    static_for<kPF>([&](auto jt) { issue(jt); });
    sched_fence();
    static_for<nElem>([&](auto jt) {
      constexpr int j = decltype(jt)::value;
      if constexpr (j + kPF < nElem) {
        if constexpr (j + kPF == jRed) asm volatile("s_barrier" ::: "memory");
        issue(std::integral_constant<int, j + kPF>{});
      }
      consume(jt);
      sched_fence();
    });
#pragma unroll
    for (int i = 0; i < kNumBases; ++i) bases[i] += (S == 0) ? T::kStage : -T::kStage;
  };

  for (int c = 0; c < nchunk; c += 2) {
    chunk(std::integral_constant<int, 0>{}, c);
    if (c + 1 < nchunk) chunk(std::integral_constant<int, 1>{}, c + 1);
  }
  block_sync();
#pragma unroll
  for (int s = 0; s < kOwn; ++s) {
    if (s + 1 < kOwn || has_last) {
      f4v x = *reinterpret_cast<const f4v*>(smem + (oown[s] - lds0));
#pragma unroll
      for (int t = 1; t < WK; ++t) x += *reinterpret_cast<const f4v*>(smem + (oown[s] - lds0) + t * 4096);
#pragma unroll
      for (int e = 0; e < 4; ++e) orow[s][(size_t)e * L + (size_t)(nchunk - 1) * T::kChunk] = x[e];
    }
  }
}

// ---------------------------------------------------------------------------------------------------
// The split scan with the operands of Q and K made once per (batch, head) ahead of it: retnet_recurrent_pmat leaves them in memory
// in the order the matrix instructions take them (three bf16 parts each), and every wave reads those of
// its own key dims straight into registers, a chunk ahead.  V, P and the factors come through LDS, requested three chunks ahead by
// a wave of their own, which also adds up and stores the waves' partial sums of O^T: a wave's loads return in order, and one that
// comes from memory holds up every one behind it.
//
// Bound by the chain of a chunk in one wave per SIMD: 52 matrix instructions (24 below 192 key dims) = 1800 (1024) of some 3000 (2600)
// cycles, the rest the barrier, LDS latency and vector work that a result of the chunk has to wait for; with 256 blocks of 256 key dims the
// operands, 96 KB per block and chunk from L2, add 15 us of 80.  Whole calls on inputs that change, the split kernel above and this one with
// its launch ahead: B2 H8 L2048 128/128 139 -> 96 us, B1 H8 L2048 256/128 157 -> 120, B4 H4 L1024 64/64 73 -> 48, B2 H8 L1056 256/512 92 -> 89
// (all operands in the caches: 87 -> 83).  Tried and not kept: 32 key dims per wave, eight waves (B2 H8 L1056 256/512 94); the operands brought into L2 by the data wave's touches
// (91 against 79 without); partial sums added and stored by the matrix waves (+8); V read straight into registers (+6).
template <int KD, int WK>
struct RetRecurrentStream {
  static constexpr int kChunk = 32;
  static constexpr int kThreads = WK * 64 + 64;
  static constexpr int kRows = KD / WK;                    // key dims of one wave
  static constexpr int kKB = kRows / 32;                   // its State tiles
  static constexpr int kSteps = 2 * kKB;                   // its k-steps over the key dims; as many (State tile, k-step over the positions)
  static constexpr int kOwn = (4 + WK - 1) / WK;           // row groups of a C tile it adds up (the last may not exist)
  static constexpr int kOpBytes = 2 * (KD / 16) * 3072;    // per (batch, head, chunk)
  static constexpr int kPOff = 4096, kFOff = 8192;
  static constexpr int kStage = kFOff + kRecFactorBytes - kRecFactorW;      // V, P and the factors (all but D) of one chunk
  static constexpr int kStages = 4;
  static constexpr int kSumOff = kStages * kStage;         // two buffers of a partial O^T tile per wave
  static constexpr int kSmemBytes = kSumOff + 2 * WK * 4096;
  static_assert(KD % (32 * WK) == 0 && WK >= 2 && WK <= 4 && kKB <= 2, "one or two State tiles per wave");
};

template <bool FP32, int KD, int WK>
AAT_DEV bool rec_stream_scan(char* smem, const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                             const char* __restrict__ factors, const char* __restrict__ pmat, const char* __restrict__ ops,
                             float* __restrict__ out, int heads, int kdim, int vdim, int L) {
  using T = RetRecurrentStream<KD, WK>;
  using Op = RecOp<FP32>;
  typedef f4v f4v_dword __attribute__((aligned(4)));       // k may start at any float

  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hi = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = xcd_remap(blockIdx.x, gridDim.x), slices = vdim / 32;
  const int bh = tile / slices, vd0 = tile % slices * 32, h = bh % heads;
  const int nchunk = L / T::kChunk;
  const uint32_t lane16 = lane * 16;
  const char* const og = ops + (size_t)bh * nchunk * T::kOpBytes;

  if (wave == WK) {
    const char* const vg = reinterpret_cast<const char*>(v + ((size_t)bh * vdim + vd0) * L);
    const char* const pg = pmat + (size_t)bh * nchunk * 4096;
    const char* const fg = factors + (size_t)h * nchunk * kRecFactorBytes + kRecFactorW;
    const int orl = lane >> 3, occ = lane & 7;
    uint32_t voff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) voff[i] = (uint32_t)((8 * i + rec_pos(orl)) * L * 4 + (occ ^ (((i & 1) << 2) | (orl >> 1))) * 16);
    const auto copy = [&](const char* g_uniform, uint32_t lane_off, char* lds) {
      const uint64_t base = (uint64_t)(uintptr_t)g_uniform;
      const uint32_t dst = (uint32_t)(uintptr_t)(AAT_AS3 char*)lds;
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                   :: "v"(lane_off), "s"(base), "s"(dst) : "memory", "m0");
    };
    const auto request = [&](int c) {
      char* const s = smem + c % T::kStages * T::kStage;
#pragma unroll
      for (int i = 0; i < 4; ++i) copy(vg + (size_t)c * T::kChunk * 4, voff[i], s + i * 1024);
#pragma unroll
      for (int i = 0; i < 4; ++i) copy(pg + (size_t)c * 4096 + i * 1024, lane16, s + T::kPOff + i * 1024);
      copy(fg + (size_t)c * kRecFactorBytes, lane16, s + T::kFOff);
    };
    // Output tile of chunk c: the waves' partial sums, registers of a C tile.
    f4v x[4];
    const auto add_sums = [&](int c) {
      const char* const part = smem + T::kSumOff + (c & 1) * WK * 4096 + lane16;
#pragma unroll
      for (int g = 0; g < 4; ++g) x[g] = *reinterpret_cast<const f4v*>(part + g * 1024);
#pragma unroll
      for (int t = 1; t < WK; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) x[g] += *reinterpret_cast<const f4v*>(part + t * 4096 + g * 1024);
    };
    uint32_t ooff[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) ooff[r] = (uint32_t)((8 * (r >> 2) + 4 * hi + (r & 3)) * L + n) * 4;
    const auto store = [&](int c) {
      const uint64_t base = (uint64_t)(uintptr_t)(out + ((size_t)bh * vdim + vd0) * L + (size_t)c * T::kChunk);
#pragma unroll
      for (int r = 0; r < 16; ++r) asm volatile("global_store_dword %0, %1, %2" :: "v"(ooff[r]), "v"(x[r >> 2][r & 3]), "s"(base) : "memory");
    };
    for (int c = 0; c < 3 && c < nchunk; ++c) request(c);
    if (nchunk > 2) wait_vmcnt<9>();
    else wait_vmcnt<0>();
    block_sync();                                          // chunks 0 and 1 have landed
    for (int c = 0; c < nchunk; ++c) {
      if (c + 3 < nchunk) request(c + 3);
      if (c > 0) {
        add_sums(c - 1);
        store(c - 1);
      }
      // chunk c + 2 has landed: younger than its copies are the stores of two chunks and the copies of chunk c + 3
      if (c > 1 && c + 3 < nchunk) wait_vmcnt<16 + 9 + 16>();
      else wait_vmcnt<0>();
      block_sync();
    }
    add_sums(nchunk - 1);
    store(nchunk - 1);
    wait_vmcnt<0>();
    return false;
  }

  int own[T::kOwn];                                        // this wave's row groups; a missing one repeats its first, with P = V = 0
#pragma unroll
  for (int s = 0; s < T::kOwn; ++s) own[s] = wave + s * WK < 4 ? wave + s * WK : wave;
  const float last = WK != 3 || wave + (T::kOwn - 1) * WK < 4 ? 1.f : 0.f;
  const char* const og_mine = og + wave * T::kSteps * 3072 + lane16;
  const int cp = rec_pos(n);

  const auto read_q = [&](int ks, int c) {
    Op o;
    if constexpr (FP32) {
      const float* const row = q + ((size_t)bh * kdim + wave * T::kRows + 16 * ks + 4 * hi) * L + (size_t)c * 32 + n;
      f4v x[2];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j >> 2][j & 3] = row[(size_t)(8 * (j >> 2) + (j & 3)) * L];
      o = rec_op<FP32>(x[0], x[1]);
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p) o.p[p] = *reinterpret_cast<const u4v*>(og_mine + (size_t)c * T::kOpBytes + ks * 3072 + p * 1024);
    }
    return o;
  };
  const auto read_k = [&](int u, int c) {                  // k-step u%2 over the positions of State tile u/2
    Op o;
    if constexpr (FP32) {
      const float* const row = k + ((size_t)bh * kdim + wave * T::kRows + 32 * (u >> 1) + n) * L + (size_t)c * 32 + 16 * (u & 1) + 4 * hi;
      o = rec_op<FP32>(*reinterpret_cast<const f4v_dword*>(row), *reinterpret_cast<const f4v_dword*>(row + 8));
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p) o.p[p] = *reinterpret_cast<const u4v*>(og_mine + (size_t)c * T::kOpBytes + (KD / 16 + u) * 3072 + p * 1024);
    }
    return o;
  };
  const auto stage_of = [&](int c) { return smem + c % T::kStages * T::kStage; };
  const auto v_at = [&](const char* sm, int g) { return *reinterpret_cast<const f4v*>(sm + cp * 128 + rec_slot(cp, 2 * g + hi) * 16); };
  f16v st[T::kKB], oacc = zero16();                        // State / lambda; T^T Q of the chunk that comes next, 0 for the first
#pragma unroll
  for (int i = 0; i < T::kKB; ++i) st[i] = zero16();
  RecFinite finite;
  Op qop[T::kSteps], kop[T::kSteps], vop[2];               // of the next chunk and of this one
  // in the order of their first uses: what the compiler waits for at the top of the loop is the worse of this order and the loop's
#pragma unroll
  for (int i = 0; i < T::kSteps; ++i) {
    kop[i] = read_k(i, 0);
    sched_fence();
  }
#pragma unroll
  for (int i = 0; i < T::kSteps; ++i) {
    qop[i] = read_q(i, nchunk > 1 ? 1 : 0);
    sched_fence();
  }
  block_sync();                                            // chunks 0 and 1 have landed
  f4v vx[4], wx[4], fx;                                    // V, w / lambda', and rescale flag, scale in the first two
  float pnx;                                               // p_n lambda
  const auto read_v = [&](const char* sm) {
#pragma unroll
    for (int g = 0; g < 4; ++g) vx[g] = v_at(sm, g);
    fx = *reinterpret_cast<const f4v*>(sm + T::kFOff + kRecFactorFlag - kRecFactorW);
    pnx = *reinterpret_cast<const float*>(sm + T::kFOff + kRecFactorPnl - kRecFactorW + n * 4);
  };
  const auto read_w = [&](const char* sm, int s) {
#pragma unroll
    for (int g = 2 * s; g < 2 * s + 2; ++g) wx[g] = *reinterpret_cast<const f4v*>(sm + T::kFOff + hi * 64 + g * 16);
  };
  const auto make_v = [&](int s) {                         // of V w / lambda'
    return rec_op<FP32>(rec_up<FP32>(vx[2 * s]) * wx[2 * s], rec_up<FP32>(vx[2 * s + 1]) * wx[2 * s + 1]);
  };
  read_v(stage_of(0));
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    read_w(stage_of(0), s);
    vop[s] = make_v(s);
  }

  // A step of the loop updates the State with chunk c, finishes chunk c's output and contracts the new State with chunk c+1's Q.
  // Every operand read ahead is used once and then read again for a chunk later in its place; behind the first branch the
  // step is one basic block, or the compiler moves those reads to its end.  Vector work goes between matrix instructions that do
  // not wait for it: the parts of a State tile that is done between those of the next one's update, those of the next chunk's V between the last
  // of T^T Q.
  for (int c = 0; c < nchunk; ++c) {
    const int next = c + 1 < nchunk ? c + 1 : nchunk - 1, next2 = c + 2 < nchunk ? c + 2 : nchunk - 1;
    const char* const sm = stage_of(c);
    const float pnl = pnx;
    if (__builtin_amdgcn_readfirstlane(__float_as_uint(fx[0])) != 0u) {     // lambda left its range: fold it into T
#pragma unroll
      for (int kb = 0; kb < T::kKB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kb][i] *= fx[1];
    }

    // ---- T += K diag(w / lambda') V^T
    f4v vo[T::kOwn], pm[T::kOwn];
#pragma unroll
    for (int t = 0; t < T::kOwn; ++t) {
      vo[t] = v_at(sm, own[t]);
      pm[t] = *reinterpret_cast<const f4v*>(sm + T::kPOff + own[t] * 1024 + lane16);
    }
    Op top[T::kSteps];
    static_for<T::kSteps>([&](auto it) {
      constexpr int u = decltype(it)::value, kb = u >> 1, s = u & 1;
      if constexpr (u == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[r] = FP32 ? oacc[r] * pnl : oacc[r] * pnl * kRecDown;
      }
      if constexpr (u >= 2) {
        top[u - 2] = rec_op_of_c<FP32>(st[0], u - 2);
        rec_pin(top[u - 2]);
      }
      st[kb] = rec_mma<FP32>(kop[u], vop[s], st[kb]);
      rec_interleave<FP32, 0, u == 0 ? 6 : 8>();
      kop[u] = read_k(u, next);
    });

    // ---- O^T = (p_n lambda) T^T Q + V P, over this wave's key dims and positions, and T^T Q of the next chunk
#pragma unroll
    for (int t = 0; t < T::kOwn; ++t) {
      const f4v a = t + 1 < T::kOwn ? vo[t] : vo[t] * last, b = t + 1 < T::kOwn ? pm[t] : pm[t] * last;
#pragma unroll
      for (int e = 0; e < 4; ++e) oacc = mfma_32x32x2_f32(a[e], b[e], oacc);
    }
    read_v(stage_of(next));
    constexpr int kMade = T::kSteps - 2;                   // operands of T made so far
    top[kMade] = rec_op_of_c<FP32>(st[T::kKB - 1], 0);
    rec_pin(top[kMade]);
    sched_fence();
    f16v tq = zero16();
    static_for<T::kSteps>([&](auto it) {
      constexpr int ks = decltype(it)::value;
      if constexpr (ks == 0) {
        top[kMade + 1] = rec_op_of_c<FP32>(st[T::kKB - 1], 1);
        rec_pin(top[kMade + 1]);
      }
      if constexpr (ks == (T::kSteps > 2 ? T::kSteps - 3 : 0)) read_w(stage_of(next), 0);
      if constexpr (ks == T::kSteps - 2) read_w(stage_of(next), 1);
      if constexpr (ks == T::kSteps - 2 && ks > 0) {
        vop[0] = make_v(0);
        rec_pin(vop[0]);
      }
      if constexpr (ks == T::kSteps - 1) {
        if constexpr (T::kSteps == 2) {
          vop[0] = make_v(0);
          rec_pin(vop[0]);
        }
        vop[1] = make_v(1);
        rec_pin(vop[1]);
      }
      tq = rec_mma<FP32>(top[ks], qop[ks], tq);
      rec_interleave<FP32, 0, T::kSteps == 2 && ks == 1 ? 16 : 8>();
      qop[ks] = read_q(ks, next2);
      if constexpr (ks == 0) {
        finite.see(oacc);
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f4v*>(smem + T::kSumOff + (c & 1) * WK * 4096 + wave * 4096 + g * 1024 + lane16) = rec_quarter(oacc, 4 * g);
      }
    });
    oacc = tq;
    block_sync();              // chunk c's partial sums are there; chunk c-1's, which the next step overwrites, have been read
  }
  return finite.broken();
}

// Grid: B * H * vdim / 32 blocks, the slices of one (batch, head) on one XCD (they read the same operands).
template <int KD, int WK>
__global__ __launch_bounds__(WK * 64 + 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void retnet_recurrent_stream_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const char* __restrict__ factors,
    const char* __restrict__ pmat, const char* __restrict__ ops, float* __restrict__ out, int heads, int kdim, int vdim, int L) {
  extern __shared__ __align__(16) char smem[];
  const bool broken = rec_stream_scan<false, KD, WK>(smem, q, k, v, factors, pmat, ops, out, heads, kdim, vdim, L);
  if (rec_any_wave(smem, broken)) rec_stream_scan<true, KD, WK>(smem, q, k, v, factors, pmat, ops, out, heads, kdim, vdim, L);
}

}  // namespace aat
