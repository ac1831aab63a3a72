"""Source text of the per-configuration wrapper for the flash-attention backward.

The reference has no such wrapper (its attention operator's ``backward`` is empty, reference
python/ops/attention_interface.py:37-58); the layout follows its RetNet backward wrapper
(csrc/kernels/retnet/bwd/profile_code.py:1-119).  One library launches two kernels: the row kernel (dQ), which also
leaves delta = rowsum(dO * O) and lse in base-2 units in the workspace, and the column kernel (dV, dK), which reads them;
with ``col_split`` the column kernel runs twice, once per output.  At 128 wide heads a column kernel with 256-row blocks
(bwd_col.h) takes the grids that fill the chip.
"""

global_vars = r"""
#define AAT_OP_ATTN_BWD 1
#include "aat_kernel_abi.h"
#include "kernels/attention/bwd/bwd_chain.h"
#define AAT_COL_WIDE ({Kd} == 128 && {D} == 128 && {Br} == 128 && {col_split} == 0)   // has the column kernel of 256-row blocks
#if AAT_COL_WIDE
#include "kernels/attention/bwd/bwd_col.h"
#endif
#include "kernels/utils/host_launch.h"

namespace {{
constexpr int Br = {Br};                 // block-resident rows of both kernels
constexpr int Bc = {Bc};                 // streamed rows per step of the column kernel
constexpr int BcRow = {row_Bc};          // streamed rows per step of the row kernel
constexpr int Kd = {Kd};
constexpr int D = {D};
constexpr int Nthreads = {Nthreads};
constexpr int num_stages = {num_stages_qk};      // LDS buffers of the streamed tiles
constexpr int waves_per_eu = {waves_per_eu};
constexpr int row_waves_per_eu = {row_waves_per_eu};   // register budget of the row kernel (one output: fits 256 registers)
#define AAT_COL_SPLIT {col_split}                      // 1: one column kernel per output (dV, dK)
constexpr int dv_waves_per_eu = {dv_waves_per_eu};
constexpr int dk_waves_per_eu = {dk_waves_per_eu};

using aat::AttnBwdPass;
using TC = aat::AttnBwdChain<Kd, D, Br, Bc, Nthreads, num_stages, AttnBwdPass::Col>;
using TR = aat::AttnBwdChain<Kd, D, Br, BcRow, Nthreads, num_stages, AttnBwdPass::Row>;
// GEN = 1: lengths the tiles do not divide
#if AAT_COL_SPLIT
template <int GEN> constexpr auto kernel_dv = &aat::attn_bwd_chain<Kd, D, Br, Bc, Nthreads, num_stages, AttnBwdPass::Col, dv_waves_per_eu, 1, GEN>;
template <int GEN> constexpr auto kernel_dk = &aat::attn_bwd_chain<Kd, D, Br, Bc, Nthreads, num_stages, AttnBwdPass::Col, dk_waves_per_eu, 2, GEN>;
#else
template <int GEN> constexpr auto kernel_col = &aat::attn_bwd_chain<Kd, D, Br, Bc, Nthreads, num_stages, AttnBwdPass::Col, waves_per_eu, 3, GEN>;
#endif
template <int GEN> constexpr auto kernel_row = &aat::attn_bwd_chain<Kd, D, Br, BcRow, Nthreads, num_stages, AttnBwdPass::Row, row_waves_per_eu, 3, GEN>;

bool bwd_shape_ok(int B, int H, int Seq_q, int Seq_k) {{ return aat::shape_ok(B, H, Seq_q, Seq_k, 32, 32); }}
bool whole_tiles(int Seq_q, int Seq_k) {{
  // every sequence length plays both roles: resident rows in one kernel, streamed rows in the other
  return Seq_q % Br == 0 && Seq_k % Br == 0 && Seq_q % Bc == 0 && Seq_k % BcRow == 0;
}}
int blocks_of(int rows) {{ return (rows + Br - 1) / Br; }}
#if AAT_COL_WIDE
// Whether 256-row column blocks are the faster ones: one takes 1.6 times as long as one of 128 rows and either fills a compute
// unit, so it is the rounds of blocks over the 256 units that decide.  Measured at 6 lengths from 256 to 8192 and 8 to 512 heads, whole
// backward, 256-row / 128-row blocks: 2 rounds for 4, 3 for 6, 4 for 8 take 0.93 to 0.95 of the time, one for two 0.92 to 0.94, 3
// for 5 1.01, 2 for 3 1.03 to 1.05, one for one 1.21 to 1.33.  The blocks of a causal walk differ in length and the longest ones
// decide as long as there are few: 256 blocks 1.03 to 1.2 (0.93 only at length 256), 384 0.97 to 1.06, 512 and more 0.94 to 0.97.
bool wide_columns(int BH, int Seq_k, int causal) {{
  constexpr long kUnits = 256;
  const long wide = (long)BH * ((Seq_k + aat::AttnBwdCol::BX - 1) / aat::AttnBwdCol::BX), narrow = (long)BH * blocks_of(Seq_k);
  return 5 * ((wide + kUnits - 1) / kUnits) < 3 * ((narrow + kUnits - 1) / kUnits) && (!causal || wide >= 2 * kUnits);
}}
#endif
size_t stats_bytes(int B, int H, int Seq_q) {{ return (size_t)2 * B * H * Seq_q * sizeof(float); }}

template <int GEN> hipError_t launch_kernels(aat_half* q, aat_half* k, aat_half* v, aat_half* o, aat_half* dO, float* lse, aat_half* dq,
                  aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, float softmax_scale, int causal,
                  void* workspace, hipStream_t stream) {{
#if AAT_COL_SPLIT
  static const hipError_t ok0 = aat::allow_lds(kernel_dv<GEN>, TC::kSmemBytes);
  static const hipError_t ok1 = aat::allow_lds(kernel_dk<GEN>, TC::kSmemBytes);
  if (ok0 != hipSuccess) return ok0;
#else
  static const hipError_t ok1 = aat::allow_lds(kernel_col<GEN>, TC::kSmemBytes);
#endif
  static const hipError_t ok2 = aat::allow_lds(kernel_row<GEN>, TR::kSmemBytes);
  if (ok1 != hipSuccess) return ok1;
  if (ok2 != hipSuccess) return ok2;
  using H16 = aat::half_t;
  const H16 *Q = reinterpret_cast<const H16*>(q), *K = reinterpret_cast<const H16*>(k), *V = reinterpret_cast<const H16*>(v),
            *O = reinterpret_cast<const H16*>(o), *G = reinterpret_cast<const H16*>(dO);
  const int rows = B * H * Seq_q;
  float* lse2 = static_cast<float*>(workspace);
  float* delta = lse2 + rows;
  const float c2 = softmax_scale * 1.4426950408889634f;
  kernel_row<GEN><<<dim3(B * H * blocks_of(Seq_q)), dim3(Nthreads), TR::kSmemBytes, stream>>>(
      Q, G, K, V, O, lse, lse2, delta, nullptr, reinterpret_cast<H16*>(dq), H, Seq_k, Seq_q, c2, softmax_scale, causal);
#if AAT_COL_SPLIT
  kernel_dv<GEN><<<dim3(B * H * blocks_of(Seq_k)), dim3(Nthreads), TC::kSmemBytes, stream>>>(
      K, V, Q, G, nullptr, nullptr, lse2, delta, reinterpret_cast<H16*>(dv), nullptr, H, Seq_k, Seq_q, c2, softmax_scale, causal);
  kernel_dk<GEN><<<dim3(B * H * blocks_of(Seq_k)), dim3(Nthreads), TC::kSmemBytes, stream>>>(
      K, V, Q, G, nullptr, nullptr, lse2, delta, nullptr, reinterpret_cast<H16*>(dk), H, Seq_k, Seq_q, c2, softmax_scale, causal);
#else
#if AAT_COL_WIDE
  if (wide_columns(B * H, Seq_k, causal)) {{
    using W = aat::AttnBwdCol;
    static const hipError_t ok3 = aat::allow_lds(aat::attn_bwd_col, W::kSmemBytes);
    if (ok3 != hipSuccess) return ok3;
    aat::attn_bwd_col<<<dim3(B * H * ((Seq_k + W::BX - 1) / W::BX)), dim3(W::Nthreads), W::kSmemBytes, stream>>>(
        K, V, Q, G, lse2, delta, reinterpret_cast<H16*>(dv), reinterpret_cast<H16*>(dk), Seq_k, Seq_q, c2, softmax_scale, causal);
    return hipGetLastError();
  }}
#endif
  kernel_col<GEN><<<dim3(B * H * blocks_of(Seq_k)), dim3(Nthreads), TC::kSmemBytes, stream>>>(
      K, V, Q, G, nullptr, nullptr, lse2, delta, reinterpret_cast<H16*>(dv), reinterpret_cast<H16*>(dk), H, Seq_k, Seq_q, c2, softmax_scale, causal);
#endif
  return hipGetLastError();
}}
hipError_t launch(aat_half* q, aat_half* k, aat_half* v, aat_half* o, aat_half* dO, float* lse, aat_half* dq,
                  aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, float softmax_scale, int causal,
                  void* workspace, hipStream_t stream) {{
  return (whole_tiles(Seq_q, Seq_k) ? launch_kernels<0> : launch_kernels<1>)(q, k, v, o, dO, lse, dq, dk, dv, B, H, Seq_q, Seq_k,
                                                                             softmax_scale, causal, workspace, stream);
}}
}}  // namespace

extern "C" int abi_version(void) {{ return AAT_ABI_VERSION; }}
extern "C" const char* config_string(void) {{ return "{config_name}"; }}
extern "C" size_t workspace_size(int B, int H, int Seq_q, int) {{ return stats_bytes(B, H, Seq_q); }}
extern "C" int column_rows(int B, int H, int Seq_q, int Seq_k, int causal) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return 0;
#if AAT_COL_WIDE
  if (wide_columns(B * H, Seq_k, causal)) return aat::AttnBwdCol::BX;
#endif
  return Br;
}}
"""

profile_func = r"""
extern "C" float profile_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* o, aat_half* dO, float* lse, aat_half* dq,
                            aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, float softmax_scale,
                            int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return -1.f;
  if (workspace == nullptr || workspace_bytes < stats_bytes(B, H, Seq_q)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{
    return launch(q, k, v, o, dO, lse, dq, dk, dv, B, H, Seq_q, Seq_k, softmax_scale, causal, workspace, s);
  }});
}}
"""

kernel_entry = r"""
extern "C" int kernel_entry_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* o, aat_half* dO, float* lse, aat_half* dq,
                               aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, float softmax_scale,
                               int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  if (workspace == nullptr || workspace_bytes < stats_bytes(B, H, Seq_q)) return AAT_ERR_WORKSPACE;
  return (int)launch(q, k, v, o, dO, lse, dq, dk, dv, B, H, Seq_q, Seq_k, softmax_scale, causal, workspace,
                     static_cast<hipStream_t>(stream));
}}
"""

profile_code = global_vars + profile_func + kernel_entry
kernel_code = profile_code
