"""Source text of the per-configuration wrapper for the register-fused RetNet forward kernel
(same role as reference csrc/kernels/retnet/regfuse/profile_code.py:1-83)."""

global_vars = r"""
#define AAT_OP_RET 1
#include "aat_kernel_abi.h"
#include "kernels/retnet/regfuse/regfuse.h"
#include "kernels/utils/host_launch.h"

namespace {{
constexpr int Br = {Br};
constexpr int Bc = {Bc};
constexpr int Kd = {Kd};
constexpr int D = {D};
constexpr int Nthreads = {Nthreads};
constexpr int num_stages_qk = {num_stages_qk};     // LDS buffers for the K tile
constexpr int num_stages_mask = {num_stages_mask}; // LDS buffers for the mask tile (fetched with K)
constexpr int num_stages_v = {num_stages_v};       // LDS buffers for the V tile
constexpr int waves_per_eu = {waves_per_eu};
constexpr int stages_mask = num_stages_mask < num_stages_qk ? num_stages_qk : num_stages_mask;

using Traits = aat::RetFwdRegfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, stages_mask>;
constexpr int shared_mem = Traits::kSmemBytes;
template <bool DECAY> constexpr auto kernel = &aat::ret_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, stages_mask, waves_per_eu, DECAY>;
// a query length the row blocks do not divide
template <bool DECAY> constexpr auto kernel_ragged = &aat::ret_ragged_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, stages_mask, waves_per_eu, DECAY>;

// The longest blocks of a decay walk in parts (utils/block_parts.h), where the call has room for their slots behind workspace_size().
using Parts = aat::PartsLaunch<aat::parts_fit(Traits::RT, Bc, waves_per_eu, Kd + D), Br, Bc, Kd + D, D, Nthreads, Traits::RT, true, waves_per_eu == 1>;
constexpr int kBlocksPerCu = aat::blocks_per_cu(Nthreads / 64, waves_per_eu, shared_mem);

aat::PartsPlan plan_of(int B, int H, int Seq_q, int Seq_k) {{
  const aat::PartsPlan p = Parts::find((long)B * H, Seq_q, Seq_k, kBlocksPerCu);
  return p.gain_us >= aat::kPrepareUs ? p : aat::PartsPlan();
}}
// ... their counts, their order and their slots
size_t parts_bytes(int B, int H, const aat::PartsPlan& p) {{
  return p.split ? aat::count_bytes((long)B * H, p) + aat::kOrderBytes + Parts::slot_bytes((long)B * H, p) : 0;
}}

bool lengths_ok(int B, int H, int Seq_q, int Seq_k) {{ return aat::shape_ok(B, H, Seq_q, Seq_k, 32, Bc); }}
int row_blocks(int Seq_q) {{ return (Seq_q + Br - 1) / Br; }}
template <bool DECAY> hipError_t allow_kernels() {{
  const hipError_t e = aat::allow_lds(kernel<DECAY>, shared_mem);
  return e != hipSuccess ? e : aat::allow_lds(kernel_ragged<DECAY>, shared_mem);
}}

hipError_t launch(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* o, float* r, int B, int H,
                  int Seq_q, int Seq_k, int mask_mode, void* workspace, hipStream_t stream) {{
  static const hipError_t lds_ok = allow_kernels<false>();
  if (lds_ok != hipSuccess) return lds_ok;
  aat::MaskWalk walk;
  const hipError_t scanned = aat::prepare_mask_walk(mask_mode, reinterpret_cast<const aat::half_t*>(mask), H, Seq_q, Seq_k,
                                                    workspace, stream, &walk);
  if (scanned != hipSuccess) return scanned;
  (Seq_q % Br == 0 ? kernel<false> : kernel_ragged<false>)<<<dim3(B * H * row_blocks(Seq_q)), dim3(Nthreads), shared_mem, stream>>>(
      reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
      reinterpret_cast<const aat::half_t*>(v), reinterpret_cast<const aat::half_t*>(mask),
      reinterpret_cast<aat::half_t*>(o), r, H, Seq_k, Seq_q, walk.causal, nullptr, walk.extents, aat::BlockParts());
  return hipGetLastError();
}}
// Decay-mask variant: the mask is gamma_h^(q + Seq_k - Seq_q - kv) below the diagonal, zero above it.
hipError_t launch_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* o, float* r, int B,
                        int H, int Seq_q, int Seq_k, void* workspace, size_t workspace_bytes, hipStream_t stream) {{
  aat::touch_thread_storage();
  static const hipError_t lds_ok = allow_kernels<true>();
  if (lds_ok != hipSuccess) return lds_ok;
  const size_t at = workspace_size(B, H, Seq_q, Seq_k);
  aat::BlockParts in_parts;
  if (aat::parts_room(workspace, workspace_bytes, at)) {{
    const aat::PartsPlan plan = plan_of(B, H, Seq_q, Seq_k);
    const size_t counts = aat::count_bytes((long)B * H, plan);
    if (plan.split > 0 && workspace_bytes >= at + parts_bytes(B, H, plan)) {{
      char* const room = static_cast<char*>(workspace) + at;
      uint32_t* const arrived = reinterpret_cast<uint32_t*>(room);
      uint16_t* const order = reinterpret_cast<uint16_t*>(room + counts);
      const int n = B * H * plan.split;
      aat::JobOrders<1> orders{{}};
      Parts::put_order(plan, Seq_q, Seq_k, orders.of[0]);
      aat::prepare_parts<1><<<dim3((n + aat::kMostJobs - 1) / aat::kMostJobs), dim3(aat::kMostJobs), 0, stream>>>(
          arrived, n, orders, order);
      in_parts = {{plan.split, plan.parts, reinterpret_cast<float*>(room + counts + aat::kOrderBytes), arrived, order}};
    }}
  }}
  const int jobs = row_blocks(Seq_q) + in_parts.split * (in_parts.parts - 1);
  (Seq_q % Br == 0 ? kernel<true> : kernel_ragged<true>)<<<dim3(B * H * jobs), dim3(Nthreads), shared_mem, stream>>>(
      reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
      reinterpret_cast<const aat::half_t*>(v), nullptr, reinterpret_cast<aat::half_t*>(o), r, H, Seq_k, Seq_q, 1,
      log2_gamma, nullptr, in_parts);
  return hipGetLastError();
}}
}}  // namespace

extern "C" int abi_version(void) {{ return AAT_ABI_VERSION; }}
extern "C" const char* config_string(void) {{ return "{config_name}"; }}
// Needed for the scanning mask modes only (AAT_MASK_SCAN / AAT_MASK_SCANNED).
extern "C" size_t workspace_size(int, int H, int Seq_q, int Seq_k) {{
  return H > 0 && Seq_q > 0 && Seq_k > 0 ? aat::mask_extent_bytes(H, Seq_q, Seq_k) : 0;
}}
static_assert(AAT_MASK_DENSE == aat::kMaskDense && AAT_MASK_CAUSAL == aat::kMaskCausal && AAT_MASK_SCAN == aat::kMaskScan &&
              AAT_MASK_SCANNED == aat::kMaskScanned, "mask modes of the header and of the kernels");
"""

profile_func = r"""
extern "C" float profile_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* o, float* r, int B, int H,
                            int Seq_q, int Seq_k, int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return -1.f;
  if (!aat::mask_mode_ok(causal, workspace, workspace_bytes, H, Seq_q, Seq_k)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{ return launch(q, k, v, mask, o, r, B, H, Seq_q, Seq_k, causal, workspace, s); }});
}}
extern "C" float profile(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* o, float* r, int B, int H,
                         int Seq_q, int Seq_k) {{
  return profile_ex(q, k, v, mask, o, r, B, H, Seq_q, Seq_k, 0, nullptr, 0, nullptr);
}}
"""

kernel_entry = r"""
extern "C" int kernel_entry_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* o, float* r, int B, int H,
                               int Seq_q, int Seq_k, int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k) || causal < 0 || causal > AAT_MASK_SCANNED) return AAT_ERR_SHAPE;
  if (!aat::mask_mode_ok(causal, workspace, workspace_bytes, H, Seq_q, Seq_k)) return AAT_ERR_WORKSPACE;
  return (int)launch(q, k, v, mask, o, r, B, H, Seq_q, Seq_k, causal, workspace, static_cast<hipStream_t>(stream));
}}
extern "C" int kernel_entry(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* o, float* r, int B, int H,
                            int Seq_k, int Seq_q) {{
  return kernel_entry_ex(q, k, v, mask, o, r, B, H, Seq_q, Seq_k, 0, nullptr, 0, nullptr);
}}
"""

decay_entry = r"""
extern "C" size_t decay_workspace_size(int B, int H, int Seq_q, int Seq_k, size_t most) {{
  const size_t at = workspace_size(B, H, Seq_q, Seq_k);
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return at;
  const size_t room = parts_bytes(B, H, plan_of(B, H, Seq_q, Seq_k));
  return room <= most ? at + room : at;
}}
extern "C" float profile_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* o, float* r,
                               int B, int H, int Seq_q, int Seq_k, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{ return launch_decay(q, k, v, log2_gamma, o, r, B, H, Seq_q, Seq_k, workspace, workspace_bytes, s); }});
}}
extern "C" int kernel_entry_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* o, float* r,
                                  int B, int H, int Seq_q, int Seq_k, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  return (int)launch_decay(q, k, v, log2_gamma, o, r, B, H, Seq_q, Seq_k, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}}
"""

profile_code = global_vars + profile_func + kernel_entry + decay_entry
kernel_code = profile_code
