"""Source text of the per-configuration wrapper for the RetNet backward passes
(same role as reference csrc/kernels/retnet/bwd/profile_code.py:1-119).

One library launches three passes of the chained-contraction kernel (dV, dK, dQ); ``Br`` is the number
of block-resident rows and ``Bc`` the number of streamed rows per step of every pass.  ``dqaccum`` is
accepted for ABI compatibility and never touched: dQ is produced directly, without atomics.

With ``ds_rows`` set the dQ pass runs before dK and stores its dS tiles in the workspace (behind the mask scan's
ranges), and dK comes from the kernel that reads them back (dk_from_ds.h); ``workspace_size`` says how much room that
takes, and without it the library runs the chained dK pass.
"""

global_vars = r"""
#define AAT_OP_RET_BWD 1
#include "aat_kernel_abi.h"
#include "kernels/retnet/bwd/bwd_chain.h"
#include "kernels/retnet/bwd/dk_from_ds.h"
#include "kernels/utils/host_launch.h"

namespace {{
constexpr int Br = {Br};                 // block-resident rows of every pass
constexpr int Bc = {Bc};                 // streamed rows per step of every pass
constexpr int Kd = {Kd};
constexpr int D = {D};
constexpr int Nthreads = {Nthreads};
constexpr int num_stages_qk = {num_stages_qk};   // LDS buffers of the first-contraction stream (+ mask)
constexpr int num_stages_dv = {num_stages_dv};   // LDS buffers of the second-contraction stream
// the same two counts for the passes that contract over d_v first (dQ, and dK when it is a chained pass): their streamed
// tiles are d_v wide, twice the dV pass's at d_v = 2 d_qk, so they often cannot afford what the dV pass can
constexpr int num_stages_ds = {num_stages_ds};
constexpr int num_stages_dq = {num_stages_dq};
constexpr int waves_per_eu = {waves_per_eu};
constexpr int ds_rows = {ds_rows};               // 0, or kv rows per block of the dK kernel that reads a stored dS
constexpr bool kStoredDs = ds_rows != 0;
// The dK kernel has four waves for 128 kv rows and two stages, eight and three where a second such block would not fit into LDS.
constexpr int kDkRows = kStoredDs ? ds_rows : 128, kDkTile = 64, kDkWaves = 2;
constexpr bool kDkAlone = kDkRows == 128 && 4 * kDkTile * (Kd + kDkRows) * 2 > 160 * 1024;
constexpr int kDkThreads = kDkAlone ? 512 : kDkRows * 2, kDkStages = kDkAlone ? 3 : 2;
// dV columns per block: the whole row when the accumulators fit the 256 accumulation registers that one
// wave per SIMD has to itself, else 256-column slices over grid.y (each repeats the first contraction).
constexpr int RTv = Br / (Nthreads / 64) / 32;
constexpr int DVB = (waves_per_eu == 1 && RTv * D <= 512) ? D : (D > 256 ? 256 : D);
constexpr int DKB = Kd;

using aat::BwdPass;
using TV = aat::RetBwdChain<Kd, D, DVB, Br, Bc, Nthreads, num_stages_qk, num_stages_dv, BwdPass::Col>;
using TK = aat::RetBwdChain<D, Kd, DKB, Br, Bc, Nthreads, num_stages_ds, num_stages_dq, BwdPass::Col>;
using TQ = aat::RetBwdChain<D, Kd, DKB, Br, Bc, Nthreads, num_stages_ds, num_stages_dq, BwdPass::Row>;
// GEN = 1: resident lengths the blocks do not divide
template <bool DECAY, int GEN> constexpr auto kernel_dv = &aat::ret_bwd_chain<Kd, D, DVB, Br, Bc, Nthreads, num_stages_qk, num_stages_dv, BwdPass::Col, waves_per_eu, GEN, DECAY, false>;
template <bool DECAY, int GEN> constexpr auto kernel_dk = &aat::ret_bwd_chain<D, Kd, DKB, Br, Bc, Nthreads, num_stages_ds, num_stages_dq, BwdPass::Col, waves_per_eu, GEN, DECAY, false>;
template <bool DECAY, int GEN> constexpr auto kernel_dq = &aat::ret_bwd_chain<D, Kd, DKB, Br, Bc, Nthreads, num_stages_ds, num_stages_dq, BwdPass::Row, waves_per_eu, GEN, DECAY, false>;
// stored dS: the row pass that writes it (the plain one again in a library without it), the dK kernel that reads it
using TKD = aat::RetBwdDk<Kd, kDkRows, kDkTile, kDkThreads, kDkStages>;
template <bool DECAY, int GEN> constexpr auto kernel_dq_ds = &aat::ret_bwd_chain<D, Kd, DKB, Br, Bc, Nthreads, num_stages_ds, num_stages_dq, BwdPass::Row, waves_per_eu, GEN, DECAY, kStoredDs>;
template <int GEN> constexpr auto kernel_dk_ds = &aat::ret_bwd_dk_from_ds<Kd, kDkRows, kDkTile, kDkThreads, kDkStages, kDkWaves, GEN>;
static_assert(!kStoredDs || Br % kDkTile == 0, "a query tile of the dK kernel lies inside one block of the row pass");

// The longest blocks of a decay walk in parts (utils/block_parts.h), where the call has room for their slots behind its other
// workspace.  The launches of a call follow each other and share the slots; each has counts of its own.
constexpr bool kPartsFit = aat::parts_fit(RTv, Bc, waves_per_eu, 0);
using PV = aat::PartsLaunch<kPartsFit, Br, Bc, Kd + D, DVB, Nthreads, 0, false, DVB == 512>;
using PQ = aat::PartsLaunch<kPartsFit, Br, Bc, Kd + D, DKB, Nthreads, 0, true, DKB == 512>;
using PK = aat::PartsLaunch<kPartsFit, Br, Bc, Kd + D, DKB, Nthreads, 0, false, DKB == 512>;
using PKD = aat::PartsLaunch<true, kDkRows, kDkTile, Kd, Kd, kDkThreads, 0, false, false, 109, kDkRows / 32>;    // it streams dS as well
struct BwdPlan {{
  aat::PartsPlan dv, dq, dk;
  size_t counts, slots;
  size_t bytes() const {{ return slots ? counts + 3 * aat::kOrderBytes + slots : 0; }}
}};
BwdPlan plan_of(int B, int H, int Seq_q, int Seq_k, bool stored) {{
  const long heads = (long)B * H;
  constexpr int waves = Nthreads / 64;
  const int row_lds = stored ? TQ::kSmemBytesDsOut : TQ::kSmemBytes;
  BwdPlan p{{}};
  if (D == DVB) p.dv = PV::find(heads, Seq_q, Seq_k, aat::blocks_per_cu(waves, waves_per_eu, TV::kSmemBytes));
  p.dq = PQ::find(heads, Seq_q, Seq_k, aat::blocks_per_cu(waves, waves_per_eu, row_lds));
  p.dk = stored ? PKD::find(heads, Seq_q, Seq_k, aat::blocks_per_cu(kDkThreads / 64, kDkWaves, TKD::kSmemBytes))
                : PK::find(heads, Seq_q, Seq_k, aat::blocks_per_cu(waves, waves_per_eu, TK::kSmemBytes));
  if (p.dv.gain_us + p.dq.gain_us + p.dk.gain_us < aat::kPrepareUs) return BwdPlan{{}};
  const size_t dk = stored ? PKD::slot_bytes(heads, p.dk) : PK::slot_bytes(heads, p.dk);
  const size_t dv = PV::slot_bytes(heads, p.dv), dq = PQ::slot_bytes(heads, p.dq);
  p.slots = dv > dq ? (dv > dk ? dv : dk) : (dq > dk ? dq : dk);
  p.counts = aat::count_bytes(heads, p.dv) + aat::count_bytes(heads, p.dq) + aat::count_bytes(heads, p.dk);
  return p;
}}

bool bwd_shape_ok(int B, int H, int Seq_q, int Seq_k) {{
  // every sequence length plays both roles: resident rows (any multiple of 32) in one pass, streamed rows in another
  return aat::shape_ok(B, H, Seq_q, Seq_k, 32, 32) && aat::shape_ok(B, H, Seq_q, Seq_k, Bc, Bc);
}}
int blocks_of(int rows) {{ return (rows + Br - 1) / Br; }}
// Whether this library stores dS for the problem: it is built for it and the lengths are whole dS blocks.  Where the kv
// length is not a multiple of the dK kernel's rows, short walks do not earn the round trip.
bool stores_ds(int B, int H, int Seq_q, int Seq_k) {{
  return kStoredDs && aat::shape_ok(B, H, Seq_q, Seq_k, kDkTile, 64) && (Seq_k % kDkRows == 0 || Seq_k >= 512);
}}

// Workspace: the mask scan's ranges (as the forward lays them out), then, with a stored dS, B*H*Seq_q*Seq_k fp16.
size_t ds_offset(int H, int Seq_q, int Seq_k) {{ return aat::mask_extent_bytes(H, Seq_q, Seq_k); }}
size_t ws_bytes_needed(int B, int H, int Seq_q, int Seq_k) {{
  const size_t scan = aat::mask_extent_bytes(H, Seq_q, Seq_k);
  return stores_ds(B, H, Seq_q, Seq_k) ? scan + (size_t)B * H * Seq_q * Seq_k * sizeof(aat::half_t) : scan;
}}
// The scanning modes need the ranges.  dS is stored when the workspace has its room too; without it (the
// reference-signature entry points have no workspace to give) dK comes from the chained pass that evaluates dS again.
bool workspace_ok(int mode, const void* workspace, size_t workspace_bytes, int H, int Seq_q, int Seq_k) {{
  return aat::mask_mode_ok(mode, workspace, workspace_bytes, H, Seq_q, Seq_k);
}}
bool room_for_ds(const void* workspace, size_t workspace_bytes, int B, int H, int Seq_q, int Seq_k) {{
  return stores_ds(B, H, Seq_q, Seq_k) && workspace != nullptr && workspace_bytes >= ws_bytes_needed(B, H, Seq_q, Seq_k);
}}

// DECAY: the mask is gamma_h^(q + Seq_k - Seq_q - kv) below the diagonal, zero above it, and `mask` and `walk` are not looked at.
template <bool DECAY> hipError_t launch_passes(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, const float* log2_gamma, aat_half* dO,
                                               float* r, aat_half* dq, aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k,
                                               aat::MaskWalk walk, void* workspace, size_t workspace_bytes, hipStream_t stream) {{
  static const hipError_t allowed[] = {{
      aat::allow_lds(kernel_dv<DECAY, 0>, TV::kSmemBytes), aat::allow_lds(kernel_dv<DECAY, 1>, TV::kSmemBytes),
      aat::allow_lds(kernel_dk<DECAY, 0>, TK::kSmemBytes), aat::allow_lds(kernel_dk<DECAY, 1>, TK::kSmemBytes),
      aat::allow_lds(kernel_dq<DECAY, 0>, TQ::kSmemBytes), aat::allow_lds(kernel_dq<DECAY, 1>, TQ::kSmemBytes),
      kStoredDs ? aat::allow_lds(kernel_dk_ds<0>, TKD::kSmemBytes) : hipSuccess,
      kStoredDs ? aat::allow_lds(kernel_dk_ds<1>, TKD::kSmemBytes) : hipSuccess,
      kStoredDs ? aat::allow_lds(kernel_dq_ds<DECAY, 0>, TQ::kSmemBytesDsOut) : hipSuccess,
      kStoredDs ? aat::allow_lds(kernel_dq_ds<DECAY, 1>, TQ::kSmemBytesDsOut) : hipSuccess}};
  for (hipError_t e : allowed)
    if (e != hipSuccess) return e;
  using H16 = aat::half_t;
  const H16 *Q = reinterpret_cast<const H16*>(q), *K = reinterpret_cast<const H16*>(k), *V = reinterpret_cast<const H16*>(v),
            *M = reinterpret_cast<const H16*>(mask), *G = reinterpret_cast<const H16*>(dO);
  H16 *DQ = reinterpret_cast<H16*>(dq), *DK = reinterpret_cast<H16*>(dk), *DV = reinterpret_cast<H16*>(dv);
  const int causal = DECAY ? 1 : walk.causal;
  const int* extents = DECAY ? nullptr : walk.extents;
  const bool whole_q = Seq_q % Br == 0, whole_k = Seq_k % Br == 0;
  const bool stored = room_for_ds(workspace, workspace_bytes, B, H, Seq_q, Seq_k);
  aat::BlockParts dv_parts, dq_parts, dk_parts;
  if constexpr (DECAY) {{
    const size_t at = stored ? ws_bytes_needed(B, H, Seq_q, Seq_k) : ds_offset(H, Seq_q, Seq_k);
    BwdPlan plan{{}};
    if (aat::parts_room(workspace, workspace_bytes, at)) plan = plan_of(B, H, Seq_q, Seq_k, stored);
    if (plan.slots > 0 && workspace_bytes >= at + plan.bytes()) {{
      char* const room = static_cast<char*>(workspace) + at;
      uint16_t* const order = reinterpret_cast<uint16_t*>(room + plan.counts);
      float* const slots = reinterpret_cast<float*>(room + plan.counts + 3 * aat::kOrderBytes);
      const int n = (int)(plan.counts / sizeof(uint32_t));
      aat::JobOrders<3> orders{{}};
      PV::put_order(plan.dv, Seq_q, Seq_k, orders.of[0]);
      PQ::put_order(plan.dq, Seq_q, Seq_k, orders.of[1]);
      if (stored) PKD::put_order(plan.dk, Seq_q, Seq_k, orders.of[2]);
      else PK::put_order(plan.dk, Seq_q, Seq_k, orders.of[2]);
      aat::prepare_parts<3><<<dim3((n + aat::kMostJobs - 1) / aat::kMostJobs), dim3(aat::kMostJobs), 0, stream>>>(
          reinterpret_cast<uint32_t*>(room), n, orders, order);
      size_t counted = 0;
      const auto take = [&](const aat::PartsPlan& p, int launch) {{
        const aat::BlockParts b{{p.split, p.parts, slots, reinterpret_cast<uint32_t*>(room + counted), order + launch * aat::kMostJobs}};
        counted += aat::count_bytes((long)B * H, p);
        return b;
      }};
      dv_parts = take(plan.dv, 0);
      dq_parts = take(plan.dq, 1);
      dk_parts = take(plan.dk, 2);
    }}
  }}
  const auto grid = [&](int blocks, const aat::BlockParts& p) {{ return (unsigned)(B * H * (blocks + p.split * (p.parts - 1))); }};
  (whole_k ? kernel_dv<DECAY, 0> : kernel_dv<DECAY, 1>)<<<dim3(grid(blocks_of(Seq_k), dv_parts), D / DVB), dim3(Nthreads), TV::kSmemBytes, stream>>>(
      K, Q, G, M, r, DV, H, Seq_k, Seq_q, causal, log2_gamma, extents, nullptr, dv_parts);
  if (stored) {{
    H16* ds = reinterpret_cast<H16*>(static_cast<char*>(workspace) + ds_offset(H, Seq_q, Seq_k));
    (whole_q ? kernel_dq_ds<DECAY, 0> : kernel_dq_ds<DECAY, 1>)<<<dim3(grid(blocks_of(Seq_q), dq_parts), Kd / DKB), dim3(Nthreads), TQ::kSmemBytesDsOut, stream>>>(
        G, V, K, M, r, DQ, H, Seq_k, Seq_q, causal, log2_gamma, extents, ds, dq_parts);
    (whole_q && Seq_k % kDkRows == 0 ? kernel_dk_ds<0> : kernel_dk_ds<1>)<<<dim3(grid((Seq_k + kDkRows - 1) / kDkRows, dk_parts)), dim3(kDkThreads), TKD::kSmemBytes, stream>>>(
        Q, ds, DK, H, Seq_k, Seq_q, causal, extents, Br, Bc, dk_parts);
  }} else {{
    (whole_k ? kernel_dk<DECAY, 0> : kernel_dk<DECAY, 1>)<<<dim3(grid(blocks_of(Seq_k), dk_parts), Kd / DKB), dim3(Nthreads), TK::kSmemBytes, stream>>>(
        V, G, Q, M, r, DK, H, Seq_k, Seq_q, causal, log2_gamma, extents, nullptr, dk_parts);
    (whole_q ? kernel_dq<DECAY, 0> : kernel_dq<DECAY, 1>)<<<dim3(grid(blocks_of(Seq_q), dq_parts), Kd / DKB), dim3(Nthreads), TQ::kSmemBytes, stream>>>(
        G, V, K, M, r, DQ, H, Seq_k, Seq_q, causal, log2_gamma, extents, nullptr, dq_parts);
  }}
  return hipGetLastError();
}}
hipError_t launch(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* dO, float* r, aat_half* dq,
                  aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, int mask_mode, void* workspace,
                  size_t workspace_bytes, hipStream_t stream) {{
  aat::MaskWalk walk;
  const hipError_t scanned = aat::prepare_mask_walk(mask_mode, reinterpret_cast<const aat::half_t*>(mask), H, Seq_q, Seq_k,
                                                    workspace, stream, &walk);
  if (scanned != hipSuccess) return scanned;
  return launch_passes<false>(q, k, v, mask, nullptr, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, walk, workspace, workspace_bytes, stream);
}}
hipError_t launch_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* dO, float* r,
                        aat_half* dq, aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, void* workspace,
                        size_t workspace_bytes, hipStream_t stream) {{
  aat::touch_thread_storage();
  return launch_passes<true>(q, k, v, nullptr, log2_gamma, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, aat::MaskWalk(), workspace, workspace_bytes, stream);
}}
}}  // namespace

extern "C" int abi_version(void) {{ return AAT_ABI_VERSION; }}
extern "C" const char* config_string(void) {{ return "{config_name}"; }}
// The ranges of the scanning mask modes (AAT_MASK_SCAN / AAT_MASK_SCANNED; the same layout as the forward's, so a scan
// the forward made can be handed over or copied to the head of a larger buffer) and, with a stored dS, its room (a
// smaller workspace is accepted: dK then comes from the chained pass).
extern "C" size_t workspace_size(int B, int H, int Seq_q, int Seq_k) {{
  return B > 0 && H > 0 && Seq_q > 0 && Seq_k > 0 ? ws_bytes_needed(B, H, Seq_q, Seq_k) : 0;
}}

static_assert(AAT_MASK_DENSE == aat::kMaskDense && AAT_MASK_CAUSAL == aat::kMaskCausal && AAT_MASK_SCAN == aat::kMaskScan &&
              AAT_MASK_SCANNED == aat::kMaskScanned, "mask modes of the header and of the kernels");
"""

profile_func = r"""
extern "C" float profile_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* dO, float* r, aat_half* dq,
                            aat_half* dk, aat_half* dv, float*, int B, int H, int Seq_q, int Seq_k, int causal,
                            void* workspace, size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return -1.f;
  if (!workspace_ok(causal, workspace, workspace_bytes, H, Seq_q, Seq_k)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{ return launch(q, k, v, mask, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, causal, workspace, workspace_bytes, s); }});
}}
extern "C" float profile(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* dO, float* r, aat_half* dq,
                         aat_half* dk, aat_half* dv, float* dqaccum, int B, int H, int Seq_q, int Seq_k) {{
  return profile_ex(q, k, v, mask, dO, r, dq, dk, dv, dqaccum, B, H, Seq_q, Seq_k, 0, nullptr, 0, nullptr);
}}
"""

kernel_entry = r"""
extern "C" int kernel_entry_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* dO, float* r,
                               aat_half* dq, aat_half* dk, aat_half* dv, float*, int B, int H, int Seq_q, int Seq_k,
                               int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k) || causal < 0 || causal > AAT_MASK_SCANNED) return AAT_ERR_SHAPE;
  if (!workspace_ok(causal, workspace, workspace_bytes, H, Seq_q, Seq_k)) return AAT_ERR_WORKSPACE;
  return (int)launch(q, k, v, mask, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, causal, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}}
extern "C" int kernel_entry(aat_half* q, aat_half* k, aat_half* v, aat_half* mask, aat_half* dO, float* r, aat_half* dq,
                            aat_half* dk, aat_half* dv, float* dqaccum, int B, int H, int Seq_k, int Seq_q) {{
  return kernel_entry_ex(q, k, v, mask, dO, r, dq, dk, dv, dqaccum, B, H, Seq_q, Seq_k, 0, nullptr, 0, nullptr);
}}
"""

decay_entry = r"""
extern "C" size_t decay_workspace_size(int B, int H, int Seq_q, int Seq_k, size_t most) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return workspace_size(B, H, Seq_q, Seq_k);
  const size_t scan = ds_offset(H, Seq_q, Seq_k), ds = ws_bytes_needed(B, H, Seq_q, Seq_k) - scan;
  const bool stored = ds > 0 && ds <= most;
  const size_t at = stored ? scan + ds : scan, room = plan_of(B, H, Seq_q, Seq_k, stored).bytes();
  return room <= most ? at + room : at;
}}
extern "C" float profile_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* dO, float* r,
                               aat_half* dq, aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k, void* workspace,
                               size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return -1.f;
  if (!workspace_ok(AAT_MASK_CAUSAL, workspace, workspace_bytes, H, Seq_q, Seq_k)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{ return launch_decay(q, k, v, log2_gamma, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, workspace, workspace_bytes, s); }});
}}
extern "C" int kernel_entry_decay(aat_half* q, aat_half* k, aat_half* v, const float* log2_gamma, aat_half* dO, float* r,
                                  aat_half* dq, aat_half* dk, aat_half* dv, int B, int H, int Seq_q, int Seq_k,
                                  void* workspace, size_t workspace_bytes, void* stream) {{
  if (!bwd_shape_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  if (!workspace_ok(AAT_MASK_CAUSAL, workspace, workspace_bytes, H, Seq_q, Seq_k)) return AAT_ERR_WORKSPACE;
  return (int)launch_decay(q, k, v, log2_gamma, dO, r, dq, dk, dv, B, H, Seq_q, Seq_k, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}}
"""

profile_code = global_vars + profile_func + kernel_entry + decay_entry
kernel_code = profile_code
