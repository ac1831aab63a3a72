"""Source text of the per-configuration wrapper for the register-fused attention forward kernel.

``str.format_map(config.__dict__)`` fills the ``{Br}``-style fields; the result is one ``.hip`` file
that instantiates the kernel template for that configuration and exports the C ABI declared in
include/aat_kernel_abi.h.  Same role as reference csrc/kernels/attention/regfuse/profile_code.py:1-79.
"""

global_vars = r"""
#define AAT_OP_ATTN 1
#include <atomic>
#include "aat_kernel_abi.h"
#include "kernels/attention/regfuse/kv_parts.h"
#include "kernels/attention/regfuse/regfuse.h"
#include "kernels/utils/host_launch.h"

namespace {{
constexpr int Br = {Br};
constexpr int Bc = {Bc};
constexpr int Kd = {Kd};
constexpr int D = {D};
constexpr int Nthreads = {Nthreads};
constexpr int num_stages_qk = {num_stages_qk};   // LDS buffers for the K tile
constexpr int num_stages_v = {num_stages_v};     // LDS buffers for the V tile
constexpr int waves_per_eu = {waves_per_eu};
constexpr int kv_splits = {kv_splits};           // > 1: a non-causal problem's kv range is cut into that many parts, a causal one's not; 1: as many as pay (kv_parts.h)
constexpr bool sw_pipeline = {sw_pipeline};      // next tile's QK^T MFMAs interleaved with this tile's exponentials
constexpr int unit_rows = sw_pipeline ? Bc : {BlockKSmem2};   // plain schedule: kv rows per scores -> softmax -> PV unit inside a tile of Bc rows
constexpr float kReferenceScale = 0.125f;        // what the reference kernels hard-code

#define AAT_KV_GROUPS {kv_groups}                // > 1: that many waves share their query rows; such a library has one kernel, for any lengths
using Traits = aat::AttnFwdRegfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, AAT_KV_GROUPS>;
constexpr int shared_mem = Traits::kSmemBytes;
#if AAT_KV_GROUPS > 1
const auto kernel_gen = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 1, AAT_KV_GROUPS, false, true>;
#else
const auto kernel = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 0, 1, sw_pipeline, false>;
const auto kernel_causal = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 0, 1, sw_pipeline, true>;
const auto kernel_causal_paired = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 0, 1, sw_pipeline, true, false, false, true>;
// any lengths that are multiples of 32, causal or not; and the same with the kv range cut into parts
const auto kernel_gen = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 1, 1, false, true>;
const auto kernel_split = &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 1, 1, false, true, true>;
constexpr int shared_mem_split = Traits::kSmemBytesSplit;

// Persistent variant (a block walks several row blocks, prefetching across them): exists for two K and two V
// buffers, the plain schedule and a tile shape that leaves room to stage the output beside the prefetched
// tiles; used for non-causal problems with an even number of kv tiles and more row blocks than the chip holds
// at once -- and with fewer than 2048 kv rows.  Measured with the Br=256 Bc=128 512-thread
// configuration under sustained load (300 launches back to back): +10 % at S=512 (B 16, H 32), +3 % at S=1024,
// +-0 at S=2048, -1.5 % at S=4096: what it removes is the 5.7 us a block spends per row block on start-up and
// drain, and on long rows the kernel runs at the chip's power limit, where idle time is not what bounds it.
constexpr int kPersistMaxKv = 1792;
using PersistTraits = Traits::Persist<waves_per_eu>;
constexpr int shared_mem_persist = PersistTraits::kSmemBytes;
template <bool OK> auto persistent_kernel() {{
  if constexpr (OK)
    return &aat::flashattn_fwd_regfuse<Kd, D, Br, Bc, Nthreads, num_stages_qk, num_stages_v, waves_per_eu, unit_rows, 0, 1, false, false, false, true>;
  else
    return static_cast<decltype(kernel)>(nullptr);
}}
const auto kernel_persist = persistent_kernel<PersistTraits::kOk && !sw_pipeline>();

// Blocks of the persistent kernel the current device holds at once (0: unknown, do not use it).
int resident_blocks() {{
  static std::atomic<int> cached[64];            // per device; threads that race here compute the same value
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  int blocks = cached[dev].load(std::memory_order_relaxed);
  if (blocks == 0) {{
    int per_cu = 0, cus = 0;
    // The persistent kernel requests the next row block's Q fragments into live registers behind the compiler's back
    // and waits for them a tile later.  That is sound only while those registers stay registers: a build whose
    // allocator spilled anything (scratch bytes per lane != 0) may have parked a fragment in memory before it arrived.
    hipFuncAttributes attr;
    if (hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(kernel_persist)) != hipSuccess || attr.localSizeBytes != 0 ||
        aat::allow_lds(kernel_persist, shared_mem_persist) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel_persist), Nthreads, shared_mem_persist) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu <= 0 || cus <= 0)
      blocks = -1;
    else
      blocks = per_cu * cus;
    cached[dev].store(blocks, std::memory_order_relaxed);
  }}
  return blocks > 0 ? blocks : 0;
}}

// Whether `n` equal workgroups come out as whole rounds over the workgroups the chip holds at this configuration's
// occupancy (registers: waves_per_eu waves per SIMD; the LDS may allow fewer, which this does not look at).
bool pairs_fill_the_chip(int n) {{
  static std::atomic<int> cus_of[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  int cus = cus_of[dev].load(std::memory_order_relaxed);
  if (cus == 0) {{
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = -1;
    cus_of[dev].store(cus, std::memory_order_relaxed);
  }}
  if (cus <= 0) return false;
  // a build of the paired kernel that keeps part of its working set in scratch memory (the second pass costs registers)
  // loses more than the pairing gains: the one-row-block-per-workgroup kernel stands in
  static const bool paired_spills = [] {{
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(kernel_causal_paired)) != hipSuccess || attr.localSizeBytes != 0;
  }}();
  if (paired_spills) return false;
  const int per_cu = waves_per_eu * 4 * 64 / Nthreads > 0 ? waves_per_eu * 4 * 64 / Nthreads : 1;
  const int resident = cus * per_cu;
  return n % resident == 0 || n >= 8 * resident;
}}
#endif

bool lengths_ok(int B, int H, int Seq_q, int Seq_k) {{ return aat::shape_ok(B, H, Seq_q, Seq_k, 32, 32); }}
bool whole_tiles(int Seq_q, int Seq_k) {{ return AAT_KV_GROUPS == 1 && Seq_q % Br == 0 && Seq_k % Bc == 0; }}
int row_blocks(int Seq_q) {{ return (Seq_q + Br - 1) / Br; }}

#if AAT_KV_GROUPS > 1
int kv_parts(int, int, int, int, int) {{ return 1; }}
#else
constexpr aat::ForwardShape kShape = {{Br, Bc, Kd, D, Nthreads / 64, aat::forward_blocks_per_cu(Nthreads / 64, waves_per_eu, shared_mem_split),
                                      (num_stages_qk == 1) + (num_stages_v == 1)}};
int kv_parts(int B, int H, int Seq_q, int Seq_k, int causal) {{
  if (kv_splits > 1) return causal ? 1 : kv_splits;
  return aat::choose_kv_parts(kShape, B, H, Seq_q, Seq_k, causal);
}}
#endif
size_t split_workspace_bytes(int parts, int B, int H, int Seq_q) {{
  return parts > 1 ? (size_t)parts * B * H * Seq_q * (D + 1) * sizeof(float) : 0;
}}
// Whether a call without room for its parts is an error.  A fixed number of parts that divides the kv tiles insists on it, as
// the caller asked for those parts; everything else runs in one part instead.
bool room_missing(int B, int H, int Seq_q, int Seq_k, int causal, const void* workspace, size_t workspace_bytes) {{
  return kv_splits > 1 && !causal && Seq_k % Bc == 0 && (Seq_k / Bc) % kv_splits == 0 &&
         (workspace == nullptr || workspace_bytes < split_workspace_bytes(kv_splits, B, H, Seq_q));
}}
size_t needed_workspace(int B, int H, int Seq_q, int Seq_k, int causal) {{
  return split_workspace_bytes(kv_parts(B, H, Seq_q, Seq_k, causal), B, H, Seq_q);
}}

hipError_t launch(aat_half* q, aat_half* k, aat_half* v, aat_half* o, int B, int H, int Seq_q, int Seq_k,
                  float softmax_scale, int causal, void* workspace, size_t workspace_bytes, hipStream_t stream, float* lse = nullptr) {{
  causal = causal != 0;                          // any value but 0 asks for the causal walk; the general kernel multiplies by it
#if AAT_KV_GROUPS == 1
  const int parts = kv_parts(B, H, Seq_q, Seq_k, causal);
  if (parts > 1 && workspace != nullptr && workspace_bytes >= split_workspace_bytes(parts, B, H, Seq_q)) {{
    static const hipError_t lds_ok_split = aat::allow_lds(kernel_split, shared_mem_split);
    if (lds_ok_split != hipSuccess) return lds_ok_split;
    const size_t rows = (size_t)B * H * Seq_q;
    float* part_o = static_cast<float*>(workspace);
    float* part_lse = part_o + (size_t)parts * rows * D;
    kernel_split<<<dim3(B * H * row_blocks(Seq_q), parts), dim3(Nthreads), shared_mem_split, stream>>>(
        reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
        reinterpret_cast<const aat::half_t*>(v), nullptr, nullptr, H, Seq_k, Seq_q, softmax_scale, part_o, part_lse, (int)rows, causal);
    const size_t threads = rows * (D / 8);
    aat::attn_split_merge<D><<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream>>>(
        part_o, part_lse, reinterpret_cast<aat::half_t*>(o), lse, (int)rows, parts);
    return hipGetLastError();
  }}
#endif
  if (!whole_tiles(Seq_q, Seq_k)) {{
    static const hipError_t lds_ok_gen = aat::allow_lds(kernel_gen, shared_mem);
    if (lds_ok_gen != hipSuccess) return lds_ok_gen;
    kernel_gen<<<dim3(B * H * row_blocks(Seq_q)), dim3(Nthreads), shared_mem, stream>>>(
        reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
        reinterpret_cast<const aat::half_t*>(v), reinterpret_cast<aat::half_t*>(o), lse, H, Seq_k, Seq_q, softmax_scale, nullptr,
        nullptr, 0, causal);
    return hipGetLastError();
  }}
#if AAT_KV_GROUPS == 1
  const int items = B * H * (Seq_q / Br);
  if (kernel_persist != nullptr && !causal && (Seq_k / Bc) % 2 == 0 && Seq_k <= kPersistMaxKv) {{
    const int resident = resident_blocks();
    if (resident > 0 && items > resident) {{
      kernel_persist<<<dim3(resident), dim3(Nthreads), shared_mem_persist, stream>>>(
          reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
          reinterpret_cast<const aat::half_t*>(v), reinterpret_cast<aat::half_t*>(o), lse, H, Seq_k, Seq_q,
          softmax_scale, nullptr, nullptr, items, 0);
      return hipGetLastError();
    }}
  }}
  static const hipError_t lds_ok = aat::allow_lds(kernel, shared_mem);
  static const hipError_t lds_ok_causal = aat::allow_lds(kernel_causal, shared_mem);
  if (lds_ok != hipSuccess) return lds_ok;
  if (lds_ok_causal != hipSuccess) return lds_ok_causal;
  // causal, an even number of row blocks per head: half the grid, every workgroup walks a long and a short row block --
  // where those workgroups fill the chip a whole number of times (or many times over); a last round that is one third
  // full costs more than the equal lengths and the shared K/V stream gain
  const bool paired = causal && (Seq_q / Br) % 2 == 0 && pairs_fill_the_chip(items / 2);
  static const hipError_t lds_ok_paired = aat::allow_lds(kernel_causal_paired, shared_mem);
  if (lds_ok_paired != hipSuccess) return lds_ok_paired;
  (paired ? kernel_causal_paired : causal ? kernel_causal : kernel)<<<dim3(paired ? items / 2 : items), dim3(Nthreads), shared_mem, stream>>>(
      reinterpret_cast<const aat::half_t*>(q), reinterpret_cast<const aat::half_t*>(k),
      reinterpret_cast<const aat::half_t*>(v), reinterpret_cast<aat::half_t*>(o), lse, H, Seq_k, Seq_q,
      softmax_scale, nullptr, nullptr, 0, causal);
#endif
  return hipGetLastError();
}}
}}  // namespace

extern "C" int abi_version(void) {{ return AAT_ABI_VERSION; }}
extern "C" const char* config_string(void) {{ return "{config_name}"; }}
extern "C" size_t workspace_size(int B, int H, int Seq_q, int Seq_k) {{   // room for either kind of call
  const size_t full = needed_workspace(B, H, Seq_q, Seq_k, 0), causal = needed_workspace(B, H, Seq_q, Seq_k, 1);
  return full > causal ? full : causal;
}}
"""

profile_func = r"""
extern "C" float profile_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* o, int B, int H, int Seq_q, int Seq_k,
                            float softmax_scale, int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return -1.f;
  if (room_missing(B, H, Seq_q, Seq_k, causal, workspace, workspace_bytes)) return -1.f;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return aat::timed_mean_ms(s, [&] {{ return launch(q, k, v, o, B, H, Seq_q, Seq_k, softmax_scale, causal, workspace, workspace_bytes, s); }});
}}
// The reference signature has no workspace argument: a kv-splitting configuration runs unsplit here.
extern "C" float profile(aat_half* q, aat_half* k, aat_half* v, aat_half* o, int B, int H, int Seq_q, int Seq_k) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return -1.f;
  return aat::timed_mean_ms(nullptr, [&] {{ return launch(q, k, v, o, B, H, Seq_q, Seq_k, kReferenceScale, 0, nullptr, 0, nullptr); }});
}}
"""

kernel_entry = r"""
extern "C" int kernel_entry_ex(aat_half* q, aat_half* k, aat_half* v, aat_half* o, int B, int H, int Seq_q, int Seq_k,
                               float softmax_scale, int causal, void* workspace, size_t workspace_bytes, void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  if (room_missing(B, H, Seq_q, Seq_k, causal, workspace, workspace_bytes)) return AAT_ERR_WORKSPACE;
  return (int)launch(q, k, v, o, B, H, Seq_q, Seq_k, softmax_scale, causal, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}}
extern "C" int kernel_entry(aat_half* q, aat_half* k, aat_half* v, aat_half* o, int B, int H, int Seq_k, int Seq_q) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  return (int)launch(q, k, v, o, B, H, Seq_q, Seq_k, kReferenceScale, 0, nullptr, 0, nullptr);
}}
extern "C" int kernel_entry_lse(aat_half* q, aat_half* k, aat_half* v, aat_half* o, float* lse, int B, int H, int Seq_q,
                                int Seq_k, float softmax_scale, int causal, void* workspace, size_t workspace_bytes,
                                void* stream) {{
  if (!lengths_ok(B, H, Seq_q, Seq_k)) return AAT_ERR_SHAPE;
  if (room_missing(B, H, Seq_q, Seq_k, causal, workspace, workspace_bytes)) return AAT_ERR_WORKSPACE;
  return (int)launch(q, k, v, o, B, H, Seq_q, Seq_k, softmax_scale, causal, workspace, workspace_bytes, static_cast<hipStream_t>(stream), lse);
}}
"""

# One library carries both halves of the ABI, so tuning and running share a single compile.
profile_code = global_vars + profile_func + kernel_entry
kernel_code = profile_code
