"""Search space and validity model for MI355X (gfx950).

The knobs that matter on CDNA4 are not the ones that matter on Ampere: tiles are built from
32x32x16 MFMAs so every wave owns whole 32-row groups; K/V reach LDS by LDS-DMA so "stages" are
whole-tile buffers; and the register file is split between the resident waves of a SIMD, so the
occupancy target (``waves_per_eu``) is itself a knob.  Validity is LDS bytes (160 KB per CU, shared by
all resident blocks) and a per-lane register estimate (512 / waves_per_eu).
"""
import math

from .configs import AttnConfig, RetConfig, RetBwdConfig, AttnBwdConfig


class NoValidConfigError(ValueError):
    """No configuration of the gfx950 space fits the problem (head sizes beyond what one wave's registers or
    the LDS hold, a sequence length no tile divides)."""

WAVE = 64
MFMA_M = 32
BR_LIST = (64, 128, 256, 512)
BC_LIST = (32, 64, 128)
THREADS = (128, 256, 512)
STAGES = ((1, 1), (2, 2), (2, 1), (1, 2))
KV_SPLITS = (2, 4, 8, 16)


def _waves(cfg):
    return cfg.Nthreads // WAVE


def rows_per_wave(cfg):
    return cfg.Br * getattr(cfg, "kv_groups", 1) // _waves(cfg)


def blocks_per_cu(cfg):
    """Resident blocks per CU implied by the occupancy target (4 SIMDs per CU)."""
    return max(1, (cfg.waves_per_eu * 4) // _waves(cfg))


def unit_rows(cfg):
    """kv rows of one scores -> softmax -> PV unit of the register-fused attention forward (plain schedule):
    ``BlockKSmem2``, a divisor of Bc; the whole tile everywhere else."""
    if cfg.operation == "attn" and cfg.fuse_type == "register" and not getattr(cfg, "sw_pipeline", 0):
        return getattr(cfg, "BlockKSmem2", cfg.Bc) or cfg.Bc
    return cfg.Bc


def dma_divisible(cfg):
    nt = cfg.Nthreads
    return (cfg.Bc * cfg.Kd // 8) % nt == 0 and (cfg.Bc * cfg.D // 8) % nt == 0


# ---- forward (attention and RetNet) ------------------------------------------------------------------
def forward_lds_bytes(cfg):
    main = cfg.num_stages_qk * cfg.Bc * cfg.Kd * 2 + cfg.num_stages_v * cfg.Bc * cfg.D * 2
    if cfg.operation == "ret":
        main += max(cfg.num_stages_mask, cfg.num_stages_qk) * cfg.Br * cfg.Bc * 2
    if cfg.fuse_type == "shared":
        main += cfg.Br * (cfg.Bc * 2 + 16)            # P tile, fp16, padded rows
        main += (cfg.warps_mma1_n * cfg.Br + cfg.Br) * 4 + 64
        return max(main, cfg.Br * (cfg.D * 2 + 16 * cfg.warps_mma_n))
    epilogue = cfg.Br * (cfg.D * 2 + 16)
    handed = (getattr(cfg, "kv_groups", 1) - 1) * cfg.Br * (cfg.D * 4 + 16)      # what waves that share rows hand over
    return max(main, epilogue, handed)


def forward_reg_estimate(cfg):
    """Per-lane 32-bit registers of the dominant live set."""
    if cfg.fuse_type == "shared":
        nw = _waves(cfg)
        rt1 = cfg.Br // (nw // cfg.warps_mma1_n) // 32
        nt1 = cfg.Bc // cfg.warps_mma1_n // 32
        o_regs = cfg.Br * cfg.D // (nw * 64)
        return rt1 * (cfg.Kd // 16) * 4 + rt1 * nt1 * 16 + o_regs + 48
    rt = rows_per_wave(cfg) // MFMA_M
    unit = unit_rows(cfg)
    q_regs = rt * (cfg.Kd // 16) * 4
    s_regs = rt * (unit // 32) * 16
    p_regs = rt * (unit // 32) * 4              # fp16 P, built while the fp32 scores retire
    if cfg.fuse_type == "register":
        o_regs = rt * (cfg.D // 32) * 16
    else:
        # shared fuse: the waves split D between them for the second contraction
        o_regs = (cfg.Br // MFMA_M) * (cfg.D // 32) * 16 // _waves(cfg)
    if getattr(cfg, "sw_pipeline", 0):
        s_regs *= 2                                   # current and next score tile are both live
    # a count of what must be live, not a prediction of what the register allocator achieves: candidates that
    # pass it and still spill are rejected by the tuning loop from the compiler's own resource report
    # (a kernel this close to its budget derives its operand addresses from one register each and keeps two-slot
    # operand rings: 24 registers besides the tiles)
    return q_regs + s_regs + p_regs + o_regs + (24 if unit < cfg.Bc else 32)


def forward_likely_spills(cfg):
    """Register-fused configurations whose accumulator alone takes half of a wave's budget have always come
    back from hipcc with hundreds of bytes of scratch.  The tuning loop lets the compiler's report decide;
    the untuned defaults stay clear of them without compiling anything."""
    if cfg.fuse_type != "register":
        return False
    rt = rows_per_wave(cfg) // MFMA_M
    o_regs = rt * (cfg.D // 32) * 16
    return o_regs > 128 and rt * (cfg.Kd // 16) * 4 + rt * (cfg.Bc // 32) * 16 + o_regs > 320


def shared_grid_ok(cfg):
    """Wave grids of the LDS-fused kernels: W1M x W1N over (rows, kv), W2M x W2N over (rows, d)."""
    nw, w1n, w2n = _waves(cfg), cfg.warps_mma1_n, cfg.warps_mma_n
    if not w1n or not w2n or nw % w1n or nw % w2n:
        return False
    w1m, w2m = nw // w1n, nw // w2n
    if cfg.Br % (32 * w1m) or cfg.Bc % (32 * w1n) or cfg.Br % (32 * w2m) or cfg.D % (32 * w2n):
        return False
    return True


def forward_valid(cfg, arch):
    if cfg.fuse_type == "shared":
        if cfg.Nthreads % WAVE or not shared_grid_ok(cfg):
            return False
    elif cfg.Nthreads % WAVE or _waves(cfg) % getattr(cfg, "kv_groups", 1) or cfg.Br % (MFMA_M * (_waves(cfg) // getattr(cfg, "kv_groups", 1))):
        return False
    if getattr(cfg, "kv_groups", 1) > 1 and not (cfg.operation == "attn" and cfg.fuse_type == "register" and not cfg.sw_pipeline and cfg.kv_splits == 1 and
                                                 rows_per_wave(cfg) == MFMA_M and cfg.num_stages_qk == cfg.num_stages_v == 2 and
                                                 cfg.Bc // unit_rows(cfg) % cfg.kv_groups == 0):
        return False
    if cfg.Bc % 32 or cfg.Kd % 64 or cfg.D % 64:
        return False
    unit = unit_rows(cfg)
    if unit % 32 or cfg.Bc % unit:
        return False
    if unit < cfg.Bc and not (cfg.num_stages_qk == 2 and cfg.num_stages_v == 2):   # no barrier between the contractions of a unit
        return False
    if _waves(cfg) > 4 * cfg.waves_per_eu:           # the block itself needs that many waves per SIMD
        return False
    if not dma_divisible(cfg):
        return False
    if getattr(cfg, "sw_pipeline", 0):
        # needs 2+2 buffers and K copies made of whole 32-row units
        rows_per_dma = cfg.Nthreads * 8 // cfg.Kd if (cfg.Nthreads * 8) % cfg.Kd == 0 else 0
        if not (cfg.num_stages_qk == 2 and cfg.num_stages_v == 2 and cfg.fuse_type == "register"):
            return False
        if rows_per_dma == 0 or rows_per_dma > 32 or 32 % rows_per_dma:
            return False
    if forward_lds_bytes(cfg) * blocks_per_cu(cfg) > arch.smem_cap:
        return False
    return forward_reg_estimate(cfg) <= arch.register_per_thread // cfg.waves_per_eu




def forward_candidates(op, br, bc, dim_qk, dim_v, fuse_types=("register", "shared"), with_splits=False):
    out = []
    for nthreads in THREADS:
        for st_qk, st_v in STAGES:
            for wpe in (1, 2, 3):
                for fuse in fuse_types:
                    if fuse == "shared":
                        if st_qk == st_v and wpe <= 2:   # the LDS-fused kernels gain little from mixed buffering
                            out.extend(_shared_candidates(op, br, bc, dim_qk, dim_v, st_qk, st_v, nthreads, wpe))
                        continue
                    if op == "attn":
                        cfg = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, st_qk, st_v, nthreads, True, waves_per_eu=wpe)
                    else:
                        cfg = RetConfig(br, bc, dim_qk, dim_v, dim_qk, bc, st_qk, st_qk, st_v, nthreads, True, waves_per_eu=wpe)
                    out.append(cfg.set_fuse_type(fuse))
                    if op == "attn" and fuse == "register" and (st_qk, st_v) == (2, 2):
                        piped = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, 2, 2, nthreads, True, waves_per_eu=wpe, sw_pipeline=1)
                        out.append(piped.set_fuse_type(fuse))
                    if op == "attn" and fuse == "register" and (st_qk, st_v) == (2, 2) and br // (nthreads // WAVE) >= 2 * MFMA_M:
                        # two or more 32-row groups per wave: a kv tile worked through in 32-row units keeps one
                        # small score tile live, which is what lets such a wave share its SIMD with a second one
                        for unit in (32, 64):
                            if unit < bc:
                                for ns in (1,) + (KV_SPLITS if with_splits else ()):
                                    u = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, unit, 2, 2, nthreads, True, waves_per_eu=wpe, kv_splits=ns)
                                    out.append(u.set_fuse_type(fuse))
                    if op == "attn" and fuse == "register" and with_splits and st_qk == st_v:
                        for ns in KV_SPLITS:   # long kv, few query rows: cut the kv range so every CU gets work
                            sp = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, st_qk, st_v, nthreads, True, waves_per_eu=wpe, kv_splits=ns)
                            out.append(sp.set_fuse_type(fuse))
    return out


def _shared_candidates(op, br, bc, dim_qk, dim_v, st_qk, st_v, nthreads, wpe):
    out = []
    nw = nthreads // WAVE
    for w1n in (1, 2, 4):
        for w2n in sorted({nw, max(1, nw // 2), max(1, nw // 4)}):
            if op == "attn":
                cfg = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, st_qk, st_v, nthreads, True, w1n, w2n, waves_per_eu=wpe)
            else:
                cfg = RetConfig(br, bc, dim_qk, dim_v, dim_qk, bc, st_qk, st_qk, st_v, nthreads, True, w1n, w2n, waves_per_eu=wpe)
            cfg.fuse_type = "shared"
            if shared_grid_ok(cfg):
                out.append(cfg)
    return out


MIN_LENGTH = 32               # the register-fused forwards and both backwards take resident lengths that are multiples of this


def _divides(tile, *seqs):
    return all(not s or s % tile == 0 for s in seqs)


# From this length on a last row block that is partial wastes less than the larger block gains.  Timed at 192 ... 1600 rows and 16
# and 96 (batch, head)s, causal and not, against the 64-row shape that divides the lengths: at 1088 and 1600 rows the forwards
# take 0.51 ... 0.97 of its time (attention 64/128, 128/192, 256/128, 128/256; RetNet 64/128, 256/128, 128/256) and the RetNet
# backward 0.81 ... 0.94; at 320 rows both directions take 0.87 ... 1.6.  256-row blocks at lengths 128 divides take up to 1.5 times
# the time of 128-row ones (640 rows), and a RetNet shape of them that spills 5.9 times (128/256), so only 128-row blocks may be partial.
PARTIAL_FROM = 1024
PARTIAL_ROWS = 128


def _rounds(cfg, arch, b, h, seq):
    return -(-b * h * -(-seq // cfg.Br) // (arch.compute_max_core * blocks_per_cu(cfg)))


def _pick(candidates, fits, partial_pays=lambda whole, partial: True):
    """The first of ``candidates`` (larger blocks first) for a length: one whose tiles divide it; where that is a block smaller than
    PARTIAL_ROWS, a partial one of PARTIAL_ROWS that pays; where nothing divides the length, the smallest that takes it.
    ``fits(cfg)``: 2 for whole tiles, 1 for partial ones, 0 for a length the kernel does not take; ``candidates`` may be a
    generator of configurations that are all valid."""
    candidates = list(candidates)
    whole = next((c for c in candidates if fits(c) == 2), None)
    if whole is not None and whole.Br >= PARTIAL_ROWS:
        return whole
    partial = next((c for c in candidates if c.Br == PARTIAL_ROWS and fits(c) == 1), None)
    if whole is None:
        return next((c for c in reversed(candidates) if fits(c)), None)
    return partial if partial is not None and partial_pays(whole, partial) else whole


def _long(*seqs):
    return all(s and s >= PARTIAL_FROM for s in seqs)


def default_forward_config(op, dim_qk, dim_v, arch, seq_q=None, seq_k=None, problem=None):
    """A configuration that is valid for every supported head size; used before/without tuning.  ``problem``: batch, heads
    and causal, for a choice that looks at the whole problem where there is a rule for one."""
    if problem is not None and covered_by_rule(op, dim_qk, dim_v):
        cfg = rule_forward_config(dim_qk, dim_v, arch, *problem[:2], seq_q, seq_k, problem[2]) if op == "attn" else \
            rule_ret_config("ret", dim_qk, dim_v, *problem[:2], seq_q, seq_k, problem[2])
        if cfg is not None:
            return cfg
    prefs = [(256, 64, 512, 2, 2, 2), (128, 64, 256, 2, 2, 2), (128, 64, 256, 1, 1, 2), (128, 64, 256, 1, 1, 1), (128, 32, 256, 1, 1, 1),
             (64, 32, 128, 1, 1, 1)]
    if op == "ret" and dim_v == 512 and _divides(128, seq_q) and _divides(64, seq_k):
        # 32 rows x 512 columns per wave fill the 256 accumulation registers of a wave that has its SIMD to itself;
        # the RetNet kernel is written so that this builds without scratch, and at d_qk 256 it leads every mask mode
        cfg = RetConfig(128, 64, dim_qk, dim_v, dim_qk, 64, 1, 1, 1, 256, True, waves_per_eu=1)
        cfg.set_fuse_type("register")
        if forward_valid(cfg, arch):
            return cfg
    def shapes():
        for br, bc, nt, sq, sv, wpe in prefs:
            if op == "attn":
                cfg = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, sq, sv, nt, True, waves_per_eu=wpe)
            else:
                cfg = RetConfig(br, bc, dim_qk, dim_v, dim_qk, bc, sq, sq, sv, nt, True, waves_per_eu=wpe)
            cfg.set_fuse_type("register")
            if forward_valid(cfg, arch) and not forward_likely_spills(cfg):
                yield cfg

    def fits(cfg):
        if _divides(cfg.Br, seq_q) and _divides(cfg.Bc, seq_k):
            return 2
        step = MIN_LENGTH if op == "attn" else cfg.Bc
        return int(_divides(MIN_LENGTH, seq_q) and _divides(step, seq_k) and (not seq_q or seq_q > cfg.Br))
    cfg = _pick(shapes(), fits, lambda whole, partial: _long(seq_q))
    if cfg is not None:
        return cfg
    # wide value heads: the LDS-fused kernel keeps the accumulator at Br*D/(64*waves) registers
    for br, bc, nt, w1n, w2n in ((128, 64, 512, 2, 8), (64, 64, 256, 2, 4)):
        if (seq_q and seq_q % br) or (seq_k and seq_k % bc):
            continue
        if op == "attn":
            cfg = AttnConfig(br, bc, dim_qk, dim_v, dim_qk, bc, 1, 1, nt, True, w1n, w2n, waves_per_eu=nt // 256)
        else:
            cfg = RetConfig(br, bc, dim_qk, dim_v, dim_qk, bc, 1, 1, 1, nt, True, w1n, w2n, waves_per_eu=nt // 256)
        cfg.fuse_type = "shared"
        if forward_valid(cfg, arch):
            return cfg
    raise NoValidConfigError(f"no default {op} configuration fits dim_qk={dim_qk} dim_v={dim_v} seq=({seq_q},{seq_k})")


# ---- attention forward without a tuned entry -----------------------------------------------------------
# Tile shapes the rule below chooses from, per pair of head sizes: (Br, Bc, unit rows, K buffers, V buffers, threads,
# waves per SIMD).  Of 38 shapes timed on 26 problems (64 ... 16384 rows, ragged lengths, 1 ... 32 kv parts) these are the ones
# without which some problem loses: with one of them at hand a problem is on the mean 4 % (d 64, 128, 192) to 6 % (d 256)
# slower than with the best of the 38.
RULE_SHAPES = {
    (64, 64): ((128, 64, 64, 2, 2, 256, 3), (256, 64, 64, 2, 1, 256, 2)),
    (128, 128): ((128, 64, 64, 2, 2, 256, 2), (256, 64, 64, 2, 2, 512, 2), (256, 64, 32, 2, 2, 256, 2), (512, 128, 32, 2, 2, 512, 2)),
    (192, 192): ((128, 32, 32, 2, 2, 256, 2), (256, 64, 64, 2, 2, 512, 2)),
    (256, 256): ((64, 64, 64, 1, 1, 128, 1), (128, 32, 32, 2, 1, 256, 2), (256, 32, 32, 2, 2, 512, 2)),
}

def covered_by_rule(op, dim_qk, dim_v):
    return (dim_qk, dim_v) in {"attn": RULE_SHAPES, "attn_bwd": ATTN_BWD_RULE, "ret": RET_RULE, "ret_bwd": RET_BWD_RULE}.get(op, ())


def rule_configs(dim_qk, dim_v):
    return [AttnConfig(br, bc, dim_qk, dim_v, dim_qk, unit, nk, nv, nt, True, waves_per_eu=wpe).set_fuse_type("register")
            for br, bc, unit, nk, nv, nt, wpe in RULE_SHAPES.get((dim_qk, dim_v), ())]


def forward_estimate_us(cfg, arch, b, h, seq_q, seq_k, causal, parts):
    """Time of one attention forward launch; the same estimate the library takes to cut the kv range into parts
    (csrc/kernels/attention/regfuse/kv_parts.h says where it comes from)."""
    waves = _waves(cfg)
    lds = cfg.Bc * (cfg.num_stages_qk * cfg.Kd + cfg.num_stages_v * cfg.D) * 2
    per_block = max(1, min(cfg.waves_per_eu * 4 // waves, 160 * 1024 // lds))
    single = (cfg.num_stages_qk == 1) + (cfg.num_stages_v == 1)
    tile = cfg.Br * cfg.Bc * 2.0 * (cfg.Kd + cfg.D) / 4.5e6 * (1.0 + 17.0 / cfg.D)
    alone = 4.55 / waves * tile
    shared = (0.72 if cfg.Br >= 512 else 0.77 if cfg.Br >= 256 else 0.87 if cfg.Br >= 128 else 1.25) * (1.0 + 0.034 * single) * tile
    start = 0.7 + 2.6e-5 * cfg.Br * (cfg.Kd + cfg.D)
    row_blocks = -(-seq_q // cfg.Br)
    tiles = -(-(-(-seq_k // cfg.Bc)) // parts)
    per_cu = b * h * row_blocks * parts / arch.compute_max_core
    us = start + tiles * alone
    if per_cu > 1.0:
        triangle = causal and seq_q == seq_k
        walked = (row_blocks + 1) / (2.0 * row_blocks) if triangle else 1.0
        queue = math.ceil(per_cu) if per_cu < 3.0 else per_cu + (0.3 if triangle else 0.6)
        rounds = math.ceil(queue / per_block) if per_cu < 3.0 * per_block else queue / per_block
        us = max(us if triangle else rounds * us, start + queue * walked * tiles * shared)
    if parts > 1:
        us += 4.0 + 1.6e-6 * parts * b * h * seq_q * cfg.D
    return us


def kv_parts(cfg, arch, b, h, seq_q, seq_k, causal):
    """Into how many parts the library of ``cfg`` cuts the kv range of a problem."""
    if cfg.kv_splits > 1:
        return 1 if causal else cfg.kv_splits
    if cfg.kv_groups > 1:
        return 1
    if seq_k < 1024 or b * h * -(-seq_q // cfg.Br) >= 2 * arch.compute_max_core:
        return 1
    return min(range(1, min(64, seq_k // 256) + 1), key=lambda p: forward_estimate_us(cfg, arch, b, h, seq_q, seq_k, causal, p))


# All queries of a (batch, head) in one row block, 160 to 256 of them: every block reads K and V of its own from memory, once, and
# what counts is how much of them it has in flight.  Blocks of eight waves have twice the copies of blocks of four under way, also
# where half of their waves have no rows, and run at 4.1 ... 4.7 TB/s where the four waves do 3.2 ... 4.1 (d 192, 160 heads of 128
# rows on 1536: 58.7 -> 46.2 us; 224 of 64 on 2176: 85.6 -> 72.8; d 256, 192 on 1024: 59.8 -> 50.7; inputs not in a cache, and 0.85
# ... 1.05 of the time where they are).  The estimate sees matrix work only and puts both within 4 %.  Fewer than 192 blocks on
# longer ranges are cut into parts by the smaller shapes, which is as good or better (d 192, 160 of 64 on 4160: 106.8 against
# 111.2); over 256 of them are more than one round.  At d 128 the gain from memory (up to 14 %) is a loss of up to 6 % from a cache.
STREAM_ROWS = 128
STREAM_BLOCKS = (160, 192, 256)
STREAM_KV = (1024, 2048)
STREAM_WIDTH = 384


def _streams_once(b, h, seq_q, seq_k):
    least, any_range, most = STREAM_BLOCKS
    return seq_q <= STREAM_ROWS and seq_k >= STREAM_KV[0] and least <= b * h <= most and (b * h >= any_range or seq_k <= STREAM_KV[1])


def rule_forward_config(dim_qk, dim_v, arch, b, h, seq_q, seq_k, causal):
    """The tile shape for an attention forward problem nobody tuned, or None (head sizes or lengths the rule does not
    cover): the one of RULE_SHAPES with the smallest estimate at the kv parts its library will take, the one of 256 rows and
    eight waves where K and V stream through once (_streams_once)."""
    if seq_q % MIN_LENGTH or seq_k % MIN_LENGTH:
        return None
    few = few_blocks_config(dim_qk, dim_v, b, h, seq_q, seq_k, causal)
    if few is not None:
        return few
    shapes = rule_configs(dim_qk, dim_v)
    if dim_qk + dim_v >= STREAM_WIDTH and _streams_once(b, h, seq_q, seq_k):
        shapes = [c for c in shapes if c.Br == 256 and c.Nthreads == 512] or shapes
    return min(shapes, default=None,
               key=lambda c: forward_estimate_us(c, arch, b, h, seq_q, seq_k, causal, kv_parts(c, arch, b, h, seq_q, seq_k, causal)))


# Launches of so few row blocks that one block's walk is their time: 32 rows a block, its waves share them and take the kv units in
# turn (``kv_groups``), or 64 rows by twice as many waves.  Per pair of head sizes, in order of preference: (rows of a block, its waves, waves per SIMD, fewest and most
# kv rows, most blocks when dense and when causal).  Kernel time against the shape taken without them, 165 problems of 2 to 32 heads, 32 to 1536
# rows: d 64 0.67 ... 0.98 up to 256 blocks of 32 rows and 0.70 ... 0.82 for the causal walks of 384 and 512, d 128 0.62 ... 0.92 up to 256;
# blocks of 64 rows up to 256 0.70 ... 0.93 (1.02 ... 1.16 on 512 keys).  Short ranges are one tile
# for every shape: 1.03 ... 1.20 on 128 keys, d 128 0.94 ... 1.08 on 256.  At d 128 a few dozen blocks on 2080 keys lose to kv parts (1.05 ... 1.23),
# at d 64 they do not (0.82 ... 0.91).
FEW_BLOCKS = {
    (64, 64): ((32, 4, 2, 160, 2112, 256, 512), (64, 8, 2, 640, 2112, 256, 256)),
    (128, 128): ((32, 4, 1, 288, 1536, 256, 256), (64, 8, 2, 640, 1536, 256, 256)),
}


def few_blocks_configs(dim_qk, dim_v):
    return [AttnConfig(br, 128, dim_qk, dim_v, dim_qk, 32, 2, 2, 64 * waves, True, waves_per_eu=wpe, kv_groups=4).set_fuse_type("register")
            for br, waves, wpe, *_ in FEW_BLOCKS.get((dim_qk, dim_v), ())]


def few_blocks_config(dim_qk, dim_v, b, h, seq_q, seq_k, causal):
    """The configuration for an attention forward of few row blocks, or None: a problem with more of them, or of other sizes.  It
    goes ahead of the entries tuned for other problems, none of which has such a kernel."""
    if seq_q % MIN_LENGTH or seq_k % MIN_LENGTH:
        return None
    for cfg, (br, _, _, least, most, dense, walked) in zip(few_blocks_configs(dim_qk, dim_v), FEW_BLOCKS.get((dim_qk, dim_v), ())):
        if least <= seq_k <= most and b * h * -(-seq_q // br) <= (walked if causal else dense):
            return cfg
    return None


# ---- backward (RetNet) ---------------------------------------------------------------------------------
# Three passes of one chained-contraction kernel (dV, dK, dQ).  Br = block-resident rows, Bc = streamed rows
# per step, for every pass; both sequence lengths must divide by both.
BWD_BR_LIST = (64, 128, 256, 512)
BWD_BC_LIST = (32, 64)


def backward_dv_cols(cfg):
    """dV columns one block produces.  With one wave per SIMD the output accumulators live in the 256
    accumulation registers, which hold a 32-row group of up to 512 columns; otherwise (or for wider
    values) the pass is sliced into 256-column blocks over grid.y and repeats its first contraction."""
    rt = cfg.Br // _waves(cfg) // MFMA_M
    if cfg.waves_per_eu == 1 and rt * cfg.D <= 512:
        return cfg.D
    return min(cfg.D, 256)


def _backward_passes(cfg):
    """(first-contraction width, output columns per block, buffers of the first stream, of the second) of the dV, dK
    and dQ passes."""
    return ((cfg.Kd, backward_dv_cols(cfg), cfg.num_stages_qk, cfg.num_stages_dv),
            (cfg.D, cfg.Kd, cfg.num_stages_ds, cfg.num_stages_dq), (cfg.D, cfg.Kd, cfg.num_stages_ds, cfg.num_stages_dq))


def backward_lds_bytes(cfg):
    worst = 0
    for kx, dzb, sy, sz in _backward_passes(cfg):
        main = sy * (cfg.Bc * kx * 2 + cfg.Br * cfg.Bc * 2) + sz * cfg.Bc * dzb * 2
        worst = max(worst, main, cfg.Br * (dzb * 2 + 16))
    return worst


def backward_reg_estimate(cfg):
    """(vector registers, accumulation registers) of the hungriest pass."""
    rt = cfg.Br // _waves(cfg) // MFMA_M
    vec = acc = 0
    for kx, dzb, _, _ in _backward_passes(cfg):
        vec = max(vec, rt * (kx // 16) * 4 + rt * (cfg.Bc // 32) * 24 + 64)
        acc = max(acc, rt * (dzb // 32) * 16)
    return vec, acc


DS_ROWS = (128, 256)          # kv rows per block of the dK kernel that reads a stored dS (64-row query tiles, two stages or more)
DS_TILE = 64


def backward_valid(cfg, arch):
    nw = _waves(cfg)
    ds_rows = getattr(cfg, "ds_rows", 0)
    if ds_rows:
        if ds_rows not in DS_ROWS or cfg.Br % DS_TILE or cfg.waves_per_eu != 1:
            return False
        # the row pass stages a dS tile behind its stream buffers; the dK kernel holds two (Q tile, dS tile) pairs
        row_lds = cfg.num_stages_ds * (cfg.Bc * cfg.D * 2 + cfg.Br * cfg.Bc * 2) + cfg.num_stages_dq * cfg.Bc * cfg.Kd * 2
        if row_lds + cfg.Br * (cfg.Bc * 2 + 16) > arch.smem_cap:
            return False
        if 2 * DS_TILE * (cfg.Kd + ds_rows) * 2 > arch.smem_cap:
            return False
    if cfg.Nthreads % WAVE or cfg.Br % (MFMA_M * nw) or cfg.Bc % 32:
        return False
    if nw > 4 * cfg.waves_per_eu:
        return False
    for sy, sz in ((cfg.num_stages_qk, cfg.num_stages_dv), (cfg.num_stages_ds, cfg.num_stages_dq)):
        if sy not in (1, 2, 3) or sz not in (1, 2):
            return False
        if sy == 3 and sz != 2:      # the three-buffer schedule prefetches Z one tile ahead
            return False
    if cfg.num_stages_mask != cfg.num_stages_qk:               # the mask tile travels with the first stream
        return False
    nt = cfg.Nthreads
    for cols in (cfg.Kd, cfg.D, backward_dv_cols(cfg), cfg.Br):   # every streamed tile must split evenly over the threads
        if (cfg.Bc * cols // 8) % nt:
            return False
    if (cfg.Br * cfg.Bc // 8) % nt:
        return False
    if backward_lds_bytes(cfg) * blocks_per_cu(cfg) > arch.smem_cap:
        return False
    vec, acc = backward_reg_estimate(cfg)
    if cfg.waves_per_eu == 1:          # 256 vector + 256 accumulation registers
        return vec <= 256 and acc <= 256
    return vec + acc <= arch.register_per_thread // cfg.waves_per_eu


BWD_STAGES = ((1, 1), (2, 2), (2, 1), (3, 2))       # (buffers of the first stream, of the second) of a pass


def backward_candidates(br, bc, dim_qk, dim_v):
    """Every combination of buffer counts for the dV pass and for the d_v-contracting passes: where d_v differs from
    d_qk the two kinds of pass stream tiles of different widths and the best counts differ with them."""
    out = []
    for nthreads in (128, 256, 512):
        for st_y, st_z in BWD_STAGES:
            for st_ds, st_dq in (BWD_STAGES if dim_qk != dim_v else ((st_y, st_z),)):
                for wpe in (1, 2):
                    n = nthreads // WAVE
                    kw = dict(BlockKSmem=dim_qk, num_stages_qk=st_y, num_stages_mask=st_y, num_stages_dv=st_z,
                              num_stages_ds=st_ds, num_stages_dq=st_dq, waves_per_eu=wpe)
                    out.append(RetBwdConfig(br, bc, dim_qk, dim_v, n, n, n, n, nthreads, True, **kw))
                    if wpe == 1:          # ... and with dS stored by the dQ pass for a dK kernel of its own (needs the workspace)
                        for ds_rows in DS_ROWS:
                            out.append(RetBwdConfig(br, bc, dim_qk, dim_v, n, n, n, n, nthreads, True, ds_rows=ds_rows, **kw))
    return out


def default_backward_config(dim_qk, dim_v, arch, seq_q=None, seq_k=None, problem=None):
    if problem is not None:
        cfg = rule_ret_config("ret_bwd", dim_qk, dim_v, *problem[:2], seq_q, seq_k, problem[2])
        if cfg is not None:
            return cfg
    prefs = ((128, 32, 256, 3, 2, 1), (128, 32, 256, 2, 2, 1), (64, 32, 128, 2, 2, 1), (64, 32, 128, 1, 1, 1), (64, 32, 128, 1, 1, 2),
             (64, 64, 128, 1, 1, 1))
    if dim_v == 512:            # measured at d_qk 256: 64-row streamed tiles with single buffers lead the three-buffer ring of 32-row tiles
        prefs = ((128, 64, 256, 1, 1, 1),) + prefs
    def shapes():
        for br, bc, nt, sy, sz, wpe in prefs:
            n = nt // WAVE
            cfg = RetBwdConfig(br, bc, dim_qk, dim_v, n, n, n, n, nt, True, BlockKSmem=dim_qk, num_stages_qk=sy,
                               num_stages_mask=sy, num_stages_dv=sz, num_stages_ds=sy, num_stages_dq=sz, waves_per_eu=wpe)
            if backward_valid(cfg, arch):
                yield cfg

    def fits(cfg):
        if not _divides(cfg.Bc, seq_q, seq_k):
            return 0
        return 2 if _divides(cfg.Br, seq_q, seq_k) else int(all(not s or s > cfg.Br for s in (seq_q, seq_k)) and _divides(MIN_LENGTH, seq_q, seq_k))

    def partial_pays(whole, partial):
        # 480 blocks of 64 rows are one round of two to a CU, the 288 blocks of 128 of the same problem are two of one: 1.6 times the time
        return _long(seq_q, seq_k) and (problem is None or all(_rounds(partial, arch, *problem[:2], s) <= _rounds(whole, arch, *problem[:2], s) for s in (seq_q, seq_k)))
    cfg = _pick(shapes(), fits, partial_pays)
    if cfg is not None:
        return cfg
    raise NoValidConfigError(f"no default ret_bwd configuration fits dim_qk={dim_qk} dim_v={dim_v} seq=({seq_q},{seq_k})")


# ---- backward (attention) ------------------------------------------------------------------------------
# A column kernel (dV, dK) and a row kernel (dQ) share Br (resident rows) and Bc (streamed rows per step).
ATTN_BWD_BR_LIST = (64, 128, 256, 512)
ATTN_BWD_BC_LIST = (32, 64)


def attn_backward_lds_bytes(cfg):
    stage = cfg.Bc * (cfg.Kd + cfg.D) * 2 + 1024            # streamed tile pair + per-row statistics slot
    return max(cfg.num_stages_qk * stage, cfg.Br * (max(cfg.Kd, cfg.D) * 2 + 16))


def attn_backward_reg_estimate(cfg):
    """(vector registers, accumulation registers) of the column kernel, the hungrier of the two."""
    rt = cfg.Br // _waves(cfg) // MFMA_M
    nt = cfg.Bc // 32
    vec = rt * ((cfg.Kd + cfg.D) // 16) * 4 + rt * nt * 16 + 72
    acc = rt * ((cfg.Kd + cfg.D) // 32) * 16                # dV + dK accumulators
    scores = rt * nt * 32                                    # S and dP tiles
    if cfg.waves_per_eu == 1 and acc + scores > 256:        # the kernel then keeps the score tiles in vector registers
        return vec + scores - rt * nt * 16, acc
    return vec, acc + scores


def attn_backward_split_reg_estimates(cfg):
    """(dV-only column kernel, dK-only column kernel) registers per lane: resident fragments, the output
    accumulators, the score tiles, the fp16 operand of the second contraction, addresses."""
    rt = cfg.Br // _waves(cfg) // MFMA_M
    nt = cfg.Bc // 32
    dv = rt * (cfg.Kd // 16) * 4 + rt * (cfg.D // 32) * 16 + rt * nt * 16 + rt * nt * 8 + 48
    dk = rt * ((cfg.Kd + cfg.D) // 16) * 4 + rt * (cfg.Kd // 32) * 16 + rt * nt * 32 + rt * nt * 8 + 48
    return dv, dk


def _one_wave_fits(rt, frag_cols, out_cols, score_tiles):
    """One wave per SIMD: 256 vector + 256 accumulation registers.  Resident fragments, the fp16 operand and
    addresses are vector registers; outputs are accumulation registers and the score tiles join them if there
    is room, else they are vector registers too."""
    vec = rt * (frag_cols // 16) * 4 + rt * 8 + 48
    acc = rt * (out_cols // 32) * 16
    scores = rt * score_tiles * 16
    if acc + scores <= 256:
        return vec <= 256 and acc <= 256
    return vec + scores <= 256 and acc <= 256


def _split_budget_ok(regs, rt, frag_cols, out_cols, score_tiles, wpe, nw, lds_bytes, arch):
    """One half of a split column kernel at ``wpe`` waves per SIMD."""
    if wpe not in (1, 2, 3) or nw > 4 * wpe:
        return False
    if lds_bytes * (max(1, (wpe * 4) // nw) if wpe > 1 else 1) > arch.smem_cap:
        return False
    if wpe == 1:
        return _one_wave_fits(rt, frag_cols, out_cols, score_tiles)
    return regs <= arch.register_per_thread // wpe


def attn_backward_valid(cfg, arch):
    nw = _waves(cfg)
    if cfg.Nthreads % WAVE or cfg.Br % (MFMA_M * nw) or cfg.Bc % 32 or cfg.Bc > 128:
        return False
    if nw > 4 * cfg.waves_per_eu or cfg.num_stages_qk not in (2, 3):
        return False
    for cols in (cfg.Kd, cfg.D):
        if cols % 64:                                              # the dual swizzle covers every multiple of 64
            return False
        if (cfg.Bc * cols // 8) % cfg.Nthreads:
            return False
    # an occupancy target above one wave per SIMD must be reachable; at one wave per SIMD a single block per CU will do
    if attn_backward_lds_bytes(cfg) * (blocks_per_cu(cfg) if cfg.waves_per_eu > 1 else 1) > arch.smem_cap:
        return False
    row_wpe = getattr(cfg, "row_waves_per_eu", cfg.waves_per_eu)
    row_bc = getattr(cfg, "row_Bc", cfg.Bc)
    if row_bc != cfg.Bc:                                     # a tile height of its own only with a budget of its own
        if row_wpe == cfg.waves_per_eu or row_bc % 32 or row_bc > 128:
            return False
        if any((row_bc * cols // 8) % cfg.Nthreads for cols in (cfg.Kd, cfg.D)):
            return False
    if row_wpe != cfg.waves_per_eu:
        if cfg.waves_per_eu != 1 or row_wpe != 2 or nw > 8:
            return False
        if attn_backward_row_reg_estimate(cfg) > arch.register_per_thread // 2:
            return False
        row_lds = max(cfg.num_stages_qk * row_bc * (cfg.Kd + cfg.D) * 2, cfg.Br * (cfg.Kd * 2 + 16))
        if row_lds * max(1, 8 // nw) > arch.smem_cap:
            return False
    elif cfg.waves_per_eu == 1:                              # the row kernel on the column kernel's budget
        if not _one_wave_fits(cfg.Br // nw // MFMA_M, cfg.Kd + cfg.D, cfg.Kd, 2 * (row_bc // 32)):
            return False
    if getattr(cfg, "col_split", 0):
        rt = cfg.Br // nw // MFMA_M
        dv, dk = attn_backward_split_reg_estimates(cfg)
        lds = attn_backward_lds_bytes(cfg)
        return (cfg.waves_per_eu == 1 and
                _split_budget_ok(dv, rt, cfg.Kd, cfg.D, cfg.Bc // 32, cfg.dv_waves_per_eu, nw, lds, arch) and
                _split_budget_ok(dk, rt, cfg.Kd + cfg.D, cfg.Kd, 2 * (cfg.Bc // 32), cfg.dk_waves_per_eu, nw, lds, arch))
    vec, acc = attn_backward_reg_estimate(cfg)
    if cfg.waves_per_eu == 1:
        return vec <= 256 and acc <= 256
    return vec + acc <= arch.register_per_thread // cfg.waves_per_eu


def attn_backward_row_reg_estimate(cfg):
    """Registers of the row kernel (resident Q and dO fragments, the dQ accumulators, S and dP, the fp16
    operand of the second contraction, addresses): 206 measured at 128/128 with 32-row tiles, 238 with 64."""
    rt = cfg.Br // _waves(cfg) // MFMA_M
    nt = getattr(cfg, "row_Bc", cfg.Bc) // 32
    return rt * ((cfg.Kd + cfg.D) // 16) * 4 + rt * (cfg.Kd // 32) * 16 + rt * nt * 32 + rt * nt * 8 + 48


def attn_backward_candidates(br, bc, dim_qk, dim_v):
    out = []
    for nthreads in (128, 256, 512):
        for stages in (2, 3):
            for wpe in (1, 2):
                out.append(AttnBwdConfig(br, bc, dim_qk, dim_v, nthreads, stages, waves_per_eu=wpe))
            for row_bc in (32, 64):
                out.append(AttnBwdConfig(br, bc, dim_qk, dim_v, nthreads, stages, waves_per_eu=1, row_waves_per_eu=2, row_Bc=row_bc))
            # one column kernel per output, each on the largest occupancy it fits
            for row_wpe in (1, 2):
                for dv_wpe, dk_wpe in ((3, 2), (2, 2), (2, 1), (1, 1)):
                    out.append(AttnBwdConfig(br, bc, dim_qk, dim_v, nthreads, stages, waves_per_eu=1, row_waves_per_eu=row_wpe,
                                             col_split=1, dv_waves_per_eu=dv_wpe, dk_waves_per_eu=dk_wpe))
    return out


def default_attn_backward_config(dim_qk, dim_v, arch, seq_q=None, seq_k=None, problem=None):
    if problem is not None:
        cfg = rule_attn_backward_config(dim_qk, dim_v, *problem[:2], seq_q, seq_k, problem[2])
        if cfg is not None:
            return cfg
    def shapes():
        for br, bc, nt, st, wpe in ((128, 32, 256, 3, 1), (128, 32, 256, 2, 1), (64, 32, 128, 3, 1), (64, 32, 128, 2, 1), (64, 32, 128, 2, 2)):
            for row_wpe in ((2, wpe) if wpe == 1 else (wpe,)):        # the row kernel at two waves per SIMD where it fits
                cfg = AttnBwdConfig(br, bc, dim_qk, dim_v, nt, st, waves_per_eu=wpe, row_waves_per_eu=row_wpe)
                if attn_backward_valid(cfg, arch):
                    yield cfg

    def split_shapes():                                               # ... or one column kernel per output
        for br, bc, nt, st in ((128, 32, 256, 3), (128, 32, 256, 2), (64, 32, 128, 2)):
            cfg = AttnBwdConfig(br, bc, dim_qk, dim_v, nt, st, waves_per_eu=1, col_split=1)
            if attn_backward_valid(cfg, arch):
                yield cfg

    def fits(cfg):
        if _divides(cfg.Br, seq_q, seq_k) and _divides(cfg.Bc, seq_q, seq_k):
            return 2
        return int(_divides(MIN_LENGTH, seq_q, seq_k) and all(not s or s > cfg.Br for s in (seq_q, seq_k)))

    def partial_pays(whole, partial):
        if problem is None:
            return _long(seq_q, seq_k)
        b, h, causal = problem
        blocks = b * h * -(-seq_k // whole.Br)
        if partial.col_split:
            # d 256/512: a block of either size has its CU to itself, so one round less is what counts (96 heads of 192 rows 0.68, of 320
            # rows 1.11 of the time; 16 of 1088 0.57), and in a causal walk, whose blocks differ in length, several rounds (96 of 1088 0.71,
            # 16 of 1088 1.08)
            per_round = arch.compute_max_core
            return -(-b * h * -(-seq_k // partial.Br) // per_round) < -(-blocks // per_round) and (not causal or blocks > 2 * per_round)
        # not causal: 0.90 ... 1.00 of the time from 1024 rows on.  Causal: 1.00 ... 1.07 at 64/128 and 256/128; 0.96 ... 1.00 at 128/192,
        # where only the larger block lets the row kernel run two waves per SIMD
        return _long(seq_q, seq_k) and _rounds(partial, arch, b, h, seq_k) <= _rounds(whole, arch, b, h, seq_k) and \
            (not causal or partial.row_waves_per_eu > whole.row_waves_per_eu)
    # head sizes whose dV and dK accumulators cannot share a wave have no shape of the first kind
    for kind in (shapes, split_shapes):
        cfg = _pick(kind(), fits, partial_pays)
        if cfg is not None:
            return cfg
    raise NoValidConfigError(f"no default attn_bwd configuration fits dim_qk={dim_qk} dim_v={dim_v} seq=({seq_q},{seq_k})")


# ---- attention backward without a tuned entry -----------------------------------------------------------
# (few blocks, many blocks) per pair of head sizes, as arguments of AttnBwdConfig behind the head sizes.  Blocks of 64 resident
# rows are two waves, two of them to a CU; blocks of 128 are four waves that share one stream.  Up to 512 blocks of 64 rows the
# smaller ones spread over more CUs (B3 H8 S1344 d 128: 112 us against 114 with two more blocks of 128 rows than there are CUs,
# d 192 156 against 235), beyond that the larger ones stream less (B4 H32 S1984 d 128 non-causal: 1026 against 1027 ... 1148), and at
# d 128 from 256 on where they all fit side by side (0.86 ... 0.91 of the time at 360 to 476 blocks of 64 rows; 1.17 and 1.22 where
# 260 blocks of 128 rows make a second round).  A causal walk's blocks are of all lengths, and finer ones end together: the line lies
# at 1600 there (from 600 to 1600 blocks the larger ones take 0.99 ... 1.10 of the time at 352 to 2112 rows).  At d 64 the smaller tile
# leaves room for four blocks to a CU, which lead beyond the line.  A causal walk at d 64 keeps the larger tile further (time of the smaller one over
# it, 18 lengths from 704 to 2048 rows): whole blocks of 64 rows, from 960 rows on, 1.00 ... 1.14 at 560 to 640 blocks and 0.98 ... 1.06 at 650 to 700; of
# 832 and 896 rows 1.01 ... 1.07 up to 611, 0.97 and 1.02 at 630; with half a block at the end, from 800 rows on, 0.99 ... 1.08 up to 576 and 0.92 ... 1.01
# around 630; shorter ones 1.0 at 550 and 0.94 ... 0.97 from 594 on.
ATTN_BWD_RULE = {
    (64, 64): (dict(Br=64, Bc=64, Nthreads=128, num_stages_qk=2, row_waves_per_eu=2, row_Bc=64),
               dict(Br=64, Bc=32, Nthreads=128, num_stages_qk=2, waves_per_eu=2, row_waves_per_eu=2)),
    (128, 128): (dict(Br=64, Bc=64, Nthreads=128, num_stages_qk=2, row_waves_per_eu=2, row_Bc=32),
                 dict(Br=128, Bc=64, Nthreads=256, num_stages_qk=2, row_waves_per_eu=2, row_Bc=32)),
    (192, 192): (dict(Br=64, Bc=32, Nthreads=128, num_stages_qk=3), dict(Br=128, Bc=32, Nthreads=256, num_stages_qk=2)),
    (256, 256): (dict(Br=128, Bc=32, Nthreads=256, num_stages_qk=2),) * 2,
}


def rule_attn_backward_configs(dim_qk, dim_v):
    return [AttnBwdConfig(Kd=dim_qk, D=dim_v, **kw) for kw in ATTN_BWD_RULE.get((dim_qk, dim_v), ())]


def rule_attn_backward_config(dim_qk, dim_v, b, h, seq_q, seq_k, causal):
    """The configuration for an attention backward problem nobody tuned, or None."""
    pair = rule_attn_backward_configs(dim_qk, dim_v)
    if not pair or seq_q % MIN_LENGTH or seq_k % MIN_LENGTH:
        return None
    blocks = b * h * -(-seq_k // 64)
    if causal:
        line = 1600 if dim_qk > 64 else 512 if seq_k < 800 else 576 if seq_k % 64 else 608 if seq_k < 960 else 640
        return pair[blocks > line]
    side_by_side = dim_qk == 128 and blocks > 256 and b * h * -(-seq_k // 128) <= 256
    return pair[blocks > 512 or side_by_side]


# ---- RetNet without a tuned entry ------------------------------------------------------------------------
# Per pair of head sizes and walk: (up to `line` blocks of 64 rows, line, beyond).  "dense" is every tile of a mask tensor;
# "skip" is a walk that leaves zero tiles out (scanned, promised, or decay rates).  Timed on 14 problems of 64 ... 3136 rows;
# a pair is 1 to 4 % slower on the mean than the best of five to seven shapes, the shape that used to stand in at lengths
# like 1344 (64 x 32 tiles, single buffers) 10 % at best and up to a half at d_v 512.  Where the line lies: two blocks of 64
# rows share a CU as one block of 128 does, so up to 512 of them the dense walk keeps more CUs busy with the smaller ones
# (B3 H8 S1344 256/256, 504 blocks: 66 us against 86 for 264 blocks of 128 rows on 32-row tiles, 102 on 64-row ones); the blocks of a skipping walk differ in length
# and balance at half as many.  Backward: blocks of 64 kv rows lead everywhere up to d 192 for the same reason, with dS stored.
#   forward  (Br, Bc, K buffers, V buffers, threads, waves per SIMD)
#   backward (Br, Bc, threads, buffers of the dV pass' two streams, of the others', waves per SIMD, ds_rows)
RET_RULE = {
    (64, 64): {"dense": ((128, 64, 2, 2, 256, 2), 0, (128, 64, 2, 2, 256, 2)), "skip": ((128, 64, 2, 2, 256, 2), 0, (128, 64, 2, 2, 256, 2))},
    (128, 128): {"dense": ((64, 64, 1, 1, 128, 2), 256, (128, 64, 1, 1, 256, 2)), "skip": ((64, 64, 1, 1, 128, 2), 256, (128, 64, 1, 1, 256, 2))},
    (192, 192): {"dense": ((64, 64, 1, 1, 128, 1), 512, (128, 64, 1, 1, 256, 2)), "skip": ((64, 64, 1, 1, 128, 1), 256, (128, 64, 2, 1, 256, 1))},
    (256, 256): {"dense": ((64, 64, 1, 1, 128, 1), 512, (128, 32, 1, 1, 256, 2)), "skip": ((64, 64, 1, 1, 128, 1), 1024, (128, 64, 1, 1, 256, 1))},
    (256, 512): {"dense": ((64, 32, 1, 1, 128, 1), 512, (128, 64, 1, 1, 256, 1)), "skip": ((64, 32, 1, 1, 128, 1), 256, (128, 64, 1, 1, 256, 1))},
}
RET_BWD_RULE = {
    (64, 64): {"dense": ((64, 64, 128, 3, 2, 3, 2, 1, 128), 512, (128, 64, 256, 2, 2, 2, 2, 2, 0)),
               "skip": ((64, 64, 128, 3, 2, 3, 2, 1, 128), 256, (128, 64, 256, 2, 2, 2, 2, 2, 0))},
    (128, 128): {"dense": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 512, (256, 64, 256, 1, 1, 1, 1, 1, 256)),
                 "skip": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 0, (64, 64, 128, 1, 1, 1, 1, 1, 128))},
    (192, 192): {"dense": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 512, (256, 32, 256, 3, 2, 3, 2, 1, 128)),
                 "skip": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 0, (64, 64, 128, 1, 1, 1, 1, 1, 128))},
    (256, 256): {"dense": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 512, (256, 32, 256, 3, 2, 3, 2, 1, 128)),
                 "skip": ((64, 64, 128, 1, 1, 1, 1, 1, 128), 512, (128, 64, 256, 1, 1, 1, 1, 1, 128))},
    (256, 512): {"dense": ((64, 32, 128, 1, 1, 1, 1, 1, 0), 128, (128, 64, 256, 1, 1, 1, 1, 1, 128)),
                 "skip": ((64, 32, 128, 1, 1, 1, 1, 1, 0), 128, (128, 64, 256, 1, 1, 1, 1, 1, 128))},
}


def _ret_config(op, dim_qk, dim_v, args):
    if op == "ret":
        br, bc, nk, nv, nt, wpe = args
        return RetConfig(br, bc, dim_qk, dim_v, dim_qk, bc, nk, nk, nv, nt, True, waves_per_eu=wpe).set_fuse_type("register")
    br, bc, nt, sy, sz, ds, dq, wpe, rows = args
    n = nt // WAVE
    return RetBwdConfig(br, bc, dim_qk, dim_v, n, n, n, n, nt, True, BlockKSmem=dim_qk, num_stages_qk=sy, num_stages_mask=sy,
                        num_stages_dv=sz, num_stages_ds=ds, num_stages_dq=dq, waves_per_eu=wpe, ds_rows=rows)


def rule_ret_configs(op, dim_qk, dim_v):
    walks = (RET_RULE if op == "ret" else RET_BWD_RULE).get((dim_qk, dim_v), {}).values()
    return [_ret_config(op, dim_qk, dim_v, args) for args in dict.fromkeys(a for few, _, many in walks for a in (few, many))]


def rule_ret_config(op, dim_qk, dim_v, b, h, seq_q, seq_k, skips):
    """The configuration for a RetNet problem nobody tuned, or None (head sizes or lengths the rule does not cover)."""
    walks = (RET_RULE if op == "ret" else RET_BWD_RULE).get((dim_qk, dim_v))
    if walks is None or seq_q % 64 or seq_k % 64:
        return None
    few, line, many = walks["skip" if skips else "dense"]
    return _ret_config(op, dim_qk, dim_v, few if b * h * (seq_q if op == "ret" else seq_k) // 64 <= line else many)
