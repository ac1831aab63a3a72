"""Attention backward at lengths its tiles do not divide: the edges of tiles, against the oracle's exact form under the
rounded-operand rule of oracle/tolerance.py."""
import math

import pytest
import torch

import attention_autotuner_amd as aat
from attention_autotuner_amd.autotuner import Runtime, codegen, gfx950_space, library, prebuilt_extra
from oracle import ref_op, tolerance

pytestmark = pytest.mark.gpu
ARCH = aat.MI355X()
# one 32-row group, one group over a tile, one short of it, either side the longer one, several blocks
SHAPES = [(1, 2, 32, 32), (2, 2, 96, 160), (1, 2, 288, 288), (1, 2, 160, 96), (1, 1, 64, 544), (1, 1, 416, 416)]


def _check(problem, dqk, dv, causal, seed, cfgs):
    b, h, sq, sk = problem
    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn(b, h, s, d, generator=g).half() for s, d in ((sq, dqk), (sk, dqk), (sk, dv), (sq, dv)))
    o, lse = ref_op.attention_ref(q, k, v, None, causal, return_lse=True)
    o = o.half()
    want = ref_op.attention_bwd_ref(q, k, v, do, None, causal)
    terms = ref_op.attention_bwd_rounding_bound(q, k, v, do, None, causal, o_stored=o)
    for cfg in cfgs:
        print(dqk, dv, causal, problem, cfg, flush=True)
        out = [torch.full_like(t, 7.0, device="cuda") for t in (q, k, v)]
        Runtime(ARCH, cfg).apply([q.cuda(), k.cuda(), v.cuda(), o.cuda(), do.cuda(), lse.cuda(), *out], softmax_scale=1 / math.sqrt(dqk), causal=causal)
        torch.cuda.synchronize()
        for name, got, ref, t in zip(("dq", "dk", "dv"), out, want, terms):
            ok, worst, ratio = tolerance.check_rounded_operand(got, ref, t)
            assert ok, (name, worst, ratio)


@pytest.mark.parametrize("d", sorted(p[0] for p in gfx950_space.ATTN_BWD_RULE))
@pytest.mark.parametrize("causal", [False, True])
def test_every_rule_shape_at_the_edges_of_its_tiles(d, causal):
    for i, problem in enumerate(SHAPES):
        _check(problem, d, d, causal, 300 + i, gfx950_space.rule_attn_backward_configs(d, d))


@pytest.mark.parametrize("causal", [False, True])
def test_two_row_groups_per_wave_and_one_column_kernel_per_output(causal):
    """A wave of the last block may have one of its two row groups; with one column kernel per output both carry the general form."""
    groups = [c for c in prebuilt_extra.ragged_row_group_configs() if c.operation == "attn_bwd"]
    assert all(c.Br // (c.Nthreads // 64) == 64 for c in groups)
    split = [prebuilt_extra.attn_bwd_split_config(*t) for t in prebuilt_extra.ATTN_BWD_SPLIT_TILES]
    wide = [gfx950_space.default_attn_backward_config(256, 512, ARCH, s, s) for s in (96, 1344)]
    assert all(c.col_split for c in split + wide)
    for i, problem in enumerate([(1, 2, 96, 160), (1, 2, 288, 288), (2, 1, 160, 96)]):
        _check(problem, 64, 64, causal, 330 + i, groups)
        _check(problem, 128, 128, causal, 340 + i, split)
        _check(problem, 256, 512, causal, 350 + i, wide)


# Heads enough for column blocks of 256 rows (130 or more blocks, 512 when causal): a last block with five 32-row groups, with six, whole
# blocks, two blocks per head; one query tile, several; either side the longer one
@pytest.mark.parametrize("problem,causal", [((10, 13, 96, 160), False), ((10, 13, 32, 256), False), ((5, 13, 64, 416), False),
                                            ((16, 32, 160, 160), True), ((16, 32, 288, 192), True), ((16, 32, 96, 256), True),
                                            ((8, 32, 352, 416), True)])
def test_column_blocks_of_256_rows(problem, causal):
    cfgs = [c for c in gfx950_space.rule_attn_backward_configs(128, 128) if c.Br == 128 and not c.col_split]
    assert cfgs
    assert library.load(codegen.compile_config(cfgs[0], ARCH), "attn_bwd").column_rows(*problem, causal) == 256
    _check(problem, 128, 128, causal, 370, cfgs[:1])


@pytest.mark.parametrize("d", sorted(p[0] for p in gfx950_space.ATTN_BWD_RULE))
def test_an_infinite_gradient_in_the_last_partial_tile_stays_an_infinity(d):
    """dV = P^T dO; the query rows a tile does not have are copies of its first 32 with P = 0, and 0 * inf must not reach dV."""
    g = torch.Generator().manual_seed(61)
    q, k, v, do = (torch.randn(1, 2, s, d, generator=g).half() for s in (160, 96, 96, 160))
    do[..., 5] = 0
    o, lse = ref_op.attention_ref(q, k, v, None, False, return_lse=True)
    o = o.half()
    want = ref_op.attention_bwd_ref(q, k, v, do, None, False)[2]
    terms = ref_op.attention_bwd_rounding_bound(q, k, v, do, None, False, o_stored=o)[2]
    do[:, :, 129, 5] = float("inf")
    for cfg in gfx950_space.rule_attn_backward_configs(d, d):
        print(d, cfg, flush=True)
        out = [torch.full_like(t, 7.0, device="cuda") for t in (q, k, v)]
        Runtime(ARCH, cfg).apply([q.cuda(), k.cuda(), v.cuda(), o.cuda(), do.cuda(), lse.cuda(), *out], softmax_scale=1 / math.sqrt(d))
        dv = out[2].cpu()
        assert (dv[..., 5] == float("inf")).all(), cfg
        dv[..., 5] = 0
        ok, worst, ratio = tolerance.check_rounded_operand(dv, want, terms)
        assert ok, (worst, ratio)
