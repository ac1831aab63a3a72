"""RetNet forward and backward at lengths their row blocks do not divide: the edges of the blocks, in every mask mode, against
the oracle's exact form under the rounded-operand rule of oracle/tolerance.py (S / r, P and dS are rounded to fp16)."""
import pytest
import torch

import attention_autotuner_amd as aat
from attention_autotuner_amd.autotuner import Runtime, gfx950_space, prebuilt_extra
from oracle import ref_op, tolerance

pytestmark = pytest.mark.gpu
ARCH = aat.MI355X()
# less than a block, one 64-row step over it, either side the longer one, and lengths at which dS is stored in part of a block
SHAPES = [(1, 2, 64, 64), (2, 2, 192, 192), (1, 2, 128, 320), (1, 2, 320, 128), (1, 2, 576, 576)]
# the configurations whose streamed tiles have 32 rows: rule shapes, and two row groups per wave in every pass
WITH_32_ROW_STREAMS = [c for op in ("ret", "ret_bwd") for d in sorted(gfx950_space.RET_RULE) for c in gfx950_space.rule_ret_configs(op, *d)
                       if c.Bc == 32] + [c for c in prebuilt_extra.ragged_row_group_configs() if c.operation != "attn_bwd"]


def _problem(b, h, sq, sk, dqk, dv, mode, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v, do = (torch.randn(b, h, s, d, generator=g).half() for s, d in ((sq, dqk), (sk, dqk), (sk, dv), (sq, dv)))
    i, j = torch.arange(sq).view(1, sq, 1) + (sk - sq), torch.arange(sk).view(1, 1, sk)
    gamma = 1.0 - torch.pow(2.0, -5.0 - torch.arange(h, dtype=torch.float64))
    decay = torch.where(j <= i, gamma.view(h, 1, 1) ** (i - j).clamp(min=0), torch.zeros((), dtype=torch.float64))
    mask = torch.randn(h, sq, sk, generator=g).half() if mode == "dense" else decay.float() if mode == "decay" else decay.float().half()
    return q, k, v, do, mask, torch.log2(gamma).float()


def _check(problem, dqk, dv, mode, seed, forward, backward):
    b, h, sq, sk = problem
    q, k, v, do, mask, lg = _problem(b, h, sq, sk, dqk, dv, mode, seed)
    o_want, r_want = ref_op.retnet_ref(q, k, v, mask, return_r=True)
    s = (q.float() @ k.float().transpose(-1, -2)) * mask.float()
    o_terms = (s.abs() / s.abs().sum(-1, keepdim=True).clamp(min=1.0)) @ v.float().abs()
    want, terms = ref_op.retnet_bwd_ref(q, k, v, mask, do), ref_op.retnet_bwd_rounding_bound(q, k, v, mask, do)
    qc, kc, vc, dc, rc = (t.cuda() for t in (q, k, v, do, r_want.reshape(b, h, sq)))
    mc = lg.cuda() if mode == "decay" else mask.cuda()
    how = dict(decay=True) if mode == "decay" else dict(causal={"dense": False, "causal": True}.get(mode, mode))
    for cfg in forward:
        print(mode, (b, h, sq, sk), cfg, flush=True)
        o, r = torch.full_like(dc, 7.0), torch.full((b, h, sq), 7.0, device="cuda")
        Runtime(ARCH, cfg).apply([qc, kc, vc, mc, o, r], **how)
        torch.cuda.synchronize()
        ok, worst, ratio = tolerance.check_rounded_operand(o, o_want, o_terms)
        assert ok, ("o", worst, ratio)
        assert ((r.cpu() - r_want.reshape(b, h, sq)).abs() / r_want.reshape(b, h, sq)).max().item() <= 1e-4
    for cfg in backward:
        print(mode, (b, h, sq, sk), cfg, flush=True)
        out = [torch.full_like(t, 7.0) for t in (qc, kc, vc)]
        Runtime(ARCH, cfg).apply([qc, kc, vc, mc, dc, rc, *out] + ([] if mode == "decay" else [torch.empty(1, device="cuda")]), **how)
        torch.cuda.synchronize()
        for name, got, ref, t in zip(("dq", "dk", "dv"), out, want, terms):
            ok, worst, ratio = tolerance.check_rounded_operand(got, ref, t)
            assert ok, (name, worst, ratio)


@pytest.mark.parametrize("dqk,dv", sorted(gfx950_space.RET_RULE))
@pytest.mark.parametrize("mode", ["dense", "causal", "scan", "decay"])
def test_every_rule_shape_at_the_edges_of_its_blocks(dqk, dv, mode):
    for i, problem in enumerate(SHAPES):
        _check(problem, dqk, dv, mode, 500 + i, gfx950_space.rule_ret_configs("ret", dqk, dv), gfx950_space.rule_ret_configs("ret_bwd", dqk, dv))


@pytest.mark.parametrize("dqk,dv", sorted({(c.Kd, c.D) for c in WITH_32_ROW_STREAMS}))
@pytest.mark.parametrize("mode", ["dense", "causal", "scan", "decay"])
def test_resident_lengths_that_are_odd_multiples_of_32(dqk, dv, mode):
    """Streams of 32-row tiles: a last block may hold one of the two row groups of a wave, and half a 64-row step of the mask."""
    cfgs = [c for c in WITH_32_ROW_STREAMS if (c.Kd, c.D) == (dqk, dv)]
    for i, problem in enumerate([(1, 2, 96, 96), (1, 2, 160, 288), (2, 1, 288, 160)]):
        _check(problem, dqk, dv, mode, 700 + i, [c for c in cfgs if c.operation == "ret"], [c for c in cfgs if c.operation == "ret_bwd"])


def test_the_scanned_walk_of_a_ragged_length_gives_the_dense_walks_bits():
    q, k, v, do, mask, _ = (t.cuda() for t in _problem(2, 3, 704, 704, 128, 128, "scan", 9))
    scan = aat.retnet_mask_scan(mask, ARCH)
    for cfg in gfx950_space.rule_ret_configs("ret", 128, 128):
        outs = []
        for how in (dict(causal=False), dict(causal="scanned", workspace=scan)):
            o, r = torch.full_like(do, 7.0), torch.full((2, 3, 704), 7.0, device="cuda")
            Runtime(ARCH, cfg).apply([q, k, v, mask, o, r], **how)
            outs.append((o, r))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]), cfg
    for cfg in gfx950_space.rule_ret_configs("ret_bwd", 128, 128):
        grads = []
        for how in (dict(causal=False), dict(causal="scanned", workspace=scan)):
            g = [torch.full_like(t, 7.0) for t in (q, k, v)]
            Runtime(ARCH, cfg).apply([q, k, v, mask, do, outs[0][1], *g, torch.empty(1, device="cuda")], **how)
            grads.append(g)
        assert all(torch.equal(a, b) for a, b in zip(*grads)), cfg
