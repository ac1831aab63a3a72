"""Attention forward at lengths its tiles do not divide and over kv ranges cut into parts: the edges of tiles, against the
oracle (the forward's own bound, 2e-3 where |ref| < 4)."""
import ctypes
import math

import pytest
import torch

import attention_autotuner_amd as aat
from attention_autotuner_amd.autotuner import Runtime, gfx950_space, library
from attention_autotuner_amd.autotuner.configs import AttnConfig
from oracle import ref_op, tolerance

pytestmark = pytest.mark.gpu
ARCH = aat.MI355X()

# (B, H, Sq, Sk): one 32-row group, a partial first tile, one row group over a tile, one short of it, more queries than keys,
# kv ranges that are cut (1024 rows and more on few row blocks), parts that see nothing under the causal mask
SHAPES = [(1, 2, 32, 32), (2, 3, 96, 160), (1, 2, 288, 288), (1, 3, 480, 544), (1, 2, 544, 96), (1, 1, 64, 1056), (1, 2, 192, 4160), (1, 1, 1088, 1088)]
PAIRS = sorted(gfx950_space.RULE_SHAPES)


def _inputs(b, h, sq, sk, d, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(b, h, s, d, generator=g).half() for s in (sq, sk, sk)]


@pytest.mark.parametrize("d", [p[0] for p in PAIRS])
@pytest.mark.parametrize("causal", [False, True])
def test_every_rule_shape_at_the_edges_of_its_tiles(d, causal):
    for i, (b, h, sq, sk) in enumerate(SHAPES):
        q, k, v = _inputs(b, h, sq, sk, d, 100 + i)
        want, want_lse = ref_op.attention_ref(q, k, v, None, causal, return_lse=True)
        qc, kc, vc = (t.cuda() for t in (q, k, v))
        for cfg in gfx950_space.rule_configs(d, d):
            print(d, causal, (b, h, sq, sk), cfg, flush=True)
            o = torch.full((b, h, sq, d), 7.0, dtype=torch.float16, device="cuda")
            lse = torch.full((b, h, sq), 7.0, device="cuda")
            Runtime(ARCH, cfg).apply([qc, kc, vc, o], softmax_scale=1 / math.sqrt(d), causal=causal, lse=lse)
            torch.cuda.synchronize()
            assert (o.float().cpu() - want).abs().max().item() <= 2e-3
            seen = torch.isfinite(want_lse)                      # rows that see no key: -inf here, output zero
            assert torch.equal(torch.isfinite(lse.cpu()), seen)
            assert (lse.cpu() - want_lse)[seen].abs().max().item() <= 1e-3


@pytest.mark.parametrize("d", sorted(p[0] for p in gfx950_space.FEW_BLOCKS))
@pytest.mark.parametrize("causal", [False, True])
def test_waves_that_share_their_rows(d, causal):
    """Units of a kv tile that a wave of the group does not have, see or is alone with; rows that see no key; an infinite value."""
    for i, (b, h, sq, sk) in enumerate(SHAPES):
        q, k, v = _inputs(b, h, sq, sk, d, 130 + i)
        want, want_lse = ref_op.attention_ref(q, k, v, None, causal, return_lse=True)
        if not causal:
            v[0, 0, sk - 1, 5] = float("inf")
        qc, kc, vc = (t.cuda() for t in (q, k, v))
        for cfg in gfx950_space.few_blocks_configs(d, d):
            print(d, causal, (b, h, sq, sk), cfg, flush=True)
            o = torch.full((b, h, sq, d), 7.0, dtype=torch.float16, device="cuda")
            lse = torch.full((b, h, sq), 7.0, device="cuda")
            Runtime(ARCH, cfg).apply([qc, kc, vc, o], softmax_scale=1 / math.sqrt(d), causal=causal, lse=lse)
            torch.cuda.synchronize()
            got, seen = o.float().cpu(), torch.isfinite(want_lse)
            if not causal:
                assert (got[0, 0, :, 5] == float("inf")).all()
                got[0, 0, :, 5] = want[0, 0, :, 5]
            assert (got - want).abs().max().item() <= 2e-3
            assert torch.equal(torch.isfinite(lse.cpu()), seen)
            assert (lse.cpu() - want_lse)[seen].abs().max().item() <= 1e-3


@pytest.mark.parametrize("b,h,sq,sk,causal", [(3, 5, 1088, 1088, True), (2, 3, 192, 4160, True), (1, 4, 64, 8192, False), (2, 3, 96, 96, False)])
def test_the_operator_takes_them_and_its_calls_agree(b, h, sq, sk, causal):
    q, k, v = (t.cuda() for t in _inputs(b, h, sq, sk, 128, 7))
    o = aat.flash_attn_func(q, k, v, ARCH, causal)
    assert torch.equal(o, aat.flash_attn_func(q, k, v, ARCH, causal))
    assert (o.float().cpu() - ref_op.attention_ref(q.cpu(), k.cpu(), v.cpu(), None, causal)).abs().max().item() <= 2e-3


def test_a_split_call_replays_from_a_captured_graph():
    q, k, v = (t.cuda() for t in _inputs(1, 2, 192, 4160, 128, 3))
    cfg = gfx950_space.rule_forward_config(128, 128, ARCH, 1, 2, 192, 4160, True)
    assert gfx950_space.kv_parts(cfg, ARCH, 1, 2, 192, 4160, True) > 1
    rt, o = Runtime(ARCH, cfg), torch.empty_like(q)
    ws = torch.empty(rt.workspace_size(1, 2, 192, 4160), dtype=torch.uint8, device="cuda")
    rt.apply([q, k, v, o], causal=True, workspace=ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rt.apply([q, k, v, o], causal=True, workspace=ws)
    for seed in (4, 5, 6):
        for t, new in zip((q, k, v), _inputs(1, 2, 192, 4160, 128, seed)):
            t.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        eager = torch.empty_like(o)
        rt.apply([q, k, v, eager], causal=True)
        torch.cuda.synchronize()
        assert torch.equal(o, eager)


@pytest.mark.parametrize("d", [p[0] for p in PAIRS])
@pytest.mark.parametrize("sq,sk", [(96, 160), (64, 1056)])
def test_an_infinite_value_in_the_last_partial_tile_stays_an_infinity(d, sq, sk):
    """The kv rows a tile does not have are copies of its first 32: their P is zero, and 0 * inf must not reach the output."""
    q, k, v = _inputs(1, 2, sq, sk, d, 40)
    v[..., 5] = 0
    want = ref_op.attention_ref(q, k, v)
    v[:, :, sk - 31, 5] = float("inf")
    for cfg in gfx950_space.rule_configs(d, d):
        print(d, (sq, sk), cfg, flush=True)
        o = torch.full((1, 2, sq, d), 7.0, dtype=torch.float16, device="cuda")
        Runtime(ARCH, cfg).apply([q.cuda(), k.cuda(), v.cuda(), o], softmax_scale=1 / math.sqrt(d))
        o = o.float().cpu()
        assert (o[..., 5] == float("inf")).all(), cfg
        o[..., 5] = 0
        assert (o - want).abs().max().item() <= 2e-3, cfg


@pytest.mark.parametrize("sk", [192, 224])
def test_a_fixed_kv_split_that_does_not_divide_the_tiles_runs_with_and_without_room(sk):
    q, k, v = _inputs(1, 2, 128, sk, 128, 77)
    want, want_lse = ref_op.attention_ref(q, k, v, return_lse=True)
    cfg = AttnConfig(128, 64, 128, 128, 128, 64, 2, 2, 256, True, waves_per_eu=2, kv_splits=4).set_fuse_type("register")
    rt = Runtime(ARCH, cfg)
    lib = library.load(rt._path(), "attn")
    qc, kc, vc = (t.cuda() for t in (q, k, v))
    room = torch.empty(rt.workspace_size(1, 2, 128, sk), dtype=torch.uint8, device="cuda")
    for ws, nbytes in ((None, 0), (room.data_ptr(), room.numel() - 1), (room.data_ptr(), room.numel())):
        o, lse = torch.full((1, 2, 128, 128), 7.0, dtype=torch.float16, device="cuda"), torch.full((1, 2, 128), 7.0, device="cuda")
        torch.cuda.synchronize()
        rc = lib.kernel_entry_lse(*[ctypes.c_void_p(t.data_ptr()) for t in (qc, kc, vc, o, lse)], 1, 2, 128, sk, ctypes.c_float(128 ** -0.5), 0,
                                  ctypes.c_void_p(ws), ctypes.c_size_t(nbytes), None)
        torch.cuda.synchronize()
        assert rc == 0
        assert (o.float().cpu() - want).abs().max().item() <= 2e-3 and (lse.cpu() - want_lse).abs().max().item() <= 1e-3


@pytest.mark.parametrize("sq,sk", [(96, 160), (64, 4160)])
def test_any_causal_flag_but_zero_asks_for_the_causal_walk(sq, sk):
    """The C entry takes an int; at lengths the tiles do not divide and over a kv range cut into parts too."""
    q, k, v = _inputs(1, 2, sq, sk, 128, 91)
    want = ref_op.attention_ref(q, k, v, None, True)
    for cfg in gfx950_space.rule_configs(128, 128):
        rt = Runtime(ARCH, cfg)
        lib = library.load(rt._path(), "attn")
        qc, kc, vc = (t.cuda() for t in (q, k, v))
        room = torch.empty(max(1, rt.workspace_size(1, 2, sq, sk)), dtype=torch.uint8, device="cuda")
        for causal in (1, 2, -1):
            o = torch.full((1, 2, sq, 128), 7.0, dtype=torch.float16, device="cuda")
            torch.cuda.synchronize()
            rc = lib.kernel_entry_ex(*[ctypes.c_void_p(t.data_ptr()) for t in (qc, kc, vc, o)], 1, 2, sq, sk, ctypes.c_float(128 ** -0.5), causal,
                                     ctypes.c_void_p(room.data_ptr()), ctypes.c_size_t(room.numel()), None)
            torch.cuda.synchronize()
            assert rc == 0 and (o.float().cpu() - want).abs().max().item() <= 2e-3, (cfg, causal)
