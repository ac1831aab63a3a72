"""RetNet with decay rates where the longest blocks are walked by several workgroups: lengths at which the library cuts, whole and
with a part of a last block, either side the longer one, against the oracle's exact form under the rounded-operand rule of
oracle/tolerance.py; the order in which the parts arrive must not show."""
import pytest
import torch

import attention_autotuner_amd as aat
from attention_autotuner_amd.autotuner import Runtime, gfx950_space, library, prebuilt, prebuilt_extra, runtime
from oracle import ref_op, tolerance
from test_retnet_ragged_gpu import _check, _problem

pytestmark = pytest.mark.gpu
ARCH = aat.MI355X()
SHAPES = [(1, 2, 1088, 1088), (1, 3, 1024, 1344), (2, 1, 1344, 1024)]


def _configs(dqk, dv, problem):
    b, h, sq, sk = problem
    return (gfx950_space.rule_ret_config("ret", dqk, dv, b, h, sq, sk, True), gfx950_space.rule_ret_config("ret_bwd", dqk, dv, b, h, sq, sk, True))


def _cuts(rt, problem):
    lib = library.load(rt._path(), rt.config.operation)
    return lib.decay_workspace_size(*problem, 1 << 40) > lib.workspace_size(*problem)


@pytest.mark.parametrize("dqk,dv", sorted(gfx950_space.RET_RULE))
def test_blocks_in_parts_against_the_oracle(dqk, dv):
    cut = 0
    for i, problem in enumerate(SHAPES):
        fwd, bwd = _configs(dqk, dv, problem)
        cut += sum(_cuts(Runtime(ARCH, cfg), problem) for cfg in (fwd, bwd))
        _check(problem, dqk, dv, "decay", 900 + i, [fwd], [bwd])
    assert cut >= 2 or dqk == 64, "nothing was cut"          # a walk of 17 tiles of 64 columns is not worth an exchange


# every RetNet shape that is built, the tuned ones among them: 2112 and 1984 rows leave half a block of 128, 2112 a quarter of one of 256
BUILT = [c for c in prebuilt.shipping_set(ARCH, prebuilt_extra.parity_configs()) if c.operation in ("ret", "ret_bwd")]


@pytest.mark.parametrize("problem", [(1, 2, 2112, 1984), (2, 1, 1984, 2112), (1, 1, 4096, 4096)])
@pytest.mark.parametrize("dqk,dv", sorted({(c.Kd, c.D) for c in BUILT}))
def test_every_shape_that_is_cut_against_the_oracle(dqk, dv, problem):
    cut = [c for c in BUILT if (c.Kd, c.D) == (dqk, dv) and not (problem[2] % c.Bc or problem[3] % c.Bc) and _cuts(Runtime(ARCH, c), problem)]
    if not cut:
        pytest.skip("no shape of these head sizes is cut at these lengths")
    _check(problem, dqk, dv, "decay", 950 + problem[2] % 7, [c for c in cut if c.operation == "ret"], [c for c in cut if c.operation == "ret_bwd"])


@pytest.mark.parametrize("op,dqk,dv,br", [("ret", 256, 512, 128), ("ret", 256, 512, 64), ("ret_bwd", 256, 512, 128), ("ret_bwd", 256, 256, 128),
                                          ("ret_bwd", 64, 64, 64)])
@pytest.mark.parametrize("sq,sk", [(2112, 2112), (2112, 1984)])
def test_the_library_cuts_with_the_room_it_asks_for_and_with_no_byte_less(op, dqk, dv, br, sq, sk):
    """The arrival counts in the workspace say which launches were cut: all of them, blocks that are partial among them."""
    problem = b, h, _, _ = 1, 2, sq, sk
    cfg = next(c for c in gfx950_space.rule_ret_configs(op, dqk, dv) if c.Br == br)
    rt = Runtime(ARCH, cfg)
    lib = library.load(rt._path(), op)
    q, k, v, do, _, lg = (t.cuda() for t in _problem(b, h, sq, sk, dqk, dv, "decay", 43))
    r = torch.full((b, h, sq), 3.0, device="cuda")
    out = [torch.empty_like(do)] if op == "ret" else [torch.empty_like(t) for t in (q, k, v)]
    arrays = [q, k, v, lg, out[0], r] if op == "ret" else [q, k, v, lg, do, r, *out]
    base, size = lib.workspace_size(*problem), lib.decay_workspace_size(*problem, 1 << 40)
    buf = torch.full((size + 4096,), 0x5a, dtype=torch.uint8, device="cuda")
    rt.apply(arrays, decay=True, workspace=buf[:size - 1])
    assert bool((buf[base:] == 0x5a).all())
    whole = [t.clone() for t in out]
    rt.apply(arrays, decay=True, workspace=buf[:size])
    torch.cuda.synchronize()
    assert bool((buf[size:] == 0x5a).all())
    launches = 1 if op == "ret" else 3
    counts = buf[base:base + 256 * (launches + 1)].view(torch.int32).cpu().view(launches + 1, 64)
    for launch in range(launches):
        words = counts[launch].tolist()
        arrived = words.count(words[0])
        assert 2 <= words[0] <= 4 and arrived % h == 0 and words[:arrived] == [words[0]] * arrived, launch
        assert set(words[arrived:]) <= {0, 0x5a5a5a5a}, launch
    for cut, one in zip(out, whole):
        assert not torch.equal(cut, one) or dqk == 64                     # other sums of fp32 values
        assert ((cut.float() - one.float()).norm() / one.float().norm()).item() < 1e-3


@pytest.mark.parametrize("dqk,dv", [(64, 64), (128, 128), (256, 512)])
def test_parts_give_the_same_bits_every_time(dqk, dv):
    problem = b, h, sq, sk = 1, 4, 2112, 2112
    q, k, v, do, _, lg = (t.cuda() for t in _problem(1, 4, sq, sk, dqk, dv, "decay", 31))
    fwd, bwd = (Runtime(ARCH, c) for c in _configs(dqk, dv, problem))
    assert _cuts(bwd, problem)
    first = None
    for _ in range(5):
        o, r = torch.full_like(do, 7.0), torch.full((b, h, sq), 7.0, device="cuda")
        grads = [torch.full_like(t, 7.0) for t in (q, k, v)]
        fwd.apply([q, k, v, lg, o, r], decay=True)
        bwd.apply([q, k, v, lg, do, r, *grads], decay=True)
        torch.cuda.synchronize()
        outs = [o, r, *grads]
        first = first or outs
        assert all(torch.equal(a, x) for a, x in zip(first, outs))


def test_a_captured_call_replays_its_parts():
    """The counts are cleared and the orders handed out by the call itself: replays between eager work give the same bits."""
    problem = b, h, sq, sk = 1, 2, 2112, 2112
    q, k, v, do, _, lg = (t.cuda() for t in _problem(b, h, sq, sk, 256, 512, "decay", 47))
    fwd, bwd = (Runtime(ARCH, c) for c in _configs(256, 512, problem))
    assert _cuts(fwd, problem) and _cuts(bwd, problem)
    o, r = torch.empty_like(do), torch.empty(b, h, sq, device="cuda")
    grads = [torch.empty_like(t) for t in (q, k, v)]

    def call():
        fwd.apply([q, k, v, lg, o, r], decay=True)
        bwd.apply([q, k, v, lg, do, r, *grads], decay=True)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seed in range(4):
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(seed)).half())
        call()
        torch.cuda.synchronize()
        want = [t.clone() for t in (o, r, *grads)]
        for t in (o, r, *grads):
            t.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, x) for a, x in zip(want, (o, r, *grads))), seed


@pytest.mark.parametrize("op", ["ret", "ret_bwd"])
def test_a_workspace_of_workspace_size_bytes_is_used_as_it_is(op):
    """... with nothing allocated beside it, every block walked in one piece, and the bytes behind it left alone; results against
    the oracle's.  So is a larger one that starts off a boundary of eight bytes; any other one that has room for the parts is used
    for them too."""
    problem = b, h, sq, sk = 1, 2, 1088, 1088
    dqk, dv = 256, 512
    q, k, v, do, mask, lg = _problem(b, h, sq, sk, dqk, dv, "decay", 37)
    rt = Runtime(ARCH, _configs(dqk, dv, problem)[op == "ret_bwd"])
    size, guard = rt.workspace_size(*problem), 1 << 26
    qc, kc, vc, dc = (t.cuda() for t in (q, k, v, do))
    o_want, r_want = ref_op.retnet_ref(q, k, v, mask, return_r=True)
    r_want = r_want.reshape(b, h, sq)
    if op == "ret":
        s = (q.float() @ k.float().transpose(-1, -2)) * mask.float()
        want, terms = [o_want], [(s.abs() / s.abs().sum(-1, keepdim=True).clamp(min=1.0)) @ v.float().abs()]
        out, r = [torch.full_like(dc, 7.0)], torch.full((b, h, sq), 7.0, device="cuda")
        arrays = [qc, kc, vc, lg.cuda(), out[0], r]
    else:
        want, terms = ref_op.retnet_bwd_ref(q, k, v, mask, do), ref_op.retnet_bwd_rounding_bound(q, k, v, mask, do)
        out = [torch.full_like(t, 7.0) for t in (qc, kc, vc)]
        arrays = [qc, kc, vc, lg.cuda(), dc, r_want.cuda(), *out]
    room = torch.full((size + guard,), 0x5a, dtype=torch.uint8, device="cuda")
    rt.apply(arrays, decay=True, workspace=room[:size])                    # the library is loaded
    for workspace in (room[:size], room[4:], room):
        torch.cuda.synchronize()
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        rt.apply(arrays, decay=True, workspace=workspace)
        torch.cuda.synchronize()
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
        untouched = bool((room[size + 4:] == 0x5a).all())
        assert untouched == (workspace is not room)                       # the parts' counts, order and slots lie there
        for got, ref, t in zip(out, want, terms):
            ok, worst, ratio = tolerance.check_rounded_operand(got, ref, t)
            assert ok, (worst, ratio)
            got.fill_(7.0)


def test_without_memory_for_the_parts_blocks_are_walked_in_one_piece(monkeypatch):
    problem = b, h, sq, sk = 1, 2, 1088, 1088
    q, k, v, _, _, lg = (t.cuda() for t in _problem(b, h, sq, sk, 256, 512, "decay", 41))
    rt = Runtime(ARCH, _configs(256, 512, problem)[0])
    assert _cuts(rt, problem)
    o, r = torch.empty(b, h, sq, 512, device="cuda", dtype=torch.float16), torch.empty(b, h, sq, device="cuda")
    rt.apply([q, k, v, lg, o, r], decay=True, workspace=torch.empty(rt.workspace_size(*problem), dtype=torch.uint8, device="cuda"))
    whole, grown, asked = o.clone(), runtime._grown, []

    def no_memory(workspace, need, device, keep):
        asked.append(need)
        if need > rt.workspace_size(*problem):
            raise torch.cuda.OutOfMemoryError("no room")
        return grown(workspace, need, device, keep)
    monkeypatch.setattr(runtime, "_grown", no_memory)
    o.fill_(7.0)
    rt.apply([q, k, v, lg, o, r], decay=True)
    torch.cuda.synchronize()
    assert torch.equal(o, whole) and asked[0] > asked[1] == rt.workspace_size(*problem)
