"""RetNet recurrent form on the GPU, through the library's C entry points and the PyTorch wrapper, against
the oracle (oracle/ref_op.py closed form for small cases, oracle/brute.c sequential recurrence for larger
ones).  Tolerance: |err| <= 2e-5 * max|ref| -- fp32 arithmetic in a different association order than the
oracle's fp64 (the reference's own block scan reassociates too, reference recurrent.h:110-131)."""
import ctypes

import numpy as np
import pytest
import torch

import attention_autotuner_amd as aat
from attention_autotuner_amd.autotuner import codegen, library
from attention_autotuner_amd.autotuner.configs import RetRecurrentConfig
from attention_autotuner_amd.ops import retnet_recurrent
from oracle import brute, ref_op

pytestmark = pytest.mark.gpu
ARCH = aat.MI355X()
RTOL_OF_MAX = 2e-5


def _inputs(seed, b, h, kdim, vdim, seqlen, lo=0.0, hi=1.0):
    g = torch.Generator().manual_seed(seed)
    q = torch.rand(b, h, kdim, seqlen, generator=g) * 2 - 1
    k = torch.rand(b, h, kdim, seqlen, generator=g) * 2 - 1
    v = torch.rand(b, h, vdim, seqlen, generator=g) * 2 - 1
    decay = torch.rand(h, seqlen, generator=g) * (hi - lo) + lo
    return q, k, v, decay


def _close(got, ref):
    err = (got.cpu().double() - ref.double()).abs().max().item()
    scale = ref.abs().max().item()
    assert err <= RTOL_OF_MAX * scale, (err, scale)


# 64, 128 and more key dims, value dims that 128 does and does not divide, few and many chunks, an odd number of them, a single
# one; all with few blocks, so the waves of a block split the key dims
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(1, 2, 128, 128, 256), (1, 3, 64, 256, 96), (2, 1, 128, 64, 32),
                                                   (1, 2, 64, 64, 160), (2, 2, 64, 192, 64), (1, 2, 256, 64, 96),
                                                   (1, 1, 192, 128, 64)])
def test_matches_the_closed_form(b, h, kdim, vdim, seqlen):
    q, k, v, decay = _inputs(0, b, h, kdim, vdim, seqlen, 0.5, 1.0)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    _close(out, ref_op.retnet_recurrent_ref(q, k, v, decay))


# blocks whose waves split the key dims: each number of key dims (192: three waves, the first with two row groups), one chunk,
# odd and even chunk counts, grids that do and do not spread over 8 chiplets, every head against the sequential recurrence;
# at 64 key dims both sides of the line to 64-wide slices (256 and 258 slices of 32)
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(1, 1, 64, 64, 32), (1, 1, 128, 64, 32), (1, 1, 192, 64, 32), (1, 1, 256, 64, 32),
                                                   (1, 3, 64, 192, 96), (3, 1, 128, 320, 160), (1, 3, 192, 192, 128),
                                                   (2, 4, 256, 128, 96), (8, 8, 64, 128, 64), (3, 43, 64, 64, 64)])
def test_split_key_dims(b, h, kdim, vdim, seqlen):
    q, k, v, decay = _inputs(11, b, h, kdim, vdim, seqlen, -0.3, 1.2)
    decay[0, seqlen // 2] = 0.0
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(h):
        _close(out[:, head], ref[:, head])


def test_zero_negative_and_vanishing_decays():
    """Zeros cut the history, negative values flip signs, long runs of small decays drive the carried
    product out of range (the state is then rescaled): all as in the recurrence."""
    q, k, v, decay = _inputs(1, 1, 4, 64, 64, 256, -1.0, 1.0)
    decay[0, 5] = 0.0
    decay[0, 64] = 0.0
    decay[1] = 0.05                      # 0.05^32 per chunk: leaves the range at once
    decay[2] = 1.0
    decay[3, :128] = 1.5                 # growth: leaves the range upwards after three chunks
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(4):
        _close(out[:, head], ref[:, head])


def test_many_blocks_take_the_wide_value_slice_and_agree_with_the_narrow_one():
    """192 or more (batch, head, 128-dim slice) blocks launch the 128-wide kernel, fewer the 64-wide one."""
    q, k, v, decay = _inputs(2, 24, 8, 64, 128, 64, 0.9, 1.0)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    _close(out, ref)
    # 64 of the value dims: 192 slices of 64 of them fit at once (two to a compute unit), 384 slices of 32 take two rounds
    narrow = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v[:, :, :64].contiguous().cuda(), decay.cuda())
    _close(narrow, ref[:, :, :64])


# more than 128 key dims where 128-wide value slices fill the chip and the split blocks would take four rounds: passes over 128 and
# 64 key dims, the second of which adds to the first one's output
@pytest.mark.parametrize("kdim", [192, 256])
def test_passes_over_the_key_dims_add_up(kdim):
    q, k, v, decay = _inputs(12, 8, 32, kdim, 128, 64, -0.3, 1.2)
    decay[0, 40] = 0.0
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(32):
        _close(out[:, head], ref[:, head])


def test_block_kdim_limits_the_contraction():
    q, k, v, decay = _inputs(3, 1, 2, 128, 64, 128, 0.8, 1.0)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda(), block_kdim=64)
    _close(out, ref_op.retnet_recurrent_ref(q, k, v, decay, block_kdim=64))


def test_reference_signature_entry_point_and_error_codes():
    """retnet_recurrent_fwd (reference recurrent.h:427: void, null stream, no workspace argument) gives the
    same result as the extended entry point; unsupported shapes and a short workspace are refused."""
    lib = library.load_recurrent(codegen.compile_config(RetRecurrentConfig(), ARCH))
    b, h, kdim, vdim, seqlen = 1, 2, 64, 64, 128
    q, k, v, decay = [t.cuda() for t in _inputs(4, b, h, kdim, vdim, seqlen, 0.7, 1.0)]
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    out_ref_sig = torch.zeros_like(v)
    torch.cuda.synchronize()
    lib.retnet_recurrent_fwd(ptr(q), ptr(k), ptr(v), ptr(decay), ptr(out_ref_sig), b, h, kdim, vdim, seqlen, kdim)
    torch.cuda.synchronize()
    out_ex = aat.retnet_recurrent_fwd(q, k, v, decay)
    assert torch.equal(out_ref_sig, out_ex)
    # a second, larger call: still within what the library's static array holds, so nothing is allocated
    q2, k2, v2, decay2 = [t.cuda() for t in _inputs(5, 1, 4, 64, 64, 256, 0.7, 1.0)]
    out2 = torch.zeros_like(v2)
    want2 = aat.retnet_recurrent_fwd(q2, k2, v2, decay2)
    torch.cuda.synchronize()
    free_before = torch.cuda.mem_get_info()[0]
    lib.retnet_recurrent_fwd(ptr(q2), ptr(k2), ptr(v2), ptr(decay2), ptr(out2), 1, 4, 64, 64, 256, 64)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free_before
    assert torch.equal(out2, want2)
    # more than 128 key dims per pass need a second output-sized buffer: the entry point allocates one and keeps it
    q3, k3, v3, decay3 = [t.cuda() for t in _inputs(6, 1, 2, 256, 64, 128, 0.7, 1.0)]
    out3 = torch.zeros_like(v3)
    lib.retnet_recurrent_fwd(ptr(q3), ptr(k3), ptr(v3), ptr(decay3), ptr(out3), 1, 2, 256, 64, 128, 256)
    torch.cuda.synchronize()
    assert torch.equal(out3, aat.retnet_recurrent_fwd(q3, k3, v3, decay3, block_kdim=256))

    need = lib.workspace_size(b, h, seqlen, seqlen)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    out = torch.empty_like(v)
    args = [ptr(q), ptr(k), ptr(v), ptr(decay), ptr(out)]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    call = lambda dims, w, nbytes: lib.retnet_recurrent_fwd_ex(*args, *dims, w, ctypes.c_size_t(nbytes), stream)
    assert call((b, h, kdim, vdim, seqlen, kdim), ptr(ws), need) == 0
    assert call((b, h, kdim, vdim, seqlen, kdim), ptr(ws), need - 1) == -3
    assert call((b, h, kdim, vdim, seqlen, kdim), ctypes.c_void_p(0), 0) == -3
    assert call((b, h, kdim, vdim, 100, kdim), ptr(ws), need) == -2         # l not a multiple of 32
    assert call((b, h, kdim, vdim, seqlen, 32), ptr(ws), need) == -2        # block_kdim
    assert call((b, h, kdim, vdim, seqlen, 128), ptr(ws), need) == -2       # block_kdim > kdim
    assert call((b, h, kdim, 32, seqlen, kdim), ptr(ws), need) == -2        # vdim
    assert call((0, h, kdim, vdim, seqlen, kdim), ptr(ws), need) == -2
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="unsupported shape"):
        aat.retnet_recurrent_fwd(q[..., :100].contiguous(), k[..., :100].contiguous(), v[..., :100].contiguous(),
                                 decay[:, :100].contiguous())


def test_deterministic_and_profile_entry():
    q, k, v, decay = [t.cuda() for t in _inputs(6, 2, 2, 128, 128, 192, 0.9, 1.0)]
    a = aat.retnet_recurrent_fwd(q, k, v, decay)
    b = aat.retnet_recurrent_fwd(q, k, v, decay)
    assert torch.equal(a, b)
    lib = library.load_recurrent(codegen.compile_config(RetRecurrentConfig(), ARCH))
    ws = torch.empty(retnet_recurrent.workspace_size(2, 192), dtype=torch.uint8, device="cuda")
    out = torch.empty_like(v)
    ms = lib.retnet_recurrent_profile(*[ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, decay, out)], 2, 2, 128, 128, 192, 128,
                                      ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(ws.numel()),
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert 0 < ms < 50
    assert torch.equal(out, a)


def test_full_size_through_size_independent_properties():
    """Benchmark shape (8, 32, 128, 128, 2048): too large for the oracle, so linearity in v, a decay-zero
    closed form and one (batch, head) slice against the sequential recurrence."""
    b, h, kdim, vdim, seqlen = 8, 32, 128, 128, 2048
    g = torch.Generator(device="cuda").manual_seed(7)
    q = torch.rand(b, h, kdim, seqlen, generator=g, device="cuda") * 2 - 1
    k = torch.rand(b, h, kdim, seqlen, generator=g, device="cuda") * 2 - 1
    v = torch.rand(b, h, vdim, seqlen, generator=g, device="cuda") * 2 - 1
    v2 = torch.rand(b, h, vdim, seqlen, generator=g, device="cuda") * 2 - 1
    gamma = 1.0 - 2.0 ** (-5.0 - torch.arange(h, dtype=torch.float32, device="cuda"))
    decay = gamma.unsqueeze(1).expand(h, seqlen).contiguous()
    o1 = aat.retnet_recurrent_fwd(q, k, v, decay)
    o2 = aat.retnet_recurrent_fwd(q, k, v2, decay)
    o12 = aat.retnet_recurrent_fwd(q, k, v + v2, decay)
    scale = o12.abs().max().item()
    assert (o12 - (o1 + o2)).abs().max().item() <= 1e-5 * scale
    o0 = aat.retnet_recurrent_fwd(q, k, v, torch.zeros_like(decay))
    expect0 = (q * k).sum(dim=2, keepdim=True) * v
    assert (o0 - expect0).abs().max().item() <= 1e-5 * expect0.abs().max().item()
    sl = (slice(3, 4), slice(17, 18))
    ref = brute.retnet_recurrent(q[sl].cpu().numpy(), k[sl].cpu().numpy(), v[sl].cpu().numpy(), decay[17:18].cpu().numpy())
    _close(o1[sl], torch.from_numpy(ref))


def test_long_sequence_and_side_stream():
    """128 chunks per head (the carried product leaves its range several times), launched on a side stream."""
    q, k, v, decay = _inputs(8, 1, 2, 64, 64, 4096, 0.6, 1.0)
    side = torch.cuda.Stream()
    qc, kc, vc, dc = q.cuda(), k.cuda(), v.cuda(), decay.cuda()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = aat.retnet_recurrent_fwd(qc, kc, vc, dc)
    side.synchronize()
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    _close(out, ref)


# one block of factors per head and a second one with a single chunk; 300 chunks: several per wave, a short last block, two
# dozen rescales; decays that do not start on 16 bytes
@pytest.mark.parametrize("seqlen", [16 * 32, 17 * 32, 300 * 32])
def test_decay_factors_over_blocks(seqlen):
    q, k, v, decay = _inputs(12, 1, 2, 64, 64, seqlen, 0.8, 1.0)
    decay[1, ::97] = -1.5
    decay[1, seqlen - 40] = 0.0
    shifted = torch.zeros(2 * seqlen + 1, device="cuda")[1:].view(2, seqlen).copy_(decay)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), shifted)
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(2):
        _close(out[:, head], ref[:, head])


# beyond 128 key dims the launch that makes P makes the records too, in blocks of four waves: a single part, a second one with a
# single chunk, several chunks per wave in as many parts as a launch has and a short last part
@pytest.mark.parametrize("kdim,seqlen", [(192, 4 * 32), (256, 5 * 32), (256, 131 * 32), (192, 259 * 32)])
def test_decay_factors_beside_the_products_of_q_and_k(kdim, seqlen):
    q, k, v, decay = _inputs(13, 2, 2, kdim, 64, seqlen, 0.8, 1.0)
    decay[1, ::97] = -1.5
    decay[1, seqlen - 40] = 0.0
    shifted = torch.zeros(2 * seqlen + 1, device="cuda")[1:].view(2, seqlen).copy_(decay)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), shifted)
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(2):
        _close(out[:, head], ref[:, head])


def test_graph_capture_replays():
    """The extended entry point allocates nothing and launches two kernels: a captured graph of it replays
    correctly with eager work and synchronisations in between, and follows new inputs written in place."""
    b, h, kdim, vdim, seqlen = 2, 2, 128, 64, 256
    q, k, v, decay = [t.cuda() for t in _inputs(9, b, h, kdim, vdim, seqlen, 0.8, 1.0)]
    out = torch.empty_like(v)
    ws = torch.empty(retnet_recurrent.workspace_size(h, seqlen, batch=b, kdim=kdim, vdim=vdim), dtype=torch.uint8, device="cuda")
    eager = aat.retnet_recurrent_fwd(q, k, v, decay)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        aat.retnet_recurrent_fwd(q, k, v, decay, out=out, workspace=ws)          # warm-up outside the capture
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        aat.retnet_recurrent_fwd(q, k, v, decay, out=out, workspace=ws)
    for rep in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), rep
        _ = (q * 2).sum().item()                                              # eager work between replays
    q2, k2, v2, decay2 = [t.cuda() for t in _inputs(10, b, h, kdim, vdim, seqlen, 0.8, 1.0)]
    q.copy_(q2), k.copy_(k2), v.copy_(v2), decay.copy_(decay2)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, aat.retnet_recurrent_fwd(q2, k2, v2, decay2))


# blocks of 128 and of 64 value dims (192 of them, so the split kernel stays away): one chunk, two, an odd number; every head
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(8, 24, 128, 128, 32), (8, 24, 64, 128, 64), (8, 24, 64, 64, 96),
                                                   (4, 24, 128, 256, 160), (8, 24, 64, 64, 32), (8, 24, 64, 128, 96)])
def test_blocks_that_split_the_value_dims(b, h, kdim, vdim, seqlen):
    q, k, v, decay = _inputs(21, b, h, kdim, vdim, seqlen, -0.3, 1.2)
    decay[0, seqlen // 2] = 0.0
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(h):
        _close(out[:, head], ref[:, head])


# fp32 products in three bf16 parts: Q, K, V, S^T, the State or outputs at the low end of fp32 (2e-37 / 2^24 lies below the smallest bf16
# subnormal, 9e-41: parts of a value that is not scaled are off by 2e-4 of it), at the high end (the State is held divided by lambda, 2^-40 at the
# least: 3e26 is as far as fp32 goes), and magnitudes that differ from key dim to key dim.
# Blocks of 128 and 64 value dims, and those with operands made ahead
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(8, 24, 128, 128, 64), (8, 24, 64, 64, 64), (1, 2, 64, 64, 512), (1, 2, 128, 64, 512),
                                                   (1, 2, 192, 64, 512), (1, 2, 256, 64, 512)])
@pytest.mark.parametrize("k_scale,q_scale,v_scale,spread", [(1e-30, 1e20, 1.0, 0.0), (2e-37, 1e26, 1.0, 0.0), (1e26, 2e-37, 1.0, 0.0), (1e20, 1.0, 2e-37, 0.0),
                                                            (1e-19, 2e-18, 1e25, 0.0), (1e-19, 1e26, 2e-18, 0.0), (1e-15, 1e-15, 2e-7, 0.0),
                                                            (1e24, 1e-20, 1.0, 0.0), (1.0, 1.0, 1.0, 12.0)])
def test_products_in_parts_keep_the_range_of_fp32(b, h, kdim, vdim, seqlen, k_scale, q_scale, v_scale, spread):
    q, k, v, decay = _inputs(22, b, h, kdim, vdim, seqlen, 0.9, 1.0)
    per_dim = 10.0 ** ((torch.arange(kdim) * 37 % kdim / (kdim - 1.0) - 0.5) * spread).view(1, 1, kdim, 1)
    q, k, v = (q * q_scale * per_dim).float(), (k * k_scale / per_dim).float(), (v * v_scale).float()
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(h):
        _close(out[:, head], ref[:, head])


# Decay factors far from one, next to values at the other end: w / lambda' of 2^-36 beside a K of 1e-28, w of 1e-30 beside a K of 1e-12, p_n of
# 1e-30 beside a Q of 1e-12.  Their products leave fp32 (or three bf16 parts) and what they are for does not: the factors go with V and with the sum.
# Blocks of 128 and 64 value dims, and those with operands made ahead.
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(8, 24, 128, 128, 64), (8, 24, 64, 128, 64), (8, 24, 64, 64, 64), (1, 2, 64, 64, 512),
                                                   (1, 2, 128, 64, 512), (1, 2, 192, 64, 512), (1, 2, 256, 64, 512)])
@pytest.mark.parametrize("where,factor,k_scale,q_scale,v_scale", [(0, 2.0 ** 36, 1e-28, 1e16, 1e12), (16, 1e-30, 1e-12, 1e12, 1e20),
                                                                  (32, 1e-30, 1e14, 1e-12, 1e12)])
def test_decay_factors_beside_values_at_the_other_end(b, h, kdim, vdim, seqlen, where, factor, k_scale, q_scale, v_scale):
    q, k, v, decay = _inputs(28, b, h, kdim, vdim, seqlen, 1.0, 1.0)
    q, k, v = (q * q_scale).float(), (k * k_scale).float(), (v * v_scale).float()
    decay[:, where] = factor
    if factor < 1:
        v[..., where:] = 0.0                              # what came before is all there is behind the factor
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(h):
        _close(out[:, head, :, where:], ref[:, head, :, where:])


# An infinity or a NaN takes its (batch, head, value slice) from the chunk it lies in on, and nothing else: the rest is as without it,
# bit for bit in other blocks, within the bound in the chunks before
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("kdim,vdim", [(128, 128), (64, 128), (64, 64)])
def test_values_that_are_not_finite(value, which, kdim, vdim):
    b, h, seqlen, pos = 8, 24, 128, 70
    q, k, v, decay = _inputs(23, b, h, kdim, vdim, seqlen, 0.9, 1.0)
    clean = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    bad = dict(q=q, k=k, v=v)
    bad[which] = bad[which].clone()
    bad[which][3, 5, 7, pos] = value
    out = aat.retnet_recurrent_fwd(bad["q"].cuda(), bad["k"].cuda(), bad["v"].cuda(), decay.cuda())
    rows = slice(7, 8) if which == "v" else slice(None)
    last = pos + 1 if which == "q" else seqlen
    assert not torch.isfinite(out[3, 5, rows, pos:last]).any()
    _close(out[3, 5, :, :64], clean[3, 5, :, :64].cpu())
    if which == "q":
        _close(out[3, 5, :, 96:], clean[3, 5, :, 96:].cpu())
    out[3, 5], clean[3, 5] = 0.0, 0.0
    assert torch.equal(out, clean)


# 3.4e38 rounds to an infinity in bf16, but is none: with small partners every product and sum stays finite
@pytest.mark.parametrize("which", ["q", "k"])
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(8, 24, 128, 128, 128), (8, 24, 64, 128, 128), (8, 24, 64, 64, 128), (4, 6, 64, 64, 512),
                                                   (4, 6, 128, 64, 512), (4, 6, 192, 64, 512), (4, 6, 256, 64, 512)])
def test_values_beyond_the_largest_of_bf16(which, b, h, kdim, vdim, seqlen):
    pos = 70
    q, k, v, decay = _inputs(24, b, h, kdim, vdim, seqlen, 0.9, 1.0)
    x = {n: t if n == which else t * 1e-6 for n, t in (("q", q), ("k", k), ("v", v))}
    x[which][3, 5, 7, pos] = 3.4e38
    out = aat.retnet_recurrent_fwd(x["q"].cuda(), x["k"].cuda(), x["v"].cuda(), decay.cuda())
    ref = torch.from_numpy(brute.retnet_recurrent(x["q"].numpy(), x["k"].numpy(), x["v"].numpy(), decay.numpy()))
    assert torch.isfinite(out).all()
    _close(out[3, 5], ref[3, 5])
    _close(out[3, 4], ref[3, 4])


def _room(b, h, kdim, vdim, seqlen, most=1 << 40):
    lib = library.load_recurrent(codegen.compile_config(RetRecurrentConfig(), ARCH))
    need = lib.retnet_recurrent_workspace_size(b, h, kdim, vdim, seqlen, kdim)
    return need, lib.retnet_recurrent_room(b, h, kdim, vdim, seqlen, kdim, ctypes.c_size_t(most))


# operands of K and Q made ahead of the scan: every number of key dims (192: three waves, the first with two row groups), the fewest chunks that
# take it, odd and even counts, decays that are 0, negative and that drive the carried product out of its range, against the recurrence
@pytest.mark.parametrize("b,h,kdim,vdim,seqlen", [(1, 2, 64, 64, 512), (1, 3, 64, 192, 544), (2, 2, 128, 64, 576), (1, 2, 128, 320, 544),
                                                   (1, 2, 192, 64, 544), (2, 1, 192, 128, 512), (1, 2, 256, 64, 512), (1, 3, 256, 128, 544)])
def test_operands_made_ahead(b, h, kdim, vdim, seqlen):
    need, room = _room(b, h, kdim, vdim, seqlen)
    assert room > need                                    # the call has the room and takes it
    q, k, v, decay = _inputs(25, b, h, kdim, vdim, seqlen, 0.6, 1.05)
    decay[0, seqlen // 2] = 0.0
    decay[0, 1::97] = -0.9
    decay[-1, 64:128] = 0.05                              # leaves the range at once
    shifted = torch.zeros(h * seqlen + 1, device="cuda")[1:].view(h, seqlen).copy_(decay)
    out = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), shifted)
    ref = torch.from_numpy(brute.retnet_recurrent(q.numpy(), k.numpy(), v.numpy(), decay.numpy()))
    for head in range(h):
        _close(out[:, head], ref[:, head])
    # without the room, and one byte short of it, the split kernel runs; the results differ by the order of additions
    for nbytes in (need, room - 1):
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        held = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda(), workspace=ws)
        for head in range(h):
            _close(held[:, head], ref[:, head])


def test_the_room_is_offered_where_it_pays_and_not_beyond_what_is_asked_for():
    for dims in [(2, 8, 256, 512, 1056), (1, 4, 64, 64, 512), (5, 6, 64, 512, 512)]:
        need, room = _room(*dims)
        assert room > need and _room(*dims, most=room) == (need, room) and _room(*dims, most=room - 1) == (need, need)
    for dims in [(8, 32, 128, 128, 2048), (1, 4, 64, 64, 480), (8, 16, 256, 64, 1024)]:
        need, room = _room(*dims)
        assert room == need
    assert _room(1, 4, 64, 64, 500) == (0, 0)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("which", ["q", "k", "v"])
@pytest.mark.parametrize("kdim", [64, 128, 192, 256])
def test_values_that_are_not_finite_with_operands_made_ahead(value, which, kdim):
    b, h, vdim, seqlen, pos = 2, 2, 64, 544, 262
    assert _room(b, h, kdim, vdim, seqlen)[1] > _room(b, h, kdim, vdim, seqlen)[0]
    q, k, v, decay = _inputs(26, b, h, kdim, vdim, seqlen, 0.9, 1.0)
    clean = aat.retnet_recurrent_fwd(q.cuda(), k.cuda(), v.cuda(), decay.cuda())
    bad = dict(q=q, k=k, v=v)
    bad[which] = bad[which].clone()
    bad[which][1, 1, 7, pos] = value
    out = aat.retnet_recurrent_fwd(bad["q"].cuda(), bad["k"].cuda(), bad["v"].cuda(), decay.cuda())
    rows = slice(7, 8) if which == "v" else slice(None)
    last = pos + 1 if which == "q" else seqlen
    assert not torch.isfinite(out[1, 1, rows, pos:last]).any()
    _close(out[1, 1, :, :256], clean[1, 1, :, :256].cpu())
    if which == "q":
        _close(out[1, 1, :, 288:], clean[1, 1, :, 288:].cpu())
    out[1, 1], clean[1, 1] = 0.0, 0.0
    assert torch.equal(out, clean)


def test_operands_made_ahead_keep_the_range_of_fp32_and_replay():
    """Magnitudes over 12 decades along the key dims; then the call in a graph, replayed with eager work in between."""
    b, h, kdim, vdim, seqlen = 1, 2, 128, 64, 512
    q, k, v, decay = _inputs(27, b, h, kdim, vdim, seqlen, 0.9, 1.0)
    per_dim = 10.0 ** ((torch.arange(kdim) * 37 % kdim / (kdim - 1.0) - 0.5) * 12).view(1, 1, kdim, 1)
    q, k, v, decay = (q * per_dim).float().cuda(), (k / per_dim).float().cuda(), v.cuda(), decay.cuda()
    out = aat.retnet_recurrent_fwd(q, k, v, decay)
    ref = torch.from_numpy(brute.retnet_recurrent(*(t.cpu().numpy() for t in (q, k, v, decay))))
    for head in range(h):
        _close(out[:, head], ref[:, head])
    ws = torch.empty(_room(b, h, kdim, vdim, seqlen)[1], dtype=torch.uint8, device="cuda")
    got = torch.empty_like(v)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        aat.retnet_recurrent_fwd(q, k, v, decay, out=got, workspace=ws)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        aat.retnet_recurrent_fwd(q, k, v, decay, out=got, workspace=ws)
    for _ in range(3):
        got.zero_(), ws.fill_(255)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, out)
        _ = (q * 2).sum().item()


def test_without_memory_for_operands_made_ahead_a_call_takes_the_least_it_needs(monkeypatch):
    dims = b, h, kdim, vdim, seqlen = 1, 2, 128, 64, 512
    need, room = _room(*dims)
    assert room > need
    q, k, v, decay = (t.cuda() for t in _inputs(29, *dims, 0.9, 1.0))
    want = aat.retnet_recurrent_fwd(q, k, v, decay, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"))
    empty, asked = torch.empty, []

    def no_memory(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            asked.append(size[0])
            if size[0] > need:
                raise torch.cuda.OutOfMemoryError("no room")
        return empty(*size, **kw)
    monkeypatch.setattr(torch, "empty", no_memory)
    assert torch.equal(aat.retnet_recurrent_fwd(q, k, v, decay), want) and asked == [room, need]
