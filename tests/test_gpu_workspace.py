"""The per-stream workspace of the device-pointer entry points: it grows by allocating (never by
freeing or waiting), so kernels and captured graphs that carry an older buffer's address stay
valid; a call that would have to allocate while its stream is being captured declines and leaves
the capture intact; cwick_hip_reserve_dev sizes it up front; cwick_hip_stream_release drops it."""
import numpy as np
import pytest

from cwick_amd import synth

pytestmark = pytest.mark.gpu


def _mla_operands(torch, n_rows, seed):
    c = synth.cfg3_mla_decode(n_rows, 128, seed=seed)
    return (c, torch.from_numpy(c["rows"]).cuda(), torch.from_numpy(c["scales"]).cuda(),
            torch.from_numpy(c["q"].view(np.int16)).cuda())


def test_growth_after_capture_keeps_the_graph_valid(hip):
    import torch
    print("[case] workspace: a graph captured before the workspace grows", flush=True)
    c, rows, scales, q = _mla_operands(torch, 700, 3200)
    out = torch.empty((128, synth.VDIM), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    sp = s.cuda_stream

    def small(ptr):
        # batch 1, 700 keys: a few slices of partials
        hip.mla_decode_dev(rows, scales, 0, 0, 700, 1, None, 700, q, 128, c["scale"], out, ptr)
    with torch.cuda.stream(s):
        small(sp)
    s.synchronize()
    want = out.clone()
    held = hip.workspace_bytes_dev(sp)
    assert held > 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        small(sp)
    # a much larger shape on the same stream: the workspace has to grow
    B = 48
    c2, rows2, scales2, _ = _mla_operands(torch, 4096, 3201)
    q2 = torch.from_numpy(np.repeat(c2["q"][None], B, 0).view(np.int16)).cuda()
    out2 = torch.empty((B, 128, synth.VDIM), dtype=torch.float32, device="cuda")
    with torch.cuda.stream(s):
        hip.mla_decode_dev(rows2, scales2, 0, 0, 4096, B, None, 4096, q2, 128, c2["scale"], out2, sp)
        hip.mla_decode_dev(rows2, scales2, 0, 0, 4096, B, None, 4096, q2, 128, c2["scale"], out2, sp)
    s.synchronize()
    assert hip.workspace_bytes_dev(sp) >= held
    big = out2.clone()
    for rep in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32)), "replay %d after the growth" % rep
        # and the large shape again between the replays (its buffer is the current one)
        with torch.cuda.stream(s):
            hip.mla_decode_dev(rows2, scales2, 0, 0, 4096, B, None, 4096, q2, 128, c2["scale"], out2, sp)
        s.synchronize()
        assert torch.equal(out2.view(torch.int32), big.view(torch.int32))
    del g
    assert hip.stream_release(sp) == 1
    assert hip.workspace_bytes_dev(sp) == 0


def test_capture_declines_instead_of_allocating_and_reserve_prevents_it(hip):
    import torch
    print("[case] workspace: first call of a stream under capture, then with a reservation", flush=True)
    c, rows, scales, q = _mla_operands(torch, 5000, 3202)
    out = torch.empty((128, synth.VDIM), dtype=torch.float32, device="cuda")
    # the kernels' one-time attributes are set by an eager call on another stream
    hip.mla_decode_dev(rows, scales, 0, 0, 5000, 1, None, 5000, q, 128, c["scale"], out, None)
    torch.cuda.synchronize()
    want = out.clone()
    s = torch.cuda.Stream()
    sp = s.cuda_stream
    assert hip.workspace_bytes_dev(sp) == 0
    marker = torch.zeros(4, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        marker.add_(1.0)                                  # the capture holds something of its own
        rc = hip.mla_decode_dev(rows, scales, 0, 0, 5000, 1, None, 5000, q, 128, c["scale"], out, sp, raw=True)
        why = hip.last_error()
    assert rc == 0 and "captured" in why, why
    assert hip.workspace_bytes_dev(sp) == 0
    g.replay()                                            # the capture survived the declined call
    torch.cuda.synchronize()
    assert float(marker[0]) == 1.0
    # with a reservation the same first call is captured and replays to the eager result
    assert hip.reserve_dev(sp, 32 << 20) == 1
    assert hip.workspace_bytes_dev(sp) >= 32 << 20
    g2 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g2, stream=s):
        hip.mla_decode_dev(rows, scales, 0, 0, 5000, 1, None, 5000, q, 128, c["scale"], out, sp)
    for rep in range(2):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g2.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32)), "replay %d" % rep
    del g, g2
    assert hip.stream_release(sp) == 1


def test_a_failed_allocation_stays_with_its_call(hip):
    """A reservation larger than the device's memory declines; the calls behind it run, whether or not they need
    workspace of their own."""
    import torch
    print("[case] workspace: a reservation of a tebibyte, then ordinary calls", flush=True)
    c = synth.cfg1_gqa_decode(500, 16, 4, 256, seed=3207)
    k, v, q = (torch.from_numpy(c[x].view(np.int16)).cuda() for x in "kvq")
    out = torch.empty((16, 256), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    for n in (100, 500):                                  # one split, then eight
        assert hip.reserve_dev(s.cuda_stream, 1 << 40, raw=True) == 0
        assert "hipMalloc" in hip.last_error()
        hip.gqa_decode_dev(k, v, n, 4, 256, q, 16, c["scale"], out, s.cuda_stream)
        s.synchronize()
        assert torch.isfinite(out).all() and hip.last_error() == ""
    assert hip.stream_release(s.cuda_stream) == 1


def _captured(torch, stream, call, out):
    """`call` as the only work of a graph captured on `stream`; the result after two replays."""
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        call(stream.cuda_stream)
    for _ in range(2):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = out.clone()
    return got


def _eager(torch, call, out):
    out.fill_(float("nan"))
    call(None)
    torch.cuda.synchronize()
    return out.clone()


def _close(got, ref, what):
    """Two plans of the same sums: fp16 or bf16 weights against other references, 2^-9 of a weight."""
    err = float((got - ref).norm() / ref.norm())
    print("[workspace] %s: rel %.2e" % (what, err), flush=True)
    assert err <= 4e-3, what


@pytest.mark.parametrize("nh,nkv,hd,first,then", [
    (64, 8, 128, 4100, 4096),      # 22 splits, then 64
    (64, 8, 128, 30000, 500),      # 32 splits, then 8 that one workgroup merges by tickets the stream has not got
    (16, 4, 256, 4096, 760),
])
def test_decode_of_fewer_keys_under_capture(hip, nh, nkv, hd, first, then):
    """A stream that has run a decode takes a shorter one under capture, which may have more splits."""
    import torch
    print("[case] workspace: gqa decode of fewer keys", first, then, flush=True)
    c = synth.cfg1_gqa_decode(first, nh, nkv, hd, seed=3203)
    k, v, q = (torch.from_numpy(c[x].view(np.int16)).cuda() for x in "kvq")
    out = torch.empty((nh, hd), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()

    def call(n):
        return lambda sp: hip.gqa_decode_dev(k, v, n, nkv, hd, q, nh, c["scale"], out, sp)
    call(first)(s.cuda_stream)
    s.synchronize()
    ref = _eager(torch, call(then), out)
    _close(_captured(torch, s, call(then), out), ref, "gqa decode")
    assert hip.stream_release(s.cuda_stream) == 1


def test_mla_decode_of_fewer_keys_under_capture(hip):
    import torch
    print("[case] workspace: mla decode of fewer keys", flush=True)
    c, rows, scales, q = _mla_operands(torch, 4097, 3204)
    out = torch.empty((128, synth.VDIM), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()

    def call(n):                                          # 4097 keys: 33 splits of two tiles; 4096: 64 of one
        return lambda sp: hip.mla_decode_dev(rows, scales, 0, 0, 4097, 1, None, n, q, 128, c["scale"], out, sp)
    call(4097)(s.cuda_stream)
    s.synchronize()
    ref = _eager(torch, call(4096), out)
    _close(_captured(torch, s, call(4096), out), ref, "mla decode")
    assert hip.stream_release(s.cuda_stream) == 1


@pytest.mark.parametrize("n,pos0", [(30, 3000), (517, 7083)])
def test_gqa_chunk_under_capture_after_a_larger_one(hip, orc, n, pos0):
    """A prompt of 4096 positions fills the chip and takes no workspace; a chunk that would be cut into slices then runs
    uncut under capture, as it does where no memory can be had."""
    import torch
    print("[case] workspace: gqa chunk under capture", n, pos0, flush=True)
    c = synth.cfg2_gqa_prefill(n, 16, 4, 256, pos0, seed=3205)
    k, v, q = (torch.from_numpy(c[x].view(np.int16)).cuda() for x in "kvq")
    big_q = torch.zeros((4096, 16, 256), dtype=torch.int16, device="cuda")
    big = torch.empty((4096, 16, 256), dtype=torch.float32, device="cuda")
    out = torch.empty((n, 16, 256), dtype=torch.float32, device="cuda")
    rows = torch.zeros((4096, 4, 256), dtype=torch.int16, device="cuda")
    s = torch.cuda.Stream()
    hip.gqa_prefill_dev(rows, rows, 0, 4096, 4, 256, big_q, 16, c["scale"], big, s.cuda_stream)
    s.synchronize()
    held = hip.workspace_bytes_dev(s.cuda_stream)

    def call(sp):
        hip.gqa_prefill_dev(k, v, pos0, n, 4, 256, q, 16, c["scale"], out, sp)
    ref = _eager(torch, call, out)
    got = _captured(torch, s, call, out)
    assert hip.workspace_bytes_dev(s.cuda_stream) == held == 0
    _close(got, ref, "gqa chunk")
    assert hip.last_error() == ""
    assert hip.stream_release(s.cuda_stream) == 1


@pytest.mark.parametrize("n,pos0,nh", [(9, 3000, 128), (5, 700, 24), (300, 700, 64)])
def test_mla_chunk_under_capture_on_a_fresh_stream(hip, n, pos0, nh):
    """The same for a chunk over the latent cache, which needs nothing of its stream when it is not cut."""
    import torch
    print("[case] workspace: mla chunk under capture", n, pos0, nh, flush=True)
    c = synth.cfg4_mla_prefill(n, pos0, nh, seed=3206)
    rows, scales = torch.from_numpy(c["rows"]).cuda(), torch.from_numpy(c["scales"]).cuda()
    q = torch.from_numpy(c["q"].view(np.int16)).cuda()
    out = torch.empty((n, nh, synth.VDIM), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()

    def call(sp):
        hip.mla_prefill_chunk_dev(rows, scales, pos0, n, q, nh, c["scale"], out, sp)
    ref = _eager(torch, call, out)
    _close(_captured(torch, s, call, out), ref, "mla chunk")
    assert hip.workspace_bytes_dev(s.cuda_stream) == 0 and hip.last_error() == ""
    assert hip.stream_release(s.cuda_stream) == 1
