"""GPU: layers committed on one context from two streams at once, back to back.

The reference runs its GPU tests under serial and concurrent dispatch (cmake/metal/tests.cmake:
330-339). Here two full prefill layers (with a shared expert, so the context's second stream is
used too) and two decode layers, each pair on different weights, are committed alternately on
two streams without a wait in between, often enough to cycle the context's 64-slot ring of
expert address tables several times. Every output must equal the same layer run alone, bit for
bit: a ring slot handed out while a launch could still read it, or a table copied for the wrong
layer, would put another layer's experts into the products.
"""
import numpy as np
import pytest

import gpu_util as gu

pytestmark = pytest.mark.gpu


def _prefill(layer, moe, seed):
    return layer.LayerConfig("concurrent", 256, 512, 64, 4, 256, 256, moe.Q4_K, moe.Q8_0, moe.F16, seed=seed)


def _decode(layer, moe, seed):
    return layer.LayerConfig("concurrent_decode", 2, 512, 64, 8, 256, 256, moe.Q4_K, moe.Q8_0, moe.F16, seed=seed)


def _out(ws):
    return gu.host(ws.out, np.float32).copy()


def test_two_streams_alternating_commits(moe, layer, gpu_ctx):
    import torch
    print("case concurrent commits on two streams", flush=True)
    pre = [layer.LayerWorkspace(gpu_ctx, c, layer.make_inputs(c)) for c in (_prefill(layer, moe, 0xC0C0A),
                                                                             _prefill(layer, moe, 0xC0C0B))]
    dec = [layer.DecodeWorkspace(gpu_ctx, c, layer.make_inputs(c)) for c in (_decode(layer, moe, 0xC0C0C),
                                                                             _decode(layer, moe, 0xC0C0D))]
    # Each layer alone first: the references.
    main = torch.cuda.current_stream().cuda_stream
    want_pre, want_dec = [], []
    for ws in pre:
        ws.run_layer(main)
        torch.cuda.synchronize()
        assert ws.read_status(main) == (0, 0, 0)
        want_pre.append(_out(ws))
    for ws in dec:
        ws.run(main)
        torch.cuda.synchronize()
        assert ws.read_status() == 0
        want_dec.append(_out(ws))
    assert not np.array_equal(want_pre[0], want_pre[1]) and not np.array_equal(want_dec[0], want_dec[1])
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]  # default priority
    for rnd in range(4):
        for _ in range(20):  # 20 x (2 prefill + 2 decode) commits of two ring slots each per round
            for i in (0, 1):
                pre[i].run_layer(streams[i].cuda_stream)
                dec[i].run(streams[i].cuda_stream)
        torch.cuda.synchronize()
        for i in (0, 1):
            assert pre[i].read_status(main) == (0, 0, 0)
            assert dec[i].read_status() == 0
            assert np.array_equal(_out(pre[i]).view(np.uint32), want_pre[i].view(np.uint32)), (rnd, "prefill", i)
            assert np.array_equal(_out(dec[i]).view(np.uint32), want_dec[i].view(np.uint32)), (rnd, "decode", i)


def test_ring_reuse_through_stage_entry_points(moe, layer, gpu_ctx, stream):
    """The standalone stages report their slots from other kernels than the layers do: 80 commits
    each of two workspaces' gate/up and routed-FFN stages, alternately, one slot per stage, so
    every slot is handed out again several times."""
    import torch
    print("case ring reuse through standalone stages", flush=True)
    pre = [layer.LayerWorkspace(gpu_ctx, c, layer.make_inputs(c)) for c in (_prefill(layer, moe, 0xC0C1A),
                                                                            _prefill(layer, moe, 0xC0C1B))]
    dec = [layer.DecodeWorkspace(gpu_ctx, c, layer.make_inputs(c)) for c in (_decode(layer, moe, 0xC0C1C),
                                                                            _decode(layer, moe, 0xC0C1D))]
    for p, d in zip(pre, dec):
        p.run_layer(stream)
        d.run(stream)
    torch.cuda.synchronize()
    outs = [b for p, d in zip(pre, dec) for b in (p.hidden, d.gate, d.parts)]
    want = [gu.host(b, np.uint32).copy() for b in outs]
    for b in outs:
        b.tensor.fill_(7)
    keep = []
    for _ in range(80):
        for p, d in zip(pre, dec):
            keep = [p.gate_up_buffers(), d.routed_buffers()]
            seg = gpu_ctx.segment()
            ok, err = seg.encode_prefill_moe_gu(p.shape, p.cfg.gate_up_fmt, keep[0])
            assert ok, err
            ok, err = seg.encode_moe_routed_ffn(d.shape, d.cfg.gate_up_fmt, d.cfg.down_fmt, keep[1])
            assert ok, err
            seg.commit(stream)
    torch.cuda.synchronize()
    for b, w in zip(outs, want):
        assert np.array_equal(gu.host(b, np.uint32), w)


def _spin(stream, ms, rate):
    """Keeps `stream` busy for about `ms` with one workgroup; the event behind it."""
    import torch
    with torch.cuda.stream(stream):
        torch.cuda._sleep(int(ms * rate))
        ev = torch.cuda.Event()
        ev.record()
    return ev


def _spin_rate():
    """Cycles of torch.cuda._sleep per millisecond."""
    import torch
    torch.cuda._sleep(1000)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    torch.cuda._sleep(10_000_000)
    b.record()
    torch.cuda.synchronize()
    return 10_000_000 / a.elapsed_time(b)


def _independent_streams(rate):
    """Two streams that run beside each other (several streams may share one hardware queue)."""
    import torch
    first = torch.cuda.Stream()
    for _ in range(8):
        other = torch.cuda.Stream()
        late, early = _spin(other, 100, rate), _spin(first, 1, rate)
        early.synchronize()
        beside = not late.query()
        torch.cuda.synchronize()
        if beside:
            return first, other
    pytest.skip("no two streams with hardware queues of their own")


def test_full_ring_waits_for_its_own_launches_only(moe, layer):
    """64 slots read by layers queued behind 1.5 s of other work: the next encode waits for the
    first of them, and for nothing else. Work on an unrelated stream is still running when it
    returns, and another thread's commit on the context is not held up while it waits."""
    import threading
    import time

    import torch
    print("case ring full behind other work", flush=True)
    ctx = moe.Context(0)
    ws = [layer.DecodeWorkspace(ctx, c, layer.make_inputs(c)) for c in (_decode(layer, moe, 0xC0C2A),
                                                                       _decode(layer, moe, 0xC0C2B))]
    main = torch.cuda.current_stream().cuda_stream
    want = []
    for w in ws:
        w.run(main)
        torch.cuda.synchronize()
        want.append(_out(w))
        w.out.tensor.fill_(7.0)
    rate = _spin_rate()
    a, b = _independent_streams(rate)
    late = _spin(b, 4000, rate)
    gate = _spin(a, 1500, rate)
    ready = ctx.segment()  # encoded ahead: two of the 64 slots, not yet committed
    ok, err = ws[1].encode(ready)
    assert ok, err
    for _ in range(31):
        ws[0].run(a.cuda_stream)
    assert not gate.query()
    done = []

    def next_layer():
        ws[0].run(a.cuda_stream)
        done.append((gate.query(), late.query()))

    t = threading.Thread(target=next_layer)
    t.start()
    time.sleep(0.2)
    assert t.is_alive() and not gate.query(), "the encode did not have to wait"
    ready.commit(a.cuda_stream)
    held_up = gate.query() or not t.is_alive()
    t.join()
    torch.cuda.synchronize()
    assert not held_up, "a commit waited for another thread's encode"
    assert done == [(True, False)], "the encode waited for an unrelated stream"
    for w, o in zip(ws, want):
        assert w.read_status() == 0
        assert np.array_equal(_out(w).view(np.uint32), o.view(np.uint32))


def test_failed_commit_keeps_its_slots(moe, layer):
    """A commit that reports an error left by an earlier call of the thread has queued its first
    launch all the same: its slot is not handed out again before that launch has read it (the 64
    claims behind the failed commit fill every slot with another layer's table)."""
    import torch
    print("case slots of a failed commit", flush=True)
    ctx = moe.Context(0)
    ws = [layer.DecodeWorkspace(ctx, c, layer.make_inputs(c)) for c in (_decode(layer, moe, 0xC0C3A),
                                                                       _decode(layer, moe, 0xC0C3B))]
    main = torch.cuda.current_stream().cuda_stream
    for w in ws:
        w.run(main)
    torch.cuda.synchronize()
    table = gu.host(ws[0].snap_gu, np.uint8).copy()
    want = _out(ws[0])
    ws[0].snap_gu.tensor.fill_(0)
    rate = _spin_rate()
    a = torch.cuda.Stream()
    hip = moe.library()  # resolves the HIP runtime that the library is linked with
    hip.hipGetLastError()
    gate = _spin(a, 400, rate)
    seg = ctx.segment()
    bufs = ws[0].routed_buffers()
    ok, err = seg.encode_moe_routed_ffn(ws[0].shape, ws[0].cfg.gate_up_fmt, ws[0].cfg.down_fmt, bufs)
    assert ok, err
    assert hip.hipSetDevice(1 << 20) != 0  # an error of the thread, left unread
    with pytest.raises(RuntimeError, match="SM_E_DEVICE"):
        seg.commit(a.cuda_stream)
    assert not gate.query()
    held = []
    for _ in range(32):
        s = ctx.segment()
        ok, err = ws[1].encode(s)
        assert ok, err
        held.append(s)
    assert gate.query(), "a slot was handed out while the failed commit's launch had not read it"
    for s in held:
        s.abort()
    torch.cuda.synchronize()
    assert np.array_equal(gu.host(ws[0].snap_gu, np.uint8), table)
    ws[0].run(main)
    torch.cuda.synchronize()
    assert ws[0].read_status() == 0 and np.array_equal(_out(ws[0]).view(np.uint32), want.view(np.uint32))
