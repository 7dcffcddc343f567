"""The status word of the device quantizers: cleared by the call whatever it held, and every
condition that the host reports by throwing (pack.hpp:64-72, mx.hpp:71-76, kvcache.hpp:60-68) found in it
wherever the element lies -- with one workgroup and with thousands, on several streams at once, and on
every replay of a captured call."""
import ctypes
import threading

import pytest
import torch

import w4amd
from devutil import DEV, ptr

pytestmark = pytest.mark.gpu
INF, BAD, RANGE = float("inf"), 1, 2


def _cache(H, S, D, gs, sym):
    G, i32 = D // gs, dict(dtype=torch.int32, device=DEV)
    side = lambda: [torch.empty(H, S, D // 8, **i32), torch.empty(H, S, G, dtype=torch.float16, device=DEV),
                    None if sym else torch.empty(H, S, (G + 7) // 8, **i32)]
    t = side() + side()
    return w4amd.capi().kv_view(H, S, D, gs, G, sym, *[ptr(a) for a in t]), t


def _kv(kind, H, S, D, gs):
    """(call(k, v, status, stream), buffers to keep) of one of the quantizers that take FP16."""
    c = w4amd.capi()
    rows = H * S
    if kind in ("w4", "w4z"):
        view, t = _cache(H, S, D, gs, kind == "w4")
        return lambda k, v, st, s: c.quantize_cache(view, ptr(k), ptr(v), st, stream=s, src_f16=True), t
    if kind == "f8":
        G = D // gs
        t = [torch.empty(H, S, D, dtype=torch.uint8, device=DEV), torch.empty(H, S, G, dtype=torch.float16, device=DEV),
             torch.empty(H, S, D, dtype=torch.uint8, device=DEV), torch.empty(H, S, G, dtype=torch.float16, device=DEV)]
        view = c.kv_f8_view(H, S, D, gs, G, *[ptr(a) for a in t])
        return lambda k, v, st, s: c.quantize_cache_f8(view, ptr(k), ptr(v), st, stream=s, src_f16=True), t
    B = D // 32
    sc = torch.empty(rows, B, dtype=torch.uint8, device=DEV)
    if kind == "mx":
        q = torch.empty(rows, D // 8, dtype=torch.int32, device=DEV)
        view = c.packed_mx_view(rows, D, B, ptr(q), ptr(sc))
        return lambda k, v, st, s: c.quantize_mx_f16(view, ptr(k), st, stream=s), (q, sc)
    q = torch.empty(rows, D, dtype=torch.uint8, device=DEV)
    view = c.act_mx8_view(rows, D, B, ptr(q), ptr(sc))
    return lambda k, v, st, s: c.quantize_mx8_f16(view, ptr(k), st, stream=s), (q, sc)


def _inputs(H, S, D):
    g = torch.Generator(device=DEV).manual_seed(H * S + D)
    return [torch.randn(H, S, D, dtype=torch.float16, device=DEV, generator=g) for _ in range(2)]


KINDS = ["w4", "w4z", "f8", "mx", "mx8"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("H,S,D,gs", [(1, 1, 64, 32), (2, 33, 128, 32), (8, 4096, 128, 64), (3, 50, 96, 32)])
def test_status_is_cleared_and_set(kind, H, S, D, gs):
    call, keep = _kv(kind, H, S, D, gs)
    k, v = _inputs(H, S, D)
    st = torch.full((1,), -1, dtype=torch.int32, device=DEV)
    n = k.numel()
    for i in (0, n // 2, n - 1, None):
        if i is not None:
            old = k.view(-1)[i].item()
            k.view(-1)[i] = float("nan")
            st.fill_(0x55)
            call(k, v, ptr(st), 0)
            assert st.item() == BAD, (kind, i)
            k.view(-1)[i] = INF
            call(k, v, ptr(st), 0)
            assert st.item() & BAD, (kind, i)
            k.view(-1)[i] = old
        call(k, v, ptr(st), 0)
        assert st.item() == 0, (kind, i)


@pytest.mark.parametrize("kind", KINDS)
def test_every_element_bad(kind):
    """Every wave reports."""
    H, S, D, gs = 8, 2048, 128, 32
    call, keep = _kv(kind, H, S, D, gs)
    k = torch.full((H, S, D), INF, dtype=torch.float16, device=DEV)
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    for _ in range(3):
        call(k, k, ptr(st), 0)
        assert st.item() == BAD | RANGE, kind


def test_calls_on_several_streams():
    """Calls that overlap, each with a word of its own: half of them with a bad element at the end."""
    H, S, D, gs = 4, 512, 128, 32
    streams = [torch.cuda.Stream() for _ in range(4)]
    jobs = []
    for i in range(64):
        call, keep = _kv(KINDS[i % 5], H, S, D, gs)
        k, v = _inputs(H, S, D)
        if i % 2:
            k.view(-1)[-1 - i] = INF
        jobs.append((call, keep, k, v))
    st = torch.full((64,), 0x77, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    for _ in range(3):
        for i, (call, _, k, v) in enumerate(jobs):
            call(k, v, ptr(st) + 4 * i, streams[i % 4].cuda_stream)
        torch.cuda.synchronize()
        got = st.tolist()
        assert [bool(x & BAD) for x in got] == [bool(i % 2) for i in range(64)], got
        st.fill_(0x33)
        torch.cuda.synchronize()


@pytest.mark.parametrize("kind", KINDS)
def test_every_element_bad_is_no_queue(kind):
    """Reports of one kind meet in one word: 256 K of them take less than 1 ms (sound input: under 0.01)."""
    H, S, D, gs = 8, 4096, 128, 32
    call, keep = _kv(kind, H, S, D, gs)
    k = torch.full((H, S, D), float("nan"), dtype=torch.float16, device=DEV)
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    call(k, k, ptr(st), 0)
    assert min(_ms(lambda: call(k, k, ptr(st), 0)) for _ in range(5)) < 1.0
    assert st.item() == BAD


@pytest.mark.parametrize("kind", KINDS)
def test_replays_of_a_captured_call(kind):
    H, S, D, gs = 2, 257, 128, 32
    call, keep = _kv(kind, H, S, D, gs)
    k, v = _inputs(H, S, D)
    good = k.clone()
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    call(k, v, ptr(st), 0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(k, v, ptr(st), torch.cuda.current_stream().cuda_stream)
    for i in range(6):
        k.copy_(good)
        if i % 2:
            k.view(-1)[i * 7919 % k.numel()] = float("nan")
        st.fill_(0x11)
        graph.replay()
        torch.cuda.synchronize()
        assert st.item() == (BAD if i % 2 else 0), (kind, i)


def _ms(fn):
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    fn()
    b.record()
    b.synchronize()
    return a.elapsed_time(b)


def test_no_other_call_clears_the_word_again():
    """A call that finds something at its start and something else at its end, and one 4096 calls later
    that runs in the middle of it on another stream: both bits of the first call are reported."""
    c = w4amd.capi()
    N, K, gs = 65536, 4800, 48  # (no power of two: the general kernel, some milliseconds)
    w = torch.ones(N, K, dtype=torch.float64, device=DEV)
    w[0, 0], w[-1, -1] = float("nan"), 1e300
    q, sc = torch.empty(N, K // 8, dtype=torch.int32, device=DEV), torch.empty(N, K // gs, dtype=torch.float16, device=DEV)
    long_view = c.packed_view(N, K, gs, K // gs, True, ptr(q), ptr(sc))
    call, keep = _kv("w4", 1, 1, 64, 32)
    k, v = _inputs(1, 1, 64)
    st = torch.zeros(3, dtype=torch.int32, device=DEV)
    c.quantize(long_view, ptr(w), ptr(st))
    long_ms = _ms(lambda: c.quantize(long_view, ptr(w), ptr(st)))
    torch.cuda._sleep(1000)
    per_ms = 1e6 / _ms(lambda: torch.cuda._sleep(1000000))  # cycles of a millisecond
    for _ in range(5):
        gate, s1, s2, s3 = [torch.cuda.Stream() for _ in range(4)]  # (some may share a hardware queue)
        st.fill_(0x55)
        torch.cuda.synchronize()
        start = torch.cuda.Event()
        with torch.cuda.stream(gate):
            torch.cuda._sleep(int(60 * per_ms))  # until everything below is enqueued
            start.record()
        s1.wait_event(start)
        s2.wait_event(start)
        c.quantize(long_view, ptr(w), ptr(st), stream=s1.cuda_stream)
        for _ in range(4095):
            call(k, v, ptr(st) + 4, s3.cuda_stream)
        with torch.cuda.stream(s2):
            torch.cuda._sleep(int(long_ms / 2 * per_ms))
        call(k, v, ptr(st) + 8, s2.cuda_stream)
        torch.cuda.synchronize()
        assert st.tolist() == [BAD | RANGE, 0, 0]


def test_threads_that_share_streams():
    """Four threads that enqueue calls on the legacy stream and on one other stream, each call with a word of its own."""
    stream = torch.cuda.Stream()
    jobs = []
    for i in range(4):
        call, keep = _kv(KINDS[i], 2, 257, 128, 32)
        k, v = _inputs(2, 257, 128)
        bad = k.clone()
        bad.view(-1)[1234 + i] = INF
        jobs.append((call, keep, k, bad, v))
    st = torch.full((4, 200), 0x44, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()

    def work(i):
        call, _, k, bad, v = jobs[i]
        for j in range(200):
            call(bad if j % 3 == i % 3 else k, v, ptr(st) + 4 * (200 * i + j), stream.cuda_stream if j % 2 else 0)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, row in enumerate(st.tolist()):
        for j, x in enumerate(row):
            assert bool(x & BAD) == (j % 3 == i % 3) and (x & BAD or x == 0), (i, j, x)


def test_more_streams_than_slots():
    """Streams past the ones that have a slot clear the word by a launch of its own."""
    hip = ctypes.CDLL(w4amd.capi().LIB_PATH)  # (the runtime that the library is linked to)
    streams = []
    for _ in range(80):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(s)) == 0
        streams.append(s.value)
    call, keep = _kv("w4z", 2, 33, 128, 32)
    k, v = _inputs(2, 33, 128)
    bad = k.clone()
    bad[0, 7, 3] = INF
    st = torch.full((80,), 0x66, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()
    for _ in range(2):
        for i, s in enumerate(streams):
            call(bad if i % 3 else k, v, ptr(st) + 4 * i, s)
        torch.cuda.synchronize()
        assert [bool(x & BAD) for x in st.tolist()] == [bool(i % 3) for i in range(80)]
        assert all(x == 0 for x in st.tolist()[::3])
    for s in streams:
        assert hip.hipStreamDestroy(ctypes.c_void_p(s)) == 0
