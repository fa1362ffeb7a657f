"""l3m_k_attend (one query head over a K/V cache) where its work is split: lane groups of 1 to 32 lanes a row,
batches of rows, one workgroup or up to 64 whose parts meet in a workspace of the stream. Against the oracle's
l3m_attend within 1e-5 absolute (the reference's own bar, tests/test_kernels.c:145)."""
import ctypes as C
import threading

import numpy as np
import pytest

import l3m_amd as A

pytestmark = pytest.mark.gpu


def inputs(seed, n, hd, stride):
    rng = np.random.default_rng(seed)
    q = (rng.standard_normal(hd) * 2).astype(np.float32)
    k, v = (rng.integers(0, 1 << 16, n * stride + 8, dtype=np.uint16) & 0xBF7F for _ in range(2))   # bf16, |v| < 2
    return q, k.astype(np.uint16), v.astype(np.uint16)


@pytest.mark.parametrize("hd", [8, 16, 40, 64, 128, 200, 256])
@pytest.mark.parametrize("n", [1, 2, 31, 33, 255, 257, 1025, 4001, 8001])
def test_attend_splits(dev, oracle, hd, n):
    stride = hd + 8 * (n % 3)
    q, k, v = inputs(hd * 10007 + n, n, hd, stride)
    got = dev.attend(q, k, v, n - 1, hd, stride)
    want = oracle.attend(q, k, v, n - 1, hd, stride)
    assert np.abs(got - want).max() <= 1e-5, np.abs(got - want).max()
    again = dev.attend(q, k, v, n - 1, hd, stride)            # whichever workgroup ends last
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))
    dev.free_all()


def test_attend_unaligned_v_rows(dev, oracle):
    """V needs no alignment beyond an element's: a V pointer one element past a 16-byte boundary."""
    n, hd = 700, 64
    q, k, v = inputs(5, n, hd, hd)
    dq, dk, dv, do = dev.put(q), dev.put(k), dev.put(v), dev.alloc(hd * 4)
    assert dev.lib.l3m_k_attend(do, dq, dk, dv + 2, n - 1, hd, hd, None) == 0
    got = dev.get(do, hd, np.float32)
    assert np.abs(got - oracle.attend(q, k, v[1:], n - 1, hd, hd)).max() <= 1e-5
    dev.free_all()


@pytest.mark.parametrize("at", [(3, 700), (515, 90), (1029, 4), (1029, 1028)])
def test_attend_large_values_and_masked_rows(dev, oracle, at):
    """Scores far past expf's range (the largest above 200, in the first, a middle and the last of nine workgroups' rows,
    and a second one just below it in another's, or its own), and rows past the last one that hold infinities: they
    are not attended. q and K are small multiples of a half, so every score is exact in f32."""
    n, hd = 1030, 64
    rng = np.random.default_rng(sum(at))
    q = rng.integers(-40, 41, hd).astype(np.float32)
    q[7] = 12
    kf = rng.integers(-2, 3, (n, hd)).astype(np.float32) / 2
    kf[at[0]] = np.where(q > 0, 1, -1) * 1.5
    kf[at[1]] = kf[at[0]]
    kf[at[1], 7] = 1                                   # its score: 12 * 0.5 / 8 lower
    s = np.sort(kf @ q / 8)
    assert s[-1] > 200 and s[-1] - s[-2] == 0.75 and s[-3] < s[-1] - 50
    k = np.full((n + 40, hd), 0x7F80, np.uint16)
    k[:n] = kf.view(np.uint32) >> 16
    v = inputs(6, n + 40, hd, hd)[2]
    v[n * hd:] = 0x7F80
    got = dev.attend(q, k.ravel(), v, n - 1, hd, hd)
    want = oracle.attend(q, k[:n].ravel(), v[:n * hd], n - 1, hd, hd)
    assert np.abs(got - want).max() <= 1e-5
    two = [(v[i * hd:(i + 1) * hd].astype(np.uint32) << 16).view(np.float32) for i in at]   # the weights: 1 and exp(-0.75)
    assert np.abs(want - (two[0] + two[1] * np.exp(-0.75)) / (1 + np.exp(-0.75))).max() <= 1e-5
    dev.free_all()


def test_attend_many_streams_and_capture(dev, oracle):
    """18 streams with a call each in flight (two more than there are workspaces), three rounds of other inputs; then a
    call recorded into a graph, replayed between other calls on the same stream."""
    hip = C.CDLL("libamdhip64.so")
    n, hd = 3000, 64
    streams = []
    for _ in range(18):
        st = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(st)) == 0
        streams.append(st)
    for rnd in range(3):
        sets = [inputs(100 * rnd + i, n, hd, hd) for i in range(18)]
        bufs = [(dev.put(q), dev.put(k), dev.put(v), dev.alloc(hd * 4)) for q, k, v in sets]
        for st, (q, k, v, o) in zip(streams, bufs):
            assert dev.lib.l3m_k_attend(o, q, k, v, n - 1, hd, hd, st) == 0
        assert hip.hipDeviceSynchronize() == 0
        for (q, k, v), b in zip(sets, bufs):
            assert np.abs(dev.get(b[3], hd, np.float32) - oracle.attend(q, k, v, n - 1, hd, hd)).max() <= 1e-5
    st, (q, k, v, o) = streams[0], bufs[0]
    graph, ex, want = C.c_void_p(), C.c_void_p(), oracle.attend(*sets[0], n - 1, hd, hd)
    assert hip.hipStreamBeginCapture(st, 1) == 0
    assert dev.lib.l3m_k_attend(o, q, k, v, n - 1, hd, hd, st) == 0
    assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    o2 = dev.alloc(hd * 4)
    for _ in range(3):
        assert hip.hipGraphLaunch(ex, st) == 0
        assert dev.lib.l3m_k_attend(o2, q, k, v, n - 1, hd, hd, st) == 0
        assert hip.hipStreamSynchronize(st) == 0
        for p in (o, o2):
            assert np.abs(dev.get(p, hd, np.float32) - want).max() <= 1e-5
    assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0
    for st in streams:
        assert hip.hipStreamDestroy(st) == 0
    dev.free_all()


def test_attend_streams_come_and_go(dev, oracle):
    """40 streams, 20 at a time, each used and destroyed, the last 20 with their calls just queued: a workspace goes back
    when its last call has ended, so a later stream's result is the library stream's bit for bit (the split's order of
    sums; one workgroup's differs), and handles that come up again are safe."""
    hip = C.CDLL("libamdhip64.so")
    n, hd = 3000, 64
    q, k, v = inputs(8, n, hd, hd)
    dq, dk, dv, do = dev.put(q), dev.put(k), dev.put(v), dev.alloc(hd * 4)

    def call(st):
        assert dev.lib.l3m_k_attend(do, dq, dk, dv, n - 1, hd, hd, st) == 0

    call(None)
    want = dev.get(do, hd, np.float32)
    assert np.abs(want - oracle.attend(q, k, v, n - 1, hd, hd)).max() <= 1e-5
    for rnd in range(3):
        streams = []
        for _ in range(20):
            st = C.c_void_p()
            assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0
            streams.append(st)
        for st in streams:
            call(st)
            if rnd < 2:
                assert hip.hipStreamSynchronize(st) == 0
                got = dev.get(do, hd, np.float32)
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (rnd, np.abs(got - want).max())
        for st in streams:
            assert hip.hipStreamDestroy(st) == 0
    st = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0
    for _ in range(50):
        call(st)
    assert hip.hipDeviceSynchronize() == 0
    got = dev.get(do, hd, np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert hip.hipStreamDestroy(st) == 0
    dev.free_all()


def test_attend_threads_on_their_own_streams(dev, oracle):
    """Four threads, each with two streams and inputs of its own, 60 calls on each while the others do the
    same: every call's output is its inputs'."""
    hip = C.CDLL("libamdhip64.so")
    n, hd, calls = 2000, 64, 60
    sets = [inputs(50 + i, n, hd, hd) for i in range(8)]
    bufs = [(dev.put(q), dev.put(k), dev.put(v)) for q, k, v in sets]
    outs = [[dev.alloc(hd * 4) for _ in range(calls)] for _ in sets]
    streams = []
    for _ in sets:
        st = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0
        streams.append(st)
    failed = []

    def work(t):
        try:
            for c in range(calls):
                for i in (2 * t, 2 * t + 1):
                    assert dev.lib.l3m_k_attend(outs[i][c], *bufs[i], n - 1, hd, hd, streams[i]) == 0
        except BaseException as e:
            failed.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed and hip.hipDeviceSynchronize() == 0
    for (q, k, v), o in zip(sets, outs):
        want = oracle.attend(q, k, v, n - 1, hd, hd)
        for p in o:
            assert np.abs(dev.get(p, hd, np.float32) - want).max() <= 1e-5
    for st in streams:
        assert hip.hipStreamDestroy(st) == 0
    dev.free_all()
