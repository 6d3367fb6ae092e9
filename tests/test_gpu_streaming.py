"""Plane streaming through fmvd_deconvolve_planes_cuda_* with a bounded
look-ahead: the reference's datasource/datasink call order
(fmvd_deconvolve.impl.cpp:216-245,288-294: nStreams gets, then a sink and a
get per plane until a get returns 0, then the remaining sinks) and results
bit-identical to the batched pipeline."""
import numpy as np
import pytest

from gpu_util import make_case

pytestmark = pytest.mark.gpu


def reference_order(D, L):
    """Callback sequence of the reference driver for D >= L planes."""
    seq = [("get", 1)] * L
    z = 0
    for _ in range(L, D):
        seq += [("put", z), ("get", 1)]
        z += 1
    seq += [("put", z), ("get", 0)]
    z += 1
    seq += [("put", k) for k in range(z, D)]
    return seq


@pytest.mark.parametrize("D,L", [(5, 3), (3, 3), (7, 2), (6, 1), (2, 3)])
def test_lookahead_call_order_and_results(fm, D, L):
    V, dh, dw, k = 2, 48, 60, 11
    data, kernels, weights = make_case(D, V, dh, dw, k, k, 16, seed=D * 10 + L)
    planes = [[data[z, v] for v in range(V)] for z in range(D)]
    print(f"\n[lookahead] D={D} L={L}", flush=True)
    with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], nstreams=L) as dec:
        batched, best = dec.run(planes, 4, want_estimate=True)
        assert dec.set_lookahead(L) == L
        out, est = dec.run(planes, 4, want_estimate=True)
        calls = dec.calls
    if D >= L:
        assert calls == reference_order(D, L)
    else:  # a source that runs dry during the first L calls ends the stream there
        assert calls == [("get", 1)] * D + [("get", 0)] + [("put", z) for z in range(D)]
    assert np.array_equal(out, batched)
    assert np.array_equal(est, best)
    # at most L planes are ever held between a get and its put
    held = 0
    for kind, ok in calls:
        held += 1 if (kind == "get" and ok) else (-1 if kind == "put" else 0)
        assert 0 <= held <= L


@pytest.mark.parametrize("D", [1, 4, 11])
def test_staging_kept_between_runs(fm, D):
    """One plan, runs of changing length, with and without the estimate sink,
    against a single-batch plan: batches of 2 planes, so 11 planes reuse each slot."""
    V, dh, dw, k = 2, 40, 52, 9
    data, kernels, weights = make_case(D, V, dh, dw, k, k, 16, seed=70 + D)
    planes = [[data[z, v] for v in range(V)] for z in range(D)]
    with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], batch_planes=64) as dec:
        out, est = dec.run(planes, 3, want_estimate=True)
    with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], nstreams=1, chunk_planes=2) as dec:
        for n, sink in ((D, False), (D, True), (0, True), (max(1, D - 3), True), (D, True)):
            o, e = dec.run(planes[:n], 3, want_estimate=sink)
            assert np.array_equal(o, out[:n])
            assert not (sink and n) or np.array_equal(e, est[:n])


@pytest.mark.parametrize("bits", [16, 8])
def test_reported_stream_batch(fm, bits):
    """What the plan reports as a stream's batch is what the first fill pulls: default, chunk, batch and look-ahead."""
    D, V, dh, dw, k = 9, 1, 40, 52, 9
    data, kernels, weights = make_case(D, V, dh, dw, k, k, bits, seed=3)
    planes = [[data[z, v] for v in range(V)] for z in range(D)]
    with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], bits=bits, nstreams=2, chunk_planes=4) as dec:
        for setting, want in ((lambda: None, 4), (lambda: dec.set_chunk_planes(1), 2), (lambda: dec.set_batch_planes(3), 3),
                              (lambda: dec.set_lookahead(5), 5)):
            setting()
            assert dec.info()["stream_batch"] == want
            dec.run(planes, 1)
            assert dec.calls.index(("put", 0)) >= want and all(c == ("get", 1) for c in dec.calls[:want])
            if want < 5:  # the pipeline pulls a second batch behind the first, then drains
                assert dec.calls.index(("put", 0)) == min(2 * want, D) + (2 * want > D)


def test_two_lanes_in_a_stream(fm, monkeypatch):
    """FMVD_LANES=2 runs the chunks of a stream on two streams: a batch holds one chunk for each, and results are the same."""
    D, V, dh, dw, k = 11, 2, 40, 52, 9
    data, kernels, weights = make_case(D, V, dh, dw, k, k, 16, seed=9)
    planes = [[data[z, v] for v in range(V)] for z in range(D)]
    got = []
    for lanes, want in ((1, 2), (2, 4)):
        monkeypatch.setenv("FMVD_LANES", str(lanes))
        with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], nstreams=1, chunk_planes=2) as dec:
            assert dec.info()["stream_batch"] == want
            got.append(dec.run(planes, 3, want_estimate=True))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


def test_timing_stride_over_a_stream(fm):
    """With kernel timing on, the launches of every 8th chunk of a stream are timed, also where a batch is one chunk."""
    D, V, dh, dw, k, it = 19, 2, 40, 52, 9, 3
    data, kernels, weights = make_case(D, V, dh, dw, k, k, 16, seed=4)
    planes = [[data[z, v] for v in range(V)] for z in range(D)]
    with fm.Deconvolver(dh, dw, list(weights), [x.copy() for x in kernels], nstreams=1, chunk_planes=1) as dec:
        assert dec.info()["stream_batch"] == 1
        with fm.KernelTiming() as kt:
            dec.run(planes, it)
            fm.device_synchronize()
            assert kt.read("ratio")[1] == 3 * V * it  # chunks 0, 8, 16
            assert kt.read("egress")[1] == 3


def test_staging_is_bounded_and_given_back(fm, monkeypatch):
    """A stream's staging stays with the plan up to the batch budget, and is given back by a new batch size and by a
    resident run that needs larger work buffers.  Free device memory tells (batches of 64 planes of 512^2, two views:
    two slots of 100 MB; a chunk with estimates: two of 42 MB)."""
    V, n, k, MB = 2, 512, 9, 1 << 20
    rng = np.random.default_rng(1)
    planes = [[rng.integers(0, 900, (n, n)).astype(np.uint16) for _ in range(V)] for _ in range(3)]
    kernels, weights = np.full((V, k, k), 1.0 / 81, np.float32), np.ones((V, n, n), np.float32)

    def given_back(plan, batch):
        before = fm.device_memory()[0]
        plan.set_batch_planes(batch)
        return fm.device_memory()[0] - before

    def plan(batch=0):
        return fm.Deconvolver(n, n, list(weights), [x.copy() for x in kernels], batch_planes=batch)

    with plan(64) as dec:
        first, _ = dec.run(planes, 2)
        assert given_back(dec, 64) >= 190 * MB
        again, _ = dec.run(planes, 2)
        assert np.array_equal(first, again)
    monkeypatch.setenv("FMVD_BATCH_BYTES", str(64 * MB))
    with plan(64) as dec:
        again, _ = dec.run(planes, 2)
        assert np.array_equal(first, again)
        assert given_back(dec, 64) < 20 * MB
    monkeypatch.delenv("FMVD_BATCH_BYTES")
    with plan() as dec:
        dec.run(planes, 2, want_estimate=True)
        assert given_back(dec, 0) >= 70 * MB
        dec.run(planes, 2, want_estimate=True)
        Z = 3 * dec.info()["stream_batch"]
        views = [fm.DeviceArray((Z, n, n), np.uint16) for _ in range(V)]
        for v in views:
            v.fill_zero()
        out = fm.DeviceArray((Z, n, n), np.uint16)
        dec.run_device([v.ptr for v in views], Z, 1, out_ptr=out.ptr)
        fm.device_synchronize()
        assert given_back(dec, 0) < 20 * MB
        again, _ = dec.run(planes, 2)
        assert np.array_equal(first, again)
