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
