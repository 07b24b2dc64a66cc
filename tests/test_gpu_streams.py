"""One plan used from several streams, threads and a graph on the GPU: what the plan
keeps for its launches (partial sums, counters, the repacked block, the packed
weight arguments) must not mix between them."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ok(rc):
    assert rc == 0


@pytest.mark.parametrize("prec,nant,nchan,npkt,nbeam", [(0, 64, 8, 32, 32), (1, 60, 16, 64, 250), (2, 100, 16, 64, 97)])
def test_beam_powers_of_small_blocks_on_several_streams_and_in_a_graph(bf, prec, nant, nchan, npkt, nbeam):
    """Small blocks, whose one launch sums the beam powers with counters that the plan
    keeps: queued on the plan's stream and two others without a wait between them, in
    a graph replayed between eager executes, and after a second pointing, each gives
    the output and powers that a plan with its variant set gives for that block."""
    hip = bf.lib                     # (the HIP runtime is among its dependencies)
    cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=16, precision=prec, weight_mode=1,
                    angle_mode=bf.ANGLE_SIN)
    freqs, scale = bf.reference_freqs(1498.75, nchan), np.full(nbeam, 2e-3 / nant, np.float32)
    plan, ref = bf.Plan(cfg), bf.Plan(cfg)
    ref.variant = ref.variant
    rng = np.random.default_rng(prec)
    blocks = [rng.integers(0, 256, bf.input_bytes(cfg), dtype=np.uint8) for _ in range(3)]
    put = lambda a: (lambda b: (b.upload(a), b)[1])(bf.DeviceBuffer(a.nbytes))  # noqa: E731
    d_scale, ins = put(scale), [put(b) for b in blocks]
    n_out = bf.output_bytes(cfg)
    outs, bps = [put(np.zeros(n_out, np.uint8)) for _ in blocks], [put(np.zeros(nbeam, np.float32)) for _ in blocks]
    streams = [None, ctypes.c_void_p(), ctypes.c_void_p()]
    for s in streams[1:]:
        _ok(hip.hipStreamCreateWithFlags(ctypes.byref(s), 1))
    run = lambda k: plan.execute(ins[k], d_scale, outs[k], None, bps[k], stream=streams[k])  # noqa: E731

    def check(want, ks=(0, 1, 2)):
        _ok(hip.hipDeviceSynchronize())
        for k in ks:
            assert np.array_equal(outs[k].download(np.empty(n_out, np.uint8)), want[k][0].ravel())
            assert np.array_equal(bps[k].download(np.empty(nbeam, np.float32)), want[k][1])
            outs[k].upload(np.zeros(n_out, np.uint8))
            bps[k].upload(np.zeros(nbeam, np.float32))

    for pointing in (5, 6):
        antpos, cal, theta = bf.synth_geometry(nant, cfg.ncal, nbeam, pointing)
        for p in (plan, ref):
            p.set_weights(antpos, cal, freqs, theta)
        want = [ref.process_block(b, scale, want_beam_power=True) for b in blocks]
        want = [(w[0], w[-1]) for w in want]
        for _ in range(3):
            for _ in range(20):
                for k in (0, 1, 2, 2, 1, 0):
                    run(k)
            check(want)
        graph, launch = ctypes.c_void_p(), ctypes.c_void_p()
        _ok(hip.hipStreamBeginCapture(streams[1], 0))
        run(1)
        _ok(hip.hipStreamEndCapture(streams[1], ctypes.byref(graph)))
        _ok(hip.hipGraphInstantiate(ctypes.byref(launch), graph, None, None, ctypes.c_size_t(0)))
        for _ in range(3):
            _ok(hip.hipGraphLaunch(launch, streams[1]))
            check(want, (1,))
            for k in (0, 2, 1):
                run(k)
            check(want)
        _ok(hip.hipGraphExecDestroy(launch))
        _ok(hip.hipGraphDestroy(graph))
    for p in (plan, ref):
        p.close()
    for s in streams[1:]:
        _ok(hip.hipStreamDestroy(s))
