"""The host side of plans, batches and the correlator's plan without a GPU:
host/bf_plan.c, host/bf_batch.c and host/xc_plan.c linked with tests/hip_stub.c,
whose device memory is host memory and whose launches, events and waits are a
log.  Checks what the plans share between calls, streams and threads."""
import ctypes as C
import os
import subprocess
import threading

import numpy as np
import pytest

from conftest import ROOT

HOST = os.path.join(ROOT, "dsa110-xengine_amd", "host")


@pytest.fixture(scope="module")
def lib(tmp_path_factory, bf):
    so = str(tmp_path_factory.mktemp("stub") / "plan.so")
    src = [os.path.join(HOST, f) for f in ("bf_plan.c", "bf_batch.c", "xc_plan.c", "bf_host.c")]
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-std=gnu11", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + HOST, "-Wl,-Bsymbolic", "-o", so, *src,
                    os.path.join(ROOT, "tests", "hip_stub.c"), "-lpthread", "-lm"], check=True)
    L = C.CDLL(so)
    L.stub_log.restype = C.c_char_p
    for f in ("dsaxbf_execute", "dsaxbf_set_variant", "dsaxbf_set_weights", "dsaxbf_destroy", "dsaxbf_get_stream"):
        getattr(L, f).argtypes = None
    L.dsaxbf_get_stream.restype = C.c_void_p
    return L


def _set(lib, **values):
    for k, v in values.items():
        t = {"stub_capturing": C.c_void_p, "stub_live": C.c_long, "stub_psum_bytes": C.c_size_t,
             "stub_packed_bytes": C.c_size_t}.get(k, C.c_int)
        t.in_dll(lib, k).value = v


def _plan(lib, bf, psum=0, packed=0):
    _set(lib, stub_psum_bytes=psum, stub_packed_bytes=packed)
    cfg = bf.config(nant=64, nchan=384, npkt=32, nbeam=64, tavg=32, weight_mode=bf.WEIGHTS_FINE)
    p = C.c_void_p()
    assert lib.dsaxbf_create(C.byref(p), C.byref(cfg)) == 0
    return p, cfg


def _weights(lib, p, cfg, v=1.0):
    arr = [np.full(n, v, t) for n, t in ((cfg.nant, np.float32), (cfg.nant * cfg.ncal * 4, np.float32),
                                         (cfg.nchan, np.float64), (cfg.nbeam, np.float64))]
    assert lib.dsaxbf_set_weights(p, *(C.c_void_p(a.ctypes.data) for a in arr), C.c_double(0)) == 0


ANY = C.c_void_p(64)         # a device pointer that the stub does not look behind


def _execute(lib, p, stream=None, power=True):
    return lib.dsaxbf_execute(p, ANY, ANY, ANY, None, ANY if power else None, stream)


def test_counters_are_zero_from_the_start_and_left_alone(lib, bf):
    """The counters of a launch that sums the beam powers are zero before the first
    launch, and dsaxbf_set_weights does not write them: a launch in flight on
    another stream would lose its count, and all later ones would sum too early."""
    p, cfg = _plan(lib, bf, psum=4096)
    _weights(lib, p, cfg)
    assert _execute(lib, p) == 0
    count = (C.c_uint32 * 32).from_address(C.c_void_p.in_dll(lib, "stub_psum").value)
    assert not any(count)
    count[3] = 7                                   # a launch has counted seven workgroups
    _weights(lib, p, cfg)
    assert count[3] == 7 and sum(count) == 7
    lib.dsaxbf_destroy(p)


def _ordered(log):
    """Whether each launch that uses plan-owned memory for one launch at a time
    starts after the one before it has ended, by its stream's order and the events."""
    clock, event, last, unordered = {}, {}, None, []
    for i, line in enumerate(log.decode().splitlines()):
        op, s, *rest = line.split()
        seen = clock.setdefault(s, set())
        if op == "record":
            event[rest[0]] = set(seen)
        elif op == "wait":
            seen |= event.get(rest[0], set())
        elif op == "launch" and rest[0] != "plain":
            if last is not None and last not in seen:
                unordered.append(line)
            last = i
            seen.add(i)
    return not unordered


STREAMS = [C.c_void_p(16 * k) for k in range(1, 4)]    # a caller's


@pytest.mark.parametrize("kind", ["sums", "packed"])
def test_launches_on_several_streams_take_the_plans_memory_in_turn(lib, bf, kind):
    """Executes of one plan on its own stream and on others, in every order of two
    and three: each launch that sums its beam powers, or reads the repacked block,
    waits for the one before it; a run on the plan's own stream needs no event for
    its sums."""
    p, cfg = _plan(lib, bf, **{"psum" if kind == "sums" else "packed": 4096})
    _weights(lib, p, cfg)
    lib.stub_reset()
    for a in (None, *STREAMS):
        for b in (None, *STREAMS):
            for c in (None, *STREAMS):
                for s in (a, b, c):
                    assert _execute(lib, p, s) == 0
    log = lib.stub_log()
    assert log.count(kind.encode()) == 3 * 64 and b"plain" not in log and _ordered(log)
    lib.stub_reset()
    for _ in range(3):
        assert _execute(lib, p) == 0
    if kind == "sums":
        assert b"".join(line[:6] for line in lib.stub_log().splitlines()[-2:]) == b"launch" * 2
    lib.dsaxbf_destroy(p)


@pytest.mark.parametrize("kind", ["sums", "packed"])
def test_captured_launches_use_none_of_it(lib, bf, kind):
    """Under capture, whose replays would not wait for other launches, a block runs
    without the plan's counters and repacked copy and records no event; so does one
    on another stream while the plan's own is captured, whose end it could not wait
    for."""
    p, cfg = _plan(lib, bf, **{"psum" if kind == "sums" else "packed": 4096})
    _weights(lib, p, cfg)
    own = lib.dsaxbf_get_stream(p)
    for captured, s, alone in [(STREAMS[0].value, STREAMS[0], True), (own, None, True), (own, STREAMS[1], kind == "sums")]:
        assert _execute(lib, p, STREAMS[2]) == 0
        _set(lib, stub_capturing=captured)
        lib.stub_reset()
        assert _execute(lib, p, s) == 0
        ops = [" ".join(x.split()[::2]) for x in lib.stub_log().decode().splitlines()]
        assert (ops == ["launch plain", "power"]) == alone
        _set(lib, stub_capturing=None)
    lib.dsaxbf_destroy(p)


def test_pointings_set_from_two_threads_do_not_mix(lib, bf):
    """dsaxbf_set_weights packs its arguments into memory that the plan keeps: calls
    from two threads each compute their weights from their own arguments."""
    p, cfg = _plan(lib, bf)
    _set(lib, stub_slow_copies=1, stub_torn=0)
    threads = [threading.Thread(target=lambda v=v: [_weights(lib, p, cfg, v) for _ in range(8)]) for v in (1.0, 2.0)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    _set(lib, stub_slow_copies=0)
    assert C.c_int.in_dll(lib, "stub_torn").value == 0
    lib.dsaxbf_destroy(p)


def test_a_launch_that_failed_half_way_keeps_its_turn(lib, bf):
    """Repacking may be queued when the launch behind it fails: the next execute, on
    another stream, still waits for it."""
    p, cfg = _plan(lib, bf, packed=4096)
    _weights(lib, p, cfg)
    lib.stub_reset()
    _set(lib, stub_fail_launch=1)
    assert _execute(lib, p, STREAMS[0]) != 0
    assert _execute(lib, p, STREAMS[1]) == 0
    assert _ordered(lib.stub_log())
    lib.dsaxbf_destroy(p)


def test_the_repacked_block_is_held_only_where_executes_use_it(lib, bf):
    """A plan gives back its repacked block once a variant is set (at the next
    pointing, the call that may free memory) and when it joins a batch, whose
    launches do not repack; the autotuner takes it again."""
    live, log = C.c_long.in_dll(lib, "stub_live"), lambda: lib.stub_log().split()[-1:]
    start = live.value

    def ran(power=False):
        lib.stub_reset()
        assert _execute(lib, p, None, power) == 0
        return [x.split()[-1] for x in lib.stub_log().splitlines() if x.startswith(b"launch")]

    size = 1 << 20
    p, cfg = _plan(lib, bf)
    _weights(lib, p, cfg)
    least = live.value - start
    lib.dsaxbf_destroy(p)
    assert live.value == start
    p, cfg = _plan(lib, bf, packed=size)
    _weights(lib, p, cfg)
    assert ran() == [b"packed"] and live.value - start == least + size
    assert lib.dsaxbf_set_variant(p, lib.dsaxbf_get_variant(p)) == 0
    assert ran() == [b"plain"]
    _weights(lib, p, cfg)
    assert ran() == [b"plain"] and live.value - start == least
    assert lib.dsaxbf_autotune(p, 1, None) == 0            # (the stub's times are equal)
    assert ran() == [b"packed"] and live.value - start == least + size
    batch, one = C.c_void_p(), (C.c_void_p * 1)
    assert lib.dsaxbf_batch_create(C.byref(batch), one(p), 1, one(64), one(64), one(64), None) == 0
    assert ran() == [b"plain"] and live.value - start == least
    _weights(lib, p, cfg)
    assert ran() == [b"plain"] and live.value - start == least
    lib.dsaxbf_batch_destroy(batch)
    lib.dsaxbf_destroy(p)
    assert live.value == start


def test_the_correlators_turned_copy_is_held_only_where_it_is_used(lib):
    """A correlator plan whose kernel reads the block itself has no turned copy (the
    input's size) until slices are set, and again none when they are the library's."""
    live = C.c_long.in_dll(lib, "stub_live")
    nin = 64 * 64 * 48 * 4
    for fused in (0, 2):
        start = live.value
        _set(lib, stub_fused_slices=fused)
        x = C.c_void_p()
        assert lib.dsaxbf_xengine_create(C.byref(x), 64, 48, 64, 0, 0) == 0
        for slices in (None, 1, 2, 0):
            if slices is not None:
                assert lib.dsaxbf_xengine_set_slices(x, slices) == 0
            turned = not fused or slices in (1, 2)
            part = 64 * (2 if slices == 2 else fused if not turned else 0)
            assert live.value - start == nin + 64 + part + (nin if turned else 0)
            lib.stub_reset()
            assert lib.dsaxbf_xengine_execute(x, ANY, ANY, None) == 0
            assert lib.stub_log() == (b"xcorr turned\n" if turned else b"xcorr fused\n")
        lib.dsaxbf_xengine_destroy(x)
        assert live.value == start
