"""GPU parity of the search-side RFI flagger (include/dsaxfl.h) against the
oracle's restatement of gpu_flagger.cu (oracle/fl_oracle.c), through the C
ABI.

Bit-exact: spectrum, maxspec, ppspec, make_ts (integer sums), the exact
variance (one rounding of the integer formula), scaley, sumpulse, flag,
flagts, the noise copy, fix_zspec and the whole block step against the oracle
step run with the exact variance.  The reference's float-order varspec is
within 1e-5 relative of the device's.  genrand: the device's FP64 log/cos may
differ from the host's in the last bit, so at most 1e-5 of the bytes may be
1 apart."""
import numpy as np
import pytest

import dsaxfl as fl
from dsaxbf import DeviceBuffer

pytestmark = pytest.mark.gpu


def _dev(a):
    a = np.ascontiguousarray(a)
    d = DeviceBuffer(max(a.nbytes, 16))
    d.upload(a)
    return d


def _get(d, shape, dtype):
    return d.download(np.empty(shape, dtype))


def _block(seed, nb, nt, nc, mean=40.0, sd=9.0):
    rng = np.random.default_rng(seed)
    x = np.clip(np.rint(rng.normal(mean, sd, (nb, nt, nc))), 0, 255).astype(np.uint8)
    x[0, :, nc // 2] = np.minimum(255, x[0, :, nc // 2].astype(int) + 60)    # a hot channel
    x[nb - 1, 1000:1100, :] = 250                                             # a burst
    return x


SHAPES = [(4, 8192, 1024), (3, 4096, 400), (2, 12288, 272)]


@pytest.mark.parametrize("nb,nt,nc", SHAPES)
def test_stats_match_oracle(orc, nb, nt, nc):
    print(f"flagger stats {nb}x{nt}x{nc}", flush=True)
    x = _block(nb + nc, nb, nt, nc)
    d = _dev(x)
    outs = {k: DeviceBuffer(nb * nc * 4) for k in ("spec", "var", "max", "pp")}
    fl.stats(d, nb, nt, nc, d_spec=outs["spec"], d_var=outs["var"], d_max=outs["max"], d_pp=outs["pp"])
    g = {k: _get(v, (nb, nc), np.float32) for k, v in outs.items()}
    spec = orc.fl_stat("spectrum", x)
    assert np.array_equal(g["spec"], spec)
    assert np.array_equal(g["max"], orc.fl_stat("maxspec", x))
    assert np.array_equal(g["pp"], orc.fl_stat("ppspec", x))
    assert np.array_equal(g["var"], orc.fl_stat("varspec_exact", x, spec))
    ref = orc.fl_stat("varspec", x, spec).astype(np.float64)
    assert (np.abs(g["var"] - ref) / ref).max() <= 1e-5
    # varspec with a spectrum argument that is not the mean
    s2 = (spec + np.float32(0.375)).astype(np.float32)
    d_s2 = _dev(s2)
    fl.stats(d, nb, nt, nc, d_var=outs["var"], d_spec_in=d_s2)
    assert np.array_equal(_get(outs["var"], (nb, nc), np.float32), orc.fl_stat("varspec_exact", x, s2))
    assert np.array_equal(_get(d, x.shape, np.uint8), x)            # the block is only read


@pytest.mark.parametrize("nc", [512, 400, 272])
def test_scaley_fused_with_stats_matches_oracle(orc, nc):
    """scaley and the statistics of the scaled block; 400 and 272 channels end
    in a part-filled 256-channel slab, whose lanes past the band must not
    write (the whole block is compared, so a stray byte anywhere fails)."""
    nb, nt = 3, 4096
    print(f"flagger scaley {nb}x{nt}x{nc}", flush=True)
    rng = np.random.default_rng(5)
    x = _block(5, nb, nt, nc)
    spec0 = rng.uniform(20, 60, (nb, nc)).astype(np.float32)
    var0 = rng.uniform(1, 200, (nb, nc)).astype(np.float32)
    var0[0, 0] = 0.0                                     # infinite scale: NaN / saturated bytes
    spec0[1, 7] = float(x[1, :, 7].mean())
    d = _dev(x)
    d_s0, d_v0 = _dev(spec0), _dev(var0)
    outs = {k: DeviceBuffer(nb * nc * 4) for k in ("spec", "var", "pp")}
    fl.scaley(d, nb, nt, nc, d_s0, d_v0, d_spec=outs["spec"], d_var=outs["var"], d_pp=outs["pp"])
    want = orc.fl_scaley(x, spec0, var0)
    got = _get(d, x.shape, np.uint8)
    assert np.array_equal(got, want)
    spec = orc.fl_stat("spectrum", want)
    assert np.array_equal(_get(outs["spec"], (nb, nc), np.float32), spec)
    assert np.array_equal(_get(outs["var"], (nb, nc), np.float32), orc.fl_stat("varspec_exact", want, spec))
    assert np.array_equal(_get(outs["pp"], (nb, nc), np.float32), orc.fl_stat("ppspec", want))
    # without statistics outputs: the scaling alone
    d2 = _dev(x)
    fl.scaley(d2, nb, nt, nc, d_s0, d_v0)
    assert np.array_equal(_get(d2, x.shape, np.uint8), want)


@pytest.mark.parametrize("nc", [1024, 400, 2048])
def test_flag_mask_with_make_ts_matches_oracle(orc, nc):
    nb, nt = 4, 4096
    print(f"flagger flag_mask + make_ts nc={nc}", flush=True)
    rng = np.random.default_rng(6)
    x = _block(6, nb, nt, nc)
    # per beam: no mask, sparse (masked chunks stored alone), 5 % and 50 %
    # (a quarter or more of a row's chunks: whole rows rewritten)
    dens = np.array([0.0, 0.005, 0.05, 0.5])[:, None]
    m = (rng.random((nb, nc)) < dens).astype(np.uint8)
    m[1, 5] = 1
    m[2, 17] = 3                                         # any nonzero byte flags
    bp = np.array([1.0, 1.3, 0.7, 4.9], np.float32)      # 48 * 4.9 = 235.2
    d, d_m, d_bp = _dev(x), _dev(m), _dev(bp)
    d_ts = DeviceBuffer(nb * nt * 4)
    fl.flag_mask(d, nb, nt, nc, d_m, d_bp, d_ts)
    midx = np.flatnonzero(m.ravel()).astype(np.int32)
    want = orc.fl_flag(x, midx, bp)
    assert np.array_equal(_get(d, x.shape, np.uint8), want)
    assert np.array_equal(_get(d_ts, (nb, nt), np.float32), _row_mean(want))
    if nc % 32 == 0:
        assert np.array_equal(_get(d_ts, (nb, nt), np.float32), orc.fl_stat("make_ts", want))
    # make_ts alone reads the block
    d2 = _dev(x)
    fl.make_ts(d2, nb, nt, nc, d_ts)
    assert np.array_equal(_get(d_ts, (nb, nt), np.float32), _row_mean(x))
    if nc % 32 == 0:
        assert np.array_equal(_get(d_ts, (nb, nt), np.float32), orc.fl_stat("make_ts", x))
    assert np.array_equal(_get(d2, x.shape, np.uint8), x)


def _row_mean(x):
    """Every row's exact integer sum over all its channels / nchan, rounded
    once to float.  The reference's make_ts (gpu_flagger.cu:419-429) gives
    each of its 32 threads nchan/32 channels, so it equals this (and the
    oracle) when nchan is a multiple of 32 and leaves the last nchan % 32
    channels out otherwise; the library sums them all."""
    return (x.sum(axis=2, dtype=np.int64) / x.shape[2]).astype(np.float32)


def test_flag_and_flagts_by_index_match_oracle(orc):
    nb, nt, nc = 3, 4096, 512
    print("flagger flag / flagts by index", flush=True)
    rng = np.random.default_rng(7)
    x = _block(7, nb, nt, nc)
    bp = np.array([1.0, 0.5, 2.0], np.float32)
    cols = np.sort(rng.choice(nb * nc, 40, replace=False)).astype(np.int32)
    rows = np.sort(rng.choice(nb * nt, 70, replace=False)).astype(np.int32)
    d, d_bp = _dev(x), _dev(bp)
    fl.flag(d, nb, nt, nc, _dev(np.append(cols, [-1, nb * nc]).astype(np.int32)), len(cols) + 2,
            d_bp)                                               # bad entries skipped
    want = orc.fl_flag(x, cols, bp)
    assert np.array_equal(_get(d, x.shape, np.uint8), want)
    fl.flagts(d, nb, nt, nc, _dev(rows), len(rows), d_bp)
    want = orc.fl_flag(want, rows, bp, ts=True)
    assert np.array_equal(_get(d, x.shape, np.uint8), want)


def test_sumpulse_matches_oracle(orc):
    print("flagger sumpulse", flush=True)
    rng = np.random.default_rng(8)
    n = 1_000_003                                        # a tail past the last 4-byte group
    x = rng.integers(0, 256, n).astype(np.uint8)
    s = rng.normal(0, 80, n).astype(np.float32)
    s[:8] = [0.25, 0.75, 1e12, -1e12, np.inf, -np.inf, np.nan, 127.5]
    d = _dev(x)
    fl.sumpulse(d, n, _dev(s))
    assert np.array_equal(_get(d, n, np.uint8), orc.fl_sumpulse(x, s))


def test_genrand_and_noise_match_oracle(orc):
    print("flagger genrand / noise", flush=True)
    nb, nt, nc = 3, 4096, 512
    n = nt * nc
    d_r = DeviceBuffer(n)
    fl.genrand(d_r, n, 12345)
    got = _get(d_r, n, np.uint8)
    want = orc.fl_genrand(n, 12345)
    diff = np.abs(got.astype(int) - want.astype(int))
    assert diff.max() <= 1 and (diff > 0).mean() <= 1e-5
    x = _block(9, nb, nt, nc)
    d = _dev(x)
    fl.noise(d, nb, nt, nc, d_r)
    assert np.array_equal(_get(d, x.shape, np.uint8), np.broadcast_to(got.reshape(nt, nc), x.shape))


@pytest.mark.parametrize("naver", [1, 3, 4, 5, 16])
def test_fix_zspec_matches_oracle(orc, naver):
    print(f"flagger fix_zspec naver={naver}", flush=True)
    rng = np.random.default_rng(naver)
    nbc = 5000
    s = rng.normal(40, 2, (naver, nbc)).astype(np.float32)
    v = rng.normal(80, 5, (naver, nbc)).astype(np.float32)
    s[:, :100] = np.round(s[:, :100])                    # ties
    d_s, d_v = _dev(s), _dev(v)
    fl.fix_zspec(d_s, d_v, nbc, naver)
    ws, wv = orc.fl_fix_zspec(s, v, naver)
    assert np.array_equal(_get(d_s, (naver, nbc), np.float32), ws)
    assert np.array_equal(_get(d_v, (naver, nbc), np.float32), wv)


def _oracle_reference(orc, blocks):
    """The start-up average: spectrum and exact varspec per block, fix_zspec,
    median_calc."""
    s = np.stack([orc.fl_stat("spectrum", b) for b in blocks])
    v = np.stack([orc.fl_stat("varspec_exact", b, sb) for b, sb in zip(blocks, s)])
    if len(blocks) > 1:
        s, v = orc.fl_fix_zspec(s, v, len(blocks))
    return orc.fl_median_calc(s[0]), orc.fl_median_calc(v[0])


@pytest.mark.parametrize("pwr,mkrand,tsflag,nc", [(1, 0, 1, 1024), (0, 0, 1, 1024), (1, 0, 0, 1024),
                                                  (0, 1, 1, 1024), (1, 0, 1, 512)])
def test_step_matches_oracle(orc, pwr, mkrand, tsflag, nc):
    nb, nt = 4, 8192
    print(f"flagger step pwr={pwr} mkrand={mkrand} tsflag={tsflag} nc={nc}", flush=True)
    cfg = fl.config(nb, nt, nc, pwr=pwr, mkrand=mkrand, tsflag=tsflag, tsthresh=6.0, seed=77)
    plan = fl.Plan(cfg)
    cal = [_block(20 + k, nb, nt, nc) for k in range(3)]
    d_cal = [_dev(b) for b in cal]
    plan.calibrate(d_cal)
    s0, v0 = plan.reference()
    ws0, wv0 = _oracle_reference(orc, cal)
    assert np.array_equal(s0, ws0) and np.array_equal(v0, wv0)
    rep = orc.fl_genrand(nt * nc, 77)
    # first block after calibration: previous total power 0, so noise (as the reference)
    x = _block(30, nb, nt, nc)
    d = _dev(x)
    info = plan.step(d)
    got = _get(d, x.shape, np.uint8)
    assert info.replaced == 1 and info.n_mask == -1
    assert (np.abs(got.astype(int) - np.broadcast_to(rep.reshape(nt, nc), x.shape).astype(int)) <= 1).all()
    # later blocks against the oracle step (exact variance)
    prev = info.tpwr
    bpwr = np.ones(nb, np.float32)
    for k in range(2):
        x = _block(40 + k, nb, nt, nc)
        x[1, :, 300 + k] += 15                          # a channel to mask (small enough to
        #                                                  stay under the power-jump test)
        d = _dev(x)
        info = plan.step(d)
        want, tp, bpwr, nm, nts = orc.fl_step(x, s0, v0, rep, prev, cfg.mod_thresh, cfg.thresh, cfg.tsthresh,
                                              pwr=pwr, mkrand=mkrand, tsflag=tsflag, perm=(10,), bpwr=bpwr,
                                              exact_var=True)
        assert info.tpwr == np.float32(tp) and info.replaced == 0
        assert (info.n_mask, info.n_tsmask) == (nm, nts), k
        got = _get(d, x.shape, np.uint8)
        if mkrand:
            diff = np.abs(got.astype(int) - want.astype(int))
            assert diff.max() <= 1 and (diff > 0).mean() <= 1e-5
        else:
            assert np.array_equal(got, want), (k, int((got != want).sum()))
            assert nm > 0
        prev = info.tpwr
    plan.close()


def test_full_reference_block_subset(orc):
    """The reference's block, 64 beams x 16384 times x 1024 channels (1 GiB),
    through the statistics pass and the fused scaley: beams 0 and 63 cut out
    and checked against the oracle bit for bit, and over the whole block the
    size-independent property that the time series of the scaled block sums
    to the spectrum's total (both integer sums of the same bytes)."""
    nb, nt, nc = 64, 16384, 1024
    print("flagger full block", flush=True)
    n = nb * nt * nc
    d = DeviceBuffer(n)
    fl.genrand(d, n, 99)                                     # N(48, 6) bytes on the device
    outs = {k: DeviceBuffer(nb * nc * 4) for k in ("spec", "var", "max", "pp")}
    fl.stats(d, nb, nt, nc, d_spec=outs["spec"], d_var=outs["var"], d_max=outs["max"], d_pp=outs["pp"])
    g = {k: _get(v, (nb, nc), np.float32) for k, v in outs.items()}
    full = _get(d, n, np.uint8).reshape(nb, nt, nc)
    for bm in (0, nb - 1):
        x = np.ascontiguousarray(full[bm:bm + 1])
        spec = orc.fl_stat("spectrum", x)
        assert np.array_equal(g["spec"][bm:bm + 1], spec), bm
        assert np.array_equal(g["var"][bm:bm + 1], orc.fl_stat("varspec_exact", x, spec)), bm
        assert np.array_equal(g["max"][bm:bm + 1], orc.fl_stat("maxspec", x)), bm
        assert np.array_equal(g["pp"][bm:bm + 1], orc.fl_stat("ppspec", x)), bm
    # scaley with the block's own spectra, then the time series of the result
    d_s0, d_v0 = _dev(g["spec"]), _dev(np.maximum(g["var"], 1.0))
    fl.scaley(d, nb, nt, nc, d_s0, d_v0, d_spec=outs["spec"])
    spec2 = _get(outs["spec"], (nb, nc), np.float32).astype(np.float64)
    d_ts = DeviceBuffer(nb * nt * 4)
    fl.make_ts(d, nb, nt, nc, d_ts)
    ts = _get(d_ts, (nb, nt), np.float32).astype(np.float64)
    assert np.allclose((ts * nc).sum(axis=1), (spec2 * nt).sum(axis=1), rtol=0, atol=0.5)
    scaled0 = _get(d, nt * nc, np.uint8).reshape(1, nt, nc)
    assert np.array_equal(scaled0, orc.fl_scaley(full[:1], g["spec"][:1], np.maximum(g["var"], 1.0)[:1]))
    for b in list(outs.values()) + [d, d_s0, d_v0, d_ts]:
        b.free()


@pytest.mark.parametrize("nb,nc", [(36, 1008), (18, 1008), (9, 1008), (2, 304)])
def test_every_slab_width_matches_oracle(orc, nb, nc):
    """Beam and channel counts on each side of the slab widths' limits (256,
    128, 64 and 32 channels a workgroup, the last slab part-filled): every
    statistic of the block as it is and scaled, and the scaled bytes.  Whole
    numbers: equal."""
    nt = 4096
    print(f"flagger slab widths {nb}x{nt}x{nc}", flush=True)
    rng = np.random.default_rng(nb)
    x = rng.integers(0, 256, (nb, nt, nc), dtype=np.uint8)
    spec0 = rng.uniform(60, 190, (nb, nc)).astype(np.float32)
    var0 = rng.uniform(500, 9000, (nb, nc)).astype(np.float32)
    d = _dev(x)
    outs = {k: DeviceBuffer(nb * nc * 4) for k in ("spec", "var", "max", "pp")}

    def check(got, data, beams):
        for b in beams:
            y = np.ascontiguousarray(data[b:b + 1])
            spec = orc.fl_stat("spectrum", y)
            want = {"spec": spec, "var": orc.fl_stat("varspec_exact", y, spec), "max": orc.fl_stat("maxspec", y),
                    "pp": orc.fl_stat("ppspec", y)}
            for k, v in want.items():
                assert np.array_equal(got[k][b:b + 1], v), (k, b)

    beams = sorted({0, 1, nb // 2, nb - 1})
    fl.stats(d, nb, nt, nc, d_spec=outs["spec"], d_var=outs["var"], d_max=outs["max"], d_pp=outs["pp"])
    check({k: _get(v, (nb, nc), np.float32) for k, v in outs.items()}, x, beams)
    fl.scaley(d, nb, nt, nc, _dev(spec0), _dev(var0), d_spec=outs["spec"], d_var=outs["var"], d_max=outs["max"],
              d_pp=outs["pp"])
    y = _get(d, x.shape, np.uint8)
    for b in beams:
        assert np.array_equal(y[b:b + 1], orc.fl_scaley(x[b:b + 1], spec0[b:b + 1], var0[b:b + 1])), b
    check({k: _get(v, (nb, nc), np.float32) for k, v in outs.items()}, y, beams)


@pytest.mark.parametrize("nb,nt,nc,pwr", [(36, 4096, 720, 0), (18, 4096, 1024, 1), (9, 8192, 1040, 0), (2, 4096, 288, 1),
                                          (1, 4096, 4496, 1)])
def test_step_over_slab_widths_matches_oracle(orc, nb, nt, nc, pwr):
    """The block step where its passes take 256, 128, 64 and 32 channels a
    workgroup (the last slab part-filled), and with more channels than a
    selection keeps in LDS.  Masked columns and rows, bytes, counts and total
    power: equal."""
    print(f"flagger step {nb}x{nt}x{nc} pwr={pwr}", flush=True)
    cfg = fl.config(nb, nt, nc, pwr=pwr, tsflag=1, tsthresh=6.0, mod_thresh=0.5, seed=3, perm=(10, 200, nc - 129, nc - 128))
    plan = fl.Plan(cfg)
    rng = np.random.default_rng(nc)
    x = _block(nc, nb, nt, nc)
    spec0 = (x.mean(axis=1) + rng.normal(0, 0.02, (nb, nc))).astype(np.float32)
    var0 = x.var(axis=1).astype(np.float32)
    x[0, :, 150 + nb] += 12
    x[nb - 1, 2000:2040, 128:] = 200
    plan.set_reference(spec0, var0)
    prev = np.float32(48.0 * nb * nc)
    plan.set_total_power(float(prev))
    d = _dev(x)
    info = plan.step(d)
    want, tp, bpwr, nm, _ = orc.fl_step(x, spec0, var0, np.zeros(nt * nc, np.uint8), prev, cfg.mod_thresh, cfg.thresh,
                                        cfg.tsthresh, pwr=pwr, mkrand=0, tsflag=0, perm=(10, 200, nc - 129, nc - 128),
                                        bpwr=np.ones(nb, np.float32), exact_var=True)
    # the series is the mean over every channel (_row_mean), also where nc % 32 != 0
    rows = np.flatnonzero(orc.fl_mask("simple_tsflag", _row_mean(want), cfg.tsthresh)).astype(np.int32)
    want, nts = orc.fl_flag(want, rows, bpwr, ts=True), len(rows)
    assert (info.replaced, info.n_mask, info.n_tsmask, info.tpwr) == (0, nm, nts, np.float32(tp))
    assert nm > 0 and nts > 0
    assert np.array_equal(_get(d, x.shape, np.uint8), want)
    plan.close()


@pytest.mark.parametrize("jump", [False, True])
def test_step_total_power_at_the_threshold(orc, jump):
    """A power jump so near its threshold that the device's own sum of the
    spectrum and the reference's float sum fall on different sides: the float
    sum decides, as in the oracle."""
    nb, nt, nc = 8, 4096, 1024
    print(f"flagger step at the power threshold jump={jump}", flush=True)
    x = _block(61, nb, nt, nc)
    spec0, var0 = x.mean(axis=1).astype(np.float32), x.var(axis=1).astype(np.float32)
    spec = orc.fl_stat("spectrum", orc.fl_scaley(x, spec0, var0))
    total = np.float32(0)
    for v in spec.ravel():
        total = np.float32(total + v)
    exact = spec.astype(np.float64).sum()
    if jump:                  # the exact sum has not moved, the float sum has
        prev, thr = np.float32(exact), 1e-7
        assert abs(exact - float(prev)) / float(prev) < thr <= abs(float(total) - float(prev)) / float(prev)
    else:                     # the float sum has not moved, the exact sum has
        prev, thr = total, 1e-9
        assert abs(exact - float(prev)) / float(prev) >= thr
    plan = fl.Plan(fl.config(nb, nt, nc, tsflag=1, tsthresh=6.0, mod_thresh=thr, seed=8))
    plan.set_reference(spec0, var0)
    plan.set_total_power(float(prev))
    d = _dev(x)
    info = plan.step(d)
    assert info.tpwr == total and info.replaced == int(jump)
    got = _get(d, x.shape, np.uint8)
    if jump:
        rep = np.broadcast_to(orc.fl_genrand(nt * nc, 8).reshape(nt, nc), x.shape).astype(int)
        assert (np.abs(got.astype(int) - rep) <= 1).all() and (info.n_mask, info.n_tsmask) == (-1, -1)
    else:
        want, _, _, nm, nts = orc.fl_step(x, spec0, var0, np.zeros(nt * nc, np.uint8), prev, thr, 5.0, 6.0, pwr=0, mkrand=0,
                                          tsflag=1, perm=(10,), bpwr=np.ones(nb, np.float32), exact_var=True)
        assert (info.n_mask, info.n_tsmask) == (nm, nts) and np.array_equal(got, want)
    plan.close()


@pytest.mark.parametrize("nc", [16, 256, 272, 512, 528])
def test_row_lanes_at_every_width(orc, nc):
    """flag_mask with make_ts and make_ts alone where 16, 32 and 64 lanes read a
    row, at the widths on each side: bytes and row means equal."""
    nb, nt = 3, 4096
    print(f"flagger row lanes nc={nc}", flush=True)
    rng = np.random.default_rng(nc)
    x = rng.integers(0, 256, (nb, nt, nc), dtype=np.uint8)
    m = (rng.random((nb, nc)) < np.array([0.0, 0.02, 0.4])[:, None]).astype(np.uint8)
    bp = np.array([1.0, 1.3, 0.7], np.float32)
    d, d_ts = _dev(x), DeviceBuffer(nb * nt * 4)
    fl.make_ts(d, nb, nt, nc, d_ts)
    assert np.array_equal(_get(d_ts, (nb, nt), np.float32), _row_mean(x))
    fl.flag_mask(d, nb, nt, nc, _dev(m), _dev(bp), d_ts)
    want = orc.fl_flag(x, np.flatnonzero(m.ravel()).astype(np.int32), bp)
    assert np.array_equal(_get(d, x.shape, np.uint8), want)
    assert np.array_equal(_get(d_ts, (nb, nt), np.float32), _row_mean(want))
