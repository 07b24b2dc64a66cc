"""The work this framework does in use, as cases that can be timed and compared.

One case is one call, or the short run of calls, that a program makes for one
block of data: the coherent beamformer (dsaX_beamformer's block), a change of
pointing, a batch of uneven blocks, the correlator X-engine and the search-side
RFI flagger.  Sizes are the ones the repository runs: the DSA-110 block (63 or 64
antennas x 384 channels x 2048 packets -> 256 beams), the 256-antenna array, the
seeded uneven batch, the 96-antenna correlator, the 64 x 16384 x 1024 filterbank,
and smaller, ragged ones of the same ranges.

Device memory is held in torch tensors, the plans' own streams run the work, and
inputs come from a seeded generator on the GPU: 4-bit complex Gaussian voltages
(sigma 2, clipped at +-7), beam weights of a random east-west array, filterbank
noise of mean 48 and standard deviation 6 with hot channels and bursts.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dsa110-xengine_amd", "python"))
import dsaxbf as bf  # noqa: E402
import dsaxfl as fl  # noqa: E402

PRECISIONS = {"fp16": bf.PREC_FP16, "fp8split": bf.PREC_FP8SPLIT, "fp6split": bf.PREC_FP6SPLIT, "fp6split3": bf.PREC_FP6SPLIT3}
WEIGHT_BYTES = {"fp16": 4.0, "fp8split": 4.0, "fp6split": 3.0, "fp6split3": 4.5}  # one complex weight
LIGHT = 299792458.0
#: Beamformer work of the largest listed case, in antennas x beams x channels x packets: no drawn case has more.
MOST_BEAM_WORK = 256 * 1024 * 384 * 2048


def listed():
    block = {"kind": "beamform", "nant": 64, "nchan": 384, "npkt": 2048, "nbeam": 256, "tavg": 32, "precision": "fp16",
             "fine": False, "sin": True, "split_order": False, "beam_major": False, "stuff": 0, "power": False}
    return [
        # the smallest block the tests and smoke() run: launches and latency
        dict(block, name="beam_small_fp16", nchan=16, npkt=64, tavg=8, fine=True, power=True),
        # the command line's own defaults: 63 antennas, FP16, one weight row per 8 channels, 8-sample bins
        dict(block, name="beam_cli_fp16", nant=63, tavg=8, sin=False),
        # the headline benchmark: FP8 voltages x split weights, one weight row per channel
        dict(block, name="beam_headline_fp8", precision="fp8split", fine=True),
        # `dsaX_split -r` input, beam-major output for the corner turn and the incoherent beam (-r -B -q)
        dict(block, name="beam_incoherent_fp6", precision="fp6split", split_order=True, beam_major=True, stuff=2),
        # a ragged array and beam set, with the unquantised power written too
        dict(block, name="beam_ragged_fp6x3", nant=100, nchan=200, npkt=1056, nbeam=300, tavg=16, precision="fp6split3", fine=True, power=True),
        # the scaled array: 256 antennas to 1024 beams
        dict(block, name="beam_scaled_fp8", nant=256, nbeam=1024, precision="fp8split", fine=True),
        # a new pointing and the first block with it: the weights re-read (-w), then the block
        dict(block, name="beam_repoint_fp16", kind="repoint", fine=True),
        # 24 uneven blocks replayed as one graph
        {"name": "batch_uneven_fp8", "kind": "batch", "nblocks": 24, "shapes": 2025, "precision": "fp8split"},
        # the correlator on the 96-antenna block, and on one node's narrow slice of a 63-antenna one
        {"name": "corr_full", "kind": "correlate", "nant": 96, "nchan": 384, "npkt": 2048, "split_order": False},
        {"name": "corr_slice", "kind": "correlate", "nant": 63, "nchan": 48, "npkt": 1024, "split_order": True},
        # the flagger's loop body on the reference's block: scale, measure, mask, replace, time series, burst rows
        {"name": "flag_step_full", "kind": "flag_step", "nbeam": 64, "ntime": 16384, "nchan": 1024, "tsflag": 1},
        # a caller's own loop over the device entry points, on a narrow filterbank
        {"name": "flag_loop_ragged", "kind": "flag_loop", "nbeam": 12, "ntime": 8192, "nchan": 400},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["beamform"] * 5 + ["repoint", "batch"] + ["correlate"] * 2 + ["flag_step", "flag_loop"])
    if kind in ("beamform", "repoint"):
        while True:
            c = {"kind": kind, "nant": round(_log(rng, 16, 256)), "nchan": 8 * round(_log(rng, 1, 48)), "npkt": 32 * round(_log(rng, 1, 64)),
                 "nbeam": round(_log(rng, 16, 1024)), "tavg": rng.choice([8, 16, 32, 64]), "precision": rng.choice(sorted(PRECISIONS)),
                 "fine": rng.random() < 0.5, "sin": rng.random() < 0.5, "split_order": rng.random() < 0.3,
                 "beam_major": rng.random() < 0.3, "stuff": rng.choice([0, 0, 0, 0, 1, 2]) if kind == "beamform" else 0,
                 "power": rng.random() < 0.3}
            if c["precision"] == "fp6split3" and c["nant"] > 128:
                continue
            if c["nant"] * c["nbeam"] * c["nchan"] * c["npkt"] <= MOST_BEAM_WORK:
                return c
    if kind == "batch":
        return {"kind": kind, "nblocks": rng.randint(3, 24), "shapes": rng.randrange(1 << 16), "precision": rng.choice(sorted(PRECISIONS))}
    if kind == "correlate":
        return {"kind": kind, "nant": round(_log(rng, 8, 96)), "nchan": 8 * round(_log(rng, 1, 48)), "npkt": 32 * round(_log(rng, 1, 64)),
                "split_order": rng.random() < 0.5}
    c = {"kind": kind, "nbeam": round(_log(rng, 2, 64)), "ntime": 4096 * rng.randint(1, 4), "nchan": 16 * rng.randint(18, 64)}
    if kind == "flag_step":
        c["tsflag"] = int(rng.random() < 0.7)
    return c


# ---- inputs -------------------------------------------------------------------

class Dev:
    """A torch tensor as the device buffer that the bindings take."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _zeros(shape, dtype):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _voltages(nbytes, seed):
    """nbytes samples of one byte: re in the low nibble, im in the high one, two's complement."""
    g = _gen(seed)
    out = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    for at in range(0, nbytes, 1 << 26):
        n = min(1 << 26, nbytes - at)
        v = torch.randn((2, n), generator=g, device="cuda").mul_(2.0).round_().clamp_(-7, 7).to(torch.int8)
        out[at:at + n] = ((v[0] & 15) | ((v[1] & 15) << 4)).view(torch.uint8)
    return out


def _geometry(nant, ncal, nbeam, seed):
    r = np.random.default_rng(seed)
    antpos = np.sort(r.uniform(-600.0, 600.0, nant)).astype(np.float32)
    amp, ph = r.uniform(0.9, 1.1, (nant, ncal, 2)), r.uniform(0.0, 2 * np.pi, (nant, ncal, 2))
    cal = np.stack([amp * np.cos(ph), amp * np.sin(ph)], -1).astype(np.float32)
    theta = np.deg2rad(np.linspace(-1.75, 1.75, nbeam) + r.uniform(-0.1, 0.1))
    return antpos, cal, theta


def _freqs(nchan):
    return (1498.75 - np.arange(nchan) * 250.0 / 8192.0) * 1e6


def _scale(nant, nbeam, tavg, seed):
    """The AGC's level of an earlier block: a mean power of about 64 in the output bytes."""
    mean = tavg * 8 * 2 * nant * 2 * 4.0
    r = np.random.default_rng(seed + 1)
    return torch.from_numpy((128.0 / mean * r.uniform(0.95, 1.05, nbeam)).astype(np.float32)).cuda()


def _beam_config(c):
    return bf.config(nant=c["nant"], nchan=c["nchan"], npkt=c["npkt"], nbeam=c["nbeam"], tavg=c["tavg"], precision=PRECISIONS[c["precision"]],
                     weight_mode=bf.WEIGHTS_FINE if c["fine"] else bf.WEIGHTS_GROUP, angle_mode=bf.ANGLE_SIN if c["sin"] else bf.ANGLE_THETA,
                     stuffants=c["stuff"], input_order=bf.ORDER_SPLIT_R if c["split_order"] else bf.ORDER_CAPTURE,
                     output_layout=bf.LAYOUT_BEAM_MAJOR if c["beam_major"] else bf.LAYOUT_TIME_MAJOR)


def _prepare_beam(c, seed):
    cfg = _beam_config(c)
    s = {"case": c, "plan": bf.Plan(cfg), "geometry": _geometry(c["nant"], cfg.ncal, c["nbeam"], seed), "freqs": _freqs(c["nchan"])}
    shape = (cfg.nbeam, cfg.nout, cfg.ngroup) if c["beam_major"] else (cfg.nout, cfg.nbeam, cfg.ngroup)
    s["in"] = Dev(_voltages(bf.input_bytes(cfg), seed))
    s["scale"] = Dev(_scale(c["nant"], c["nbeam"], c["tavg"], seed))
    s["out"], s["beam_power"] = Dev(_zeros(shape, torch.uint8)), Dev(_zeros(c["nbeam"], torch.float32))
    s["power"] = Dev(_zeros(shape, torch.float32)) if c["power"] else None
    if c["kind"] == "beamform":
        antpos, cal, theta = s["geometry"]
        s["plan"].set_weights(antpos, cal, s["freqs"], theta)
    return s


def _batch_cases(c):
    return [{"kind": "beamform", "nant": 64, "nchan": nchan, "npkt": nsamp // 2, "nbeam": nbeam, "tavg": 32, "precision": c["precision"], "fine": True,
             "sin": True, "split_order": False, "beam_major": False, "stuff": 0, "power": False}
            for nchan, nbeam, nsamp in bf.uneven_batch_shapes(c["shapes"], c["nblocks"])]


def _filterbank(c, seed):
    """Scaled filterbank noise with hot channels and a few bright bursts; the reference spectra are its own mean and variance."""
    nb, nt, nc = c["nbeam"], c["ntime"], c["nchan"]
    g = _gen(seed)
    r = np.random.default_rng(seed)
    x = torch.empty((nb, nt, nc), dtype=torch.uint8, device="cuda")
    hot = torch.from_numpy((r.random((nb, nc)) < 0.02) * r.uniform(2.0, 20.0, (nb, nc))).to(device="cuda", dtype=torch.float32)
    for b in range(nb):
        v = torch.randn((nt, nc), generator=g, device="cuda").mul_(6.0).add_(48.0).add_(hot[b])
        for _ in range(2):
            t = int(r.integers(0, nt - 40))
            v[t:t + int(r.integers(4, 40))] += 30.0
        x[b] = v.round_().clamp_(0, 255).to(torch.uint8)
    return x


def _flags(c, seed):
    """3 % of the columns, 1 % of the rows and each beam's level: what the caller's own masks give."""
    r = np.random.default_rng(seed + 2)
    cols, rows = (np.flatnonzero(r.random(c["nbeam"] * n) < share).astype(np.int32) for n, share in ((c["nchan"], 0.03), (c["ntime"], 0.01)))
    return cols, rows, r.uniform(0.95, 1.05, c["nbeam"]).astype(np.float32)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("beamform", "repoint"):
        return _prepare_beam(c, seed)
    if kind == "batch":
        blocks = [_prepare_beam(b, seed + 1000 * k) for k, b in enumerate(_batch_cases(c))]
        batch = bf.Batch([b["plan"] for b in blocks], *([b[k] for b in blocks] for k in ("in", "scale", "out", "beam_power")))
        return {"case": c, "blocks": blocks, "batch": batch, "stream": blocks[0]["plan"].stream}
    if kind == "correlate":
        x = bf.XEngine(c["nant"], c["nchan"], c["npkt"], bf.ORDER_SPLIT_R if c["split_order"] else bf.ORDER_CAPTURE)
        return {"case": c, "plan": x, "in": Dev(_voltages(c["npkt"] * c["nant"] * c["nchan"] * 4, seed)),
                "vis": Dev(_zeros((x.nbase, c["nchan"], 2, 2), torch.float32))}
    nb, nt, nc = c["nbeam"], c["ntime"], c["nchan"]
    s = {"case": c, "block": Dev(_filterbank(c, seed))}
    spec0, var0 = np.full((nb, nc), 48.0, np.float32), np.full((nb, nc), 36.0, np.float32)
    if kind == "flag_step":
        # steady state: the last block's power is known, and a block's own is within 5 % of it
        s["plan"] = fl.Plan(fl.config(nb, nt, nc, tsflag=c["tsflag"], mod_thresh=0.05, seed=1 + seed % 1000))
        s["plan"].set_reference(spec0, var0)
        s["plan"].set_total_power(48.3 * nb * nc)
        return s
    cols, rows, bpwr = _flags(c, seed)
    put = lambda a: Dev(torch.from_numpy(a).cuda())  # noqa: E731
    s |= {"spec0": put(spec0), "var0": put(var0), "cols": put(cols), "ncol": len(cols), "rows": put(rows), "nrow": len(rows), "bpwr": put(bpwr)}
    s |= {k: Dev(_zeros((nb, nc), torch.float32)) for k in ("spec", "var", "pp")}
    s["ts"] = Dev(_zeros((nb, nt), torch.float32))
    return s


# ---- one pass -----------------------------------------------------------------

def run(state):
    s, kind = state, state["case"]["kind"]
    if kind in ("beamform", "repoint"):
        if kind == "repoint":
            antpos, cal, theta = s["geometry"]
            s["plan"].set_weights(antpos, cal, s["freqs"], theta)
        s["plan"].execute(s["in"].ptr.value, s["scale"].ptr.value, s["out"].ptr.value, s["power"] and s["power"].ptr.value, s["beam_power"].ptr.value)
        out = {"out": s["out"].t, "beam_power": s["beam_power"].t}
        return dict(out, power=s["power"].t) if s["power"] else out
    if kind == "batch":
        s["batch"].launch(s["stream"])
        return {"out": [b["out"].t for b in s["blocks"]], "beam_power": [b["beam_power"].t for b in s["blocks"]]}
    if kind == "correlate":
        s["plan"].execute(s["in"], s["vis"])
        return s["vis"].t
    c = s["case"]
    shape = c["nbeam"], c["ntime"], c["nchan"]
    p = lambda k: s[k].ptr.value  # noqa: E731
    if kind == "flag_step":
        info = s["plan"].step(p("block"))
        return {"block": s["block"].t, "tpwr": info.tpwr, "replaced": info.replaced, "n_mask": info.n_mask, "n_tsmask": info.n_tsmask}
    fl.scaley(p("block"), *shape, p("spec0"), p("var0"), p("spec"), p("var"), None, p("pp"))
    fl.flag(p("block"), *shape, p("cols"), s["ncol"], p("bpwr"))
    fl.make_ts(p("block"), *shape, p("ts"))
    fl.flagts(p("block"), *shape, p("rows"), s["nrow"], p("bpwr"))
    return {k: s[k].t for k in ("block", "spec", "var", "pp", "ts")}


def work(case):
    c, kind = case, case["kind"]
    if kind == "batch":
        each = [work(b) for b in _batch_cases(c)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    if kind in ("beamform", "repoint"):
        nin, nout = 4 * c["npkt"] * c["nant"] * c["nchan"], 2 * c["npkt"] // c["tavg"] * c["nbeam"] * (c["nchan"] // 8)
        weights = WEIGHT_BYTES[c["precision"]] * 2 * c["nant"] * c["nbeam"] * (c["nchan"] if c["fine"] else c["nchan"] // 8)
        live = 0 if c["stuff"] == 1 else 1
        return {"bytes": nin + live * weights + nout * (5 if c["power"] else 1) + 8 * c["nbeam"],
                "flops": live * 8.0 * c["nbeam"] * c["nant"] * c["nchan"] * 2 * 2 * c["npkt"]}
    if kind == "correlate":
        nbase = c["nant"] * (c["nant"] + 1) // 2
        return {"bytes": 4 * c["npkt"] * c["nant"] * c["nchan"] + 16 * nbase * c["nchan"], "flops": 8.0 * nbase * c["nchan"] * 2 * 2 * c["npkt"]}
    n = c["nbeam"] * c["ntime"] * c["nchan"]
    return {"bytes": 2 * n + 12 * c["nbeam"] * c["nchan"] + 4 * c["nbeam"] * c["ntime"], "flops": 0}


# ---- in 64 bits ---------------------------------------------------------------

def _decode(raw, c):
    """[nchan][pol][sample][antenna] complex128 of a packed block, a channel at a time."""
    na, nc, npk = c["nant"], c["nchan"], c["npkt"]
    v = raw.view(npk, nc // 8, na, 8, 2, 2).permute(0, 2, 1, 3, 4, 5) if c["split_order"] else raw.view(npk, na, nc // 8, 8, 2, 2)
    for ch in range(nc):
        x = v[:, :, ch // 8, ch % 8].permute(3, 0, 2, 1).reshape(2, 2 * npk, na).to(torch.int32)  # pol, sample, antenna
        re, im = ((x & 15) ^ 8) - 8, ((x >> 4) ^ 8) - 8
        yield torch.complex(re.double(), im.double())


def _exact_beam(c, seed):
    antpos, cal, theta = _geometry(c["nant"], c["nchan"] if c["fine"] else c["nchan"] // 8, c["nbeam"], seed)
    f, x = _freqs(c["nchan"]), torch.from_numpy(antpos).cuda().double()
    ang = torch.from_numpy(np.sin(theta) if c["sin"] else theta).cuda()
    k = torch.from_numpy(cal).cuda().double()
    k = torch.complex(k[..., 0], k[..., 1])
    nout, ng = 2 * c["npkt"] // c["tavg"], c["nchan"] // 8
    power = _zeros((nout, c["nbeam"], ng), torch.float64)
    beam = torch.arange(c["nbeam"], device="cuda")
    ant = ((beam // 16) % 4) * 16 + beam % 16
    for ch, d in enumerate(_decode(_voltages(4 * c["npkt"] * c["nant"] * c["nchan"], seed), c)):
        wc = ch if c["fine"] else ch // 8
        ph = -2.0 * math.pi * f[ch if c["fine"] else ch // 8 * 8 + 4] / LIGHT * ang[None, :] * x[:, None]
        for pol in range(2):
            bins = lambda p: p.view(nout, c["tavg"], -1).sum(1)  # noqa: E731
            if c["stuff"] != 1:
                b = d[pol] @ (torch.polar(torch.ones_like(ph), ph) * k[:, wc, pol, None])
                p = bins(b.real.square() + b.imag.square())
            if c["stuff"]:
                a = bins(d[pol].real.square() + d[pol].imag.square())
                if c["stuff"] == 1:
                    p = torch.where(ant < c["nant"], a[:, ant.clamp(max=c["nant"] - 1)], 0.0)
                else:
                    p[:, 0] = a.sum(1)
            power[:, :, ch // 8] += p
    out = {"out": None, "beam_power": power.sum((0, 2))}
    if c["power"]:
        out["power"] = power.permute(1, 0, 2).contiguous() if c["beam_major"] else power
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("beamform", "repoint"):
        return _exact_beam(c, seed)
    if kind == "batch":
        each = [_exact_beam(b, seed + 1000 * k) for k, b in enumerate(_batch_cases(c))]
        return {"out": [None] * len(each), "beam_power": [e["beam_power"] for e in each]}
    if kind == "correlate":
        i = torch.arange(c["nant"], device="cuda")
        jj, ii = torch.meshgrid(i, i, indexing="xy")  # row i, column j <= i
        low = jj <= ii
        vis = _zeros((c["nant"] * (c["nant"] + 1) // 2, c["nchan"], 2, 2), torch.float64)
        for ch, d in enumerate(_decode(_voltages(c["npkt"] * c["nant"] * c["nchan"] * 4, seed), c)):
            for pol in range(2):
                v = d[pol].T.contiguous() @ d[pol].conj().resolve_conj().contiguous()  # [i][j] = sum of d_i conj(d_j)
                vis[:, ch, pol] = torch.view_as_real(v[low].contiguous())
        return vis
    x = _filterbank(c, seed)
    nb, nt, nc = x.shape
    sums = torch.stack([x[b].double().sum(0) for b in range(nb)])
    if kind == "flag_step":
        return {"block": None, "tpwr": (sums / nt).sum(), "replaced": None, "n_mask": None, "n_tsmask": None}
    mean = sums / nt
    var = torch.stack([(x[b].double() - mean[b]).square().mean(0) for b in range(nb)])
    seg = x.view(nb, 32, nt // 32 // 128, 128, nc).double().sum(3).amax(2) / 128.0
    pp = seg.amax(1) - seg[:, 16:].amin(1)
    cols, _, bpwr = _flags(c, seed)
    flagged = _zeros(nb * nc, torch.bool)
    flagged[torch.from_numpy(cols).long().cuda()] = True
    level = torch.from_numpy(np.floor(48.0 * bpwr.astype(np.float64))).cuda()
    ts = torch.stack([torch.where(m, level[b], x[b].double()).mean(1) for b, m in enumerate(flagged.view(nb, nc))])
    return {"block": None, "spec": mean, "var": var, "pp": pp, "ts": ts}
