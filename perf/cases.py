"""Timed cases of the matched filter: what a search program has it do.

Each case is one call (or one call plus the upload or the derivative that
belongs to it) through the public classes: ``MatchedFilter.run``,
``HierarchicalFilter.run``, ``run_series``, ``RefineQueue.run_async`` and
``PeakFilter``.  The units are the usual ones of a matched-filter search:
templates of unit norm (``sum |T|^2 = 1``) against spectra of complex N(0, 1)
noise (real and imaginary part of variance 1), so ``|z|`` is a signal-to-noise
ratio, the reporting threshold is 5.5 and a signal has amplitude 8: about 1%
of the white templates, or one chirp in every 16th segment (its neighbours in
the bank respond to it too).

``listed()`` are the named cases, ``draw(rng)`` further ones of the same
ranges, ``prepare`` what the program holds before the call (filter, resident
banks, gate calibration, plan), ``run`` the call, ``exact`` its values in 64
bits without this package, ``work`` the bytes and operations it cannot do
without.
"""
import math

import numpy as np
import torch

SNR = 8.0          # amplitude of the injected signals
DEV = "cuda:0"


# ------------------------------------------------------------------- cases
def listed():
    """The named cases, smallest calls first."""
    return [
        # one segment against one template, both resident: the latency of a
        # call (a follow-up of a single trigger)
        dict(name="one_pair_1024", kind="run", n=1024, nd=1, nt=1, binsize=1024, threshold=5.5, raw=False,
             lo=0, hi=1024, ingest="resident"),
        # a live analysis: each new segment arrives in host memory and is
        # filtered against a small bank, with clustered (8-bin) output, the
        # usable middle of the segment only and the per-template counts
        dict(name="live_segment_4096", kind="run", n=4096, nd=1, nt=37, binsize=512, threshold=5.5, raw=False,
             lo=0, hi=4096, ingest="host"),
        # many short segments (transients) against a bank of short templates,
        # odd counts, results as plain arrays
        dict(name="short_rows_256", kind="run", n=256, nd=64, nt=501, binsize=256, threshold=5.5, raw=True,
             lo=0, hi=256, ingest="resident"),
        # the headline search block
        dict(name="search_block_4096", kind="run", n=4096, nd=16, nt=1024, binsize=4096, threshold=5.5, raw=False,
             lo=0, hi=4096, ingest="resident"),
        # longer segments, the same number of samples in all
        dict(name="long_rows_16384", kind="run", n=16384, nd=16, nt=256, binsize=16384, threshold=5.5, raw=False,
             lo=0, hi=16384, ingest="resident"),
        # lengths past one workgroup's memory
        dict(name="four_step_65536", kind="run", n=65536, nd=4, nt=128, binsize=1024, threshold=5.5, raw=False,
             lo=0, hi=65536, ingest="resident"),
        # minutes-long segments against a few templates
        dict(name="four_step_262144", kind="run", n=262144, nd=2, nt=31, binsize=4096, threshold=5.5, raw=False,
             lo=0, hi=262144, ingest="resident"),
        # the hierarchical search as it is configured by default: FP32 screen,
        # band chosen for the bank
        dict(name="screened_auto_4096", kind="hier", n=4096, nd=16, nt=1024, band=0, precision="fp32",
             threshold=5.5, fd=1e-2),
        # the same block with the matrix-core screen
        dict(name="screened_fp16_4096", kind="hier", n=4096, nd=16, nt=1024, band=512, precision="fp16",
             threshold=5.5, fd=1e-2),
        # a stretch of strain on the device, half-overlapping blocks, the
        # first and last block searched to their edges (three windows)
        dict(name="series_4096", kind="series", n=4096, blocks=16, nt=1024, binsize=4096, threshold=5.5, where="device"),
        # follow-up of a coarse stage: requests of mixed length, a few
        # candidate templates each
        dict(name="refine_queue", kind="queue", requests=4000, threshold=5.5),
        # gradient descent on template spectra: peak values and their gradient
        dict(name="peak_fit_4096", kind="fit", n=4096, nd=64, nt=32, binsize=512, both=False),
    ]


_POINTS = 16 * 1024 * 4096      # samples correlated by the largest listed block


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["run", "run", "run", "hier", "series", "queue", "fit"])
    if kind == "run":
        n = 1 << rng.randint(6, 18)
        points = _POINTS if n <= 65536 else _POINTS // 4
        pairs = min(_log_int(rng, 1, points // n), 32768)
        nd = min(_log_int(rng, 1, max(1.0, math.sqrt(pairs))), pairs)
        nt = max(1, pairs // nd)
        lo, hi = 0, n
        if rng.random() < 0.4:      # the uncorrupted middle, not always aligned
            lo = rng.randint(1, n // 4)
            hi = n - rng.randint(0, n // 4)
        nbins = rng.choice([1, 1, 8, rng.randint(2, 24)])
        while nbins > 1 and nd * nt * nbins > 131072:
            nbins -= 1
        return dict(kind="run", n=n, nd=nd, nt=nt, binsize=max(1, -(-(hi - lo) // nbins)), threshold=5.5,
                    raw=rng.random() < 0.3, lo=lo, hi=hi, ingest=rng.choice(["resident", "resident", "host", "device"]))
    if kind == "hier":
        n = 1 << rng.randint(10, 14)
        pairs = min(_log_int(rng, 64, _POINTS // n), 16384)
        nd = min(_log_int(rng, 1, math.sqrt(pairs)), pairs)
        precision = rng.choice(["fp32", "fp16", "bf16"])
        return dict(kind="hier", n=n, nd=nd, nt=max(1, pairs // nd), threshold=5.5, fd=1e-2, precision=precision,
                    band=512 if precision != "fp32" else rng.choice([0, 0, 128, 256, 512]))
    if kind == "series":
        n = 1 << rng.randint(8, 16)
        blocks = rng.randint(1, 40)
        return dict(kind="series", n=n, blocks=blocks,
                    nt=max(1, min(_log_int(rng, 1, max(1, _POINTS // (n * blocks))), 32768 // blocks)),
                    binsize=n, threshold=5.5, where=rng.choice(["device", "host"]))
    if kind == "queue":
        return dict(kind="queue", requests=_log_int(rng, 3, 3000), threshold=5.5)
    n = 1 << rng.randint(9, 13)
    pairs = _log_int(rng, 4, 64 * 32 * 4096 // n)
    nd = min(_log_int(rng, 1, 64), pairs)
    return dict(kind="fit", n=n, nd=nd, nt=max(1, min(pairs // nd, 4096)), binsize=n // rng.choice([1, 4, 8]),
                both=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _noise(g, rows, n):
    """Spectra of complex N(0, 1) noise (variance 1 per component)."""
    return torch.randn((rows, n), dtype=torch.complex64, device=DEV, generator=g) * math.sqrt(2.0)


def _white_bank(g, nt, n):
    t = torch.randn((nt, n), dtype=torch.complex64, device=DEV, generator=g)
    return t / torch.linalg.vector_norm(t, dim=1, keepdim=True)


def _edges(n):
    """First and last bin of the inspiral band of a length-n spectrum (20 and
    1500 of 4096)."""
    return max(1, n * 20 // 4096), max(2, n * 1500 // 4096)


def _profile(n):
    """Mean power of a chirp spectrum: f^-7/3 inside the band."""
    f = np.arange(n, dtype=np.float64)
    lo, hi = _edges(n)
    return np.where((f >= lo) & (f <= hi), np.where(f > 0, f, 1.0) ** (-7.0 / 3.0), 0.0).astype(np.float32)


def _chirp_bank(g, nt, n):
    """Inspiral-like chirps, amplitude f^-7/6, unit norm."""
    f = torch.arange(n, dtype=torch.float64, device=DEV)
    lo, hi = _edges(n)
    band = (f >= lo) & (f <= hi)
    ff = torch.where(band, f, torch.ones_like(f))
    amp = torch.where(band, ff ** (-7.0 / 6.0), torch.zeros_like(f))
    amp = amp / torch.linalg.vector_norm(amp)
    u = torch.rand((3, nt, 1), dtype=torch.float64, device=DEV, generator=g)
    phase = (2 * math.pi * ff * u[0] + (1e3 + 9e3 * u[1]) * (ff * (4096.0 / n)) ** (-5.0 / 3.0)
             + (2 * u[2] - 1) * ff * (4096.0 / n))
    return torch.polar(amp.expand(nt, n).contiguous(), phase).to(torch.complex64)


def _inject(g, data, bank, count):
    """Adds SNR times `bank[t]`, shifted to a random lag, to every row of
    `data`, for `count` random t each."""
    nd, n = data.shape
    f = torch.arange(n, dtype=torch.int64, device=DEV)
    for _ in range(count):
        t = torch.randint(0, bank.shape[0], (nd,), device=DEV, generator=g)
        lag = torch.randint(0, n, (nd,), device=DEV, generator=g)
        phase = ((f[None, :] * lag[:, None]) % n).to(torch.float64) * (-2.0 * math.pi / n)
        data += (SNR * bank[t] * torch.polar(torch.ones_like(phase), phase)).to(torch.complex64)
    return data


def _pair_inputs(case, seed):
    g = _generator(seed)
    n, nd, nt = case["n"], case["nd"], case["nt"]
    if case["kind"] == "hier":
        bank, data = _chirp_bank(g, nt, n), _noise(g, nd, n)
        _inject(g, data[::16], bank, 1)
    else:
        bank = _white_bank(g, nt, n)
        data = _inject(g, _noise(g, nd, n), bank, max(1, nt // 100))
    return data, bank


def _series_inputs(case, seed):
    """A real-valued stretch of noise with one template added per block, the
    bank, and the half-overlapping layout: the middle half of every block,
    the first from its start and the last to its end."""
    g = _generator(seed)
    n, blocks, nt = case["n"], case["blocks"], case["nt"]
    bank = _white_bank(g, nt, n)
    # block spectra are FFT/n, so noise of variance 2n per sample gives
    # spectra of complex N(0, 1)
    x = torch.randn(blocks * n // 2 + n // 2, dtype=torch.float32, device=DEV, generator=g) * math.sqrt(2.0 * n)
    x = x.to(torch.complex64)
    wave = torch.fft.ifft(bank[:blocks]) * (SNR * n)
    for b in range(wave.shape[0]):
        x[b * n // 2:b * n // 2 + n] += wave[b]
    starts = np.arange(blocks, dtype=np.int64) * (n // 2)
    lo = np.full(blocks, n // 4, np.int64)
    hi = np.full(blocks, 3 * n // 4, np.int64)
    lo[0], hi[-1] = 0, n
    return x, bank, starts, lo, hi


def _queue_inputs(case, seed):
    """Requests of length 1024, 4096, 16384 and 65536 (weights .4/.3/.2/.1)
    with geometric(1/3) candidates, back to back in one pool: each data
    spectrum is noise with the first candidate at SNR 8.  The layout belongs
    to the case, the spectra and lags to the seed."""
    nreq = case["requests"]
    rng = np.random.default_rng(nreq)
    n = rng.choice(np.array([1024, 4096, 16384, 65536], np.int64), size=nreq, p=[.4, .3, .2, .1])
    cand = np.minimum(rng.geometric(1.0 / 3.0, size=nreq), 16).astype(np.int64)
    doff = np.concatenate([[0], np.cumsum(n * (1 + cand))[:-1]]).astype(np.int64)
    lag = np.random.default_rng(seed).integers(0, n)
    g = _generator(seed)
    pool = torch.randn(int((n * (1 + cand)).sum()), dtype=torch.complex64, device=DEV, generator=g)
    for length in (1024, 4096, 16384, 65536):
        rows = np.nonzero(n == length)[0]
        f = torch.arange(length, device=DEV)
        for part in np.array_split(rows, max(1, len(rows) * length // (1 << 24))):
            if not len(part):
                continue
            base = torch.from_numpy(doff[part]).to(DEV)[:, None]
            k = torch.from_numpy(lag[part]).to(DEV)[:, None]
            phase = ((f[None, :] * k) % length).to(torch.float64) * (-2.0 * math.pi / length)
            first = pool[base + length + f] / math.sqrt(length)
            pool[base + f] = (pool[base + f] * math.sqrt(2.0)
                              + (SNR * first * torch.polar(torch.ones_like(phase), phase)).to(torch.complex64))
            # scale each request's candidates to unit norm on average
            for j in range(int(cand[part].max())):
                sub = part[cand[part] > j]
                at = torch.from_numpy(doff[sub]).to(DEV)[:, None] + (1 + j) * length + f
                pool[at] = pool[at] / math.sqrt(length)
    plan = dict(n=n, data_offset=doff, template_offset=doff + n, candidates=cand, binsize=n // 8,
                threshold=case["threshold"])
    return pool, plan


def prepare(case, seed):
    """Filter, resident banks and whatever else the program keeps."""
    import apogee_amd as mf
    kind = case["kind"]
    if kind == "run":
        data, bank = _pair_inputs(case, seed)
        f = mf.MatchedFilter(case["n"], case["nd"], case["nt"])
        f.set_templates(bank)
        state = dict(case=case, filter=f, bank=bank)
        if case["ingest"] == "host":
            state["data"] = data.cpu().numpy()
        else:
            state["data"] = data
            f.set_data(data)
        return state
    if kind == "hier":
        data, bank = _pair_inputs(case, seed)
        f = mf.HierarchicalFilter(case["n"], case["nd"], case["nt"], snr=5.5, fd=case["fd"],
                                  band=case["band"] or None)
        f.set_reference(_profile(case["n"]))
        f.set_coarse_precision(case["precision"])
        f.set_templates(bank)
        f.set_data(data)
        f.coarse_threshold      # calibrated once per bank
        return dict(case=case, filter=f, bank=bank, data=data)
    if kind == "series":
        x, bank, starts, lo, hi = _series_inputs(case, seed)
        f = mf.MatchedFilter(case["n"], 1, case["nt"])
        f.set_templates(bank)
        return dict(case=case, filter=f, bank=bank, layout=(starts, lo, hi),
                    series=x if case["where"] == "device" else x.cpu().numpy())
    if kind == "queue":
        pool, plan = _queue_inputs(case, seed)
        q = mf.RefineQueue()
        q.plan(pool, **plan)
        return dict(case=case, queue=q, pool=pool,
                    index=torch.empty(q.total, dtype=torch.int64, device=DEV),
                    value=torch.empty(q.total, dtype=torch.complex64, device=DEV))
    from apogee_amd.autograd import PeakFilter
    g = _generator(seed)
    data = _noise(g, case["nd"], case["n"])
    bank = _white_bank(g, case["nt"], case["n"])
    return dict(case=case, filter=PeakFilter(case["n"], case["nd"], case["nt"]),
                data=data.requires_grad_(case["both"]), bank=bank.requires_grad_(True))


# ------------------------------------------------------------------- calls
def run(state):
    """One pass through the public entry points."""
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        f = state["filter"]
        if case["ingest"] != "resident":
            f.set_data(state["data"])
        out = f.run(binsize=case["binsize"], threshold=case["threshold"], window=(case["lo"], case["hi"]),
                    raw=case["raw"], counts=case["ingest"] == "host")
        if case["ingest"] == "host":
            body, counts = out
            return _peaks(body, case["raw"]) + (counts,)
        return _peaks(out, case["raw"])
    if kind == "hier":
        return _peaks(state["filter"].run(threshold=case["threshold"]), False)
    if kind == "series":
        starts, lo, hi = state["layout"]
        return _peaks(state["filter"].run_series(state["series"], starts, lo, hi, binsize=case["binsize"],
                                                 threshold=case["threshold"]), False)
    if kind == "queue":
        q = state["queue"]
        q.run_async(state["index"], state["value"])
        q.sync()
        return state["index"], state["value"]
    value, index = state["filter"](state["data"], state["bank"], binsize=case["binsize"])
    loss = -(value.abs() ** 2).sum()
    wrt = (state["data"], state["bank"]) if case["both"] else (state["bank"],)
    return (index, value.detach()) + torch.autograd.grad(loss, wrt)


def _peaks(out, raw):
    return tuple(out) if raw else (out["index"], out["value"])


# ------------------------------------------------------- values in 64 bits
def _select(z, binsize, threshold, lo, hi):
    """Loudest sample per bin of `z` (..., n) over lags [lo, hi), 0 where
    nothing exceeds the threshold."""
    z = z[..., lo:hi]
    nb = -(-(hi - lo) // binsize)
    z = torch.nn.functional.pad(z, (0, nb * binsize - (hi - lo)))
    z = z.reshape(z.shape[:-1] + (nb, binsize))
    best, at = z.abs().max(dim=-1, keepdim=True)
    return torch.where(best > threshold, torch.gather(z, -1, at), torch.zeros_like(best, dtype=z.dtype))[..., 0]


def _exact_pairs(data, bank, binsize, threshold, lo, hi):
    n = data.shape[1]
    data = data.to(torch.complex128)
    step = max(1, (1 << 25) // (data.shape[0] * n))
    parts = []
    for t in range(0, bank.shape[0], step):
        z = torch.fft.ifft(data[:, None, :] * bank[None, t:t + step].to(torch.complex128).conj()) * n
        parts.append(_select(z, binsize, threshold, lo, hi))
    return torch.cat(parts, dim=1)


def exact(case, seed):
    """What `run` returns, in 64 bits; None for lags, and for the
    hierarchical filter, whose omissions depend on its calibrated gate."""
    kind = case["kind"]
    if kind == "hier":
        return None
    if kind == "run":
        data, bank = _pair_inputs(case, seed)
        value = _exact_pairs(data, bank, case["binsize"], case["threshold"], case["lo"], case["hi"]).cpu().numpy()
        return (None, value, None) if case["ingest"] == "host" else (None, value)
    if kind == "series":
        x, bank, starts, lo, hi = _series_inputs(case, seed)
        n = case["n"]
        x = torch.nn.functional.pad(x.to(torch.complex128), (0, n))
        rows = [_exact_pairs((torch.fft.fft(x[s:s + n]) / n)[None], bank, case["binsize"], case["threshold"],
                             int(a), int(b)) for s, a, b in zip(starts, lo, hi)]
        return None, torch.cat(rows).cpu().numpy()
    if kind == "queue":
        pool, plan = _queue_inputs(case, seed)
        parts = []
        for n, doff, toff, c in zip(*(plan[k].tolist() for k in ("n", "data_offset", "template_offset", "candidates"))):
            parts.append(_exact_pairs(pool[doff:doff + n][None], pool[toff:toff + c * n].reshape(c, n), n // 8,
                                      case["threshold"], 0, n).reshape(-1))
        return None, torch.cat(parts)
    g = _generator(seed)
    data = _noise(g, case["nd"], case["n"]).to(torch.complex128).requires_grad_(case["both"])
    bank = _white_bank(g, case["nt"], case["n"]).to(torch.complex128).requires_grad_(True)
    n = case["n"]
    z = torch.fft.ifft(data[:, None, :] * bank[None].conj()) * n
    value = _select(z, case["binsize"], 0.0, 0, n)
    wrt = (data, bank) if case["both"] else (bank,)
    grads = torch.autograd.grad(-(value.abs() ** 2).sum(), wrt)
    return (None, value.detach()) + tuple(x.resolve_conj() for x in grads)


# -------------------------------------------------------------------- work
def _pair_flops(n):
    """Product, inverse transform and |z|^2 of one pair."""
    return 6 * n + 5 * n * math.log2(n) + 3 * n


def work(case):
    """Bytes and operations of one pass: each input read once, each 16-byte
    result written once."""
    kind = case["kind"]
    if kind == "run":
        n, nd, nt = case["n"], case["nd"], case["nt"]
        cells = nd * nt * -(-(case["hi"] - case["lo"]) // case["binsize"])
        return {"bytes": 8 * n * (nd + nt) + 16 * cells, "flops": nd * nt * _pair_flops(n)}
    if kind == "hier":
        # the screen reads one band of every row; only the pairs of a segment
        # that carries a signal need their whole spectra
        n, nd, nt = case["n"], case["nd"], case["nt"]
        band = case["band"] or 128
        rows = -(-nd // 16)
        return {"bytes": 8 * band * (nd + nt) + 8 * n * (rows + nt) + 16 * nd * nt,
                "flops": nd * nt * _pair_flops(band) + rows * nt * _pair_flops(n)}
    if kind == "series":
        n, blocks, nt = case["n"], case["blocks"], case["nt"]
        samples = blocks * n // 2 + n // 2
        return {"bytes": 8 * samples + 8 * n * nt + 16 * blocks * nt,
                "flops": blocks * 5 * n * math.log2(n) + blocks * nt * _pair_flops(n)}
    if kind == "queue":
        # expected pool: three candidates per request over the length mix
        mix = {1024: .4, 4096: .3, 16384: .2, 65536: .1}
        r = case["requests"]
        return {"bytes": r * (sum(w * 8 * 4 * n for n, w in mix.items()) + 3 * 8 * 16),
                "flops": r * 3 * sum(w * _pair_flops(n) for n, w in mix.items())}
    n, nd, nt = case["n"], case["nd"], case["nt"]
    bins = n // case["binsize"]
    sides = 2 if case["both"] else 1
    return {"bytes": 8 * n * (nd + nt) * 2 + 8 * n * (nd + nt if case["both"] else nt) + 32 * nd * nt * bins,
            "flops": nd * nt * _pair_flops(n) + sides * 8 * nd * nt * bins * n}
