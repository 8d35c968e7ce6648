"""The work a program has this library do, as cases that can be timed and compared.

Every case goes through the public entry points (``fdas_amd.host.FDAS``, ``fdas_amd.engine.Engine``,
``fdas_amd.io.FrontEnd`` and the C ABI's ``fdas_hsum_noalloc``).  Spectra are white noise of unit mean power
with up to two drifting tones, thresholds the six-sigma rule of ``synth.noise_thresholds``, banks the drift grid
z = 2 (j - c); sizes are those of the tests and of ``bench.py`` (emulator size 32,768 bins, full trials of
2^19 .. 2^22) and odd ones between.  Tile, rows per item and rows per summing workgroup of an engine are
fixed, as in a program that reads a tuning cache, so that no pass depends on an autotuner's timings.

``exact`` gives the same outputs in 64 bits.  A candidate list of thousands of noise entries per plane has
no such value: which of two neighbours at its cut it keeps, and so where every later entry stands, is
decided by FP32 rounding; lists of at most 512 entries per plane are far enough apart.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from fdas_amd import _native, synth
from fdas_amd.engine import Engine, Trial
from fdas_amd.host import FDAS, make_drift_bank
from fdas_amd.io import FrontEnd

MAX_TAPS = 421
NOISE_SIGMA = 6.0
EXACT_LIST = 512  # longest per-plane list that exact() lays out


def listed():
    return [
        # The smallest call: a short ragged spectrum, few templates, host in and lists out; launches and
        # latency decide.
        {"name": "launch_n4999", "kind": "launch", "n": 4999, "templates": 33, "harmonics": 4, "tile": 1024,
         "cap": 64, "part": 2, "sets": 1},
        # One emulator-size trial through the drop-in class at its defaults (2048-point tiles, 85 templates,
        # 8 planes, 512 per plane): the host flow of a program written against the reference.
        {"name": "launch_n32768", "kind": "launch", "n": 32768, "templates": 85, "harmonics": 8, "tile": 2048,
         "cap": 512, "part": 2, "sets": 1},
        # Two ragged mid-size trials pipelined over the buffer sets A and B, spectra already on the GPU, the
        # non-negative drifts only.
        {"name": "resident_n700001_ab", "kind": "resident", "n": 700001, "templates": 85, "harmonics": 8,
         "tile": 2048, "cap": 512, "part": 1, "sets": 2},
        # One full trial, spectrum on the GPU, one launch and one wait: what a search of single trials costs.
        {"name": "resident_n2p21", "kind": "resident", "n": 1 << 21, "templates": 85, "harmonics": 8,
         "tile": 1024, "cap": 4096, "part": 2, "sets": 1},
        # The staged calls with the long bank and the largest tile, tiles and the whole plane read back: how a
        # program checks a bank, or takes the plane elsewhere.
        {"name": "stages_n20011_t169", "kind": "stages", "n": 20011, "templates": 169, "tile": 4096, "part": 2},
        # Thresholds taken from the data (about 256 candidates per plane), then the search with them.
        {"name": "quantile_n2p18", "kind": "quantile", "n": 1 << 18, "templates": 85, "harmonics": 8,
         "tile": 2048, "cap": 512, "part": 2, "per_plane": 256},
        # Summing and selection alone over a plane in the caller's memory, ragged length (no row is aligned).
        {"name": "hsum_n100003", "kind": "hsum", "n": 100003, "templates": 85, "harmonics": 8, "cap": 512,
         "part": 2},
        # The batched throughput form: 16 full trials in groups of 8.
        {"name": "batch16_n2p21", "kind": "plan", "mix": ",".join(["2097152:85:8"] * 16), "graph": False},
        # An uneven batch as a replayed graph: sizes, banks and plane counts mixed.
        {"name": "uneven8_graph", "kind": "plan", "graph": True,
         "mix": "524288:85:8,524288:169:16,1048576:85:16,1048576:169:8,2097152:85:8,700001:85:8,2097152:169:8,"
                "4194304:85:16"},
        # A burst of requests to the server.
        {"name": "served12", "kind": "served",
         "mix": "1048576:85:8,2097152:169:8,2097152:85:8,1048576:169:8,2097152:85:8,4194304:85:8,1048576:85:8,"
                "2097152:169:8,1048576:85:8,2097152:85:8,1048576:169:8,2097152:85:8"},
        # Front end, largest series, GPU to GPU: upstream of every resident search.
        {"name": "frontend_n2p22", "kind": "frontend", "n": 1 << 22, "host": False},
        # Front end, a short series.
        {"name": "frontend_n2p15", "kind": "frontend", "n": 1 << 15, "host": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["launch", "resident", "stages", "quantile", "hsum", "plan", "served", "frontend"])
    part = rng.choice([0, 1, 2, 2])
    templates = rng.choice([33, 85, 85, 169])
    harmonics = rng.choice([4, 8, 8, 16])
    tile = rng.choice([1024, 2048, 2048, 4096])
    if kind in ("launch", "resident"):
        # the 32-bit lists hold up to 127 templates and 8 planes
        lo, hi = (4000, 300_000) if kind == "launch" else (30_000, 1 << 21)
        return {"kind": kind, "n": _log_int(rng, lo, hi), "templates": min(templates, 85),
                "harmonics": min(harmonics, 8), "tile": tile, "cap": rng.choice([64, 512]), "part": part,
                "sets": rng.choice([1, 2])}
    if kind == "stages":
        return {"kind": kind, "n": _log_int(rng, 4000, 60_000), "templates": templates, "tile": tile, "part": part}
    if kind == "quantile":
        return {"kind": kind, "n": _log_int(rng, 20_000, 600_000), "templates": templates, "harmonics": harmonics,
                "tile": tile, "cap": 512, "part": part, "per_plane": rng.randint(50, 400)}
    if kind == "hsum":
        n = _log_int(rng, 5000, 300_000)
        return {"kind": kind, "n": n - n % 8 if rng.random() < 0.5 else n, "templates": templates,
                "harmonics": harmonics, "cap": rng.choice([64, 512]), "part": part}
    if kind in ("plan", "served"):
        mix = []
        for _ in range(rng.randint(3, 9)):
            n = rng.choice([1 << 18, 1 << 19, 1 << 20, 1 << 21, _log_int(rng, 50_000, 2_000_000)])
            mix.append("%d:%d:%d" % (n, rng.choice([85, 85, 169]), rng.choice([8, 8, 16])))
        case = {"kind": kind, "mix": ",".join(mix)}
        if kind == "plan":
            case["graph"] = rng.random() < 0.5
        return case
    n = 1 << rng.randint(10, 22)
    return {"kind": kind, "n": n, "host": n in (1 << 15, 1 << 22) or rng.random() < 0.3}


# --------------------------------------------------------------------------- inputs


def _workload(n, templates, seed):
    """White noise with 0-2 drifting tones of 8 harmonics.  A tone of amplitude A stands at A^2 n / 2 times
    the noise's mean power: 20 .. 100 for short series (the emulator workload's is 41), up to 400 for full
    trials (bench.py's lie between 105 and 943)."""
    r = np.random.default_rng([seed, n, templates])
    top = min(400.0, max(100.0, n / 5000.0))
    tones = [synth.Tone(float(r.uniform(0.02, 0.9) * n), float(r.uniform(1 - templates, templates - 1)), 8,
                        math.sqrt(2.0 * float(r.uniform(20.0, top)) / n)) for _ in range(int(r.integers(0, 3)))]
    return synth.Workload("trial", n, int(r.integers(1, 1 << 40)), tones)


def _spectrum(n, templates, seed):
    """The trial's spectrum, normalised to unit mean noise power."""
    return (synth.device_spectrum(_workload(n, templates, seed)) * math.sqrt(2.0 * n)).contiguous()


def _noise_thresholds(x, harmonics):
    """synth.noise_thresholds with the mean taken on the GPU."""
    p = float((x.real.double() ** 2 + x.imag.double() ** 2).mean())
    k = np.arange(1, harmonics + 1, dtype=np.float64)
    return ((k + NOISE_SIGMA * np.sqrt(k)) * p).astype(np.float32)


def _bank(templates):
    return make_drift_bank(synth.drift_grid(templates), MAX_TAPS)


def _plane(case, seed):
    """A filter-output plane: exponential noise of unit mean and two drifting tones with their harmonics."""
    n, T = case["n"], case["templates"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    fop = torch.empty((T, n), dtype=torch.float32, device="cuda").exponential_(generator=g)
    r = np.random.default_rng([seed, n, T])
    for _ in range(2):
        f0, z = r.uniform(0.02, 0.12) * n, r.uniform(-T / 16, T / 16)
        for h in range(1, 9):
            row, f = int(T // 2 + h * z), int(h * f0)
            for dr in range(-2, 3):
                if 0 <= row + dr < T and f + 8 < n:
                    fop[row + dr, f:f + 8] += float(r.uniform(5.0, 30.0)) / (1 + abs(dr))
    return fop


def _context(case, n_harmonics=8, cap=512):
    f = FDAS(log=lambda level, message: None)
    if not f.initialise_accelerator(case["n"], n_templates=case["templates"], max_taps=MAX_TAPS, tile=case["tile"],
                                    n_harmonics=n_harmonics, cands_per_harmonic=cap):
        raise RuntimeError("the accelerator could not be initialised")
    bank = _bank(case["templates"])
    for ab in range(case.get("sets", 1)):
        _ok(f, f.upload_template_taps(bank, ab))
    return f


def _ok(f, good):
    if not good:
        raise RuntimeError(f.last_error)


def _mix(case):
    return [tuple(int(v) for v in one.split(":")) for one in case["mix"].split(",")]


def _rows(templates, part):
    """First row and row count of a part."""
    c = templates // 2
    return {0: (0, c + 1), 1: (c, c + 1), 2: (0, templates)}[part]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("launch", "resident"):
        f = _context(case, case["harmonics"], case["cap"])
        spectra = [_spectrum(case["n"], case["templates"], seed + 1000003 * s) for s in range(case["sets"])]
        thresholds = [_noise_thresholds(x, case["harmonics"]) for x in spectra]
        if kind == "launch":
            spectra = [x.cpu().numpy() for x in spectra]
        size = f.get_candidate_list_sz()
        lists = [(np.zeros(size, np.uint32), np.zeros(size, np.float32)) for _ in spectra]
        torch.cuda.synchronize()
        return {"case": case, "fdas": f, "spectra": spectra, "thresholds": thresholds, "lists": lists}
    if kind == "stages":
        f = _context(case)
        x = _spectrum(case["n"], case["templates"], seed).cpu().numpy()
        return {"case": case, "fdas": f, "x": x, "tiles": np.zeros(f.get_tiles_sz(), np.complex64),
                "fop": np.zeros(f.get_fop_sz(), np.float32)}
    if kind == "quantile":
        f = _context(case, case["harmonics"], case["cap"])
        x = _spectrum(case["n"], case["templates"], seed)
        torch.cuda.synchronize()
        return {"case": case, "fdas": f, "x": x}
    if kind == "hsum":
        H, cap = case["harmonics"], case["cap"]
        k = np.arange(1, H + 1, dtype=np.float64)
        return {"case": case, "fop": _plane(case, seed), "log": _native.LOG_FN(lambda level, message, user: None),
                "thresholds": (k + NOISE_SIGMA * np.sqrt(k)).astype(np.float32),
                "key": torch.zeros(H * cap, dtype=torch.int32, device="cuda"),
                "power": torch.zeros(H * cap, dtype=torch.float32, device="cuda"),
                "counts": torch.zeros(2 * H, dtype=torch.int32, device="cuda")}
    if kind in ("plan", "served"):
        eng = Engine(tile=1024, rows_per_item=16, hsum_rows=11, log=lambda level, message: None)
        banks, trials = {}, []
        for i, (n, T, H) in enumerate(_mix(case)):
            if T not in banks:
                banks[T] = eng.add_bank(_bank(T))
            x = _spectrum(n, T, seed + 1000003 * i)
            trials.append(Trial(x, banks[T], _noise_thresholds(x, H), FDAS.AllAccelerations, tag=i))
            eng.prepare(n, banks[T])
        torch.cuda.synchronize()
        state = {"case": case, "engine": eng, "trials": trials}
        if kind == "plan":
            state["plan"] = eng.plan(trials, graph=case["graph"])
        return state
    n = case["n"]
    series = synth.device_series(_workload(n, 85, seed))
    state = {"case": case, "front": FrontEnd(n)}
    if case["host"]:
        state["series"] = series.cpu().numpy()
    else:
        state["series"], state["out"] = series, torch.zeros(n, dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    return state


# --------------------------------------------------------------------------- one pass


def _trial_outputs(results, cap):
    """Per trial: the plane-major lists, each plane's padded to `cap` entries, and the detections per plane."""
    out = []
    for r in results:
        key = np.zeros((len(r.keys), cap), np.uint32)
        power = np.full(key.shape, -1.0, np.float32)
        for p, (k, v) in enumerate(zip(r.keys, r.powers)):
            key[p, :len(k)] = k
            power[p, :len(v)] = v
        out.append({"key": key, "power": power, "detected": r.n_detected})
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    f = state.get("fdas")
    if kind == "launch":
        for ab, (x, thr, (loc, pwr)) in enumerate(zip(state["spectra"], state["thresholds"], state["lists"])):
            _ok(f, f.launch(x, thr, loc, pwr, case["part"], ab))
        for ab in range(case["sets"]):
            _ok(f, f.wait(ab))
        return [{"location": loc, "power": pwr} for loc, pwr in state["lists"]]
    if kind == "resident":
        for ab, (x, thr, (loc, pwr)) in enumerate(zip(state["spectra"], state["thresholds"], state["lists"])):
            _ok(f, f.set_input_device(x.data_ptr(), ab))
            _ok(f, f.launch_resident(thr, loc, pwr, case["part"], ab))
        for ab in range(case["sets"]):
            _ok(f, f.wait(ab))
        return [{"location": loc, "power": pwr} for loc, pwr in state["lists"]]
    if kind == "stages":
        _ok(f, f.perform_input_tiling(state["x"], FDAS.A))
        _ok(f, f.perform_ft_convolution(case["part"], FDAS.A))
        _ok(f, f.retrieve_tiles(state["tiles"], FDAS.A))
        _ok(f, f.retrieve_FOP(state["fop"], FDAS.A))
        return {"tiles": state["tiles"], "fop": state["fop"]}
    if kind == "quantile":
        _ok(f, f.set_input_device(state["x"].data_ptr(), FDAS.A))
        _ok(f, f.perform_ft_convolution(case["part"], FDAS.A))
        thr = f.quantile_thresholds(case["per_plane"], case["part"], FDAS.A)
        if thr is None:
            raise RuntimeError(f.last_error)
        _ok(f, f.perform_harmonic_summing(thr, case["part"], FDAS.A))
        harmonic, template, freq, power, detected = f.retrieve_candidates_wide(FDAS.A)
        return {"thresholds": thr, "harmonic": harmonic, "template": template, "bin": freq, "power": power,
                "detected": detected}
    if kind == "hsum":
        # the spill the default rule would take, within the entry point's fixed scratch
        H, cap = case["harmonics"], case["cap"]
        status = _native.load().fdas_hsum_noalloc(
            ctypes.c_void_p(state["fop"].data_ptr()), case["n"], case["templates"], case["part"], H,
            _native.fptr(state["thresholds"]), cap, 262144 if H <= 8 else 131072,
            ctypes.c_void_p(state["key"].data_ptr()), ctypes.c_void_p(state["power"].data_ptr()),
            ctypes.c_void_p(state["counts"].data_ptr()),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), state["log"], None)
        if status != _native.FDAS_OK:
            raise RuntimeError(f"fdas_hsum_noalloc: status {status}")
        return {"key": state["key"], "power": state["power"], "counts": state["counts"]}
    if kind == "plan":
        return _trial_outputs(state["plan"].run(), state["engine"].cap)
    if kind == "served":
        for t in state["trials"]:
            state["engine"].submit(t)
        return _trial_outputs(sorted(state["engine"].drain(), key=lambda r: r.tag), state["engine"].cap)
    if case["host"]:
        return state["front"].run(state["series"])
    return state["front"].run(state["series"], out=state["out"])


# --------------------------------------------------------------------------- what a pass cannot do without


def _conv_flops(n, rows):
    """Overlap-save convolution of `rows` templates: the inverse transform of a 1024-point tile per
    five-sixths of its points, the spectrum product and |x|^2."""
    return n * rows * (1.2 * 5 * 10 + 1.2 * 6 + 3)


def _search_work(n, templates, harmonics, cap, part):
    rows = _rows(templates, part)[1]
    return {"bytes": 8 * n + 8 * templates * MAX_TAPS + 8 * harmonics * cap,
            "flops": _conv_flops(n, rows) + n * rows * (2 * harmonics - 1)}


def work(case):
    kind = case["kind"]
    if kind in ("launch", "resident", "quantile"):
        w = _search_work(case["n"], case["templates"], case["harmonics"], case["cap"], case["part"])
        return {k: v * case.get("sets", 1) for k, v in w.items()}
    if kind == "stages":
        n, rows = case["n"], _rows(case["templates"], case["part"])[1]
        tiles = -(-n // (case["tile"] - MAX_TAPS + 1)) * case["tile"]
        return {"bytes": 8 * n + 8 * case["templates"] * MAX_TAPS + 8 * tiles + 4 * case["templates"] * n,
                "flops": _conv_flops(n, rows) + 5 * tiles * math.log2(case["tile"])}
    if kind == "hsum":
        n, rows, H = case["n"], _rows(case["templates"], case["part"])[1], case["harmonics"]
        return {"bytes": 4 * n * rows + 8 * H * case["cap"], "flops": n * rows * (2 * H - 1)}
    if kind in ("plan", "served"):
        each = [_search_work(n, T, H, 4096, 2) for n, T, H in _mix(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    n = case["n"]
    return {"bytes": 8 * n + 8 * n, "flops": 5 * n * math.log2(n) + 14 * n}


# --------------------------------------------------------------------------- the same in 64 bits


def _exact_fop(x, case):
    """FOP[r][f] = |sum_m taps[r][m] X[f - m]|^2 in FP64, rows outside the part zero."""
    n, T = case["n"], case["templates"]
    size = 1 << (n + MAX_TAPS - 1).bit_length()
    spec = torch.fft.fft(x.to(torch.complex128), size)
    taps = torch.from_numpy(_bank(T)).to("cuda", torch.complex128)
    fop = torch.zeros((T, n), dtype=torch.float64, device="cuda")
    begin, count = _rows(T, case["part"])
    for r in range(begin, begin + count):
        y = torch.fft.ifft(spec * torch.fft.fft(taps[r], size))[:n]
        fop[r] = y.real ** 2 + y.imag ** 2
    return fop


def _exact_planes(fop, case):
    """HP_1 .. HP_H of the part: HP_k = HP_(k-1) + FOP[trunc(t / k)][f // k]."""
    n, T = case["n"], case["templates"]
    begin, count = _rows(T, case["part"])
    f = torch.arange(n, device="cuda")
    t = torch.arange(begin, begin + count, device="cuda") - T // 2
    hp = fop[begin:begin + count].clone()
    yield hp
    for k in range(2, case["harmonics"] + 1):
        hp += fop[T // 2 + torch.div(t, k, rounding_mode="trunc")][:, f // k]
        yield hp


def _exact_list(hp, threshold, cap):
    """Powers of the plane's strongest `cap` values above the threshold, in (row, bin) order."""
    flat = hp.reshape(-1)
    at = torch.nonzero(flat > float(threshold)).reshape(-1)
    if at.numel() > cap:
        at = at[torch.topk(flat[at], cap).indices].sort().values
    return flat[at].cpu().numpy()


def _padded(values, cap, fill):
    out = np.full(cap, fill, np.float64)
    out[:len(values)] = values
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("launch", "resident") and case["cap"] <= EXACT_LIST and case["n"] <= 800_000:
        out = []
        for s in range(case["sets"]):
            x = _spectrum(case["n"], case["templates"], seed + 1000003 * s)
            thr = _noise_thresholds(x, case["harmonics"])
            planes = _exact_planes(_exact_fop(x, case), case)
            out.append({"location": None, "power": np.concatenate(
                [_padded(_exact_list(hp, t, case["cap"]), case["cap"], -1.0) for hp, t in zip(planes, thr)])})
        return out
    if kind == "stages":
        x = _spectrum(case["n"], case["templates"], seed)
        overlap = -(-(MAX_TAPS - 1) // 4) * 4
        payload = case["tile"] - overlap
        n_tiles = -(-case["n"] // payload)
        padded = torch.zeros(overlap + n_tiles * payload, dtype=torch.complex128, device="cuda")
        padded[overlap:overlap + case["n"]] = x
        tiles = torch.fft.fft(padded.unfold(0, case["tile"], payload), dim=1).reshape(-1)
        return {"tiles": tiles.cpu().numpy(), "fop": _exact_fop(x, case).reshape(-1).cpu().numpy()}
    if kind == "quantile":
        fop = _exact_fop(_spectrum(case["n"], case["templates"], seed), case)
        thr, powers = [], []
        for hp in _exact_planes(fop, case):
            place = (1.0 - case["per_plane"] / hp.numel()) * (hp.numel() - 1)
            below = math.floor(place)
            top = torch.topk(hp.reshape(-1), hp.numel() - below).values
            lo, hi = float(top[-1]), float(top[-2])
            thr.append(lo + (place - below) * (hi - lo))
            powers.append(_exact_list(hp, thr[-1], case["cap"]))
        return {"thresholds": np.array(thr), "harmonic": None, "template": None, "bin": None,
                "power": np.concatenate(powers), "detected": None}
    if kind == "hsum":
        fop = _plane(case, seed).double()
        k = np.arange(1, case["harmonics"] + 1, dtype=np.float64)
        thr = (k + NOISE_SIGMA * np.sqrt(k)).astype(np.float32)
        return {"key": None, "counts": None, "power": np.concatenate(
            [_padded(_exact_list(hp, t, case["cap"]), case["cap"], 0.0)
             for hp, t in zip(_exact_planes(fop, case), thr)])}
    if kind == "frontend":
        series = synth.device_series(_workload(case["n"], 85, seed)).double()
        spec = torch.fft.rfft(series)[:case["n"]] / (2 * case["n"])
        return spec.cpu().numpy() if case["host"] else spec
    return None
