"""Performance cases of the AAK waveform and likelihood path.

Each case is one call that a user's program makes, through the package's
public entry points: batches of likelihoods (a sampler's step), single
likelihoods, waveforms and phases (the reference's calling pattern), the inner
product on the caller's own device buffers, an uneven batch over several
grids, and one training gradient and one inference of the frequency-map
network.  Templates are either drawn from the production prior (log10 M ~
U[5, 7], mu ~ U[5, 50], a ~ U[0, 0.95], e0 ~ U[1e-3, 0.5], p0 ~ U[7, 15],
iota0 = 0.5, angles over the sphere), as a search does, or scattered about
one source (10^5.8 to 10^6.6 solar masses), as a sampler's walkers are.  The
data are an injected source plus Gaussian noise of the analytic LISA PSD,
weighted on the rFFT grid.
"""
import ctypes as C

import numpy as np
import torch

from emri_kludge_suite_amd import GPUAAK, _lib
from emri_kludge_suite_amd import AAKwrapper
from emri_kludge_suite_amd import freqmap_mlp as F
from emri_kludge_suite_amd import multigrid as MG

KEYS = ("iota", "s", "p", "e", "M", "mu", "gamma", "psi", "alpha", "theta_S", "phi_S", "theta_K", "phi_K", "D")
GRIDS = tuple((1 << k, dt) for k in (19, 20, 21) for dt in (10.0, 15.0))  # of the uneven batch


def _case(name, kind, N=0, dt=15.0, n=1, precision="fp64", nmax=0, LISA=True, backint=False,
          around="source"):
    return {"name": name, "kind": kind, "N": N, "dt": dt, "n": n, "precision": precision, "nmax": nmax,
            "LISA": LISA, "backint": backint, "around": around}


def listed():
    return [
        # a search's step on one year of data, the headline: 256 templates over the prior, mixed precision
        _case("batch_1yr_prior_mixed", "batch", 1 << 21, 15.0, 256, "mixed", 50, around="prior"),
        # a sampler's step on the same data: 128 walkers, mixed precision
        _case("batch_1yr_mixed", "batch", 1 << 21, 15.0, 128, "mixed", 50),
        # the same in the default precision, evolved back to the start of the data
        _case("batch_1yr_fp64_backint", "batch", 1 << 21, 15.0, 128, "fp64", 50, True, True),
        # one month at 10 s, the reference's harmonic rule
        _case("batch_month_fp64", "batch", 1 << 18, 10.0, 256, "fp64", 0),
        # exactly 365.25 days at 15 s: a length that is no power of two
        _case("batch_ragged_fp64", "batch", 2103840, 15.0, 64, "fp64", 30),
        # templates of uneven duration and step over the prior, learned map start
        _case("uneven_prior_mixed", "uneven", 1 << 21, 15.0, 192, "mixed", 0, around="prior"),
        # one likelihood per call, as the reference's caller loops over them
        _case("like_1yr_fp64", "like", 1 << 21, 15.0, 1, "fp64", 50),
        # a short waveform without the detector's response, copied to the host
        _case("wave_week_ldc", "wave", 1 << 16, 10.0, 1, "fp64", 0, False, False),
        # phases and frequencies of one source
        _case("phases_4months", "phases", 1 << 20, 10.0),
        # the inner product alone on series that are on the GPU already: smallest and one year
        _case("inner_4096", "inner", 1 << 12),
        _case("inner_1yr", "inner", 1 << 21),
        # gradient of the map network over one training batch
        _case("map_gradient", "gradient", 0, 15.0, 4096, "bf16"),
    ]


def draw(rng):
    kind = rng.choice(("batch", "batch", "batch", "batch", "like", "like", "wave", "phases", "inner", "inner",
                       "gradient", "predict", "uneven"))
    if kind in ("gradient", "predict"):
        return _unnamed(_case("", kind, 0, 15.0, int(2 ** rng.uniform(6, 14)), "bf16"))
    if kind == "inner":
        return _unnamed(_case("", kind, 1 << rng.randint(8, 21), 15.0, rng.randint(2, 8)))
    if kind == "uneven":
        return _unnamed(_case("", kind, 1 << 21, 15.0, rng.randint(8, 192), rng.choice(("mixed", "fp64")), around="prior"))
    N = int(2 ** rng.uniform(15, 21))
    N = 1 << (N.bit_length() - 1) if rng.random() < 0.7 else N - N % 2
    n = 1
    if kind == "batch":
        n = max(1, min(256, int(2 ** rng.uniform(0, 8)), (1 << 28) // N))
    if kind == "phases":
        return _unnamed(_case("", kind, N, rng.choice((10.0, 15.0)), backint=rng.random() < 0.4))
    return _unnamed(_case("", kind, N, rng.choice((10.0, 15.0)), n, rng.choice(("mixed", "fp64")),
                          rng.choice((0, 10, 30, 50, rng.randint(4, 60))), rng.random() < 0.75, rng.random() < 0.4,
                          "prior" if kind == "batch" and rng.random() < 0.2 else "source"))


def _unnamed(c):
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs
def _prior(rng, n):
    """n draws from the production prior, clear of the last stable orbit."""
    out = []
    while len(out) < n:
        s, p, e = rng.uniform(0, 0.95), rng.uniform(7, 15), rng.uniform(1e-3, 0.5)
        if p < F.p_lso(s, e, 0.5) + 0.2:
            continue
        ang = rng.uniform(0, 2 * np.pi, 5)
        out.append([0.5, s, p, e, 10 ** rng.uniform(5, 7), rng.uniform(5, 50), ang[0], ang[1], ang[2],
                    np.arccos(rng.uniform(-1, 1)), ang[3], np.arccos(rng.uniform(-1, 1)), ang[4], 1.0])
    return np.array(out)


def _source(rng):
    """A source in the middle of the band, clear of the last stable orbit at t = 0."""
    while True:
        q = _prior(rng, 1)[0]
        q[4] = 10 ** rng.uniform(5.8, 6.6)
        if q[2] > F.p_lso(q[1], q[3], 0.5) + 1.0:
            return q


def _walkers(rng, n):
    """n templates about one source: intrinsic parameters to 1e-4, angles to 0.1."""
    P = np.tile(_source(rng), (n, 1))
    P[:, 1:6] *= 1.0 + 1e-4 * rng.standard_normal((n, 5))
    P[:, 6:13] += 0.1 * rng.standard_normal((n, 7))
    P[:, (9, 11)] = np.clip(P[:, (9, 11)], 0.01, np.pi - 0.01)
    return P


def _data(g, rng, N, dt):
    """Weighted data of an injected source plus noise, loaded into the handle."""
    w = MG.psd_weights(N, dt, 1)
    g.gpu_gen_AAK(*_source(rng))
    _, hI, hII = g.GetWaveform()
    d = []
    for h in (hI[:N], hII[:N]):
        noise = rng.standard_normal((w.size, 2)).view(np.complex128)[:, 0]
        d.append(np.fft.rfft(h) * w + 0.5 * noise)  # 4 <n|n> of unit weight per bin and component
    g.input_data(d[0], d[1], w, w)


def _network_inputs(rng, n):
    """Normalised features and targets as the training set has them."""
    X = rng.uniform(-1.7, 1.7, (n, 4)).astype(np.float32)
    T = (np.sin(X[:, :3] + 0.5 * X[:, 3:]) + 0.05 * rng.standard_normal((n, 3))).astype(np.float32)
    return X, T


def _inner_inputs(case, seed):
    """Both channels of n coloured series, their weighted data and weights, in the scale the path meets."""
    N = case["N"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    h, d, w = [], [], []
    f = torch.linspace(1.0 / N, 0.5, N // 2 + 1, device="cuda", dtype=torch.float64)
    t = torch.arange(N, device="cuda", dtype=torch.float64)
    for k in range(2):
        noise = torch.randn((case["n"], N), device="cuda", dtype=torch.float64, generator=gen)
        wk = 1e18 / (1.0 + (0.02 / f) ** 2 + (f / 0.2) ** 2)
        hk = 1e-21 * (torch.sin(0.37 * t + 1e-8 * t * t + k) + 0.1 * noise)
        dk = (torch.fft.rfft(hk[0]) + 1e-21 * N ** 0.5 * torch.randn(N // 2 + 1, device="cuda", dtype=torch.complex128,
                                                                     generator=gen)) * wk
        h.append(hk)
        d.append(dk.contiguous())
        w.append(wk.contiguous())
    return h, d, w


def prepare(case, seed):
    kind, N, dt = case["kind"], case["N"], case["dt"]
    rng = np.random.default_rng([seed, 77])
    if kind in ("gradient", "predict"):
        st = {"kind": kind, "model": F.FreqMapModel.load()}
        if kind == "gradient":
            st["X"], st["T"] = _network_inputs(rng, case["n"])
        else:
            st["pts"] = F.sample_points(case["n"], seed)
        return st
    if kind == "inner":
        f = _lib.lib().aak_inner_product_noalloc
        f.restype, f.argtypes = C.c_int, [C.c_void_p] * 6 + [C.c_int, C.c_void_p, C.c_void_p]
        h, d, w = _inner_inputs(case, seed)
        return {"kind": kind, "f": f, "N": N, "h": h, "data": d + w,
                "out": torch.empty((case["n"], 2), device="cuda", dtype=torch.float64)}
    if kind == "uneven":
        mg = MG.MultiGridBatch(precision=case["precision"], map_model=F.FreqMapModel.load())
        for n_, dt_ in GRIDS:
            _data(mg.handle(n_, dt_), rng, n_, dt_)
        P = _prior(rng, case["n"])
        g = np.array(GRIDS)[rng.integers(0, len(GRIDS), case["n"])]
        nmax = np.clip(np.rint(100 * P[:, 3]), 10, 60).astype(np.int32)
        return {"kind": kind, "mg": mg, "P": P, "N": g[:, 0].astype(np.int64), "dt": g[:, 1], "nmax": nmax}
    if kind == "phases":
        p = dict(zip(KEYS, _source(rng).tolist()))
        p.update(T_fit=1.0, length=N, dt=dt, LISA=case["LISA"], backint=case["backint"])
        return {"kind": kind, "pars": p}
    g = GPUAAK(1.0, max(1, N // 100), N, 100.0, dt, case["LISA"], case["backint"])
    g.set_nmax(case["nmax"])
    if kind != "wave":
        _data(g, rng, N, dt)
    g.set_precision(case["precision"])
    return {"kind": kind, "g": g, "P": (_prior if case["around"] == "prior" else _walkers)(rng, case["n"])}


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "batch":
        return state["g"].LikelihoodBatch(state["P"])
    if kind == "uneven":
        return state["mg"].likelihood(state["P"], state["N"], state["dt"], state["nmax"])[0]
    if kind == "like":
        return state["g"].WaveformThroughLikelihood(*state["P"][0])
    if kind == "wave":
        state["g"].gpu_gen_AAK(*state["P"][0])
        return state["g"].GetWaveform()
    if kind == "phases":
        return AAKwrapper.phase(state["pars"])[:8]
    if kind == "gradient":
        return state["model"].gradient(state["X"], state["T"])
    if kind == "predict":
        return state["model"].predict_maps(state["pts"])
    stream = torch.cuda.current_stream().cuda_stream
    fixed = [b.data_ptr() for b in state["data"]]
    for hI, hII, out in zip(*state["h"], state["out"]):
        _lib.check(state["f"](hI.data_ptr(), hII.data_ptr(), *fixed, state["N"], out.data_ptr(), stream),
                   "inner_product_noalloc")
    return state["out"]


def work(case):
    """Inputs read once, outputs written once, and the arithmetic of one pass:
    per sample the phase rates (400 operations), 26 per harmonic (rotation and
    three second-order sums) and the response (300); the FFT's 2.5 N log2 N
    per channel; per likelihood bin the weighting and two sums."""
    kind, N, n = case["kind"], case["N"], case["n"]
    if kind in ("gradient", "predict"):
        macs = 4 * 128 + 2 * 128 * 128 + 3 * 128
        par = 4 * (2 * 128 * 128 + 11 * 128 + 3)
        if kind == "predict":
            return {"bytes": n * 56 + par, "flops": 2 * n * macs}
        return {"bytes": n * 28 + 2 * par, "flops": 6 * n * macs}
    nb = N // 2 + 1
    fft = 2 * (2.5 * N * np.log2(max(N, 2)) + 14 * nb)
    if kind == "inner":
        return {"bytes": n * (16 * N + 16) + 48 * nb, "flops": n * fft}
    if kind == "uneven":
        mean = sum(g[0] for g in GRIDS) / len(GRIDS)
        per = mean * (700 + 26 * 30) + fft * mean / N
        return {"bytes": sum(48 * (g[0] // 2 + 1) for g in GRIDS) + 128 * n, "flops": n * per}
    wave = N * (700.0 + 26 * (case["nmax"] or 8))
    if kind == "phases":
        return {"bytes": 64 * N, "flops": 400.0 * N}
    if kind == "wave":
        return {"bytes": 24 * (N + 2), "flops": wave}
    return {"bytes": 48 * nb + 128 * n, "flops": n * (wave + fft)}


# ------------------------------------------------------------------ 64 bits
def _network(p):
    o, out = 0, []
    for shape in ((4, 128), (128,), (128, 128), (128,), (128, 128), (128,), (128, 3), (3,)):
        k = int(np.prod(shape))
        out.append(p[o:o + k].astype(np.float64).reshape(shape))
        o += k
    return out


def _gelu(z):
    t = np.tanh(np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3))
    return 0.5 * z * (1 + t), 0.5 * (1 + t) + 0.5 * z * (1 - t * t) * np.sqrt(2 / np.pi) * (1 + 3 * 0.044715 * z * z)


def exact(case, seed):
    kind = case["kind"]
    if kind == "inner":
        h, d, w = _inner_inputs(case, seed)
        out = torch.zeros((case["n"], 2), dtype=torch.float64)
        for hk, dk, wk in zip(h, d, w):
            x = torch.fft.rfft(hk.cpu()) * wk.cpu()
            out[:, 0] += 4 * (x.conj() * dk.cpu()).real.sum(1)
            out[:, 1] += 4 * (x.conj() * x).real.sum(1)
        return out
    if kind not in ("gradient", "predict"):
        return None  # waveforms: no closed form in plain numpy
    with np.load(F.WEIGHTS, allow_pickle=False) as z:
        W1, b1, W2, b2, W3, b3, W4, b4 = _network(z["params"])
        norm = z["norm"].astype(np.float64)
    if kind == "predict":
        pts = F.sample_points(case["n"], seed)
        X = (F.features(pts) - norm[:4]) / norm[4:8]
    else:
        X, T = _network_inputs(np.random.default_rng([seed, 77]), case["n"])
        X, T = X.astype(np.float64), T.astype(np.float64)
    A1, G1 = _gelu(X @ W1 + b1)
    A2, G2 = _gelu(A1 @ W2 + b2)
    A3, G3 = _gelu(A2 @ W3 + b3)
    Y = A3 @ W4 + b4
    if kind == "predict":
        c = norm[8:11] + norm[11:14] * Y
        return np.column_stack([1 / np.sqrt(pts[:, 1]), np.ones(len(pts)), pts[:, 0]]) + c
    D = Y - T
    dY = 2 * D / D.size
    d3 = dY @ W4.T * G3
    d2 = d3 @ W3.T * G2
    d1 = d2 @ W2.T * G1
    g = [X.T @ d1, d1.sum(0), A1.T @ d2, d2.sum(0), A2.T @ d3, d3.sum(0), A3.T @ dY, dY.sum(0)]
    return np.concatenate([x.ravel() for x in g]), float(np.mean(D * D))
