"""The work that is measured: data passes, pede iterations (data pass + global solve) and served
alignment jobs, through the entry points a program calls (mpgpu.Pede, mpgpu.Server).

`listed()` are the cases, `draw(rng)` one more of the same ranges, `prepare` the context a program
keeps (records in device memory, structure built), `run` one pass through the public calls, and
`exact` the same numbers from plain torch in 64 bits."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "millepede-ii_amd"))

import mpgpu  # noqa: E402

SIGMA = 0.002          # measurement error of the module detectors (20 um), as in bench.py
EXTENT = 100.0         # layer size in x and y (cm): module size = EXTENT / modules


# ------------------------------------------------------------------------------------------------
# cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a planar test detector with two parameters per module and the first
        # and last plane fixed, pede's default method; launches and host work count
        _step("toy_inversion", "toy", 2000, method="inversion"),
        # pede's default method on a detector of a few hundred modules, with parameter errors
        _step("inversion_1800", "pixel", 20000, layers=10, nx=6, ny=5, method="inversion"),
        # decomposition with Lagrange multipliers: the size of the smaller served jobs
        _step("decomposition_4500", "pixel", 40000, layers=10, nx=15, ny=5, method="decomposition"),
        # dense detector above the size where the FP32 factor with FP64 refinement is used
        _step("fp32_refine_18000", "dense", 20000, layers=40, nx=15, ny=5, method="fp32"),
        # matrix-building pass into full storage: every track crosses every layer
        _pass("pass_dense_6000", "dense", 100000, layers=40, nx=5, ny=5, storage="full"),
        # matrix-building pass of the large sparse detector (the benchmark's detector; half its tracks)
        _pass("pass_block_120k", "pixel", 1000000, layers=20, nx=50, ny=20),
        # line search: vector and chi^2 only, parameters close to the solution
        _pass("pass_chi2_60k", "pixel", 400000, layers=20, nx=25, ny=20, icalcm=0, nloopn=2, near=True),
        # a later iteration with outlier down-weighting and a chi^2 cut, FP64 records
        _pass("pass_huber_f64_12k", "pixel", 100000, layers=20, nx=10, ny=10, nloopn=2, lhuber=3, chicut=30.0, f64=True,
              near=True),
        # broken-lines tracks: bordered-band local fits of up to 44 local parameters
        _pass("pass_lines_6k", "lines", 20000, layers=20, nx=10, ny=5, hmin=8, hmax=20),
        # one pede iteration of a large detector: pass and MINRES with the band preconditioner,
        # solved to the accuracy of the benchmark's metric
        _step("minres_24k", "pixel", 200000, layers=20, nx=20, ny=10, method="minres", mrestl=1e-14),
        # the same with pede's default treatment of the constraints (elimination)
        _step("minres_elim_6k", "pixel", 50000, layers=20, nx=10, ny=5, method="minres", mrestl=1e-14, elim=True),
        # several detector subsets aligned at once: records from host memory to corrections
        _serve("serve_8_jobs", 8, 500, 12000, 1000, 30000),
    ]


def _case(name, kind, det, tracks, **kw):
    c = dict(name=name, kind=kind, det=det, tracks=tracks, layers=10, nx=5, ny=1, hmin=8, hmax=30, storage="full", icalcm=1,
             nloopn=1, lhuber=0, chicut=0.0, f64=False, near=False, method="", mrestl=1e-12, elim=False)
    if det == "dense":
        c["hmin"] = c["hmax"] = kw["layers"]
    c.update(kw)
    return c


def _pass(name, det, tracks, **kw):
    kw.setdefault("storage", "block")
    return _case(name, "pass", det, tracks, **kw)


def _step(name, det, tracks, **kw):
    kw.setdefault("storage", "block" if kw["method"] == "minres" else "full")
    return _case(name, "step", det, tracks, **kw)


def _serve(name, jobs, gmin, gmax, tmin, tmax):
    return dict(name=name, kind="serve", jobs=jobs, gmin=gmin, gmax=gmax, tmin=tmin, tmax=tmax)


def draw(rng):
    """One more case of the listed ranges."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def grid(lo, hi):
        n = log(lo, hi)
        ny = max(1, int(round(math.sqrt(n / rng.uniform(1.0, 3.0)))))
        return dict(nx=max(1, n // ny), ny=ny)

    what = rng.choice(["toy", "inversion", "decomposition", "fp32", "full", "block", "block", "block", "lines", "minres",
                       "elim", "serve"])
    if what == "toy":
        c = _step("", "toy", log(200, 20000), method="inversion")
    elif what == "inversion":
        c = _step("", "pixel", log(4000, 20000), layers=10, method="inversion", **grid(4, 30))
    elif what == "decomposition":
        c = _step("", "pixel", log(10000, 40000), layers=10, method="decomposition", **grid(6, 75))
    elif what == "fp32":
        nx = rng.randrange(70, 76)
        c = _step("", "dense", log(8000, 20000), layers=40, nx=nx, ny=1, method="fp32")
    elif what == "full":
        layers = rng.randrange(10, 41)
        c = _pass("", "dense", log(2000, 100000), layers=layers, storage="full", **grid(6, 1000 // layers))
    elif what == "block":
        layers = rng.randrange(10, 21)
        lhuber = rng.choice([0, 0, 2, 3, 5])
        g = grid(30, 1000)
        c = _pass("", "pixel", log(g["nx"] * g["ny"] * 50, min(1000000, g["nx"] * g["ny"] * 5000)), layers=layers,
                  hmin=rng.randrange(5, 9), hmax=rng.randrange(10, 31), icalcm=rng.choice([1, 1, 1, 0]),
                  nloopn=2 if lhuber else rng.choice([1, 2]), lhuber=lhuber, chicut=rng.choice([0.0, 30.0]),
                  f64=rng.random() < 0.3, near=True, **g)
    elif what == "lines":
        c = _pass("", "lines", log(1000, 20000), layers=20, hmin=rng.randrange(6, 11), hmax=rng.randrange(12, 21),
                  storage=rng.choice(["block", "full"]), **grid(10, 50))
    elif what in ("minres", "elim"):
        g = grid(40, 200 if what == "minres" else 50)
        c = _step("", "pixel", g["nx"] * g["ny"] * rng.randrange(600, 1001), layers=20, method="minres",
                  mrestl=1e-14, elim=what == "elim", **g)
    else:
        c = _serve("", rng.randrange(2, 9), 500, log(2000, 12000), 1000, log(4000, 30000))
    c.pop("name")
    return c


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def _records(c, seed):
    """(rec_ptr, words, values, true parameters in label order or None)"""
    if c["det"] == "toy":
        rp, ii, gg, truth = mpgpu.toy_records(seed, c["tracks"])
    elif c["det"] == "pixel":
        rp, ii, gg, truth = mpgpu.pixel_records(seed, c["layers"], c["nx"], c["ny"], c["tracks"], c["hmin"], c["hmax"],
                                                wx=EXTENT / c["nx"], wy=EXTENT / c["ny"], sigma=SIGMA)
    elif c["det"] == "dense":
        rp, ii, gg, truth = mpgpu.dense_records(seed, c["layers"], c["nx"], c["ny"], c["tracks"], sigma=SIGMA)
    else:
        rp, ii, gg = mpgpu.brokenlines_records(seed, c["layers"], c["nx"], c["ny"], c["tracks"], c["hmin"], c["hmax"],
                                               wx=EXTENT / c["nx"], wy=EXTENT / c["ny"], sigma=SIGMA)
        truth = None
    return rp, ii, gg, truth


def _labels(c):
    """every label of the detector, in order"""
    return mpgpu.toy_labels() if c["det"] == "toy" else mpgpu.pixel_labels(c["layers"], c["nx"], c["ny"])


def _steering(c):
    """(labels, pre-sigmas) of the Parameter lines and the constraint blocks"""
    labels = _labels(c)
    if c["det"] == "toy":
        lab = labels[(labels < 200) | (labels > 1000)]           # first and last plane fixed
        return lab, -np.ones(len(lab)), []
    if c["det"] == "pixel":
        lab = np.array(mpgpu.pixel_weak_labels(c["layers"], c["nx"], c["ny"]), dtype=np.int32)
        return lab, np.array(mpgpu.pixel_presigma(lab)), mpgpu.pixel_constraints(c["layers"], c["nx"], c["ny"])
    return labels, np.array([0.1 if q % 10 <= 3 else 0.01 for q in labels]), []


METHODS = dict(inversion=mpgpu.INVERSION, decomposition=mpgpu.DECOMPOSITION, fp32=mpgpu.CHOLESKY_FP32_IR,
               minres=mpgpu.MINRES)


def _entries(c):
    """the entries cut ('entries n'): broken-lines tracks seldom reach the outer modules, whose
    parameters stay variable with their pre-sigmas"""
    return 0 if c["det"] == "lines" else 5


def _start(c, truth, n):
    """start parameters by label: zero in a first pass, near the solution in a later one"""
    return 0.9 * truth if c["near"] and truth is not None else np.zeros(n)


def _jobs(c):
    """the detectors of the served jobs, from the smallest to the largest"""
    jobs = []
    for k in range(c["jobs"]):
        f = k / max(1, c["jobs"] - 1)
        g = c["gmin"] ** (1 - f) * c["gmax"] ** f
        t = int(c["tmin"] ** (1 - f) * c["tmax"] ** f)
        nmod = max(1, int(round(g / 60)))
        ny = max(1, int(round(math.sqrt(nmod / 2.5))))
        nx = max(1, -(-nmod // ny))
        full = 60 * nx * ny <= 5000
        jobs.append(_case("", "job", "pixel", t, layers=10, nx=nx, ny=ny, storage="full" if full else "block",
                          method="fp32" if full else "minres", mrestl=1e-12))
    return jobs


class _Served:
    pass


def prepare(case, seed):
    c = case
    if c["kind"] == "serve":
        s = _Served()
        s.case = c
        s.server = mpgpu.Server(nworkers=8, budget_bytes=60 << 30)
        s.jobs = []
        for k, j in enumerate(_jobs(c)):
            rp, ii, gg, _ = _records(j, seed * 1000 + k)
            lab, sig, cons = _steering(j)
            full = j["storage"] == "full"
            opt = dict(matsto=mpgpu.FULL if full else mpgpu.SPARSE, metsol=METHODS[j["method"]], mreqenf=_entries(j), mcount=1,
                       mrestl=j["mrestl"], mbandw=6, withmultipliers=1)
            s.jobs.append(((rp, ii, gg), (lab, np.zeros(len(lab)), sig), cons, opt, 60 * j["nx"] * j["ny"]))
        return s
    rp, ii, gg, truth = _records(c, seed)
    opt = dict(matsto=mpgpu.FULL if c["storage"] == "full" else mpgpu.SPARSE, mreqenf=_entries(c), mcount=1, lhuber=c["lhuber"])
    if c["method"]:
        opt["metsol"] = METHODS[c["method"]]
    elif c["storage"] == "block":
        opt["metsol"] = mpgpu.MINRES
    if c["storage"] == "block":
        opt.update(mbandw=6, mrestl=c["mrestl"], withmultipliers=0 if c["elim"] else 1)
    P = mpgpu.Pede(**opt)
    P.add_records(rp, ii, gg.astype(np.float64) if c["f64"] else gg)
    lab, sig, cons = _steering(c)
    P.set_steering_parameters(lab, np.zeros(len(lab)), sig)
    if cons:
        P.add_constraints(cons)
    P.build_structure()
    by_label = dict(zip(_labels(c).tolist(), _start(c, truth, len(_labels(c))).tolist()))
    P.set_parameters(np.array([by_label[q] for q in P.labels()[0].tolist()]))
    P.case = c
    P.probe = _probe(seed, P.nall)
    return P


def _probe(seed, n):
    """a vector the matrix of a pass is applied to"""
    return np.random.default_rng(seed + 17).standard_normal(n)


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------
def _pass_out(st, vec, cnt):
    return dict(vec=vec, cnt=cnt, chi2=np.array([st["chi2"]]), counts=np.array([st["ndf"], st["naccept"], st["nrec"]] + st["nrej"]))


def run(state):
    if isinstance(state, _Served):
        # all jobs are handed over, then waited for in order
        ids = [state.server.submit(rec, par, cons, **opt) for rec, par, cons, opt, _ in state.jobs]
        out = dict(corr=[], labels=[], chi2=[], ndf=[])
        for i, job in zip(ids, state.jobs):
            rc, st, lab, corr = state.server.wait(i, job[4])
            if rc:
                raise RuntimeError(f"job failed with exit code {rc}")
            out["corr"].append(corr)
            out["labels"].append(lab)
            out["chi2"].append(st["chi2"])
            out["ndf"].append(st["ndf"])
        out["chi2"] = np.array(out["chi2"])
        out["ndf"] = np.array(out["ndf"])
        return out
    P, c = state, state.case
    st = P.loopn(c["icalcm"], c["nloopn"], c["chicut"])
    if c["kind"] == "pass":
        # the matrix stays on the device: a program sees it through its product
        y = P.avprod(P.probe) if c["icalcm"] == 1 else None
        vec, cnt = P.vector()
        out = _pass_out(st, vec, cnt)
        if y is not None:
            out["product"] = y
        return out
    x, _ = P.solve()
    vec, cnt = P.vector()
    out = _pass_out(st, vec, cnt)
    out["x"] = x
    if c["method"] == "inversion":
        out["err"], out["gcor"] = P.errors()
    return out


# ------------------------------------------------------------------------------------------------
# the work a pass cannot do without, and how exact its results are
# ------------------------------------------------------------------------------------------------
def _sizes(c):
    """expected words and equations per record, parameters per record, parameters, stored matrix words"""
    if c["det"] == "toy":
        return 81.0, 10.0, 16.0, 80, 80 * 81 / 2, 2
    n = 6 * c["layers"] * c["nx"] * c["ny"]
    if c["det"] == "lines":
        np_ = 0.5 * (c["hmin"] + min(c["hmax"], c["layers"]))
        words, neq, hits, nalc = 1 + 20 * np_ + 10 * (np_ - 2), 4 * np_ - 4, np_, 4 + 2 * np_
    elif c["det"] == "dense":
        hits = c["layers"]
        words, neq, nalc = 1 + 18 * hits, 2 * hits, 4
    else:
        hs = [min(h, c["layers"]) + max(0, min(h - c["layers"], c["layers"])) for h in range(c["hmin"], c["hmax"] + 1)]
        hits = 0.93 * sum(hs) / len(hs)
        words, neq, nalc = 1 + 18 * hits, 2 * hits, 4
    full = n * (n + 1) / 2
    if c["storage"] == "full":
        return words, neq, 6 * hits, n, full, nalc
    # group blocks: modules of two layers d apart that one straight track (slope 0.1 rms) can cross
    stored, nmod = 0.0, c["nx"] * c["ny"]
    for d in range(c["layers"]):
        reach = 2.0 * 2.5 * 0.1 * 5.0 * d
        kx = min(c["nx"], 1 + reach * c["nx"] / EXTENT)
        ky = min(c["ny"], 1 + reach * c["ny"] / EXTENT)
        stored += (c["layers"] - d) * nmod * kx * ky * 36
    return words, neq, 6 * hits, n, min(full, stored, c["tracks"] * 36 * hits * (hits + 1) / 2), nalc


def _pass_work(c):
    words, neq, nalg, n, stored, nalc = _sizes(c)
    build = c["icalcm"] == 1
    per_word = 12 if c["f64"] else 8
    b = c["tracks"] * words * per_word + 16 * n + (8 * stored if build else 0)
    # normal equations of the local fit, its inversion, and the update of the global matrix: the
    # lower triangle of G Gamma^-1 G^T
    f = c["tracks"] * (neq * nalc * (nalc + 3) * max(1, c["lhuber"]) + nalc ** 3 + (nalg * (nalg + 1) * nalc if build else 0))
    return b, f, n, stored


# MINRES iterations to the tolerance on these detectors (pede's algorithm needs one matrix product in each)
ITERATIONS = {1e-14: 300, 1e-12: 200}


def work(case):
    if case["kind"] == "serve":
        g = math.sqrt(case["gmin"] * case["gmax"])
        t = math.sqrt(case["tmin"] * case["tmax"])
        j = _case("", "step", "pixel", t, layers=10, nx=g / 60, ny=1, storage="block", method="minres")
        b, f, n, stored = _pass_work(j)
        return {"bytes": case["jobs"] * (b + 8 * stored * 100), "flops": case["jobs"] * (f + 4 * stored * 100)}
    b, f, n, stored = _pass_work(case)
    if case["method"] == "inversion":
        b, f = b + 16 * stored, f + float(n) ** 3
    elif case["method"] in ("decomposition", "fp32"):
        b, f = b + 16 * stored, f + float(n) ** 3 / 3
    elif case["method"] == "minres":
        it = ITERATIONS[case["mrestl"]]
        b, f = b + 8 * stored * it, f + 4 * stored * it
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the largest error against 64-bit torch seen on these ranges, per kind."""
    if case["kind"] == "pass":
        return {"rel": 1e-9}
    if case["kind"] == "serve":
        # MINRES stops within its tolerance; the weakly determined modes are then known to a percent
        return {"rel": 0.03}
    # inversion: the parameter errors are REAL(4) numbers, as pede's are
    return {"rel": {"inversion": 1e-6, "decomposition": 1e-8, "fp32": 1e-6,
                    "minres": 2e-4 if case["elim"] else 1e-7}[case["method"]]}


# ------------------------------------------------------------------------------------------------
# the same numbers in plain torch, 64 bits
# ------------------------------------------------------------------------------------------------
class _Ref:
    """Records as padded arrays per chunk, the parameter tables, and the sums of a data pass."""

    def __init__(self, c, seed, dev):
        self.c, self.dev = c, dev
        rp, ii, gg, truth = _records(c, seed)
        self.rp = torch.from_numpy(rp).to(dev)
        self.ii = torch.from_numpy(ii).to(dev)
        self.gg = torch.from_numpy(gg).to(dev)
        self.nrec = len(rp) - 1
        self.host_rp = rp
        lab, sig, cons = _steering(c)
        every = _labels(c)
        self.labels = torch.from_numpy(np.ascontiguousarray(every)).to(dev)
        n = len(every)
        self.ntot = n
        # entries per record of every label
        cnt = torch.zeros(n, dtype=torch.int64, device=dev)
        for lo, hi in self.chunks(200000):
            w0, w1 = int(rp[lo]), int(rp[hi])
            words = self.ii[w0:w1]
            rec = torch.repeat_interleave(torch.arange(hi - lo, device=dev), self.rp[lo + 1:hi + 1] - self.rp[lo:hi])
            g = words > 99            # labels are above every local index
            key = torch.unique(rec[g] * n + torch.searchsorted(self.labels, words[g]))
            cnt += torch.bincount(key % n, minlength=n)
        presig = np.zeros(n)
        at = {int(q): k for k, q in enumerate(every)}
        for q, s in zip(lab.tolist(), sig.tolist()):
            presig[at[q]] = s
        entries = cnt.cpu().numpy()
        variable = (presig >= 0) & (entries >= _entries(c))
        named = np.zeros(n, bool)          # labels the context knows
        named[entries > 0] = True
        for q in lab.tolist():
            named[at[q]] = True
        for _, _, ls, _ in cons:
            for q in ls:
                named[at[q]] = True
        self.var = np.where(variable, np.cumsum(variable) - 1, -1)
        self.nvar = int(variable.sum())
        self.varlab = every[variable]
        self.par = _start(c, truth, n) * named
        self.prew = np.where(presig[variable] > 0, 1.0 / np.maximum(presig[variable], 1e-100) ** 2, 0.0)
        rows, rhs = [], []
        for r, _, ls, fs in cons:
            row = np.zeros(self.nvar)
            d = r
            for q, f in zip(ls, fs):
                k = at[q]
                d -= f * self.par[k]
                if self.var[k] >= 0:
                    row[self.var[k]] += f
            rows.append(row)
            rhs.append(d)
        self.cons = torch.tensor(np.array(rows).reshape(len(rows), self.nvar), device=dev)
        self.crhs = torch.tensor(np.array(rhs).reshape(-1), dtype=torch.float64, device=dev)

    def chunks(self, size):
        return [(lo, min(self.nrec, lo + size)) for lo in range(0, self.nrec, size)]

    def padded(self, lo, hi):
        """per record of [lo, hi): residuals r[B,M], errors s, mask, local derivatives L[B,M,K],
        global derivatives G[B,M,V] and the total index of each of the V columns (-1: none)"""
        dev, B = self.dev, hi - lo
        w0 = int(self.host_rp[lo])
        words, vals = self.ii[w0:int(self.host_rp[hi])], self.gg[w0:int(self.host_rp[hi])].double()
        ptr = self.rp[lo:hi + 1] - w0
        mark = words == 0
        mark[ptr[:-1]] = False
        z = torch.nonzero(mark).flatten()
        meas, sig = z[0::2].contiguous(), z[1::2].contiguous()               # every equation: value, locals, error, globals
        rec_of = torch.repeat_interleave(torch.arange(B, device=dev), ptr[1:] - ptr[:-1])
        erec = rec_of[meas]
        first = torch.searchsorted(erec, torch.arange(B + 1, device=dev))
        neq = first[1:] - first[:-1]
        M = max(1, int(neq.max()))
        e_in = torch.arange(len(meas), device=dev) - first[erec]
        r = torch.zeros(B, M, dtype=torch.float64, device=dev)
        s = torch.ones_like(r)
        ok = torch.zeros(B, M, dtype=torch.bool, device=dev)
        r[erec, e_in] = vals[meas]
        s[erec, e_in] = vals[sig]
        ok[erec, e_in] = True
        pos = torch.arange(len(words), device=dev)
        eq = torch.searchsorted(meas, pos, right=True) - 1
        inside = (eq >= 0) & ~mark
        inside[ptr[:-1]] = False
        eqc = eq.clamp(min=0)
        if len(meas) == 0:
            inside = torch.zeros_like(inside)
        isl = inside.clone()
        isl[inside] = pos[inside] < sig[eqc[inside]]
        isg = inside & ~isl
        K = max(1, int(words[isl].max())) if bool(isl.any()) else 1
        L = torch.zeros(B, M, K, dtype=torch.float64, device=dev)
        L[rec_of[isl], e_in[eqc[isl]], words[isl].long() - 1] = vals[isl]
        nalc = torch.zeros(B, dtype=torch.int64, device=dev)
        nalc.scatter_reduce_(0, rec_of[isl], words[isl].long(), "amax")
        tix = torch.searchsorted(self.labels, words[isg])
        key, inv = torch.unique(rec_of[isg] * self.ntot + tix, return_inverse=True)
        kfirst = torch.searchsorted(key // self.ntot, torch.arange(B + 1, device=dev))
        V = max(1, int((kfirst[1:] - kfirst[:-1]).max()))
        G = torch.zeros(B, M, V, dtype=torch.float64, device=dev)
        G[rec_of[isg], e_in[eqc[isg]], inv - kfirst[rec_of[isg]]] = vals[isg]
        cols = torch.full((B, V), -1, dtype=torch.int64, device=dev)
        cols[key // self.ntot, torch.arange(len(key), device=dev) - kfirst[key // self.ntot]] = key % self.ntot
        return r, s, ok, L, G, cols, neq, nalc

    def run(self, probe=None, dense=False):
        c, dev = self.c, self.dev
        n = self.nvar
        vec = torch.zeros(n + 1, dtype=torch.float64, device=dev)
        cnt = torch.zeros(n + 1, dtype=torch.float64, device=dev)
        y = torch.zeros(n + 1, dtype=torch.float64, device=dev) if probe is not None else None
        px = torch.cat([torch.as_tensor(probe[:n], device=dev), torch.zeros(1, dtype=torch.float64, device=dev)]) if probe is not None else None
        A = torch.zeros((n + 1) * (n + 1), dtype=torch.float64, device=dev) if dense else None
        par = torch.as_tensor(self.par, device=dev)
        var = torch.as_tensor(self.var, device=dev)
        chi2, ndf_sum, nacc, nrej = 0.0, 0, 0, [0] * 6
        _, neq, nalg, _, _, nalc = _sizes(c)
        big = 1.7 * nalg
        size = max(64, int(1.0e8 / (big * max(2.0 * neq, big if dense else 1.0))))
        eps = 2.0 ** -52
        robust = c["nloopn"] != 1 and c["lhuber"] != 0
        nter = c["lhuber"] if robust else 1
        for lo, hi in self.chunks(min(size, 100000)):
            r, s, ok, L, G, cols, neq, nalc = self.padded(lo, hi)
            K = L.shape[2]
            known = cols >= 0
            pc = torch.where(known, par[cols.clamp(min=0)], torch.zeros((), dtype=torch.float64, device=dev))
            r = r - torch.einsum("bmv,bv->bm", G, pc)
            w0 = torch.where(ok, 1.0 / (s * s), torch.zeros_like(s))
            fit = torch.zeros_like(r)
            status = torch.where(nalc <= 0, 7, 0)
            for it in range(1, nter + 1):
                w = w0
                if robust and it > 1:
                    w = w0 * _down(r - fit, s, it)
                N = torch.bmm((L * w[:, :, None]).transpose(1, 2).contiguous(), L)
                pad = torch.arange(K, device=dev)[None, :] >= nalc[:, None]
                N = N + torch.diag_embed(pad.double())
                Ni, good = _inverse(N, 16 * eps)
                Ni = torch.where(good[:, None, None], Ni, torch.zeros_like(Ni))
                x = torch.einsum("bij,bj->bi", Ni, torch.einsum("bmk,bm->bk", L, w * r))
                fit = torch.einsum("bmk,bk->bm", L, x)
                res = r - fit
                dchi = w0 * res * res
                suwt = ok.double()
                if robust and it > 1:
                    dchi, suwt = _dchi(res, s, it, dchi), torch.sqrt(_down(res, s, it)) * ok
                    dchi = torch.where(ok, dchi, torch.zeros_like(dchi))
                summ = dchi.sum(1)
                ndf = neq - nalc
                status = torch.where((status == 0) & ~good, 2, status)
                status = torch.where((status == 0) & (ndf <= 0), 4, status)
            lim = _chindl(ndf, dev)
            if c["chicut"] >= 0:
                huge = (torch.tensor(50.0, dtype=torch.float32, device=dev) * lim).double()
                status = torch.where((status == 0) & (summ > huge), 5, status)
                if c["chicut"] > 0:
                    cut = (torch.tensor(c["chicut"], dtype=torch.float32, device=dev) * lim).double()
                    over = (status == 0) & (summ > cut)
                    status = torch.where(over, 6, status)
                    chi2 += float(cut[over].sum())
                    ndf_sum += int(ndf[over].sum())
            acc = status == 0
            for k in range(6):
                nrej[k] += int((status == k + 1).sum())
            nacc += int(acc.sum())
            wf = w if robust else w0
            last = w0 * res * res
            if robust:
                last = torch.where(ok, _dchi(res, s, nter, last), torch.zeros_like(last))
            chi2 += float(last.sum(1)[acc].sum())
            ndf_sum += int(ndf[acc].sum())
            wf = wf * acc[:, None]
            # columns of variable parameters; the others go to a spare row
            vcol = torch.where(known, var[cols.clamp(min=0)], torch.full_like(cols, -1))
            vidx = torch.where(vcol >= 0, vcol, torch.full_like(vcol, n))
            vec.index_add_(0, vidx.flatten(), torch.einsum("bmv,bm->bv", G, wf * res).flatten())
            cnt.index_add_(0, vidx.flatten(), torch.einsum("bmv,bm->bv", (G != 0).double(), (ok & acc[:, None]).double()).flatten())
            if probe is None and not dense:
                continue
            GL = torch.bmm((G * wf[:, :, None]).transpose(1, 2).contiguous(), L)
            if probe is not None:
                xg = px[vidx] * (vcol >= 0)
                t = torch.einsum("bmv,bv->bm", G, xg)
                u = torch.einsum("bmv,bm->bv", G, wf * t)
                u = u - torch.einsum("bvk,bk->bv", GL, torch.einsum("bij,bj->bi", Ni, torch.einsum("bvk,bv->bk", GL, xg)))
                y.index_add_(0, vidx.flatten(), u.flatten())
            if dense:
                C = torch.bmm((G * wf[:, :, None]).transpose(1, 2).contiguous(), G)
                C -= torch.bmm(torch.bmm(GL, Ni), GL.transpose(1, 2).contiguous())
                A.index_add_(0, (vidx[:, :, None] * (n + 1) + vidx[:, None, :]).flatten(), C.flatten())
        self.chi2, self.counts = chi2, [ndf_sum, nacc, self.nrec] + nrej
        self.vec, self.cnt = vec[:n], torch.round(cnt[:n]).long()
        prew = torch.as_tensor(self.prew, device=dev)
        if y is not None:
            self.y = y[:n] + prew * px[:n]
        if dense:
            self.A = A.view(n + 1, n + 1)[:n, :n].contiguous()
            self.A.diagonal().add_(prew)

    def solve(self):
        """(x, multipliers, A^-1 C^T and C A^-1 C^T) of the constrained system; self.inv(B) is A^-1 B
        of the augmented parameter block, refined with residuals in more than 64 bits"""
        rho = 0.0
        A = self.A
        m = len(self.crhs)
        if m:
            rho = float(A.diagonal().abs().max() / (self.cons * self.cons).sum(0).max())
            A = A + rho * (self.cons.T.contiguous() @ self.cons)
        F = torch.linalg.cholesky(A)

        parts = _slices(A, 1)

        def inv(B):
            X = torch.cholesky_solve(B, F)
            for _ in range(3):
                X = X + torch.cholesky_solve(_residual(B, parts, X), F)
            return X
        self.inv = inv
        b = self.vec[:, None]
        if not m:
            return inv(b)[:, 0], None, None
        Z = inv(self.cons.T.contiguous())
        d = self.crhs[:, None]
        yb = inv(b + rho * (self.cons.T.contiguous() @ d))
        S = self.cons @ Z
        lam = torch.linalg.solve(S, self.cons @ yb - d)
        return (yb - Z @ lam)[:, 0], lam[:, 0], (Z, S)


def _slices(M, dim):
    """M as a sum of three matrices of 20 bits each (relative to the largest value along dim), so that
    64-bit products of the slices of two matrices are free of rounding"""
    out, R = [], M
    for _ in range(3):
        top = R.abs().amax(dim, keepdim=True).clamp(min=1e-250)
        sigma = 0.75 * torch.exp2(torch.ceil(torch.log2(top)) + 53 - 20)
        H = (R + sigma) - sigma
        out.append(H)
        R = R - H
    return out


def _residual(B, parts, X):
    """B - A X from the slices of A, with the products of the leading slices exact"""
    xs = _slices(X, 0)
    for order in range(3):
        for i in range(order + 1):
            B = B - parts[i] @ xs[order - i]
    return B


def _down(res, s, it):
    """weight factor of the outlier down-weighting (Huber in the second and third iteration, Cauchy after)"""
    if it <= 3:
        a = res.abs()
        return torch.where(a > 1.345 * s, 1.345 * s / a.clamp(min=1e-300), torch.ones_like(a))
    t = res / s / 2.3849
    return 1.0 / (1.0 + t * t)


def _dchi(res, s, it, plain):
    if it <= 3:
        a = res.abs()
        return torch.where(a > 1.345 * s, 2.0 * 1.345 * (a / s - 0.5 * 1.345), plain)
    t = res / s / 2.3849
    return torch.log(1.0 + t * t) * 2.3849 * 2.3849


def _inverse(N, eps):
    """inverses of symmetric positive definite matrices [B,K,K], and which have full rank"""
    K = N.shape[1]
    d = N.diagonal(dim1=1, dim2=2).clamp(min=1e-300)
    sc = 1.0 / torch.sqrt(d)
    X = N * sc[:, :, None] * sc[:, None, :]
    good = torch.ones(N.shape[0], dtype=torch.bool, device=N.device)
    for k in range(K):
        p = X[:, k, k]
        good = good & (p > eps)
        ip = 1.0 / torch.where(p > eps, p, torch.ones_like(p))
        row = X[:, k, :] * ip[:, None]
        col = X[:, :, k].clone()
        X = X - col[:, :, None] * row[:, None, :]
        X[:, k, :] = row
        X[:, :, k] = -col * ip[:, None]
        X[:, k, k] = ip
    X = 0.5 * (X + X.transpose(1, 2))
    return X * sc[:, :, None] * sc[:, None, :], good


def _chindl(ndf, dev):
    """three-sigma limit of chi^2 for ndf degrees of freedom, with pede's REAL(4) table"""
    tab = torch.tensor([9.0000, 5.9146, 4.7184, 4.0628, 3.6410, 3.3436, 3.1209, 2.9468, 2.8063, 2.6902, 2.5922, 2.5082,
                        2.4352, 2.3711, 2.3143, 2.2635, 2.2178, 2.1764, 2.1386, 2.1040, 2.0722, 2.0428, 2.0155, 1.9901,
                        1.9665, 1.9443, 1.9235, 1.9040, 1.8855, 1.8681], dtype=torch.float32, device=dev)
    f = ndf.float()
    t = 2.782170 + torch.sqrt((2 * ndf - 1).clamp(min=1).float())
    c = torch.where(ndf <= 30, tab[(ndf - 1).clamp(0, 29)], t * t / (2 * ndf).clamp(min=1).float())
    return torch.where(ndf < 1, torch.zeros_like(c), c) * f


def _job_exact(c, seed, dev):
    R = _Ref(c, seed, dev)
    R.run(dense=True)
    return R, R.solve()


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    c = case
    if c["kind"] == "serve":
        out = dict(corr=[], labels=[], chi2=[], ndf=[])
        for k, j in enumerate(_jobs(c)):
            R, (x, _, _) = _job_exact(j, seed * 1000 + k, dev)
            out["corr"].append(x.cpu().numpy())
            out["labels"].append(np.ascontiguousarray(R.varlab, dtype=np.int32))
            out["chi2"].append(R.chi2)
            out["ndf"].append(R.counts[0])
        out["chi2"] = np.array(out["chi2"])
        out["ndf"] = np.array(out["ndf"])
        return out
    R = _Ref(c, seed, dev)
    mult = len(R.crhs) if not c["elim"] else 0
    if c["kind"] == "pass":
        probe = _probe(seed, R.nvar + mult) if c["icalcm"] == 1 else None
        R.run(probe=probe)
    else:
        R.run(dense=True)
    vec = R.vec
    if mult:
        vec = torch.cat([vec, R.crhs])
    out = dict(vec=vec.cpu().numpy(), cnt=R.cnt.cpu().numpy(), chi2=np.array([R.chi2]), counts=np.array(R.counts))
    if c["kind"] == "pass":
        if c["icalcm"] == 1:
            y = R.y
            if mult:
                p = torch.as_tensor(probe, device=dev)
                y = torch.cat([y + R.cons.T @ p[R.nvar:], R.cons @ p[:R.nvar]])
            out["product"] = y.cpu().numpy()
        return out
    x, lam, ZS = R.solve()
    out["x"] = (torch.cat([x, lam]) if mult else x).cpu().numpy()
    if c["method"] == "inversion":
        inv = R.inv(torch.eye(R.nvar, dtype=torch.float64, device=dev)).diagonal()
        if ZS is not None:
            inv = inv - (ZS[0] * torch.linalg.solve(ZS[1], ZS[0].T.contiguous()).T).sum(1)
        inv = inv.cpu().numpy()
        diag = R.A.diagonal().cpu().numpy()
        g2 = 1.0 - 1.0 / (inv * diag)
        out["err"] = np.sqrt(np.abs(inv))
        out["gcor"] = np.where((g2 >= 0) & (g2 <= 1), np.sqrt(np.clip(g2, 0, 1)), -1.0)
    return out
