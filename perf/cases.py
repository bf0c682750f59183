"""The calls whose speed this library answers for, as a user's program makes them.

Five kinds of call, each through the package's public entry points (song_amd.lib):

  los     Engine.run on resident inputs: source re-layout, k3 spline, line-of-sight integral of
          every loaded (k1,k2) pair; the transfers stay in device memory (device_output)
  host    Engine.load + run + store on host arrays: what transfer2_init does per k1 batch
          (upload, device layouts, run, scatter into ptr2->transfer), on a kept engine
  serve   Server.submit / wait: a burst of jobs of 1..n pairs, each with its own l_max
  k3int   K3Integral.run + result: the bispectrum module's k3 integral of the transfers
  cl2     Cl2.run + result: the second-order C_l sum over (k1, k2, k3)

Inputs are seeded: the los, host and serve kinds take SONG's structures from the package's own
generator (k and tau grids, source tables, J tables), the consumers take transfers that
oscillate in k3 and fall with it, as the stage's output does.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from song_amd import lib as L

FORMS = {"fp64": L.FORM_FP64, "fp64fast": L.FORM_FP64_FAST, "fp32c": L.FORM_FP32C}

# values shared by every configuration unless a case says otherwise
_GRID = dict(kind="los", form="fp64", m="0,1,2", E=True, L=6, k_size=32, k_min=1e-5, k_max=0.1,
             k3_size=60, tau_size=600, l_size=96, l_max=2000, dk_fine=1.5e-4,
             xx_max=1500.0, cubic_k3=True, extrap=False, pairs=0, graph=False)


def listed():
    return [
        # the quick check of the benchmark: 21 pairs, every launch latency shows
        dict(_GRID, name="los_tiny", L=4, k_size=6, k3_size=16, tau_size=128, l_size=12,
             l_max=400, dk_fine=1e-3),
        # the reference's CPU configuration: T only, m = 0, 136 pairs
        dict(_GRID, name="los_c1", m="0", E=False, L=4, k_size=16, k_min=1e-4, k_max=0.05,
             tau_size=400, l_size=48, l_max=1000, dk_fine=2e-4, xx_max=750.0),
        # odd sizes and the options: m = 0, 2, linear k3 interpolation, flat extrapolation
        dict(_GRID, name="los_ragged", m="0,2", L=5, k_size=13, k3_size=23, tau_size=251,
             l_size=37, l_max=1500, dk_fine=4.3e-4, cubic_k3=False, extrap=True),
        # the benchmark's headline workload: every pair of a 32 x 32 grid, T + E + B, plain FP64
        dict(_GRID, name="los_c2"),
        # the other two forms on a grid of half as many k
        dict(_GRID, name="los_fma", form="fp64fast", k_size=16),
        # the precision study: l to 3000, 128 l
        dict(_GRID, name="los_fp32c", form="fp32c", k_size=16, l_size=128, l_max=3000),
        # a batch of pairs picked from a wider grid, few coarse k3, one captured graph
        dict(_GRID, name="los_batch", k_size=40, k_max=0.2, k3_size=8, dk_fine=3.5e-4,
             pairs=512, graph=True, xx_max=3000.0),
        # a host-resident k1 batch, uploaded, run and scattered back
        dict(_GRID, name="host_batch", kind="host", k_size=10),
        # a burst of serving jobs
        dict(_GRID, name="serve_burst", kind="serve", k_size=16, k_max=0.2, k3_size=8,
             dk_fine=3.5e-4, l_size=128, l_max=3000, xx_max=3000.0, jobs=24, job_pairs=32),
        # the bispectrum's k3 integral: 48 l3 rows x 136 pairs x 100 r
        dict(name="k3int", kind="k3int", k_size=16, k_min=1e-5, k_max=0.1, dk_fine=1.5e-4,
             l_size=48, l_max=2000, n_r=100, step=0.3),
        # the C_l sums: a small spectrum and the benchmark's (96 l x 3 m x 528 pairs)
        dict(name="cl2_small", kind="cl2", k_size=12, k_min=1e-4, k_max=0.1, dk_fine=1e-3,
             l_size=25, m="0,2", rescale=True, cross=True),
        dict(name="cl2", kind="cl2", k_size=32, k_min=1e-5, k_max=0.1, dk_fine=1.5e-4,
             l_size=96, m="0,1,2", rescale=True, cross=False),
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _logi(rng, a, b):
    return int(round(_log(rng, a, b)))


def draw(rng):
    kind = rng.choice(["los", "los", "los", "los", "los", "los", "host", "serve", "k3int", "cl2"])
    if kind == "k3int":
        return dict(kind=kind, k_size=rng.randint(4, 16), k_min=1e-5, k_max=0.1,
                    dk_fine=_log(rng, 1.5e-4, 1e-3), l_size=_logi(rng, 5, 48), l_max=2000,
                    n_r=_logi(rng, 9, 100), step=0.3)
    if kind == "cl2":
        return dict(kind=kind, k_size=rng.randint(5, 30), k_min=1e-4, k_max=0.1,
                    dk_fine=_log(rng, 1.5e-4, 1e-3), l_size=_logi(rng, 6, 96),
                    m=rng.choice(["0", "0,1", "0,2", "0,1,2"]), rescale=rng.random() < 0.5,
                    cross=rng.random() < 0.5)
    l_max = rng.choice([500, 1000, 1500, 2000, 3000])
    c = dict(_GRID, kind=kind, k_size=rng.randint(5, 18),
             k_max=rng.choice([0.05, 0.1, 0.2]), k3_size=_logi(rng, 6, 60), tau_size=_logi(rng, 90, 600),
             l_size=_logi(rng, 9, 128), l_max=l_max,
             dk_fine=_log(rng, 1.5e-4, 1e-3), L=rng.randint(2, 7),
             m=rng.choice(["0", "0,1", "0,2", "0,1,2"]), E=rng.random() < 0.75,
             cubic_k3=rng.random() < 0.8,
             form=rng.choice(["fp64", "fp64", "fp64fast", "fp32c"]))
    c["xx_max"] = c["k_max"] * 15000.0
    if kind == "host":
        c.update(k_size=rng.randint(5, 10), form="fp64")
    if kind == "serve":
        c.update(k_size=rng.randint(6, 14), k3_size=_logi(rng, 6, 16),
                 jobs=rng.randint(3, 24), job_pairs=rng.randint(2, 20))
    if kind == "los" and rng.random() < 0.3:
        c.update(pairs=rng.randint(10, c["k_size"] * (c["k_size"] + 1) // 2),
                 graph=rng.random() < 0.5)
    return c


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _m(case):
    return [int(v) for v in case["m"].split(",")]


def _config(case, seed):
    return L.Config(has_T=1, has_E=int(case["E"]), m_list=_m(case), l_max_los_t=case["L"],
                    l_max_los_p=case["L"], k_size=case["k_size"], k_min=case["k_min"],
                    k_max=case["k_max"], k3_size=case["k3_size"],
                    tau_size=case["tau_size"], l_size=case["l_size"], l_max=case["l_max"],
                    dk_fine=case["dk_fine"], xx_max=case["xx_max"],
                    k3_interpolation=L.CUBIC if case["cubic_k3"] else L.LINEAR,
                    extrapolation=L.FLAT_EXTRAP if case["extrap"] else L.NO_EXTRAP,
                    extra_osc_left=3.0 if case["extrap"] else 0.0,
                    extra_osc_right=3.0 if case["extrap"] else 0.0, seed=1000 + int(seed))


def _all_pairs(case):
    return [(i1, i2) for i1 in range(case["k_size"]) for i2 in range(i1 + 1)]


def _pairs(case):
    allp = _all_pairs(case)
    if not case["pairs"] or case["pairs"] >= len(allp):
        return allp
    pick = np.sort(np.random.default_rng(7).choice(len(allp), case["pairs"], replace=False))
    return [allp[i] for i in pick]


def _jobs(case):
    allp = _all_pairs(case)
    rng = np.random.default_rng(7)
    jobs = []
    for _ in range(case["jobs"]):
        n = int(rng.integers(1, min(case["job_pairs"], len(allp)) + 1))
        lmax = int(case["l_max"] * rng.choice([0.25, 0.5, 1.0]))
        jobs.append(([allp[i] for i in rng.choice(len(allp), n, replace=False)], lmax))
    return jobs


def _triangle(case):
    """k grid, (k1,k2) pairs with k2 <= k1, offsets and k3 grid of every pair."""
    n = case["k_size"]
    k = np.exp(np.linspace(math.log(case["k_min"]), math.log(case["k_max"]), n))
    grids = []
    for i1 in range(n):
        for i2 in range(i1 + 1):
            lo = max(k[i1] - k[i2], k[0]) * (1 + 1e-6)
            hi = min(k[i1] + k[i2], k[-1]) * (1 - 1e-6)
            grids.append(np.linspace(lo, hi, max(4, int((hi - lo) / case["dk_fine"]))))
    off = np.concatenate([[0], np.cumsum([g.size for g in grids])])
    return k, off, np.concatenate(grids)


def _transfers(rng, rows, off, k3):
    """[rows][k3 of all pairs]: an amplitude per (row, pair), oscillating in k3 and falling."""
    n = np.diff(off)
    amp = np.repeat(rng.normal(size=(rows, n.size)), n, axis=1)
    phase = np.repeat(rng.uniform(0, 2 * np.pi, size=(rows, n.size)), n, axis=1)
    return amp * np.cos(k3 * 280.0 + phase) * (k3 / 0.01) ** -1.5


def _k3_bounds(k, i1, i2):
    """Ends of a pair's coarse k3 grid: the triangle's, kept inside the k grid."""
    lo = max(k[i1] - k[i2] + 1e-10, (k[i1] + k[i2]) / 100.0, k[0])
    return lo, min(k[i1] + k[i2] - 1e-10, k[-1])


def _l_list(n, l_max):
    return sorted({int(round(2.0 * (l_max / 2.0) ** (i / max(1, n - 1)))) for i in range(n)})


def _j_tables(case, kr_max):
    """j_l(x) on the x grid of every l, from its first value above the cut on."""
    lib, ls = L.load(), _l_list(case["l_size"], case["l_max"])
    nx = int(kr_max / case["step"]) + 3
    row = np.empty(max(ls) + 1)
    jl = np.empty((nx, len(ls)))
    for ix in range(nx):
        lib.los_sph_bessel_array(max(ls), ix * case["step"],
                                 row.ctypes.data_as(C.POINTER(C.c_double)))
        jl[ix] = row[ls]
    off, vals, x_min = [0], [], []
    for q in range(len(ls)):
        i0 = max(int(np.argmax(np.abs(jl[:, q]) >= 1e-12)) - 1, 0)
        vals.append(jl[i0:, q])
        x_min.append(i0 * case["step"])
        off.append(off[-1] + nx - i0)
    return off, np.concatenate(vals), np.array(x_min)


def _consumer_inputs(case, seed):
    rng = np.random.default_rng(seed)
    k, off, k3 = _triangle(case)
    if case["kind"] == "k3int":
        r = np.linspace(13600.0, 14400.0, case["n_r"])
        j_off, j, x_min = _j_tables(case, k3.max() * r.max())
        T = _transfers(rng, len(x_min), off, k3)
        return dict(off=off, k3=k3, T=T, index_L=np.arange(len(x_min)), j_off=j_off, j=j,
                    x_min=x_min, step=case["step"], r=r)
    m = _m(case)
    T1 = _transfers(rng, case["l_size"] * len(m), off, k3)
    T2 = _transfers(rng, case["l_size"] * len(m), off, k3) if case["cross"] else T1
    pk = 2.1e-9 * (k / 0.05) ** (0.965 - 1)
    return dict(k=k, pk=pk, off=off, k3=k3, m=m, T1=T1, T2=T2,
                used=np.ones((case["l_size"], len(m)), dtype=np.int32), rescale=case["rescale"])


def prepare(case, seed):
    if case["kind"] == "k3int":
        a = _consumer_inputs(case, seed)
        return "k3int", L.K3Integral(a["off"], a["k3"], a["T"], a["index_L"], a["j_off"], a["j"],
                                     a["x_min"], a["step"], a["r"])
    if case["kind"] == "cl2":
        a = _consumer_inputs(case, seed)
        return "cl2", L.Cl2(a["k"], a["pk"], a["off"], a["k3"], a["m"], a["T1"], a["T2"],
                            a["used"], a["rescale"])
    scen = L.Scenario(_config(case, seed))
    scen.prepare()
    if case["kind"] == "serve":
        srv = L.Server(scen, FORMS[case["form"]], budget_bytes=4.0 * 2 ** 30, slots=3)
        return "serve", srv, scen, _jobs(case)
    eng = L.Engine(0)
    eng.set_form(FORMS[case["form"]])
    if case["kind"] == "host":
        eng.load(scen)
        eng.autotune()
        return "host", eng, scen
    eng.load_pairs(scen, _pairs(case))
    scen.close()
    eng.autotune()
    if case["graph"]:
        eng.capture()
    return "los", eng


class _Device:
    """The engine's transfers in device memory, for torch.as_tensor; the tensor keeps this object
    and so the engine, whose memory it is."""

    def __init__(self, engine):
        self.engine = engine
        ptr, rows, cols = engine.device_output()
        self.__cuda_array_interface__ = {"shape": (rows, cols), "typestr": "<f8",
                                         "data": (ptr, False), "version": 2}


def run(state):
    kind, h = state[0], state[1]
    if kind == "los":
        h.run()
        out = torch.as_tensor(_Device(h), device="cuda")
        out.engine = h
        return out
    if kind == "host":
        h.load(state[2])
        h.run()
        h.store(state[2])
        return state[2].gather()
    if kind == "serve":
        ids = [h.submit(p, lmax) for p, lmax in state[3]]
        return [h.wait(i)[0] for i in ids]
    h.run()
    return h.result()


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _los_sizes(case):
    """Coarse and fine k3 counts and the mean k3 of the pairs a pass works on."""
    k = np.exp(np.linspace(math.log(case["k_min"]), math.log(case["k_max"]), case["k_size"]))
    if case["kind"] == "serve":
        pairs = [p for ps, _ in _jobs(case) for p in ps]
    else:
        pairs = _pairs(case)
    fine, k3 = [], []
    for i1, i2 in pairs:
        lo, hi = _k3_bounds(k, i1, i2)
        nc = case["k3_size"]
        gap = (hi - lo) / (nc - 1)
        n = nc if gap < case["dk_fine"] else int((hi - lo) / case["dk_fine"]) + 1
        fine.append(n)
        k3.append(np.linspace(lo, hi, n))
    return len(pairs), int(sum(fine)), np.concatenate(k3)


def work(case):
    if case["kind"] == "k3int":
        k, off, k3 = _triangle(case)
        n_l = len(_l_list(case["l_size"], case["l_max"]))
        nx = k3.max() * 14400.0 / case["step"]
        terms = 0.0
        for l in _l_list(case["l_size"], case["l_max"]):
            terms += float(np.mean(k3 * 14000.0 > 0.8 * l)) * k3.size * case["n_r"]
        return {"bytes": 8.0 * (k3.size * (2 + n_l) + nx * n_l + n_l * case["n_r"] * (off.size - 1)),
                "flops": 16.0 * terms}
    if case["kind"] == "cl2":
        k, off, k3 = _triangle(case)
        rows = case["l_size"] * len(_m(case))
        return {"bytes": 8.0 * k3.size * (1 + rows * (2 if case["cross"] else 1)) + 8.0 * rows,
                "flops": 10.0 * rows * k3.size}
    n_pairs, F, k3 = _los_sizes(case)
    m, Lm = _m(case), case["L"]
    ls = np.array(_l_list(case["l_size"], case["l_max"]), dtype=float)
    n_mL = sum(Lm + 1 - v for v in m if v <= Lm)
    has_B = case["E"] and m[-1] > 0
    fields = 1 + (1 + int(has_B) if case["E"] else 0)
    n_lm = len(ls) * len(m)
    # live time steps: x = k3 (tau0 - tau) above about l
    tau = np.exp(np.linspace(math.log(200.0), math.log(14000.0), case["tau_size"]))
    x = np.sort(k3)[:: max(1, F // 512), None] * (14200.0 - tau[None, :])
    live = float(np.mean([np.mean(x > 0.95 * l) for l in ls]))
    J_rows = n_mL * len(ls) * (1 + (1 + int(has_B) if case["E"] else 0))
    X = k3.max() * 14000.0 / 0.3
    flops = 0.0
    for v in m:
        nL = max(0, Lm + 1 - v)
        per = 5.0 * nL + 2.0
        n_int = 1 + ((2 if (v and has_B) else 1) + (2 if has_B else 0) if case["E"] else 0)
        flops += n_int * per * len(ls) * F * case["tau_size"] * live
    jb = 4.0 if case["form"] == "fp32c" else 8.0
    src = 8.0 * n_mL * fields * case["tau_size"] * n_pairs * case["k3_size"]
    if case["kind"] == "serve":  # sources and tables are resident and prepared: F values per type
        src = 8.0 * n_mL * fields * case["tau_size"] * F
    return {"bytes": src + jb * J_rows * X * 0.6 + 8.0 * fields * n_lm * F, "flops": flops}


# ---------------------------------------------------------------------------------------------
# the same values in 64 bits, from the inputs alone
# ---------------------------------------------------------------------------------------------
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64,
                           device="cuda" if torch.cuda.is_available() else "cpu")


def _spline_operator(x):
    """Matrix D with D y the second derivatives of the cubic spline through (x, y) whose end
    slopes are those of the parabolas through the three end points."""
    n = x.size
    A, B = np.zeros((n, n)), np.zeros((n, n))
    h = np.diff(x)
    for i in range(1, n - 1):
        A[i, i - 1:i + 2] = h[i - 1] / 6, (h[i - 1] + h[i]) / 3, h[i] / 6
        B[i, i - 1:i + 2] = 1 / h[i - 1], -1 / h[i - 1] - 1 / h[i], 1 / h[i]

    def slope(a, b, c):  # derivative at x[a] of the parabola through a, b, c
        xa, xb, xc = x[a], x[b], x[c]
        s = np.zeros(n)
        s[a] = (2 * xa - xb - xc) / ((xa - xb) * (xa - xc))
        s[b] = (xa - xc) / ((xb - xa) * (xb - xc))
        s[c] = (xa - xb) / ((xc - xa) * (xc - xb))
        return s

    A[0, :2] = h[0] / 3, h[0] / 6
    B[0, 0], B[0, 1] = -1 / h[0], 1 / h[0]
    B[0] -= slope(0, 1, 2)
    A[-1, -2:] = h[-1] / 6, h[-1] / 3
    B[-1, -2], B[-1, -1] = 1 / h[-1], -1 / h[-1]
    B[-1] += slope(n - 1, n - 2, n - 3)
    return np.linalg.solve(A, B)


def _k3_grids(scen, case, pairs):
    """(coarse grid, fine grid, first and last physical fine point) of each pair."""
    lib, s = L.load(), scen.s
    sizes, k = scen.k3_sizes(), scen.grids()[1]
    out = []
    for i1, i2 in pairs:
        n, first, phys = (int(v) for v in sizes[i1 * (i1 + 1) // 2 + i2])
        buf, last = np.zeros(n + case["k3_size"]), C.c_int()
        lib.transfer2_get_k3_list(s["ppr"], s["ppr2"], s["ppt2"], s["pbs"], s["pbs2"], s["ptr2"],
                                  i1, i2, buf.ctypes.data_as(C.POINTER(C.c_double)),
                                  C.byref(last))
        lo, hi = _k3_bounds(k, i1, i2)
        nc = case["k3_size"]
        out.append((lo + np.arange(nc) * (hi - lo) / (nc - 1), buf[:n], first, first + phys - 1))
    return out


def _exact_los(case, seed, pairs):
    """{pair: [tt][fine k3]} from the scenario's inputs."""
    scen = L.Scenario(_config(case, seed))
    scen.prepare()
    m, Lm, nt = _m(case), case["L"], case["tau_size"]
    ls, _, tau = scen.grids()
    ls = [int(v) for v in ls]
    lm = [(il, im) for il, l in enumerate(ls) for im, v in enumerate(m) if v <= l]
    src_lm = [(Lv, im) for Lv in range(Lm + 1) for im, v in enumerate(m) if v <= Lv]
    n_src, n_lm = len(src_lm), len(lm)
    has_E, has_B = case["E"], case["E"] and m[-1] > 0
    fields = 1 + int(has_E) + int(has_B)
    grids = _k3_grids(scen, case, pairs)
    off = np.concatenate([[0], np.cumsum([g[1].size for g in grids])])
    F = int(off[-1])
    t0mt = 14200.0 - tau
    dtau = np.empty(nt)
    dtau[0], dtau[-1] = tau[1] - tau[0], tau[-1] - tau[-2]
    dtau[1:-1] = tau[2:] - tau[:-2]
    X = int(max(g[1].max() for g in grids) * t0mt[0] / 0.3) + 3
    # sources at the fine k3: a linear map of the coarse values, [tp][F][tau]
    S = torch.empty((n_src * fields, F, nt), dtype=torch.float64, device=_t([0.0]).device)
    for q, (p, (kc, fine, first, last)) in enumerate(zip(pairs, grids)):
        ks = np.clip(fine, fine[first], fine[last])
        br = np.clip(np.searchsorted(kc, ks, side="left") - 1, 0, kc.size - 2)
        h = kc[br + 1] - kc[br]
        b = (ks - kc[br]) / h
        a = 1 - b
        A = np.zeros((fine.size, kc.size))
        r = np.arange(fine.size)
        A[r, br] += a
        A[r, br + 1] += b
        if case["cubic_k3"]:
            D = _spline_operator(kc)
            A += ((a ** 3 - a) * h * h / 6)[:, None] * D[br]
            A += ((b ** 3 - b) * h * h / 6)[:, None] * D[br + 1]
        src = _t(np.stack([scen.source(tp, *p) for tp in range(n_src * fields)]))
        S[:, off[q]:off[q + 1]] = torch.matmul(_t(A)[None], src.transpose(1, 2).contiguous())
    S *= _t(dtau)
    # J rows: [X][l] of each (type, L, m), zero where the row is skipped, at the left and at the
    # right node
    def rows(jt, Lv, im):
        left, right = np.zeros((X, len(ls))), np.zeros((X, len(ls)))
        for il, l in enumerate(ls):
            if m[im] > l:
                continue
            xm, v = scen.J_row(jt, Lv, il, im)
            n = min(v.size, X - xm)
            if n > 1:
                left[xm:xm + n, il] = v[:n]
                right[xm:xm + n - 1, il] = v[1:n]
        return _t(left), _t(right)

    kf = _t(np.concatenate([g[1] for g in grids]))
    x = kf[:, None] * _t(t0mt)
    ix = (x / 0.3).to(torch.int64)
    a = (0.3 * (ix + 1).double() - x) / 0.3
    out = torch.zeros((fields * n_lm, F), dtype=torch.float64, device=S.device)
    step = max(1, int(1.5e8 / X))
    rank = [[lm.index((il, im)) if (il, im) in lm else -1 for il in range(len(ls))]
            for im in range(len(m))]
    for sp, (Lv, im) in enumerate(src_lm):
        J = [rows(jt, Lv, im) for jt in range(fields)]  # TT, EE, EB
        idx = [r for r in rank[im]]
        keep = [il for il, r in enumerate(idx) if r >= 0]
        dest = torch.tensor([idx[il] for il in keep], device=S.device)
        for f0 in range(0, F, step):
            f1 = min(F, f0 + step)

            def integral(field, jt):
                s = S[field * n_src + sp, f0:f1]
                res = 0
                for w, Jm in ((a[f0:f1] * s, J[jt][0]), ((1 - a[f0:f1]) * s, J[jt][1])):
                    W = torch.zeros((f1 - f0, X), dtype=torch.float64, device=S.device)
                    W.scatter_add_(1, ix[f0:f1], w)
                    res = res + W @ Jm
                return res.T[keep]

            out[dest, f0:f1] += integral(0, 0)
            if has_E:
                out[n_lm + dest, f0:f1] += integral(1, 1)
            if has_B:
                if m[im]:
                    out[n_lm + dest, f0:f1] += integral(2, 2)
                out[2 * n_lm + dest, f0:f1] += integral(2, 1) - integral(1, 2)
    den = _t([2.0 * ls[il] + 1 for il, _ in lm])
    out = out.view(fields, n_lm, F) * (0.5 / 4 / 2) / den[:, None]
    scen.close()
    return out, off, [ls[il] for il, _ in lm]


def exact(case, seed):
    if case["kind"] == "k3int":
        return _exact_k3int(_consumer_inputs(case, seed))
    if case["kind"] == "cl2":
        return _exact_cl2(_consumer_inputs(case, seed))
    if case["kind"] == "serve":
        allp = _all_pairs(case)
        out, off, l_of = _exact_los(case, seed, allp)
        where = {p: q for q, p in enumerate(allp)}
        res = []
        for ps, lmax in _jobs(case):
            keep = [i for i, l in enumerate(l_of) if l <= lmax]
            cols = np.concatenate([np.arange(off[where[p]], off[where[p] + 1]) for p in ps])
            r = out[:, keep][:, :, torch.as_tensor(cols, device=out.device)]
            res.append(r.reshape(-1, cols.size).cpu().numpy())
        return res
    out, off, _ = _exact_los(case, seed, _pairs(case))
    if case["kind"] == "host":  # (tt, k1, k2 <= k1, k3) order is the load order
        return out.reshape(-1).cpu().numpy()
    return out.reshape(-1, out.shape[-1])


def _exact_k3int(a):
    off, k3, r = a["off"], _t(a["k3"]), _t(a["r"])
    n = np.diff(off)
    dk = np.empty(a["k3"].size)
    dk[1:-1] = a["k3"][2:] - a["k3"][:-2]
    for b, e in zip(off[:-1], off[1:]):
        dk[b], dk[e - 1] = a["k3"][b + 1] - a["k3"][b], a["k3"][e - 1] - a["k3"][e - 2]
    pair = torch.repeat_interleave(torch.arange(n.size), torch.as_tensor(n)).to(k3.device)
    x = k3[None, :] * r[:, None]
    res = torch.zeros((len(a["x_min"]), r.numel(), n.size), dtype=torch.float64, device=k3.device)
    for q, xm in enumerate(a["x_min"]):
        j = _t(a["j"][a["j_off"][q]:a["j_off"][q + 1]])
        y = (x - float(xm)).clamp(min=0) / a["step"]
        i = y.to(torch.int64).clamp(max=j.numel() - 2)
        w = y - i
        f = torch.where(x >= float(xm), (1 - w) * j[i] + w * j[i + 1], 0.0)
        f = f * (k3 * k3 * _t(dk) * _t(a["T"][q]))
        res[q].index_add_(1, pair, f)
    return res.cpu().numpy()


def _exact_cl2(a):
    k, pk, off, k3 = a["k"], a["pk"], a["off"], a["k3"]
    n = k.size
    P = 2 * np.pi ** 2 / k ** 3 * pk

    def half_steps(g, i):  # trapezoid weight of point i of grid g
        lo = g[i] - g[i - 1] if i > 0 else 0.0
        hi = g[i + 1] - g[i] if i + 1 < len(g) else 0.0
        return (lo + hi) / 2

    w = np.zeros(k3.size)
    c2 = np.zeros(k3.size)
    q = 0
    for i1 in range(n):
        for i2 in range(i1 + 1):
            g = k3[off[q]:off[q + 1]]
            dk3 = np.empty(g.size)
            dk3[1:-1] = (g[2:] - g[:-2]) / 2
            dk3[0], dk3[-1] = (g[1] - g[0]) / 2, (g[-1] - g[-2]) / 2
            dk3[0] += g[0] - (k[i1] - k[i2])
            dk3[-1] += (k[i1] + k[i2]) - g[-1]
            d1 = half_steps(k, i1)
            d2 = half_steps(k[:i1 + 1], i2)
            w[off[q]:off[q + 1]] = (2 * k[i1] * k[i2] * g * d1 * d2 * dk3 * P[i1] * P[i2])
            cos = (k[i1] ** 2 + g ** 2 - k[i2] ** 2) / (2 * k[i1] * g)
            c2[off[q]:off[q + 1]] = 1 - cos ** 2
            q += 1
    w *= 2 / np.pi / 2 / np.pi / 2 / np.pi / 2 / np.pi
    n_l, n_m = a["used"].shape
    T1, T2 = _t(a["T1"]).view(n_l, n_m, -1), _t(a["T2"]).view(n_l, n_m, -1)
    res = []
    for im, m in enumerate(a["m"]):
        s = c2 ** m if a["rescale"] else np.ones_like(c2)
        res.append((T1[:, im] * T2[:, im]) @ _t(w * s))
    return torch.stack(res, 1).cpu().numpy()
