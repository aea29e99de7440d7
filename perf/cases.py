"""Measured workloads of the solver library.

Each case is one thing a program does with this package through its public
entry points: a history sum or a history block product on device arrays, the
reference program's "Sum" call sequence on the device layer, a whole 1D, 3D,
distributed-order or space-fractional solve, an ensemble in one batch, and a
few requests through the server.  `listed()` gives fixed sizes (those of the
repository's workloads where it names one), `draw()` other sizes of the same
ranges.  `exact()` restates the mathematics in 64 bits with numpy and torch.
"""
import ctypes
import math

import numpy as np
import torch

import fpde_hpc_amd as F

DEV = "cuda:0"
MODE_ID = {"mfma_f64": 1, "split_bf16": 2, "split_f16": 3, "split_bf16x3": 4}


def listed():
    return [
        # a short history summed for one new level: launch and call latency
        {"name": "sum_small", "kind": "sum", "nodes": 1000, "levels": 64, "alpha": 0.8},
        # the longest plain FP64 history sum of the large 1D workload: HBM streaming
        {"name": "sum_large", "kind": "sum", "nodes": 10000, "levels": 20000, "alpha": 0.7},
        # one block of future steps in split bf16 at half of that history
        {"name": "block_bf16", "kind": "block", "mode": "split_bf16", "nodes": 10000, "levels": 9984, "block": 64,
         "alpha": 0.7},
        # a step of the reference program's GPU path: newest level and weights
        # up, "Sum", result down (ragged node count, padded level stride)
        {"name": "device_sum", "kind": "facade", "nodes": 9999, "levels": 4000, "alpha": 0.7, "sum_alg": 0,
         "keep": 1.0},
        # the small 1D workload: N = 1000, M = 2000, Picard
        {"name": "solve_1d_small", "kind": "solve1d", "hist": "split_bf16", "nodes": 1000, "steps": 2000,
         "tau": 1e-3, "alpha": 0.8, "block": 64, "picard": 3, "gamma": 0.0, "orders": 0},
        # the large 1D workload (the benchmark's default): N = 10^4, M = 2 10^4, Picard
        {"name": "solve_1d_large", "kind": "solve1d", "hist": "split_bf16", "nodes": 10000, "steps": 20000,
         "tau": 5e-4, "alpha": 0.7, "block": 64, "picard": 3, "gamma": 0.0, "orders": 0},
        # the distributed-order workload: 32 orders, split fp16
        {"name": "solve_1d_orders", "kind": "solve1d", "hist": "split_f16", "nodes": 4000, "steps": 10000,
         "tau": 5e-4, "alpha": 0.5, "block": 64, "picard": 3, "gamma": 0.0, "orders": 32},
        # the default history form (plain FP64), lagged coefficients as the reference steps
        {"name": "solve_1d_plain", "kind": "solve1d", "hist": "plain", "nodes": 3001, "steps": 1500,
         "tau": 5e-4, "alpha": 0.7, "block": 64, "picard": 1, "gamma": 0.0, "orders": 0},
        # the space-fractional scheme in 1D
        {"name": "solve_1d_space", "kind": "solve1d", "hist": "split_bf16", "nodes": 4000, "steps": 600,
         "tau": 1e-3, "alpha": 0.8, "block": 64, "picard": 1, "gamma": 0.8, "orders": 0},
        # the 3D workload: 128^3, M = 1000
        {"name": "solve_3d_large", "kind": "solve3d", "hist": "split_bf16", "nodes": 128, "steps": 1000,
         "tau": 1e-3, "alpha": 0.85, "block": 64},
        # an ensemble over alpha in one batch: six N = 10^4 solves
        {"name": "ensemble", "kind": "batch", "count": 6, "nodes": 10000, "steps": 2000, "tau": 5e-4, "block": 64,
         "hist": "split_bf16"},
        # sixteen uneven requests through the server (80% 1D, 20% 3D, a quarter distributed order)
        {"name": "serve", "kind": "serve", "count": 16, "nodes": 20000, "steps": 3000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sum", "block", "facade", "solve1d", "solve1d", "solve1d", "solve3d", "solve3d", "batch",
                       "serve"])
    alpha = round(rng.uniform(0.3, 0.95), 3)
    if kind == "sum":
        nodes = _log(rng, 300, 20000)
        return {"kind": kind, "nodes": nodes, "levels": _log(rng, 16, min(20000, 200000000 // nodes)), "alpha": alpha}
    if kind == "block":
        mode = rng.choice(["mfma_f64", "split_bf16", "split_f16", "split_bf16x3"])
        nodes = _log(rng, 300, 20000)
        levels = _log(rng, 64, min(20000, 150000000 // nodes))
        if mode != "mfma_f64":
            levels = max(32, levels // 32 * 32)
        return {"kind": kind, "mode": mode, "nodes": nodes, "levels": levels, "block": rng.choice([16, 32, 64, 128]),
                "alpha": alpha}
    if kind == "facade":
        nodes = _log(rng, 300, 20000)
        return {"kind": kind, "nodes": nodes, "levels": _log(rng, 32, min(8000, 40000000 // nodes)), "alpha": alpha,
                "sum_alg": rng.choice([0, 0, 1]), "keep": round(rng.uniform(0.2, 0.9), 3)}
    if kind == "solve1d":
        hist = rng.choice(["plain", "mfma_f64", "split_bf16", "split_bf16", "split_f16", "split_bf16x3"])
        gamma = round(rng.uniform(0.5, 0.95), 3) if rng.random() < 0.2 else 0.0
        slow = hist == "plain" or gamma > 0.0
        return {"kind": kind, "hist": hist, "nodes": _log(rng, 300, 16000), "steps": _log(rng, 200, 1500 if slow else 6000),
                "tau": rng.choice([5e-4, 1e-3]), "alpha": alpha, "block": rng.choice([32, 64, 64, 128]),
                "picard": rng.choice([1, 3, 3]), "gamma": gamma, "orders": rng.choice([0, 0, 0, 16])}
    if kind == "solve3d":
        return {"kind": kind, "hist": rng.choice(["plain", "mfma_f64", "split_bf16", "split_bf16", "split_f16"]),
                "nodes": _log(rng, 24, 128), "steps": _log(rng, 60, 300), "tau": 1e-3, "alpha": alpha,
                "block": rng.choice([32, 64])}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(2, 10), "nodes": _log(rng, 1000, 10000),
                "steps": _log(rng, 300, 2000), "tau": 5e-4, "block": rng.choice([64, 128]),
                "hist": rng.choice(["split_bf16", "split_bf16", "split_f16", "mfma_f64"])}
    return {"kind": kind, "count": rng.randint(4, 12), "nodes": _log(rng, 2000, 20000), "steps": _log(rng, 500, 2500)}


# ---------------------------------------------------------------------------
# inputs
def _head_1d(n, rng):
    """Initial head -1 + four sine modes of random amplitude and phase."""
    z = np.linspace(0.0, 1.0, n)
    u = np.full(n, -1.0)
    for k in range(1, 5):
        u += rng.uniform(0.0, 0.05) * np.sin(k * np.pi * z + rng.uniform(0.0, 2.0 * np.pi))
    return u


def _head_3d(n, rng):
    """Initial head -1 + eight Gaussian blobs, depth fastest, then x, then y."""
    z = np.linspace(0.0, 1.0, n)
    u = np.full((n, n, n), -1.0)
    for _ in range(8):
        c, s, a = rng.uniform(0.2, 0.8, 3), rng.uniform(0.05, 0.15), rng.uniform(0.0, 0.05)
        g = [np.exp(-(z - c[d]) ** 2 / (2.0 * s * s)) for d in range(3)]
        u += a * g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    return u.reshape(-1)


def _lags(n, alpha, tau=5e-4):
    """Toeplitz L1 weights (times 1/(Gamma(1-alpha) tau)) of lags 1..n."""
    j = np.arange(1, n + 1, dtype=np.float64)
    e = 1.0 - alpha
    return tau ** e / e * j ** e * np.expm1(e * np.log1p(1.0 / j)) / (math.gamma(e) * tau)


def _history(nodes, ld, levels, seed):
    """Level differences D[t][i] of a relaxing field, smooth in both, padded to ld."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    t = torch.arange(levels, dtype=torch.float64, device=DEV)[:, None]
    D = torch.zeros(levels, ld, dtype=torch.float64, device=DEV)
    z = torch.linspace(0.0, 1.0, nodes, dtype=torch.float64, device=DEV)[None, :]
    p = torch.rand(6, generator=g, dtype=torch.float64, device=DEV).cpu().numpy()
    D[:, :nodes] = torch.sin(6.0 * z + 6.28 * p[0]) * (1e-3 * (t + 1.0) ** (-0.5 - 0.3 * p[1]))
    D[:, :nodes] += 1e-6 * (0.5 + p[2]) * torch.cos(40.0 * z * p[3] + 0.01 * t)
    return D


def _facade_inputs(case, seed):
    """Levels U^0..U^n [levels+1][os], weights kb, step lengths, the cut of sum_alg 1."""
    nodes, n = case["nodes"], case["levels"]
    os_ = -(-nodes // 16) * 16
    U = torch.cumsum(_history(nodes, os_, n + 1, seed), 0) - 1.0
    U[:, nodes:] = 0.0
    tau = 5e-4 * (1.0 + 0.2 * np.random.default_rng(seed + 7).random(n + 1))
    T = np.concatenate([[0.0], np.cumsum(tau)])
    e = 1.0 - case["alpha"]
    kb = ((T[n + 1] - T[:n]) ** e - (T[n + 1] - T[1:n + 1]) ** e) / e
    cut = float(kb[int((1.0 - case["keep"]) * (n - 1))])
    return os_, U, tau, T, kb, cut


def _spec_1d(case, u0):
    kw = dict(do_q=case["orders"], do_rule=0, do_a0=0.1, do_a1=1.0) if case["orders"] else {}
    return F.make_spec(case["nodes"], case["steps"], case["tau"], alpha=case["alpha"], hist_mode=case["hist"],
                       block=case["block"], picard_max=case["picard"], picard_tol=1e-12 if case["picard"] > 1 else 0.0,
                       u_top=float(u0[0]), gamma=case["gamma"], **kw)


def _specs_batch(case, seed):
    rng = np.random.default_rng(seed)
    specs, u0s = [], []
    for i in range(case["count"]):
        u0 = _head_1d(case["nodes"], rng)
        specs.append(F.make_spec(case["nodes"], case["steps"], case["tau"], hist_mode=case["hist"],
                                 alpha=0.5 + 0.4 * i / max(1, case["count"] - 1), block=case["block"], picard_max=3,
                                 picard_tol=1e-12, u_top=float(u0[0]), chunk_rows=256))
        u0s.append(u0)
    return specs, u0s


def _requests(case, seed):
    """A mix of requests: the shapes follow from the case alone, the fields and orders from the seed."""
    shape = np.random.default_rng(case["count"] * 1000003 + case["nodes"] * 31 + case["steps"])
    rng = np.random.default_rng(seed)
    reqs = []
    for i in range(case["count"]):
        alpha = float(rng.uniform(0.3, 0.95))
        kw = dict(do_q=16, do_rule=0, do_a0=0.1, do_a1=1.0) if i % 4 == 3 else {}
        if i % 5 == 4:
            n, m = int(shape.integers(32, 65)), int(shape.integers(100, 301))
            u0 = _head_3d(n, rng)
            spec = F.make_spec(n, m, 1e-3, alpha=alpha, dims=3, block=32, hist_mode="split_bf16", u_top=float(u0[0]), **kw)
        else:
            n = int(shape.integers(500, case["nodes"] + 1))
            m = int(shape.integers(case["steps"] // 3, case["steps"] + 1))
            u0 = _head_1d(n, rng)
            spec = F.make_spec(n, m, 5e-4, alpha=alpha, block=128, chunk_rows=256, hist_mode="split_bf16",
                               u_top=float(u0[0]), **kw)
        reqs.append((spec, u0))
    return reqs


class _Facade:
    """The device-layer objects of the reference program's history sum."""

    def __init__(self, case, seed):
        self.L = L = F.lib()
        self.n, self.nodes = case["levels"], case["nodes"]
        self.os, U, self.tau, self.T, self.kb, cut = _facade_inputs(case, seed)
        self.alpha, self.cut = case["alpha"], cut
        host = U.cpu().numpy()
        self.newest = host[self.n].copy()
        self.ctx, self.prog, self.kern = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        F.check(L.fpde_cl_ctx_create(0, ctypes.byref(self.ctx)))
        text = f"#define sum_alg {case['sum_alg']}\n#define OS {self.os}\n#define BS 16\n"
        F.check(L.fpde_cl_program_create(self.ctx, text.encode(), ctypes.byref(self.prog)))
        F.check(L.fpde_cl_kernel_create(self.prog, b"Sum", ctypes.byref(self.kern)))
        self.S, self.old = self._buf(np.zeros(self.os)), self._buf(host)
        self.btau, self.bkb = self._buf(self.tau), self._buf(np.zeros(self.n + 1))
        self.bH, self.bC = self._buf(np.zeros(8)), self._buf(np.zeros(8))

    def _buf(self, a):
        b = ctypes.c_void_p()
        F.check(self.L.fpde_cl_buf_alloc(self.ctx, a.nbytes, a.ctypes.data, ctypes.byref(b)))
        return b

    def call(self):
        L, k, n, os_ = self.L, self.kern, self.n, self.os
        F.check(L.fpde_cl_buf_write(self.ctx, self.bkb, 0, 8 * n, self.kb.ctypes.data))
        F.check(L.fpde_cl_buf_write(self.ctx, self.old, 8 * n * os_, 8 * os_, self.newest.ctypes.data))
        F.check(L.fpde_cl_buf_write(self.ctx, self.btau, 8 * n, 8, self.tau[n:].ctypes.data))
        for i, b in ((0, self.S), (1, self.old), (3, self.btau), (4, self.bH), (5, self.bC), (6, self.bkb)):
            F.check(L.fpde_cl_kernel_set_buffer_arg(k, i, b))
        for i, v in ((2, n + 1), (11, n)):
            F.check(L.fpde_cl_kernel_set_arg(k, i, 4, ctypes.byref(ctypes.c_int(v))))
        for i, v in ((7, self.cut), (8, self.T[n + 1]), (9, self.T[n]), (10, self.alpha)):
            F.check(L.fpde_cl_kernel_set_arg(k, i, 8, ctypes.byref(ctypes.c_double(v))))
        g, l = (ctypes.c_size_t * 1)(os_), (ctypes.c_size_t * 1)(16)
        F.check(L.fpde_cl_launch(self.ctx, k, 1, g, l))
        F.check(L.fpde_cl_finish(self.ctx))
        out = np.empty(self.nodes)
        F.check(L.fpde_cl_buf_read(self.ctx, self.S, 0, 8 * self.nodes, out.ctypes.data))
        return out

    def __del__(self):
        for b in (self.S, self.old, self.btau, self.bkb, self.bH, self.bC):
            self.L.fpde_cl_buf_free(b)
        self.L.fpde_cl_kernel_destroy(self.kern)
        self.L.fpde_cl_program_destroy(self.prog)
        self.L.fpde_cl_ctx_destroy(self.ctx)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("sum", "block"):
        nodes, n = case["nodes"], case["levels"]
        ld = -(-nodes // 64) * 64
        s.update(ld=ld, D=_history(nodes, ld, -(-n // 32) * 32, seed))
        if kind == "sum":
            s["w"] = torch.from_numpy(_lags(n, case["alpha"])).to(DEV)
            s["S"] = torch.zeros(nodes, dtype=torch.float64, device=DEV)
        else:
            w = np.zeros(n + case["block"] + 512)
            w[:n + case["block"]] = _lags(n + case["block"], case["alpha"])
            s["w"] = torch.from_numpy(w).to(DEV)
            s["P"] = torch.zeros(case["block"], ld, dtype=torch.float64, device=DEV)
        torch.cuda.synchronize()
    elif kind == "facade":
        s["facade"] = _Facade(case, seed)
    elif kind in ("solve1d", "solve3d"):
        rng = np.random.default_rng(seed)
        if kind == "solve1d":
            s["u0"] = _head_1d(case["nodes"], rng)
            spec = _spec_1d(case, s["u0"])
        else:
            s["u0"] = _head_3d(case["nodes"], rng)
            spec = F.make_spec(case["nodes"], case["steps"], case["tau"], alpha=case["alpha"], dims=3,
                               hist_mode=case["hist"], block=case["block"], u_top=float(s["u0"][0]))
        s["solver"] = F.Solver(spec)
    elif kind == "batch":
        specs, s["u0"] = _specs_batch(case, seed)
        s["solvers"] = [F.Solver(sp) for sp in specs]
    else:
        s["requests"] = _requests(case, seed)
        s["server"] = F.Server(48 << 30, max_active=16)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    L = F.lib()
    if kind == "sum":
        F.check(L.fpde_history_sum_f64(state["S"].data_ptr(), state["D"].data_ptr(), case["levels"], case["nodes"],
                                       state["ld"], state["w"].data_ptr()))
        return state["S"]
    if kind == "block":
        F.check(L.fpde_history_block_gemm(MODE_ID[case["mode"]], state["D"].data_ptr(), state["ld"], case["nodes"],
                                          state["D"].shape[0], case["levels"], case["levels"], case["block"],
                                          state["w"].data_ptr(), state["P"].data_ptr()))
        return state["P"][:, :case["nodes"]]
    if kind == "facade":
        return state["facade"].call()
    if kind in ("solve1d", "solve3d"):
        sv = state["solver"]
        sv.reset(state["u0"])
        sv.advance()
        return sv.solution()
    if kind == "batch":
        for sv, u0 in zip(state["solvers"], state["u0"]):
            sv.reset(u0)
        F.advance_batch(state["solvers"])
        return [sv.solution() for sv in state["solvers"]]
    srv = state["server"]
    ids = [srv.submit(spec, u0) for spec, u0 in state["requests"]]
    srv.run()
    return [srv.result(i) for i in ids]


def _solve_work(unknowns, steps, iters):
    # every level kept once and read once at least; the history products and
    # about 100 operations per unknown and line solve
    return {"bytes": 16.0 * unknowns * steps, "flops": 1.0 * unknowns * steps * (steps + 100.0 * iters)}


def work(case):
    kind = case["kind"]
    if kind == "sum":
        n, m = case["nodes"], case["levels"]
        return {"bytes": 8.0 * (n * m + m + n), "flops": 2.0 * n * m}
    if kind == "block":
        n, m, b = case["nodes"], case["levels"], case["block"]
        return {"bytes": 8.0 * (n * m + m + b + n * b), "flops": 2.0 * n * m * b}
    if kind == "facade":
        n, m = case["nodes"], case["levels"] * (case["keep"] if case["sum_alg"] == 1 else 1.0)
        return {"bytes": 8.0 * (n * m + 2 * m + 2 * n), "flops": 4.0 * n * m}
    if kind == "solve1d":
        w = _solve_work(case["nodes"], case["steps"], 1 if case["picard"] == 1 else 2)
        if case["gamma"] > 0.0:
            w["flops"] += 1.0 * case["nodes"] ** 2 * case["steps"]
        return w
    if kind == "solve3d":
        return _solve_work(case["nodes"] ** 3, case["steps"], 3)
    if kind == "batch":
        w = _solve_work(case["nodes"], case["steps"], 2)
        return {k: v * case["count"] for k, v in w.items()}
    total = {"bytes": 0.0, "flops": 0.0}
    for spec, u0 in _requests(case, 0):
        w = _solve_work(u0.size, spec.steps, 3 if spec.dims == 3 else 1)
        total = {k: total[k] + w[k] for k in total}
    return total


# ---------------------------------------------------------------------------
# the same quantities in 64 bits, by plain array code
def _vgm(u, z, ksat):
    """K and 1/C of the van Genuchten-Mualem soil (n = 5/4, a = 0.066, s0 = 0.0736, s1 = 0.55)."""
    m = 0.2
    P = np.maximum(z - u, 1e-300)
    y = 100.0 * 0.066 * P
    x = y ** 1.25
    w = 1.0 + x
    r = w ** -m
    c = r * y ** 0.25
    t = 1.0 / (w * ((((c + 1.0) * c + 1.0) * c + 1.0) * c + 1.0))     # 1 - c, without cancellation
    dry = z - u > 0.0
    return (np.where(dry, ksat * np.sqrt(r) * t * t, ksat),
            np.where(dry, 4.0 * w * P / ((0.55 - 0.0736) * x * r), 1e20))


def _orders(case):
    """(order, weight) pairs of the discrete derivative."""
    if not case.get("orders"):
        return [(case["alpha"], 1.0)]
    x, w = np.polynomial.legendre.leggauss(case["orders"])
    a = 0.1 + 0.9 * (x + 1.0) / 2.0
    return [(float(p), float(0.45 * q * math.gamma(3.0 - p) / 2.0)) for p, q in zip(a, w)]


def _series_weight(a, p0, p1, pa, eps=1e-5):
    """Weight of an old interval by its binomial series, stopped at the first term within eps."""
    total, v1, v2, v6, i = 0.0, 1.0, pa ** -a * p1, p0 / p1, 0
    while True:
        if i == 0:
            v3 = (p1 - p0) / p1
        else:
            v1 *= (a + i - 1.0) / i
            v2 *= p1 / pa
            v6 *= p0 / p1
            v3 = (1.0 - v6) / (i + 1.0)
        term = v1 * v2 * v3
        total += term
        i += 1
        if abs(term) <= eps:
            return total


def _weights(orders, h, n):
    """Coefficient of the newest interval, lag weights 1..n, weights of the
    two oldest intervals per row [n][2] (their series), on a uniform grid h."""
    local, lag, old = 0.0, np.zeros(n), np.zeros((n, 2))
    for a, c in orders:
        if a == 1.0:
            continue
        g = c / math.gamma(1.0 - a)
        local += g * h ** (1.0 - a) / (1.0 - a) / h
        lag += c * _lags(n, a, h)
        for k in range(1, n):
            old[k, 0] += g / h * _series_weight(a, 0.0, h, (k + 1) * h)
            if k >= 2:
                old[k, 1] += g / h * _series_weight(a, h, 2.0 * h, (k + 1) * h)
    return local, lag, old


def _tridiag(a, b, c, d):
    """Cyclic reduction of a x_{i-1} + b x_i + c x_{i+1} = d."""
    n = len(d)
    a, c, d = a / b, c / b, d / b
    s = 1
    while s < n:
        z = np.zeros(s)
        am, cm, dm = (np.concatenate([z, v[:-s]]) for v in (a, c, d))
        ap, cp, dp = (np.concatenate([v[s:], z]) for v in (a, c, d))
        q = 1.0 / (1.0 - a * cm - c * ap)
        a, c, d = -a * am * q, -c * cp * q, (d - a * dm - c * dp) * q
        s *= 2
    return d


def _solve_1d(case, u0):
    N, M, tau, gamma = case["nodes"], case["steps"], case["tau"], case["gamma"]
    h = 1.0 / (N - 1)
    spec = _spec_1d(case, u0)
    ksat, z = spec.ksat, h * np.arange(N)
    L, lag, old = _weights(_orders(case), tau, M)
    kap, T = 1.0, None
    if gamma > 0.0:
        # rows i: sum over j = 1..i-1 of the interval weights (Toeplitz lag i-j, series for j = 1, 2)
        loc, sl, so = _weights([(gamma, 1.0)], h, N)
        kap = loc * h
        idx = torch.arange(N, device=DEV)
        d = idx[:, None] - idx[None, :]
        lagt = torch.from_numpy(np.concatenate([[0.0], sl * h, [0.0]])).to(DEV)
        T = torch.where((d >= 1) & (idx[None, :] >= 1), lagt[d.clamp(0, N)], torch.zeros((), dtype=torch.float64, device=DEV))
        so = torch.from_numpy(so * h).to(DEV)
        T[2:, 1] = so[1:N - 1, 0]
        T[3:, 2] = so[2:N - 1, 1]
    u, top = u0.copy(), u0[0]
    D = torch.zeros(M, N, dtype=torch.float64, device=DEV)
    w = torch.from_numpy(lag).to(DEV).flip(0)
    prev = None
    for n in range(M):
        S = np.zeros(N)
        if n >= 1:
            wt = w[M - n:].clone()
            wt[0] = old[n, 0]
            if n >= 2:
                wt[1] = old[n, 1]
            S = (wt @ D[:n]).cpu().numpy()
        E = None
        if T is not None:
            K, _ = _vgm(u, z, ksat)
            Fl = np.zeros(N)
            Fl[1:-1] = (K[1:-1] * (u[2:] - u[1:-1]) - K[:-2] * (u[1:-1] - u[:-2])) / h ** 2
            E = (T @ torch.from_numpy(Fl).to(DEV)).cpu().numpy()
        it = 2.0 * u - prev if case["picard"] > 1 and prev is not None else u
        for k in range(case["picard"]):
            K, iC = _vgm(it, z, ksat)
            a, b, c, d = np.zeros(N), np.ones(N), np.zeros(N), np.zeros(N)
            a[1:-1] = K[:-2] * iC[1:-1] / h ** 2 * kap
            c[1:-1] = K[1:-1] * iC[1:-1] / h ** 2 * kap
            b[1:-1] = -(a[1:-1] + c[1:-1] + L)
            d[1:-1] = -L * u[1:-1] + S[1:-1] - (iC[1:-1] * E[1:-1] if E is not None else 0.0)
            d[0], a[-1] = top, -1.0
            new = _tridiag(a, b, c, d)
            step, it = np.max(np.abs(new - it)), new
            if step <= 1e-12 and case["picard"] > 1:
                break
        prev, u = u, it
        D[n] = torch.from_numpy(u - prev).to(DEV)
    return u


def _lines(A, B, C, Dr):
    """Thomas along the last axis for many lines (torch, in 64 bits)."""
    n = Dr.shape[-1]
    cs, ds = [C[..., 0] / B[..., 0]], [Dr[..., 0] / B[..., 0]]
    for i in range(1, n):
        q = 1.0 / (B[..., i] - A[..., i] * cs[-1])
        cs.append(C[..., i] * q)
        ds.append((Dr[..., i] - A[..., i] * ds[-1]) * q)
    x = [ds[-1]]
    for i in range(n - 2, -1, -1):
        x.append(ds[i] - cs[i] * x[-1])
    return torch.stack(x[::-1], -1)


def _vgm_t(u, z, ksat):
    K, iC = _vgm(u.cpu().numpy(), z.cpu().numpy(), ksat)
    return torch.from_numpy(K).to(DEV), torch.from_numpy(iC).to(DEV)


def _solve_3d(case, u0):
    n, M, tau = case["nodes"], case["steps"], case["tau"]
    h = 1.0 / (n - 1)
    ksat = F.make_spec(n, M, tau, dims=3, u_top=float(u0[0])).ksat
    L, lag, old = _weights([(case["alpha"], 1.0)], tau, M)
    u = torch.from_numpy(u0.reshape(n, n, n)).to(DEV)            # [y][x][z]
    z = (h * torch.arange(n, dtype=torch.float64, device=DEV)).expand(n, n, n)
    top = u[:, :, 0].clone()
    D = torch.zeros(M, n ** 3, dtype=torch.float64, device=DEV)
    w = torch.from_numpy(lag).to(DEV).flip(0)

    def sweep(u, axis, S):
        v, zz = u.movedim(axis, 2), z.movedim(axis, 2)
        K, iC = _vgm_t(v.contiguous(), zz.contiguous(), ksat)
        a, b, c, d = torch.zeros_like(K), torch.ones_like(K), torch.zeros_like(K), torch.zeros_like(K)
        a[..., 1:-1] = K[..., :-2] * iC[..., 1:-1] / h ** 2
        c[..., 1:-1] = K[..., 1:-1] * iC[..., 1:-1] / h ** 2
        b[..., 1:-1] = -(a[..., 1:-1] + c[..., 1:-1] + L)
        d[..., 1:-1] = -L * v[..., 1:-1]
        if S is not None:
            d[..., 1:-1] += S.movedim(axis, 2)[..., 1:-1]
        a[..., -1] = -1.0
        if axis == 2:
            d[..., 0] = top
        else:
            c[..., 0] = -1.0
        return _lines(a, b, c, d).movedim(2, axis)

    for m in range(M):
        S = None
        if m >= 1:
            wt = w[M - m:].clone()
            wt[0] = old[m, 0]
            if m >= 2:
                wt[1] = old[m, 1]
            S = (wt @ D[:m]).reshape(n, n, n)
        before = u
        u = sweep(sweep(sweep(u, 0, S), 1, None), 2, None)
        D[m] = (u - before).reshape(-1)
    return u.cpu().numpy().reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sum", "block"):
        nodes, n = case["nodes"], case["levels"]
        D = _history(nodes, -(-nodes // 64) * 64, -(-n // 32) * 32, seed)[:n, :nodes]
        if kind == "sum":
            w = torch.from_numpy(_lags(n, case["alpha"])).to(DEV).flip(0)
            return w @ D
        lag = torch.from_numpy(_lags(n + case["block"], case["alpha"])).to(DEV)
        # row r: weight of lag n + r - t at level t
        r, t = torch.arange(case["block"], device=DEV)[:, None], torch.arange(n, device=DEV)[None, :]
        return lag[n + r - t - 1] @ D
    if kind == "facade":
        _, U, tau, _, kb, cut = _facade_inputs(case, seed)
        n = case["levels"]
        lo = 0
        if case["sum_alg"] == 1:
            # newest first in chunks of 16; a full chunk with every |kb| < cut is the last one taken
            t = n - 1
            while t >= 0:
                if t >= 15 and np.all(np.abs(kb[t - 15:t + 1]) < cut):
                    lo = t - 15
                    break
                t -= 16
        c = torch.from_numpy(kb[lo:] / tau[lo:n]).to(DEV)
        return (c @ (U[lo + 1:n + 1] - U[lo:n]))[:case["nodes"]].cpu().numpy()
    if kind == "solve1d":
        rows = case["steps"] * (1 if case["picard"] == 1 else 2)
        cost = rows * (6e-4 + 3e-7 * case["nodes"]) + case["steps"] * (2e-4 + 1e-5 * max(1, case["orders"]))
        return _solve_1d(case, _head_1d(case["nodes"], np.random.default_rng(seed))) if cost < 10.0 else None
    if kind == "solve3d":
        cost = case["steps"] * (3 * case["nodes"] * 1.5e-4 + 8e-7 * case["nodes"] ** 3)
        if cost > 12.0:
            return None
        return _solve_3d(case, _head_3d(case["nodes"], np.random.default_rng(seed)))
    return None
