"""Workloads of the event-loop engine, for timing it and comparing its outputs.

A case is a plain dict.  Its "path" says which public entry point it goes through:

  closure     Engine.simulate_batch: the drop-in for one call of the reference's per-batch closure, as a host
              program that keeps its own scheduler calls it (one accumulator back, the generator state advanced)
  run         Engine.run: a whole run, per-batch accumulators and their fold back on the host, what the
              command-line tool and run_simulation do
  device      Engine.run_device: the same run with accumulators and fold left in device memory
  adjoint     Engine.adjoint_device: integrand and its derivatives at points of a stream or at given points
  flow-train  Flow.set_params, Flow.train, Flow.get_params: training of the proposal from given weights
  flow-run    Flow.run_device: the weighted event loop on the trained proposal

The run configuration is the shipped `valeurs`; the generator seeds, given points and flow weights come from the
seed.  exact() evaluates the same quantities in float64 with torch alone.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "3photons-rust_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "3photons-rust_amd"))

import trois_photons as tp  # noqa: E402

VALEURS = os.path.join(ROOT, "tests", "golden", "valeurs")
BATCH = tp.BATCH_SIZE
PRECISIONS = {"f64": tp.PREC_F64, "mixed": tp.PREC_MIXED, "f32": tp.PREC_F32}

# Algorithmic operations of one plain event (each +, -, *, /, sqrt, sin, cos, ln counted once, pass rate 0.708) and
# of one pass of a sample through the flow's six networks (two per multiply-add, without the biases).
EVENT_FLOPS = 852.3
FLOW_FLOPS = 2 * 6 * (16 * 64 + 64 * 64 + 64 * 32)
ACC_BYTES = 104
FLOW_CHUNK = 6144 * BATCH  # a weighted run takes its flow share from every chunk of this many events


def _sim(name, path, rng, events, precision="f64", seeding="skipahead", sort=True, faster=False):
    return {"name": name, "path": path, "rng": rng, "events": events, "precision": precision, "seeding": seeding,
            "sort": sort, "faster": faster}


def listed():
    return [
        # One closure call of 10 000 events, the reference's batch, on its default stream: a scheduler of the
        # user's own in sequential mode.  Launches and latency count here.
        _sim("closure-ranf", "closure", "ranf", 10_000),
        # The same on the standard-random stream, an odd number of events.
        _sim("closure-xoshiro", "closure", "xoshiro", 4_321),
        # The reference's default build on the shipped configuration: 1e7 events, RANF, f64.
        _sim("run-default-1e7", "run", "ranf", 10_000_000),
        # standard-random with faster-threading seeding, a short ragged run (a scan over parameters takes many).
        _sim("run-xoshiro-jump", "run", "xoshiro", 1_234_567, seeding="jump"),
        # The f32 build of the reference on the shipped configuration.
        _sim("run-f32-1e7", "run", "ranf", 10_000_000, precision="f32"),
        # The faster-evgen build on the shipped configuration.
        _sim("run-faster-evgen-1e7", "run", "ranf", 10_000_000, faster=True),
        # High statistics, the headline benchmark: 1e9 events, accumulators left in device memory.
        _sim("device-xoshiro-1e9", "device", "xoshiro", 1_000_000_000),
        # Mixed precision, a tenth of that and not a whole number of batches.
        _sim("device-mixed-1e8", "device", "xoshiro", 99_999_999, precision="mixed"),
        # Everything the reference's fastest build turns on: f32, faster-evgen, faster-threading, standard-random.
        _sim("device-faster-f32-5e7", "device", "xoshiro", 50_000_000, precision="f32", seeding="jump", faster=True),
        # Values and derivatives of the integrand at a million points of the stream.
        {"name": "adjoint-f64", "path": "adjoint", "precision": "f64", "points": 1 << 20, "given": False},
        # Training of the proposal at the default batch (64 of its 2000 steps).
        {"name": "flow-train", "path": "flow-train", "batch": 65536, "steps": 64},
        # The weighted event loop at the default mixture share.
        {"name": "flow-run-2e7", "path": "flow-run", "events": 20_000_000, "alpha": 0.7},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["closure", "closure", "run", "run", "run", "device", "device", "adjoint", "flow-train", "flow-run"])
    if path == "adjoint":
        return {"path": path, "precision": rng.choice(["f64", "f32"]), "points": _log_int(rng, 64, 1 << 21),
                "given": rng.random() < 0.5}
    if path == "flow-train":
        return {"path": path, "batch": 16 * _log_int(rng, 64, 4096), "steps": rng.randint(16, 64)}
    if path == "flow-run":
        return {"path": path, "events": _log_int(rng, 10_000, 60_000_000), "alpha": rng.choice([0.7, 0.7, 0.9, 0.5])}
    c = {"path": path, "rng": rng.choice(["ranf", "xoshiro"]), "precision": rng.choice(["f64", "f64", "f64", "mixed", "f32"]),
         "seeding": "skipahead" if path == "closure" else rng.choice(["skipahead", "jump"]),
         "sort": rng.random() < 0.8, "faster": rng.random() < 0.25}
    if c["precision"] == "mixed":
        c["faster"] = False
    if path == "closure":
        c["events"] = _log_int(rng, 1, 640_000)
    elif path == "run":
        c["events"] = _log_int(rng, 10_000, 100_000_000)
    else:
        c["events"] = _log_int(rng, 1_000_000, 600_000_000 if c["rng"] == "xoshiro" and c["precision"] != "f32" else 200_000_000)
    if c["faster"]:
        c["events"] = min(c["events"], 100_000_000 - rng.randint(0, 50_000_000))
    return c


# ---- what a program keeps ---------------------------------------------------------------------------------------

_state = {}


def _engine():
    if "engine" not in _state:
        _state["engine"] = tp.Engine(0)
    return _state["engine"]


def _kind(case):
    if case["rng"] == "ranf":
        return tp.RNG_RANF
    return tp.RNG_XOSHIRO128 if case["precision"] == "f32" else tp.RNG_XOSHIRO


def _rng(case, seed):
    # RANF's seeds lie below its modulus, 1e9 (faster-threading adds 123 456 a batch)
    return tp.rng_state(_kind(case), seed % 500_000_000 if case["rng"] == "ranf" else seed)


def _params(events, precision="f64", sort=True, faster=False):
    cfg = tp.Configuration.load(VALEURS).with_events(events)
    return tp.params_from_config(cfg, sort=sort, precision=PRECISIONS[precision], faster_evgen=faster)


def _points(case, seed):
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    return torch.rand(case["points"], 12, dtype=torch.float64, device="cuda:0", generator=g)


def _flow_weights(seed):
    """Hidden layers as they are initialised, and an output layer of the size training gives it."""
    r = np.random.default_rng(seed)
    w = np.zeros((6, 7328), np.float32)
    b1, b2 = 1 / math.sqrt(12), 1 / math.sqrt(64)
    w1 = r.uniform(-b1, b1, (6, 64, 16))
    w1[:, :, 12:] = 0
    w[:, :1024] = w1.reshape(6, -1)
    w[:, 1024:1088] = r.uniform(-b1, b1, (6, 64))
    w[:, 1088:5184] = r.uniform(-b2, b2, (6, 4096))
    w[:, 5184:5248] = r.uniform(-b2, b2, (6, 64))
    w3 = r.normal(0, 0.02, (6, 32, 64))
    b3 = r.normal(0, 0.02, (6, 32))
    for a in (w3, b3):
        a[:, 12:16] = 0
        a[:, 28:] = 0
    w[:, 5248:7296] = w3.reshape(6, -1)
    w[:, 7296:] = b3
    return w.reshape(-1)


def prepare(case, seed):
    eng, path, dev = _engine(), case["path"], torch.device("cuda:0")
    s = {"case": case, "path": path, "engine": eng}
    if path == "adjoint":
        n, dt = case["points"], torch.float32 if case["precision"] == "f32" else torch.float64
        s["params"] = _params(n)
        s["rng"] = tp.rng_state(tp.RNG_XOSHIRO, seed)
        s["u"] = _points(case, seed) if case["given"] else None
        s["out"] = [torch.empty(n, 5, dtype=dt, device=dev), torch.empty(n, 5, 12, dtype=dt, device=dev),
                    torch.empty(n, 5, 12, dtype=dt, device=dev)]
        return s
    if path == "flow-train":
        s["params"] = _params(case["batch"])
        s["flow"], s["weights"] = tp.Flow(eng), _flow_weights(seed)
        s["opts"] = tp.flow_default_opts(batch=case["batch"], steps=case["steps"], seed=seed)
        return s
    n = case["events"]
    nb = -(-n // BATCH)
    if path == "flow-run":
        s["params"] = _params(n)
        s["flow"] = tp.Flow(eng)
        s["flow"].set_params(_flow_weights(seed))
        s["key"] = seed
    else:
        s["params"] = _params(n, case["precision"], case["sort"], case["faster"])
        s["rng"] = _rng(case, seed)
    if path in ("device", "flow-run"):
        s["per"] = torch.empty(nb, 13, dtype=torch.float64, device=dev)
        s["merged"] = torch.empty(13, dtype=torch.float64, device=dev)
    return s


def _accs(words):
    """Accumulators, an array or tensor (.., 13) of float64, as their fields."""
    whole = words.view(torch.int64) if isinstance(words, torch.Tensor) else words.view(np.int64)
    return {"selected": whole[..., 0], "spm2": words[..., 1:6], "vars": words[..., 6:11], "sigma": words[..., 11],
            "variance": words[..., 12]}


def run(s):
    case, path, eng = s["case"], s["path"], s["engine"]
    if path == "closure":
        st = type(s["rng"]).from_buffer_copy(s["rng"])
        acc = eng.simulate_batch(s["params"], _kind(case), st, case["events"])
        return {"acc": _accs(np.frombuffer(acc, np.float64)), "rng": np.frombuffer(st, np.int32)}
    if path == "run":
        per, merged, _ = eng.run(s["params"], _kind(case), tp.SEEDINGS[case["seeding"]], s["rng"], case["events"])
        return {"batches": _accs(per.view(np.float64).reshape(-1, 13)), "run": _accs(np.frombuffer(merged, np.float64))}
    if path == "device":
        eng.run_device(s["params"], _kind(case), tp.SEEDINGS[case["seeding"]], s["rng"], case["events"],
                       s["per"].data_ptr(), s["merged"].data_ptr())
        return {"batches": _accs(s["per"]), "run": _accs(s["merged"])}
    if path == "flow-run":
        s["flow"].run_device(s["params"], case["alpha"], s["key"], case["events"], s["per"].data_ptr(),
                             s["merged"].data_ptr())
        return {"batches": _accs(s["per"]), "run": _accs(s["merged"])}
    if path == "flow-train":
        s["flow"].set_params(s["weights"])
        loss, _ = s["flow"].train(s["params"], s["opts"])
        return {"loss": loss, "weights": s["flow"].get_params()}
    prec = PRECISIONS[case["precision"]]
    ptrs = [t.data_ptr() for t in s["out"]]
    if s["u"] is None:
        eng.adjoint_device(s["params"], case["points"], prec, s["rng"], *ptrs)
    else:
        v = ctypes.c_void_p
        eng._check(tp.lib.tp_adjoint(eng.h, ctypes.byref(s["params"]), tp.RNG_XOSHIRO, None, v(s["u"].data_ptr()),
                                     case["points"], prec, 1, *(v(p) for p in ptrs)), "tp_adjoint")
    return {"F": s["out"][0], "dF_du": s["out"][1], "dF_dp": s["out"][2]}


def work(case):
    path = case["path"]
    if path == "adjoint":
        n, size = case["points"], 4 if case["precision"] == "f32" else 8
        # one forward pass and, for each of the five contributions, a reverse sweep of about twice its work
        return {"bytes": n * (125 * size + (96 if case["given"] else 0)), "flops": n * 11 * EVENT_FLOPS}
    if path == "flow-train":
        n = case["batch"] * case["steps"]
        # network forward and twice that backward, the integrand and its derivative
        return {"bytes": 2 * 4 * tp.FLOW_NPARAM + 4 * case["steps"], "flops": n * (3 * FLOW_FLOPS + 3 * EVENT_FLOPS)}
    n = case["events"]
    out = ACC_BYTES * (1 if path == "closure" else -(-n // BATCH) + 1)
    if path == "flow-run":
        return {"bytes": out + 4 * tp.FLOW_NPARAM, "flops": n * (FLOW_FLOPS + EVENT_FLOPS)}
    return {"bytes": out + 256, "flops": n * EVENT_FLOPS}


# ---- the same quantities in 64 bits -----------------------------------------------------------------------------

def _dev():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _momenta(P, u):
    """RAMBO: photon momenta (n, 3, 4) as (X, Y, Z, E), sorted by decreasing energy if the run sorts."""
    c, phi, e1, e2 = u.reshape(-1, 3, 4).unbind(2)
    cos = 2 * c - 1
    sin = torch.sqrt(1 - cos * cos)
    en = -torch.log(e1 * e2 + 2.2250738585072014e-308)
    q = en.unsqueeze(2) * torch.stack([sin * torch.sin(2 * math.pi * phi), sin * torch.cos(2 * math.pi * phi), cos,
                                       torch.ones_like(cos)], 2)
    r = q.sum(1, keepdim=True)
    rv, re = r[..., :3], r[..., 3]
    m2 = re * re - (rv * rv).sum(2)
    m = torch.sqrt(m2)
    alpha, beta = P.e_total / m2, 1 / (m + re)
    rq = (q[..., :3] * rv).sum(2)
    e = alpha * (re * q[..., 3] - rq)
    v = alpha.unsqueeze(2) * (m.unsqueeze(2) * q[..., :3] + (beta * rq - q[..., 3]).unsqueeze(2) * rv)
    p = torch.cat([v, e.unsqueeze(2)], 2)
    if P.sort_photons:
        order = torch.argsort(p[..., 3].detach(), dim=1, descending=True, stable=True)
        p = torch.gather(p, 1, order.unsqueeze(2).expand(-1, -1, 4))
    return p


def _cuts(P, p):
    e = p[..., 3]
    bad = e.min(1).values < P.e_min
    bad |= (p[..., 0].abs() > P.cut_beam * e).any(1)
    for i, j in ((0, 1), (0, 2), (1, 2)):
        bad |= (p[:, i, :3] * p[:, j, :3]).sum(1) > P.cut_pp * (e[:, i] * e[:, j])
    if P.cut_plane > 0:
        n = torch.linalg.cross(p[:, 0, :3], p[:, 1, :3])
        bad |= n[:, 0].abs() < P.cut_plane * torch.linalg.norm(n, dim=1)
    return ~bad


def _helicity_sums(P, p):
    """The five contributions (n, 5) of events with photon momenta p."""
    half = P.e_total / 2
    xx = [math.sqrt(half), math.sqrt(half)] + [torch.sqrt(p[:, k, 3] + p[:, k, 2]) for k in range(3)]
    fx = [-half / xx[0], half / xx[1]] + [torch.complex(p[:, k, 0], p[:, k, 1]) / xx[2 + k] for k in range(3)]
    s = {(i, j): fx[i] * xx[j] - fx[j] * xx[i] for i in range(5) for j in range(5) if i != j}
    t = {ij: -(v.conj() if isinstance(v, torch.Tensor) else v) for ij, v in s.items()}
    k8 = -2 * math.sqrt(2.)
    ns, nt = k8 * s[0, 1], k8 * t[0, 1]
    mA = mP = X = 0
    for a, b, c in ((2, 3, 4), (2, 4, 3), (3, 4, 2)):  # photons a, b of one helicity, c of the other
        for A, B in ((ns * s[0, c] ** 2 / (s[0, a] * s[0, b] * s[1, a] * s[1, b]), nt * (t[a, b] * s[c, 0]) ** 2),
                     (nt * t[1, c] ** 2 / (t[1, a] * t[1, b] * t[0, a] * t[0, b]), ns * (t[c, 1] * s[a, b]) ** 2)):
            A, B = A * P.g_a, B * P.g_beta_p
            mA = mA + (A * A.conj()).real
            mP = mP + (B * B.conj()).real
            X = X + 2 * A * B.conj()
    Bp = ns * ((t[2, 3] * t[4, 1]) ** 2 + (t[2, 4] * t[3, 1]) ** 2 + (t[3, 4] * t[2, 1]) ** 2) * P.g_beta_m
    Bm = nt * ((s[2, 0] * s[3, 4]) ** 2 + (s[3, 0] * s[2, 4]) ** 2 + (s[4, 0] * s[2, 3]) ** 2) * P.g_beta_m
    return torch.stack([mA, mP, (Bp * Bp.conj()).real + (Bm * Bm.conj()).real, X.real, X.imag], 1)


class _Sums:
    def __init__(self, P, nb):
        self.P, self.nb = P, nb
        self.sel = torch.zeros(nb, dtype=torch.int64, device=_dev())
        self.s = torch.zeros(nb, 12, dtype=torch.float64, device=_dev())
        self.sc = torch.tensor(list(P.sigma_contribs), dtype=torch.float64, device=_dev())

    def add(self, u, batch, weight=None):
        p = _momenta(self.P, u)
        keep = _cuts(self.P, p)
        p, batch = p[keep], batch[keep]
        m = _helicity_sums(self.P, p)
        if weight is not None:
            m = m * weight[keep].unsqueeze(1)
        w = (m * self.sc).sum(1, keepdim=True)
        self.s.index_add_(0, batch, torch.cat([m, m * m, w, w * w], 1))
        self.sel += torch.bincount(batch, minlength=self.nb)

    def fields(self):
        def of(sel, s):
            return {"selected": sel, "spm2": s[..., :5], "vars": s[..., 5:10], "sigma": s[..., 10], "variance": s[..., 11]}
        return of(self.sel, self.s), of(self.sel.sum(), self.s.sum(0))


def _ranf_mul(A, B):
    """A B mod 1e9 for integer matrices below 1e9, each partial sum exact in float64."""
    hi, lo = torch.div(A, 32768, rounding_mode="floor"), A % 32768
    part = [(x.double() @ B.double()).to(torch.int64) % 1_000_000_000 for x in (hi, lo)]
    return (part[0] * 32768 + part[1]) % 1_000_000_000


def _ranf_round(x):
    """The next 55 values of the subtractive generator from x (55, lanes)."""
    a = (x[:24] - x[31:]) % 1_000_000_000
    b = (x[24:48] - a) % 1_000_000_000
    return torch.cat([a, b, (x[48:] - b[:7]) % 1_000_000_000])


def _ranf_uniforms(x, rounds):
    """Uniforms (lanes, 55 rounds) from round states x (55, lanes), each round handed out backwards."""
    out = torch.empty(x.shape[1], rounds, 55, dtype=torch.int32, device=x.device)
    for r in range(rounds):
        out[:, r] = x.flip(0).t()
        x = _ranf_round(x)
    return out.reshape(x.shape[1], -1)


def _ranf_events(st, seeding, n):
    """(uniforms, batch) pieces of a RANF run."""
    dev = _dev()
    x0 = torch.tensor(list(st.numbers)[1:], dtype=torch.int64, device=dev).reshape(55, 1)
    first = 55 - st.index
    if seeding == "jump":
        nb = -(-n // BATCH)
        seed = (torch.arange(nb, dtype=torch.int64) * 123456 + st.seed + 2 ** 31) % 2 ** 32 - 2 ** 31
        x = torch.zeros(56, nb, dtype=torch.int64)
        x[55] = seed
        j, k = seed.clone(), torch.ones(nb, dtype=torch.int64)
        for i in range(1, 55):
            x[21 * i % 55] = k
            j, k = x[21 * i % 55].clone(), j - k
            k = torch.where(k < 0, k + 1_000_000_000, k)
        x = x[1:].to(dev)
        for _ in range(10):
            x = _ranf_round(x)
        x[:, 0] = x0[:, 0]  # the first batch runs on the caller's state
        for b0 in range(0, nb, 500):
            d = _ranf_uniforms(x[:, b0:b0 + 500].contiguous(), 12 * BATCH // 55 + 3)
            for b in range(b0, min(nb, b0 + 500)):
                off, m = first if b == 0 else 0, min(BATCH, n - b * BATCH)
                u = d[b - b0, off:off + 12 * m].reshape(m, 12).double() * 1e-9
                yield u, torch.full((m,), b, device=dev)
        return
    total = -(-(first + 12 * n) // 55)
    rounds = max(1, min(512, -(-total // 256)))
    step = torch.zeros(55, 55, dtype=torch.int64)
    for c in range(55):
        e = torch.zeros(55, 1, dtype=torch.int64)
        e[c] = 1
        step[:, c:c + 1] = _ranf_round(e)
    step, J, k = step.to(dev), torch.eye(55, dtype=torch.int64, device=dev), rounds
    while k:
        J = _ranf_mul(step, J) if k & 1 else J
        step, k = _ranf_mul(step, step), k >> 1
    x = x0
    while x.shape[1] * rounds < total:
        x, J = torch.cat([x, _ranf_mul(J, x)], 1), _ranf_mul(J, J)
    d = _ranf_uniforms(x, rounds).reshape(-1)[first:first + 12 * n].reshape(n, 12)
    for e0 in range(0, n, 1 << 20):
        u = d[e0:e0 + (1 << 20)].double() * 1e-9
        yield u, torch.arange(e0, e0 + len(u), device=dev) // BATCH


def _xo_step(s, bits):
    """One xoshiro256+ (64-bit words) or xoshiro128+ (32-bit words) update of a list of four integers."""
    mask, (a, r) = (1 << bits) - 1, ((17, 45) if bits == 64 else (9, 11))
    t = (s[1] << a) & mask
    s[2] ^= s[0]
    s[3] ^= s[1]
    s[1] ^= s[2]
    s[0] ^= s[3]
    s[2] ^= t
    s[3] = ((s[3] << r) | (s[3] >> (bits - r))) & mask


def _xo_matrix(bits):
    M = torch.zeros(4 * bits, 4 * bits, dtype=torch.float64)
    for c in range(4 * bits):
        s = [0, 0, 0, 0]
        s[c // bits] = 1 << (c % bits)
        _xo_step(s, bits)
        for r in range(4 * bits):
            M[r, c] = (s[r // bits] >> (r % bits)) & 1
    return M.to(_dev())


def _gf2_pow(M, n):
    R = torch.eye(len(M), dtype=torch.float64, device=M.device)
    while n:
        R = (M @ R) % 2 if n & 1 else R
        M, n = (M @ M) % 2, n >> 1
    return R


def _gf2_orbit(M, S, count):
    """[S, M S, M^2 S, ...], `count` blocks of S's columns."""
    width = S.shape[1]
    while S.shape[1] < count * width:
        S, M = torch.cat([S, (M @ S) % 2], 1), (M @ M) % 2
    return S[:, :count * width]


def _shr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def _xo_draw(s, bits):
    """Uniforms of a tensor of states (4, lanes), which step."""
    x = s[0] + s[3]
    if bits == 64:
        u = _shr(x, 11).double() * 2. ** -53
        t = s[1] << 17
    else:
        u = ((x & 0xFFFFFFFF) >> 8).double() * 2. ** -24
        t = (s[1] << 9) & 0xFFFFFFFF
    s[2] ^= s[0]
    s[3] ^= s[1]
    s[1] ^= s[2]
    s[0] ^= s[3]
    s[2] ^= t
    s[3] = (s[3] << 45) | _shr(s[3], 19) if bits == 64 else ((s[3] << 11) | (s[3] >> 21)) & 0xFFFFFFFF
    return u


def _xo_events(st, seeding, n, batch, per=125):
    """(uniforms, batch) pieces of a xoshiro run in batches of `batch` events."""
    bits = 64 if isinstance(st, tp.XoshiroState) else 32
    M, nb, dev = _xo_matrix(bits), -(-n // batch), _dev()
    s0 = torch.tensor([[float((int(w) >> k) & 1)] for w in st.s for k in range(bits)], dtype=torch.float64, device=dev)
    lanes = -(-min(n, batch) // per)
    B = _gf2_pow(M, 12 * batch if seeding == "skipahead" else 1 << (128 if bits == 64 else 64))
    S = _gf2_orbit(_gf2_pow(M, 12 * per), _gf2_orbit(B, s0, nb), lanes)
    place = torch.arange(bits, device=dev).reshape(1, bits, 1)
    s = list((S.reshape(4, bits, -1).to(torch.int64) << place).sum(1))
    at = torch.arange(nb, device=dev).repeat(lanes)
    first = torch.arange(lanes, device=dev).repeat_interleave(nb) * per
    size = torch.clamp(n - at * batch, max=batch)
    for i in range(per):
        u = torch.stack([_xo_draw(s, bits) for _ in range(12)], 1)
        ok = first + i < size
        yield u[ok], at[ok]


def _mix(key, k):
    z = (k + 1) * (0x9E3779B97F4A7C15 - (1 << 64)) + (key if key < 1 << 63 else key - (1 << 64))
    z = (z ^ _shr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ _shr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ _shr(z, 31)


def _flow_layers(seed):
    w = torch.tensor(_flow_weights(seed), dtype=torch.float64, device=_dev()).reshape(6, 7328)
    for l in range(6):
        c = torch.tensor([(tp.FLOW_COND_MASKS[l] >> j) & 1 == 1 for j in range(12)], device=_dev())
        W1, W2, W3 = w[l, :1024].reshape(64, 16)[:, :12], w[l, 1088:5184].reshape(64, 64), w[l, 5248:7296].reshape(32, 64)

        def net(z, c=c, W1=W1, W2=W2, W3=W3, l=l):
            h = torch.nn.functional.hardswish(torch.where(c, z, 0.) @ W1.T + w[l, 1024:1088])
            h = torch.nn.functional.hardswish(h @ W2.T + w[l, 5184:5248])
            o = h @ W3.T + w[l, 7296:]
            return torch.where(c, 0., 1.5 * torch.tanh(o[:, :12])), torch.where(c, 0., o[:, 16:28])
        yield net


def _flow_events(case, seed):
    n, alpha, dev = case["events"], case["alpha"], _dev()
    nets = list(_flow_layers(seed))
    nf = int(math.floor(alpha * n + 0.5))

    def inv(logq):
        return 1 / (alpha * torch.exp(logq) + (1 - alpha))
    for e0 in range(0, nf, 1 << 20):
        k = 12 * torch.arange(e0, min(nf, e0 + (1 << 20)), device=dev).unsqueeze(1) + torch.arange(12, device=dev)
        v = _shr(_mix(seed, k), 41).double() * 2. ** -23 + 2. ** -24
        z, logq = torch.log(v) - torch.log1p(-v), (torch.log(v) + torch.log1p(-v)).sum(1)
        for net in nets:
            sc, t = net(z)
            z, logq = z * torch.exp(sc) + t, logq - sc.sum(1)
        logq = logq + (torch.nn.functional.softplus(z) + torch.nn.functional.softplus(-z)).sum(1)
        yield torch.sigmoid(z), torch.arange(e0, e0 + len(z), device=dev) // BATCH, inv(logq)
    for e0 in range(nf, n, 1 << 20):
        k = 12 * torch.arange(e0 - nf, min(n, e0 + (1 << 20)) - nf, device=dev).unsqueeze(1) + torch.arange(12, device=dev)
        u = _shr(_mix(seed ^ tp.UNIFORM_KEY_XOR, k), 12).double() * 2. ** -52 + 2. ** -53
        z, logq = torch.log(u) - torch.log1p(-u), -(torch.log(u) + torch.log1p(-u)).sum(1)
        for net in reversed(nets):
            sc, t = net(z)
            z, logq = (z - t) * torch.exp(-sc), logq - sc.sum(1)
        logq = logq - (torch.nn.functional.softplus(z) + torch.nn.functional.softplus(-z)).sum(1)
        yield u, torch.arange(e0, e0 + len(z), device=dev) // BATCH, inv(logq)


def _exact_adjoint(case, seed):
    P, n = _params(case["points"]), case["points"]
    if case["given"]:
        u = _points(case, seed)
    else:
        parts = list(_xo_events(tp.rng_state(tp.RNG_XOSHIRO, seed), "skipahead", n, n, per=256))
        lanes = -(-n // 256)
        u = torch.empty(lanes, 256, 12, dtype=torch.float64, device=_dev())
        for i, (x, _) in enumerate(parts):
            u[:len(x), i] = x
        u = u.reshape(-1, 12)[:n]
    out = [torch.empty(n, 5, dtype=torch.float64, device=_dev()), torch.empty(n, 5, 12, dtype=torch.float64, device=_dev()),
           torch.empty(n, 5, 12, dtype=torch.float64, device=_dev())]
    for a in range(0, n, 1 << 18):
        b = min(n, a + (1 << 18))
        v = u[a:b].clone().requires_grad_(True)
        p = _momenta(P, v)
        keep = _cuts(P, p.detach()).unsqueeze(1)
        F = P.ev_weight * _helicity_sums(P, p)
        out[0][a:b] = torch.where(keep, F.detach(), 0.)
        for c in range(5):
            gu, gp = torch.autograd.grad(F[:, c].sum(), (v, p), retain_graph=True)
            out[1][a:b, c] = torch.where(keep, gu, 0.)
            out[2][a:b, c] = torch.where(keep, gp.reshape(-1, 12), 0.)
    return {"F": out[0], "dF_du": out[1], "dF_dp": out[2]}


def exact(case, seed):
    path = case["path"]
    if path == "adjoint":
        return _exact_adjoint(case, seed)
    # training is a chain of rounded steps; faster-evgen runs consume their stream by rejection, one event after
    # another; the rest is left out above sizes that take too long
    if path == "flow-train" or case.get("faster") or case["events"] > 30_000_000:
        return None
    n = case["events"]
    batch = n if path == "closure" else BATCH
    sums = _Sums(_params(n, "f64", case.get("sort", True)), -(-n // batch))
    if path == "flow-run":
        for u, b, w in _flow_events(case, seed):
            sums.add(u, b, w)
    else:
        st = _rng(case, seed)
        if case["rng"] == "ranf":
            for u, b in _ranf_events(st, case["seeding"], n):
                sums.add(u, b if path != "closure" else torch.zeros_like(b))
        else:
            for u, b in _xo_events(st, case["seeding"], n, batch):
                sums.add(u, b)
    per, merged = sums.fields()
    if path == "closure":
        return {"acc": {k: v[0] for k, v in per.items()}, "rng": None}
    return {"batches": per, "run": merged}
