"""Performance cases of the P3T hot path: what is timed, on which inputs, and what a pass
returns.

    listed()            the cases, from the smallest device call to the N = 1M disk
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call (inputs, device state)
    run(state)          one pass through the public entry points (gplum_amd.gpu / the C ABI)
    exact(case, seed)   the same outputs in 64 bits from plain torch, where that is possible
    work(case)          bytes and flops that a pass cannot do without

Kinds of case:

    epep      gplum_calc_force_epep_noalloc: direct EP-EP force and neighbour counts on
              device arrays and the caller's stream
    functor   the per-group functors FDPS calls on host arrays (EP-EP, EP-SP quadrupole and
              monopole in FP32, EP-SP quadrupole in FP64)
    walk      the FDPS MultiWalk dispatch / retrieve pair (list and index form)
    run       a whole small run: particles in, initialisation, 64 soft steps, particles out
    step      the device-resident system: 16 soft steps, then the particles and energies
    hard      batched block-step Hermite of independent clusters (host arrays in place)
    train     the forecaster network's training (forward, backward, Adam) on the device
"""
import ctypes
import math

import numpy as np
import torch

from gplum_amd import abi, gpu, ic

# Parameters of the benchmark's disk (reference parameter file; the power-of-two soft step
# nearest below 2 pi / 64) and of the batched hard workload.
DISK = dict(R_cut0=3.0 * 2 ** (1 / 3), R_cut1=8.0, R_search0=1.1, R_search1=6.0, R_search2=1.1, R_search3=2.0,
            gamma=0.1, eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -4, dt_min=2.0 ** -30,
            n_leaf_limit=8, theta=0.5, collision=1)
HARD = dict(eta=0.01, eta_sun=0.01, eta_0=0.002, eta_sun0=0.002, dt_tree=2.0 ** -4, dt_min=2.0 ** -30, gamma=0.1,
            collision=1)
STEPS = {"step": 16,  # soft steps between two outputs: one time unit (1 / 2 pi year) of dt_tree = 2^-4
         "run": 64}   # the sample run's length
LR = 3e-3             # the forecaster's learning rate
ADAM = (0.9, 0.999, 1e-8)


def listed():
    return [
        # one i-group of a tree walk against its EP list, on device arrays: the smallest call,
        # where latency and the number of workgroups count
        {"name": "epep_group", "kind": "epep", "ni": 117, "nj": 731},
        # a few thousand bodies against a larger set, ragged in both sizes
        {"name": "epep_ragged", "kind": "epep", "ni": 3001, "nj": 10007},
        # direct summation over a whole patch of a disk (the check of a tree force)
        {"name": "epep_patch", "kind": "epep", "ni": 65536, "nj": 65536},
        # one FDPS functor call on host arrays: EP-SP quadrupole of one i-group
        {"name": "functor_epsp", "kind": "functor", "fn": "quad", "ni": 124, "nj": 340},
        # one MultiWalk dispatch of a force call: walks of the sizes that the N = 1M tree has
        {"name": "walk_lists", "kind": "walk", "walks": 200, "quad": 1, "index": 0},
        # the reference's sample run: 64 steps of a ring of 3000 planetesimals, monopole,
        # i-groups of 64
        {"name": "run_ring_3k", "kind": "run", "n": 3000, "mass": 1e-9, "a_in": 0.9, "a_out": 1.1, "quad": 0,
         "group": 64, "forecast": "off"},
        # an ordinary disk on one GPU
        {"name": "step_disk_100k", "kind": "step", "n": 100003, "mass": 1e-11, "a_in": 0.5, "a_out": 2.0, "quad": 1,
         "group": 256, "forecast": "off"},
        # the headline workload: N = 1M, quadrupole, learned candidate sizing
        {"name": "step_disk_1m", "kind": "step", "n": 1000000, "mass": 1e-12, "a_in": 0.5, "a_out": 2.0, "quad": 1,
         "group": 256, "forecast": "network"},
        # the clusters of a disk before runaway growth: pairs to quadruples, many of them
        {"name": "hard_pairs", "kind": "hard", "clusters": 20000, "lo": 2, "hi": 4},
        # clusters of the batched workload's lower range
        {"name": "hard_small", "kind": "hard", "clusters": 300, "lo": 2, "hi": 32},
        # crowded clusters around the one-wave limit and above it
        {"name": "hard_crowded", "kind": "hard", "clusters": 6, "lo": 33, "hi": 100},
        # the forecaster's training at the system's default batch
        {"name": "train_8k", "kind": "train", "n": 8192, "steps": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["epep", "epep", "functor", "walk", "step", "step", "hard", "hard", "train"])
    if kind == "epep":
        ni = _log_int(rng, 1, 65536)
        return {"kind": kind, "ni": ni, "nj": _log_int(rng, 1, min(1 << 20, (1 << 32) // ni))}
    if kind == "functor":
        return {"kind": kind, "fn": rng.choice(["ep", "quad", "mono", "quad64"]), "ni": _log_int(rng, 1, 4096),
                "nj": _log_int(rng, 1, 8192)}
    if kind == "walk":
        return {"kind": kind, "walks": _log_int(rng, 1, 400), "quad": rng.randint(0, 1), "index": rng.randint(0, 1)}
    if kind == "step":
        n = _log_int(rng, 1000, 1000000)
        ring = n < 10000
        return {"kind": "run" if ring else "step", "n": n, "mass": 1e-9 if ring else 1e-6 / n, "a_in": 0.9 if ring else 0.5,
                "a_out": 1.1 if ring else 2.0, "quad": rng.randint(0, 1), "group": rng.choice([64, 128, 256]),
                "forecast": rng.choice(["off", "network", "uniform"])}
    if kind == "hard":
        lo = _log_int(rng, 2, 64)
        hi = min(128, _log_int(rng, lo, 4 * lo))
        most = max(4, int(40000 / hi ** 2))
        return {"kind": kind, "clusters": _log_int(rng, 1, most), "lo": lo, "hi": hi}
    return {"kind": "train", "n": _log_int(rng, 200, 50000), "steps": rng.randint(1, 30)}


# ------------------------------------------------------------------------------ inputs

def _ep_lists(ni, nj, seed):
    """A patch of a planetesimal disk 1e-3 AU wide and two search radii thick: ni i-particles and
    the EP list (its first entries are the i-particles themselves, as in FDPS); a few neighbours
    within the search radius for each, whatever the number of bodies."""
    rng = np.random.default_rng(seed)
    epi, epj = np.zeros(ni, dtype=abi.EPI), np.zeros(nj, dtype=abi.EPJ)
    n = max(ni, nj)
    size = 1e-3
    r0 = size * math.sqrt(4.0 / (math.pi * n))
    pos = np.array([1.0, 0.2, 0.01]) + rng.uniform(-0.5, 0.5, (n, 3)) * np.array([size, size, 2.0 * r0])
    r_search = r0 * rng.uniform(0.8, 1.2, n)
    r_out = r_search / 2.5
    for e, m in ((epi, ni), (epj, nj)):
        e["id_local"] = np.arange(m)
        e["pos"], e["r_out"], e["r_search"] = pos[:m], r_out[:m], r_search[:m]
    epj["id"] = np.arange(nj)
    epj["mass"] = rng.uniform(0.5e-12, 2e-12, nj)
    return epi, epj


def _sp_list(ns, quad, seed):
    """Tree nodes around the patch of _ep_lists: clumps of planetesimals 0.02 to 1 AU away, with
    the second moments of clumps a tenth of their distance wide."""
    rng = np.random.default_rng(seed)
    sp = np.zeros(ns, dtype=abi.SPJ_QUAD if quad else abi.SPJ_MONO)
    d = np.exp(rng.uniform(math.log(0.02), 0.0, ns))
    phi = rng.uniform(0, 2 * math.pi, ns)
    sp["pos"] = np.array([1.0, 0.2, 0.01]) + np.stack([d * np.cos(phi), d * np.sin(phi),
                                                       0.02 * d * rng.normal(size=ns)], 1)
    sp["mass"] = rng.uniform(1e-11, 1e-9, ns)
    if quad:
        a = 0.1 * d[:, None, None] * rng.normal(size=(ns, 3, 3)) / 3.0
        q = sp["mass"][:, None, None] * (a @ a.transpose(0, 2, 1))
        for k, (u, v) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            sp["quad"][:, k] = q[:, u, v]
    return sp


def _walks(case, seed):
    """The walks' particles and lists: i-groups of 16 to 256, EP lists of 100 to 700 and SP
    lists of 100 to 600 (the N = 1M tree: 124, 390 and 340 on average), the sizes fixed by the
    case."""
    rng = np.random.default_rng(1)
    out = []
    for w in range(case["walks"]):
        ni, nj, ns = int(rng.integers(16, 257)), int(rng.integers(100, 701)), int(rng.integers(100, 601))
        epi, epj = _ep_lists(ni, max(ni, nj), [seed, 2, w])
        out.append((epi, epj, _sp_list(ns, case["quad"], [seed, 3, w])))
    return out


def _clusters(case, seed):
    """The batched hard workload's clusters (ic.clusters' law: sizes log-uniform in [lo, hi],
    members Gaussian with sigma = 2 Hill radii of 1e-10 around circular 1 AU orbits, masses
    log-uniform in [1e-12, 1e-8]), the sizes fixed by the case."""
    lo, hi, nc = case["lo"], case["hi"], case["clusters"]
    size = np.random.default_rng(1).uniform(math.log(lo), math.log(hi + 1), nc)
    size = np.clip(np.exp(size).astype(np.int64), lo, hi)
    parts = []
    off = np.concatenate([[0], np.cumsum(size)])
    for n in np.unique(size):
        # the clusters of one size in one call of the generator
        sub, _ = ic.clusters(int((size == n).sum()), seed=[seed, int(n)], size_min=int(n), size_max=int(n))
        parts.append((np.flatnonzero(size == n), sub.reshape(-1, int(n))))
    pp = np.zeros(off[-1], dtype=abi.PARTICLE)
    for which, sub in parts:
        for c, members in zip(which, sub):
            pp[off[c]:off[c + 1]] = members
    pp["id"] = np.arange(off[-1])
    pp["id_cluster"] = np.repeat(off[:-1], size)
    ic.cluster_acc0(pp, off)
    return pp, off


def _train_data(case, seed):
    """Standardised features and Poisson counts of a smooth rate, and the network's initial
    weights (variance 1 / fan-in)."""
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(case["n"], 4)).astype(np.float32)
    y = rng.poisson(np.exp(0.5 * x[:, 0] - 0.3 * x[:, 1] + 0.2 * x[:, 2] * x[:, 3])).astype(np.float32)
    theta = np.zeros(4545, np.float32)
    theta[0:256] = rng.normal(size=256) / 2.0
    theta[320:4416] = rng.normal(size=4096) / 8.0
    theta[4480:4544] = rng.normal(size=64) / 8.0
    return x, y, theta


def _device(a):
    return torch.from_numpy(a.view(np.uint8).reshape(-1).copy()).cuda()


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "epep":
        epi, epj = _ep_lists(case["ni"], case["nj"], seed)
        s["epi"], s["epj"] = _device(epi), _device(epj)
        s["clear"] = _device(abi.cleared_force(case["ni"]))
        s["force"] = torch.empty_like(s["clear"])
    elif kind == "functor":
        epi, s["epj"] = _ep_lists(case["ni"], max(case["ni"], case["nj"]), seed)
        s["epi"] = epi
        s["epj"] = s["epj"][:case["nj"]]
        s["spj"] = _sp_list(case["nj"], case["fn"] != "mono", [seed, 1])
        s["clear"] = abi.cleared_force(case["ni"])
        s["force"] = s["clear"].copy()
    elif kind == "walk":
        walks = _walks(case, seed)
        nw = len(walks)
        s["walks"] = walks
        s["force"] = np.zeros(sum(len(w[0]) for w in walks), dtype=abi.FORCE)

        def table(arrays):
            return (ctypes.c_void_p * nw)(*[a.ctypes.data for a in arrays])

        def counts(arrays):
            return (ctypes.c_int * nw)(*[len(a) for a in arrays])
        s["p_epi"], s["n_epi"] = table([w[0] for w in walks]), counts([w[0] for w in walks])
        s["p_force"] = table(np.split(s["force"], np.cumsum(s["n_epi"])[:-1]))
        s["n_epj"], s["n_spj"] = counts([w[1] for w in walks]), counts([w[2] for w in walks])
        if case["index"]:
            # the tree's whole arrays and each walk's indices into them
            s["epj"] = np.concatenate([w[1] for w in walks])
            s["spj"] = np.concatenate([w[2] for w in walks])
            nj, ns = np.cumsum([0] + list(s["n_epj"])), np.cumsum([0] + list(s["n_spj"]))
            s["idj"] = [np.arange(nj[w], nj[w + 1], dtype=np.int32) for w in range(nw)]
            s["ids"] = [np.arange(ns[w], ns[w + 1], dtype=np.int32) for w in range(nw)]
            s["p_epj"], s["p_spj"] = table(s["idj"]), table(s["ids"])
        else:
            s["p_epj"], s["p_spj"] = table([w[1] for w in walks]), table([w[2] for w in walks])
    elif kind in ("step", "run"):
        pp = ic.disk(case["n"], case["mass"], case["a_in"], case["a_out"], seed=seed)
        s["system"] = gpu.System(gpu.params(quadrupole=case["quad"], n_group_limit=case["group"], **DISK), pp)
        s["system"].set_forecast(case["forecast"])
        if kind == "step":
            s["system"].initialize()
        s["start"] = pp
        s["pp"] = np.zeros(case["n"], dtype=abi.PARTICLE)      # the program's output buffer
    elif kind == "hard":
        s["p"] = gpu.params(**HARD)
        s["pp"], s["off"] = _clusters(case, seed)
    else:
        s["x"], s["y"], s["theta"] = _train_data(case, seed)
    return s


# -------------------------------------------------------------------------------- runs

def _forces(f):
    return {"acc": f["acc"], "phi": f["phi"], "number": f["neighbor"]["number"], "rank": f["neighbor"]["rank"],
            "id_max": f["neighbor"]["id_max"], "id_min": f["neighbor"]["id_min"]}


def run(s):
    case, kind = s["case"], s["kind"]
    if kind == "epep":
        # the caller clears the forces (ForceGrav::clear) and calls on its own stream
        s["force"].copy_(s["clear"])
        gpu.check(gpu.lib().gplum_calc_force_epep_noalloc(
            s["epi"].data_ptr(), case["ni"], s["epj"].data_ptr(), case["nj"], s["force"].data_ptr(), 0.0,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        f = s["force"].view(torch.float32).view(-1, 8)
        return {"acc": f[:, :3], "phi": f[:, 3], "neighbor": f.view(torch.int32)[:, 4:]}
    if kind == "functor":
        np.copyto(s["force"], s["clear"])
        if case["fn"] == "ep":
            gpu.calc_force_epep(s["epi"], s["epj"], s["force"])
        elif case["fn"] == "mono":
            gpu.calc_force_epsp_mono(s["epi"], s["spj"], s["force"])
        elif case["fn"] == "quad":
            gpu.calc_force_epsp_quad(s["epi"], s["spj"], s["force"])
        else:
            acc, phi = gpu.calc_force_epsp_quad_f64(s["epi"], s["spj"], s["force"])
            return dict(_forces(s["force"]), acc64=acc, phi64=phi)
        return _forces(s["force"])
    if kind == "walk":
        L, nw = gpu.lib(), case["walks"]
        mono = "" if case["quad"] else "_mono"
        if case["index"]:
            rc = getattr(L, "gplum_multiwalk_dispatch_index" + mono)(
                0, nw, s["p_epi"], s["n_epi"], s["p_epj"], s["n_epj"], s["p_spj"], s["n_spj"], abi.ptr(s["epj"]),
                len(s["epj"]), abi.ptr(s["spj"]), len(s["spj"]), 1)
        else:
            rc = getattr(L, "gplum_multiwalk_dispatch" + mono)(
                0, nw, s["p_epi"], s["n_epi"], s["p_epj"], s["n_epj"], s["p_spj"], s["n_spj"])
        gpu.check(rc)
        gpu.check(L.gplum_multiwalk_retrieve(0, nw, s["n_epi"], s["p_force"]))
        return _forces(s["force"])
    if kind in ("step", "run"):
        if kind == "run":
            s["system"].set_particles(s["start"])
            s["system"].initialize()
        # the steps between two outputs, then what a snapshot and the energy log hold (mergers
        # leave fewer particles than the buffer holds)
        s["system"].step(STEPS[kind])
        e, n, pp = s["system"].energy(), s["system"].count(), s["pp"]
        gpu.check(gpu.lib().gplum_system_get_particles(s["system"].h, abi.ptr(pp), len(pp)))
        return {"n": n, "id": pp["id"], "mass": pp["mass"], "r_planet": pp["r_planet"], "f": pp["f"], "pos": pp["pos"],
                "vel": pp["vel"], "number": pp["neighbor"]["number"], "flags": pp["flags"], "energy": e}
    if kind == "hard":
        pp = s["pp"].copy()          # integrated in place
        edisp, nblock, _, pairs = gpu.hard_integrate(s["p"], pp, s["off"], prepare=True, counts=True)
        out = {k: pp[k] for k in ("id", "mass", "r_planet", "pos", "vel", "acc_s", "jerk_s", "acc_d", "jerk_d", "phi_s",
                                  "phi_d", "time", "dt", "flags", "n_cluster")}
        return dict(out, edisp=edisp, block_steps=nblock, pairs=pairs)
    theta, first, last = gpu.mlp_train(s["theta"], s["x"], s["y"], case["steps"], LR)
    return {"theta": theta, "first": first, "last": last}


# ------------------------------------------------------------------------------- exact

def _cuda64(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def _ep64(epi, epj, chunk=1 << 25):
    """acc and phi of the EP-EP law in 64 bits: -m / r and m dr / r^3 with r^2 clamped at the
    larger r_out^2."""
    xi, xj, m, ro_i, ro_j = (_cuda64(a) for a in (epi["pos"], epj["pos"], epj["mass"], epi["r_out"], epj["r_out"]))
    acc, phi = torch.zeros_like(xi), torch.zeros(len(xi), dtype=torch.float64, device=xi.device)
    step = max(1, chunk // max(1, len(xj)))
    for b in range(0, len(xi), step):
        d = [xj[None, :, k] - xi[b:b + step, None, k] for k in range(3)]
        r2 = torch.maximum(d[0] ** 2 + d[1] ** 2 + d[2] ** 2, torch.maximum(ro_i[b:b + step, None], ro_j[None]) ** 2)
        mr = m[None] * torch.rsqrt(r2)
        phi[b:b + step] = -mr.sum(1)
        mr /= r2
        for k in range(3):
            acc[b:b + step, k] = (mr * d[k]).sum(1)
    return acc.cpu().numpy(), phi.cpu().numpy()


def _sp64(epi, spj):
    """acc and phi of the EP-SP law in 64 bits (monopole, plus quadrupole where given)."""
    x = spj["pos"][None].astype(np.float64) - epi["pos"][:, None]
    r2 = (x * x).sum(2)
    ri = 1.0 / np.sqrt(r2)
    m = spj["mass"][None]
    acc, phi = (m * ri ** 3)[:, :, None] * x, -m * ri
    if "quad" in spj.dtype.names:
        q = spj["quad"]
        t = np.empty((len(spj), 3, 3))
        for k, (u, v) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            t[:, u, v] = t[:, v, u] = 3.0 * q[:, k]
        t -= (q[:, 0] + q[:, 1] + q[:, 2])[:, None, None] * np.eye(3)
        qr = np.einsum("juv,ijv->iju", t, x)
        rqr = (qr * x).sum(2)
        phi = phi - 0.5 * rqr * ri ** 5
        acc = acc + (2.5 * rqr * ri ** 7)[:, :, None] * x - (ri ** 5)[:, :, None] * qr
    return acc.sum(1), phi.sum(1)


def exact(case, seed):
    kind = case["kind"]
    none = {"number": None, "rank": None, "id_max": None, "id_min": None}
    if kind == "epep":
        acc, phi = _ep64(*_ep_lists(case["ni"], case["nj"], seed))
        return {"acc": acc, "phi": phi, "neighbor": None}
    if kind == "functor":
        epi, epj = _ep_lists(case["ni"], max(case["ni"], case["nj"]), seed)
        if case["fn"] == "ep":
            acc, phi = _ep64(epi, epj[:case["nj"]])
        else:
            acc, phi = _sp64(epi, _sp_list(case["nj"], case["fn"] != "mono", [seed, 1]))
        out = dict(none, acc=acc, phi=phi)
        return dict(out, acc64=acc, phi64=phi) if case["fn"] == "quad64" else out
    if kind == "walk":
        a, f = [], []
        for epi, epj, spj in _walks(case, seed):
            (a0, p0), (a1, p1) = _ep64(epi, epj), _sp64(epi, spj)
            a.append(a0 + a1)
            f.append(p0 + p1)
        return dict(none, acc=np.concatenate(a), phi=np.concatenate(f))
    if kind == "train":
        x, y, theta = _train_data(case, seed)
        x, y, th = _cuda64(x), _cuda64(y), _cuda64(theta).requires_grad_()

        def loss():
            h = torch.tanh(x @ th[0:256].view(64, 4).T + th[256:320])
            h = torch.tanh(h @ th[320:4416].view(64, 64).T + th[4416:4480])
            lam = torch.nn.functional.softplus(h @ th[4480:4544] + th[4544])
            return (lam - y * torch.log(lam + 1e-6)).mean()
        m, v, first = torch.zeros_like(th), torch.zeros_like(th), None
        for t in range(1, case["steps"] + 1):
            now = loss()
            first = float(now.detach()) if first is None else first
            g, = torch.autograd.grad(now, th)
            m = ADAM[0] * m + (1 - ADAM[0]) * g
            v = ADAM[1] * v + (1 - ADAM[1]) * g * g
            with torch.no_grad():
                th -= LR * (m / (1 - ADAM[0] ** t)) / (torch.sqrt(v / (1 - ADAM[1] ** t)) + ADAM[2])
        with torch.no_grad():
            last = float(loss())
        return {"theta": th.detach().cpu().numpy(), "first": first, "last": last}
    return None          # block-step integrations have no closed value


# -------------------------------------------------------------------------------- work

def work(case):
    """Flops per pair: 28 EP-EP, 60 EP-SP quadrupole, 25 EP-SP monopole, 75 FP64 per Hermite pair
    evaluation; the numbers of pairs of trees and of Hermite runs are estimates."""
    kind = case["kind"]
    if kind == "epep":
        return {"bytes": 48 * case["ni"] + 112 * case["nj"] + 64 * case["ni"], "flops": 28.0 * case["ni"] * case["nj"]}
    if kind == "functor":
        size, flop = {"ep": (112, 28), "quad": (80, 60), "mono": (32, 25), "quad64": (80, 60)}[case["fn"]]
        return {"bytes": 112 * case["ni"] + size * case["nj"], "flops": float(flop) * case["ni"] * case["nj"]}
    if kind == "walk":
        w, sp = case["walks"], (80, 60) if case["quad"] else (32, 25)
        return {"bytes": w * (136 * 80 + 400 * 112 + 350 * sp[0]), "flops": w * 136.0 * (400 * 28 + 350 * sp[1])}
    if kind in ("step", "run"):
        # per step: the particles read and written once (pos, vel, soft force and radii), and the
        # interactions of one tree force (their number per particle grows with log N)
        n, per, steps = case["n"], (60 if case["quad"] else 25), STEPS[kind]
        pairs = n * steps * (1.5 * case["group"] * 28 + 17.0 * math.log2(n) * per)
        return {"bytes": steps * n * 2.0 * 150 + 408.0 * n, "flops": pairs}
    if kind == "hard":
        # block steps grow with the cluster: about 25 n^3 pair evaluations per cluster and soft step
        lo, hi = case["lo"], case["hi"] + 1.0
        cube = (hi ** 3 - lo ** 3) / (3.0 * math.log(hi / lo))
        mean = (hi - lo) / math.log(hi / lo)
        return {"bytes": 2 * 408.0 * case["clusters"] * mean, "flops": 75.0 * 25.0 * case["clusters"] * cube}
    n, s = case["n"], case["steps"] + 1
    return {"bytes": 20.0 * n + 2 * 4 * 4545, "flops": s * n * 6.0 * (4 * 64 + 64 * 64 + 64)}
