"""Performance cases: what a program that uses this engine has it do.

Five kinds of case, each through public entry points:

  step     advance a loaded simulation by `steps` full steps and read the
           state back (the particle records of a snapshot)
  force    one force evaluation of a loaded simulation (Engine.init, the first
           call of every run) and its accelerations
  adjoint  reverse mode: a recorded run and the gradient of its loss with
           respect to the initial state
  abi      the reference host program's sequence over its own C entry points,
           on device arrays: smoothing lengths, list offsets, SPH forces,
           gravity
  sort     the stable (key, value) sort of particle keys

Workloads are the engine's seeded configurations: 1 uniform cube, 2 and 4
Plummer spheres, 3 two polytropes on an encounter, 5 turbulent sphere.
Particles are put in Peano-Hilbert order once, as the engine itself does every
`ph_period` steps.  The repeatedly advanced cases take the bound systems: a
pass is then much the same after some hundred steps (the hot cube and the
turbulent sphere disperse).
"""
import ctypes
import math

import numpy as np
import torch

import cudasph_amd as cs

REAL = {"plain": 4, "mixed": 4, "fp64": 8}
# smoothed neighbour targets give these mean list lengths (self included)
NGB = {0: 34, 1: 33, 2: 51, 3: 66, 4: 51, 5: 65}
PAIR_FLOPS = 20      # one softened gravity pair: distance, 1/s, 1/s^3, four sums
NGB_FLOPS = 150      # one neighbour over density, EOS viscosity, hydro, reaction


def _step(name, form, config, n, steps, far=False):
    return {"name": name, "kind": "step", "form": form, "config": config, "n": n, "steps": steps, "far": far}


def listed():
    return [
        # a test problem: so small that launches and waits are all there is
        _step("step_mixed_1k", "mixed", 2, 1000, 1),
        # a small Plummer sphere, advanced between two outputs
        _step("step_mixed_16k", "mixed", 2, 16384, 5),
        # the Plummer sphere of the adjoint workload, run forward
        _step("step_mixed_65k", "mixed", 4, 65536, 4),
        # the first force evaluation of a Plummer sphere whose size is no
        # multiple of anything
        {"name": "force_mixed_250k", "kind": "force", "form": "mixed", "config": 2, "n": 250007},
        # the headline: two polytropes at 2^20, one step
        _step("step_mixed_1M", "mixed", 3, 1048576, 1),
        # the drop-in FP32 form, small and in a ragged middle size
        _step("step_plain_16k", "plain", 2, 16384, 5),
        _step("step_plain_100k", "plain", 2, 100003, 2),
        # the FP64 reference run that the others are checked against
        _step("step_fp64_50k", "fp64", 4, 50021, 2),
        # the optional multipole far field on the turbulent sphere
        _step("step_far_1M", "mixed", 5, 1048576, 1, far=True),
        # gradient of 20 steps, checkpointed every 5
        {"name": "adjoint_65k", "kind": "adjoint", "config": 4, "n": 65536, "steps": 20, "ckpt": 5},
        # the reference's host program on its own constants (spline softening)
        {"name": "abi_16k", "kind": "abi", "config": 0, "n": 16384},
        # Peano-Hilbert or cell keys of a large simulation
        {"name": "sort_1M", "kind": "sort", "n": 1000003, "bits": 30},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mixed", "mixed", "plain", "fp64", "far", "force", "adjoint", "abi", "sort"])
    config = rng.choice([1, 2, 3, 5])
    if kind in ("mixed", "plain", "fp64", "far"):
        lo, hi = {"mixed": (700, 1000000), "plain": (700, 300000), "fp64": (700, 200000), "far": (70000, 1000000)}[kind]
        n = _size(rng, lo, hi)
        # the polytropes only where their particles resolve them
        config = rng.choice([3, 5] if kind == "far" else [2, 3] if n >= 20000 else [2])
        steps = rng.randint(1, 5 if n < 40000 else 2 if n < 200000 else 1)
        c = _step("", "mixed" if kind == "far" else kind, config, n, steps, kind == "far")
        del c["name"]
        return c
    if kind == "force":
        form = rng.choice(["mixed", "plain", "fp64"])
        return {"kind": kind, "form": form, "config": config, "n": _size(rng, 700, 400000 if form == "mixed" else 150000)}
    if kind == "adjoint":
        n = _size(rng, 1000, 60000)
        steps = rng.randint(1, 12)
        return {"kind": kind, "config": rng.choice([1, 4]), "n": n, "steps": steps, "ckpt": rng.randint(1, 6)}
    if kind == "abi":
        return {"kind": kind, "config": rng.choice([0, 1, 4]), "n": 256 * _size(rng, 4, 250)}
    return {"kind": "sort", "n": _size(rng, 300, 8000000), "bits": rng.choice([16, 22, 30, 32])}


# ---------------------------------------------------------------------------
def _engine(form, config, n, seed):
    e = cs.make_engine(form, config, n, seed, ph_sort=True, i_order=0)
    e.sync()
    return e


def _n_norm(c, j):      # the list slot layout: counts rounded up to j, at least j
    return torch.clamp((c + j - 1) // j * j, min=j)


def _abi_params(config, n):
    return cs.default_params(n) if config == 0 else cs.preset_params(config, n)


def _prepare_abi(case, seed):
    n = case["n"]
    p = _abi_params(case["config"], n)
    pos, vel, hyd = cs.generate_ic(case["config"] or 1, n, seed)
    nd = p.n_dev
    tree, _ = cs.build_kd_tree(pos.astype(np.float32), nd)

    def dev(a, pad=0.0):
        out = torch.full((nd, 4), pad, dtype=torch.float32, device="cuda")
        out[:n] = torch.from_numpy(np.ascontiguousarray(a)).to(device="cuda", dtype=torch.float32)
        return out

    ids = torch.arange(nd, dtype=torch.int32, device="cuda")
    far = torch.tensor([1e10, 1e10, 1e10, 0.0], device="cuda")
    s = {"p": p, "n": n, "nd": nd, "pos": dev(pos), "vel": dev(vel), "hydro": dev(hyd),
         "tree": torch.from_numpy(tree[: nd + 1].copy()).cuda(), "hash": torch.stack([ids, ids], 1).contiguous(),
         "map": torch.zeros(nd, dtype=torch.int32, device="cuda"),
         "n_ngb": torch.zeros(nd, dtype=torch.int32, device="cuda"),
         "list": torch.zeros(100 * nd, dtype=torch.int32, device="cuda"),
         "acc": torch.zeros(100 * nd, dtype=torch.float32, device="cuda"),
         "off": torch.zeros(nd, dtype=torch.int32, device="cuda")}
    s["pos"][n:] = far
    s["vel"][n:] = far
    for name in ("dots", "bdots", "hydro2", "grav", "gpos", "gvel"):
        s[name] = torch.zeros((nd, 4), dtype=torch.float32, device="cuda")
    L = cs.lib()
    vp, ci, cf = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    L.host_solve_range.argtypes = [ci, ci, cf] + [vp] * 6 + [ci]
    L.host_solve_range.restype = cf
    L.host_sph_accelerations.argtypes = [ci, ci, cf, cf] + [vp] * 10 + [ci]
    L.host_sph_accelerations.restype = cf
    L.compute_CUDA_gravity.argtypes = [ci, vp, vp, vp, ci, ci, ci]
    L.compute_CUDA_gravity.restype = None
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "abi":
        return dict(_prepare_abi(case, seed), kind=kind)
    if kind == "sort":
        g = torch.Generator(device="cuda").manual_seed(seed)
        n = case["n"]
        keys = torch.randint(0, 1 << case["bits"], (n,), generator=g, device="cuda").to(torch.int32)
        src = torch.stack([keys, torch.arange(n, dtype=torch.int32, device="cuda")], 1).contiguous()
        L = cs.lib()
        L.sph_radix_sort_noalloc.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_uint] * 2 + [ctypes.c_void_p]
        L.sph_radix_sort_noalloc.restype = ctypes.c_int
        return {"kind": kind, "src": src, "data": torch.empty_like(src), "alt": torch.empty_like(src),
                "bits": case["bits"]}
    e = _engine("fp64" if kind == "adjoint" else case["form"], case["config"], case["n"], seed)
    if case.get("far"):
        e.set_scalar("grav_far", 1)
    if kind == "step":
        e.init()
        e.sync()
    return dict(case, engine=e)


def run(s):
    kind = s["kind"]
    if kind == "step":
        e, n = s["engine"], s["n"]
        e.step(s["steps"])
        return {k: e.get(k, n) for k in ("pos", "vel", "hydro")}
    if kind == "force":
        e, n = s["engine"], s["n"]
        e.init()
        return {k: e.get(k, n) for k in ("grav", "bdots", "hydro")}
    if kind == "adjoint":
        e = s["engine"]
        loss = e.adjoint_forward(s["steps"], s["ckpt"])
        gx, gv, gu = e.adjoint_backward()
        return {"loss": np.array([loss]), "gx": gx, "gv": gv, "gu": gu}
    L = cs.lib()
    if kind == "sort":
        s["data"].copy_(s["src"])
        stream = torch.cuda.current_stream().cuda_stream
        if L.sph_radix_sort_noalloc(s["data"].data_ptr(), s["alt"].data_ptr(), len(s["data"]), s["bits"], stream):
            raise RuntimeError(L.sph_last_error().decode())
        return s["data"]
    p, n, nd = s["p"], s["n"], s["nd"]
    at = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}
    L.sph_abi_set_params(ctypes.byref(p), 0)
    L.host_solve_range(nd, n, p.rel_err, at["hash"], at["map"], at["pos"], at["vel"], at["tree"], at["n_ngb"], 0)
    ends = torch.cumsum(_n_norm(s["n_ngb"], 4), 0, dtype=torch.int32)
    s["off"][1:] = ends[:-1]
    total = int(ends[-1])
    L.host_sph_accelerations(nd, total, p.av_alpha, p.av_beta, at["hash"], None, at["map"], at["list"], at["off"],
                             at["hydro"], at["dots"], at["bdots"], at["hydro2"], at["acc"], 0)
    s["gpos"][:, :3] = s["pos"][:, :3]
    s["gpos"][:, 3] = s["vel"][:, 3]
    s["gvel"][:, :3] = s["vel"][:, :3]
    s["gvel"][:, 3] = s["pos"][:, 3] ** 2
    L.compute_CUDA_gravity(nd, at["grav"], at["gpos"], at["gvel"], 256, 1, 0)
    return {"pos": s["pos"][:n], "hydro": s["hydro"][:n], "dots": s["dots"][:n], "bdots": s["bdots"][:n],
            "grav": s["grav"][:n], "n_ngb": s["n_ngb"][:n]}


# ---------------------------------------------------------------------------
def _sizes(case):
    """(particles, list entries, gravity pairs) of one force evaluation."""
    n = case["n"]
    return n, n * NGB[case["config"]], 0 if case.get("far") else n * n


def work(case):
    """One pass: the state in and out (and its copy to the host), and the
    arithmetic of the neighbour and gravity pairs.  The far field has no
    fixed count of gravity pairs: only its neighbours are counted."""
    kind = case["kind"]
    if kind == "sort":
        passes = -(-case["bits"] // 8)
        return {"bytes": 16 * case["n"], "flops": passes * case["n"]}
    n, entries, pairs = _sizes(case)
    evaluation = NGB_FLOPS * entries + PAIR_FLOPS * pairs
    if kind == "abi":
        return {"bytes": 16 * 9 * n, "flops": evaluation}
    if kind == "adjoint":
        # forward evaluations with gravity; backward the same pairs' gradients
        # (about twice a pair's arithmetic) over every evaluation
        evals = case["steps"] + 1
        return {"bytes": evals * 32 * 12 * n, "flops": 3 * evals * evaluation}
    record = 4 * REAL[case["form"]]
    return {"bytes": 12 * record * n, "flops": case.get("steps", 1) * evaluation}


def exact(case, seed):
    """The Plummer accelerations and potentials in 64 bits for one force
    evaluation.  Everything else goes through the smoothing lengths, which the
    solver fixes only to its tolerance, so no other value is exact for it."""
    n = case["n"]
    if case["kind"] != "force" or n > 400000:
        return None
    s = prepare(case, seed)
    e = s["engine"]
    x = torch.from_numpy(e.get("pos64" if case["form"] == "mixed" else "pos")[:n, :3].copy()).double().cuda()
    m = torch.from_numpy(e.get("vel")[:n, 3].copy()).double().cuda()
    eps2 = float(np.float32(s["engine"].params.grav_eps)) ** 2
    out = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    chunk = max(1, (1 << 27) // n)
    for i0 in range(0, n, chunk):
        xi = x[i0:i0 + chunk]
        d2 = torch.full((len(xi), n), eps2, dtype=torch.float64, device="cuda")
        for k in range(3):
            d2 += (x[:, k][None, :] - xi[:, k][:, None]).square_()
        inv = d2.rsqrt_()
        out[i0:i0 + chunk, 3] = -(inv @ m)
        w = inv * inv * inv * m
        out[i0:i0 + chunk, :3] = w @ x - w.sum(1, keepdim=True) * xi
    return {"grav": out, "bdots": None, "hydro": None}
