"""The work that is timed when the framework's speed is measured.

Each case is one call (or one step) that a simulation program makes through `lib.Context`, on
inputs that already live on the GPU.  `listed()` names the cases, `draw()` gives more of the same
ranges, `prepare()` makes the inputs and the context, `run()` is one pass, `work()` what a pass
cannot do without and `exact()` the result in plain 64-bit torch where that is affordable.

Kinds:
  gravity    one Barnes-Hut RHS of a Plummer sphere
  leapfrog   one drift-RHS-kick step of the same
  sph        one SPH RHS of the Sedov start (a slightly jittered lattice, energy in the centre)
  blast      one predictor-corrector Euler step of a blast wave half-way through its run
  cloud      one self-gravitating SPH RHS of a turbulent isothermal cloud
  train      Adam steps of the learned smoothing length on a finished RHS's pairs
  sums       energies, momenta and centre of mass of a particle set
  keys       the allocation-free sort of space-filling-curve keys
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from miluphpc_amd import ics, lib

N_NB = 64          # target neighbour count
FLOAT_OUT = ("ax", "ay", "az", "rho", "p", "drhodt", "dedt", "dsmldt")


def listed() -> list[dict]:
    return [
        # an interactive or test-sized N-body run: one leapfrog step of a few thousand bodies,
        # where launches and latency are everything
        dict(name="nbody_step_2048", kind="leapfrog", n=2048, theta=0.5, eps2=1e-6, curve=1, mac=0, quad=0,
             accept=1, fp32=0, dt=5e-4),
        # the plain method's standard size: FP64 monopole Barnes-Hut with potential
        dict(name="plummer_65536_fp64", kind="gravity", n=65536, theta=0.5, eps2=1e-6, curve=1, mac=0, quad=0,
             accept=1, fp32=0, potential=1),
        # a mid-size sphere of a ragged count in the mixed-precision form, the library's default vote
        dict(name="plummer_300007_quad", kind="gravity", n=300007, theta=0.6, eps2=4e-8, curve=1, mac=0, quad=1,
             accept=1, fp32=1, potential=0),
        # the large production sphere: quadrupole, box acceptance, FP32 pair sums
        dict(name="plummer_16m_quad_box", kind="gravity", n=16777216, theta=0.6, eps2=4e-8, curve=1, mac=0, quad=1,
             accept=0, fp32=1, potential=0),
        # the smallest SPH run: a 16^3 test blast's RHS
        dict(name="sedov_16_rhs", kind="sph", side=16, curve=0, kernel=1, fp32=0, lists=1),
        # an ordinary odd-sized SPH RHS in the reference's structure (count, then a full list walk)
        dict(name="sedov_47_two_walks", kind="sph", side=47, curve=0, kernel=1, fp32=0, lists=0),
        # the headline: one predictor-corrector step (two RHS) of the evolving 2M-particle blast
        dict(name="blast_128_step", kind="blast", side=128, curve=0, kernel=1, fp32=0, lists=1),
        # the largest SPH RHS
        dict(name="sedov_256_rhs", kind="sph", side=256, curve=0, kernel=1, fp32=0, lists=1),
        # collapse run: self-gravity and SPH together, FP32 pair sums, Hilbert order
        dict(name="cloud_1m_rhs", kind="cloud", n=1048576, theta=0.5, curve=1, kernel=1, fp32=1, lists=1),
        # online training of the learned smoothing length between two steps
        dict(name="train_65536x20", kind="train", n=262144, samples=65536, iters=20),
        # the conservation log of every output step
        dict(name="sums_2m", kind="sums", n=2097152),
        # key sort in a serving loop that must not allocate, an odd count
        dict(name="keys_1000003", kind="keys", n=1000003),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng) -> dict:
    kind = rng.choice(["gravity", "gravity", "leapfrog", "sph", "sph", "blast", "cloud", "train", "sums", "keys"])
    if kind in ("gravity", "leapfrog"):
        c = dict(kind=kind, n=_log_int(rng, 1000, 2000000), theta=round(rng.uniform(0.4, 0.8), 3), eps2=1e-6,
                 curve=rng.randrange(2), mac=0, quad=rng.randrange(2), accept=rng.randrange(2), fp32=rng.randrange(2))
        if kind == "gravity":
            c["potential"] = rng.randrange(2)
        else:
            c["dt"] = 5e-4
        return c
    if kind == "sph":
        return dict(kind=kind, side=_log_int(rng, 10, 150), curve=rng.randrange(2), kernel=rng.choice([1, 1, 2, 4]),
                    fp32=rng.randrange(2), lists=rng.randrange(2))
    if kind == "blast":
        return dict(kind=kind, side=_log_int(rng, 14, 130), curve=rng.randrange(2), kernel=1, fp32=0, lists=1)
    if kind == "cloud":
        return dict(kind=kind, n=_log_int(rng, 4000, 1000000), theta=round(rng.uniform(0.4, 0.8), 3), curve=1,
                    kernel=1, fp32=rng.randrange(2), lists=rng.randrange(2))
    if kind == "train":
        return dict(kind=kind, n=_log_int(rng, 8000, 300000), samples=_log_int(rng, 1000, 200000),
                    iters=rng.randrange(5, 41))
    if kind == "sums":
        return dict(kind=kind, n=_log_int(rng, 1000, 16000000))
    return dict(kind=kind, n=_log_int(rng, 256, 2097152))


# ---- inputs --------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(0x5eed0000 + seed)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _isotropic(g, n):
    ct = _rand(g, n) * 2.0 - 1.0
    ph = _rand(g, n) * (2.0 * math.pi)
    st = torch.sqrt(1.0 - ct * ct)
    return torch.stack([st * torch.cos(ph), st * torch.sin(ph), ct])


def _plummer(n: int, seed: int) -> dict:
    """Plummer sphere, G = M = a = 1, cut at 10 a, equal masses, isotropic velocities drawn from the
    distribution function, in the centre-of-mass frame."""
    g = _gen(seed)
    umax = (1.0 + 1.0 / 100.0) ** -1.5
    r = 1.0 / torch.sqrt((_rand(g, n) * umax + 1e-12) ** (-2.0 / 3.0) - 1.0)
    pos = _isotropic(g, n) * r
    q = torch.linspace(0.0, 1.0, 4097, device="cuda", dtype=torch.float64)
    cdf = torch.cumsum(q * q * (1.0 - q * q) ** 3.5, 0)
    cdf = cdf / cdf[-1]
    speed = q[torch.searchsorted(cdf, _rand(g, n)).clamp(max=4096)] * math.sqrt(2.0) * (1.0 + r * r) ** -0.25
    vel = _isotropic(g, n) * speed
    pos = pos - pos.mean(1, keepdim=True)
    vel = vel - vel.mean(1, keepdim=True)
    m = torch.full((n,), 1.0 / n, device="cuda", dtype=torch.float64)
    return dict(x=pos[0].contiguous(), y=pos[1].contiguous(), z=pos[2].contiguous(), vx=vel[0].contiguous(),
                vy=vel[1].contiguous(), vz=vel[2].contiguous(), mass=m)


def _lattice(side: int, jitter: float, g) -> torch.Tensor:
    c = -0.5 + (torch.arange(side, device="cuda", dtype=torch.float64) + 0.5) / side
    z, y, x = torch.meshgrid(c, c, c, indexing="ij")
    pos = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)])
    return pos + jitter / side * (_rand(g, *pos.shape) - 0.5)


def _sedov(side: int, seed: int) -> dict:
    """The Sedov start: unit mass on a lattice (jittered by a hundredth of its spacing), background
    energy 1e-6, unit energy deposited around the centre, every h at 64 neighbours."""
    g = _gen(seed)
    pos = _lattice(side, 0.02, g)
    n = side ** 3
    h0 = ics.h_for_neighbours(float(n), N_NB)
    r = torch.sqrt((pos * pos).sum(0))
    q = r / (2.0 * h0)
    w = torch.where(q <= 0.5, 6 * q ** 3 - 6 * q ** 2 + 1, 2 * (1 - q).clamp(min=0.0) ** 3)
    m = torch.full((n,), 1.0 / n, device="cuda", dtype=torch.float64)
    e = 1e-6 * (1.0 + 0.1 * _rand(g, n)) + w / (m * w).sum()
    v = 1e-3 * _randn(g, 3, n)
    one = torch.ones_like(m)
    return dict(x=pos[0].contiguous(), y=pos[1].contiguous(), z=pos[2].contiguous(), vx=v[0].contiguous(),
                vy=v[1].contiguous(), vz=v[2].contiguous(), mass=m, sml=h0 * one, e=e, rho=one.clone(),
                p=(2.0 / 3.0) * e, cs=torch.sqrt(10.0 / 9.0 * e))


def _blast(side: int, seed: int) -> dict:
    """The blast half-way through its run: the inner 0.3 swept outwards (the density rises towards the
    front and falls towards the centre), expanding and hot inside, at rest and cold outside, every h
    near the one its density needs (one per cent off, as after a time step)."""
    g = _gen(seed)
    pos = _lattice(side, 0.02, g)
    n = side ** 3
    h0 = ics.h_for_neighbours(float(n), N_NB)
    r = torch.sqrt((pos * pos).sum(0)).clamp(min=1e-9)
    rs, pw = 0.3, 0.6
    inside = r < rs
    t = (r / rs).clamp(max=1.0)
    pos = torch.where(inside, pos * (t ** (pw - 1.0)), pos)
    rho = torch.where(inside, t ** (3.0 - 3.0 * pw) / pw, torch.ones_like(r))
    v = torch.where(inside, pos * (0.8 / rs), torch.zeros_like(pos)) + 1e-3 * _randn(g, 3, n)
    e = torch.where(inside, 0.3 / (2.0 / 3.0 * rho), torch.full_like(r, 1e-4)) * (1.0 + 0.01 * _rand(g, n))
    sml = (h0 * rho ** (-1.0 / 3.0) * (1.0 + 0.01 * _randn(g, n))).clamp(max=4.0 * h0)
    p = (2.0 / 3.0) * rho * e
    m = torch.full((n,), 1.0 / n, device="cuda", dtype=torch.float64)
    return dict(x=pos[0].contiguous(), y=pos[1].contiguous(), z=pos[2].contiguous(), vx=v[0].contiguous(),
                vy=v[1].contiguous(), vz=v[2].contiguous(), mass=m, sml=sml, e=e, rho=rho, p=p,
                cs=torch.sqrt(5.0 / 3.0 * p / rho))


def _cloud(n: int, seed: int) -> dict:
    """A uniform unit sphere of unequal masses in solid rotation plus turbulent velocities."""
    g = _gen(seed)
    pos = _isotropic(g, n) * _rand(g, n) ** (1.0 / 3.0)
    phi = torch.atan2(pos[1], pos[0])
    w = 1.0 + 0.1 * torch.cos(2.0 * phi)
    v = torch.stack([-0.72 * pos[1], 0.72 * pos[0], torch.zeros_like(w)]) + 0.3 * _randn(g, 3, n)
    h0 = ics.h_for_neighbours(n / (4.0 / 3.0 * math.pi), N_NB)
    one = torch.ones_like(w)
    return dict(x=pos[0].contiguous(), y=pos[1].contiguous(), z=pos[2].contiguous(), vx=v[0].contiguous(),
                vy=v[1].contiguous(), vz=v[2].contiguous(), mass=w / w.sum(), sml=h0 * one, e=0.0 * one,
                rho=one.clone(), p=0.0 * one, cs=0.167 * one)


def _keys(n: int, seed: int) -> torch.Tensor:
    """21-level Lebesgue keys (63 bits) of a Plummer sphere in particle order."""
    s = _plummer(n, seed)
    key = torch.zeros(n, device="cuda", dtype=torch.int64)
    lo = min(float(s[a].min()) for a in "xyz")
    hi = max(float(s[a].max()) for a in "xyz")
    for axis, a in enumerate("xyz"):
        i = ((s[a] - lo) / (hi - lo) * 2097151.0).to(torch.int64).clamp(0, 2097151)
        for b in range(21):
            key |= ((i >> b) & 1) << (3 * b + axis)
    return key


class _Buffer:
    """A context's own array as torch sees foreign device memory; holds the context."""

    def __init__(self, ctx, field: str):
        self.ctx = ctx
        t = np.dtype(lib.FIELD_DTYPE[field])
        self.__cuda_array_interface__ = dict(shape=(ctx.n,), typestr=t.str, data=(ctx.field_ptr(field), False),
                                             strides=None, version=2)


def _view(ctx, field: str) -> torch.Tensor:
    return torch.as_tensor(_Buffer(ctx, field), device="cuda")


def _load(ctx, fields: dict) -> None:
    ctx.set_num_particles(len(fields["x"]))
    torch.cuda.synchronize()
    for k, v in fields.items():
        ctx.upload_device(k, v.data_ptr())
    ctx.synchronize()


def _params(c: dict) -> lib.Params:
    prec = lib.PREC_FP32_KAHAN if c.get("fp32") else lib.PREC_FP64
    if c["kind"] in ("gravity", "leapfrog"):
        return lib.default_params(theta=c["theta"], smoothing=c["eps2"], curve=c["curve"], mac=c["mac"],
                                  quadrupole=c["quad"], bh_accept=c["accept"], precision=prec)
    if c["kind"] in ("sph", "blast"):
        h0 = ics.h_for_neighbours(float(c["side"] ** 3), N_NB)
        return ics.params_sedov(sml_max=4.0 * h0, curve=c["curve"], smoothing_kernel=c["kernel"], precision=prec)
    p = ics.params_boss_bodenheimer()
    h0 = ics.h_for_neighbours(c["n"] / (4.0 / 3.0 * math.pi), N_NB)
    p.sml_max = 4.0 * h0
    if c["kind"] == "cloud":
        p.theta, p.curve, p.smoothing_kernel, p.precision = c["theta"], c["curve"], c["kernel"], prec
    return p


def _inputs(c: dict, seed: int) -> dict:
    k = c["kind"]
    if k == "sums":
        f = _plummer(c["n"], seed)
        g = _gen(seed + 1)
        for a in "xyz":   # off centre and moving, so that no sum cancels
            f[a] += 0.5 + 0.1 * float(_rand(g, 1))
            f["v" + a] += 0.7
        f["e"] = _rand(g, c["n"])
        f["u"] = -_rand(g, c["n"]) / c["n"]
        return f
    if k in ("gravity", "leapfrog"):
        return _plummer(c["n"], seed)
    if k == "sph":
        return _sedov(c["side"], seed)
    if k == "blast":
        return _blast(c["side"], seed)
    return _cloud(c["n"], seed)


def prepare(case: dict, seed: int) -> dict:
    c = dict(case)
    kind = c["kind"]
    if kind == "keys":
        k = _keys(c["n"], seed)
        s = dict(case=c, keys=k, out=torch.empty_like(k), perm=torch.empty(c["n"], device="cuda", dtype=torch.int32))
        torch.cuda.synchronize()
        return s
    if kind == "sums":
        ctx = lib.Context(c["n"])
        _load(ctx, _inputs(c, seed))
        return dict(case=c, ctx=ctx)
    f = _inputs(c, seed)
    ctx = lib.Context(len(f["x"]), _params(c))
    s = dict(case=c, ctx=ctx)
    if kind == "train":
        g = _gen(seed + 1)
        mean = [-2.0, 1.0, 0.0, 0.0, 0.0, 0.0, 0.01, 0.0]
        std = [0.1, 0.2, 0.3, 1.0, 1.0, 1.0, 0.01, 1.0]
        ctx.mlp_init(seed)
        ctx.mlp_set_norm(np.array(mean + std + [0.0, 0.05], np.float32))
        f["sml"] = f["sml"] * (1.0 + 0.1 * _randn(g, c["n"])).clamp(0.7, 1.3)
        _load(ctx, f)
        flags = lib.RHS_SPH | lib.RHS_VARIABLE_SML | lib.RHS_FEATURES | lib.RHS_SPECULATIVE_NN
        ctx.rhs(flags)
        _load(ctx, dict(x=f["x"], sml=f["sml"]))
        ctx.rhs(flags)   # features of a state whose derivatives are known
        return s
    _load(ctx, f)
    if kind == "leapfrog":
        ctx.rhs(lib.RHS_GRAVITY)
        s["out"] = {k: _view(ctx, k) for k in ("x", "y", "z", "vx", "vy", "vz", "g_ax", "g_ay", "g_az")}
    elif kind == "gravity":
        s["flags"] = lib.RHS_GRAVITY | (lib.RHS_POTENTIAL if c["potential"] else 0)
        s["out"] = {k: _view(ctx, k) for k in ("g_ax", "g_ay", "g_az") + (("u",) if c["potential"] else ())}
    else:
        s["flags"] = lib.RHS_SPH | lib.RHS_VARIABLE_SML | (lib.RHS_SPECULATIVE_NN if c["lists"] else 0)
        out = FLOAT_OUT + ("sml", "noi")
        if kind == "cloud":
            s["flags"] |= lib.RHS_GRAVITY
            out += ("g_ax", "g_ay", "g_az")
        if kind == "blast":
            out += ("x", "y", "z", "vx", "vy", "vz", "e")
        s["out"] = {k: _view(ctx, k) for k in out}
        # what a pass overwrites of its own inputs: set back before the next one
        keep = ("sml", "p", "cs") if kind != "blast" else ("x", "y", "z", "vx", "vy", "vz", "e", "sml", "p", "cs")
        s["keep"] = {k: f[k] for k in keep}
    return s


def _results(s: dict):
    """The fields as the program keeps them: FP32 pair sums are kept in FP32."""
    if not s["case"].get("fp32"):
        return s["out"]
    return {k: v if k in ("sml", "noi") else v.float() for k, v in s["out"].items()}


def run(state: dict):
    c = state["case"]
    kind = c["kind"]
    if kind == "keys":
        st = lib.LIB.mhpc_sort_keys_noalloc(state["keys"].data_ptr(), c["n"], state["out"].data_ptr(),
                                            state["perm"].data_ptr(),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if st != lib.OK:
            raise lib.MhpcError(st, "mhpc_sort_keys_noalloc")
        return {"keys": state["out"], "perm": state["perm"]}
    ctx = state["ctx"]
    if kind == "sums":
        return ctx.diagnostics()
    if kind == "train":
        loss = ctx.mlp_train(nsamples=c["samples"], iters=c["iters"], lr=1e-3, seed=7)
        return {"params": ctx.mlp_get_params(), "loss": np.float32(loss)}
    if kind == "leapfrog":
        ctx.leapfrog_update_x(c["dt"])
        ctx.rhs(lib.RHS_GRAVITY)
        ctx.leapfrog_update_v(c["dt"])
        return _results(state)
    if kind == "gravity":
        ctx.rhs(state["flags"])
        return _results(state)
    for k, v in state["keep"].items():
        ctx.upload_device(k, v.data_ptr())
    if kind == "blast":
        dt = ctx.pc_euler_step(state["flags"], courant_fact=0.3)[0]
        return {"dt": dt, **_results(state)}
    ctx.rhs(state["flags"])
    return _results(state)


# ---- what a pass cannot do without -----------------------------------------------------
def work(case: dict) -> dict:
    c = case
    kind = c["kind"]
    if kind == "keys":
        return {"bytes": 20.0 * c["n"], "flops": 0.0}
    if kind == "sums":
        return {"bytes": 72.0 * c["n"], "flops": 45.0 * c["n"]}
    if kind == "train":
        return {"bytes": c["iters"] * (40.0 * c["samples"] + 16.0 * lib.MLP_NPARAM),
                "flops": c["iters"] * c["samples"] * 3.0 * 2.0 * (64 * 8 + 64 * 64 + 64)}
    n = float(c.get("n") or c["side"] ** 3)
    nbytes, flops = 0.0, 0.0
    if kind in ("gravity", "leapfrog", "cloud"):
        # interactions per particle of a per-particle walk, about 28 log2(n) / theta^2 (all of them at most)
        inter = min(n, 28.0 * math.log2(n) / c["theta"] ** 2)
        nbytes += 32.0 * n + 24.0 * n + (8.0 * n if c.get("potential") else 0.0)
        flops += n * inter * (68.0 if c.get("quad") else 23.0)
        if kind == "leapfrog":
            nbytes += 13 * 8.0 * n
    if kind in ("sph", "blast", "cloud"):
        rhs = 2.0 if kind == "blast" else 1.0
        nbytes += rhs * (10 * 8.0 + 11 * 8.0) * n
        flops += rhs * n * N_NB * (8.0 + 25.0 + 70.0)
        if kind == "blast":
            nbytes += 30 * 8.0 * n
    return {"bytes": nbytes, "flops": flops}


# ---- the same in plain 64-bit torch ----------------------------------------------------
def _direct(x, m, eps2):
    """Accelerations and potentials of every particle by direct summation."""
    n = x.shape[1]
    acc, phi = torch.empty_like(x), torch.empty_like(m)
    step = max(1, min(n, (1 << 26) // n))
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [x[k][None, :] - x[k][a:b, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + eps2
        i = torch.arange(a, b, device="cuda")
        ri = torch.where(r2 > 0.0, 1.0 / torch.sqrt(r2), torch.zeros_like(r2))
        mr = m[None, :] * ri
        mr3 = mr * ri * ri
        for k in range(3):
            acc[k, a:b] = (mr3 * d[k]).sum(1)
        mr[torch.arange(b - a, device="cuda"), i] = 0.0
        phi[a:b] = -mr.sum(1)
    return acc, phi


def _pairs(x, h, rows):
    """Ordered pairs (i, j), i in rows, with d^2 < h_i^2 and d^2 < h_j^2."""
    n = x.shape[1]
    step = max(1, (1 << 26) // n)
    h2 = h * h
    ii, jj = [], []
    for a in range(0, len(rows), step):
        r = rows[a:a + step]
        d2 = torch.zeros(len(r), n, device="cuda", dtype=torch.float64)
        for k in range(3):
            t = x[k][r][:, None] - x[k][None, :]
            d2 += t * t
        hit = (d2 < h2[r][:, None]) & (d2 < h2[None, :])
        hit[torch.arange(len(r), device="cuda"), r] = False
        at = hit.nonzero()
        ii.append(r[at[:, 0]])
        jj.append(at[:, 1])
    return torch.cat(ii), torch.cat(jj)


def _sph_exact(f: dict, p: lib.Params) -> dict:
    n = len(f["x"])
    x = torch.stack([f["x"], f["y"], f["z"]])
    v = torch.stack([f["vx"], f["vy"], f["vz"]])
    m, h = f["mass"], f["sml"].clone()
    rows = torch.arange(n, device="cuda")
    for it in range(p.max_counts):
        i, _ = _pairs(x, h, rows)
        cnt = torch.bincount(i, minlength=n)[rows]
        done = ((cnt >= p.band_lo) & (cnt <= p.band_hi)) | (it == p.max_counts - 1)
        grow = 0.5 * (1.0 + (p.n_target / cnt.clamp(min=1).double()) ** (1.0 / 3.0))
        new = h[rows] * torch.where(done & (cnt < p.max_nb), torch.ones_like(grow), grow)
        if p.sml_max > 0.0:
            new = new.clamp(max=p.sml_max)
        h[rows] = new
        rows = rows[~done]
        if len(rows) == 0:
            break
    i, j = _pairs(x, h, torch.arange(n, device="cuda"))
    d = x[:, i] - x[:, j]
    r2 = (d * d).sum(0)
    r = torch.sqrt(r2)
    hb = 0.5 * (h[i] + h[j])
    q = r / hb
    f8 = 8.0 / math.pi / hb ** 3
    w = torch.where(q <= 0.5, f8 * (6 * q ** 3 - 6 * q ** 2 + 1), 2 * f8 * (1 - q).clamp(min=0.0) ** 3)
    dw = torch.where(q <= 0.5, 6 * f8 / hb * (3 * q * q - 2 * q), -6 * f8 / hb * (1 - q).clamp(min=0.0) ** 2)

    def add(t):
        return torch.zeros(n, device="cuda", dtype=torch.float64).index_add_(0, i, t)

    rho = m * (8.0 / math.pi) / h ** 3 + add(m[j] * w)
    if p.eos == lib.EOS_IDEAL_GAS:
        cs = torch.sqrt(p.gamma * f["p"] / rho)
        pr = (p.gamma - 1.0) * rho * f["e"]
    else:
        cs = torch.full_like(rho, p.cs_const)
        pr = cs * cs * rho
    g = dw / r * d
    dv = v[:, i] - v[:, j]
    vv, vr = (dv * g).sum(0), (dv * d).sum(0)
    mu = hb * vr / (r2 + 0.01 * hb * hb)
    visc = m[j] * (p.beta * mu - p.alpha * 0.5 * (cs[i] + cs[j])) * mu / (0.5 * (rho[i] + rho[j]))
    visc = torch.where(vr < 0.0, visc, torch.zeros_like(visc))
    pf = -m[j] * (pr[i] / rho[i] ** 2 + pr[j] / rho[j] ** 2)
    a = [add((pf - visc) * g[k]) for k in range(3)]
    dvv = add(m[j] / rho[j] * vv)
    return dict(ax=a[0], ay=a[1], az=a[2], rho=rho, p=pr, drhodt=rho * dvv, dedt=0.5 * add((visc - pf) * vv),
                dsmldt=-h / 3.0 * dvv, sml=h, noi=None)


def exact(case: dict, seed: int):
    c = case
    kind = c["kind"]
    n = c.get("n") or c["side"] ** 3
    if kind == "sums":
        f = {k: v.cpu().numpy().astype(np.longdouble) for k, v in _inputs(c, seed).items()}
        m = f["mass"]
        kin = 0.5 * (m * (f["vx"] ** 2 + f["vy"] ** 2 + f["vz"] ** 2)).sum()
        pot, inner = f["u"].sum(), (m * f["e"]).sum()
        mom = [(m * f["v" + a]).sum() for a in "xyz"]
        ang = [(m * (f[b] * f["v" + d] - f[d] * f["v" + b])).sum() for b, d in ("yz", "zx", "xy")]
        out = dict(kinetic=kin, potential=pot, internal=inner, total=kin + pot + inner, momentum=mom,
                   angular_momentum=ang, angular_momentum_norm=np.sqrt(sum(a * a for a in ang)), mass=m.sum(),
                   com=[(m * f[a]).sum() / m.sum() for a in "xyz"])
        return {k: [float(t) for t in v] if isinstance(v, list) else float(v) for k, v in out.items()}
    if kind in ("keys", "train", "blast") or n > 310000:
        return None
    f = _inputs(c, seed)
    p = _params(c)
    if kind in ("gravity", "leapfrog"):
        x = torch.stack([f["x"], f["y"], f["z"]])
        acc, phi = _direct(x, f["mass"], c["eps2"])
        if kind == "gravity":
            out = dict(g_ax=acc[0], g_ay=acc[1], g_az=acc[2])
            if c["potential"]:
                out["u"] = 0.5 * f["mass"] * phi
            return out
        dt = c["dt"]
        v = torch.stack([f["vx"], f["vy"], f["vz"]])
        x = x + dt * (v + 0.5 * dt * acc)
        acc1, _ = _direct(x, f["mass"], c["eps2"])
        v = v + 0.5 * dt * (acc + acc1)
        out = {}
        for k, a in enumerate("xyz"):
            out.update({a: x[k], "v" + a: v[k], "g_a" + a: acc1[k]})
        return out
    if c["kernel"] != 1 or n > 120000:
        return None
    out = _sph_exact(f, p)
    if kind == "cloud":
        acc, _ = _direct(torch.stack([f["x"], f["y"], f["z"]]), f["mass"], p.smoothing)
        out.update(g_ax=acc[0], g_ay=acc[1], g_az=acc[2])
    return out
