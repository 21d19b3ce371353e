"""The workloads that a user of this library runs, as measured cases.

A case is a dict of plain values.  `path` names the public entry point that it goes through, `dims`
the lattice (x, y, z, t) and the rest the options of the call:

  wilson     wilson_apply: the Wilson operator D, D^dagger, DD or DD^dagger on a full field
  schur      wilson_schur: the even-site Schur complement that even-odd solves iterate on
  ks         ks_apply: the staggered operator on a full field
  wforce     the Wilson fermion force of one molecular dynamics step (force cleared, then formed)
  ksforce    the staggered fermion force of one step over the poles of a rational approximation
  quenched   hmc_evolve with the plaquette action alone: gauge forces, momentum and link updates
  solve      solve: even-odd GMRES to a true residual, plain or in mixed precision
  multishift multishift_solve: all shifted systems of a rational approximation at once
  batch      solve_batch: the spin-colour point sources of a propagator plus uneven lattices
  hmc        hmc_evolve with the plaquette and the two-flavour Wilson action: one short trajectory

Gauge links, sources, momenta and solution vectors are drawn with torch on the GPU from the seed, put
into device fields through the upload entry point, and kept in the state together with the output
fields, as a user's program keeps them.  `exact` repeats a call on the same inputs with plain torch
operations in 64 bits.
"""
import math

import numpy as np
import torch

import cudalatticegauge_amd as clg

BC = (1, 1, 1, -1)  # antiperiodic in time, the fermion boundary of every configuration here
PREC = {"f64": clg.F64, "f32": clg.F32}
INNER = {"f64": (clg.F64, 0.0), "f32": (clg.F32, 1e-4), "f16": (clg.INNER_F16_VECTORS, 1e-2)}
OPS = {"D": clg.EFO_F_D, "Ddagger": clg.EFO_F_Ddagger, "DD": clg.EFO_F_DD, "DDdagger": clg.EFO_F_DDdagger}
KAPPA = 0.1355
MASS = 0.05
BETA = 5.5

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = clg.Context(0)
    return _context


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: one D on the lattice of the library's unit tests, where a launch's latency counts
        dict(name="d_8x8x8x8_f64", path="wilson", lx=8, ly=8, lz=8, lt=8, prec="f64", links=18, op="D"),
        # one D at the library's benchmark size
        dict(name="d_32x32x32x16_f64", path="wilson", lx=32, ly=32, lz=32, lt=16, prec="f64", links=18, op="D"),
        # the inner operator of mixed even-odd solves on a production shape whose planes are no power of two
        dict(name="schur_24x24x24x48_f32", path="schur", lx=24, ly=24, lz=24, lt=48, prec="f32", links=18, op="D"),
        # staggered D D^dagger on odd, ragged extents
        dict(name="ks_21x19x25x18_f64", path="ks", lx=21, ly=19, lz=25, lt=18, prec="f64", links=18, op="DDdagger"),
        # the fermion forces at the sizes of the Wilson and the staggered trajectories
        dict(name="wforce_32x32x32x16", path="wforce", lx=32, ly=32, lz=32, lt=16),
        dict(name="ksforce_24x24x24x8", path="ksforce", lx=24, ly=24, lz=24, lt=8, poles=12),
        # a pure gauge trajectory: what the inner steps of every nested integrator consist of
        dict(name="quenched_16x16x16x32", path="quenched", lx=16, ly=16, lz=16, lt=32, steps=8, exp=8),
        # a solve on a small lattice: many short launches and host reads
        dict(name="solve_8x8x8x8_f64", path="solve", lx=8, ly=8, lz=8, lt=8, inner="f64", op="D"),
        # the largest: a quark propagator component at 32^4 in mixed precision
        dict(name="solve_32x32x32x32_f16", path="solve", lx=32, ly=32, lz=32, lt=32, inner="f16", op="D"),
        # the shifted solves of a staggered trajectory's force in single precision
        dict(name="multishift_24x24x24x8_f32", path="multishift", lx=24, ly=24, lz=24, lt=8, prec="f32", shifts=12),
        # a full propagator (12 point sources) with three more uneven lattices in one batch
        dict(name="batch_16x16x16x32_f16", path="batch", lx=16, ly=16, lz=16, lt=32, sources=12,
             others="8x8x8x8,12x12x12x12,10x14x6x12", inner="f16"),
        # a whole call: a short two-flavour Wilson trajectory (nested force gradient) in mixed precision
        dict(name="hmc_16x16x16x16_f32", path="hmc", lx=16, ly=16, lz=16, lt=16, steps=2, nested=3, inner="f32"),
    ]


def _extent(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(rng, lo, hi):
    return 2 * _extent(rng, lo / 2, hi / 2)


def draw(rng):
    path = rng.choice(["wilson", "schur", "ks", "wforce", "ksforce", "quenched", "solve", "multishift", "batch", "hmc"])
    c = dict(path=path)
    if path in ("wilson", "ks"):
        c.update(lx=_extent(rng, 6, 32), ly=_extent(rng, 6, 32), lz=_extent(rng, 6, 32), lt=_even(rng, 6, 32),
                 prec=rng.choice(["f64", "f32"]), links=rng.choice([18, 12]),
                 op=rng.choice(["D", "Ddagger", "DD", "DDdagger"]))
    elif path == "schur":
        c.update(lx=_even(rng, 6, 32), ly=_even(rng, 6, 32), lz=_even(rng, 6, 32), lt=_even(rng, 6, 48),
                 prec=rng.choice(["f64", "f32"]), links=rng.choice([18, 12]), op=rng.choice(["D", "Ddagger"]))
    elif path == "wforce":
        c.update(lx=_extent(rng, 6, 32), ly=_extent(rng, 6, 32), lz=_extent(rng, 6, 32), lt=_even(rng, 6, 32))
    elif path == "ksforce":
        c.update(lx=_extent(rng, 6, 28), ly=_extent(rng, 6, 28), lz=_extent(rng, 6, 28), lt=_even(rng, 6, 28),
                 poles=rng.randint(1, 16))
    elif path == "quenched":
        c.update(lx=_extent(rng, 4, 24), ly=_extent(rng, 4, 24), lz=_extent(rng, 4, 24), lt=_even(rng, 4, 24),
                 steps=rng.randint(4, 10), exp=rng.choice([0, 8]))
    elif path == "solve":
        c.update(lx=_even(rng, 6, 28), ly=_even(rng, 6, 28), lz=_even(rng, 6, 28), lt=_even(rng, 6, 28),
                 inner=rng.choice(["f64", "f32", "f16"]), op=rng.choice(["D", "Ddagger", "DDdagger"]))
    elif path == "multishift":
        c.update(lx=_even(rng, 6, 20), ly=_even(rng, 6, 20), lz=_even(rng, 6, 20), lt=_even(rng, 6, 16),
                 prec=rng.choice(["f64", "f32"]), shifts=rng.randint(4, 14))
    elif path == "batch":
        c.update(lx=_even(rng, 6, 16), ly=_even(rng, 6, 16), lz=_even(rng, 6, 16), lt=_even(rng, 6, 24),
                 sources=rng.randint(1, 12), inner=rng.choice(["f32", "f16"]),
                 others=",".join("x".join(str(_even(rng, 4, 12)) for _ in range(4)) for _ in range(rng.randint(0, 3))))
    else:
        c.update(lx=_even(rng, 6, 16), ly=_even(rng, 6, 16), lz=_even(rng, 6, 16), lt=_even(rng, 6, 16),
                 steps=rng.randint(1, 2), nested=rng.randint(1, 3), inner=rng.choice(["f64", "f32", "f16"]))
    return c


def _dims(case):
    return (case["lx"], case["ly"], case["lz"], case["lt"])


def _lattices(case):
    """Lattice, source kind (spin-colour index of a point source, or -1 for a Gaussian one) of each system."""
    out = [(_dims(case), k) for k in range(case["sources"])]
    for text in case["others"].split(","):
        if text:
            out.append((tuple(int(v) for v in text.split("x")), -1))
    return out


def _shifts(case):
    return np.logspace(-4, 1, case["shifts"])


# ------------------------------------------------------------------ inputs (torch, 64 bits, from the seed alone)
def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _mm(a, b):
    """Products of 3x3 matrices in the last two dimensions, column by column."""
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(3))


def _dag(a):
    return a.mH


def _normal(g, shape):
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, device="cuda", dtype=torch.float64))


def _links(dims, seed, eps, stream=0):
    """exp(i eps H), H traceless Hermitian with unit Gaussian entries: [x, y, z, t, mu, 3, 3]."""
    h = _normal(_gen(seed, stream), (*dims, 4, 3, 3))
    h = (h + _dag(h)) / 2
    h = h - torch.diag_embed(h.diagonal(dim1=-2, dim2=-1).sum(-1, keepdim=True).expand(*dims, 4, 3) / 3)
    a, eye = 0.25j * eps * h, torch.eye(3, device="cuda", dtype=torch.complex128)
    u = eye.expand_as(a)
    for k in range(14, 0, -1):
        u = eye + _mm(a, u) / k
    for _ in range(2):
        u = _mm(u, u)
    return _reunit(u)


def _reunit(u):
    """Gram-Schmidt on rows 0 and 1, row 2 = conj(r0 x r1)."""
    r0 = u[..., 0, :] / torch.linalg.vector_norm(u[..., 0, :], dim=-1, keepdim=True)
    r1 = u[..., 1, :] - (r0.conj() * u[..., 1, :]).sum(-1, keepdim=True) * r0
    r1 = r1 / torch.linalg.vector_norm(r1, dim=-1, keepdim=True)
    return torch.stack([r0, r1, torch.linalg.cross(r0, r1).conj()], dim=-2)


def _momenta(dims, seed):
    """Traceless anti-Hermitian, Gaussian generator weights of variance 1/4 (the heat bath's)."""
    h = _normal(_gen(seed, 1), (*dims, 4, 3, 3)) * math.sqrt(0.125)
    return _ta(1j * (h + _dag(h)))


def _spinor(dims, seed, stream, kind="wilson"):
    """Gaussian, E|psi_i|^2 = 1: [x, y, z, t, 4, 3] or, for staggered fields, [x, y, z, t, 3]."""
    return _normal(_gen(seed, stream), (*dims, 4, 3) if kind == "wilson" else (*dims, 3)) / math.sqrt(2)


def _source(dims, k, seed, stream):
    if k < 0:
        return _spinor(dims, seed, stream)
    b = torch.zeros(*dims, 4, 3, device="cuda", dtype=torch.complex128)
    b[0, 0, 0, 0, k // 3, k % 3] = 1
    return b


def _host(t):
    return torch.view_as_real(t.contiguous()).cpu().numpy().ravel()


def _put(kind, prec, dims, values=None, subset=clg.FULL):
    f = clg.Field(_ctx(), kind, prec, dims, subset=subset, bc=None if kind in (clg.GAUGE, clg.GAUGE12) else BC)
    if values is not None:
        f.upload(_host(values))
    return f


def _even_sites(dims):
    """Flat index of the e-th even site (whichever of the lexicographic sites 2e, 2e+1 is even)."""
    x, y, z, t = (torch.arange(n, device="cuda") for n in dims)
    odd = (x[:, None, None, None] + y[None, :, None, None] + z[None, None, :, None] + t) % 2
    odd = odd.reshape(-1, 2)
    return torch.arange(odd.shape[0], device="cuda") * 2 + odd[:, 0]


def _inputs(case, seed):
    """The call's inputs as torch tensors."""
    path, dims = case["path"], _dims(case)
    if path == "wilson":
        return _links(dims, seed, 0.5), _spinor(dims, seed, 2)
    if path == "schur":
        psi = _spinor(dims, seed, 2).reshape(-1, 4, 3)
        return _links(dims, seed, 0.5), psi[_even_sites(dims)]
    if path in ("ks", "multishift"):
        return _links(dims, seed, 0.4), _spinor(dims, seed, 2, "ks")
    if path == "wforce":
        return _links(dims, seed, 0.5), _spinor(dims, seed, 2), _spinor(dims, seed, 3)
    if path == "ksforce":
        phis = [_spinor(dims, seed, 2 + 2 * k, "ks") for k in range(case["poles"])]
        ds = [_spinor(dims, seed, 3 + 2 * k, "ks") for k in range(case["poles"])]
        return _links(dims, seed, 0.4), phis, ds, np.linspace(0.1, 1.0, case["poles"])
    if path == "quenched":
        return _links(dims, seed, 0.4), _momenta(dims, seed)
    if path == "solve":
        return _links(dims, seed, 0.5), _spinor(dims, seed, 2)
    if path == "batch":
        systems, links = _lattices(case), {}
        for i, (d, _) in enumerate(systems):
            if d not in links:
                links[d] = _links(d, seed, 0.5, 32 + len(links))
        return links, [_source(d, k, seed, 2 + i) for i, (d, k) in enumerate(systems)]
    return _links(dims, seed, 0.5), _momenta(dims, seed), _spinor(dims, seed, 2)


def prepare(case, seed):
    path, dims, ctx = case["path"], _dims(case), _ctx()
    s = dict(case=case, ctx=ctx)
    given = _inputs(case, seed)
    if path in ("wilson", "ks"):
        kind, prec = (clg.WILSON if path == "wilson" else clg.KS), PREC[case["prec"]]
        s["gauge"] = _put(clg.GAUGE if case["links"] == 18 else clg.GAUGE12, prec, dims, given[0])
        s["in"], s["out"] = _put(kind, prec, dims, given[1]), _put(kind, prec, dims)
    elif path == "schur":
        prec = PREC[case["prec"]]
        s["gauge"] = _put(clg.GAUGE if case["links"] == 18 else clg.GAUGE12, prec, dims, given[0])
        s["in"] = _put(clg.WILSON, prec, dims, given[1], clg.EVEN)
        s["out"] = _put(clg.WILSON, prec, dims, subset=clg.EVEN)
    elif path == "wforce":
        s["gauge"], s["force"] = _put(clg.GAUGE, clg.F64, dims, given[0]), _put(clg.GAUGE, clg.F64, dims)
        s["x"], s["y"] = (_put(clg.WILSON, clg.F64, dims, v) for v in given[1:])
    elif path == "ksforce":
        s["gauge"], s["force"] = _put(clg.GAUGE, clg.F64, dims, given[0]), _put(clg.GAUGE, clg.F64, dims)
        s["phi"], s["d"] = ([_put(clg.KS, clg.F64, dims, v) for v in vs] for vs in given[1:3])
        s["a"] = given[3]
    elif path in ("quenched", "hmc"):
        s["u0"], s["p0"] = (_put(clg.GAUGE, clg.F64, dims, v) for v in given[:2])
        s["u"], s["p"] = (_put(clg.GAUGE, clg.F64, dims) for _ in range(2))
        s["actions"] = [dict(kind=clg.ACTION_GAUGE_PLAQUETTE, beta=BETA)]
        if path == "quenched":
            s["params"] = clg.hmc_params(integrator=clg.INT_LEAPFROG, step_length=0.4, steps=case["steps"],
                                         exp_precision=case["exp"], metropolis=0)
        else:
            s["phi"] = _put(clg.WILSON, clg.F64, dims, given[2])
            s["actions"].append(dict(kind=clg.ACTION_FERMION_WILSON_NF2, kappa_or_mass=KAPPA, phi=s["phi"],
                                     solver=_solver(case["inner"], 1e-8), energy_accuracy=1e-10))
            s["params"] = clg.hmc_params(integrator=clg.INT_NESTED_FORCE_GRADIENT, step_length=0.25,
                                         steps=case["steps"], nested_steps=case["nested"], exp_precision=8,
                                         metropolis=0)
    elif path == "solve":
        s["gauge"], s["b"] = _put(clg.GAUGE, clg.F64, dims, given[0]), _put(clg.WILSON, clg.F64, dims, given[1])
        s["x"] = _put(clg.WILSON, clg.F64, dims)
        s["params"] = _solver(case["inner"], 1e-10)
    elif path == "multishift":
        s["gauge"], s["b"] = _put(clg.GAUGE, clg.F64, dims, given[0]), _put(clg.KS, clg.F64, dims, given[1])
        s["xs"] = [_put(clg.KS, clg.F64, dims) for _ in range(case["shifts"])]
        s["params"] = clg.solver_params(kind=clg.KS, max_dim=40, restart=200, absolute_accuracy=1,
                                        accuracy=1e-8 if case["prec"] == "f64" else 1e-5)
    else:
        gauges = {d: _put(clg.GAUGE, clg.F64, d, u) for d, u in given[0].items()}
        dd = [d for d, _ in _lattices(case)]
        s["gauges"] = [gauges[d] for d in dd]
        s["bs"] = [_put(clg.WILSON, clg.F64, d, b) for d, b in zip(dd, given[1])]
        s["xs"] = [_put(clg.WILSON, clg.F64, d) for d in dd]
        s["params"] = _solver(case["inner"], 1e-10)
    ctx.sync()
    return s


def _solver(inner, accuracy):
    prec, inner_accuracy = INNER[inner]
    return clg.solver_params(max_dim=12, restart=500, accuracy=accuracy, stop_rule=clg.STOP_TRUE_RESIDUAL, even_odd=1,
                             inner_prec=prec, inner_accuracy=inner_accuracy, max_outer=60)


# ------------------------------------------------------------------ one pass
class Outputs(dict):
    """The outputs of a call by name.  Device fields stay on the device: whoever looks one up gets its whole
    contents through the library's download, in the host order, at that moment."""

    def __getitem__(self, name):
        v = dict.__getitem__(self, name)
        return v.download() if isinstance(v, clg.Field) else v


def run(s):
    case, ctx = s["case"], s["ctx"]
    path = case["path"]
    if path == "wilson":
        clg.wilson_apply(ctx, s["out"], s["in"], s["gauge"], KAPPA, OPS[case["op"]])
        return Outputs(out=s["out"])
    if path == "schur":
        clg.wilson_schur(ctx, s["out"], s["in"], s["gauge"], KAPPA, OPS[case["op"]])
        return Outputs(out=s["out"])
    if path == "ks":
        clg.ks_apply(ctx, s["out"], s["in"], s["gauge"], MASS, OPS[case["op"]])
        return Outputs(out=s["out"])
    if path == "wforce":
        s["force"].zero()
        clg.wilson_force_kernel(ctx, s["force"], s["gauge"], s["x"], s["y"], KAPPA)
        return Outputs(force=s["force"])
    if path == "ksforce":
        s["force"].zero()
        clg.ks_force_kernel(ctx, s["force"], s["gauge"], s["phi"], s["d"], s["a"])
        return Outputs(force=s["force"])
    if path in ("quenched", "hmc"):
        s["u"].copy_from(s["u0"])
        s["p"].copy_from(s["p0"])
        rep = clg.hmc_evolve(ctx, s["u"], s["p"], s["params"], s["actions"])
        return Outputs(u=s["u"], p=s["p"], h_before=rep.h_before, h_after=rep.h_after)
    if path == "solve":
        clg.solve(ctx, s["params"], s["x"], s["b"], s["gauge"], KAPPA, clg.EFO_F_InverseD + OPS[case["op"]])
        return Outputs(x=s["x"])
    if path == "multishift":
        clg.multishift_solve(ctx, s["params"], s["xs"], _shifts(case), s["b"], s["gauge"], MASS, clg.EFO_F_DDdagger,
                             kind=clg.MS_BICGSTAB, prec=PREC[case["prec"]])
        return Outputs({"x%02d" % k: x for k, x in enumerate(s["xs"])})
    clg.solve_batch(ctx, s["params"], s["xs"], s["bs"], s["gauges"], KAPPA, clg.EFO_F_InverseD)
    return Outputs({"x%02d" % k: x for k, x in enumerate(s["xs"])})


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Every input read once and every output written once; the flops of one operator application (solves and
    trajectories: of the least that touches every input, since how many they take is the algorithm's affair)."""
    path, v = case["path"], math.prod(_dims(case))
    r = 4 if case.get("prec") == "f32" else 8
    if path in ("wilson", "ks"):
        n, fl = (24, 1368) if path == "wilson" else (6, 582)
        return dict(bytes=(2 * n + 4 * case["links"]) * r * v, flops=fl * v * (2 if case["op"].startswith("DD") else 1))
    if path == "schur":
        return dict(bytes=(24 + 4 * case["links"]) * r * v, flops=(2 * 1320 + 48) * v / 2)
    if path == "wforce":
        return dict(bytes=(48 + 72 + 72) * r * v, flops=4 * 1000 * v)
    if path == "ksforce":
        return dict(bytes=(12 * case["poles"] + 144) * r * v, flops=400 * case["poles"] * v)
    if path in ("quenched", "hmc"):
        # each step's force reads the links; momenta and links are read and written once
        return dict(bytes=(4 * 72 + (24 if path == "hmc" else 0)) * r * v, flops=4 * 2900 * v * case["steps"])
    if path == "solve":
        return dict(bytes=(72 + 48) * 8 * v, flops=1368 * v)
    if path == "multishift":
        return dict(bytes=(72 + 6 + 6 * case["shifts"]) * 8 * v, flops=2 * 582 * v)
    systems = _lattices(case)
    links = sum(72 * math.prod(d) for d in {d for d, _ in systems})
    return dict(bytes=8 * (links + sum(48 * math.prod(d) for d, _ in systems)),
                flops=sum(1368 * math.prod(d) for d, _ in systems))


def tolerance(case):
    path = case["path"]
    if path in ("wilson", "schur", "ks"):
        return {"rel": 4e-7} if case["prec"] == "f32" else {"rel": 1e-15}
    if path in ("wforce", "ksforce"):
        return {"rel": 2e-15}
    if path == "quenched":
        return {"rel": 1e-13}
    if path in ("solve", "batch"):
        return {"rel": 1e-9}  # the stop rule's 1e-10 times the condition of D
    if path == "multishift":
        return {"rel": 4e-6} if case["prec"] == "f32" else {"rel": 1e-9}
    return {"rel": 1e-7}  # force solves to a residual of 1e-8


# ------------------------------------------------------------------ the same in plain torch, 64 bits
# gamma_mu of the chiral representation: (gamma_mu psi)[r] = phase[r] psi[index[r]]
GAMMA = [([3, 2, 1, 0], [-1j, -1j, 1j, 1j]), ([3, 2, 1, 0], [-1, 1, 1, -1]), ([2, 3, 0, 1], [-1j, 1j, 1j, -1j]),
         ([2, 3, 0, 1], [1, 1, 1, 1])]


def _gamma(mu, psi):
    idx, ph = GAMMA[mu]
    return psi[..., idx, :] * torch.tensor(ph, device=psi.device, dtype=psi.dtype)[:, None]


def _ahead(f, mu, bc=1):
    """f(x + mu), times the boundary sign where it wraps."""
    g = torch.roll(f, -1, mu)
    if bc != 1:
        g.select(mu, g.shape[mu] - 1).mul_(bc)
    return g


def _behind(f, mu, bc=1):
    g = torch.roll(f, 1, mu)
    if bc != 1:
        g.select(mu, 0).mul_(bc)
    return g


def _mv(u, v):
    """u v on the colour index (the last one) of v."""
    if v.dim() == u.dim():  # a spin index before the colour
        u = u[..., None, :, :]
    return sum(u[..., :, k] * v[..., k, None] for k in range(3))


def _wilson_hop(u, psi, sign):
    out = torch.zeros_like(psi)
    for mu in range(4):
        um = u[..., mu, :, :]
        f = _ahead(psi, mu, BC[mu])
        out += _mv(um, f - sign * _gamma(mu, f))
        b = psi + sign * _gamma(mu, psi)
        out += _behind(_mv(_dag(um), b), mu, BC[mu])
    return out


def _wilson(u, psi, op):
    if op in ("DD", "DDdagger"):
        return _wilson(u, _wilson(u, psi, "Ddagger" if op == "DDdagger" else "D"), "D")
    return psi - KAPPA * _wilson_hop(u, psi, 1 if op == "D" else -1)


def _eta(dims, mu):
    """(-1)^(x_0 + ... + x_{mu-1}), one value a site and a colour index to broadcast over."""
    e = torch.ones(*dims, 1, device="cuda", dtype=torch.float64)
    for nu in range(mu):
        shape = [1] * 5
        shape[nu] = dims[nu]
        e = e * (1 - 2 * (torch.arange(dims[nu], device="cuda") % 2)).reshape(shape)
    return e


def _ks_hop(u, psi):
    out = torch.zeros_like(psi)
    for mu in range(4):
        um = u[..., mu, :, :]
        out += _eta(psi.shape[:4], mu) * (_mv(um, _ahead(psi, mu, BC[mu])) - _behind(_mv(_dag(um), psi), mu, BC[mu]))
    return out


def _ks(u, psi, op):
    if op in ("DD", "DDdagger"):
        return _ks(u, _ks(u, psi, "Ddagger" if op == "DDdagger" else "D"), "D")
    return MASS * psi + (1 if op == "D" else -1) * _ks_hop(u, psi)


def _ta(m):
    m = (m - _dag(m)) / 2
    return m - torch.diag_embed(m.diagonal(dim1=-2, dim2=-1).sum(-1, keepdim=True).expand(*m.shape[:-1]) / 3)


def _outer(a, b):
    """a b^dagger over colour, summed over spin where there is one."""
    m = a[..., :, None] * b[..., None, :].conj()
    return m.sum(-3) if a.dim() == 6 else m


def _wilson_force(u, x, y):
    out = torch.empty_like(u)
    for mu in range(4):
        # the wrap sign stands once in each product, through the forward neighbour
        yf, xf = _ahead(y, mu, BC[mu]), _ahead(x, mu, BC[mu])
        mid = _outer(yf - _gamma(mu, yf), x) + _outer(xf, y + _gamma(mu, y))
        out[..., mu, :, :] = KAPPA * _ta(_mm(u[..., mu, :, :], mid))
    return out


def _ks_force(u, phis, ds, a):
    out = torch.zeros_like(u)
    for mu in range(4):
        um, eta = u[..., mu, :, :], _eta(u.shape[:4], mu)
        for phi, d, w in zip(phis, ds, a):
            t = _outer(_mv(um, _ahead(phi, mu, BC[mu])), d) + _outer(phi, _mv(um, _ahead(d, mu, BC[mu])))
            out[..., mu, :, :] -= _ta(w * eta[..., None] * t)
    return out


def _gauge_force(u):
    out = torch.empty_like(u)
    for mu in range(4):
        um, c = u[..., mu, :, :], 0
        for nu in range(4):
            if nu == mu:
                continue
            un = u[..., nu, :, :]
            c = c + _mm(_mm(_ahead(un, mu), _dag(_ahead(um, nu))), _dag(un))
            c = c + _behind(_mm(_dag(_mm(um, _ahead(un, mu))), un), nu)
        out[..., mu, :, :] = -BETA / 6 * _ta(_mm(um, c))
    return out


def _plaquette_energy(u):
    e = 0.0
    for mu in range(4):
        for nu in range(mu + 1, 4):
            um, un = u[..., mu, :, :], u[..., nu, :, :]
            p = _mm(um, _ahead(un, mu)) * _mm(un, _ahead(um, nu)).conj()
            e += 3 * p[..., 0, 0].numel() - float(p.real.sum())
    return BETA / 3 * e


def _cayley(i, j, y, z, m):
    """m with rows i, j multiplied by (1 + X)(1 - X)^-1, X = [[i y, z], [-z*, -i y]]."""
    n = y * y + z.abs() ** 2
    c, o = torch.complex((1 - n) / (1 + n), 2 * y / (1 + n))[..., None], (2 * z / (1 + n))[..., None]
    m = m.clone()
    a, b = m[..., i, :].clone(), m[..., j, :].clone()
    m[..., i, :] = c * a + o * b
    m[..., j, :] = -o.conj() * a + c.conj() * b
    return m


def _expm(p, a, order):
    eye = torch.eye(3, device="cuda", dtype=torch.complex128).expand_as(p)
    if order == 0:  # the symmetric product of five SU(2) Cayley maps
        d = p.diagonal(dim1=-2, dim2=-1).imag
        y1, y2, y3 = a * (d[..., 0] - d[..., 1]) / 12, a * (d[..., 0] - d[..., 2]) / 12, a * (d[..., 1] - d[..., 2]) / 6
        z1, z2, z3 = a / 4 * p[..., 0, 1], a / 4 * p[..., 0, 2], a / 2 * p[..., 1, 2]
        m = _cayley(0, 1, y1, z1, eye)
        m = _cayley(1, 2, y3, z3, _cayley(0, 2, y2, z2, m))
        return _cayley(0, 1, y1, z1, _cayley(0, 2, y2, z2, m))
    m = eye
    for k in range(order, 0, -1):
        m = eye + a / k * _mm(p, m)
    return m


def _bicgstab(apply, b, tol=1e-14, most=2000):
    x, r = torch.zeros_like(b), b.clone()
    rh, p = r.clone(), r.clone()
    rho, bn = torch.sum(rh.conj() * r), float(torch.linalg.vector_norm(b))
    for _ in range(most):
        v = apply(p)
        alpha = rho / torch.sum(rh.conj() * v)
        s = r - alpha * v
        t = apply(s)
        omega = torch.sum(t.conj() * s) / torch.sum(t.conj() * t)
        x = x + alpha * p + omega * s
        r = s - omega * t
        if float(torch.linalg.vector_norm(r)) < tol * bn:
            break
        new = torch.sum(rh.conj() * r)
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
    return x


def _shifted_cg(apply, b, shifts, tol=1e-13, most=8000):
    """(A + c_k)^-1 b for all c_k >= c_0, A Hermitian positive definite: conjugate gradients on A + c_0."""
    base = float(shifts[0])
    n = len(shifts)
    x, p = [torch.zeros_like(b) for _ in range(n)], [b.clone() for _ in range(n)]
    zo, z, r = [1.0] * n, [1.0] * n, b.clone()
    rr, ao, beta = float(torch.sum(r.abs() ** 2)), 1.0, 0.0
    stop = tol * math.sqrt(rr)
    live = list(range(n))
    for _ in range(most):
        q = apply(p[0]) + base * p[0]
        a = rr / float(torch.sum(p[0].conj() * q).real)
        r = r - a * q
        new = float(torch.sum(r.abs() ** 2))
        keep = []
        for k in live:
            s = float(shifts[k]) - base
            zn = z[k] * zo[k] * ao / (a * beta * (zo[k] - z[k]) + zo[k] * ao * (1 + s * a))
            ak = a * zn / z[k]
            x[k] = x[k] + ak * p[k]
            bk = new / rr * (zn / z[k]) ** 2
            p[k] = zn * r + bk * p[k]
            zo[k], z[k] = z[k], zn
            if k == 0 or abs(zn) * math.sqrt(new) > stop:
                keep.append(k)
        live, beta, ao, rr = keep, new / rr, a, new
        if math.sqrt(rr) < stop:
            break
    return x


def _real(t):
    return torch.view_as_real(t.contiguous()).reshape(-1)


def exact(case, seed):
    path, dims = case["path"], _dims(case)
    if path == "hmc":
        return None
    given = _inputs(case, seed)
    if path == "wilson":
        return dict(out=_real(_wilson(given[0], given[1], case["op"])))
    if path == "schur":
        at, sign = _even_sites(dims), 1 if case["op"] == "D" else -1
        full = torch.zeros(math.prod(dims), 4, 3, device="cuda", dtype=torch.complex128)
        full[at] = given[1]
        hop = _wilson_hop(given[0], _wilson_hop(given[0], full.reshape(*dims, 4, 3), sign), sign).reshape(-1, 4, 3)
        return dict(out=_real(given[1] - KAPPA * KAPPA * hop[at]))
    if path == "ks":
        return dict(out=_real(_ks(given[0], given[1], case["op"])))
    if path == "wforce":
        return dict(force=_real(_wilson_force(*given)))
    if path == "ksforce":
        return dict(force=_real(_ks_force(*given)))
    if path == "quenched":
        u, p = given
        eps = 0.4 / case["steps"]
        before = float((p.abs() ** 2).sum()) + _plaquette_energy(u)
        for k in range(case["steps"]):  # half a step of momenta, links and forces in turn, half a step at the end
            p = p + (eps / 2 if k == 0 else eps) * _gauge_force(u)
            u = _mm(_expm(p, eps, case["exp"]), u)
        p, u = p + eps / 2 * _gauge_force(u), _reunit(u)
        after = float((p.abs() ** 2).sum()) + _plaquette_energy(u)
        return dict(u=_real(u), p=_real(p), h_before=before, h_after=after)
    if path == "solve":
        u, x = given
        for op in ("D", "Ddagger") if case["op"] == "DDdagger" else (case["op"],):
            x = _bicgstab(lambda v, op=op: _wilson(u, v, op), x)
        return dict(x=_real(x))
    if path == "multishift":
        xs = _shifted_cg(lambda v: _ks(given[0], v, "DDdagger"), given[1], _shifts(case))
        return {"x%02d" % k: _real(x) for k, x in enumerate(xs)}
    out = {}
    for k, ((d, _), b) in enumerate(zip(_lattices(case), given[1])):
        out["x%02d" % k] = _real(_bicgstab(lambda v, u=given[0][d]: _wilson(u, v, "D"), b))
    return out
