"""The engine's timed workloads: what a program that uses it has it do, through
the C ABI and its Python binding.

Kinds of case (sizes are those of bench.py, mgmol_amd/measure.py, the tests,
or of the same ranges):

  solve      mgx_solver_run: steps of the orbital iteration on a box set from
             its initial orbitals (Anderson, zero-start V-cycle, graph replay),
             with the plain FP64 path, the mixed path (FP32 V-cycle, hi/lo-split
             S/H) or the Mehrstellen discretisation
  cnn_apply  mgx_cnn_apply: the learned preconditioner over a box set
  cnn_grad   mgx_cnn_grad: forward and backward pass of one training batch
  hloc       mgx_hloc_apply: H psi of full-grid orbitals
  precond    mgx_precond_mg: the V-cycle preconditioner of full-grid orbitals
  hartree    mgx_poisson_mg: the Hartree potential by multigrid V-cycles
  gram       mgx_local_gram + mgx_local_product: S and H of full-grid orbitals
  density    mgx_box_density: the electron density of a box set
"""
import ctypes as C
import itertools
import math

import numpy as np
import torch
import torch.nn.functional as F

from mgmol_amd import learned, mgx

FP64 = torch.float64
_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(mgx.Ctx(0))
    return _CTX[0]


def _dev():
    return torch.device("cuda", 0)


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a small molecule: few small boxes of several edges, every launch a few microseconds
        dict(name="solve_small", kind="solve", nbox=24, gdim=40, edges="8,12,16", path="mixed", steps=12),
        # orbitals with uneven localisation regions (512 boxes, edges 24-40, 192^3), all FP64
        dict(name="solve_uneven", kind="solve", nbox=512, gdim=192, edges="24,28,32,36,40", path="plain", steps=16),
        # the flagship: 2048 orbitals in 32^3 boxes on 256^3, the mixed path
        dict(name="solve_large", kind="solve", nbox=2048, gdim=256, edges="32", path="mixed", steps=24),
        # the reference's default discretisation (FDtype = Mehrstellen)
        dict(name="solve_mehr", kind="solve", nbox=128, gdim=96, edges="20,24", path="mehr", steps=6),
        # one application of the network to every box of the flagship set
        dict(name="cnn_apply", kind="cnn_apply", nbox=2048, edge=32),
        # one batch of the network's training
        dict(name="cnn_grad", kind="cnn_grad", nbox=64, edge=32),
        # delocalised orbitals through the drop-in entry points: 64 on 96^3
        dict(name="hloc_grid", kind="hloc", n=64, d0=96, d1=96, d2=96, lap=2, dtype="f64"),
        dict(name="precond_grid", kind="precond", n=64, d0=96, d1=96, d2=96, lap=2, dtype="f64", levels=2),
        # a few orbitals on a small uneven grid, the reference's FP32 preconditioner and default operator
        dict(name="precond_small", kind="precond", n=6, d0=48, d1=40, d2=36, lap=0, dtype="f32", levels=2),
        # the Hartree potential on the flagship's grid
        dict(name="hartree", kind="hartree", d0=256, d1=256, d2=256, lap=0, bc=1),
        # S and H of the 64 orbitals on 96^3
        dict(name="gram_grid", kind="gram", n=64, rows=884736, prec="f64"),
        # the electron density of the flagship set
        dict(name="density", kind="density", nbox=2048, gdim=256, edges="32"),
    ]


def _logint(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _boxes_for(rng, lo, hi, edge_sets, ratio, gstep):
    """nbox, edges and a grid edge such that the boxes cover each point `ratio`
    times on average, within the geometry a box set accepts."""
    edges = rng.choice(edge_sets)
    ev = [int(e) for e in edges.split(",")]
    vol = sum(e ** 3 for e in ev) / len(ev)
    nbox = _logint(rng, lo, hi)
    nbox = max(1, min(nbox, int(2.0e7 / vol)))
    g = (nbox * vol / rng.uniform(*ratio)) ** (1.0 / 3.0)
    g = max(int(math.ceil(g / gstep)) * gstep, int(math.ceil((2 * max(ev) + 4) / gstep)) * gstep)
    return nbox, min(g, 256), edges


def draw(rng):
    kind = rng.choice(["solve", "solve", "mehr", "cnn_apply", "cnn_grad", "hloc", "precond", "hartree", "gram",
                       "density"])
    if kind in ("solve", "mehr"):
        path = "mehr" if kind == "mehr" else rng.choice(["mixed", "mixed", "plain"])
        sets = ["8,12,16", "16", "12,20", "20,24", "24,28,32,36,40", "32", "28,36"]
        nbox, g, edges = _boxes_for(rng, 6, 128 if path == "mehr" else 800, sets[:4] if path == "mehr" else sets,
                                    (1.5, 3.0), rng.choice([8, 8, 8, 4]))
        return dict(kind="solve", nbox=nbox, gdim=g, edges=edges, path=path,
                    steps=rng.randint(3, 6) if path == "mehr" else rng.randint(6, 12))
    if kind in ("cnn_apply", "cnn_grad"):
        edge = rng.choice([16, 20, 24, 28, 32, 36, 40])
        most = 2.0e7 if kind == "cnn_apply" else 2.0e6
        return dict(kind=kind, nbox=_logint(rng, 4, max(5, int(most / edge ** 3))), edge=edge)
    if kind == "hartree":
        step = rng.choice([4, 8, 16])
        bc = rng.choice([1, 1, 0])
        d = [_logint(rng, 32, 200, step) for _ in range(3)]
        return dict(kind=kind, d0=d[0], d1=d[1], d2=d[2], lap=rng.choice([0, 0, 2]), bc=bc)
    if kind == "density":
        nbox, g, edges = _boxes_for(rng, 16, 1200, ["20,24", "24,28,32", "32"], (1.2, 2.2), 8)
        return dict(kind=kind, nbox=nbox, gdim=g, edges=edges)
    if kind == "gram":
        n = _logint(rng, 3, 240)
        rows = _logint(rng, 20000, max(20001, int(5.0e7 / n)))
        return dict(kind=kind, n=n, rows=rows, prec=rng.choice(["f64", "f64", "split"]))
    step = 4 if kind == "precond" else 1
    d = [_logint(rng, 16, 112, step) for _ in range(3)]
    n = _logint(rng, 1, max(2, min(96, int(4.5e7 / (d[0] * d[1] * d[2])))))
    case = dict(kind=kind, n=n, d0=d[0], d1=d[1], d2=d[2], lap=rng.choice([0, 2, 2]), dtype=rng.choice(["f64", "f32"]))
    if kind == "precond":
        case["levels"] = 2
    return case


# ------------------------------------------------------------ seeded inputs
H_GRID = 0.25  # bohr


def _rngs(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed))
    return np.random.default_rng(int(seed)), g


def _uniform(shape, g, a):
    return (2.0 * torch.rand(shape, generator=g, device=_dev(), dtype=FP64) - 1.0) * a


def _centers(n, L, sep, rng):
    """n positions at least `sep` apart (periodic), by random sequential addition"""
    out = np.zeros((n, 3))
    k = tries = 0
    while k < n:
        c = rng.uniform(0.0, L, 3)
        tries += 1
        d = np.abs(out[:k] - c)
        d = np.minimum(d, L - d)
        if k == 0 or tries > 200 * n or np.min(np.sum(d * d, axis=1)) >= sep * sep:
            out[k] = c
            k += 1
    return out


def _wells(dims, n, rng):
    """Gaussian wells in Rydberg on the periodic grid: depth 1-4 Ry, width 1.5 bohr"""
    h = H_GRID
    dep = torch.as_tensor(2.0 * rng.uniform(-2.0, -0.5, n), device=_dev(), dtype=FP64)
    f = []
    for d in dims:
        c = torch.as_tensor(rng.uniform(0.0, d * h, n), device=_dev(), dtype=FP64)
        x = torch.arange(d, device=_dev(), dtype=FP64) * h
        r = (x[None, :] - c[:, None]).abs()
        r = torch.minimum(r, d * h - r)
        f.append(torch.exp(-r * r / (2.0 * 1.5 ** 2)))
    xy = (dep[:, None, None] * f[0][:, :, None] * f[1][:, None, :]).reshape(n, -1)
    return (xy.t().contiguous() @ f[2]).reshape(dims)


class Geometry:
    """Box layout of a case: origins, edges, offsets (host) and box groups of one edge."""

    def __init__(self, case, rng):
        self.g, self.h = int(case["gdim"]), H_GRID
        ev = np.array([int(e) for e in case["edges"].split(",")])
        self.n = int(case["nbox"])
        self.edge = rng.permutation(np.resize(ev, self.n)).astype(np.int64)
        L = self.g * self.h
        spacing = L / self.n ** (1.0 / 3.0)
        self.cen = _centers(self.n, L, 0.5 * spacing, rng)
        self.sigma = min(0.155 * float(np.mean(ev)) * self.h, 0.25 * spacing)
        o = np.floor(self.cen / self.h).astype(np.int64) - (self.edge // 2)[:, None]
        self.origin = np.mod((o // 4) * 4, self.g)
        self.off = np.zeros(self.n + 1, dtype=np.int64)
        self.off[1:] = np.cumsum(self.edge ** 3)
        self.groups = []
        for e in sorted(set(self.edge.tolist())):
            idx = np.nonzero(self.edge == e)[0]
            pos = torch.as_tensor(self.off[idx], device=_dev())[:, None] + torch.arange(e ** 3, device=_dev())[None, :]
            self.groups.append((e, idx, None if len(idx) == self.n else pos.reshape(-1)))

    def split(self, flat):
        """packed boxes -> one (m, e, e, e) tensor per group"""
        return [(flat if pos is None else flat[pos]).reshape(len(idx), e, e, e) for e, idx, pos in self.groups]

    def join(self, parts):
        if self.groups[0][2] is None:
            return parts[0].reshape(-1)
        out = torch.empty(int(self.off[-1]), device=_dev(), dtype=parts[0].dtype)
        for (_e, _i, pos), p in zip(self.groups, parts):
            out[pos] = p.reshape(-1)
        return out

    def orbitals(self, gen):
        """Gaussians about the centres with 1e-3 noise, normalised"""
        parts = []
        L = self.g * self.h
        for e, idx, _pos in self.groups:
            f = []
            for d in range(3):
                x = (torch.as_tensor(self.origin[idx, d], device=_dev())[:, None]
                     + torch.arange(e, device=_dev())[None, :]).to(FP64) * self.h
                r = x - torch.as_tensor(self.cen[idx, d], device=_dev())[:, None]
                r = r - L * torch.round(r / L)
                f.append(torch.exp(-r * r / (2.0 * self.sigma ** 2)))
            v = f[0][:, :, None, None] * f[1][:, None, :, None] * f[2][:, None, None, :]
            v = v + _uniform(v.shape, gen, 1e-3)
            nrm = (self.h ** 3 * (v * v).sum(dim=(1, 2, 3), keepdim=True)).sqrt()
            parts.append(v / nrm)
        return self.join(parts)

    def boxset(self, levels=3):
        return mgx.BoxSet(_ctx(), self.origin, self.edge, self.g, self.h, levels)


def _box_inputs(case, seed):
    rng, gen = _rngs(seed)
    geo = Geometry(case, rng)
    psi = geo.orbitals(gen)
    v = _wells((geo.g,) * 3, max(3, geo.n // 32), rng)
    return geo, psi, v, gen


def _grid_orbitals(n, dims, rng, gen):
    """full-grid orbitals: Gaussians of width 1 bohr with 1e-3 noise"""
    h = H_GRID
    f = []
    for d in dims:
        c = torch.as_tensor(rng.uniform(0.0, d * h, n), device=_dev(), dtype=FP64)
        r = torch.arange(d, device=_dev(), dtype=FP64)[None, :] * h - c[:, None]
        r = r - d * h * torch.round(r / (d * h))
        f.append(torch.exp(-0.5 * r * r))
    v = f[0][:, :, None, None] * f[1][:, None, :, None] * f[2][:, None, None, :]
    return (v + _uniform(v.shape, gen, 1e-3)).reshape(n, -1)


def _dims(case):
    return (case["d0"], case["d1"], case["d2"])


def _grid(case, ghosts, bc=1):
    return mgx.Grid.make(_dims(case), ghosts, (H_GRID,) * 3, (bc,) * 3)


def _block(t, grid):
    b = mgx.Block()
    b.data, b.dtype, b.nfunc, b.grid = t.data_ptr(), mgx.F64, t.shape[0], grid
    return b


def _net_params(rng):
    p = learned.init_params(seed=int(rng.integers(1 << 30)))
    for k in range(4):
        b = p["b%d" % k]
        p["b%d" % k] = (0.05 * rng.standard_normal(b.shape)).astype(np.float32)
    return p


def _cnn_fields(case, seed):
    """residual-like boxes: a smooth Gaussian part and noise, amplitudes over decades"""
    rng, gen = _rngs(seed)
    nb, e = case["nbox"], case["edge"]
    x = (torch.arange(e, device=_dev(), dtype=FP64) - 0.5 * e) / (0.2 * e)
    g = torch.exp(-0.5 * x * x)
    sm = g[:, None, None] * g[None, :, None] * g[None, None, :]
    amp = 10.0 ** (-1.0 - 4.0 * torch.rand(nb, 1, 1, 1, generator=gen, device=_dev(), dtype=FP64))
    noise = torch.randn(nb, e, e, e, generator=gen, device=_dev(), dtype=FP64)
    return _net_params(rng), sm[None], amp, noise, gen


SOLVER = {
    "plain": dict(precond_dtype=mgx.F64, gram_prec=mgx.PREC_F64),
    "mixed": dict(precond_dtype=mgx.F32, gram_prec=mgx.PREC_SPLIT),
    "mehr": dict(precond_dtype=mgx.F64, gram_prec=mgx.PREC_F64, lap_type=mgx.LAP_MEHRSTELLEN),
}


class _Net(learned.Cnn):
    """a network whose device memory goes with the object"""

    def __del__(self):
        self.close()


class _View:
    """a device buffer of the engine as torch sees it; its tensors keep the owner, and so the buffer, alive"""

    def __init__(self, owner, p, n):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(p, False), shape=(n,), typestr="<f8", version=2)


# ----------------------------------------------------------------- prepare
def _in_solve(case, seed):
    geo, psi, v, _gen = _box_inputs(case, seed)
    bs = geo.boxset()
    s = mgx.Solver(_ctx(), bs, v.cpu().numpy(), psi.cpu().numpy(), mg_levels=2, anderson_m=1, **SOLVER[case["path"]])
    s.set_graph(True)
    return dict(solver=s, steps=case["steps"], npts=int(geo.off[-1]))


def _in_cnn_apply(case, seed):
    p, sm, amp, noise, _gen = _cnn_fields(case, seed)
    R = (amp * (sm + 0.1 * noise)).contiguous()
    net = _Net(_ctx(), case["edge"], min(256, case["nbox"]), p)
    return dict(net=net, nb=case["nbox"], R=R, out=torch.empty_like(R))


def _train_pairs(case, seed):
    p, sm, _amp, noise, gen = _cnn_fields(case, seed)
    x = sm + 0.3 * noise
    x = x / x.square().mean(dim=(1, 2, 3), keepdim=True).sqrt()
    t = 0.2 * x + 0.05 * torch.randn(x.shape, generator=gen, device=_dev(), dtype=FP64)
    return p, x.to(torch.float32).contiguous(), t.to(torch.float32).contiguous()


def _in_cnn_grad(case, seed):
    p, x, t = _train_pairs(case, seed)
    return dict(net=_Net(_ctx(), case["edge"], case["nbox"], p), nb=case["nbox"], x=x, t=t)


def _torch_type(case):
    return torch.float32 if case["dtype"] == "f32" else FP64


def _hloc_inputs(case, seed):
    rng, gen = _rngs(seed)
    psi = _grid_orbitals(case["n"], _dims(case), rng, gen).to(_torch_type(case))
    return psi, _wells(_dims(case), 16, rng).reshape(-1)


def _in_hloc(case, seed):
    psi, v = _hloc_inputs(case, seed)
    return dict(lap=case["lap"], grid=_grid(case, 2), psi=psi, v=v, out=torch.empty_like(psi), n=case["n"],
                code=mgx.F32 if case["dtype"] == "f32" else mgx.F64)


def _residual_inputs(case, seed):
    """residuals of orbitals: the orbital times a smooth factor, plus noise"""
    rng, gen = _rngs(seed)
    psi = _grid_orbitals(case["n"], _dims(case), rng, gen)
    r = 0.05 * psi + _uniform(psi.shape, gen, 2e-3)
    return r, float(mgx.lib().mgx_gamma((C.c_double * 3)(*(H_GRID,) * 3), 2, 0.0, -3.0))


def _in_precond(case, seed):
    r, gam = _residual_inputs(case, seed)
    return dict(lap=case["lap"], levels=case["levels"], gamma=gam, grid=_grid(case, 2), res=r, n=case["n"],
                out=torch.empty_like(r), code=mgx.F32 if case["dtype"] == "f32" else mgx.F64)


def _charge(case, seed):
    """4 pi rho of Gaussian charges with a little noise, of zero mean on a periodic grid"""
    rng, gen = _rngs(seed)
    q = -_wells(_dims(case), 24, rng) + _uniform(_dims(case), gen, 1e-3)
    if case["bc"] == 1:
        q = q - q.mean()
    return 4.0 * math.pi * q


def _in_hartree(case, seed):
    ng = 2 if case["lap"] == 2 else 1
    grid = _grid(case, ng, case["bc"])
    rho = F.pad(_charge(case, seed)[None], (ng,) * 6).contiguous()
    vh = torch.zeros_like(rho)
    return dict(lap=case["lap"], rho=rho, vh=vh, brho=_block(rho, grid), bvh=_block(vh, grid), ng=ng,
                stats=mgx.PoissonStats())


def _gram_inputs(case, seed):
    _rng, gen = _rngs(seed)
    n, k = case["n"], case["rows"]
    a = torch.randn(n, k, generator=gen, device=_dev(), dtype=FP64)
    # neighbouring orbitals overlap; H psi is psi scaled plus its own part
    a[1:] += 0.5 * a[:-1]
    b = torch.randn(n, k, generator=gen, device=_dev(), dtype=FP64) * 0.5 - 1.5 * a
    return a, b


def _in_gram(case, seed):
    a, b = _gram_inputs(case, seed)
    n = case["n"]
    return dict(a=a, b=b, n=n, k=case["rows"], vel=1.0 / case["rows"], S=torch.empty(n, n, device=_dev(), dtype=FP64),
                H=torch.empty(n, n, device=_dev(), dtype=FP64),
                prec=mgx.PREC_SPLIT if case["prec"] == "split" else mgx.PREC_F64)


def _density_inputs(case, seed):
    geo, psi, _v, gen = _box_inputs(case, seed)
    a = torch.randn(geo.n, geo.n, generator=gen, device=_dev(), dtype=FP64) * 0.1
    return geo, psi, (2.0 * torch.eye(geo.n, device=_dev(), dtype=FP64) + a + a.t()).contiguous()


def _in_density(case, seed):
    geo, psi, dm = _density_inputs(case, seed)
    return dict(bs=geo.boxset(), psi=psi, dm=dm, rho=torch.empty((geo.g,) * 3, device=_dev(), dtype=FP64))


def prepare(case, seed):
    state = globals()["_in_" + case["kind"]](case, seed)
    state["kind"] = case["kind"]
    torch.cuda.synchronize()
    return state


# --------------------------------------------------------------------- run
def _run_solve(s):
    sol = s["solver"]
    sol.reset()
    st = sol.run(0.0, s["steps"])
    p = C.c_void_p()
    _ctx().check(mgx.lib().mgx_solver_buffers(sol.h, C.byref(p), None, None, None, None), "mgx_solver_buffers")
    return dict(energy=np.float64(st.band_energy), residual=np.float64(st.residual),
                psi=torch.as_tensor(_View(sol, p.value, s["npts"]), device=_dev()))


def _run_cnn_apply(s):
    s["net"].apply(s["nb"], s["R"], s["out"])
    return s["out"]


def _run_cnn_grad(s):
    loss, g = s["net"].grad(s["x"], s["t"], s["nb"])
    return dict(g, loss=np.float64(loss))


def _run_hloc(s):
    ld = s["psi"].shape[1]
    _ctx().call("mgx_hloc_apply", s["lap"], C.byref(s["grid"]), s["code"], mgx.ptr(s["psi"]), ld, s["n"], mgx.ptr(s["v"]),
                mgx.ptr(s["out"]), ld)
    return s["out"]


def _run_precond(s):
    ld = s["res"].shape[1]
    _ctx().call("mgx_precond_mg", s["lap"], s["levels"], s["gamma"], s["code"], C.byref(s["grid"]), mgx.ptr(s["res"]), ld,
                s["n"], None, mgx.ptr(s["out"]), ld)
    return s["out"]


def _run_hartree(s):
    # from zero: torch clears on its own stream, the engine runs on another
    s["vh"].zero_()
    torch.cuda.current_stream().synchronize()
    _ctx().call("mgx_poisson_mg", s["lap"], C.byref(s["brho"]), C.byref(s["bvh"]), 2, 2, 10, 1e-16, 10,
                C.byref(s["stats"]))
    n = s["ng"]
    return s["vh"][0, n:-n, n:-n, n:-n]


def _run_gram(s):
    c = _ctx()
    c.call("mgx_local_gram", s["prec"], mgx.ptr(s["a"]), s["k"], s["k"], s["n"], 1, s["vel"], mgx.ptr(s["S"]))
    c.call("mgx_local_product", s["prec"], mgx.ptr(s["a"]), mgx.ptr(s["b"]), s["k"], s["k"], s["n"], 1, s["vel"],
           mgx.ptr(s["H"]))
    return s["S"], s["H"]


def _run_density(s):
    q = s["bs"].density(s["psi"], s["dm"], s["rho"])
    return dict(rho=s["rho"], charge=np.float64(q))


def run(state):
    return globals()["_run_" + state["kind"]](state)


# -------------------------------------------------------------------- work
def _npts(case):
    e = np.resize([int(x) for x in case["edges"].split(",")], case["nbox"])
    return float(np.sum(e ** 3))


def work(case):
    k = case["kind"]
    if k == "solve":
        # the state one step hands to the next: psi and the previous psi (FP64),
        # the previous correction; each read and written once a step, V read once
        np_, g3 = _npts(case), float(case["gdim"]) ** 3
        s = 4.0 if case["path"] == "mixed" else 8.0
        cover = np_ / g3
        # H psi, four fine sweeps and the coarse ones, S and H over the boxes that
        # cover a point, the residual, the update
        flops = np_ * (28 + 4.6 * 30 + 3 * cover + 2 * cover + 12)
        return dict(bytes=case["steps"] * ((8 + 8 + 8 + 2 * s) * np_ + 8 * g3), flops=case["steps"] * flops)
    if k in ("cnn_apply", "cnn_grad"):
        m = case["nbox"] * float(case["edge"]) ** 3
        fwd = 2.0 * 27 * (16 + 256 + 256 + 16) * m
        if k == "cnn_apply":
            return dict(bytes=16.0 * m, flops=fwd)
        return dict(bytes=8.0 * m, flops=2 * fwd + 2.0 * 27 * (256 + 256 + 16) * m)
    if k == "gram":
        n, r = case["n"], float(case["rows"])
        return dict(bytes=16.0 * n * r + 16.0 * n * n, flops=r * n * (n + 1) + 2.0 * r * n * n)
    if k == "density":
        np_, g3 = _npts(case), float(case["gdim"]) ** 3
        return dict(bytes=8 * np_ + 8 * g3, flops=2 * np_ * (np_ / g3) + 2 * np_)
    m = float(case["d0"] * case["d1"] * case["d2"])
    if k == "hartree":
        # rho read, the potential read and written once
        return dict(bytes=24.0 * m, flops=10 * m * (5 * 30 * 8.0 / 7.0 + 60))
    if k == "hloc":
        s = 4.0 if case["dtype"] == "f32" else 8.0
        return dict(bytes=2 * s * m * case["n"] + 8 * m, flops=30.0 * m * case["n"])
    return dict(bytes=16.0 * m * case["n"], flops=m * case["n"] * (4 * 30 + 40) * 8.0 / 7.0)


def tolerance(case):
    return TOLERANCE[case["kind"]](case)


# about four times the largest differences from exact() seen over the ranges
TOLERANCE = {
    # mixed: FP32 corrections and split S/H, carried through the Anderson steps
    "solve": lambda c: {"rel": 4e-7, "max": 1e-5} if c["path"] == "mixed" else {"rel": 2e-12, "max": 2e-11},
    # BF16 weights and activations, FP32 sums
    "cnn_apply": lambda c: {"rel": 1.5e-3, "max": 0.035},
    "cnn_grad": lambda c: {"rel": 0.03, "max": 0.1},
    "hloc": lambda c: {"rel": 1e-7, "max": 3e-7} if c["dtype"] == "f32" else {"rel": 3e-14, "max": 1.5e-12},
    "precond": lambda c: {"rel": 1.5e-7, "max": 7e-7} if c["dtype"] == "f32" else {"rel": 8e-15, "max": 2e-14},
    "hartree": lambda c: {"rel": 1e-12, "max": 3e-12},
    # split: products of 32-bit halves
    "gram": lambda c: {"rel": 1e-8, "max": 3e-8} if c["prec"] == "split" else {"rel": 1.2e-13, "max": 4e-13},
    "density": lambda c: {"rel": 1e-15, "max": 3e-15},
}


# ---------------------------------------------------- the same in 64 bits
def _sh(u, d, wrap):
    """out[i] = u[i + d] over the last three axes: periodic, or zero outside"""
    for ax, o in zip((-3, -2, -1), d):
        if o == 0:
            continue
        if wrap:
            u = torch.roll(u, -o, ax)
        else:
            n = u.shape[ax]
            z = torch.zeros_like(u)
            if abs(o) < n:
                src, dst = (o, 0) if o > 0 else (0, -o)
                z.narrow(ax, dst, n - abs(o)).copy_(u.narrow(ax, src, n - abs(o)))
            u = z
    return u


def _axis(k, o):
    return tuple(o if a == k else 0 for a in range(3))


def _lap(u, lap, h, wrap):
    """-Laplacian: 0 Mehrstellen (19 points), 1 second order, 2 fourth order; spacing h in every direction"""
    ih = 1.0 / (h * h)
    if lap == 1:
        out = 6.0 * ih * u
        for k in range(3):
            out -= ih * (_sh(u, _axis(k, 1), wrap) + _sh(u, _axis(k, -1), wrap))
        return out
    if lap == 2:
        out = 7.5 * ih * u
        for k in range(3):
            out -= 4.0 / 3.0 * ih * (_sh(u, _axis(k, 1), wrap) + _sh(u, _axis(k, -1), wrap))
            out += ih / 12.0 * (_sh(u, _axis(k, 2), wrap) + _sh(u, _axis(k, -2), wrap))
        return out
    out = 4.0 * ih * u
    for k in range(3):
        out -= ih / 3.0 * (_sh(u, _axis(k, 1), wrap) + _sh(u, _axis(k, -1), wrap))
    for a, b in ((0, 1), (1, 2), (0, 2)):
        for s, t in itertools.product((1, -1), (1, -1)):
            d = [0, 0, 0]
            d[a], d[b] = s, t
            out -= ih / 6.0 * _sh(u, d, wrap)
    return out


def _bop(u, wrap):
    """the Mehrstellen right-hand-side operator"""
    out = 0.5 * u
    for k in range(3):
        out += (_sh(u, _axis(k, 1), wrap) + _sh(u, _axis(k, -1), wrap)) / 12.0
    return out


def _omega(lap, h):
    d = (4.0, 6.0, 7.5)[lap] / (h * h)
    return (1.0, 6.0 / 7.0, 2.0 / 3.0)[lap] / d


def _restrict(u, wrap):
    for k in range(3):
        u = 0.25 * (_sh(u, _axis(k, 1), wrap) + _sh(u, _axis(k, -1), wrap)) + 0.5 * u
        u = u.index_select(k - 3, torch.arange(0, u.shape[k - 3], 2, device=u.device))
    return u


def _extend(c, wrap):
    for k in range(3):
        c = _interleave(c, 0.5 * (c + _sh(c, _axis(k, 1), wrap)), k - 3)
    return c


def _interleave(a, b, ax):
    ax = ax % a.dim()
    shape = list(a.shape)
    shape[ax] *= 2
    return torch.stack([a, b], dim=ax + 1).reshape(shape)


def _vcycle_pre(v, f, lap, level, top, h, wrap):
    """the orbital preconditioner's V-cycle: the residual before the last pre-sweep is restricted"""
    om = _omega(lap, h)
    w = None
    for _ in range(4 if level == top else 2):
        w = _lap(v, lap, h, wrap) - f
        v = v - om * w
    if level == top:
        return v
    rc = _restrict(w, wrap)
    v = v - _extend(_vcycle_pre(torch.zeros_like(rc), rc, 1, level + 1, top, 2 * h, wrap), wrap)
    for _ in range(2):
        v = v - om * (_lap(v, lap, h, wrap) - f)
    return v


class _Cells:
    """8^3 blocks of the periodic grid with the boxes (grown by `reach`) that cover each"""

    B = 8

    def __init__(self, geo, reach):
        self.geo, self.reach = geo, reach
        g, B = geo.g, self.B
        nc = -(-g // B)
        cells, boxes = [], []
        for j in range(geo.n):
            e = int(geo.edge[j]) + 2 * reach
            ax = [np.unique(np.mod(np.arange(e) + geo.origin[j, d] - reach, g) // B) for d in range(3)]
            c = ((ax[0][:, None, None] * nc + ax[1][None, :, None]) * nc + ax[2][None, None, :]).reshape(-1)
            cells.append(c)
            boxes.append(np.full(len(c), j))
        cells, boxes = np.concatenate(cells), np.concatenate(boxes)
        order = np.argsort(cells, kind="stable")
        cells, boxes = cells[order], boxes[order]
        ids, first, count = np.unique(cells, return_index=True, return_counts=True)
        slot = np.arange(len(cells)) - np.repeat(first, count)
        table = np.full((len(ids), int(count.max())), -1)
        table[np.repeat(np.arange(len(ids)), count), slot] = boxes
        self.nc, dev = nc, _dev()
        self.ids, self.table = torch.as_tensor(ids, device=dev), torch.as_tensor(table, device=dev)
        self.origin = torch.as_tensor(geo.origin, device=dev)
        self.edge = torch.as_tensor(geo.edge, device=dev)
        self.off = torch.as_tensor(geo.off[:-1], device=dev)
        eext = geo.edge + 2 * reach
        self.off_ext = torch.as_tensor(np.concatenate([[0], np.cumsum(eext ** 3)[:-1]]), device=dev)

    def chunks(self, budget=1 << 26):
        step = max(1, budget // (self.table.shape[1] * self.B ** 3))
        for a in range(0, self.table.shape[0], step):
            yield self.ids[a:a + step], self.table[a:a + step]

    def points(self, ids):
        c = [ids // (self.nc * self.nc), (ids // self.nc) % self.nc, ids % self.nc]
        return [x[:, None] * self.B + torch.arange(self.B, device=ids.device)[None, :] for x in c]

    def index(self, ids, tab, ext):
        """flat index (0 where outside) and mask, (cells, slots, 8^3), into packed boxes grown by `reach` if ext"""
        g, r = self.geo.g, self.reach if ext else 0
        p, b = self.points(ids), tab.clamp(min=0)
        e = self.edge[b] + 2 * r
        loc, ok = [], []
        for d in range(3):
            q = p[d][:, None, :]
            x = torch.remainder(q - self.origin[b][:, :, d, None] + r, g)
            loc.append(x)
            ok.append((x < e[:, :, None]) & (q < g) & (tab >= 0)[:, :, None])
        m = ok[0][:, :, :, None, None] & ok[1][:, :, None, :, None] & ok[2][:, :, None, None, :]
        o = (self.off_ext if ext else self.off)[b]
        e = e[:, :, None, None, None]
        i = (loc[0][:, :, :, None, None] * e + loc[1][:, :, None, :, None]) * e + loc[2][:, :, None, None, :]
        i = torch.where(m, i + o[:, :, None, None, None], torch.zeros_like(i))
        return i.flatten(2), m.flatten(2)

    def grown(self, parts, reach):
        """box groups grown by `reach` -> packed in box order"""
        out = torch.empty(int((self.off_ext[-1] + (self.edge[-1] + 2 * reach) ** 3).item()), device=_dev(), dtype=FP64)
        for (e, idx, _pos), p in zip(self.geo.groups, parts):
            n = (e + 2 * reach) ** 3
            pos = self.off_ext[torch.as_tensor(idx, device=_dev())][:, None] + torch.arange(n, device=_dev())[None, :]
            out[pos.reshape(-1)] = p.reshape(-1)
        return out


def _inv(a):
    return torch.as_tensor(np.linalg.inv(a.cpu().numpy()), device=_dev())


def _box_v(geo, v, reach):
    """V on every box grown by `reach`, per group"""
    out = []
    for e, idx, _pos in geo.groups:
        ax = [torch.as_tensor(np.mod(geo.origin[idx, d][:, None] + np.arange(e + 2 * reach)[None, :] - reach, geo.g),
                              device=_dev()) for d in range(3)]
        out.append(v[ax[0][:, :, None, None], ax[1][:, None, :, None], ax[2][:, None, None, :]])
    return out


def _exact_solve(case, seed):
    geo, psi, v, _gen = _box_inputs(case, seed)
    lap = 0 if case["path"] == "mehr" else 2
    reach = 1 if lap == 0 else 2
    n, h, vel = geo.n, geo.h, geo.h ** 3
    cells = _Cells(geo, reach)
    vext = _box_v(geo, v, reach)
    inner = (slice(None),) + (slice(reach, -reach),) * 3
    boxid = torch.as_tensor(np.repeat(np.arange(n), geo.edge ** 3), device=_dev())

    def box(x):  # the sum over each box
        out = torch.empty(n, device=_dev(), dtype=FP64)
        for (_e, idx, _pos), u in zip(geo.groups, geo.split(x)):
            out[torch.as_tensor(idx, device=_dev())] = u.sum(dim=(1, 2, 3))
        return out

    alpha, prev, accel, hist = 0.75, None, False, None
    deig, deig2 = 1e9, 1e9
    for it in range(case["steps"]):
        parts = [F.pad(u, (reach,) * 6) for u in geo.split(psi)]
        if lap == 2:
            hext = [_lap(u, 2, h, False) + vv * u for u, vv in zip(parts, vext)]
            bext = parts
        else:
            hext = [_lap(u, 0, h, False) + _bop(vv * u, False) for u, vv in zip(parts, vext)]
            bext = [_bop(u, False) for u in parts]
        hpsi = geo.join([u[inner].contiguous() for u in hext])
        he = cells.grown(hext, reach)
        be = cells.grown(bext, reach) if lap == 0 else None
        S, Hm, Bm = (torch.zeros(n * n, device=_dev(), dtype=FP64) for _ in range(3))
        for ids, tab in cells.chunks():
            i0, m0 = cells.index(ids, tab, False)
            ie, me = cells.index(ids, tab, True)
            P, Q = psi[i0] * m0, he[ie] * me
            pair = (tab[:, :, None] * n + tab[:, None, :]).reshape(-1)
            both = ((tab[:, :, None] >= 0) & (tab[:, None, :] >= 0)).reshape(-1).nonzero()[:, 0]
            pair = pair[both]
            for M, X in ((S, P), (Hm, Q)) + (((Bm, be[ie] * me),) if lap == 0 else ()):
                M.index_add_(0, pair, torch.bmm(P, X.transpose(1, 2).contiguous()).reshape(-1)[both])
        S, Hm, Bm = (vel * x.reshape(n, n) for x in (S, Hm, Bm))
        if lap == 2:
            Hm = 0.5 * (Hm + Hm.t())
        Sinv = _inv(S)
        theta = (Sinv if lap == 2 else _inv(Bm)) @ Hm
        energy = 0.5 * float(torch.trace(theta))
        R = torch.zeros_like(psi)
        for ids, tab in cells.chunks():
            i0, m0 = cells.index(ids, tab, False)
            ie, me = cells.index(ids, tab, True)
            P = (be[ie] * me) if lap == 0 else psi[i0] * m0
            b = tab.clamp(min=0)
            T = theta[b[:, None, :], b[:, :, None]]  # (cells, j, a) = theta[a, j]
            R[i0[m0]] = torch.bmm(T, P)[m0]
        R -= hpsi
        sd = torch.diagonal(Sinv)
        rnorm = 0.5 * math.sqrt(float((sd * vel * box(R * R)).sum()))
        if it > 0:
            old, deig = deig, abs(energy - prev)
            deig2 = max(deig, old)
        prev = energy
        accel = accel or 4.0 * deig2 < 1e-2 * n
        f = alpha * geo.join([_vcycle_pre(torch.zeros_like(u), u, lap, 0, 2, h, False) for u in geo.split(R)])
        if not accel:
            psi = psi + f
        else:
            x0, f0, t = psi, f, 0.0
            if hist is not None:
                x0, f0 = hist
                df = f - f0
                mat, rhs = float((sd * box(df * df)).sum()), float((sd * box(df * f)).sum())
                t = rhs / mat if mat > 0.0 else 0.0
                t = (-0.5 if t > 1.0 else 0.0) if t > 0.5 else max(t, -3.0)
            hist = (psi, f)
            psi = (1.0 - t) * psi + t * x0 + (1.0 - t) * f + t * f0
        psi = psi / torch.sqrt(vel * box(psi * psi))[boxid]
    return dict(energy=np.float64(energy), residual=np.float64(rnorm), psi=psi)


def _cols(x):
    """the 27 zero-padded neighbours of every voxel: (m, e, e, e, c) -> (voxels, 27 c)"""
    e, c = x.shape[1], x.shape[4]
    xp = F.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    t = [xp[:, i:i + e, j:j + e, k:k + e] for i, j, k in itertools.product(range(3), repeat=3)]
    return torch.stack(t, dim=4).reshape(-1, 27 * c)


def _conv(x, w):
    """3^3 convolution, channels last: x (m, e, e, e, ci), w (27, co, ci)"""
    out = _cols(x) @ w.permute(0, 2, 1).reshape(-1, w.shape[1]).contiguous()
    return out.reshape(x.shape[:4] + (w.shape[1],))


def _net(p, x):
    """the network's output and the input of every layer"""
    h = [x[..., None]]
    for k in range(4):
        z = _conv(h[-1], p["w%d" % k]) + p["b%d" % k]
        h.append(torch.relu(z) if k < 3 else z)
    return p["s"] * x + h[4][..., 0], h


def _net_exact(p):
    return {k: torch.as_tensor(np.asarray(v), device=_dev(), dtype=FP64) for k, v in p.items()}


def _exact_cnn_apply(case, seed):
    p, sm, amp, noise, _gen = _cnn_fields(case, seed)
    q = _net_exact(p)
    R = amp * (sm + 0.1 * noise)
    out = torch.empty_like(R)
    step = max(1, int(2 ** 21 / case["edge"] ** 3))
    for a in range(0, case["nbox"], step):
        r = R[a:a + step]
        rms = r.square().mean(dim=(1, 2, 3), keepdim=True).sqrt()
        out[a:a + step] = rms * _net(q, r / rms)[0]
    return out


def _exact_cnn_grad(case, seed):
    p, x, t = _train_pairs(case, seed)
    q = _net_exact(p)
    g = {k: torch.zeros_like(v) for k, v in q.items()}
    loss = 0.0
    step = max(1, int(2 ** 20 / case["edge"] ** 3))
    for a in range(0, case["nbox"], step):
        xc, tc = x[a:a + step].to(FP64), t[a:a + step].to(FP64)
        y, h = _net(q, xc)
        loss += float((y - tc).square().sum()) / x.numel()
        dz = (2.0 / x.numel()) * (y - tc)
        g["s"] += (dz * xc).sum()
        dz = dz[..., None]
        for k in (3, 2, 1, 0):
            w = q["w%d" % k]
            g["b%d" % k] += dz.sum(dim=(0, 1, 2, 3))
            dw = _cols(h[k]).t().contiguous() @ dz.reshape(-1, w.shape[1])
            g["w%d" % k] += dw.reshape(27, w.shape[2], w.shape[1]).permute(0, 2, 1)
            if k:
                dz = _conv(dz, w.flip(0).permute(0, 2, 1)) * (h[k] > 0)
    return dict(g, loss=np.float64(loss))


def _exact_hloc(case, seed):
    psi, v = _hloc_inputs(case, seed)
    u = psi.to(FP64).reshape((case["n"],) + _dims(case))
    v = v.reshape(_dims(case))
    out = _lap(u, case["lap"], H_GRID, True) + (_bop(v * u, True) if case["lap"] == 0 else v * u)
    return out.reshape(case["n"], -1)


def _exact_precond(case, seed):
    r, gam = _residual_inputs(case, seed)
    r = r.reshape((case["n"],) + _dims(case))
    return _vcycle_pre(gam * r, r, case["lap"], 0, case["levels"], H_GRID, True).reshape(case["n"], -1)


def _exact_hartree(case, seed):
    wrap = case["bc"] == 1

    def edge(u):  # a non-periodic grid holds zero on its index-0 planes
        if wrap:
            return u
        u = u.clone()
        u[0], u[:, 0], u[:, :, 0] = 0.0, 0.0, 0.0
        return u

    def cycle(x, f, lap, h, ghosts, level):
        om = _omega(lap, h)

        def sweep(x):
            x = edge(x)
            return x - om * (_lap(x, lap, h, wrap) - f)

        x = sweep(sweep(x))
        if level < 10 and all(d % 2 == 0 and d >= 2 * ghosts for d in x.shape):
            x = edge(x)
            rc = _restrict(edge(_lap(x, lap, h, wrap) - f), wrap)
            c = cycle(torch.zeros_like(rc), rc, 1 if lap == 2 else lap, 2 * h, 1, level + 1)
            x = x - _extend(edge(c), wrap)
        return sweep(sweep(x))

    lap, h = case["lap"], H_GRID
    f = edge(_charge(case, seed))
    if lap == 0:
        f = _bop(f, wrap)
    vh = torch.zeros_like(f)
    for _ in range(10):
        vh = edge(vh)
        vh = vh + cycle(torch.zeros_like(vh), f - _lap(vh, lap, h, wrap), lap, h, 2 if lap == 2 else 1, 0)
    vh = edge(vh)
    return vh - vh.mean() if wrap else vh


def _exact_gram(case, seed):
    a, b = _gram_inputs(case, seed)
    at, bt = a.t().contiguous(), b.t().contiguous()
    # column-major results: H(i, j) = <a_i, b_j> is H^T row by row
    return a @ at / case["rows"], (a @ bt).t().contiguous() / case["rows"]


def _exact_density(case, seed):
    geo, psi, dm = _density_inputs(case, seed)
    cells = _Cells(geo, 0)
    g = geo.g
    rho = torch.zeros(g ** 3, device=_dev(), dtype=FP64)
    for ids, tab in cells.chunks():
        i0, m0 = cells.index(ids, tab, False)
        P = psi[i0] * m0
        b = tab.clamp(min=0)
        val = (torch.bmm(dm[b[:, :, None], b[:, None, :]], P) * P).sum(dim=1)
        p = cells.points(ids)
        at = ((p[0][:, :, None, None] * g + p[1][:, None, :, None]) * g + p[2][:, None, None, :]).reshape(len(ids), -1)
        ok = ((p[0] < g)[:, :, None, None] & (p[1] < g)[:, None, :, None] & (p[2] < g)[:, None, None, :])
        ok = ok.reshape(len(ids), -1)
        rho[at[ok]] = val[ok]
    return dict(rho=rho.reshape(g, g, g), charge=np.float64(float(rho.sum()) * geo.h ** 3))


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)
