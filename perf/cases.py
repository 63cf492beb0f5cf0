"""Performance cases: the linear solves a CFD program hands to cfdrs_amd.

Each case is a dict of plain values; ``prepare`` makes its inputs from a
seed, ``run`` is one pass through the package's public entry points, and
``exact`` computes the same result in float64 with plain torch.

The families:

* ``spmv``      y = A x on a 2D 5-point or 3D 7-point operator;
* ``cg_jacobi`` a small 2D pressure correction by Jacobi-PCG;
* ``cg_amg``    2D / 3D pressure Poisson solves by smoothed-aggregation
                AMG-PCG, in FP64 or with the automatic precision;
* ``gs_amg``    a small 2D pressure solve by BiCGSTAB with the default AMG
                (Ruge-Stueben, classical interpolation, Gauss-Seidel);
* ``momentum``  the upwind momentum system of a lid-driven cavity by
                BiCGSTAB + Jacobi or GMRES(30) + SOR;
* ``simple``    the pressure half of one SIMPLE iteration on the device;
* ``networks``  a batch of Kirchhoff channel networks;
* ``widths``    outlet flux of a batch of networks and its gradient with
                respect to the channel widths (forward and backward);
* ``adjoint``   outlet flux of a porous 2D domain and its gradient with
                respect to the log-permeability (forward and backward).
"""
import math

import numpy as np
import torch

import cfdrs_amd as ca
from cfdrs_amd import adjoint as adj
from cfdrs_amd import network as net
from cfdrs_amd import simple as simple_mod

DEV = "cuda"
WEST, EAST, BOTTOM = 1, 2, 16  # Dirichlet faces of the grid operators


def listed():
    return [
        # one product of the 128 x 128 pressure correction: latency only
        {"name": "spmv_pressure_128x128", "op": "spmv", "nx": 128, "ny": 128, "nz": 1, "dtype": "f64"},
        # one product of a 2M-row 3D operator with odd sides: memory bandwidth
        {"name": "spmv_varcoef_127x129x125", "op": "spmv", "nx": 127, "ny": 129, "nz": 125, "dtype": "f64"},
        # pressure correction of a small 2D cavity, the cheapest preconditioner
        {"name": "cg_jacobi_128x128", "op": "cg_jacobi", "nx": 128, "ny": 128, "tol": 1e-10},
        # pressure Poisson solve of a mid-sized 2D channel with odd sides
        {"name": "cg_amg_383x255", "op": "cg_amg", "nx": 383, "ny": 255, "nz": 1, "precision": "fp64", "tol": 1e-10},
        # the largest single solve: 2M unknowns, two decades of coefficients
        {"name": "cg_amg_128x128x128_auto", "op": "cg_amg", "nx": 128, "ny": 128, "nz": 128, "precision": "auto",
         "tol": 1e-10},
        # a solver's default AMG below 10,000 rows: many small levels
        {"name": "gs_amg_96x80", "op": "gs_amg", "nx": 96, "ny": 80, "tol": 1e-12},
        # momentum predictor of a 512 x 512 cavity at Re = 1000 (the lid's unit
        # rows dominate the norm of b, so interior velocities need 1e-13)
        {"name": "momentum_bicgstab_512", "op": "momentum", "nx": 512, "method": "bicgstab", "tol": 1e-13},
        # the same predictor as the reference solves it, GMRES(30) with SOR
        {"name": "momentum_gmres_sor_384", "op": "momentum", "nx": 384, "method": "gmres", "tol": 1e-13},
        # one SIMPLE pressure step: refresh, AMG recompute, solve, corrections
        {"name": "simple_step_320x256", "op": "simple", "nx": 320, "ny": 256, "tol": 1e-11},
        # a screening batch of channel networks, the largest batch
        {"name": "networks_4096", "op": "networks", "count": 4096, "nmin": 50, "nmax": 2000, "tol": 1e-10},
        # a design step of a small batch: forward solve and adjoint gradient
        {"name": "widths_600", "op": "widths", "count": 600, "nmin": 30, "nmax": 700},
        # permeability gradient on a 256 x 256 Gaussian random field
        {"name": "adjoint_256x256", "op": "adjoint", "nx": 256, "ny": 256, "corr": 16.0, "tol": 1e-12},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "cg_jacobi", "cg_amg", "gs_amg", "momentum", "simple", "networks", "widths", "adjoint"])
    if op == "spmv":
        if rng.random() < 0.5:
            nx, ny, nz = _log_int(rng, 64, 1500), _log_int(rng, 64, 1500), 1
        else:
            nx, ny, nz = (_log_int(rng, 20, 128) for _ in range(3))
        return {"op": op, "nx": nx, "ny": ny, "nz": nz, "dtype": rng.choice(["f64", "f32"])}
    if op == "cg_jacobi":
        return {"op": op, "nx": rng.randint(24, 192), "ny": rng.randint(24, 192), "tol": 1e-10}
    if op == "cg_amg":
        if rng.random() < 0.6:
            nx, ny, nz = _log_int(rng, 64, 640), _log_int(rng, 64, 640), 1
        else:
            nx, ny, nz = (rng.randint(24, 112) for _ in range(3))
        return {"op": op, "nx": nx, "ny": ny, "nz": nz, "precision": rng.choice(["fp64", "auto"]), "tol": 1e-10}
    if op == "gs_amg":
        return {"op": op, "nx": rng.randint(24, 100), "ny": rng.randint(24, 100), "tol": 1e-12}
    if op == "momentum":
        return {"op": op, "nx": rng.randint(64, 512), "method": rng.choice(["bicgstab", "gmres"]), "tol": 1e-13}
    if op == "simple":
        return {"op": op, "nx": rng.randint(80, 400), "ny": rng.randint(80, 400), "tol": 1e-11}
    if op == "networks":
        nmax = _log_int(rng, 100, 2000)
        return {"op": op, "count": _log_int(rng, 32, 3000), "nmin": rng.randint(20, 60), "nmax": nmax, "tol": 1e-10}
    if op == "widths":
        nmax = _log_int(rng, 100, 1500)
        return {"op": op, "count": _log_int(rng, 32, 800), "nmin": rng.randint(20, 60), "nmax": nmax}
    return {"op": op, "nx": rng.randint(64, 288), "ny": rng.randint(64, 288), "corr": rng.uniform(6.0, 24.0),
            "tol": 1e-12}


# ---- grid operators as diagonals ------------------------------------------------
def _faces(k, inv_h2, mask):
    """{offset: coefficients} of the variable-coefficient Poisson
    operator on the cells of k (nz, ny, nx): harmonic face coefficients, and
    k / h^2 added to the diagonal at the Dirichlet faces in ``mask``."""
    nz, ny, nx = k.shape
    diag = torch.zeros_like(k)
    out = {}
    for axis, step in ((0, nx * ny), (1, nx), (2, 1)):
        if k.shape[axis] == 1:
            continue
        a = k.narrow(axis, 0, k.shape[axis] - 1)
        b = k.narrow(axis, 1, k.shape[axis] - 1)
        face = 2.0 * a * b / (a + b) * inv_h2
        edge = torch.zeros_like(k.narrow(axis, 0, 1))
        lower, upper = torch.cat([edge, face], axis), torch.cat([face, edge], axis)
        diag = diag + lower + upper
        out[-step], out[step] = -lower, -upper
    wall = torch.zeros_like(k)
    if mask & WEST:
        wall[:, :, 0] += 1.0
    if mask & EAST:
        wall[:, :, -1] += 1.0
    if mask & BOTTOM:
        wall[0] += 1.0
    out[0] = diag + wall * k * inv_h2
    return {o: out[o].reshape(-1) for o in sorted(out)}


def _csr(diags):
    """(row_ptr, columns, values) of nonzero entries, columns ascending."""
    offsets = sorted(diags)
    vals = torch.stack([diags[o] for o in offsets], 1).cpu()
    n = vals.shape[0]
    keep = vals != 0.0
    cols = torch.arange(n)[:, None] + torch.tensor(offsets)[None, :]
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(keep.sum(1).numpy(), out=rp[1:])
    return rp, cols[keep].numpy(), vals[keep].numpy()


def _matvec(diags, x):
    pad = max(abs(o) for o in diags)
    xp = torch.nn.functional.pad(x, (pad, pad))
    y = torch.zeros_like(x)
    for o, d in diags.items():
        y += d * xp[pad + o:pad + o + x.numel()]
    return y


def _field(case, seed):
    """Cell coefficients (nz, ny, nx) on the GPU: uniform in 2D, two decades
    of log-uniform contrast in 3D."""
    shape = (case.get("nz", 1), case["ny"], case["nx"])
    if shape[0] == 1:
        return torch.ones(shape, dtype=torch.float64, device=DEV)
    g = np.random.default_rng([seed, 1]).uniform(-math.log(10.0), math.log(10.0), shape)
    return torch.exp(torch.from_numpy(g).to(DEV))


def _grid_operator(case, seed):
    return _faces(_field(case, seed), float(case["nx"]) ** 2, EAST if case.get("nz", 1) == 1 else BOTTOM)


def _rand(seed, tag, n):
    return torch.from_numpy(np.random.default_rng([seed, tag]).uniform(-1.0, 1.0, n)).to(DEV)


def _device_matrix(diags):
    rp, ci, v = _csr(diags)
    n = rp.size - 1
    return ca.CsrMatrix.from_parts(v, ci, rp, n, n)


def _momentum(case, seed):
    """First-order upwind x-momentum operator and right-hand side of the
    lid-driven cavity (unit square, Re = 1000, dt = 0.05)."""
    n = case["nx"]
    h, mu, dt = 1.0 / (n - 1), 1e-3, 0.05
    rng = np.random.default_rng([seed, 2])
    y = np.linspace(0.0, 1.0, n)
    u = np.tile((y ** 4)[:, None], (1, n))
    v = np.zeros((n, n))
    u[1:-1, 1:-1] += 0.05 * rng.uniform(-1.0, 1.0, (n - 2, n - 2))
    v[1:-1, 1:-1] += 0.05 * rng.uniform(-1.0, 1.0, (n - 2, n - 2))
    u[0, :] = u[:, 0] = u[:, -1] = 0.0
    u[-1, :] = 1.0
    inner = np.zeros((n, n), bool)
    inner[1:-1, 1:-1] = True
    fx = u * h
    fy = np.zeros((n, n))
    fy[:, :-1] = 0.5 * (v[:, :-1] + v[:, 1:]) * h
    aw, ae = mu + np.maximum(fx, 0.0), mu + np.maximum(-fx, 0.0)
    a_s, an = mu + np.maximum(fy, 0.0), mu + np.maximum(-fy, 0.0)
    ap = aw + ae + a_s + an + h * h / dt
    z = np.zeros((n, n))
    parts = {-n: np.where(inner, -a_s, z), -1: np.where(inner, -aw, z), 0: np.where(inner, ap, 1.0),
             1: np.where(inner, -ae, z), n: np.where(inner, -an, z)}
    b = np.where(inner, h * h / dt * u, u)
    return {o: torch.from_numpy(p.reshape(-1)).to(DEV) for o, p in parts.items()}, torch.from_numpy(b.reshape(-1)).to(DEV)


# ---- networks ---------------------------------------------------------------------
def _networks(case, seed):
    """Planar channel networks: each node joins the grid node left of or above
    it (a spanning tree), and about a third close a loop to the other one."""
    lo, hi, count = case["nmin"], case["nmax"], case["count"]
    sizes = np.random.default_rng([lo, hi, count]).integers(lo, hi + 1, count)
    rng = np.random.default_rng([seed, 3])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    sys = np.repeat(np.arange(sizes.size), sizes)
    loc = np.arange(off[-1]) - off[sys]
    w = np.ceil(np.sqrt(sizes)).astype(np.int64)[sys]
    left, up = loc % w > 0, loc >= w
    coin = rng.random(loc.size)
    both = left & up
    loop = np.zeros(loc.size, bool)
    loop[rng.permutation(np.nonzero(both)[0])[:int(0.36 * np.count_nonzero(both))]] = True
    take_left = left & (~both | (coin < 0.5) | loop)
    take_up = up & (~both | (coin >= 0.5) | loop)
    nodes = np.concatenate([loc[take_left], loc[take_up]])
    other = np.concatenate([loc[take_left] - 1, (loc - w)[take_up]])
    of = np.concatenate([sys[take_left], sys[take_up]])
    order = np.argsort(of, kind="stable")
    ei, ej, of = other[order], nodes[order], of[order]
    eoff = np.concatenate([[0], np.cumsum(np.bincount(of, minlength=sizes.size))]).astype(np.int64)
    width = rng.uniform(50e-6, 500e-6, ei.size)
    length = rng.uniform(1e-3, 10e-3, ei.size)
    inlet, outlet = off[:-1], off[1:] - 1
    fixed = np.zeros(off[-1], np.uint8)
    fixed[inlet] = fixed[outlet] = 1
    value = np.zeros(off[-1])
    value[inlet] = net.INLET_PRESSURE
    return {"off": off, "eoff": eoff, "ei": ei, "ej": ej, "of": of, "sys": sys, "width": width, "length": length,
            "fixed": fixed, "value": value, "outlet": outlet}


def _batch(n):
    g, _ = net.rect_conductance(n["width"], net.CHANNEL_HEIGHT, n["length"])
    return net.NetworkBatch(n["off"], n["eoff"], n["ei"], n["ej"], g, n["fixed"], n["value"])


def _conductance(width, length):
    """G(w) of rectangular ducts of the package's default height."""
    h = torch.full_like(width, net.CHANNEL_HEIGHT)
    eps = torch.minimum(width, h) / torch.maximum(width, h)
    po = 96.0 / ((1.0 + eps) ** 2 * (1.0 - 192.0 * eps / math.pi ** 5 * torch.tanh(math.pi / (2.0 * eps))))
    area = width * h
    dh = 2.0 * area / (width + h)
    return 2.0 * area * dh ** 2 / (po * net.WATER_VISCOSITY * length)


class _NetworkMath:
    """Kirchhoff systems of all networks at once, by segmented Jacobi-CG on
    vectors padded to one row per network."""

    def __init__(self, n, g):
        count, m = n["off"].size - 1, int(np.diff(n["off"]).max())
        slot = n["sys"] * m + np.arange(n["off"][-1]) - n["off"][:-1][n["sys"]]
        i, j = n["ei"] + n["of"] * m, n["ej"] + n["of"] * m
        # up to four (edge, neighbour) pairs per node
        ends, others = np.concatenate([i, j]), np.concatenate([j, i])
        order = np.argsort(ends, kind="stable")
        first = np.concatenate([[0], np.cumsum(np.bincount(ends, minlength=count * m))])
        rank = np.arange(ends.size) - first[ends[order]]
        nb = np.tile(np.arange(count * m)[:, None], (1, 4))
        edge = np.full((count * m, 4), i.size)
        nb[ends[order], rank] = others[order]
        edge[ends[order], rank] = order % i.size
        t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
        self.shape, self.slot, self.nb = (count, m), t(slot), t(nb)
        self.g = torch.cat([g, torch.zeros_like(g[:1])])[t(edge)]
        self.free = self.pad(t(1.0 - n["fixed"].astype(np.float64)))
        self.diag = self.g.sum(1)
        self.diag = torch.where(self.diag > 0, self.diag, torch.ones_like(self.diag))

    def pad(self, v):
        out = torch.zeros(self.shape[0] * self.shape[1], dtype=v.dtype, device=v.device)
        out[self.slot] = v
        return out

    def apply(self, x):
        return (self.g * (x[:, None] - x[self.nb])).sum(1)

    def solve(self, x, rhs):
        """x with fixed nodes as given and (apply(x) = rhs) on free nodes."""
        x, rhs = self.pad(x), self.pad(rhs)
        total = lambda v: v.view(self.shape).sum(1, keepdim=True)  # noqa: E731
        scale = lambda a, v: (a * v.view(self.shape)).view(-1)  # noqa: E731
        for _ in range(2):  # the restart removes what the recurrence has lost
            r = (rhs - self.apply(x)) * self.free
            z = r / self.diag
            p, rz = z, total(r * z)
            first, one, zero = rz.clone(), torch.ones_like(rz), torch.zeros_like(rz)
            for it in range(6000):
                q = self.apply(p) * self.free
                pq = total(p * q)
                live = (rz > 1e-30 * first) & (pq > 0)
                if it % 50 == 0 and not bool(live.any()):
                    break
                alpha = torch.where(live, rz / torch.where(live, pq, one), zero)
                x = x + scale(alpha, p)
                r = r - scale(alpha, q)
                z = r / self.diag
                new = torch.where(live, total(r * z), rz)
                p = z + scale(torch.where(live, new / torch.where(live, rz, one), zero), p)
                rz = new
        return x[self.slot]


# ---- what a program has in hand ---------------------------------------------------
_PRECISION = {"fp64": ca.Precision.FP64, "auto": ca.Precision.AUTO}


def _config(case, max_it=20000):
    c = ca.IterativeSolverConfig.new(case["tol"]).with_max_iterations(max_it)
    return c.with_precision(_PRECISION[case.get("precision", "fp64")])


def _grf(case, seed):
    """Log-permeability: Gaussian random field, mean 0, deviation 1."""
    ny, nx = case["ny"], case["nx"]
    noise = np.random.default_rng([seed, 4]).standard_normal((ny, nx))
    ky, kx = np.fft.fftfreq(ny)[:, None], np.fft.rfftfreq(nx)[None, :]
    s = case["corr"] / math.sqrt(2.0)
    f = np.fft.irfft2(np.fft.rfft2(noise) * np.exp(-2.0 * (math.pi * s) ** 2 * (kx ** 2 + ky ** 2)), s=(ny, nx))
    return torch.from_numpy(((f - f.mean()) / f.std()).reshape(-1)).to(DEV)


def _simple_fields(case, seed):
    n = case["nx"] * case["ny"]
    u, v, p = (_rand(seed, 10 + q, n) for q in range(3))
    du, dv = (1e-2 * (1.0 + 0.5 * _rand(seed, 13 + q, n)) for q in range(2))
    return u, v, p, du, dv, torch.ones_like(u)


SIDES = (simple_mod.SIDE_PLAIN, simple_mod.SIDE_PRESSURE, simple_mod.SIDE_PLAIN, simple_mod.SIDE_PLAIN)


def prepare(case, seed):
    op = case["op"]
    s = {"case": case}
    if op == "spmv":
        d = _grid_operator(case, seed)
        s["a"] = _device_matrix(d)
        s["x"] = _rand(seed, 5, s["a"].nrows)
        if case["dtype"] == "f32":
            s["x"] = s["x"].float()
        s["y"] = torch.empty_like(s["x"])
    elif op in ("cg_jacobi", "cg_amg", "gs_amg"):
        s["a"] = _device_matrix(_grid_operator(case, seed))
        s["b"] = _rand(seed, 5, s["a"].nrows)
        s["config"] = _config(case)
        if op == "cg_jacobi":
            s["m"] = ca.JacobiPreconditioner(s["a"])
        elif op == "gs_amg":
            s["m"] = ca.AlgebraicMultigrid(s["a"], ca.AMGConfig.default())
        else:
            amg = ca.AMGConfig.smoothed_aggregation()
            amg.galerkin_on_device = True
            s["m"] = ca.AlgebraicMultigrid(s["a"], amg)
    elif op == "momentum":
        d, s["b"] = _momentum(case, seed)
        s["a"] = _device_matrix(d)
        s["config"] = _config(case)
        s["m"] = (ca.JacobiPreconditioner(s["a"]) if case["method"] == "bicgstab"
                  else ca.SuccessiveOverRelaxation(s["a"], 1.0))
    elif op == "simple":
        s["fields"] = _simple_fields(case, seed)
        h = 1.0 / (case["nx"] - 1)
        host = [f.cpu().numpy() for f in s["fields"]]
        s["system"] = simple_mod.SimplePressureCorrection(case["nx"], case["ny"], h, h, SIDES, fields=host,
                                                          positive_diagonal=True)
        amg = ca.AMGConfig.smoothed_aggregation()
        amg.galerkin_on_device = True
        s["m"] = ca.AlgebraicMultigrid(s["system"].matrix, amg)
        s["config"] = _config(case, 2000)
    elif op == "networks":
        s["batch"] = _batch(_networks(case, seed))
        s["config"] = _config(case, 50000)
    elif op == "widths":
        n = _networks(case, seed)
        s["batch"] = _batch(n)
        outlet = np.zeros(n["off"][-1], np.uint8)
        outlet[n["outlet"]] = 1
        s["design"] = net.WidthDesign(s["batch"], net.CHANNEL_HEIGHT, torch.from_numpy(n["length"]).to(DEV),
                                      torch.from_numpy(outlet).to(DEV))
        s["width"] = torch.from_numpy(n["width"]).to(DEV).requires_grad_(True)
        s["weight"] = _rand(seed, 6, case["count"])
    else:
        s["problem"] = adj.FluxProblem(case["nx"], case["ny"], case["tol"])
        s["g"] = _grf(case, seed).requires_grad_(True)
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "spmv":
        s["a"].spmv_into(s["x"], s["y"])
        return s["y"]
    if op in ("cg_jacobi", "cg_amg"):
        x = torch.zeros_like(s["b"])
        ca.cg_preconditioned(s["a"], s["b"], s["m"], x, s["config"])
        return x
    if op == "gs_amg":
        x = torch.zeros_like(s["b"])
        ca.bicgstab_preconditioned(s["a"], s["b"], s["m"], x, s["config"])
        return x
    if op == "momentum":
        x = torch.zeros_like(s["b"])
        if case["method"] == "bicgstab":
            ca.bicgstab_preconditioned(s["a"], s["b"], s["m"], x, s["config"])
        else:
            ca.gmres_preconditioned(s["a"], s["b"], s["m"], x, s["config"], 30)
        return x
    if op == "simple":
        u, v, p, du, dv, rho = s["fields"]
        u, v, p = u.clone(), v.clone(), p.clone()  # the step updates them in place
        rhs, pp = torch.empty_like(p), torch.zeros_like(p)
        imbalance = s["system"].assemble_device(u, v, p, du, dv, rho, rhs)
        s["m"].recompute_device(s["system"].matrix)
        ca.bicgstab_preconditioned(s["system"].matrix, rhs, s["m"], pp, s["config"])
        s["system"].apply_corrections_device(pp, du, dv, p, u, v, 0.3)
        return {"u": u, "v": v, "p": p, "correction": pp, "imbalance": imbalance}
    if op == "networks":
        x = torch.zeros(s["batch"].n_rows, dtype=torch.float64, device=DEV)
        s["batch"].solve(x, s["config"])
        return x
    if op == "widths":
        s["width"].grad = None
        flux = s["design"].flux(s["width"])
        flux.backward(s["weight"])
        return {"flux": flux.detach(), "gradient": s["width"].grad}
    s["g"].grad = None
    flux = adj.outlet_flux(s["g"], s["problem"])
    flux.backward()
    return {"flux": flux.detach(), "gradient": s["g"].grad}


# ---- the least work -----------------------------------------------------------------
def work(case):
    """Matrix values and vectors once each, two operations per matrix entry
    and product; a solve cannot do with less than one product."""
    op = case["op"]
    if op in ("networks", "widths"):
        n = case["count"] * (case["nmin"] + case["nmax"]) / 2.0
        edges = 1.33 * n
        nnz = n + 2.0 * edges
        if op == "networks":
            return {"bytes": 12.0 * nnz + 16.0 * n, "flops": 2.0 * nnz}
        return {"bytes": 2.0 * 12.0 * nnz + 32.0 * edges, "flops": 4.0 * nnz}
    nx, ny, nz = case["nx"], case.get("ny", case["nx"]), case.get("nz", 1)
    n = nx * ny * nz
    nnz = n * (7 if nz > 1 else 5)
    s = 4 if case.get("dtype") == "f32" else 8
    if op == "simple":
        return {"bytes": 8.0 * (nnz + 15 * n), "flops": 2.0 * nnz + 60.0 * n}
    if op == "adjoint":
        return {"bytes": 8.0 * (2 * nnz + 8 * n), "flops": 4.0 * nnz + 40.0 * n}
    return {"bytes": float(s * (nnz + 2 * n)), "flops": 2.0 * nnz}


# ---- float64 results with plain torch -------------------------------------------------
def _cg(diags, b):
    """Jacobi-PCG to the floor of float64, restarted from the true residual."""
    x = torch.zeros_like(b)
    dinv = 1.0 / diags[0]
    bb = float(b.dot(b))
    for _ in range(3):
        r = b - _matvec(diags, x)
        z = dinv * r
        p, rz = z, r.dot(z)
        for it in range(20000):
            q = _matvec(diags, p)
            alpha = rz / p.dot(q)
            x = x + alpha * p
            r = r - alpha * q
            z = dinv * r
            new = r.dot(z)
            p = z + (new / rz) * p
            rz = new
            if it % 25 == 0 and not float(r.dot(r)) > 1e-30 * bb:
                break
    return x


def _bicgstab(diags, b):
    """Jacobi-preconditioned BiCGSTAB, restarted until the residual stops falling."""
    x = torch.zeros_like(b)
    dinv = 1.0 / diags[0]
    best, best_x = math.inf, x
    for _ in range(8):
        r = b - _matvec(diags, x)
        norm = float(r.norm())
        if not norm < 0.5 * best:
            break
        best, best_x = norm, x
        rhat, p, v = r.clone(), torch.zeros_like(b), torch.zeros_like(b)
        rho = alpha = omega = torch.ones((), dtype=b.dtype, device=b.device)
        for it in range(4000):
            new = rhat.dot(r)
            p = r + (new / rho) * (alpha / omega) * (p - omega * v)
            rho = new
            ph = dinv * p
            v = _matvec(diags, ph)
            alpha = rho / rhat.dot(v)
            t0 = r - alpha * v
            sh = dinv * t0
            t = _matvec(diags, sh)
            omega = t.dot(t0) / t.dot(t)
            x = x + alpha * ph + omega * sh
            r = t0 - omega * t
            if it % 10 == 0 and not float(r.norm()) > 1e-6 * norm:
                break
        if not bool(torch.isfinite(x).all()):
            break
    return best_x


def _exact_simple(case, seed):
    nx, ny = case["nx"], case["ny"]
    h = 1.0 / (nx - 1)
    u, v, p, du, dv, rho = (f.reshape(ny, nx) for f in _simple_fields(case, seed))

    def grown(a):  # one linearly extrapolated node beyond each side
        a = torch.cat([2 * a[:, :1] - a[:, 1:2], a, 2 * a[:, -1:] - a[:, -2:-1]], 1)
        return torch.cat([2 * a[:1] - a[1:2], a, 2 * a[-1:] - a[-2:-1]], 0)

    pg = grown(p)
    gx = (pg[1:-1, 2:] - pg[1:-1, :-2]) / (2 * h)  # cell-centred gradients at every node
    gy = (pg[2:, 1:-1] - pg[:-2, 1:-1]) / (2 * h)
    dx_face, dy_face = 0.5 * (du[:, 1:] + du[:, :-1]), 0.5 * (dv[1:] + dv[:-1])
    uf = 0.5 * (u[:, 1:] + u[:, :-1]) + dx_face * (0.5 * (gx[:, 1:] + gx[:, :-1]) - (p[:, 1:] - p[:, :-1]) / h)
    vf = 0.5 * (v[1:] + v[:-1]) + dy_face * (0.5 * (gy[1:] + gy[:-1]) - (p[1:] - p[:-1]) / h)
    imbalance = ((uf[1:-1, 1:] - uf[1:-1, :-1]) + (vf[1:, 1:-1] - vf[:-1, 1:-1])) * h
    # interior unknowns; plain sides copy the node across, the east side is 0
    mx, my = nx - 2, ny - 2
    aw, ae = dx_face[1:-1, :-1].clone(), dx_face[1:-1, 1:].clone()
    a_s, an = dy_face[:-1, 1:-1].clone(), dy_face[1:, 1:-1].clone()
    aw[:, 0] = 0.0
    a_s[0] = 0.0
    an[-1] = 0.0
    ap = aw + ae + a_s + an
    ae = ae.clone()
    ae[:, -1] = 0.0
    diags = {-mx: -a_s, -1: -aw, 0: ap, 1: -ae, mx: -an}
    sol = _cg({o: d.reshape(-1) for o, d in diags.items()}, -imbalance.reshape(-1)).reshape(my, mx)
    pp = torch.zeros_like(p)
    pp[1:-1, 1:-1] = sol
    pp[1:-1, 0] = pp[1:-1, 1]
    pp[0, 1:-1], pp[-1, 1:-1] = pp[1, 1:-1], pp[-2, 1:-1]
    pp[0, 0], pp[-1, 0] = 0.5 * (pp[0, 1] + pp[1, 0]), 0.5 * (pp[-1, 1] + pp[-2, 0])
    u, v, p = u.clone(), v.clone(), p.clone()
    p[1:-1, 1:-1] += 0.3 * pp[1:-1, 1:-1]
    u[1:-1, 1:-1] -= du[1:-1, 1:-1] * 0.5 * (pp[1:-1, 2:] - pp[1:-1, :-2])
    v[1:-1, 1:-1] -= dv[1:-1, 1:-1] * 0.5 * (pp[2:, 1:-1] - pp[:-2, 1:-1])
    return {"u": u.reshape(-1), "v": v.reshape(-1), "p": p.reshape(-1), "correction": pp.reshape(-1),
            "imbalance": float(imbalance.abs().max())}


def _exact_adjoint(case, seed):
    nx, ny = case["nx"], case["ny"]
    ih2 = float(nx * nx)
    g = _grf(case, seed).requires_grad_(True)
    k = torch.exp(g).reshape(1, ny, nx)
    diags = _faces(k, ih2, WEST | EAST)
    inlet = torch.zeros_like(k)
    inlet[:, :, 0] = 1.0
    east = torch.zeros_like(k)
    east[:, :, -1] = 1.0
    b = (inlet * k * ih2).reshape(-1)
    flux_of = (east * k).reshape(-1)
    fixed = {o: d.detach() for o, d in diags.items()}
    p = _cg(fixed, b.detach())
    lam = _cg(fixed, flux_of.detach())
    flux = flux_of.detach().dot(p)
    (flux_of.dot(p) + lam.dot(b - _matvec(diags, p))).backward()
    return {"flux": flux, "gradient": g.grad}


def _exact_widths(case, seed):
    n = _networks(case, seed)
    width = torch.from_numpy(n["width"]).to(DEV).requires_grad_(True)
    g = _conductance(width, torch.from_numpy(n["length"]).to(DEV))
    m = _NetworkMath(n, g.detach())
    value = torch.from_numpy(n["value"]).to(DEV)
    p = m.solve(value, torch.zeros_like(value))
    weight = _rand(seed, 6, case["count"])
    out = torch.zeros_like(value)
    out[torch.from_numpy(n["outlet"]).to(DEV)] = 1.0
    of = torch.from_numpy(n["of"]).to(DEV)
    base = n["off"][:-1][n["of"]]
    i, j = (torch.from_numpy(n[e] + base).to(DEV) for e in ("ei", "ej"))
    drop = (out[j] - out[i]) * (p[i] - p[j])  # flow into an outlet node, per conductance
    flux = torch.zeros(case["count"], dtype=p.dtype, device=DEV).index_add_(0, of, g.detach() * drop)
    # d(sum weight flux)/dp on free nodes, then the adjoint of the free system
    c = weight[of] * g.detach() * (out[j] - out[i])
    dp = torch.zeros_like(p).index_add_(0, i, c).index_add_(0, j, -c)
    dp *= torch.from_numpy(1.0 - n["fixed"]).to(DEV)
    lam = m.solve(torch.zeros_like(p), dp)
    dg = weight[of] * drop - (lam[i] - lam[j]) * (p[i] - p[j])
    g.backward(dg)
    return {"flux": flux, "gradient": width.grad}


def exact(case, seed):
    op = case["op"]
    if op == "spmv":
        x = _rand(seed, 5, case["nx"] * case["ny"] * case["nz"])
        return _matvec(_grid_operator(case, seed), x.float().double() if case["dtype"] == "f32" else x)
    if op in ("cg_jacobi", "cg_amg", "gs_amg"):
        return _cg(_grid_operator(case, seed), _rand(seed, 5, case["nx"] * case["ny"] * case.get("nz", 1)))
    if op == "momentum":
        return _bicgstab(*_momentum(case, seed))
    if op == "simple":
        return _exact_simple(case, seed)
    if op == "networks":
        n = _networks(case, seed)
        value = torch.from_numpy(n["value"]).to(DEV)
        g = _conductance(torch.from_numpy(n["width"]).to(DEV), torch.from_numpy(n["length"]).to(DEV))
        return _NetworkMath(n, g).solve(value, torch.zeros_like(value))
    if op == "widths":
        return _exact_widths(case, seed)
    return _exact_adjoint(case, seed)
