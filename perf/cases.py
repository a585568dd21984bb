"""The calls whose speed is followed: timesteps of the dynamics kernels, the DG transport on
its own and the warm-start network, over the sizes, meshes and options they are used with.

A case names its path ("kind"):
  mevp       MEVPDynamicsKernel: one model step as the benchmark takes it (DG0 reset of h and
             A, wind, update of 100 mEVP subcycles, cell means read back)
  module     the same through the model-level MEVPDynamics module: every field is exchanged
             with host arrays in both directions
  bbm        BBMDynamicsKernel: the same step with the brittle rheology
  transport  DGTransport: a velocity, then many RK steps of one field
  train      WarmStartNet: loss, gradient and Adam step on a batch
  predict    WarmStartNet: forward pass
Meshes: "box" (uniform), "warped" (the box with non-affine elements), "sphere" (a
longitude-latitude patch). Cells are 4 km and more: at that spacing a step with the
reference's fixed mEVP parameters does not amplify rounding errors.
"""
import ctypes
import math

import numpy as np
import torch

from nextsimdg_amd import learned
from nextsimdg_amd import module as modules
from nextsimdg_amd.dynamics import BBMDynamicsKernel, DGTransport, MEVPDynamicsKernel, ParametricMesh

SUBCYCLES = 100
R_EARTH = 6371000.0
STORMS = 3


def listed():
    return [
        # the small box of the tests and of parameter studies: a step is launches and latency
        dict(name="mevp_box_24", kind="mevp", mesh="box", cg=2, nx=24, ny=24, dx=16e3, dt=120.0, fp32=False),
        # the 128 x 128 CG1/DG1 box that the benchmark runs for 24 h, with its host exchange
        dict(name="module_cg1_128", kind="module", mesh="box", cg=1, nx=128, ny=128, dx=4e3, dt=120.0, fp32=False),
        # the grid of the 25 km northern hemisphere mesh, spherical, with land
        dict(name="mevp_sphere_154x121", kind="mevp", mesh="sphere", cg=2, nx=154, ny=121, dx=25e3, dt=600.0,
             fp32=False),
        # the headline box
        dict(name="mevp_box_512", kind="mevp", mesh="box", cg=2, nx=512, ny=512, dx=4e3, dt=120.0, fp32=False),
        # single precision rheology at the size it was built for
        dict(name="mevp_fp32_1024", kind="mevp", mesh="box", cg=2, nx=1024, ny=1024, dx=4e3, dt=120.0, fp32=True),
        # the largest box of the benchmark, under several storms
        dict(name="mevp_box_2048", kind="mevp", mesh="box", cg=2, nx=2048, ny=2048, dx=4e3, dt=120.0, fp32=False),
        # a regional spherical model at high resolution
        dict(name="mevp_sphere_512", kind="mevp", mesh="sphere", cg=2, nx=512, ny=512, dx=6e3, dt=120.0, fp32=False),
        # brittle rheology on the headline box
        dict(name="bbm_box_512", kind="bbm", mesh="box", cg=2, nx=512, ny=512, dx=8e3, dt=120.0, fp32=False),
        # brittle rheology on non-affine elements, ragged size
        dict(name="bbm_warped_397x263", kind="bbm", mesh="warped", cg=2, nx=397, ny=263, dx=8e3, dt=120.0, fp32=False),
        # advection alone, as the reference's convergence tests run it, on a distorted mesh
        dict(name="transport_warped_500x333", kind="transport", mesh="warped", dg=6, scheme="rk2", limit=True, nx=500,
             ny=333, dx=4e3, dt=600.0, steps=100),
        # one optimiser step of the warm-start network at its training size and batch
        dict(name="train_256_b16", kind="train", batch=16, nx=256, ny=256),
        # the trained network applied to the 1024 x 1024 box
        dict(name="predict_1024", kind="predict", batch=1, nx=1024, ny=1024),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["mevp", "mevp", "mevp", "mevp", "bbm", "bbm", "transport", "module", "train", "predict"])
    if kind in ("train", "predict"):
        batch = rng.choice([1, 2, 5, 16]) if kind == "train" else 1
        return dict(kind=kind, batch=batch, nx=16 * log(2, 16 if batch > 5 else 40), ny=log(30, 256 if batch > 5 else 700))
    mesh = rng.choice(["box", "box", "warped", "sphere"])
    if kind == "transport":
        nx = log(24, 700)
        dg = rng.choice([1, 3, 6])
        return dict(kind=kind, mesh=mesh, dg=dg, scheme=rng.choice(["rk1", "rk2", "rk2", "rk3"]),
                    limit=rng.choice([True, False]), nx=nx, ny=max(8, int(nx * rng.uniform(0.5, 1.2))), dx=4e3,
                    dt=rng.choice([120.0, 300.0]), steps=rng.randint(40, 120))
    if kind == "bbm":
        mesh = rng.choice(["box", "warped"])  # the reference's brittle update grows without bound on the sphere
    nx = log(20, {"mevp": 1400 if mesh == "box" else 900, "bbm": 700, "module": 400}[kind])
    ny = max(12, int(nx * rng.uniform(0.5, 1.3)))
    cg = rng.choice([1, 2, 2, 2])
    fp32 = kind == "mevp" and mesh == "box" and rng.random() < 0.35
    return dict(kind=kind, mesh=mesh, cg=cg, nx=nx, ny=ny, dx=8e3 if kind == "bbm" else rng.choice([4e3, 8e3, 16e3]),
                dt=120.0, fp32=fp32)


# ---------------------------------------------------------------- inputs, from the seed
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _waves(g, x, y, n=6, top=7.0):
    """A smooth field of order one on [0, 1]^2: n plane waves."""
    k, p = _uniform(g, (n, 2), -top, top), _uniform(g, n, 0.0, 2 * math.pi)
    out = torch.zeros_like(x)
    for i in range(n):
        out += torch.sin(2 * math.pi * (k[i, 0] * x + k[i, 1] * y) + p[i])
    return out / math.sqrt(n)


def _grid(nx, ny, ox=0.0, oy=0.0, px=0, py=0):
    j, i = torch.meshgrid(torch.arange(ny + py, device="cuda", dtype=torch.float64),
                          torch.arange(nx + px, device="cuda", dtype=torch.float64), indexing="ij")
    return (i.reshape(-1) + ox) / nx, (j.reshape(-1) + oy) / ny


def _coords(case):
    """Vertices [(ny+1)(nx+1), 2] as the kernel's operators see them (metres, or longitude and
    latitude in radians of the rotated pole)."""
    nx, ny, dx = case["nx"], case["ny"], case["dx"]
    x, y = _grid(nx, ny, px=1, py=1)
    if case["mesh"] == "sphere":
        h, w = ny * dx / R_EARTH, nx * dx / R_EARTH
        mid = 0.95
        h, w = min(h, 0.9), min(w / math.cos(mid), 4.0)
        return torch.stack([(x - 0.5) * w, mid + (y - 0.5) * h], dim=1)
    c = torch.stack([x * nx * dx, y * ny * dx], dim=1)
    if case["mesh"] == "warped":
        i, j = x * nx, y * ny
        c = c + 0.12 * dx * torch.stack([torch.sin(0.9 * j + 0.3 * i), torch.cos(0.7 * i - 0.2 * j)], dim=1)
    return c


def _given(case, coords):
    """The vertices as a user passes them: on the sphere before the kernel's pole rotation."""
    if case["mesh"] != "sphere":
        return coords.cpu().numpy()
    lon, lat = coords[:, 0], coords[:, 1]
    x, y, z = torch.cos(lat) * torch.cos(lon), torch.cos(lat) * torch.sin(lon), torch.sin(lat)
    aw, bw = math.radians(-40.0), math.radians(-15.0)
    x, z = math.cos(bw) * x - math.sin(bw) * z, math.sin(bw) * x + math.cos(bw) * z
    x, y = math.cos(aw) * x - math.sin(aw) * y, math.sin(aw) * x + math.cos(aw) * y
    return torch.stack([torch.atan2(y, x), torch.asin(z)], dim=1).cpu().numpy()


def _mask(case):
    """1 on ocean: the outer ring of cells is land, and on the sphere also smooth islands."""
    nx, ny = case["nx"], case["ny"]
    m = torch.ones((ny, nx), device="cuda", dtype=torch.float64)
    if case["mesh"] == "sphere":
        x, y = _grid(nx, ny, 0.5, 0.5)
        land = torch.sin(9 * x + 2) * torch.sin(11 * y + 1) + 0.4 * torch.sin(31 * x + 17 * y) > 0.95
        m[land.reshape(ny, nx)] = 0.0
    m[0, :] = m[-1, :] = m[:, 0] = m[:, -1] = 0.0
    return m.reshape(-1)


def _inputs(case, seed):
    g = _gen(seed)
    nx, ny = case["nx"], case["ny"]
    x, y = _grid(nx, ny, 0.5, 0.5)
    n = nx * ny
    f = dict(coords=_coords(case), mask=_mask(case))
    if case["kind"] == "bbm":  # smooth thick ice
        f["hice"] = 1.0 + 0.2 * _waves(g, x, y, top=3.0) + 0.01 * _uniform(g, n, -1, 1)
        f["cice"] = 0.96 + 0.03 * _uniform(g, n, -1, 1)
    else:  # heterogeneous ice: log-normal thickness, concentrations below one
        f["hice"] = 0.3 + torch.exp(0.3 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64))
        f["cice"] = 1.0 - 0.2 * _uniform(g, n, 0, 1) ** 3
    f["uocean"], f["vocean"] = 0.01 * (2 * y - 1), 0.01 * (1 - 2 * x)
    f["ssh"] = 0.05 * _waves(g, x, y, n=3, top=2.0)
    f["uwind"], f["vwind"] = 9.0 * _waves(g, x, y, top=3.0), 9.0 * _waves(g, x, y, top=3.0)
    if "cg" in case:
        X, Y = _grid(case["cg"] * nx, case["cg"] * ny, px=1, py=1)
        w = torch.sin(math.pi * X) * torch.sin(math.pi * Y)
        f["u"], f["v"] = 0.05 * w * _waves(g, X, Y, top=3.0), 0.05 * w * _waves(g, X, Y, top=3.0)
    s = _uniform(g, (STORMS, 3), -1.0, 1.0).cpu().numpy()
    L = nx * case["dx"]
    f["storms"] = [(0.3 * L * a, 0.3 * L * b, (17.0 + 7.0 * c) * math.e) for a, b, c in s]
    return f


def _host(t):
    return t.cpu().numpy()


def _net_inputs(case, seed):
    g = _gen(seed)
    shape = (case["batch"], case["ny"], case["nx"])
    x = torch.zeros(shape + (32,), device="cuda", dtype=torch.bfloat16)
    x[..., :19] = torch.randn(shape + (19,), generator=g, device="cuda").to(torch.bfloat16)  # 19 of 32 are used
    # He-normal weights, the last layer's scaled down and its unused rows zero, as the network starts
    p = []
    for layer in range(4):
        w = torch.randn((32, 32, 3, 3), generator=g, device="cuda") * math.sqrt(2.0 / 288)
        b = 0.05 * torch.randn(32, generator=g, device="cuda")
        if layer == 3:
            w[8:], b[8:] = 0.0, 0.0
        p += [w.reshape(-1), b]
    t = 0.3 * torch.randn(shape + (8,), generator=g, device="cuda")
    w = (torch.rand(shape, generator=g, device="cuda") > 0.1).float()  # 1 on ocean, 0 on land
    return x, torch.cat(p), t, w


class _Memory:
    """A torch tensor in the form the network's calls take (shape, dtype, address)."""

    def __init__(self, t, dtype):
        self.t, self.shape, self.dtype, self.ptr = t, tuple(t.shape), np.dtype(dtype), ctypes.c_void_p(t.data_ptr())


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "predict"):
        x, p, t, w = _net_inputs(case, seed)
        net = learned.WarmStartNet(0)
        net.set_params(_host(p))
        y = torch.empty(x.shape[:3] + (8,), device="cuda", dtype=torch.float32)
        torch.cuda.synchronize()
        return dict(kind=kind, net=net, x=_Memory(x, np.uint16), y=_Memory(y, np.float32), t=_Memory(t, np.float32),
                    w=_Memory(w, np.float32))
    f = _inputs(case, seed)
    nx, ny, sph = case["nx"], case["ny"], case["mesh"] == "sphere"
    given, mask = _given(case, f["coords"]), _host(f["mask"])
    if kind == "transport":
        m = ParametricMesh(nx, ny, given, sph)
        m.landmaskFromModelArray(mask)
        m.dirichletFromMask()
        t = DGTransport(m, case["dg"])
        t.settimesteppingscheme(case["scheme"])
        u, v, phi = _transport_inputs(case, seed)
        return dict(kind=kind, case=case, t=t, u=_host(u), v=_host(v), phi=_host(phi))
    if kind == "module":
        store = modules.ModelStore()
        d = modules.MEVPDynamics(store, case["cg"], 3 if case["cg"] == 1 else 6)
        zero = np.zeros(nx * ny)
        d.setData({"nx": nx, "ny": ny, ("longitude" if sph else "x"): None, ("latitude" if sph else "y"): None,
                   "coords": np.degrees(given) if sph else given, "mask": mask, "hice": _host(f["hice"]),
                   "cice": _host(f["cice"]), "u": zero, "v": zero})
        for key, n in ((modules.H_ICE, "hice"), (modules.C_ICE, "cice"), (modules.WIND_U, "uwind"),
                       (modules.WIND_V, "vwind"), (modules.OCEAN_U, "uocean"), (modules.OCEAN_V, "vocean"),
                       (modules.SSH, "ssh")):
            store[key] = _host(f[n])
        return dict(kind=kind, case=case, d=d, store=store, n=0)
    k = (BBMDynamicsKernel if kind == "bbm" else MEVPDynamicsKernel)(case["cg"], 3 if case["cg"] == 1 else 6)
    k.initialise(given, sph, mask, nx, ny)
    for n in ("hice", "cice", "uocean", "vocean", "ssh", "uwind", "vwind"):
        k.setData(n, _host(f[n]), 1)
    for n in ("u", "v") + (("avgU", "avgV") if kind == "bbm" else ()):
        k.set_cg(n, _host(f[n[-1].lower()]))
    if case["fp32"]:
        k.set_precision(1)
    return dict(kind=kind, case=case, k=k, n=0, storms=f["storms"])


def run(state):
    kind = state["kind"]
    if kind == "predict":
        state["net"].forward(state["x"], state["y"])
        return state["y"].t
    if kind == "train":
        loss, grad = state["net"].loss_grad(state["x"], state["t"], state["w"], want_grad=True)
        state["net"].adam(1e-3)
        return {"loss": np.float32(loss), "grad": grad}
    case = state["case"]
    if kind == "transport":
        t = state["t"]
        t.prepareAdvection(2, state["u"], state["v"])
        return t.run(case["dt"], state["phi"], case["steps"], case["limit"], case["limit"])
    state["n"] += 1
    if kind == "module":
        d, s = state["d"], state["store"]
        d.update(modules.TimestepTime((state["n"] - 1) * case["dt"], case["dt"]))
        return {"hice": s[modules.H_ICE], "cice": s[modules.C_ICE], "u": d.uice, "v": d.vice, "taux": d.taux,
                "tauy": d.tauy}
    k = state["k"]
    k.reset_dg0("hice")
    k.reset_dg0("cice")
    if case["mesh"] == "box":
        k.storm_wind(case["nx"] * case["dx"], (state["n"] - 1) * case["dt"], state["storms"])
    k.update(case["dt"])
    names = ("hice", "cice", "u", "v") + (("damage",) if kind == "bbm" else ())
    return {n: k.getDG0Data(n) for n in names}


def _transport_inputs(case, seed):
    g = _gen(seed)
    nx, ny, D = case["nx"], case["ny"], case["dg"]
    X, Y = _grid(2 * nx, 2 * ny, px=1, py=1)
    w = torch.sin(math.pi * X) * torch.sin(math.pi * Y)
    u, v = 0.3 * w * _waves(g, X, Y, top=2.0), 0.3 * w * _waves(g, X, Y, top=2.0)
    x, y = _grid(nx, ny, 0.5, 0.5)
    phi = torch.zeros((nx * ny, D), device="cuda", dtype=torch.float64)
    phi[:, 0] = 0.5 + 0.3 * _waves(g, x, y, top=3.0) + 0.05 * _uniform(g, nx * ny, -1, 1)
    if D > 1:
        phi[:, 1:] = 0.05 * torch.randn((nx * ny, D - 1), generator=g, device="cuda", dtype=torch.float64)
    return u, v, phi


def work(case):
    kind = case["kind"]
    ne = case["nx"] * case["ny"]
    if kind in ("train", "predict"):
        px = ne * case["batch"]
        conv = 2 * 9 * 32 * 32 * px
        if kind == "predict":
            return {"bytes": px * (64 + 32), "flops": 4 * conv}
        return {"bytes": px * (64 + 32 + 4), "flops": (4 + 3 + 4) * conv}  # forward, data gradient, weight gradient
    if kind == "transport":
        D = case["dg"]
        stages = {"rk1": 1, "rk2": 2, "rk3": 3}[case["scheme"]]
        per = {1: 60, 3: 350, 6: 1100}[D]  # cell term, four edge fluxes, inverse mass, per element and stage
        return {"bytes": 16 * ne * D + 16 * 4 * ne, "flops": case["steps"] * ne * (stages * per + 30 * D)}
    cg = case["cg"]
    D, S, N = (3, 3, 1) if cg == 1 else (6, 8, 4)
    state = 2 * 8 * ne * (2 * D + 3 * S) + 8 * ne * N * 2 * 2  # h, A, stress; u, v: read and written
    forcing = 8 * ne * 8
    geometry = 0 if case["mesh"] == "box" else 8 * 2 * ne
    # per element and subcycle: strain, rheology and projection at the Gauss points, weak
    # divergence, and the node update of the N nodes per element
    flops = {1: 350, 2: 1700}[cg] + (0 if kind != "bbm" else {1: 500, 2: 1400}[cg])
    if case["mesh"] != "box":
        flops = flops * 3 // 2
    return {"bytes": state + forcing + geometry, "flops": SUBCYCLES * ne * flops}


# ---------------------------------------------------------------- the same in plain torch, 64 bits
def _gauss(n):
    p, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (p + 1.0), 0.5 * w


def _psi(D, x, y, d=0):
    """The first D DG basis functions (d = 1, 2: their x and y derivatives) at points: [D, points]."""
    X, Y = np.asarray(x) - 0.5, np.asarray(y) - 0.5
    o, z, t = np.ones_like(X), np.zeros_like(X), 1.0 / 12.0
    if d == 0:
        b = [o, X, Y, X * X - t, Y * Y - t, X * Y, Y * (X * X - t), X * (Y * Y - t)]
    elif d == 1:
        b = [z, o, z, 2 * X, z, Y, 2 * X * Y, Y * Y - t]
    else:
        b = [z, z, o, z, 2 * Y, X, X * X - t, 2 * X * Y]
    return np.stack(b[:D])


def _phi(cg, x, y, d=0):
    """The CG basis (node jx + (cg+1) jy) at points: [nodes, points]."""
    def one(t, dd):
        t = np.asarray(t)
        if cg == 1:
            return [1 - t, t] if not dd else [-np.ones_like(t), np.ones_like(t)]
        if dd:
            return [4 * t - 3, 4 - 8 * t, 4 * t - 1]
        return [2 * (t - 0.5) * (t - 1), 4 * t * (1 - t), 2 * t * (t - 0.5)]
    a, b = one(x, d == 1), one(y, d == 2)
    return np.stack([a[i] * b[j] for j in range(cg + 1) for i in range(cg + 1)])


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda", dtype=torch.float64)


class _Rule:
    """G x G Gauss points of the unit square, x fastest."""

    def __init__(self, G):
        p, w = _gauss(G)
        self.x, self.y = np.tile(p, G), np.repeat(p, G)
        self.w = _t(np.tile(w, G) * np.repeat(w, G))


class _Exact:
    def __init__(self, case, f):
        self.nx, self.ny, self.sph = case["nx"], case["ny"], case["mesh"] == "sphere"
        nx, ny = self.nx, self.ny
        c = f["coords"].reshape(ny + 1, nx + 1, 2)
        self.vert = c
        self.c = [q.reshape(-1, 2) for q in (c[:-1, :-1], c[:-1, 1:], c[1:, :-1], c[1:, 1:])]
        self.ocean = f["mask"].reshape(ny, nx) == 1.0
        oc = torch.zeros((ny + 2, nx + 2), dtype=torch.bool, device="cuda")
        oc[1:-1, 1:-1] = self.ocean
        mid = oc[1:-1, 1:-1]
        # an ocean element next to land or the edge of the domain: bottom, right, top, left
        self.wall = [mid & ~oc[:-2, 1:-1], mid & ~oc[1:-1, 2:], mid & ~oc[2:, 1:-1], mid & ~oc[1:-1, :-2]]
        if case["kind"] == "transport":  # walls from the mask only: not at the edge of the domain
            self.wall[0][0], self.wall[1][:, -1], self.wall[2][-1], self.wall[3][:, 0] = 4 * (False,)
        self.iR = 1.0 / R_EARTH if self.sph else 1.0

    def geometry(self, R):
        """Map gradients x_xi, x_eta, y_xi, y_eta, J and the latitude at the points of R: [ne, Q]."""
        px, py, p = _t(_phi(1, R.x, R.y, 1)), _t(_phi(1, R.x, R.y, 2)), _t(_phi(1, R.x, R.y))
        C = torch.stack(self.c, dim=1)  # ne, 4, 2
        xxi, xeta, yxi, yeta = C[..., 0] @ px, C[..., 0] @ py, C[..., 1] @ px, C[..., 1] @ py
        lat = C[..., 1] @ p if self.sph else None
        return xxi, xeta, yxi, yeta, xxi * yeta - xeta * yxi, lat

    def inverse_mass(self, D, R, J, lat):
        B = _t(_psi(D, R.x, R.y))
        W = R.w * J * (torch.cos(lat) if self.sph else 1.0)
        P = torch.stack([B[i] * B[j] for i in range(D) for j in range(D)], dim=1)  # Q, D D
        return torch.linalg.inv((W @ P).reshape(-1, D, D))

    @staticmethod
    def solve(Mi, b):
        return (Mi * b[:, None, :]).sum(-1)

    # ---- CG nodes
    def local(self, cg, w):
        """The node values of every element: [ne, nodes]."""
        W = w.reshape(cg * self.ny + 1, cg * self.nx + 1)
        e = [W[j:j + cg * self.ny:cg, i:i + cg * self.nx:cg] for j in range(cg + 1) for i in range(cg + 1)]
        return torch.stack([q.reshape(-1) for q in e], dim=1)

    def add(self, cg, t):
        """The sum of the elements' contributions [ne, nodes] at the CG nodes."""
        W = torch.zeros((cg * self.ny + 1, cg * self.nx + 1), device="cuda", dtype=torch.float64)
        for j in range(cg + 1):
            for i in range(cg + 1):
                W[j:j + cg * self.ny:cg, i:i + cg * self.nx:cg] += t[:, i + (cg + 1) * j].reshape(self.ny, self.nx)
        return W.reshape(-1)

    def walls(self, cg):
        m = torch.zeros((cg * self.ny + 1, cg * self.nx + 1), dtype=torch.bool, device="cuda")
        for k in range(cg + 1):
            a = (slice(k, k + cg * self.ny, cg), slice(k, k + cg * self.nx, cg))
            m[0:cg * self.ny:cg, a[1]] |= self.wall[0]
            m[cg::cg, a[1]] |= self.wall[2]
            m[a[0], cg::cg] |= self.wall[1]
            m[a[0], 0:cg * self.nx:cg] |= self.wall[3]
        return m.reshape(-1)

    def to_dg(self, cg, D, w):
        G = {1: 1, 3: 2, 6: 3, 8: 3}[D]
        R = _Rule(G)
        *_, J, lat = self.geometry(R)
        val = self.local(cg, w) @ _t(_phi(cg, R.x, R.y))
        b = (val * R.w * J * (torch.cos(lat) if self.sph else 1.0)) @ _t(_psi(D, R.x, R.y)).T
        return self.solve(self.inverse_mass(D, R, J, lat), b)

    def to_cg(self, cg, c):
        p = np.linspace(0.0, 1.0, cg + 1)
        B = _psi(c.shape[1], np.tile(p, cg + 1), np.repeat(p, cg + 1))
        one = np.array([0.5, 0.5]) if cg == 1 else np.array([0.5, 1.0, 0.5])
        w = self.add(cg, (c @ _t(B)) * _t(np.tile(one, cg + 1) * np.repeat(one, cg + 1)))
        W = w.reshape(cg * self.ny + 1, -1)
        W[0] *= 2.0
        W[-1] *= 2.0
        W[:, 0] *= 2.0
        W[:, -1] *= 2.0
        return w

    # ---- transport
    def trace(self, D, c, side):
        """Restriction of [ny, nx, D] to a side, in the edge basis."""
        s = -0.5 if side in (0, 3) else 0.5
        a = (1, 2, 3, 4, 6, 7) if side in (1, 3) else (2, 1, 4, 3, 7, 6)  # normal, tangential, their squares, cubics
        if D == 1:
            return c
        if D == 3:
            return torch.stack([c[..., 0] + s * c[..., a[0]], c[..., a[1]]], dim=-1)
        o = [c[..., 0] + s * c[..., a[0]] + c[..., a[2]] / 6.0, c[..., a[1]] + s * c[..., 5], c[..., a[3]]]
        if D == 8:
            o[1] = o[1] + c[..., a[4]] / 6.0
            o[2] = o[2] + s * c[..., a[5]]
        return torch.stack(o, dim=-1)

    def advection(self, D, vx, vy):
        """The transport operator of the velocity (DG coefficients): phi -> dphi per unit time."""
        G = {1: 1, 3: 2, 6: 3, 8: 3}[D]
        nx, ny = self.nx, self.ny
        R = _Rule(G)
        xxi, xeta, yxi, yeta, J, lat = self.geometry(R)
        Mi = self.inverse_mass(D, R, J, lat) * self.iR
        B, Bx, By = (_t(_psi(D, R.x, R.y, d)) for d in (0, 1, 2))
        VX, VY = vx @ B, vy @ B
        fx, fy = R.w * (VX * yeta - VY * xeta), R.w * (VY * xxi - VX * yxi)  # against psi_xi, psi_eta
        oc = self.ocean.reshape(ny, nx, 1).double()
        ux, uy = vx.reshape(ny, nx, D), vy.reshape(ny, nx, D)
        V = self.vert
        ev, eh = V[1:] - V[:-1], V[:, 1:] - V[:, :-1]  # edges along y [ny, nx+1], along x [ny+1, nx]
        E = {1: 1, 3: 2, 6: 3, 8: 3}[D]
        nY = torch.zeros((ny, nx + 1, E), device="cuda", dtype=torch.float64)
        nX = torch.zeros((ny + 1, nx, E), device="cuda", dtype=torch.float64)
        for at, side in ((slice(0, nx), 3), (slice(1, nx + 1), 1)):
            t = ev[:, at]
            nY[:, at] += 0.5 * oc * (t[..., 1:] * self.trace(D, ux, side) - t[..., :1] * self.trace(D, uy, side))
        for at, side in ((slice(0, ny), 0), (slice(1, ny + 1), 2)):
            t = eh[at]
            nX[at] += 0.5 * oc * (t[..., :1] * self.trace(D, uy, side) - t[..., 1:] * self.trace(D, ux, side))
        wall = [w[..., None].double() for w in self.wall]
        nX[:-1] *= 1 + wall[0]
        nY[:, 1:] *= 1 + wall[1]
        nX[1:] *= 1 + wall[2]
        nY[:, :-1] *= 1 + wall[3]
        p, w1 = _gauss(G)
        T = np.asarray(p) - 0.5
        PE = _t(np.stack([np.ones_like(T), T, T * T - 1.0 / 12.0][:E]))
        gX, gY = nX @ PE, nY @ PE
        ends = [(p, 0 * p), (0 * p + 1, p), (p, 0 * p + 1), (0 * p, p)]
        PW = [_t(w1[:, None] * _psi(D, *e).T) for e in ends]
        both_y, both_x = oc[:, :-1] * oc[:, 1:], oc[:-1] * oc[1:]

        def op(phi):
            c = phi.reshape(ny, nx, D)
            ph = phi @ B
            out = ((fx * ph) @ Bx.T + (fy * ph) @ By.T).reshape(ny, nx, D) * oc
            tr = [self.trace(D, c, s) @ PE for s in range(4)]
            g = gY[:, 1:-1]
            flux = both_y * (g.clamp(min=0) * tr[1][:, :-1] + g.clamp(max=0) * tr[3][:, 1:])
            out[:, :-1] -= flux @ PW[1]
            out[:, 1:] += flux @ PW[3]
            g = gX[1:-1]
            flux = both_x * (g.clamp(min=0) * tr[2][:-1] + g.clamp(max=0) * tr[0][1:])
            out[:-1] -= flux @ PW[2]
            out[1:] += flux @ PW[0]
            for s, g in ((0, -gX[:-1]), (1, gY[:, 1:]), (2, gX[1:]), (3, -gY[:, :-1])):
                out -= (wall[s] * g.clamp(min=0) * tr[s]) @ PW[s]
            return self.solve(Mi, out.reshape(-1, D))
        return op

    @staticmethod
    def step(op, dt, phi, scheme="rk2"):
        if scheme == "rk1":
            return phi + dt * op(phi)
        if scheme == "rk2":
            k = dt * op(phi)
            return phi + 0.5 * (k + dt * op(phi + k))
        a = phi + dt * op(phi)
        b = 0.75 * phi + 0.25 * (a + dt * op(a))
        return phi / 3.0 + 2.0 / 3.0 * (b + dt * op(b))

    @staticmethod
    def limit(c, bound, upper):
        """LimitMax / LimitMin of the reference (the sign that LimitMin gives to a DG2 cell included)."""
        c = c.clone()
        D = c.shape[1]
        c[:, 0] = c[:, 0].clamp(max=bound) if upper else c[:, 0].clamp(min=bound)
        if D == 1:
            return c
        if D == 3:
            l0 = 2.0 * torch.maximum((c[:, 1] + c[:, 2]).abs(), (c[:, 1] - c[:, 2]).abs())
            room = bound - c[:, 0] if upper else c[:, 0] - bound
            cut = (l0 > 0) & (l0 > room)
        else:
            g = c @ _t(_psi(6, _Rule(3).x, _Rule(3).y))
            m = g.max(dim=1).values if upper else g.min(dim=1).values
            l0 = m - c[:, 0]
            room = bound - c[:, 0] if upper else c[:, 0] - bound
            cut = m > bound if upper else m < bound
        r = torch.where(cut, room / torch.where(cut, l0, torch.ones_like(l0)), torch.ones_like(l0))
        c[:, 1:] *= r[:, None]
        return c

    # ---- momentum
    def momentum(self, cg):
        self.cg, self.S = cg, 3 if cg == 1 else 8
        G = 2 if cg == 1 else 3
        R = self.R = _Rule(G)
        self.xxi, self.xeta, self.yxi, self.yeta, self.J, lat = self.geometry(R)
        self.cl = torch.cos(lat) if self.sph else torch.ones(1, device="cuda", dtype=torch.float64)
        self.sl = torch.sin(lat) if self.sph else None
        self.Mi = self.inverse_mass(self.S, R, self.J, lat)
        self.B = _t(_psi(self.S, R.x, R.y))
        self.F = [_t(_phi(cg, R.x, R.y, d)) for d in (0, 1, 2)]
        L = _Rule(1 if cg == 1 else 4)
        *_, J, la = self.geometry(L)
        self.lumped = self.add(cg, (J * L.w * (torch.cos(la) if self.sph else 1.0)) @ _t(_phi(cg, L.x, L.y)).T)
        self.wallnode = self.walls(cg)
        self.sea = self.ocean.reshape(-1, 1)

    def strain(self, u, v, old):
        def grads(w):
            l = self.local(self.cg, w)
            a, b = l @ self.F[1], l @ self.F[2]
            gx = (a * self.yeta - b * self.yxi) * self.R.w * self.iR
            gy = (b * self.xxi - a * self.xeta) * self.R.w * self.cl * self.iR
            return gx, gy, l @ self.F[0]
        ux, uy, uq = grads(u)
        vx, vy, vq = grads(v)
        g11, g22, g12 = ux, vy, 0.5 * (vx + uy)
        if self.sph:
            js = self.J * self.R.w * self.sl * self.iR
            g11, g12 = g11 - js * vq, g12 + 0.5 * js * uq
        return [torch.where(self.sea, self.solve(self.Mi, g @ self.B.T), o) for g, o in zip((g11, g12, g22), old)]

    def project(self, r):
        return self.solve(self.Mi, (r * self.J * self.R.w) @ self.B.T)

    def divergence(self, s):
        s11, s12, s22 = (c @ self.B * self.sea for c in s)
        a, b = self.yeta * self.R.w * self.iR, self.yxi * self.R.w * self.iR
        c, d = self.xxi * self.R.w * self.cl * self.iR, self.xeta * self.R.w * self.cl * self.iR

        def weak(p, q, extra):
            t = (a * p - d * q) @ self.F[1].T + (c * q - b * p) @ self.F[2].T
            return t + extra @ self.F[0].T if extra is not None else t
        js = self.J * self.R.w * self.sl * self.iR if self.sph else None
        dx = -self.add(self.cg, weak(s11, s12, js * s12 if self.sph else None))
        dy = -self.add(self.cg, weak(s12, s22, -js * s11 if self.sph else None))
        dx[self.wallnode] = 0.0
        dy[self.wallnode] = 0.0
        return dx, dy

    def ssh_gradient(self, ssh):
        nx, ny = self.nx, self.ny
        R = self.R
        val = self.local(1, self.to_cg(1, ssh.reshape(-1, 1))) @ _t(_phi(1, R.x, R.y))
        Fx, Fy = _t(_phi(1, R.x, R.y, 1)), _t(_phi(1, R.x, R.y, 2))
        a, b = self.yeta * R.w * self.iR, self.yxi * R.w * self.iR
        c, d = self.xxi * R.w * self.cl * self.iR, self.xeta * R.w * self.cl * self.iR
        L = _Rule(2)
        *_, J, la = self.geometry(L)
        ML = self.add(1, (J * L.w * (torch.cos(la) if self.sph else 1.0)) @ _t(_phi(1, L.x, L.y)).T)
        out = []
        for t in ((val * a) @ Fx.T - (val * b) @ Fy.T, (val * c) @ Fy.T - (val * d) @ Fx.T):
            g = (-self.add(1, t) / ML).reshape(ny + 1, nx + 1)
            g[0, 1:-1], g[-1, 1:-1] = g[1, 1:-1].clone(), g[-2, 1:-1].clone()
            g[1:-1, 0], g[1:-1, -1] = g[1:-1, 1].clone(), g[1:-1, -2].clone()
            g[0, 0], g[0, -1], g[-1, 0], g[-1, -1] = (g[1, 1].clone(), g[1, -2].clone(), g[-2, 1].clone(),
                                                      g[-2, -2].clone())
            if self.cg == 2:
                h = torch.empty((2 * ny + 1, 2 * nx + 1), device="cuda", dtype=torch.float64)
                h[::2, ::2] = g
                h[::2, 1::2] = 0.5 * (g[:, 1:] + g[:, :-1])
                h[1::2] = 0.5 * (h[2::2] + h[:-2:2])
                g = h
            out.append(g.reshape(-1))
        return out


P = dict(rho=900.0, Fa=1.2e-3 * 1.3, Fo=5.5e-3 * 1026.0, fc=1.45842e-4, g=9.81, Pstar=27500.0, dmin=2e-9, alpha=1500.0,
         beta=1500.0)
BBM = dict(comp=-20.0, nu=1.0 / 3.0, young=5.96e8, P0=10e3, t0=1e7, ex=5.0, ec=1.5, tan=0.7, strength=1e10, clab=2e6)


def _exact_step(case, f):
    """One model step from the inputs f: cell means, and the ice-ocean stress for the module."""
    X = _Exact(case, f)
    kind, cg, dt = case["kind"], case["cg"], case["dt"]
    D = 3 if cg == 1 else 6
    X.momentum(cg)
    S, ne = X.S, case["nx"] * case["ny"]
    zero = torch.zeros((ne, 1), device="cuda", dtype=torch.float64)

    def dg0(w, n):
        return torch.cat([w.reshape(-1, 1)] + [zero] * (n - 1), dim=1)
    if kind == "module":
        u = v = torch.zeros_like(X.lumped)
    else:
        u, v = f["u"], f["v"]
    uw, vw = f["uwind"], f["vwind"]
    if case["mesh"] == "box" and kind != "module":
        x, y = _grid(case["nx"], case["ny"])
        x, y = x * case["nx"] * case["dx"], y * (case["nx"] * case["dx"])  # both axes of the wind span L
        uw, vw = torch.zeros_like(x), torch.zeros_like(x)
        L, a = case["nx"] * case["dx"], 72.0 / 180.0 * math.pi
        for ox, oy, vm in f["storms"]:
            xp, yp = x - 0.5 * L - ox, y - 0.5 * L - oy
            sc = 1e-5 * torch.exp(-1e-5 * torch.hypot(xp, yp))
            uw = uw - sc * vm * (math.cos(a) * xp + math.sin(a) * yp)
            vw = vw - sc * vm * (-math.sin(a) * xp + math.cos(a) * yp)
    ua, va, uo, vo = (X.to_cg(cg, w.reshape(-1, 1)) for w in (uw, vw, f["uocean"], f["vocean"]))
    op = X.advection(D, X.to_dg(cg, D, u), X.to_dg(cg, D, v))
    A, h = X.step(op, dt, dg0(f["cice"], D)), X.step(op, dt, dg0(f["hice"], D))
    A = X.limit(X.limit(A, 1.0, True), 0.0, False)
    h = X.limit(h, 0.0, False)
    H, C = X.to_cg(cg, h).clamp(min=1e-4), X.to_cg(cg, A).clamp(min=1e-4, max=1.0)
    gx, gy = X.ssh_gradient(f["ssh"])
    Bd = _t(_psi(D, X.R.x, X.R.y))
    hg, ag = (h @ Bd).clamp(min=0.0), (A @ Bd).clamp(min=0.0, max=1.0)
    sig = [torch.zeros((ne, S), device="cuda", dtype=torch.float64) for _ in range(3)]
    eps = [torch.zeros_like(q) for q in sig]
    ML, rho = X.lumped, P["rho"]
    wind = torch.hypot(ua, va)
    if kind == "bbm":
        dmg = X.limit(X.limit(X.step(op, dt, dg0(torch.ones(ne, device="cuda", dtype=torch.float64), D)), 1.0, True),
                      1e-12, False)
        a, b, c, d = X.c[0], X.c[1], X.c[3], X.c[2]

        def sq(p, q):
            return ((p - q) ** 2).sum(-1)
        k = sq(b, c) + sq(a, d) - sq(a, b) - sq(d, c)
        hE = torch.sqrt(0.25 * torch.sqrt(4 * sq(a, c) * sq(b, d) - k * k)).reshape(-1, 1)
        Md = X.inverse_mass(D, X.R, X.J, None)
        sub, nu = dt / SUBCYCLES, BBM["nu"]
        scale, expC = torch.sqrt(0.1 / hE), torch.exp(BBM["comp"] * (1 - ag))
        Pmax = BBM["P0"] * hg ** (BBM["ec"] + 1) * expC
        for _ in range(SUBCYCLES):
            eps = X.strain(u, v, eps)
            e11, e12, e22 = (e @ X.B for e in eps)
            s11, s12, s22 = (q @ X.B for q in sig)
            dg = (dmg @ Bd).clamp(min=1e-12, max=1.0)
            tv = BBM["t0"] * (dg * expC) ** (BBM["ex"] - 1)
            sn = 0.5 * (s11 + s22)
            tilde = torch.where(sn < 0, (-Pmax / sn).clamp(max=1.0), torch.zeros_like(sn))
            mult = tv / (tv + (1 - tilde) * sub)
            el = hg * BBM["young"] * dg * expC
            K = sub * el / (1 - nu * nu)
            s11, s22, s12 = ((s11 + K * (e11 + nu * e22)) * mult, (s22 + K * (nu * e11 + e22)) * mult,
                             (s12 + K * e12 * (1 - nu)) * mult)
            sn, tau = 0.5 * (s11 + s22), torch.hypot(0.5 * (s11 - s22), s12)
            mc, cs = tau + BBM["tan"] * sn, BBM["strength"] * scale * hg
            crit = torch.where(mc > 0, BBM["clab"] * scale * hg / mc, torch.ones_like(mc))
            crit = torch.where(sn < -cs, -cs / sn, crit).clamp(max=1.0)
            cut = 1 - (1 - crit) * sub / (hE * math.sqrt(2 * (1 + nu) * rho) / torch.sqrt(el))
            sig = [X.project(q * cut) for q in (s11, s12, s22)]
            dmg = X.solve(Md, (dg * cut * X.J * X.R.w) @ Bd.T)
            dx, dy = X.divergence(sig)
            m = sub / (rho * H)
            co = C * P["Fo"] * torch.hypot(uo - u, vo - v)
            al, be = 1 + m * co, sub * P["fc"]
            X1 = dx / ML - rho * H * P["g"] * gx + C * P["Fa"] * wind * ua + co * uo
            Y1 = dy / ML - rho * H * P["g"] * gy + C * P["Fa"] * wind * va + co * vo
            u, v = ((al * u + be * v + m * (al * X1 + be * Y1)) / (al * al + be * be),
                    (al * v - be * u + m * (al * Y1 + be * X1)) / (al * al + be * be))
            u, v = u.masked_fill(X.wallnode, 0.0), v.masked_fill(X.wallnode, 0.0)
    else:
        u0, v0, c1 = u, v, rho * H / dt
        Pg = P["Pstar"] * hg * torch.exp(-20.0 * (1.0 - ag))
        for _ in range(SUBCYCLES):
            eps = X.strain(u, v, eps)
            e11, e12, e22 = (e @ X.B for e in eps)
            delta = torch.sqrt(P["dmin"] ** 2 + 1.25 * (e11 * e11 + e22 * e22) + 1.5 * e11 * e22 + e12 * e12)
            z = Pg / (8.0 * delta)
            r = (z * (5 * e11 + 3 * e22) - 0.5 * Pg, 2 * z * e12, z * (5 * e22 + 3 * e11) - 0.5 * Pg)
            sig = [(1 - 1 / P["alpha"]) * q + X.project(t) / P["alpha"] for q, t in zip(sig, r)]
            dx, dy = X.divergence(sig)
            drag = C * P["Fo"] * torch.hypot(uo - u, v - vo)
            den = c1 * (1 + P["beta"]) + drag
            u, v = ((c1 * (P["beta"] * u + u0) + C * P["Fa"] * wind * ua + drag * uo - rho * H * P["fc"] * u
                     - rho * H * P["g"] * gx + dx / ML) / den,
                    (c1 * (P["beta"] * v + v0) + C * P["Fa"] * wind * va + drag * vo + rho * H * P["fc"] * v
                     - rho * H * P["g"] * gy + dy / ML) / den)
            u, v = u.masked_fill(X.wallnode, 0.0), v.masked_fill(X.wallnode, 0.0)
    out = {"hice": h[:, 0], "cice": A[:, 0], "u": X.to_dg(cg, D, u)[:, 0], "v": X.to_dg(cg, D, v)[:, 0]}
    if kind == "bbm":
        out["damage"] = dmg[:, 0]
    if kind == "module":
        s = P["Fo"] * torch.hypot(u - uo, v - vo)
        out["taux"], out["tauy"] = X.to_dg(cg, D, s * (u - uo))[:, 0], X.to_dg(cg, D, s * (v - vo))[:, 0]
    return out


def _exact_net(case, seed):
    x, p, t, w = _net_inputs(case, seed)
    n, ny, nx = x.shape[:3]
    params, at = [], 0
    for _ in range(4):
        # the kernels multiply bfloat16 copies of the weights
        W = p[at:at + 9216].to(torch.bfloat16).double().reshape(32, 32, 3, 3).requires_grad_(True)
        b = p[at + 9216:at + 9248].double().requires_grad_(True)
        params += [W, b]
        at += 9248
    a = x.double()
    for layer in range(4):
        W, b = params[2 * layer], params[2 * layer + 1]
        pad = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        out = b.expand(n * ny * nx, 32)
        for ky in range(3):
            for kx in range(3):
                out = out + pad[:, ky:ky + ny, kx:kx + nx].reshape(-1, 32) @ W[:, :, ky, kx].T
        a = out.reshape(n, ny, nx, 32)
        if layer < 3:
            a = a.clamp(min=0.0)
    y = a[..., :8]
    if case["kind"] == "predict":
        return y.detach()
    loss = (w.double()[..., None] * (y - t.double()) ** 2).sum() / (8 * n * ny * nx)
    loss.backward()
    return {"loss": loss.detach(), "grad": torch.cat([q.grad.reshape(-1) for q in params])}


def exact(case, seed):
    if case["kind"] in ("train", "predict"):
        return _exact_net(case, seed)
    f = _inputs(case, seed)
    if case["kind"] == "transport":
        u, v, phi = _transport_inputs(case, seed)
        X = _Exact(case, f)
        D = case["dg"]
        op = X.advection(D, X.to_dg(2, D, u), X.to_dg(2, D, v))
        for _ in range(case["steps"]):
            phi = X.step(op, case["dt"], phi, case["scheme"])
            if case["limit"]:
                phi = X.limit(X.limit(phi, 1.0, True), 0.0, False)
        return phi
    return _exact_step(case, f)
