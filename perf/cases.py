"""Timed workloads of the framework: what a flow solver's program has it do in
a run, through the public entry points.

Families (the `path` of a case) and what they stand for:

  solve    the pressure solve of a constant-density run: operator set up once,
           one DeviceSolve.solve per step from a zero guess (rcvg 1e-10), the
           mean removed from the result as shift_p does
  host     the same solve as an existing Fortran program calls it: host arrays
           through NgapStr, copies included
  twophase setup + solve of a density-ratio-1000 operator, as a two-phase run
           does every step
  step     one whole device-resident projection step of a two-phase run:
           operator from face densities, setup, divergence, right-hand side,
           solve, shift_p, pressure gradient, velocity correction
  implicit the nonsymmetric velocity solve (flexible GMRES)
  fourier  the FFT direct solve on a periodic uniform grid
  uns      hypre_uns: PCG with algebraic multigrid around solid bodies in a
           duct with an outflow (p = 0) at its end
  forward  the U-Net correction of a residual
  train    forward and backward pass of the U-Net, gradients out
  layer    one 3x3x3 BF16 layer: forward, data gradient, weight gradient

Grids run from 32 cells a side, where launches and latency count, to 256^3,
the size of the benchmark's solve; odd and ragged sizes wherever the path
takes them.
"""
import ctypes as C
import math

import numpy as np
import torch

from nga2_amd import incomp, unet
from nga2_amd._lib import GMRES_PFMG, PCG_PFMG
from nga2_amd.config import Config, tanh_stretched, uniform
from nga2_amd.fourier import DeviceFourier
from nga2_amd.linsol import DeviceSolve, NgapStr
from nga2_amd.proj import DeviceProjection
from nga2_amd.uns import PCG_AMG, DeviceUns

RCVG = 1e-10
MAXIT = 300
F64 = torch.float64

# (level, input, output channels) of the network's MFMA layers
LAYERS = [(1, 32, 32), (2, 32, 64), (2, 64, 64), (3, 64, 64), (2, 128, 64), (1, 96, 32), (0, 64, 32)]


def listed():
    return [
        # the benchmark's solve: channel box, walls in y, stretched, 256^3
        dict(name="channel_256_mixed", path="solve", nx=256, ny=256, nz=256, walls="y", stretch=2.0, mixed=1),
        # a two-phase step's setup + solve at the same size
        dict(name="twophase_256_mixed", path="twophase", nx=256, ny=256, nz=256, spheres=50, mixed=1),
        # a whole projection step of a medium run in the reference's precision
        dict(name="step_128_fp64", path="step", nx=128, ny=128, nz=128, spheres=30, mixed=0),
        # a small periodic box: launches and latency
        dict(name="periodic_64_fp64", path="solve", nx=64, ny=64, nz=64, walls="", stretch=0.0, mixed=0),
        # a closed box with odd sizes, from a host program
        dict(name="host_odd_mixed", path="host", nx=131, ny=99, nz=75, walls="xyz", stretch=0.0, mixed=1),
        # implicit velocity solve of a channel run
        dict(name="implicit_128_mixed", path="implicit", nx=128, ny=128, nz=128, walls="y", stretch=2.0, mixed=1),
        # FFT solves: the benchmark's size and a small ragged one
        dict(name="fourier_256", path="fourier", nx=256, ny=256, nz=256),
        dict(name="fourier_ragged", path="fourier", nx=90, ny=75, nz=64),
        # flow around solid bodies
        dict(name="uns_96_fp64", path="uns", nx=96, ny=96, nz=96, walls="x", spheres=27, mixed=0),
        # the learned stage: one correction, one training pass, its widest layer
        dict(name="unet_forward_128", path="forward", nx=128, ny=128, nz=128),
        dict(name="unet_train_128x64x64", path="train", nx=128, ny=64, nz=64),
        dict(name="unet_layer_128", path="layer", nx=128, ny=128, nz=128, cin=64, cout=32),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        c = _draw(rng)
        if c not in known:
            return c


def _draw(rng):
    path = rng.choice(["solve", "solve", "host", "twophase", "step", "implicit", "fourier", "fourier", "uns",
                       "forward", "train", "layer"])
    even = [32, 40, 48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256]  # periodic lengths the cycle can halve
    if path in ("solve", "implicit"):
        mixed = rng.randint(0, 1)
        walls = rng.choice(["", "y", "xyz", "xy"]) if path == "solve" else rng.choice(["", "y"])
        most = 192 ** 3 if mixed and path == "solve" else 128 ** 3
        while True:
            n = [_log_size(rng, 32, 256) if a in walls else rng.choice(even) for a in "xyz"]
            if n[0] * n[1] * n[2] <= most:
                break
        return dict(path=path, nx=n[0], ny=n[1], nz=n[2], walls=walls,
                    stretch=rng.choice([0.0, 1.0, 2.0]) if walls == "y" else 0.0, mixed=mixed)
    if path == "host":
        while True:
            n = [_log_size(rng, 32, 160) for _ in range(3)]
            if n[0] * n[1] * n[2] <= 128 ** 3:
                break
        return dict(path=path, nx=n[0], ny=n[1], nz=n[2], walls="xyz", stretch=0.0, mixed=rng.randint(0, 1))
    if path in ("twophase", "step"):
        n = rng.choice([48, 64, 96, 112, 128, 160] if path == "twophase" else [48, 64, 96, 112])
        return dict(path=path, nx=n, ny=n, nz=n, spheres=rng.randint(8, 50), mixed=rng.randint(0, 1))
    if path == "fourier":
        while True:
            n = [_log_size(rng, 16, 256) for _ in range(3)]
            if n[0] * n[1] * n[2] <= 200 ** 3:
                break
        return dict(path=path, nx=n[0], ny=n[1], nz=n[2])
    if path == "uns":
        n = _log_size(rng, 24, 96)
        return dict(path=path, nx=n, ny=n, nz=n, walls="x", spheres=rng.choice([8, 27, 64]), mixed=rng.randint(0, 1))
    if path == "layer":
        lvl, cin, cout = rng.choice(LAYERS)
        return dict(path=path, nx=16 * rng.randint(1, 8), ny=4 * rng.randint(1, max(4, 32 >> lvl)),
                    nz=4 * rng.randint(1, max(4, 32 >> lvl)), cin=cin, cout=cout)
    while True:
        n = [128 * rng.randint(1, 3), 32 * rng.randint(1, 8), 32 * rng.randint(1, 8)]
        if n[0] * n[1] * n[2] <= (128 ** 3 if path == "forward" else 128 * 64 * 64):
            return dict(path=path, nx=n[0], ny=n[1], nz=n[2])


# ------------------------------------------------------------------ grids, fields, operators (torch, FP64)

def _vertices(case):
    """Vertices of the box [0, n/nmax] per direction (cubic cells), y stretched on request."""
    n = (case["nx"], case["ny"], case["nz"])
    h = 1.0 / max(n)
    v = [uniform(m, m * h) for m in n]
    if case.get("stretch", 0.0) > 0.0:
        v[1] = tanh_stretched(n[1], 1.0, case["stretch"])
    return v


def _periodic(case):
    return tuple(a not in case.get("walls", "") for a in "xyz")


def _config(case):
    x, y, z = _vertices(case)
    px, py, pz = _periodic(case)
    return Config(x, y, z, no=1, xper=px, yper=py, zper=pz, name="perf")


def _spacing(case):
    return [torch.from_numpy(np.diff(v)).cuda() for v in _vertices(case)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, dtype=F64, device="cuda")


# interior fields are [k, j, i]; axis a of x, y, z is tensor dimension 2 - a
def _roll(t, a, s):
    return torch.roll(t, s, 2 - a)


def _shape3(v, a):
    s = [1, 1, 1]
    s[2 - a] = -1
    return v.reshape(s)


def _faces(case, rho=None, fluid=None):
    """Face couplings area / distance (/ density) between each cell and its
    lower neighbour, one [k, j, i] tensor per direction; 0 across walls."""
    d = _spacing(case)
    per = _periodic(case)
    out = []
    for a in range(3):
        area = torch.ones((), dtype=F64, device="cuda")
        for b in range(3):
            if b != a:
                area = area * _shape3(d[b], b)
        dm = 0.5 * (d[a] + torch.roll(d[a], 1))
        inv = 1.0 / dm
        if not per[a]:
            inv[0] = 0.0
        f = (_shape3(inv, a) * area).expand(case["nz"], case["ny"], case["nx"]).clone()
        if rho is not None:
            f /= 0.5 * (rho + _roll(rho, a, 1))
        if fluid is not None:
            f *= fluid * _roll(fluid, a, 1)
        out.append(f)
    return out


def _outflow(case, fluid):
    """What p = 0 on the last x face adds to the diagonal: area over half a cell."""
    d = _spacing(case)
    out = torch.zeros_like(fluid)
    out[:, :, -1] = fluid[:, :, -1] * (d[2][:, None] * d[1][None, :] * 2.0 / d[0][-1])
    return out


def _operator(faces, outflow=None):
    """The ghosted 7-entry array (centre, +x, -x, +y, -y, +z, -z) of -vol div grad."""
    nz, ny, nx = faces[0].shape
    opr = torch.zeros((nz + 2, ny + 2, nx + 2, 7), dtype=F64, device="cuda")
    o = opr[1:-1, 1:-1, 1:-1]
    for a in range(3):
        up = _roll(faces[a], a, -1)
        o[..., 0] += faces[a] + up
        o[..., 1 + 2 * a] = -up
        o[..., 2 + 2 * a] = -faces[a]
    if outflow is not None:
        o[..., 0] += outflow
    return opr.reshape(-1)


def _apply(faces, x, outflow=None):
    y = torch.zeros_like(x) if outflow is None else outflow * x
    for a in range(3):
        flux = faces[a] * (x - _roll(x, a, 1))  # through the lower face
        y += flux - _roll(flux, a, -1)
    return y


def _ghosted(t, per=(False, False, False)):
    g = torch.zeros([n + 2 for n in t.shape], dtype=t.dtype, device=t.device)
    g[1:-1, 1:-1, 1:-1] = t
    for a in range(3):
        if per[a]:
            dim = 2 - a
            g.select(dim, 0).copy_(g.select(dim, -2))
            g.select(dim, -1).copy_(g.select(dim, 1))
    return g.reshape(-1)


def _volume(case):
    d = _spacing(case)
    return _shape3(d[0], 0) * _shape3(d[1], 1) * _shape3(d[2], 2)


def _source(case, gen):
    """vol times the divergence of Gaussian face velocities, 0 on walls: sums to zero."""
    per = _periodic(case)
    d = _spacing(case)
    b = torch.zeros((case["nz"], case["ny"], case["nx"]), dtype=F64, device="cuda")
    for a in range(3):
        area = torch.ones((), dtype=F64, device="cuda")
        for e in range(3):
            if e != a:
                area = area * _shape3(d[e], e)
        u = _randn(gen, *b.shape) * area
        if not per[a]:
            u.select(2 - a, 0).zero_()
        b -= _roll(u, a, -1) - u
    return b


def _spheres(case, gen):
    """Liquid fraction of spheres in the periodic unit cube, one cell wide interfaces."""
    n = case["nx"]
    c = torch.rand(case["spheres"], 3, generator=gen, dtype=F64, device="cuda").cpu().numpy()
    r = 0.05 + 0.10 * torch.rand(case["spheres"], generator=gen, dtype=F64, device="cuda").cpu().numpy()
    xc = (torch.arange(n, dtype=F64, device="cuda") + 0.5) / n
    s = torch.full((n, n, n), -1.0, dtype=F64, device="cuda")
    for q in range(case["spheres"]):
        e = [(torch.remainder(xc - c[q, a] + 0.5, 1.0) - 0.5) ** 2 for a in range(3)]
        dist = (_shape3(e[0], 0) + _shape3(e[1], 1) + _shape3(e[2], 2)).sqrt_()
        torch.maximum(s, r[q] - dist, out=s)
    return (0.5 + s * n).clamp_(0.0, 1.0)


def _solids(case, gen):
    """Fluid indicator around a jittered lattice of solid spheres that do not touch."""
    n = case["nx"]
    m = round(case["spheres"] ** (1.0 / 3.0))
    jit = torch.rand(case["spheres"], 4, generator=gen, dtype=F64, device="cuda").cpu().numpy()
    xc = (torch.arange(n, dtype=F64, device="cuda") + 0.5) / n
    fluid = torch.ones((n, n, n), dtype=F64, device="cuda")
    for q in range(case["spheres"]):
        at = (q % m, (q // m) % m, q // (m * m))
        e = []
        for a in range(3):
            c = (at[a] + 0.4 + 0.2 * jit[q, a]) / m
            e.append((torch.remainder(xc - c + 0.5, 1.0) - 0.5) ** 2)
        r = (0.18 + 0.12 * jit[q, 3]) / m
        fluid[_shape3(e[0], 0) + _shape3(e[1], 1) + _shape3(e[2], 2) < r * r] = 0.0
    return fluid


def _convection(case, gen):
    """rho + dt/2 (convection - viscosity) per unit volume with Gaussian face
    velocities (|u|max 1, CFL 1, viscosity 0.02): the 7 ghosted coefficients
    and the interior ones [k, j, i, 7]."""
    d = _spacing(case)
    per = _periodic(case)
    dt = min(float(v.min()) for v in d)
    shape = (case["nz"], case["ny"], case["nx"])
    u = [_randn(gen, *shape) for _ in range(3)]
    top = max(float(v.abs().max()) for v in u)
    opr = torch.zeros([n + 2 for n in shape] + [7], dtype=F64, device="cuda")
    o = opr[1:-1, 1:-1, 1:-1]
    o[..., 0] = 1.0
    for a in range(3):
        uf = u[a] / top
        dm = 0.5 * (d[a] + torch.roll(d[a], 1))
        g = 0.02 / dm
        if not per[a]:
            uf.select(2 - a, 0).zero_()
            g[0] = 0.0
        inv = _shape3(1.0 / d[a], a)
        g = _shape3(g, a)
        gup = _roll(g, a, -1)
        uup = _roll(uf, a, -1)
        o[..., 0] += 0.5 * dt * inv * (0.5 * uup - 0.5 * uf + g + gup)
        o[..., 1 + 2 * a] = 0.5 * dt * inv * (0.5 * uup - gup)
        o[..., 2 + 2 * a] = 0.5 * dt * inv * (-0.5 * uf - g)
    return opr.reshape(-1)


def _unet_weights(gen):
    w = {}
    for name, _lvl, cin, cout, kind in unet.LAYERS:
        taps = 1 if kind == "1x1" else 27
        std = math.sqrt((1.0 if kind == "1x1" else 2.0) / (taps * cin))
        w[name] = (torch.randn(taps * cin * cout, generator=gen, device="cuda") * std).cpu().numpy()
    return w


def _layer_inputs(case, gen):
    v = case["nx"] * case["ny"] * case["nz"]
    x = torch.relu(torch.randn(v, case["cin"], generator=gen, device="cuda")).to(torch.bfloat16)
    w = (torch.randn(27, case["cout"], case["cin"], generator=gen, device="cuda")
         * math.sqrt(2.0 / (27 * case["cin"]))).to(torch.bfloat16)
    g = torch.randn(v, case["cout"], generator=gen, device="cuda").to(torch.bfloat16)
    return x, w, g


class _Held:
    """A handle that gives its device memory back with the state."""

    def __init__(self, obj):
        self.obj = obj

    def __del__(self):
        try:
            (self.obj.close if hasattr(self.obj, "close") else self.obj.destroy)()
        except Exception:
            pass


def _inputs(case, seed):
    """The device inputs of a case, from the seed alone."""
    torch.zeros(1, device="cuda")
    gen = _gen(seed)
    path = case["path"]
    if path in ("solve", "host", "fourier"):
        return dict(faces=_faces(case), b=_source(case, gen))
    if path in ("twophase", "step"):
        rho = 1.0 + 999.0 * _spheres(case, gen)
        if path == "twophase":
            return dict(rho=rho, faces=_faces(case, rho), b=_source(case, gen))
        return dict(rho=rho, u=[_randn(gen, *rho.shape) for _ in range(3)])
    if path == "implicit":
        return dict(opr=_convection(case, gen), b=_randn(gen, case["nz"], case["ny"], case["nx"]))
    if path == "uns":
        fluid = _solids(case, gen)
        return dict(faces=_faces(case, fluid=fluid), outflow=_outflow(case, fluid), b=_randn(gen, *fluid.shape) * fluid)
    if path == "layer":
        return dict(zip(("x", "w", "g"), _layer_inputs(case, gen)))
    r = torch.randn(case["nz"], case["ny"], case["nx"], generator=gen, device="cuda")
    t = r  # the target of a training pass: the residual's smooth part
    for _ in range(4):
        for a in range(3):
            t = (t + _roll(t, a, 1) + _roll(t, a, -1)) / 3.0
    return dict(w=_unet_weights(gen), r=r.reshape(-1), target=(t / t.std()).reshape(-1))


def prepare(case, seed):
    path = case["path"]
    q = _inputs(case, seed)
    st = dict(case=case)
    if path in ("solve", "twophase", "implicit"):
        cfg = _config(case)
        ds = DeviceSolve(cfg, method=GMRES_PFMG if path == "implicit" else PCG_PFMG)
        st["ds"] = ds
        st["opr"] = q["opr"] if path == "implicit" else _operator(q["faces"])
        st["rhs"] = _ghosted(q["b"])
        st["sol"] = torch.zeros_like(st["rhs"])
        if path != "implicit":
            w = _volume(case)
            st["weight"] = _ghosted((w / w.sum()).expand_as(q["b"]).contiguous())
        if path != "twophase":
            ds.setup(st["opr"], maxit=MAXIT, rcvg=RCVG, precision=case["mixed"])
            del st["opr"]
    elif path == "host":
        cfg = _config(case)
        ps = NgapStr(cfg, "Pressure", PCG_PFMG, 7)
        ps.stc[:] = incomp.STC7
        ps.maxit, ps.rcvg, ps.precision = MAXIT, RCVG, case["mixed"]
        ps.opr = _operator(q["faces"]).cpu().numpy().reshape((7,) + cfg.shape, order="F")
        ps.init()
        ps.setup()
        ps.rhs[...] = _ghosted(q["b"]).cpu().numpy().reshape(cfg.shape, order="F")
        w = _volume(case)
        st["weight"] = _ghosted((w / w.sum()).expand_as(q["b"]).contiguous()).cpu().numpy()
        st["ps"] = ps
    elif path == "step":
        cfg = _config(case)
        per = (True, True, True)
        st["proj"] = DeviceProjection(incomp.Metrics(cfg))
        st["ds"] = DeviceSolve(cfg)
        st["u0"] = [_ghosted(u, per) for u in q["u"]]
        st["faces"] = tuple(_ghosted(0.5 * (q["rho"] + _roll(q["rho"], a, 1)), per) for a in range(3))
        z = torch.zeros_like(st["u0"][0])
        st.update(u=[z.clone() for _ in range(3)], g=[z.clone() for _ in range(3)], div=z.clone(), rhs=z.clone(),
                  sol=z.clone(), P=z.clone(), opr=torch.zeros(7 * z.numel(), dtype=F64, device="cuda"))
    elif path == "fourier":
        st["f"] = DeviceFourier(_config(case))
        st["held"] = _Held(st["f"])
        st["f"].setup(_operator(q["faces"]))
        st["rhs"] = _ghosted(q["b"])
        st["sol"] = torch.zeros_like(st["rhs"])
    elif path == "uns":
        cfg = _config(case)
        opr = _operator(q["faces"], q["outflow"]).cpu().numpy().reshape((7,) + cfg.shape, order="F")
        st["s"] = DeviceUns(cfg, opr, method=PCG_AMG, maxit=MAXIT, rcvg=RCVG, precision=case["mixed"])
        st["held"] = _Held(st["s"])
        st["rhs"] = _ghosted(q["b"])
        st["sol"] = torch.zeros_like(st["rhs"])
    elif path == "layer":
        L = unet.lib()
        cin, cout = case["cin"], case["cout"]
        dims = (case["nx"], case["ny"], case["nz"])
        v = dims[0] * dims[1] * dims[2]
        parts = L.ngapnet_wgrad_parts(*dims, cin, cout)
        st.update(q, y=torch.empty(v, cout, dtype=torch.bfloat16, device="cuda"),
                  wd=torch.empty(27, cin, cout, dtype=torch.bfloat16, device="cuda"),
                  dx=torch.empty(v, cin, device="cuda"), dw=torch.empty(27, cout, cin, device="cuda"),
                  part=torch.empty(parts * 27 * cin * cout, device="cuda"))
    else:
        net = unet.UNet((case["nx"], case["ny"], case["nz"]))
        net.set_weights(q["w"])
        st.update(net=net, held=_Held(net), r=q["r"], target=q["target"])
    return st


def _interior(case, flat):
    return flat.reshape(case["nz"] + 2, case["ny"] + 2, case["nx"] + 2)[1:-1, 1:-1, 1:-1]


def run(st):
    case = st["case"]
    path = case["path"]
    if path in ("solve", "twophase", "implicit"):
        if path == "twophase":
            st["ds"].setup(st["opr"], maxit=MAXIT, rcvg=RCVG, precision=case["mixed"])
        st["sol"].zero_()
        st["ds"].solve(st["rhs"], st["sol"])
        if path != "implicit":
            _interior(case, st["sol"]).sub_(torch.dot(st["sol"], st["weight"]))
        return st["sol"]
    if path == "host":
        ps = st["ps"]
        ps.sol[...] = 0.0
        ps.solve()
        ps.sol[ps.cfg.interior] -= np.dot(ps.sol.reshape(-1, order="F"), st["weight"])
        return ps.sol
    if path == "step":
        proj, ds = st["proj"], st["ds"]
        for u, u0 in zip(st["u"], st["u0"]):
            u.copy_(u0)
        st["P"].zero_()
        proj.laplacian(st["opr"], st["faces"])
        ds.setup(st["opr"], maxit=MAXIT, rcvg=RCVG, precision=case["mixed"])
        proj.div(*st["u"], st["div"])
        proj.rhs(st["div"], 1.0, 1.0, st["rhs"])
        st["sol"].zero_()
        ds.solve(st["rhs"], st["sol"])
        proj.shift_p(st["sol"])
        proj.pgrad(st["sol"], *st["g"])
        proj.correct(1.0, 1.0, st["g"], st["u"], st["faces"], P=st["P"], sol=st["sol"])
        return st["u"] + [st["P"]]
    if path == "fourier":
        st["f"].solve(st["rhs"], st["sol"])
        return st["sol"]
    if path == "uns":
        st["sol"].zero_()
        st["s"].solve(st["rhs"], st["sol"])
        return st["sol"]
    if path == "layer":
        L = unet.lib()
        a = (case["nx"], case["ny"], case["nz"], case["cin"], case["cout"])
        t = (a[0], a[1], a[2], a[4], a[3])

        def p(x):
            return C.c_void_p(x.data_ptr())

        unet._enter()
        rc = L.ngapnet_conv3_fwd(p(st["x"]), p(st["w"]), None, p(st["y"]), *a, 1, None)
        rc |= L.ngapnet_conv3_wgrad(p(st["x"]), p(st["g"]), p(st["dw"]), p(st["part"]), *a, None)
        rc |= L.ngapnet_flip_transpose(p(st["w"]), p(st["wd"]), a[3], a[4], None)
        rc |= L.ngapnet_conv3_fwd(p(st["g"]), p(st["wd"]), p(st["dx"]), None, *t, 0, None)
        unet._leave()
        if rc:
            raise RuntimeError(f"layer call failed ({rc})")
        return dict(y=st["y"], dx=st["dx"], dw=st["dw"])
    y = st["net"].forward(st["r"])
    if path == "forward":
        return y
    st["net"].backward((y - st["target"]) * (2.0 / y.numel()))  # mean squared error
    g = st["net"].grads()
    return dict(y=y, g=np.concatenate([g[name] for name, *_ in unet.LAYERS]))


def work(case):
    """Bytes: each input read and each output written once (the symmetric
    operator as 4 values a cell where the path takes any, 8 for face densities
    and velocities). Flops: one operator product for the solves, the transform
    for fourier, the multiply-adds of the network's layers."""
    path = case["path"]
    v = case["nx"] * case["ny"] * case["nz"]
    if path in ("solve", "host"):
        return dict(bytes=8.0 * v * 6, flops=13.0 * v)
    if path == "twophase":
        return dict(bytes=8.0 * v * 9, flops=13.0 * v)
    if path == "step":
        return dict(bytes=8.0 * v * (3 + 3 + 3 + 1), flops=60.0 * v)
    if path == "implicit":
        return dict(bytes=8.0 * v * 9, flops=13.0 * v)
    if path == "fourier":
        return dict(bytes=8.0 * v * 2, flops=5.0 * v * math.log2(v))
    if path == "uns":
        return dict(bytes=(8.0 * 9 + 4.0 * 7) * v, flops=14.0 * v)
    if path == "layer":
        mul = 2.0 * 27 * case["cin"] * case["cout"]
        return dict(bytes=v * (2.0 * 2 * case["cin"] + 3.0 * 2 * case["cout"] + 4.0 * case["cin"]), flops=3 * mul * v)
    fl = 0.0
    for _n, lvl, cin, cout, kind in unet.LAYERS:
        fl += 2.0 * (1 if kind == "1x1" else 27) * cin * cout * v / 8 ** lvl
    if path == "forward":
        return dict(bytes=8.0 * v, flops=fl)
    return dict(bytes=12.0 * v, flops=3.0 * fl)


def tolerance(case):
    path = case["path"]
    if path in ("solve", "host", "twophase", "step", "uns"):
        return {"rel": 1.5e-8}
    if path == "implicit":
        return {"rel": 1e-9}
    if path == "fourier":
        return {"rel": 1e-12}
    if path == "layer":
        return {"rel": 2e-3}
    if path == "forward":
        return {"rel": 1.2e-2}
    return {"rel": 3e-2}


# ------------------------------------------------------------------ 64-bit results in plain torch and numpy

def _fast_diag(case):
    """b -> A^-1 b of the constant-coefficient operator by diagonalising each direction."""
    d = _spacing(case)
    per = _periodic(case)
    Q, lam = [], []
    for a in range(3):
        n = d[a].numel()
        h = d[a].cpu().numpy()
        dm = 0.5 * (h + np.roll(h, 1))
        f = 1.0 / dm
        if not per[a]:
            f[0] = 0.0
        K = np.zeros((n, n))
        i = np.arange(n)
        np.add.at(K, (i, i), f + np.roll(f, -1))
        np.add.at(K, (i, (i - 1) % n), -f)
        np.add.at(K, ((i - 1) % n, i), -f)
        s = 1.0 / np.sqrt(h)
        e, v = np.linalg.eigh(K * s[:, None] * s[None, :])
        Q.append(torch.from_numpy(v).cuda())
        e[0] = 0.0
        lam.append(torch.from_numpy(e).cuda())
    s = [1.0 / v.sqrt() for v in d]
    S = _shape3(s[0], 0) * _shape3(s[1], 1) * _shape3(s[2], 2)
    L = _shape3(lam[0], 0) + _shape3(lam[1], 1) + _shape3(lam[2], 2)
    L[0, 0, 0] = 1.0

    def along(t, m, a):  # t contracted with m[:, new] over direction a
        dim = 2 - a
        t = t.movedim(dim, -1)
        sh = t.shape
        return (t.reshape(-1, sh[-1]) @ m).reshape(sh).movedim(-1, dim).contiguous()

    def solve(b):
        t = b * S
        for a in range(3):
            t = along(t, Q[a], a)
        t = t / L
        t[0, 0, 0] = 0.0
        for a in range(3):
            t = along(t, Q[a].T.contiguous(), a)
        return t * S

    return solve


def _cg(A, b, M, project, tol, most=3000):
    x = torch.zeros_like(b)
    r = project(b.clone())
    z = project(M(r))
    p = z.clone()
    rz = (r * z).sum()
    stop = tol * float(b.norm())
    for i in range(most):
        Ap = A(p)
        al = rz / (p * Ap).sum()
        x += al * p
        r -= al * Ap
        if i % 10 == 9 and float(r.norm()) <= stop:
            break
        z = project(M(r))
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x


def _bicgstab(A, b, M, tol, most=2000):
    x = torch.zeros_like(b)
    r = b.clone()
    rh = r.clone()
    rho = al = om = torch.ones((), dtype=F64, device="cuda")
    v = torch.zeros_like(b)
    p = torch.zeros_like(b)
    stop = tol * float(b.norm())
    for _ in range(most):
        new = (rh * r).sum()
        p = r + (new / rho) * (al / om) * (p - om * v)
        rho = new
        ph = M(p)
        v = A(ph)
        al = rho / (rh * v).sum()
        s = r - al * v
        sh = M(s)
        t = A(sh)
        om = (t * s).sum() / (t * t).sum()
        x += al * ph + om * sh
        r = s - om * t
        if float(r.norm()) <= stop:
            break
    return x


def _taps(x, dims):
    """x[v][c] at the 27 periodic neighbours, tap = (dz+1)*9 + (dy+1)*3 + (dx+1)."""
    g = x.reshape(dims[2], dims[1], dims[0], -1)
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                yield torch.roll(g, (-dz, -dy, -dx), (0, 1, 2)).reshape(x.shape)


def _conv(x, w, dims):
    """sum over taps of x[v + off] w[tap]^T, w [27][cout][cin]"""
    y = None
    for t, xs in enumerate(_taps(x, dims)):
        m = xs @ w[t].T
        y = m if y is None else y + m
    return y


def _net64(case, w, r):
    n = (case["nx"], case["ny"], case["nz"])
    dims = [tuple(v >> l for v in n) for l in range(4)]

    def conv(name, x, l):
        return torch.relu(_conv(x, w[name], dims[l]))

    def pool(x, l):
        d = dims[l]
        return x.reshape(d[2] // 2, 2, d[1] // 2, 2, d[0] // 2, 2, -1).mean((1, 3, 5)).reshape(-1, x.shape[1])

    def up(x, l):
        d = dims[l + 1]
        g = x.reshape(d[2], 1, d[1], 1, d[0], 1, -1).expand(d[2], 2, d[1], 2, d[0], 2, x.shape[1])
        return g.reshape(-1, x.shape[1])

    c0 = conv("c0", r.reshape(-1, 1), 0)
    c1 = conv("c1", pool(c0, 0), 1)
    c2 = conv("c2", conv("c2a", pool(c1, 1), 2), 2)
    b = conv("b", conv("b1", pool(c2, 2), 3), 3)
    d2 = conv("d2", torch.cat((up(b, 2), c2), 1), 2)
    d1 = conv("d1", torch.cat((up(d2, 1), c1), 1), 1)
    d0 = conv("d0", torch.cat((up(d1, 0), c0), 1), 0)
    return (d0 @ w["out"].reshape(-1, 1)).reshape(-1)


def exact(case, seed):
    path = case["path"]
    q = _inputs(case, seed)
    if path == "fourier":
        lam = torch.zeros((), dtype=F64, device="cuda")
        for a, n in enumerate((case["nx"], case["ny"], case["nz"])):
            k = torch.arange(n, dtype=F64, device="cuda")
            lam = lam + _shape3(4.0 * q["faces"][a][0, 0, 0] * torch.sin(math.pi * k / n) ** 2, a)
        lam[0, 0, 0] = 1.0
        t = torch.fft.fftn(q["b"]) / lam
        t[0, 0, 0] = 0.0
        return _ghosted(torch.fft.ifftn(t).real, (True, True, True))
    if path in ("solve", "host"):
        fast = _fast_diag(case)
        x = fast(q["b"])
        for _ in range(2):
            x = x + fast(q["b"] - _apply(q["faces"], x))
        w = _volume(case)
        x = x - (x * (w / w.sum())).sum()
        if path == "solve":
            return _ghosted(x)
        shape = (case["nx"] + 2, case["ny"] + 2, case["nz"] + 2)
        return _ghosted(x).cpu().numpy().reshape(shape, order="F")
    if path in ("twophase", "step"):
        fast = _fast_diag(case)
        faces = _faces(case, q["rho"])
        w = _volume(case)
        if path == "twophase":
            b = q["b"]
        else:
            d = _spacing(case)
            b = torch.zeros_like(q["rho"])
            for a in range(3):
                b -= w * (_roll(q["u"][a], a, -1) - q["u"][a]) / _shape3(d[a], a)

        def centred(t):
            return t - t.mean()

        x = _cg(lambda t: _apply(faces, t), b, fast, centred, 1e-13)
        x = centred(x)  # uniform cells
        if path == "twophase":
            return _ghosted(x)
        per = (True, True, True)
        out = []
        for a in range(3):
            h = _spacing(case)[a][0]
            rf = 0.5 * (q["rho"] + _roll(q["rho"], a, 1))
            out.append(_ghosted(q["u"][a] - (x - _roll(x, a, 1)) / h / rf, per))
        return out + [_ghosted(x, per)]
    if path == "implicit":
        shape = (case["nz"] + 2, case["ny"] + 2, case["nx"] + 2, 7)
        o = q["opr"].reshape(shape)[1:-1, 1:-1, 1:-1].movedim(-1, 0).contiguous()

        def A(t):
            y = o[0] * t
            for a in range(3):
                y = y + o[1 + 2 * a] * _roll(t, a, -1) + o[2 + 2 * a] * _roll(t, a, 1)
            return y

        x = _bicgstab(A, q["b"], lambda t: t / o[0], 1e-14)
        x = x + _bicgstab(A, q["b"] - A(x), lambda t: t / o[0], 1e-4)
        return _ghosted(x)
    if path == "uns":
        faces, out = q["faces"], q["outflow"]
        diag = out + sum(f + _roll(f, a, -1) for a, f in enumerate(faces))
        inv = torch.where(diag > 0, 1.0 / diag, 0.0)
        return _ghosted(_cg(lambda t: _apply(faces, t, out), q["b"], lambda t: inv * t, lambda t: t, 1e-13))
    if path == "layer":
        dims = (case["nx"], case["ny"], case["nz"])
        x, w, g = (q[k].to(F64) for k in ("x", "w", "g"))
        y = torch.relu(_conv(x, w, dims))
        dw = torch.stack([g.T @ xs for xs in _taps(x, dims)])
        wd = torch.stack([w[26 - t].T for t in range(27)])
        return dict(y=y, dx=_conv(g, wd, dims), dw=dw)
    w = {}
    for name, _lvl, cin, cout, kind in unet.LAYERS:
        t = torch.from_numpy(q["w"][name]).cuda().to(F64)
        w[name] = (t if kind == "1x1" else t.reshape(27, cout, cin)).requires_grad_(path == "train")
    y = _net64(case, w, q["r"].to(F64))
    if path == "forward":
        return y
    ((y - q["target"].to(F64)) ** 2).mean().backward()
    return dict(y=y.detach(), g=np.concatenate([w[name].grad.cpu().numpy().reshape(-1) for name, *_ in unet.LAYERS]))
