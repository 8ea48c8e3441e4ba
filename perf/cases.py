"""Workloads of the channel solver, as programs that use it run them.

A case is a dict of plain values; `prepare` makes the inputs from a seed and
sets up what a program keeps (the context with its resident fields, the body,
the network, page-locked host buffers for its output), `run` is one pass
through the public entry points, and `exact` is the same pass in plain torch
at 64 bits.

kind "channel"    the time loop of a channel run at constant flow rate:
                  compute_dt and compute_time_step_RK3 each step, divergence
                  and monitor every `every` steps, plane statistics and the
                  fields at the end.
kind "cylinders"  RK3 steps around two rotating cylinders (immersed boundary,
                  a BiCGSTAB solve per stage).
kind "waves"      RK3 steps between moving walls (operators set up anew at
                  every stage).
kind "poisson"    solve_poisson_equation on a host array, as a host program
                  that keeps its own arrays calls it.
kind "train"      the learned start of the body's solve: training epochs, then
                  a prediction for every marker.
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

from channel3d_parallel_amd import Channel
from channel3d_parallel_amd._lib import PREC_FP64, PREC_MIXED, ptr

DEV = "cuda"
NU = 1.0 / 2800.0
LX, LZ, LY = 2 * math.pi, math.pi, 2.0
CFL = 0.4
FFT_LENGTHS = (16, 32, 48, 64, 96, 128, 192, 256, 384, 512)


def listed():
    return [
        # the smallest call: one Poisson solve of a host program's own array
        dict(name="poisson 34x65x34", kind="poisson", nx=34, ny=65, nz=34),
        # a small channel (32x64x32 cells), where launches and latency count
        dict(name="channel 34x65x34", kind="channel", nx=34, ny=65, nz=34, steps=20, every=10,
             mixed=False, bitwise=False),
        # a wall-normal resolution chosen freely (100 rows), lengths that differ per axis
        dict(name="channel 98x101x50", kind="channel", nx=98, ny=101, nz=50, steps=20, every=10,
             mixed=False, bitwise=False),
        # an ordinary channel
        dict(name="channel 194x129x194", kind="channel", nx=194, ny=129, nz=194, steps=20, every=10,
             mixed=False, bitwise=False),
        # the same kind of run reproducing the reference's arithmetic to the last bit
        dict(name="channel bitwise 130x97x130", kind="channel", nx=130, ny=97, nz=130, steps=20,
             every=10, mixed=False, bitwise=True),
        # the largest grid of the benchmark, in FP64
        dict(name="channel 386x193x386", kind="channel", nx=386, ny=193, nz=386, steps=16, every=8,
             mixed=False, bitwise=False),
        # the same grid with the mixed-precision solver
        dict(name="channel mixed 386x193x386", kind="channel", nx=386, ny=193, nz=386, steps=12,
             every=6, mixed=True, bitwise=False),
        # a small body: each iteration of its solve is a chain of short kernels
        dict(name="cylinders 66x65x66", kind="cylinders", nx=66, ny=65, nz=66, nth=48, nzb=64,
             steps=2, guess=4, dt=0.01),
        # the two-cylinder case of the benchmark (24,576 markers)
        dict(name="cylinders 130x129x130", kind="cylinders", nx=130, ny=129, nz=130, nth=96, nzb=128,
             steps=2, guess=0, dt=0.01),
        # the moving walls of the benchmark (16,384 markers)
        dict(name="waves 130x129x66", kind="waves", nx=130, ny=129, nz=66, nxb=128, nzb=64, steps=1,
             dt=0.005),
        # the learned start of the benchmark: its 20,000 training pairs, its 24,576 markers
        dict(name="train 20000", kind="train", pairs=20000, batch=256, rows=24576, epochs=2),
    ]


def draw(rng):
    kind = rng.choices(("channel", "poisson", "cylinders", "waves", "train"), (8, 2, 4, 1, 1))[0]
    if kind == "train":
        n = int(math.exp(rng.uniform(math.log(2000), math.log(20000))))
        return dict(kind="train", pairs=n, batch=rng.choice((128, 256, 512)),
                    rows=int(math.exp(rng.uniform(math.log(1500), math.log(24576)))), epochs=2)
    if kind == "cylinders":
        n = rng.choice((64, 96, 128))
        ny = rng.randint(n - 6, n + 1)
        return dict(kind="cylinders", nx=n + 2, ny=ny, nz=n + 2, nth=3 * n // 4, nzb=n, steps=1,
                    guess=rng.choice((0, 4, 5)), dt=0.01)
    if kind == "waves":
        n = rng.choice((96, 128))
        return dict(kind="waves", nx=n + 2, ny=rng.randint(100, 129), nz=rng.choice((50, 66)), nxb=n,
                    nzb=rng.choice((32, 48)), steps=1, dt=0.005)
    while True:
        nxp, nzp = rng.choice(FFT_LENGTHS[1:9]), rng.choice(FFT_LENGTHS[1:9])
        ny = rng.choice((65, 129, 193, int(math.exp(rng.uniform(math.log(33), math.log(193))))))
        cells = nxp * nzp * (ny - 1)
        if kind == "poisson" and cells <= 128 ** 3:
            return dict(kind="poisson", nx=nxp + 2, ny=ny, nz=nzp + 2)
        if kind == "channel" and cells <= 10_000_000:
            mixed = ny in (65, 129, 193) and rng.random() < 0.3
            return dict(kind="channel", nx=nxp + 2, ny=ny, nz=nzp + 2, steps=rng.randint(8, 20),
                        every=rng.choice((4, 5, 8)), mixed=mixed,
                        bitwise=not mixed and rng.random() < 0.2)


def work(case):
    k = case["kind"]
    if k == "train":
        per = 2.0 * (54 * 256 + 2 * 256 * 256 + 256 * 4)
        params = 54 * 256 + 256 + 2 * (256 * 256 + 256) + 256 * 4 + 4
        steps = case["epochs"] * (case["pairs"] // case["batch"])
        seen = case["epochs"] * (3 * case["batch"] * (case["pairs"] // case["batch"]) + case["pairs"])
        return dict(bytes=4.0 * (case["epochs"] * case["pairs"] * 58 * 2 + steps * 7 * params + case["rows"] * 58),
                    flops=per * (seen + case["rows"]))
    cells = float((case["nx"] - 2) * (case["ny"] - 1) * (case["nz"] - 2))
    solve = 10.0 * cells * math.log2((case["nx"] - 2) * (case["nz"] - 2)) / 2 + 30 * cells
    if k == "poisson":
        return dict(bytes=16.0 * cells, flops=solve)
    # words of 8 bytes per cell and step: the three stages' right-hand sides and updates read the
    # velocity, its start and the earlier stage's right-hand side and write the velocity and theirs
    # (9 + 15 + 12), each projection reads and writes the fields and the spectrum (17)
    bytes_ = case["steps"] * 8.0 * cells * (36 + 3 * 17)
    flops = case["steps"] * 3 * (solve + 250 * cells)
    if k == "channel":
        per = cells * 8.0 * 3 * (case["steps"] + 2 * (case["steps"] // case["every"]) + 1)
        return dict(bytes=bytes_ + per + 32.0 * cells, flops=flops)
    # an immersed body: two Schur products in each of the (about 25, between the walls 50)
    # iterations of a stage's solve, each a Poisson solve with its fields (10 words per cell) and
    # the markers' four stencils and three spreading maps
    nb = 2.0 * case["nzb"] * (case["nth"] if k == "cylinders" else case["nxb"])
    products = case["steps"] * 3 * (50.0 if k == "cylinders" else 100.0)
    return dict(bytes=bytes_ + products * (80.0 * cells + nb * (375 * 12 + 4 * 15 * 12 + 64)),
                flops=flops + products * (solve + nb * 500 * 8))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def grid_args(case):
    if case["kind"] == "cylinders":
        return dict(grid_type=0)
    if case["kind"] == "waves":
        return dict(grid_type=2, alpha=2.6, min_buffer_width=0.1)
    return dict(grid_type=1, alpha=2.0)


def faces_y(ny, grid_type, alpha=2.0, min_buffer_width=0.0):
    if grid_type == 0:
        return LY * np.arange(ny) / (ny - 1)
    if grid_type == 1:
        y = np.tanh(alpha * (LY * np.arange(ny) / (ny - 1) - 1.0)) / np.tanh(alpha)
        y = y - y.min()
        return y * LY / y.max()
    nbuf = 1
    while True:  # uniform layers beyond the walls, as many points as hold the body
        m = ny - 2 * (nbuf - 1)
        s = 2.0 * np.arange(m) / (m - 1) - 1.0
        s = np.tanh(alpha * s) / np.tanh(alpha)
        hu = s[1] - s[0]
        h = LY * hu / (2.0 + (nbuf - 1) * hu)
        y = np.zeros(ny)
        y[nbuf - 1:nbuf - 1 + m] = s * h / hu
        for b in range(1, nbuf):
            y[ny - nbuf + b] = y[ny - nbuf + b - 1] + h
            y[nbuf - 1 - b] = y[nbuf - b] - h
        h1 = y[1] - y[0]
        if nbuf * h1 >= min_buffer_width + 6 * h1:
            return y + 1.0
        nbuf += 1


def flow(case, seed, pert=0.1):
    """Laminar profile of bulk velocity 1 plus a divergence-free perturbation (RMS `pert`, energy
    falling as k^(-5/3)): U(nzg, nyg, nx), V(nzg, ny, nxg), W(nz, nyg, nxg) on the GPU."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    nxp, nzp = nx - 2, nz - 2
    y = torch.tensor(faces_y(ny, **grid_args(case)), dtype=torch.float64, device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kz = torch.fft.fftfreq(nzp, 1.0 / nzp, device=DEV, dtype=torch.float64)
    ky = torch.fft.fftfreq(ny, 1.0 / ny, device=DEV, dtype=torch.float64)
    kx = torch.fft.rfftfreq(nxp, 1.0 / nxp, device=DEV, dtype=torch.float64)
    k2 = kz[:, None, None] ** 2 + ky[None, :, None] ** 2 + kx[None, None, :] ** 2
    amp = torch.where(k2 > 0, k2, 1.0) ** (-17.0 / 12.0)
    amp[0, 0, 0] = 0.0
    wall = torch.zeros(ny, dtype=torch.float64, device=DEV)
    inside = (y > 0) & (y < LY)
    wall[inside] = torch.sin(math.pi * y[inside] / LY)
    A = []
    for c in range(3):
        n = torch.randn((nzp, ny, nxp), generator=gen, device=DEV, dtype=torch.float64)
        A.append(torch.fft.irfftn(torch.fft.rfftn(n) * amp, s=(nzp, ny, nxp)) * wall[:, None])
    del amp, k2, n
    Ax, Ay, Az = A
    Ay = 0.5 * (Ay[:, 1:] + Ay[:, :-1])
    hx, hz, hy = LX / nxp, LZ / nzp, (y[1:] - y[:-1])[:, None]
    Up = (Az[:, 1:] - Az[:, :-1]) / hy - (Ay - Ay.roll(1, 0)) / hz
    Vp = (Ax - Ax.roll(1, 0)) / hz - (Az - Az.roll(1, 2)) / hx
    Wp = (Ay - Ay.roll(1, 2)) / hx - (Ax[:, 1:] - Ax[:, :-1]) / hy
    s = pert / torch.sqrt((Up.square().mean() + Vp[:, 1:-1].square().mean() + Wp.square().mean()) / 3)
    yc = 0.5 * (y[1:] + y[:-1])
    lam = torch.where((yc > 0) & (yc < LY), 1.5 * yc * (LY - yc) * 4 / LY ** 2, 0.0)
    U = torch.zeros((nz + 1, ny + 1, nx), dtype=torch.float64, device=DEV)
    V = torch.zeros((nz + 1, ny, nx + 1), dtype=torch.float64, device=DEV)
    W = torch.zeros((nz, ny + 1, nx + 1), dtype=torch.float64, device=DEV)
    U[1:nzp + 1, 1:ny, 1:nxp + 1] = lam[:, None] + s * Up
    V[1:nzp + 1, :, 1:nxp + 1] = s * Vp
    W[1:nzp + 1, 1:ny, 1:nxp + 1] = s * Wp
    return U, V, W


def cylinders(case, seed):
    """Two rotating cylinders along z, radius 0.2, their speeds within [0.3, 0.7]."""
    r = np.random.RandomState(seed % (1 << 31))
    nth, nzb = case["nth"], case["nzb"]
    nb = 2 * nth * nzb
    th = 2 * math.pi * np.arange(nth) / nth
    c, s = np.cos(th), np.sin(th)
    rad, dzb = 0.2, LZ / nzb
    slab = dict(x=[], y=[], ux=[], uy=[], n=[])
    for (xc, yc), speed in zip(((2.0, 0.7), (4.0, 1.3)), (r.uniform(0.3, 0.7), -r.uniform(0.3, 0.7))):
        slab["x"].append(xc + rad * c)
        slab["y"].append(yc + rad * s)
        slab["ux"].append(-s * speed)
        slab["uy"].append(c * speed)
        slab["n"].append(np.stack((c, s)))
    rep = lambda v: np.tile(np.concatenate(v), nzb)  # noqa: E731
    nrm = np.concatenate(slab["n"], 1)
    zero = np.zeros(nb)
    return SimpleNamespace(
        nb=nb, xb=rep(slab["x"]), yb=rep(slab["y"]),
        zb=np.repeat((np.arange(nzb) + 0.5) * dzb, 2 * nth),
        normals=np.concatenate((np.tile(nrm[0], nzb), np.tile(nrm[1], nzb), zero)),
        sb=np.full(nb, 2 * math.pi * rad / nth * dzb),
        ub=np.concatenate((rep(slab["ux"]), rep(slab["uy"]), zero)), nzb=nzb, nxb=2 * nth, nxb1=nth,
        yref=np.ones(nb, dtype=np.int32))


WAVE = (0.03, 2.0, 1.0)  # standing wave: amplitude, angular frequency, wavelengths in x


def pairs(case, seed):
    g = torch.Generator().manual_seed(int(seed))
    X = torch.randn((case["pairs"], 54), generator=g)
    mix = torch.randn((54, 4), generator=g) / 54 ** 0.5
    T = torch.tanh(X @ mix) + 0.05 * torch.randn((case["pairs"], 4), generator=g)
    R = torch.randn((case["rows"], 54), generator=g)
    P = []
    for i, o in ((54, 256), (256, 256), (256, 256), (256, 4)):
        P += [((2 * torch.rand((o, i), generator=g) - 1) * math.sqrt(6.0 / i)).reshape(-1), torch.zeros(o)]
    return X, T, R, torch.cat(P)


def pinned(shape):
    return torch.zeros(shape, dtype=torch.float64, pin_memory=True)


def poisson_rhs(case, seed):
    """A divergence-like right-hand side: the reference's array, x fastest."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    r = torch.randn((case["nz"], case["ny"] - 1, case["nx"] - 1), generator=g, device=DEV, dtype=torch.float64)
    r[:, :, -1] = r[:, :, 0]
    r[-2] = r[0]
    r[-1] = 0.0
    return r


def prepare(case, seed):
    k = case["kind"]
    if k == "train":
        X, T, R, P = pairs(case, seed)
        ch = Channel(18, 17, 18)
        ch.mlp_init(1)
        ch.mlp_set_params(P.numpy())
        return dict(case=case, ch=ch, X=X.numpy(), T=T.numpy(), R=R.numpy(), seed=int(seed) % 1000 + 1)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ch = Channel(nx, ny, nz, nu=NU, precision=PREC_MIXED if case.get("mixed") else PREC_FP64,
                 **grid_args(case))
    if k == "poisson":
        rhs, out = pinned((nz, ny - 1, nx - 1)), pinned((nz, ny - 1, nx - 1))
        rhs.copy_(poisson_rhs(case, seed))
        return dict(case=case, ch=ch, rhs=rhs, out=out)
    out = [pinned((nz + 1, ny + 1, nx)), pinned((nz + 1, ny, nx + 1)), pinned((nz, ny + 1, nx + 1)),
           pinned((nz + 1, ny + 1, nx + 1))]
    for o, f in zip(out, flow(case, seed)):
        o.copy_(f)
    if k == "cylinders":
        ch.setup_IB(cylinders(case, seed))
    if k == "waves":
        ch.setup_IB_wave("standing_wave", case["nxb"], case["nzb"], *WAVE, 0.0, 0.0)
    ch.set_fields(*[o.numpy().T for o in out])
    ch.apply_boundary_conditions()
    ch.set_pressure_gradient(3.0 * NU, 0.0, 0.0)
    state = dict(case=case, ch=ch, out=out, ptrs=[ptr(o.numpy().T) for o in out] + [None])
    if k == "channel":
        ch.set_rhs_exact(case["bitwise"])
        state["q0"] = ch.mean_mass_flow_u()
    else:
        # velocities and forces determined to ten digits
        ch.set_IB_solver(tol=1e-12, maxit=2000, guess_mode=case.get("guess", 0))
    return state


def step_limit(case):
    """The time step the convection of these flows bears."""
    return 0.15 * min(LX / (case["nx"] - 2), LZ / (case["nz"] - 2))


def run(state):
    case, ch = state["case"], state["ch"]
    k = case["kind"]
    if k == "train":
        hist = ch.mlp_train(state["X"], state["T"], case["epochs"], batch=case["batch"], lr=1e-3,
                            seed=state["seed"])
        return dict(hist=hist, params=ch.mlp_params(), pred=ch.mlp_forward(state["R"]))
    if k == "poisson":
        state["out"].copy_(state["rhs"])
        ch.solve_poisson_equation(state["out"].numpy().T)
        return dict(phi=state["out"])
    res = {}
    if k == "channel":
        limit = step_limit(case)
        for s in range(case["steps"]):
            dt = min(ch.compute_dt(CFL), limit)
            ch.compute_time_step_RK3(dt, 1, state["q0"])
            if (s + 1) % case["every"] == 0:
                ch.check_divergence()
                res["monitor"] = ch.monitor()["maxU"]
        stats = ch.plane_statistics()
        for q in ("Umean", "U2mean", "V2mean", "W2mean", "UVmean"):
            res[q] = stats[q]
    else:
        for _ in range(case["steps"]):
            ch.compute_time_step_RK3(case["dt"])
    ch._chk(ch.L.c3d_get_fields(ch.h, *state["ptrs"]))
    res.update(zip("UVWP", state["out"]))
    if k != "channel":
        # P is then the potential of the body's force alone, whose additive part the solve's
        # tolerance leaves open: it stays in the buffer
        del res["P"]
        res["fb"] = ch.get_IB_force()
    return res


# ---------------------------------------------------------------------------
# the same passes in plain torch, 64 bits; arrays are (z, y, x), index 0 the
# reference's index 1
# ---------------------------------------------------------------------------
def centres(f):
    g = np.zeros(f.size + 1)
    g[1:-1] = 0.5 * (f[:-1] + f[1:])
    g[0] = 2 * f[0] - g[1]
    g[-1] = 2 * f[-1] - g[-2]
    return g


class Grid:
    def __init__(self, case):
        self.nx, self.ny, self.nz = nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.nxp, self.nzp, self.nym = nx - 2, nz - 2, ny - 1
        self.x, self.z = LX * np.arange(nx) / (nx - 2), LZ * np.arange(nz) / (nz - 2)
        self.y = faces_y(ny, **grid_args(case))
        self.yg = centres(self.y)
        self.dx, self.dz = (np.diff(centres(f)).min() for f in (self.x, self.z))
        self.dymin = np.diff(self.yg).min()
        dev = lambda v: torch.tensor(v, dtype=torch.float64, device=DEV)  # noqa: E731
        self.hyf = dev(np.diff(self.y))[:, None]        # of the cell rows (ny - 1)
        self.hyg = dev(np.diff(self.yg))[:, None]       # between the centre rows (ny)
        wave = lambda n, d: 2 * (np.cos(2 * np.pi * np.arange(n) / n) - 1) / d ** 2  # noqa: E731
        lam = dev(wave(self.nzp, self.dz))[:, None] + dev(wave(self.nxp, self.dx)[:self.nxp // 2 + 1])
        hf, hg = np.diff(self.y), np.diff(self.yg)
        up, lo = 1 / hf / hg[1:], 1 / hf / hg[:-1]
        up[-1] = lo[0] = 0.0
        self.lo, self.inv, self.cp = lo, [], []
        for j in range(self.nym):
            d = lam - (up[j] + lo[j])
            if j == 0:
                d[0, 0] = 1.5 * d[0, 0]
            else:
                d = d - lo[j] * self.cp[-1]
            self.inv.append(1 / d)
            self.cp.append(up[j] / d)

    def poisson(self, rhs):
        """rhs on the cells (nzp, nym, nxp)."""
        b = torch.fft.fft(torch.fft.rfft(rhs, dim=2), dim=0).permute(1, 0, 2).contiguous()
        b[0] *= self.inv[0]
        for j in range(1, self.nym):
            b[j] = (b[j] - self.lo[j] * b[j - 1]) * self.inv[j]
        for j in range(self.nym - 2, -1, -1):
            b[j] -= self.cp[j] * b[j + 1]
        return torch.fft.irfft(torch.fft.ifft(b.permute(1, 0, 2), dim=0), n=self.nxp, dim=2)

    def bc(self, U, V, W):
        for a, ax, face in ((U, 2, 1), (V, 2, 0), (W, 2, 0), (U, 0, 0), (V, 0, 0), (W, 0, 1)):
            v = a.transpose(0, ax)
            if face:
                v[0] = v[-2]
                v[-1] = v[1]
            else:
                v[0] = v[-3]
                v[-2] = v[1]
                v[-1] = v[2]
        for a in (U, W):
            a[:, 0] = -a[:, 1]
            a[:, -1] = -a[:, -2]
        V[:, 0] = 0
        V[:, -1] = 0

    def div(self, U, V, W):
        c = slice(1, self.nzp + 1), slice(1, self.nym + 1), slice(1, self.nxp + 1)
        return ((U[c] - U[c[0], c[1], 0:self.nxp]) / self.dx
                + (V[c[0], 1:self.ny, c[2]] - V[c[0], 0:self.ny - 1, c[2]]) / self.hyf
                + (W[c] - W[0:self.nzp, c[1], c[2]]) / self.dz)

    def subtract_gradient(self, U, V, W, phi):
        """From the faces of the periodic cells; their images follow with the boundary conditions."""
        c = slice(1, self.nzp + 1), slice(1, self.nym + 1), slice(1, self.nxp + 1)
        U[c] -= (phi.roll(-1, 2) - phi) / self.dx
        V[c[0], 1:self.ny - 1, c[2]] -= (phi[:, 1:] - phi[:, :-1]) / self.hyg[1:-1]
        W[c] -= (phi.roll(-1, 0) - phi) / self.dz

    def pressure(self, phi, dt):
        p = phi / (dt * 8 / 15)
        p = torch.cat((p, p[:1]), 0)
        p = torch.cat((p, p[:, :, :1]), 2)
        p = torch.cat((p[:, :, :1], p, p[:, :, -1:]), 2)
        p = torch.cat((p[:, :1], p, p[:, -1:]), 1)
        return torch.cat((p[:1], p, p[-1:]), 0)

    def rhs(self, U, V, W, dpdx):
        """Right-hand sides on the interiors of U, V, W (the reference's fully conservative form)."""
        nx, ny, nz, dx, dz, hyf, hyg = self.nx, self.ny, self.nz, self.dx, self.dz, self.hyf, self.hyg
        ax = lambda a: 0.5 * (a[:, :, 1:] + a[:, :, :-1])  # noqa: E731
        ay = lambda a: 0.5 * (a[:, 1:] + a[:, :-1])  # noqa: E731
        az = lambda a: 0.5 * (a[1:] + a[:-1])  # noqa: E731
        dX, dY, dZ = (lambda a: a[:, :, 1:] - a[:, :, :-1]), (lambda a: a[:, 1:] - a[:, :-1]), (lambda a: a[1:] - a[:-1])
        I = slice(1, -1)  # noqa: E741
        uv = ay(U) * ax(V)                     # x faces, y faces, z centres
        uw = az(U) * ax(W)                     # x faces, y centres, z faces
        vw = az(V) * ay(W)                     # x centres, y faces, z faces
        Fu = (-dX(ax(U)[I, I].square()) / dx - dY(uv[I, :, I]) / hyf - dZ(uw[:, I, I]) / dz
              + NU * (dX(dX(U[I, I])) / dx ** 2 + dY(dY(U[I, :, I]) / hyg) / hyf + dZ(dZ(U[:, I, I])) / dz ** 2) + dpdx)
        Fv = (-dX(uv[I, I]) / dx - dY(ay(V)[I, :, I].square()) / hyg[1:-1] - dZ(vw[:, I, I]) / dz
              + NU * (dX(dX(V[I, I])) / dx ** 2 + dY(dY(V[I, :, I]) / hyf) / hyg[1:-1] + dZ(dZ(V[:, I, I])) / dz ** 2))
        Fw = (-dX(uw[I, I]) / dx - dY(vw[I, :, I]) / hyf - dZ(az(W)[:, I, I].square()) / dz
              + NU * (dX(dX(W[I, I])) / dx ** 2 + dY(dY(W[I, :, I]) / hyg) / hyf + dZ(dZ(W[:, I, I])) / dz ** 2))
        return Fu, Fv, Fw

    def flow_rate(self, U):
        h = self.hyg[1:-1]
        u = U[1:-1, 1:-1, 1:-1]
        return float(((u[:, 1:] + u[:, :-1]) * 0.5 * h).sum() / (h.sum() * u.shape[0] * u.shape[2]))

    def statistics(self, U, V, W):
        n = self.nx - 2
        u = 0.5 * (U[1:-2, :, :n] + U[1:-2, :, 1:n + 1])
        v = V[1:-2, :, 1:n + 1]
        v = 0.5 * (v[:, 1:] + v[:, :-1])
        v = torch.cat((-v[:, :1], v, -v[:, -1:]), 1)
        w = W[1:-1, :, 1:n + 1]
        m = lambda a: a.mean(dim=(0, 2))  # noqa: E731
        return dict(Umean=m(u), U2mean=m(u * u), V2mean=m(v * v), W2mean=m(w * w), UVmean=m(u * v))


class Body:
    """Immersed-boundary operators of one marker set: 5x5x5 delta kernels on the four staggered
    positions, interpolation and spreading, the Heaviside coefficients, the Schur product."""

    def __init__(self, g, m):
        self.g, self.nb = g, m.nb
        dev = lambda v: torch.as_tensor(np.asarray(v), dtype=torch.float64, device=DEV)  # noqa: E731
        self.n, self.ub, self.sb = dev(m.normals).view(3, -1), dev(m.ub).view(3, -1), dev(m.sb)
        self.first = torch.as_tensor(np.arange(m.nb) % m.nxb < m.nxb1, device=DEV)
        nx, ny, nz = g.nx, g.ny, g.nz
        shapes = ((nz + 1, ny + 1, nx), (nz + 1, ny, nx + 1), (nz, ny + 1, nx + 1), (nz + 1, ny + 1, nx + 1))
        self.shapes, self.idx, self.w, self.dxn = shapes, [], [], []
        yr = np.asarray(m.yref) - 1
        o = np.arange(-2, 3)
        for s in range(4):
            if s == 0:  # node index 0 is the face x = 0
                i = np.floor(m.xb / g.dx).astype(int)[:, None] + o
                x, X = i * g.dx, np.where(i % g.nxp == 0, g.nxp, i % g.nxp)
            else:
                i = np.floor((m.xb + 0.5 * g.dx) / g.dx).astype(int)[:, None] - (2 if s == 2 else 1) + o
                x, X = (i + 0.5) * g.dx, i % g.nxp + 1
            if s == 1:
                j = (np.floor((m.yb - g.y[yr]) / g.dymin).astype(int) + yr)[:, None] + o
                y, Y = g.y[j], j
            else:
                j = (np.floor((m.yb - (g.y[yr] + 0.5 * g.dymin)) / g.dymin).astype(int) + yr)[:, None] + o
                y, Y = g.yg[j + 1], j + 1
            if s == 2:
                kk = np.floor(m.zb / g.dz).astype(int)[:, None] + o
                z, Z = kk * g.dz, np.where(kk % g.nzp == 0, g.nzp, kk % g.nzp)
            else:
                kk = np.floor((m.zb + 0.5 * g.dz) / g.dz).astype(int)[:, None] - 1 + o
                z, Z = (kk + 0.5) * g.dz, kk % g.nzp + 1
            d = [dev(a) for a in (x - m.xb[:, None], y - m.yb[:, None], z - m.zb[:, None])]
            f = [delta(a, h) for a, h in zip(d, (g.dx, g.dymin, g.dz))]
            X, Y, Z = (torch.as_tensor(a, device=DEV) for a in (X, Y, Z))
            _, ly, lx = shapes[s]
            out = lambda a, b, c: (a[:, :, None, None], b[:, None, :, None], c[:, None, None, :])  # noqa: E731
            a, b, c = out(Z, Y, X)
            self.idx.append(((a * ly + b) * lx + c).reshape(self.nb, 125))
            a, b, c = out(f[2], f[1], f[0])
            self.w.append((a * b * c * (g.dx * g.dymin * g.dz)).reshape(self.nb, 125))
            a, b, c = out(self.n[2][:, None] * d[2], self.n[1][:, None] * d[1], self.n[0][:, None] * d[0])
            self.dxn.append((a + b + c).reshape(self.nb, 125))
        phi = g.poisson(-g.div(*self.spread(self.n)))
        h = 1 - phi
        face = [torch.zeros(s, dtype=torch.float64, device=DEV) for s in shapes[:3]]
        c = slice(1, g.nzp + 1), slice(1, g.nym + 1), slice(1, g.nxp + 1)
        face[0][c] = 0.5 * (h + h.roll(-1, 2))
        face[1][c[0], 1:g.ny - 1, c[2]] = 0.5 * (h[:, 1:] + h[:, :-1])
        face[2][c] = 0.5 * (h + h.roll(-1, 0))
        g.bc(*face)
        self.e1h = self.interpolate(face, True)
        self.e1hc = self.centre(h)

    def interpolate(self, F, distance=False):
        return torch.stack([((self.w[s] * self.dxn[s] if distance else self.w[s]) * F[s].reshape(-1)[self.idx[s]]).sum(1)
                            for s in range(3)])

    def centre(self, p):
        f = torch.zeros(self.shapes[3], dtype=torch.float64, device=DEV)
        f[1:self.g.nzp + 1, 1:self.g.nym + 1, 1:self.g.nxp + 1] = p
        return (self.w[3] * self.dxn[3] * f.reshape(-1)[self.idx[3]]).sum(1)

    def spread(self, f):
        out = []
        for s in range(3):
            a = torch.zeros(self.shapes[s], dtype=torch.float64, device=DEV)
            v = self.w[s] * (self.sb * f[s] / (self.g.dx * self.g.dymin * self.g.dz))[:, None]
            a.view(-1).index_add_(0, self.idx[s].reshape(-1), v.reshape(-1))
            out.append(a)
        self.g.bc(*out)
        return out

    def zero_mean(self, f):
        other = ~self.first
        f = f.clone()
        f[self.first] -= f[self.first].mean()
        f[other] -= f[other].mean()
        return f

    def regularised(self, f, dt):
        f = f.view(4, -1)
        R = self.spread(dt * NU * f[:3] - dt * f[3] * self.n)
        return R, self.g.poisson(self.g.div(*R))

    def schur(self, f, dt):
        R, phi = self.regularised(f, dt)
        G = [torch.zeros(s, dtype=torch.float64, device=DEV) for s in self.shapes[:3]]
        self.g.subtract_gradient(*G, phi)
        f = f.view(4, -1)
        u = self.interpolate([-a - r for a, r in zip(G, R)]) - self.e1h * f[:3]
        p = self.zero_mean(-self.centre(phi / dt)) - self.e1hc * f[3]
        return torch.cat((u.reshape(-1), p))

    def solve(self, b, x, dt, tol=1e-13, most=600):
        r = b - self.schur(x, dt)
        rh, rho, alpha, om = r.clone(), 1.0, 1.0, 1.0
        p, v = torch.zeros_like(r), torch.zeros_like(r)
        for _ in range(most):
            rn = float(rh @ r)
            p = r + rn / rho * alpha / om * (p - om * v)
            v = self.schur(p, dt)
            alpha = rn / float(rh @ v)
            h, s = x + alpha * p, r - alpha * v
            t = self.schur(s, dt)
            om = float(t @ s) / float(t @ t)
            x, r, rho = h + om * s, s - om * t, rn
            if float(r @ r) < tol * tol:
                break
        return x


def delta(d, h):
    r = d.abs() / h
    s3, pi = math.sqrt(3.0), math.pi
    a = torch.clamp(r, max=1.0)
    one = (17 / 48 + s3 * pi / 108 + a / 4 - a ** 2 / 4 + (1 - 2 * a) / 16 * torch.sqrt(-12 * a ** 2 + 12 * a + 1)
           - s3 / 12 * torch.asin(s3 / 2 * (2 * a - 1)))
    b = torch.clamp(r, min=1.0, max=2.0)
    two = (55 / 48 - s3 * pi / 108 - 13 * b / 12 + b ** 2 / 4
           + (2 * b - 3) / 48 * torch.sqrt(torch.clamp(-12 * b ** 2 + 36 * b - 23, min=0.0))
           + s3 / 36 * torch.asin(s3 / 2 * (2 * b - 3)))
    return torch.where(r <= 1, one, torch.where(r <= 2, two, torch.zeros_like(r))) / h


def wave_markers(case, g, t):
    """Standing-wave walls at time t: bottom and top move alike."""
    nxb, nzb = case["nxb"], case["nzb"]
    a, om, k = WAVE
    # markers midway between faces sit on the windows' edges: the same operations as the solver's
    x = (np.arange(nxb) + 0.5) * ((g.x[-1] - g.x[0] - g.dx) / nxb)
    ph = 2 * math.pi * k * x / LX
    yb, vy = a * np.sin(ph) * math.cos(om * t), -a * om * np.sin(ph) * math.sin(om * t)
    s = a * 2 * math.pi * k / LX * np.cos(ph) * math.cos(om * t)
    t1, t2 = 1 / np.sqrt(1 + s * s), s / np.sqrt(1 + s * s)
    chord = np.sqrt((LX / nxb) ** 2 + (np.roll(yb, -1) - yb) ** 2)
    area = LZ / nzb * 0.5 * (chord + np.roll(chord, 1))
    rep = lambda lo, up: np.tile(np.concatenate((lo, up)), nzb)  # noqa: E731
    nb = 2 * nxb * nzb
    zero = np.zeros(nb)
    return SimpleNamespace(nb=nb, xb=rep(x, x), yb=rep(yb, LY + yb),
                           zb=np.repeat((np.arange(nzb) + 0.5) * LZ / nzb, 2 * nxb),
                           normals=np.concatenate((rep(t2, -t2), rep(-t1, t1), zero)), sb=rep(area, area),
                           ub=np.concatenate((zero, rep(vy, vy), zero)), nzb=nzb, nxb=2 * nxb, nxb1=nxb,
                           yref=rep(np.full(nxb, 1), np.full(nxb, case["ny"])))


def exact_train(case, seed):
    X, T, R, P = (a.double() for a in pairs(case, seed))
    n, batch = case["pairs"], case["batch"]
    X, T, R = X.to(DEV), T.to(DEV), R.to(DEV)
    P = P.to(DEV).requires_grad_(True)
    dims = ((54, 256), (256, 256), (256, 256), (256, 4))

    def net(p, a):
        o = 0
        for q, (i, j) in enumerate(dims):
            a = a @ p[o:o + i * j].view(j, i).T + p[o + i * j:o + i * j + j]
            o += i * j + j
            a = a if q == 3 else torch.relu(a)
        return a

    st, mask = int(seed) % 1000 + 1, (1 << 64) - 1
    perm, hist = list(range(n)), []
    m, v, t = torch.zeros_like(P), torch.zeros_like(P), 0
    for _ in range(case["epochs"]):
        for i in range(n - 1, 0, -1):  # SplitMix64 and Fisher-Yates
            st = (st + 0x9E3779B97F4A7C15) & mask
            z = ((st ^ (st >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = (z ^ (z >> 31)) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        at = torch.tensor(perm, device=DEV)
        for b in range(n // batch):
            e = at[b * batch:(b + 1) * batch]
            g, = torch.autograd.grad((net(P, X[e]) - T[e]).square().mean(), P)
            t += 1
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            lr = 1e-3 * math.sqrt(1 - 0.999 ** t) / (1 - 0.9 ** t)
            P = (P.detach() - lr * m / (v.sqrt() + 1e-8)).requires_grad_(True)
        hist.append(float((net(P, X) - T).square().mean()))
    P = P.detach()
    return dict(hist=torch.tensor(hist, dtype=torch.float64), params=P, pred=net(P, R))


def exact(case, seed):
    k = case["kind"]
    if k == "train":
        return exact_train(case, seed)
    g = Grid(case)
    if k == "poisson":
        rhs = poisson_rhs(case, seed)
        phi = g.poisson(rhs[:g.nzp, :, :g.nxp])
        phi = torch.cat((phi, phi[:, :, :1]), 2)
        return dict(phi=torch.cat((phi, phi[:1], torch.zeros_like(phi[:1])), 0))
    X = list(flow(case, seed))
    g.bc(*X)
    q0, dpdx, t = g.flow_rate(X[0]), 3.0 * NU, 0.0
    body = Body(g, cylinders(case, seed)) if k == "cylinders" else None
    fb = torch.zeros(8 * case["nzb"] * (case["nth"] if body else case["nxb"]), dtype=torch.float64, device=DEV) if k != "channel" else None
    I = (slice(1, -1),) * 3  # noqa: E741
    res, P = {}, None
    for s in range(case["steps"]):
        if k == "channel":
            # the reference's convective limit is the largest of spacing / |velocity|: never the
            # smallest of the limits where some velocity is near zero
            dt = min(CFL * min(g.dx, g.dymin, g.dz) ** 2 / NU, 0.1, step_limit(case))
        else:
            dt = case["dt"]
        X0, F = [a.clone() for a in X], []
        for st, tk in ((1, 8 / 15), (2, 2 / 3), (3, 1.0)):
            F.append(g.rhs(*X, dpdx))
            co = ((8 / 15,), (1 / 4, 5 / 12), (1 / 4, 0.0, 3 / 4))[st - 1]
            for q in range(3):
                X[q][I] = X0[q][I] + dt * sum(a * f[q] for a, f in zip(co, F))
            if k == "waves":
                body = Body(g, wave_markers(case, g, t + tk * dt))
            g.bc(*X)
            inner = [a.clone() for a in X] if body else None
            phi = g.poisson(g.div(*X))
            g.subtract_gradient(*X, phi)
            if st == 1:
                P = g.pressure(phi, dt)
            g.bc(*X)
            if body:
                b = torch.cat(((body.ub - body.interpolate(X)).reshape(-1), body.zero_mean(-body.centre(phi / dt))))
                fb = body.solve(b, fb, dt)
                R, psi = body.regularised(fb, dt)
                X = [a - r for a, r in zip(inner, R)]
                g.subtract_gradient(*X, phi - psi)
                g.bc(*X)
        t += dt
        if k == "channel":
            d = q0 - g.flow_rate(X[0])
            X[0][I] += d
            g.bc(*X)
            dpdx = 0.5 * (dpdx + d / dt)
            if (s + 1) % case["every"] == 0:
                res["monitor"] = float(X[0][1:-1, 1:-1, 1:-1].max())
    if k == "channel":
        res.update(g.statistics(*X))
    else:
        res["fb"] = fb
    res.update(zip("UVW", X))
    if k == "channel":
        res["P"] = P
    return res
