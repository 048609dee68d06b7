"""Performance cases of the DNS time step: what programs that use this package have it do.

A case is one of three kinds of work, over the grids, nonlinear forms, time-stepping schemes and flows that
the package serves:

  dns         one integration on the plain path: `steps` time steps of a resident DNS (the interval between two
              looks at the state), its velocity and pressure left on the device; `cfl` adds the CFL number a
              variable-dt loop asks for after each interval
  batch       an ensemble of integrations on uneven grids advanced together over a horizon, every member's
              velocity and pressure read back, as edge-tracking and ensemble programs do
  multishoot  one residual of a multiple-shooting search: a Batch built from the shots, advanced over T and the
              G_i = f^T(u_i) - u_{i+1} returned

Initial fields are seeded divergence-free no-slip perturbations. Each flow runs at a dt and a perturbation norm at
which it stays finite however long it is integrated. `exact` integrates the same equations in 64 bits from their
definition: FFTs of numpy, dense Chebyshev matrices, and per Fourier mode one dense linear system for (u, v, w, q).
"""
import ctypes
import math

import numpy as np
import torch

import channelflow_amd as cfa
from channelflow_amd.dsi import MultiShooting

LX, LZ = 2 * math.pi / 1.14, 2 * math.pi / 2.5  # the plane Couette box
SBDF = {"SBDF1": 1, "SBDF2": 2, "SBDF3": 3, "SBDF4": 4, "CNFE1": 1}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _dns(name, nx, ny, nz, flow, form, step, steps=10, dealias=True, cfl=False, dt=0.01, norm=0.05):
    return {"name": name, "kind": "dns", "Nx": nx, "Ny": ny, "Nz": nz, "flow": flow, "form": form, "stepping": step,
            "steps": steps, "dealias": dealias, "cfl": cfl, "dt": dt, "norm": norm}


def listed():
    return [
        # the smallest call: one small Couette integration, where launches and latency count
        _dns("couette_32", 32, 33, 32, "couette", "SkewSymmetric", "SBDF3"),
        # the grid, flow and form of channelflow's own time-integration test (suction boundary layer), all modes kept,
        # in a variable-dt loop that asks for the CFL number after each interval
        _dns("suction_48x35x48_cfl", 48, 35, 48, "suction", "Rotational", "SBDF3", dealias=False, cfl=True),
        # Runge-Kutta start-up scheme as the main one, the divergence form, on a ragged grid
        _dns("ragged_54x57x72_smrk2", 54, 57, 72, "couette", "Divergence", "SMRK2", steps=4),
        # an ordinary Couette integration
        _dns("couette_64", 64, 65, 64, "couette", "SkewSymmetric", "SBDF3"),
        # a served Couette request and a served Poiseuille request on the two larger grids, and the convection form
        _dns("couette_96", 96, 97, 96, "couette", "SkewSymmetric", "SBDF3", dt=0.005),
        _dns("poiseuille_128", 128, 129, 128, "poiseuille", "Rotational", "SBDF3", dt=0.005, norm=0.02),
        _dns("couette_128_conv_sbdf2", 128, 129, 128, "couette", "Convection", "SBDF2", dt=0.004),
        # the largest: the 192x129x192 channel
        _dns("channel_192", 192, 129, 192, "channel", "Rotational", "SBDF3", dt=0.004, norm=0.02),
        # one bisection round of edge tracking: many small integrations of one grid
        {"name": "batch_24x32", "kind": "batch", "grids": "24*32x33x32", "flow": "couette", "form": "SkewSymmetric",
         "stepping": "SBDF3", "steps": 200, "dt": 0.01, "norm": 0.05},
        # the uneven ensemble (32^3 : 48^3 : 64^3 = 3 : 3 : 2) over an interval of 400 steps
        {"name": "batch_uneven", "kind": "batch", "grids": "9*32x33x32 9*48x49x48 6*64x65x64", "flow": "couette",
         "form": "SkewSymmetric", "stepping": "SBDF3", "steps": 400, "dt": 0.01, "norm": 0.05},
        # a multiple-shooting residual: 16 shots of 32x49x32 over T = 4
        {"name": "multishoot_16", "kind": "multishoot", "grids": "16*32x49x32", "flow": "couette",
         "form": "SkewSymmetric", "stepping": "SBDF3", "steps": 200, "dt": 0.02, "norm": 0.05},
    ]


def draw(rng):
    sizes = [16, 18, 24, 32, 36, 48, 54, 64, 72, 96, 108, 128, 144, 162, 192]

    def size(lo, hi):
        s = [n for n in sizes if lo <= n <= hi]
        return s[min(len(s) - 1, int(rng.random() * len(s)))]

    def odd(lo, hi):
        return 2 * int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)) + 1

    form = rng.choice(["SkewSymmetric", "SkewSymmetric", "Rotational", "Rotational", "Convection", "Divergence"])
    kind = rng.choice(["dns"] * 6 + ["batch"] * 2)
    if kind == "batch":
        groups = [f"{rng.randint(4, 16)}*{size(16, 54)}x{odd(16, 60)}x{size(16, 54)}" for _ in range(rng.randint(1, 2))]
        return {"kind": "batch", "grids": " ".join(groups), "flow": "couette", "form": form, "stepping": "SBDF3",
                "steps": 10 * rng.randint(10, 20), "dt": 0.01, "norm": 10 ** rng.uniform(-3, -1.7)}
    step = rng.choice(["SBDF3"] * 5 + ["SBDF2", "SBDF4", "CNAB2", "SMRK2", "CNRK2"])
    flow = rng.choice(["couette", "couette", "poiseuille", "channel", "suction"])
    # a pressure-driven channel is unstable on fewer than about 30 Chebyshev points
    nx, nz, ny = size(16, 192), size(16, 192), odd(32 if flow in ("poiseuille", "channel") else 16, 128)
    c = _dns("", nx, ny, nz, flow, form, step, steps=3 if step in ("SMRK2", "CNRK2") else rng.randint(6, 12),
             dealias=max(nx, nz) > 96 or rng.random() < 0.85, cfl=rng.random() < 0.25,
             dt=0.01 if max(nx, nz) <= 48 else 0.004, norm=10 ** rng.uniform(-3, -1.7))
    del c["name"]
    return c


def _flags(case):
    f = {"nonlinearity": case["form"], "timestepping": case["stepping"], "initstepping": "SMRK2",
         "dealiasing": "DealiasXZ" if case.get("dealias", True) else "NoDealiasing", "dt": case["dt"],
         "baseflow": "LaminarBase", "variabledt": False}
    flow = case["flow"]
    if flow == "couette":
        f.update(nu=1 / 400, constraint="BulkVelocity", Ubulk=0.0, ulowerwall=-1.0, uupperwall=1.0)
    elif flow == "poiseuille":  # bulk velocity 1 held by its pressure gradient
        f.update(nu=1 / 2000, constraint="PressureGradient", dPdx=-3.0 / 2000)
    elif flow == "channel":  # the same at Re_bulk = 2800, in the 4 pi x 2 pi box
        f.update(nu=1 / 2800, constraint="PressureGradient", dPdx=-3.0 / 2800)
    else:  # suction boundary layer between a resting and a moving wall
        f.update(nu=1 / 300, constraint="PressureGradient", Vsuck=1 / 300, ulowerwall=0.0, uupperwall=1.0)
    return f


def _box(case):
    return (4 * math.pi, 2 * math.pi) if case["flow"] == "channel" else (LX, LZ)


def _groups(case):
    """[(count, Nx, Ny, Nz)] of a batch's member classes."""
    out = []
    for g in case["grids"].split():
        n, s = g.split("*")
        out.append((int(n),) + tuple(int(v) for v in s.split("x")))
    return out


def _live(nx, nz, dealias):
    kxd, kzd = (nx // 3 - 1, nz // 3 - 1) if dealias else (nx // 2 - 1, nz // 2 - 1)
    kx = np.concatenate([np.arange(kxd + 1), np.arange(-kxd, 0)])
    return kx, np.arange(kzd + 1)


# ---------------------------------------------------------------------------
# initial fields
# ---------------------------------------------------------------------------
def _field(seed, nx, ny, nz, box, norm, dealias=True, decay=0.5):
    """Seeded divergence-free no-slip perturbation, (3, Ny, Nx, Nz/2+1) Chebyshev-Fourier coefficients: per mode a
    wall-normal velocity (1-y^2)^2 p(y) and vorticity (1-y^2) r(y), spectra decaying in every direction."""
    rng = np.random.default_rng(seed)
    kx, kz = _live(nx, nz, dealias)
    top = 12  # higher modes are below rounding at this decay
    mx, mz = np.meshgrid(kx[np.abs(kx) <= top], kz[kz <= top], indexing="ij")
    keep = (mz > 0) | (mx > 0)
    mx, mz = mx[keep], mz[keep]
    cheb = np.polynomial.chebyshev

    def profile(factor, n):
        a = rng.standard_normal((n, mx.size)) + 1j * rng.standard_normal((n, mx.size))
        a *= decay ** (np.abs(mx) + mz) * decay ** (np.arange(n)[:, None] / 3.0)
        f = np.zeros((ny, mx.size), dtype=np.complex128)
        for i in range(n):
            e = np.zeros(n)
            e[i] = 1.0
            f += np.pad(cheb.chebmul(factor, e), (0, ny))[:ny, None] * a[i]
        return f

    one = np.array([0.5, 0.0, -0.5])  # 1 - y^2
    v, eta = profile(cheb.chebmul(one, one), min(ny - 4, 40)), profile(one, min(ny - 2, 40))
    dv = np.zeros_like(v)
    dv[:-1] = cheb.chebder(v)
    ax, az = 2 * math.pi * mx / box[0], 2 * math.pi * mz / box[1]
    k2 = ax * ax + az * az
    u = np.zeros((3, ny, nx, nz // 2 + 1), dtype=np.complex128)
    for c, w in enumerate((1j * (ax * dv - az * eta) / k2, v, 1j * (az * dv + ax * eta) / k2)):
        u[c][:, mx % nx, mz] = w
        z0 = mz == 0
        u[c][:, (-mx[z0]) % nx, 0] = np.conj(w[:, z0])
    return u * (norm / math.sqrt(2.0 * float(np.sum(u.real ** 2 + u.imag ** 2))))


def _fields(u, nx, ny, nz, box):
    return [cfa.FlowField(nx, ny, nz, 3, *box, data=u), cfa.FlowField(nx, ny, nz, 1, *box)]


class _DeviceArray:
    """A device buffer of the library as torch sees it, without a copy. The tensor made from it holds this object,
    and with it the owner of the memory."""

    def __init__(self, pointer, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f8", "data": (pointer, False), "version": 2}


def _device_state(dns, ny):
    """The resident velocity and pressure (cfg_dns_device_state): live modes, [component][y][kz][kx][re, im]."""
    P = ctypes.POINTER(ctypes.c_double)
    u, q, nkx, nkz = P(), P(), ctypes.c_int(), ctypes.c_int()
    rc = cfa.library().cfg_dns_device_state(dns._h, ctypes.byref(u), ctypes.byref(q), ctypes.byref(nkx),
                                            ctypes.byref(nkz))
    if rc:
        raise RuntimeError("cfg_dns_device_state: %d" % rc)
    out = []
    for p, n in ((u, 3), (q, 1)):
        a = _DeviceArray(ctypes.cast(p, ctypes.c_void_p).value, (n, ny, nkz.value, nkx.value, 2), dns)
        out.append(torch.as_tensor(a, device="cuda"))
    return out


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    box, fl = _box(case), _flags(case)
    if case["kind"] == "dns":
        nx, ny, nz = case["Nx"], case["Ny"], case["Nz"]
        u = _field(seed, nx, ny, nz, box, case["norm"], case["dealias"])
        return {"case": case, "dns": cfa.DNS(_fields(u, nx, ny, nz, box), cfa.DNSFlags(**fl))}
    rng = np.random.default_rng(seed + 1)
    if case["kind"] == "multishoot":
        (n, nx, ny, nz), = _groups(case)
        shots = [_field(seed * 64 + i, nx, ny, nz, box, case["norm"] * rng.uniform(0.5, 1.0)) for i in range(n)]
        return {"case": case, "shots": shots,
                "ms": MultiShooting(nx, ny, nz, *box, cfa.DNSFlags(**fl), case["steps"] * case["dt"])}
    batch, ids = cfa.Batch(), []
    for k, (n, nx, ny, nz) in enumerate(_groups(case)):
        one, two = (_field(seed * 64 + 2 * k + i, nx, ny, nz, box, case["norm"]) for i in range(2))
        for _ in range(n):  # blends of two states, as a bisection's members are, norms log-uniform
            t, s = rng.uniform(0.0, 1.0), math.exp(rng.uniform(math.log(0.02), 0.0))
            ids.append(batch.add(_fields(s * (t * one + (1 - t) * two), nx, ny, nz, box), cfa.DNSFlags(**fl)))
    return {"case": case, "batch": batch, "ids": ids}


def run(state):
    case = state["case"]
    if case["kind"] == "dns":
        dns = state["dns"]
        dns.advance_resident(case["steps"])
        out = _device_state(dns, case["Ny"])
        if case["cfl"]:
            out.append(dns.CFL())
        return out
    if case["kind"] == "multishoot":
        return state["ms"].eval(state["shots"])
    state["batch"].advance(case["steps"])
    return [x for m in state["ids"] for x in state["batch"].state(m)]


def work(case):
    """Bytes: every step reads the state's velocity and nonlinear-term histories and writes the new velocity,
    pressure and nonlinear term once (live modes only). Flops: the FFTs of the form's fields at 5 N log2 N, the
    Chebyshev transforms as matrix products of the upper half of the points, and the solves."""
    if case["kind"] == "dns":
        groups, dealias = [(1, case["Nx"], case["Ny"], case["Nz"])], case["dealias"]
    else:
        groups, dealias = _groups(case), True
    evals = case["steps"] * (3 if case["stepping"] in ("SMRK2", "CNRK2") else 1)
    order = SBDF.get(case["stepping"], 2)
    fin, fout, src = {"Rotational": (6, 3, 6), "Convection": (12, 3, 6), "SkewSymmetric": (12, 9, 6),
                      "Divergence": (3, 6, 3)}[case["form"]]
    total_bytes = total_flops = 0.0
    for n, nx, ny, nz in groups:
        kx, kz = _live(nx, nz, dealias)
        field = 16.0 * ny * kx.size * kz.size
        total_bytes += n * evals * field * (3 * 2 * order + 3 + 1 + 3)
        fft = 5.0 * nx * nz * math.log2(nx * nz) / 2
        y = 4.0 * ny * ny / 2 * kx.size * kz.size
        total_flops += n * evals * (ny * fft * (fin + fout) + y * (src + fout) + 300.0 * ny * kx.size * kz.size)
    if case["kind"] != "dns":  # the members' states as they are handed over and back
        total_bytes += sum(n * 4 * 16.0 * ny * nx * (nz // 2 + 1) for n, nx, ny, nz in groups)
    return {"bytes": total_bytes, "flops": total_flops}


# ---------------------------------------------------------------------------
# the same in 64 bits, from the equations
# ---------------------------------------------------------------------------
class _Reference:
    def __init__(self, case):
        self.nx, self.ny, self.nz = nx, ny, nz = case["Nx"], case["Ny"], case["Nz"]
        self.fl, self.form, (self.lx, self.lz) = _flags(case), case["form"], _box(case)
        self.nu, self.dt = self.fl["nu"], case["dt"]
        self.kx, self.kz = _live(nx, nz, case["dealias"])
        n = np.arange(ny)
        self.T = np.cos(math.pi * np.outer(n, n) / (ny - 1))
        self.Ti = np.linalg.inv(self.T)
        self.D = np.zeros((ny, ny))
        self.D[:-1] = np.polynomial.chebyshev.chebder(np.eye(ny))
        self.ax, self.az = 2 * math.pi * self.kx / self.lx, 2 * math.pi * self.kz / self.lz
        self.U = self.base()
        self.rhsU = self.nu * (self.D @ (self.D @ self.U))
        self.bulk = self.fl["constraint"] == "BulkVelocity"
        w = np.zeros(ny)
        w[::2] = 1.0 / (1.0 - n[::2] ** 2.0)
        self.mean = w  # mean over y of each Chebyshev polynomial
        self.systems = {}

    def base(self):
        """The laminar streamwise profile: nu U'' - V U' = dPdx with its wall values (here V is -Vsuck)."""
        fl, n = self.fl, np.arange(self.ny)
        A = fl["nu"] * self.D @ self.D + fl.get("Vsuck", 0.0) * self.D
        r = np.full(self.ny, 0.0)
        r[0] = fl.get("dPdx", 0.0)
        A[-2], A[-1] = np.ones(self.ny), (-1.0) ** n
        r[-2], r[-1] = fl.get("uupperwall", 0.0), fl.get("ulowerwall", 0.0)
        return np.linalg.solve(A, r)

    def physical(self, c):  # (ny, nkx, nkz) coefficients at y points -> (ny, nx, nz)
        full = np.zeros((self.ny, self.nx, self.nz // 2 + 1), dtype=np.complex128)
        full[:, self.kx[:, None] % self.nx, self.kz[None, :]] = c
        return np.fft.irfft2(full, s=(self.nx, self.nz), axes=(1, 2)) * (self.nx * self.nz)

    def spectral(self, p):  # and back, with the y transform
        full = np.fft.rfft2(p, axes=(1, 2)) / (self.nx * self.nz)
        return np.tensordot(self.Ti, full[:, self.kx[:, None] % self.nx, self.kz[None, :]], 1)

    def dx(self, a):
        return 1j * self.ax[:, None] * a

    def dz(self, a):
        return 1j * self.az * a

    def dy(self, a):
        return np.tensordot(self.D, a, 1)

    def nonlinear(self, u):
        tot = u.copy()
        tot[0][:, 0, 0] += self.U
        tot[1][0, 0, 0] -= self.fl.get("Vsuck", 0.0)
        phys = lambda a: self.physical(np.tensordot(self.T, a, 1))  # noqa: E731
        up = [phys(a) for a in tot]
        if self.form == "Rotational":
            w = [phys(self.dy(tot[2]) - self.dz(tot[1])), phys(self.dz(tot[0]) - self.dx(tot[2])),
                 phys(self.dx(tot[1]) - self.dy(tot[0]))]
            return np.stack([self.spectral(w[1] * up[2] - w[2] * up[1]), self.spectral(w[2] * up[0] - w[0] * up[2]),
                             self.spectral(w[0] * up[1] - w[1] * up[0])])
        conv = div = 0.0
        if self.form != "Divergence":
            conv = np.stack([self.spectral(up[0] * phys(self.dx(a)) + up[1] * phys(self.dy(a)) +
                                           up[2] * phys(self.dz(a))) for a in tot])
        if self.form != "Convection":
            div = np.stack([self.dx(self.spectral(up[0] * a)) + self.dy(self.spectral(up[1] * a)) +
                            self.dz(self.spectral(up[2] * a)) for a in up])
        return conv if self.form == "Convection" else div if self.form == "Divergence" else 0.5 * (conv + div)

    def linear(self, u, q):
        out = np.empty_like(u)
        k2 = self.ax[:, None] ** 2 + self.az ** 2
        for c, g in enumerate((self.dx, self.dy, self.dz)):
            out[c] = self.nu * (self.dy(self.dy(u[c])) - k2 * u[c]) - g(q)
        for c, extra in ((0, self.rhsU), (2, 0.0)):
            out[c][:, 0, 0] += extra
            if self.bulk:
                d = self.D @ u[c][:, 0, 0].real + (self.D @ self.U if c == 0 else 0.0)
                out[c][0, 0, 0] -= self.nu * (d.sum() - (d * (-1.0) ** np.arange(self.ny)).sum()) / 2.0
            elif c == 0:
                out[c][0, 0, 0] -= self.fl.get("dPdx", 0.0)
        return out

    def system(self, lam):
        """Per mode: the momentum equations on the first Ny - 2 Chebyshev rows, no slip, and div u = 0 on all rows."""
        if lam not in self.systems:
            N, r = self.ny, self.ny - 2
            ax = np.repeat(self.ax, self.kz.size)[1:]
            az = np.tile(self.az, self.kx.size)[1:]
            A = torch.zeros((ax.size, 4 * N, 4 * N), dtype=torch.complex128)
            I, D = torch.eye(N, dtype=torch.complex128), torch.from_numpy(self.D).to(torch.complex128)
            tx, tz = torch.from_numpy(1j * ax)[:, None, None], torch.from_numpy(1j * az)[:, None, None]
            H = self.nu * (D @ D) - lam * I + (self.nu * (tx * tx + tz * tz)) * I
            for c, G in enumerate((tx * I, D.expand(ax.size, N, N), tz * I)):
                A[:, c * r:(c + 1) * r, c * N:(c + 1) * N] = H[:, :r]
                A[:, c * r:(c + 1) * r, 3 * N:] = -G[:, :r]
                A[:, 3 * r + 2 * c, c * N:(c + 1) * N] = 1.0
                A[:, 3 * r + 2 * c + 1, c * N:(c + 1) * N] = torch.from_numpy((-1.0) ** np.arange(N) + 0j)
                A[:, 3 * N:, c * N:(c + 1) * N] = G
            self.systems[lam] = torch.linalg.lu_factor(A)
        return self.systems[lam]

    def solve(self, R, lam):
        N, r, nk = self.ny, self.ny - 2, self.kx.size * self.kz.size
        b = np.zeros((nk - 1, 4 * N, 1), dtype=np.complex128)
        for c in range(3):
            b[:, c * r:(c + 1) * r, 0] = -R[c].reshape(N, nk)[:r, 1:].T
        x = torch.linalg.lu_solve(*self.system(lam), torch.from_numpy(b)).numpy()[:, :, 0]
        u, q = np.zeros_like(R), np.zeros_like(R[0])
        for c in range(4):
            (u[c] if c < 3 else q).reshape(N, nk)[:, 1:] = x[:, c * N:(c + 1) * N].T
        # the mean mode: u and w with the given pressure gradient or mean, v = 0
        bc = np.stack([np.ones(N), (-1.0) ** np.arange(N)])
        H = np.concatenate([(self.nu * self.D @ self.D - lam * np.eye(N))[:r], bc])
        for c, extra in ((0, self.rhsU), (2, np.zeros(N))):
            f = R[c][:, 0, 0].real + extra
            if not self.bulk and c == 0:
                f[0] -= self.fl.get("dPdx", 0.0)
            one = np.zeros(N)
            one[0] = 1.0
            p, s = (np.linalg.solve(H, np.concatenate([-v[:r], [0.0, 0.0]])) for v in (f, one))
            if self.bulk:
                goal = self.fl.get("Ubulk", 0.0) - self.mean @ self.U if c == 0 else 0.0
                p = p + s * (goal - self.mean @ p) / (self.mean @ s)
            u[c][:, 0, 0] = p
        H = np.concatenate([(self.D @ self.D)[:r], bc])
        q[:, 0, 0] = np.linalg.solve(H, np.concatenate([(self.D @ R[1][:, 0, 0].real)[:r], [0.0, 0.0]]))
        return u, q

    def smrk2(self, u, q):
        f0 = 0.0
        for a, b, g, z in ((29 / 96, 37 / 160, 8 / 15, 0.0), (-3 / 40, 5 / 24, 5 / 12, -17 / 60),
                           (1 / 6, 1 / 6, 3 / 4, -5 / 12)):
            f1, f0 = f0, self.nonlinear(u)
            lam = 1.0 / (b * self.dt)
            u, q = self.solve(lam * u + (a / b) * self.linear(u, q) - (g / b) * f0 - (z / b) * f1, lam)
        return u, q

    def advance(self, u, q, stepping, steps):
        if stepping == "SMRK2":
            for _ in range(steps):
                u, q = self.smrk2(u, q)
            return u, q
        eta, al, be = {1: (1.0, (-1,), (1,)), 2: (1.5, (-2, 0.5), (2, -1)), 3: (11 / 6, (-3, 1.5, -1 / 3), (3, -3, 1)),
                       4: (25 / 12, (-4, 3, -4 / 3, 0.25), (4, -6, 4, -1))}[SBDF[stepping]]
        hist = []
        for _ in range(steps):
            hist.insert(0, (u, self.nonlinear(u)))
            if len(hist) < len(al):
                u, q = self.smrk2(u, q)
            else:
                R = sum(-a / self.dt * v - b * f for a, b, (v, f) in zip(al, be, hist))
                u, q = self.solve(R, eta / self.dt)
                hist.pop()
        return u, q

    def cfl(self, u, scale):
        y = np.cos(math.pi * np.arange(self.ny) / (self.ny - 1))
        dy = np.concatenate([[y[0] - y[1]], (y[:-2] - y[2:]) / 2, [y[0] - y[1]]])[:, None, None]
        tot = u.copy()
        tot[0][:, 0, 0] += self.U
        p = [self.physical(np.tensordot(self.T, a, 1)) for a in tot]
        return scale * max(0.0, (p[0] / (self.lx / self.nx)).max(), (p[1] / dy).max(), (p[2] / (self.lz / self.nz)).max())


def exact(case, seed):
    if case["kind"] != "dns" or case["stepping"] not in ("SMRK2", "SBDF1", "SBDF2", "SBDF3", "SBDF4"):
        return None
    kx, kz = _live(case["Nx"], case["Nz"], case["dealias"])
    if kx.size * kz.size * (4.0 * case["Ny"]) ** 3 > 4e9:  # larger grids take too long
        return None
    ref = _Reference(case)
    u = _field(seed, case["Nx"], case["Ny"], case["Nz"], _box(case), case["norm"], case["dealias"])
    u = u[:, :, kx[:, None] % case["Nx"], kz[None, :]]
    u, q = ref.advance(u, np.zeros_like(u[0]), case["stepping"], case["steps"])

    def compact(a):
        return np.ascontiguousarray(np.swapaxes(a, -1, -2)).view(np.float64).reshape(*a.shape[:-2], kz.size, kx.size, 2)

    out = [compact(u), compact(q)[None]]
    if case["cfl"]:
        out.append(ref.cfl(u, (2 / 3 if case["dealias"] else 1.0) * math.pi * case["dt"]))
    return out
