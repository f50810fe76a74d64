"""Performance cases of the shot-profile migration library.

Each case is one call (or one batched launch) that a user of the library makes: migration (adjoint)
and modelling (forward), split-step Fourier and PSPI, 2-D and 3-D, resident plans and plain host
calls, and the elastic pair's migration.  Sizes are those of the repository's own workloads
(seiswem.synth) and generic ones in between.

`exact` restates the operators in 64-bit torch: the sampling, source index, reference velocities and
selection are evaluated in the float arithmetic that defines them, everything else in double.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "seismic.jl_amd"))

DEV = "cuda"
F32 = np.float32

# op:   "adj" migrates records into the stacked image, "fwd" models records from an image
# kind: "ssf" split step, "pspi" the reference's PSPI, "linear" interpolating PSPI (the least-squares
#       pair), "elastic" elastic migration
# call: "plan" a resident plan on device buffers, "host" one plain call on host arrays
DEFAULTS = dict(op="adj", kind="ssf", call="plan", ny=1, dt=0.004, dx=10.0, dz=10.0, fmin=2, fmax=60, nref=4, f0=20.0)

LISTED = (
    # the smallest request of a served mix: one 2-D shot, where launches and latency count
    dict(name="ssf2d_one_small", nx=128, nz=200, nt=1000, shots=1),
    # modelling half of a least-squares iteration: all shots of a small survey
    dict(name="ssf2d_model_32", op="fwd", nx=256, nz=200, nt=1000, shots=32),
    # a survey's batch of shots through a resident plan, the headline workload's grid
    dict(name="pspi2d_batch_32", kind="pspi", nx=1024, nz=500, nt=2000, dt=0.002, dz=5.0, fmin=0, fmax=80, f0=25.0, shots=32),
    # the drop-in call of a driver that migrates shot by shot from host arrays
    dict(name="pspi2d_host_call", kind="pspi", call="host", nx=1024, nz=500, nt=2000, dt=0.002, dz=5.0, fmin=0, fmax=80, f0=25.0, shots=1),
    # modelled records of a few shots over the headline grid
    dict(name="pspi2d_model_8", op="fwd", kind="pspi", nx=1024, nz=500, nt=2000, dt=0.002, dz=5.0, fmin=0, fmax=80, f0=25.0, shots=8),
    # adjoint half of a least-squares iteration with the interpolating extrapolator
    dict(name="linear2d_batch_8", kind="linear", nx=512, nz=400, nt=2000, shots=8),
    # a line whose padded length is no power of two (2000 = 2^4 5^3)
    dict(name="pspi2d_nx1000", kind="pspi", nx=1000, nz=400, nt=1500, dt=0.002, dz=5.0, fmin=3, fmax=70, f0=25.0, shots=4),
    # the 3-D workload: one shot on the full grid
    dict(name="ssf3d_full", nx=256, ny=256, nz=300, nt=1500, dx=12.5, fmin=3, fmax=50, f0=15.0, shots=1),
    # 3-D modelling of one shot
    dict(name="ssf3d_model_128", op="fwd", nx=128, ny=128, nz=150, nt=1000, dx=12.5, fmin=3, fmax=50, f0=15.0, shots=1),
    # a 3-D grid with ragged sides (transforms of 200 and 160 points)
    dict(name="ssf3d_100x80", nx=100, ny=80, nz=150, nt=1000, dx=12.5, fmin=3, fmax=50, f0=15.0, shots=2),
    # 3-D PSPI migration
    dict(name="pspi3d_128", kind="pspi", nx=128, ny=128, nz=80, nt=1000, dx=12.5, fmin=3, fmax=50, f0=15.0, shots=1),
    # elastic migration of two-component records from host arrays
    dict(name="elastic2d_host_4", kind="elastic", call="host", nx=512, nz=300, nt=1500, fmin=2, fmax=50, shots=4),
)


def listed():
    return [{**DEFAULTS, **c} for c in LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A grid side: mostly a round number, as grids are laid out, else any; now and then a power of two."""
    n, how = _log(rng, lo, hi), rng.random()
    if how < 0.3:
        return min(hi, 1 << round(math.log2(n)))
    return n if how > 0.8 else max(lo, 10 * round(n / 10))


def _slow(n):
    """Rough cost of a transform of n points against one of the next power of two."""
    while n % 2 == 0:
        n //= 2
    if n == 1:
        return 1.0
    for p in (3, 5):
        while n % p == 0:
            n //= p
    return 3.0 if n == 1 else 14.0


def draw(rng):
    """One more case of the listed ranges: 2-D lines of 64 to 1024 traces (elastic ones from 200), no deeper
    than they are long in samples, and 3-D grids of 40 to 200 a side."""
    three = rng.random() < 0.35
    kind = rng.choice(("ssf", "ssf", "pspi") if three else ("ssf", "ssf", "pspi", "pspi", "linear", "elastic"))
    op = "adj" if kind == "elastic" or rng.random() < 0.65 else "fwd"
    c = dict(DEFAULTS, kind=kind, op=op, call="host" if kind == "elastic" or rng.random() < 0.25 else "plan")
    if three:
        c.update(nx=_side(rng, 40, 200), ny=_side(rng, 40, 200), nz=_log(rng, 40, 200), nt=_log(rng, 400, 1200), dx=12.5,
                 fmin=3, fmax=rng.randint(25, 50), f0=15.0, shots=rng.randint(1, 2))
    else:
        nx = _side(rng, 200 if kind == "elastic" else 64, 1024)
        c.update(nx=nx, nz=min(_log(rng, 100, 500), nx), nt=2 * _log(rng, 250, 1000), dt=rng.choice((0.002, 0.004)),
                 dz=rng.choice((5.0, 10.0)), fmin=rng.randint(0, 4), fmax=rng.randint(40, 80), nref=rng.randint(3, 6),
                 shots=1 if rng.random() < 0.35 else _log(rng, 2, 32))
    most = 0.25 * max(work(x)["flops"] for x in listed())
    for key, least in (("shots", 1), ("nz", 30), ("fmax", 20)):
        while c[key] > least and work(c)["flops"] * max(_slow(2 * c["nx"]), _slow(2 * c["ny"])) > most:
            c[key] = max(least, int(0.8 * c[key]))
    return c


# ------------------------------------------------------------------------------- inputs
def _geometry(case):
    from seiswem import WemGeometry

    return WemGeometry(nt=case["nt"], dt=case["dt"], nmx=case["nx"], dmx=case["dx"], nz=case["nz"], dz=case["dz"],
                       nmy=case["ny"], dmy=case["dx"] if case["ny"] > 1 else 0.0, nref=case["nref"],
                       fmin=float(case["fmin"]), fmax=float(case["fmax"]), pspi=case["kind"] in ("pspi", "linear"))


def _wavelet(case):
    """Ricker wavelet from time zero on, the length of a trace."""
    n = int(1.0 / (case["f0"] * case["dt"]))
    b = (math.pi * case["f0"] * case["dt"] * np.arange(-n, n + 1)) ** 2
    w = np.zeros(case["nt"], F32)
    r = ((1.0 - 2.0 * b) * np.exp(-b)).astype(F32)[: case["nt"]]
    w[: r.size] = r
    return w


def _velocity(case, rng):
    """[nm, nz]: 2-D a background with smooth anomalies, 3-D a gradient with one; in m/s."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    x, z = np.arange(nx) * case["dx"], np.arange(nz) * case["dz"]
    if ny == 1:
        v = np.full((nx, nz), 1800.0)
        for _ in range(12):
            a, s = rng.uniform(-800.0, 800.0), rng.uniform(100.0, 300.0)
            r2 = (x[:, None] - rng.uniform(0, x[-1])) ** 2 + (z[None, :] - rng.uniform(0, z[-1])) ** 2
            v += a * np.exp(-r2 / (2 * s * s))
        return np.clip(v, 1500.0, 4000.0).astype(F32)
    y = np.arange(ny) * case["dx"]
    c = [rng.uniform(0.3, 0.7) * q[-1] for q in (x, y, z)]
    g = [np.exp(-(q - m) ** 2 / (2 * 400.0 ** 2)) for q, m in zip((x, y, z), c)]
    v = 1600.0 + 0.6 * z[None, None, :] + rng.uniform(300, 600) * g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    return v.astype(F32).reshape(nx * ny, nz)


def _shots(case, rng):
    """Source positions spread over the line, or inside the grid."""
    n, nx, ny, dx = case["shots"], case["nx"], case["ny"], case["dx"]
    ix = (np.arange(n) * nx) // n + int(rng.integers(0, max(1, nx // n)))
    sx = (ix * dx).astype(F32)
    sy = np.zeros(n, F32) if ny == 1 else (rng.integers(ny // 4, 3 * ny // 4, n) * dx).astype(F32)
    return sx, sy


def _records(case, gen, sx, sy):
    """[shots, nm, nt] on the card: echoes of the ground around each source, weaker with distance as waves
    are, over faint noise (records as modelling gives them: most of the energy comes from nearby)."""
    nx, ny, nt, dt, dx = case["nx"], case["ny"], case["nt"], case["dt"], case["dx"]
    g = torch.arange(nx * ny, device=DEV)
    gx, gy, t = (g // ny) * dx, (g % ny) * dx, torch.arange(nt, device=DEV) * dt
    noise = torch.Generator(DEV).manual_seed(int(gen.initial_seed()) + 1)
    d = torch.empty(len(sx), nx * ny, nt, device=DEV)
    for s in range(len(sx)):
        d[s].normal_(0.0, 1e-4, generator=noise)
        off, depth, amp = torch.randn(20, 2, generator=gen), torch.rand(20, generator=gen), torch.rand(20, generator=gen)
        for (ox, oy), q, a in zip(off.tolist(), depth.tolist(), amp.tolist()):
            pz = dx + q ** 2 * case["nz"] * case["dz"]
            ox, oy = 0.5 * ox * pz, 0.5 * oy * pz if ny > 1 else 0.0
            down = math.sqrt(ox ** 2 + oy ** 2 + pz ** 2)
            up = torch.sqrt((gx - float(sx[s]) - ox) ** 2 + (gy - float(sy[s]) - oy) ** 2 + pz ** 2)
            b = (math.pi * case["f0"] * (t[None, :] - ((down + up) / 1800.0)[:, None])) ** 2
            d[s] += ((a + 0.5) * 1e4 / (down * up))[:, None] * (1.0 - 2.0 * b) * torch.exp(-b)
    return d


def _image(case, gen):
    """[nm, nz] on the card: sparse reflectivity."""
    on_card = torch.Generator(DEV).manual_seed(int(gen.initial_seed()) + 2)
    r = torch.rand(2, case["nx"] * case["ny"], case["nz"], generator=on_card, device=DEV)
    return torch.where(r[0] < 0.05, 0.2 * (r[1] - 0.5), torch.zeros_like(r[0]))


def _inputs(case, seed):
    """(velocity, wavelet, sx, sy, x): x is the records or the image of the call, on the card."""
    rng, gen = np.random.default_rng([seed, 7]), torch.Generator().manual_seed(seed)
    vel, (sx, sy) = _velocity(case, rng), _shots(case, rng)
    if case["op"] == "fwd":
        return vel, _wavelet(case), sx, sy, _image(case, gen)
    x = _records(case, gen, sx, sy)
    if case["kind"] == "elastic":  # the horizontal component: the same events, weaker and turned
        x = torch.stack([0.5 * torch.roll(x, 3, -1), x])
    return vel, _wavelet(case), sx, sy, x


class Buffer:
    """A tensor as the plan calls take it: memory on the card with a `ptr`."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


def prepare(case, seed):
    import seiswem

    vel, wav, sx, sy, x = _inputs(case, seed)
    geom = _geometry(case)
    state = dict(case=case, geom=geom, vel=vel, wav=wav, sx=sx, sy=sy if case["ny"] > 1 else None)
    state["mode"] = seiswem.PSPI_LINEAR if case["kind"] == "linear" else seiswem.PSPI_COMPAT
    if case["call"] == "host":
        state["x"] = x.cpu().numpy()
        if case["kind"] == "elastic":
            state["vs"] = (vel / 1.8).astype(F32)
        return state
    x = x.contiguous()
    shape = (geom.nm, geom.nz) if case["op"] == "adj" else (len(sx), geom.nm, geom.nt)
    state.update(plan=seiswem.Plan(geom, vel, wav, pspi_mode=state["mode"]), x=Buffer(x), out=Buffer(torch.zeros(shape, device=DEV)))
    return state


def run(state):
    import seiswem

    case, adj = state["case"], state["case"]["op"] == "adj"
    if case["kind"] == "elastic":
        ux, uz = state["x"]
        return seiswem.ShotProfileEWEM((ux, uz, uz), True, vp=state["vel"], vs=state["vs"], wav=state["wav"],
                                       geom=state["geom"], sx=state["sx"])
    if case["call"] == "host":
        return seiswem.ShotProfileWEM(state["x"], adj, vel=state["vel"], wav=state["wav"], geom=state["geom"],
                                      sx=state["sx"], sy=state["sy"], pspi_mode=state["mode"])
    call = state["plan"].migrate if adj else state["plan"].model
    return call(state["x"], state["sx"], state["sy"], state["out"]).tensor


# --------------------------------------------------------------------------- sampling and work
def _sampling(case):
    """(ntfft, first bin, end bin), with the casts that define them."""
    nt, dt = case["nt"], F32(case["dt"])
    ntfft = 2 * nt  # padt = 2
    nw = ntfft // 2 + 1
    hi, lo = F32(F32(case["fmax"]) * dt) * F32(ntfft), F32(F32(case["fmin"]) * dt) * F32(ntfft)
    end = int(F32(hi + F32(1)))
    return ntfft, int(lo), min(end, nw)


def work(case):
    nx, ny, nz, nm = case["nx"], case["ny"], case["nz"], case["nx"] * case["ny"]
    nk = 2 * nx * (2 * ny if ny > 1 else 1)
    _, lo, hi = _sampling(case)
    fft = 5.0 * nk * math.log2(nk)
    if case["kind"] == "ssf":
        steps = 2 * (2 * fft + 6 * nk + 8 * nm)
    elif case["kind"] == "elastic":  # source, two potentials and four maps of a pair
        steps = 14 * fft + 18 * nk + 24 * nm
    else:
        steps = 2 * (fft * (1 + case["nref"]) + 6 * case["nref"] * nk + 8 * nm)
    data = case["shots"] * nm * case["nt"] * (2 if case["kind"] == "elastic" else 1)
    return {"bytes": 4.0 * (data + 2 * nm * nz), "flops": float(case["shots"] * (hi - lo) * nz * (steps + 4 * nm))}


# ----------------------------------------------------------------------------- 64-bit operators
class _Exact:
    """The one-way operators in complex128 over fields [frequency, shot, x, y]."""

    def __init__(self, case, vel, freqs):
        self.nx, self.ny, self.nz, self.nref = case["nx"], case["ny"], case["nz"], case["nref"]
        self.dims = (-2, -1) if self.ny > 1 else (-2,)
        self.size = (2 * self.nx, 2 * self.ny)[: len(self.dims)]
        self.nk = (2 * self.nx, 2 * self.ny if self.ny > 1 else 1)
        self.dz, self.kind = case["dz"], case["kind"]
        k = [2 * math.pi * torch.fft.fftfreq(n, case["dx"], dtype=torch.float64, device=DEV) for n in self.nk]
        self.kx = k[0][:, None]
        self.k2 = k[0][:, None] ** 2 + k[1][None, :] ** 2
        self.w = freqs[:, None, None, None]
        v = torch.from_numpy(vel).to(DEV).double().reshape(self.nx, self.ny, self.nz)
        self.po = 1.0 / v.mean((0, 1))
        self.pd = 1.0 / v - self.po
        taper = []
        for n in (self.nx, self.ny):
            i, l = torch.arange(n, dtype=torch.float64, device=DEV), 30 if n > 100 else 0
            far = torch.where(i < l, l - i, torch.where(i > n - l, i - n + l, torch.zeros_like(i)))
            taper.append(torch.exp(-((0.015 * far) ** 2)))
        self.taper = taper[0][:, None] * taper[1][None, :]
        if case["kind"] in ("pspi", "linear"):
            self._ladder(vel)

    def _ladder(self, vel):
        """Reference velocities and the choice at each point, in float as they are defined."""
        n1, lo, hi = F32(self.nref - 1), vel[: self.nx].min(0), vel.max(0)
        ir = (F32(self.nref - 1) * (vel - lo) / np.maximum(hi - lo, F32(1e-3))).astype(np.int64)
        ir = np.maximum(ir, 0)
        i1, i2 = np.where(ir > self.nref - 2, self.nref - 1, ir), np.where(ir > self.nref - 2, self.nref - 1, ir + 1)
        flat = ~(hi > lo + F32(10))
        i1[:, flat], i2[:, flat] = 0, 0
        vref = np.stack([lo + (F32(r) * (hi - lo)) / n1 for r in range(self.nref)])
        iz = np.arange(self.nz)[None, :]
        cut = (vref[i2, iz] - vref[i1, iz]).astype(np.float64) > 10.0
        v64 = lo.astype(np.float64) + np.arange(self.nref)[:, None] * (vref[-1].astype(np.float64) - lo) / (self.nref - 1.0)
        a, b = v64[i1, iz], v64[i2, iz]
        w2 = np.where(cut, (vel - a) / np.where(cut, b - a, 1.0), 0.0)
        self.v64 = v64
        self.i1, self.i2, self.cut, self.w2 = (torch.from_numpy(q).to(DEV).reshape(self.nx, self.ny, self.nz) for q in (i1, i2, cut, w2))
        self.used = [sorted(set(np.unique(i1[:, z])) | (set(np.unique(i2[:, z])) if self.kind == "linear" else set())) for z in range(self.nz)]

    def fft(self, u):
        return torch.fft.fftn(u, s=self.size, dim=self.dims)

    def ifft(self, a):
        return torch.fft.ifftn(a, dim=self.dims)[..., : self.nx, : self.ny]

    def phase(self, p2, dz):
        s = self.w ** 2 * p2 - self.k2
        r = s.abs().sqrt()
        return torch.where(s >= 0, torch.polar(torch.ones_like(r), r * dz), torch.exp(-0.2 * r * abs(dz)).to(torch.complex128))

    def step(self, u, iz, dz, adj):
        if self.kind in ("ssf", "elastic"):
            p = self.w * self.pd[..., iz] * dz
            split = torch.polar(torch.ones_like(p), p) * self.taper
            if adj:
                return self.ifft(self.fft(u) * self.phase(self.po[iz] ** 2, dz)) * split
            return self.ifft(self.fft(u * split) * self.phase(self.po[iz] ** 2, dz))
        i1, i2, cut, w2 = (q[..., iz] for q in (self.i1, self.i2, self.cut, self.w2))
        if self.kind == "linear" and not adj:
            acc = 0
            for r in self.used[iz]:
                acc = acc + self.fft(u * ((i1 == r) * (1.0 - w2) + (i2 == r) * w2)) * self.phase(self.v64[r, iz] ** -2, dz)
            return self.ifft(acc)
        a, out = self.fft(u), torch.zeros_like(u)
        for r in self.used[iz]:
            b = self.ifft(a * self.phase(self.v64[r, iz] ** -2, dz))
            if self.kind == "linear":
                out += b * ((i1 == r) * (1.0 - w2) + (i2 == r) * w2)
            else:
                out = torch.where(i1 == r, torch.where(cut, b.real.to(b.dtype), b), out)
        return out

    def separate(self, a, c, vp, vs, sep):
        """Separation of (ux, uz) into P and S potentials, or back, at every kx (adjoint forms)."""
        a, c, w, kx = self.fft(a), self.fft(c), self.w, self.kx
        kzp, kzs = (torch.sqrt(torch.clamp(w ** 2 / v ** 2 - kx ** 2, min=0.0)) for v in (vp, vs))
        n_p, n_s = torch.sqrt(kx ** 2 + kzp ** 2), torch.sqrt(kx ** 2 + kzs ** 2)
        kxp, kxs, kzp, kzs = kx / n_p, kx / n_s, kzp / n_p, kzs / n_s
        norm = kxp * kxs + kzp * kzs
        use = (norm >= 0.1) & (w >= 20.0)
        one = torch.where(use, norm, torch.ones_like(norm))
        kxp, kxs, kzp, kzs = (torch.where(use, q, torch.zeros_like(q)) for q in (kxp, kxs, kzp, kzs))
        if sep:
            r, s = kxp * a + kzp * c, -kzs * a + kxs * c
        else:
            r, s = (kxs * a - kzp * c) / one, (kzs * a + kxp * c) / one
        return self.ifft(torch.where(use, r, c)), self.ifft(torch.where(use, s, a))


def exact(case, seed):
    field = 32.0 * case["nx"] * case["ny"] * (2 if case["ny"] > 1 else 1)
    vel, wav, sx, sy, x = _inputs(case, seed)
    ntfft, lo, hi = _sampling(case)
    nx, ny, nz, nt, ns, nf = case["nx"], case["ny"], case["nz"], case["nt"], len(sx), hi - lo
    transforms = 2 * (1 + case["nref"]) if case["kind"] in ("pspi", "linear") else 14 if case["kind"] == "elastic" else 4
    if field * nf * ns * nz * transforms * (2 if ny > 1 else 1) * 5 > 4e13:
        return None  # too long in 64 bits
    omega = 2 * math.pi * torch.arange(lo, hi, dtype=torch.float64, device=DEV) / (ntfft * float(F32(case["dt"])))
    source = torch.fft.rfft(torch.from_numpy(wav).to(DEV).double(), n=ntfft)[lo:hi] / math.sqrt(ntfft)
    ix, iy = ([int(F32(int(q)) / F32(case["dx"])) for q in s] for s in (sx, sy))
    adj = case["op"] == "adj"
    elastic = case["kind"] == "elastic"
    if adj:
        spec = torch.stack([torch.fft.rfft(x.reshape(-1, ns, nx * ny, nt)[:, s].double(), n=ntfft)[..., lo:hi] for s in range(ns)]) / math.sqrt(ntfft)
        spec = spec.permute(1, 3, 0, 2).reshape(-1, nf, ns, nx, ny)  # [component, f, shot, x, y]
        m = torch.zeros(2 if elastic else 1, nx, ny, nz, dtype=torch.float64, device=DEV)
    else:
        m = x.double().reshape(nx, ny, nz)
        out = torch.zeros(nf, ns, nx, ny, dtype=torch.complex128, device=DEV)
    per = max(1, int(2e9 // (field * ns)))
    if not adj:
        per = max(1, min(per, int(4e10 // (16.0 * nx * ny * nz * ns))))
    for f in range(0, nf, per):
        at = slice(f, min(nf, f + per))
        ex = _Exact(case, vel, omega[at])
        factor = torch.where(omega[at] == 0, 1.0, 2.0)[:, None, None, None]
        us = torch.zeros(omega[at].numel(), ns, nx, ny, dtype=torch.complex128, device=DEV)
        for s in range(ns):
            us[:, s, ix[s], iy[s]] = source[at]
        dz = ex.dz
        if elastic:
            es = _Exact(case, (vel / 1.8).astype(F32), omega[at])
            peak = float(np.abs(wav).max()) / math.sqrt(ntfft)
            rx, rz = spec[0, at], spec[1, at]
            for iz in range(nz):
                us = ex.step(us, iz, -dz, True)
                p, s = ex.separate(rx, rz, 1 / ex.po[iz], 1 / es.po[iz], True)
                p, s = ex.step(p, iz, dz, True), es.step(s, iz, dz, True)
                rx, rz = ex.separate(p, s, 1 / ex.po[iz], 1 / es.po[iz], False)
                for q, u in enumerate((p, s)):
                    m[q, ..., iz] += (factor * (u * us.conj()).real).sum((0, 1)) / peak
        elif adj:
            ur = spec[0, at] * ex.w ** 2
            for iz in range(nz):
                us, ur = ex.step(us, iz, -dz, True), ex.step(ur, iz, dz, True)
                m[0, ..., iz] += (factor * (ur * us.conj()).real).sum((0, 1))
        else:
            down = []
            for iz in range(nz):
                us = ex.step(us, iz, -dz, True)
                down.append(us)
            ur = torch.zeros_like(us)
            for iz in reversed(range(nz)):
                ur = ex.step(ur + m[..., iz] * down[iz], iz, -dz, False)
            out[at] = ur * ex.w ** 2 / math.sqrt(ntfft)
            del down
    if elastic:
        return tuple(q.reshape(nx * ny, nz).cpu().numpy() for q in (m[0], torch.zeros_like(m[0]), m[1]))
    if adj:
        r = m[0].reshape(nx * ny, nz)
    else:
        band = torch.zeros(ns, nx * ny, ntfft // 2 + 1, dtype=torch.complex128, device=DEV)
        band[..., lo:hi] = out.reshape(nf, ns, nx * ny).permute(1, 2, 0)
        r = torch.fft.irfft(band, n=ntfft)[..., :nt] * ntfft
    return r.cpu().numpy() if case["call"] == "host" else r
