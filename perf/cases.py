"""What a user of this framework has it do, as timed cases: reconstruction calls of the engine's
algorithms over the range of scans it takes, from a 64-pixel tutorial scan to 512-pixel frames,
in both precisions, with ragged batch and frame counts, through one object slice or several, in
the far and the near field, with and without refined positions, and the cost's gradient for an
outer torch loop.

A state is an engine on its scan (counts resident on the GPU, as a program keeps it); a pass is
one call of an algorithm for a few epochs or cycles and the download of what it updated, which
is how a program takes the result. A second pass goes on from where the first one left.

`exact` restates each algorithm in 64 bits with plain torch operations.
"""

import math

import numpy as np
import torch

import ptyrs_amd as pa
from ptyrs_amd import autograd, sim

LAM, DIST, DPIX = sim.WAVELENGTH, sim.DISTANCE, sim.DETECTOR_PIXEL
POWERS = {1: (1.0,), 2: (0.8, 0.2), 3: (0.7, 0.2, 0.1), 4: (0.7, 0.15, 0.1, 0.05),
          5: (0.6, 0.15, 0.1, 0.1, 0.05), 6: (0.5, 0.15, 0.1, 0.1, 0.1, 0.05)}
GAP = 2e-6  # metres between object slices

_BASE = dict(alg="rpie", n=256, modes=4, frames=1024, step=24, batch=100, passes=5, dtype="c64",
             counts="float", optics="far", slices=1, positions="none", cost="poisson",
             psi_f16=False, probe=True)


def _case(name, **kw):
    return dict(_BASE, name=name, **kw)


def listed():
    return [
        # The smallest run anybody makes: one mode, a 10x10 scan of 64-pixel frames, every frame
        # in one batch; launches and latency are all of it.
        _case("rpie_64x1", n=64, modes=1, frames=100, step=8, passes=10),
        # The headline workload of bench.py: 256-pixel frames, four modes, a 32x32 scan.
        _case("rpie_256x4", passes=5),
        # The same step in double precision on a smaller scan.
        _case("rpie_256x4_double", frames=420, passes=2, dtype="c128"),
        # Detector counts as uint16 with masked pixels, a side that is no power of two, batches
        # that do not divide the scan.
        _case("rpie_96x3_masked", n=96, modes=3, frames=317, step=10, batch=37, passes=5,
              counts="u16"),
        # Near field, the object little larger than the frame: the whole plane is sampled at
        # sub-pixel positions, which are refined.
        _case("rpie_near_positions", n=128, modes=2, frames=64, step=3, batch=32, passes=1,
              optics="near", positions="refine"),
        # Least-squares maximum likelihood on the headline scan.
        _case("lsqml_256x4", alg="lsqml", passes=2),
        # Thick samples: three slices, positions refined with the reconstruction.
        _case("lsqml_slices_positions", alg="lsqml", n=128, modes=2, frames=400, step=8, batch=50,
              passes=1, slices=3, positions="refine"),
        # Alternating projections, object and probe, the usual start of a reconstruction.
        _case("ap_256x4", alg="ap", passes=3),
        # Difference map on large frames.
        _case("dm_512x2", alg="dm", n=512, modes=2, frames=300, step=40, passes=3),
        # Relaxed averaged alternating reflections with half-precision carried waves, an uneven
        # number of frames.
        _case("raar_256x2_half", alg="raar", modes=2, frames=799, passes=3, psi_f16=True),
        # The conjugate-gradient refinement at the end of a reconstruction.
        _case("ml_128x2", alg="ml", n=128, modes=2, frames=400, step=12, passes=5),
        # The cost and its gradient through three slices for an optimiser written in torch.
        _case("grad_128x2_slices", alg="grad", n=128, modes=2, frames=400, step=8, passes=1,
              slices=3),
    ]


def _weight(c):
    """Relative work of a pass, for keeping drawn cases under the listed ones."""
    w = c["frames"] * c["n"] ** 2 * c["modes"] * c["passes"] * (2 if c["dtype"] == "c128" else 1)
    w *= {"rpie": 1, "ap": 1, "dm": 1.6, "raar": 1.6, "ml": 2.2, "lsqml": 2, "grad": 2}[c["alg"]]
    if c["slices"] > 1:
        w *= 1.5 * c["slices"]
    if c["positions"] != "none":
        w *= 3
    if c["optics"] == "near":
        w *= 12
    return w


def draw(rng):
    limit = 0.8 * max(_weight(c) for c in listed())
    kinds = ["rpie"] * 4 + ["lsqml"] * 2 + ["ap", "dm", "raar", "ml", "grad", "near", "slices"]
    while True:
        kind = rng.choice(kinds)
        c = dict(_BASE, alg=kind, probe=True)
        c["n"] = rng.choice([64, 96, 128, 128, 256, 256, 512])
        c["modes"] = rng.randint(1, 5)
        c["frames"] = int(round(math.exp(rng.uniform(math.log(60), math.log(1200)))))
        c["step"] = max(3, int(c["n"] * rng.uniform(0.07, 0.12)))
        c["batch"] = rng.randint(24, 128)
        c["passes"] = rng.randint(1, 4)
        c["dtype"] = rng.choice(["c64", "c64", "c128"])
        c["counts"] = rng.choice(["float", "u16"])
        if kind in ("ap", "dm", "raar", "ml"):
            c.update(n=rng.choice([64, 128, 128, 256, 256, 512]), modes=rng.choice([1, 2, 4]))
        if kind == "lsqml":
            c["cost"] = rng.choice(["poisson", "amplitude"])
        elif kind in ("dm", "raar"):
            c["psi_f16"] = c["dtype"] == "c64" and rng.random() < 0.5
        elif kind == "ml":
            c["probe"] = rng.random() < 0.6
        elif kind == "grad":
            c.update(slices=rng.randint(1, 3), passes=1, n=rng.choice([64, 128, 256]),
                     modes=rng.randint(1, 3))
        elif kind == "near":
            c.update(alg="rpie", optics="near", positions="refine", passes=1, step=3,
                     n=rng.choice([64, 96, 128]), modes=rng.randint(1, 3),
                     frames=rng.randint(16, 64), batch=rng.randint(8, 40))
        elif kind == "slices":
            c.update(alg="lsqml", slices=rng.randint(2, 3), positions="refine", passes=1,
                     n=rng.choice([64, 128, 256]), modes=rng.randint(1, 3))
        if _weight(c) <= limit:
            return c


# ---- inputs --------------------------------------------------------------------------------------


def _geometry(c):
    """Object pixel and, with slices or in the near field, the exit model's numbers."""
    if c["optics"] == "near":
        return 1e-6, 1.24e-10, 2e-3          # pixel, wavelength, propagation distance
    return sim.pixel_size(c["n"]), LAM, DIST


def _side(c, reach):
    """Object side: the scan's extent, the frame and a margin, a multiple of 4. In the near
    field no more than 5/4 of the frame, where the whole object plane is sampled."""
    side = (2 * reach + c["n"] + 8 + 3) // 4 * 4
    if c["optics"] == "near":
        side = min(side, (5 * c["n"] - 1) // 4 // 2 * 2)
    return side


def _smooth(gen, shape, sigma):
    """Gaussian-filtered white noise (periodic) scaled to [0, 1]."""
    w = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)
    fy = torch.fft.fftfreq(shape[-2], device="cuda", dtype=torch.float64)[:, None]
    fx = torch.fft.fftfreq(shape[-1], device="cuda", dtype=torch.float64)[None]
    s = torch.fft.ifft2(torch.fft.fft2(w) * torch.exp(-2 * (math.pi * sigma) ** 2
                                                      * (fy * fy + fx * fx))).real
    lo, hi = s.amin((-2, -1), keepdim=True), s.amax((-2, -1), keepdim=True)
    return (s - lo) / (hi - lo)


def _inputs(c, seed):
    """The scan: corners, counts (detector order), start object and probe, position errors.
    Everything from the seed; probe and frames on the GPU until the counts are downloaded."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    rng = np.random.default_rng(int(seed))
    n, f = c["n"], c["frames"]
    k = np.arange(f)
    r = 0.56 * c["step"] * np.sqrt(k)  # a Fermat spiral, about one position per step squared
    th = k * math.pi * (3 - math.sqrt(5)) + rng.uniform(0, 6)
    y = np.round(r * np.sin(th)) + rng.integers(-1, 2, f)
    x = np.round(r * np.cos(th)) + rng.integers(-1, 2, f)
    side = _side(c, int(0.56 * c["step"] * math.sqrt(f)) + 2)
    half = (side - n) // 2
    oy = np.clip(y, -half, half).astype(np.int64) + half
    ox = np.clip(x, -half, half).astype(np.int64) + half
    ph = _smooth(gen, (c["slices"], side, side), 4.0)
    if c["slices"] > 1:
        truth = torch.exp(torch.complex(-0.015 * ph, 0.3 * ph))
    else:
        amp = 0.9 + 0.1 * torch.rand(ph.shape, generator=gen, device="cuda", dtype=torch.float64)
        truth = torch.polar(amp, ph - 0.5)
    probe = torch.from_numpy(sim.hermite_gauss_probe(n, powers=POWERS[c["modes"]])).cuda()
    m = _Model(c, torch.from_numpy(oy).cuda(), torch.from_numpy(ox).cuda(), side)
    photons = 10 ** rng.uniform(5.5, 7)
    offs = np.zeros((f, 2))
    if c["positions"] != "none":
        offs = rng.normal(0.0, 0.3, (f, 2))
    total = torch.tensor(0.0, device="cuda", dtype=torch.float64)
    counts = torch.empty((f, n, n), device="cuda")
    for s in range(0, f, 64):
        fr = list(range(s, min(f, s + 64)))
        e = m.exit_waves([t[None] for t in truth], probe, fr, None)
        counts[s:s + 64] = m.to_detector((m.forward(e).abs() ** 2).sum(1)).float()
    total = counts.double().sum() / f
    scale = photons / total
    counts = torch.poisson(counts * scale.float(), generator=gen)
    if c["counts"] == "u16":
        # a counting detector saturates; a dead stripe and dead pixels are masked
        counts = counts.clamp(max=60000.0)
        dead = torch.rand((n, n), generator=gen, device="cuda") < 0.004
        dead[:, n // 3] = True
        counts = torch.where(dead[None], torch.full_like(counts, pa.MASKED), counts)
        host = counts.to(torch.int32).cpu().numpy().astype(np.uint16)
    else:
        host = counts.cpu().numpy()
    probe = probe * torch.sqrt(scale)
    start = torch.rand(truth.shape, generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    if c["slices"] > 1 or c["alg"] in ("lsqml", "ml", "grad"):
        start = truth * torch.polar(torch.ones_like(start), 0.1 * start)  # late in a run
    else:
        start = torch.polar(torch.ones_like(start), start)
    probe = probe * torch.exp(0.02j * torch.randn(probe.shape, generator=gen, device="cuda",
                                                  dtype=torch.float64))
    return dict(counts=host, oy=oy, ox=ox, side=side, obj=start[:, None], probe=probe, offs=offs,
                model=m)


def _optics(c):
    n = c["n"]
    pixel, lam, dist = _geometry(c)
    if c["optics"] == "near":
        o = pa.Optics.free_space(pa.Wavefield([n, n], lam, [pixel, pixel], dist))
    else:
        o = pa.Optics.far_field(lam, dist, DPIX, [n, n])
    if c["slices"] > 1:
        o = o.with_slices([pa.Wavefield([n, n], lam, [pixel, pixel], GAP)] * (c["slices"] - 1))
    return o


def prepare(case, seed):
    c = dict(_BASE, **case)
    d = _inputs(c, seed)
    pixel, _, _ = _geometry(c)
    corners = np.stack([d["oy"], d["ox"]], axis=1)
    scan = pa.Scan(d["counts"], d["oy"] * pixel, d["ox"] * pixel, LAM, DIST, DPIX, corners=corners)
    obj = d["obj"].cpu().numpy()
    opts = dict(dtype=c["dtype"])
    if c["psi_f16"]:
        opts["psi_f16"] = True
    g = pa.GpuPtycho(scan, obj if c["slices"] > 1 else obj[0], d["probe"].cpu().numpy(),
                     optics=_optics(c), **opts)
    if c["positions"] == "refine":
        g.set_features(position=d["offs"])
    s = dict(case=c, engine=g)
    if c["alg"] == "grad":
        dt = torch.complex64 if c["dtype"] == "c64" else torch.complex128
        s["objects"] = d["obj"].to(dt).requires_grad_(True)
        s["probe"] = d["probe"].to(dt).requires_grad_(True)
    return s


def run(state):
    c, g = state["case"], state["engine"]
    k, alg = c["passes"], c["alg"]
    if alg == "grad":
        o, p = state["objects"], state["probe"]
        o.grad = p.grad = None
        loss = autograd.cost(g, o, p, c["cost"])
        loss.backward()
        return dict(loss=loss.detach(), objects=o.grad, probe=p.grad)
    if alg == "rpie":
        g.rpie(k, batch_size=c["batch"])
    elif alg == "lsqml":
        g.lsqml(k, 0, c["batch"], c["cost"], 7)
    elif alg == "ap":
        g.ap(k, probe_inertia=0.01)
    elif alg == "dm":
        g.dm(k)
    elif alg == "raar":
        g.raar(k)
    elif alg == "ml":
        g.ml(k, update_probe=c["probe"])
    out = dict(objects=g.objects, probe=g.probe)
    if c["positions"] == "refine":
        out["position"] = g.features["position"]
    return out


def work(case):
    """A pass reads the scan's counts once per epoch or cycle, reads and writes the object and
    the probe (and, of the algorithms that carry them, every exit wave once per cycle); its
    operations are the transforms, a line of N values at 5 N log2 N."""
    c = dict(_BASE, **case)
    n2, m, f, k = c["n"] ** 2, c["modes"], c["frames"], c["passes"]
    cb = 8 if c["dtype"] == "c64" else 16
    side = _side(c, int(0.56 * c["step"] * math.sqrt(f)) + 2)
    state = 2 * cb * (c["slices"] * side * side + m * n2)
    b = k * (4 * f * n2 + state)
    if c["alg"] in ("dm", "raar"):
        b += k * 2 * f * m * n2 * (4 if c["psi_f16"] else cb)
    # 2D transforms per frame and mode: out and back; between slices two 2D transforms a gap each
    # way; the Poisson step of LSQML needs no more; ML forwards its directions too
    pairs = 2 * (2 * c["slices"] - 1) + (3 if c["alg"] == "ml" else 0)
    if c["optics"] == "near":
        pairs *= 2
    fl = k * f * m * pairs * 5 * n2 * math.log2(n2)
    return {"bytes": float(b), "flops": float(fl)}


def tolerance(case):
    """Relative errors, about four times what complex64 runs over these ranges are from `exact`:
    5e-6 after a few steps of most cases; up to 5e-5 of rPIE with a single mode or in the near
    field, whose steps divide by small overlaps; 2e-4 of a gradient (and of what ML adds along
    it), a small difference of large terms; 1.5e-4 with half-precision carried waves.
    complex128 runs are within 2e-13, and the bound leaves room for the same amplification."""
    c = dict(_BASE, **case)
    rel = 2e-5
    if c["dtype"] == "c128":
        rel = 1e-10
    elif c["psi_f16"]:
        rel = 6e-4
    elif c["alg"] in ("ml", "grad"):
        rel = 1e-3
    elif c["alg"] == "rpie" and (c["modes"] == 1 or c["optics"] == "near"):
        rel = 2e-4
    return {"rel": rel, "max": 50 * rel}


# ---- the algorithms in 64 bits -------------------------------------------------------------------


class _Model:
    """The exit-wave model in plain torch, complex128: views' windows, plane phase, gaps between
    slices, the exit transform. Planes are natural (centred); the detector plane of the far
    field is in DFT index order, of the near field spatial."""

    def __init__(self, c, oy, ox, side):
        n = c["n"]
        self.c, self.n, self.oy, self.ox, self.side = c, n, oy, ox, side
        self.near = c["optics"] == "near"
        dev = oy.device
        pixel, lam, dist = _geometry(c)
        d = torch.arange(n, device=dev, dtype=torch.float64) - n // 2
        ph = math.pi * pixel * pixel / (lam * dist) * (d[:, None] ** 2 + d[None] ** 2)
        self.q = torch.polar(torch.ones_like(ph), torch.zeros_like(ph) if self.near else ph)
        self.curv = math.pi * pixel * pixel / (lam * dist)
        self.d = d
        f = torch.fft.fftfreq(n, device=dev, dtype=torch.float64)
        self.f = f

        def transfer(z):
            r = (f[:, None] ** 2 + f[None] ** 2) * (lam / pixel) ** 2
            return torch.polar((r < 1).double(), 2 * math.pi * z / lam
                               * torch.sqrt((1 - r).clamp(min=0)))
        self.t_exit = transfer(dist) if self.near else None
        self.t_gap = transfer(GAP) if c["slices"] > 1 else None
        self.scale = 1.0 if self.near else float(n * n)
        ar = torch.arange(n, device=dev)
        self.index = (((oy[:, None] + ar)[:, :, None]) * side + (ox[:, None] + ar)[:, None, :])

    # exit transform, unitary
    def forward(self, e):
        if self.near:
            return torch.fft.ifft2(torch.fft.fft2(e) * self.t_exit)
        return torch.fft.fft2(e, norm="ortho")

    def back(self, e):
        if self.near:
            return torch.fft.ifft2(torch.fft.fft2(e) * self.t_exit.conj())
        return torch.fft.ifft2(e, norm="ortho")

    def gap(self, w, adjoint=False):
        t = self.t_gap.conj() if adjoint else self.t_gap
        return torch.fft.ifft2(torch.fft.fft2(w) * t)

    def to_detector(self, i):
        return i if self.near else torch.fft.fftshift(i, dim=(-2, -1))

    def observed(self, counts):
        """Intensities in the detector plane's index order, NaN where masked."""
        if counts.dtype == np.uint16:
            t = torch.from_numpy(counts.astype(np.float64)).cuda()
            t[t == pa.MASKED] = math.nan
        else:
            t = torch.from_numpy(counts).cuda().double()
            t[t < 0] = math.nan
        return t if self.near else torch.fft.ifftshift(t, dim=(-2, -1))

    def read(self, plane, fr):
        """Windows [frames, n, n] of an object plane [side, side]."""
        return plane.reshape(-1)[self.index[fr]]

    def add(self, plane, fr, patches):
        """Patches [frames, n, n] added onto `plane` at the frames' corners."""
        plane.view(-1).index_add_(0, self.index[fr].reshape(-1), patches.reshape(-1))
        return plane

    def ramps(self, offs):
        """exp(-2 pi i f.d) of each frame's offset, [frames, n, n]."""
        a = -2 * math.pi * self.f
        return torch.polar(torch.ones(len(offs), self.n, self.n, device=a.device,
                                      dtype=torch.float64),
                           offs[:, 0, None, None] * a[None, :, None]
                           + offs[:, 1, None, None] * a[None, None, :])

    def exit_waves(self, objects, probe, fr, _):
        """Exit waves [frames, modes, n, n] through every slice ([1, side, side] each)."""
        w = probe[None]
        for s, o in enumerate(objects):
            w = w * self.read(o[0], fr)[:, None]
            if s + 1 < len(objects):
                w = self.gap(w)
        return w * self.q


def _batches(nframe, size, seed, epoch):
    """The engine's seeded random batches: Fisher-Yates from the end with SplitMix64 draws."""
    u = (1 << 64) - 1

    def mix(z):
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & u
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & u
        return z ^ (z >> 31)
    state, order = (seed ^ mix(epoch)) & u, list(range(nframe))
    for i in range(nframe - 1, 0, -1):
        state = (state + 0x9E3779B97F4A7C15) & u
        j = (mix(state) * (i + 1)) >> 64
        order[i], order[j] = order[j], order[i]
    return [sorted(order[s:s + size]) for s in range(0, nframe, size)]


def _sq(z):
    return z.real ** 2 + z.imag ** 2


def _amplitude(io, far, eps, floor):
    """far times sqrt(io + eps)/max or + of the modelled amplitude, unchanged where masked."""
    a = torch.sqrt(_sq(far).sum(1))
    r = torch.sqrt(io + eps) / (a.clamp(min=floor) if eps == 0 else a + eps)
    return far * torch.where(torch.isnan(io), torch.ones_like(r), r)[:, None]


def _position_directions(sums, eps):
    num, den = sums
    return num / (den + den.amax(0).clamp(min=eps))


def _position_step(offs, fr, delta):
    dx = torch.zeros_like(offs)
    dx[fr] = 0.3 * delta
    mad = (dx - dx.mean(0)).abs().mean(0)
    lim = torch.clamp(10 * mad, max=0.1)
    return offs + torch.minimum(torch.maximum(dx, -lim), lim)


class _Sampled:
    """Whole-plane Fourier sampling at sub-pixel positions and its adjoint."""

    def __init__(self, m, offs, fr):
        self.m = m
        f = torch.fft.fftfreq(m.side, device=offs.device, dtype=torch.float64)
        ty, tx = m.oy[fr] + offs[fr, 0], m.ox[fr] + offs[fr, 1]
        ang = 2 * math.pi * (ty[:, None, None] * f[None, :, None] + tx[:, None, None]
                             * f[None, None, :])
        self.e = torch.polar(torch.ones_like(ang), ang)
        self.df = 2j * math.pi * f

    def read(self, plane, axis=None):
        s = torch.fft.fft2(plane)
        if axis is not None:
            s = s * (self.df[:, None] if axis == 0 else self.df[None])
        n = self.m.n
        return torch.fft.ifft2(s * self.e)[:, :n, :n]

    def place(self, patches):
        full = torch.zeros(self.e.shape, dtype=torch.complex128, device=self.e.device)
        full[:, :self.m.n, :self.m.n] = patches
        return torch.fft.ifft2((torch.fft.fft2(full) * self.e.conj()).sum(0))


def _rpie(c, m, io, obj, probe, offs):
    a, near = 0.1, c["optics"] == "near"
    obj = obj[0, 0].clone()
    for ep in range(c["passes"]):
        for fr in _batches(c["frames"], c["batch"], 7, ep):
            sm = _Sampled(m, offs, fr) if near else None
            win = sm.read(obj) if near else m.read(obj, fr)
            w = probe * m.q
            psi = w * win[:, None]
            far = _amplitude(io[fr], m.forward(psi), 1e-7, 0)
            delta = m.back(far) - psi
            w2 = _sq(probe)
            dens = []
            for k in range(len(probe)):
                one = w2[k].expand(len(fr), -1, -1)
                if near:
                    dens.append(sm.read(sm.place(one.to(obj.dtype))).real.clamp(min=0))
                else:
                    dens.append(m.read(m.add(torch.zeros_like(obj.real), fr, one.contiguous()),
                                       fr))
            dens = torch.stack(dens, 1)
            step = w.conj() / ((1 - a) * dens + a * dens.sum(1).max()) * delta
            if near:
                d_obj = sm.place(step.sum(1))
            else:
                d_obj = m.add(torch.zeros_like(obj), fr, step.sum(1))
            o2 = _sq(win)
            wgt = (win * m.q).conj() / ((1 - a) * o2 + a * o2.amax((1, 2), keepdim=True))
            d_probe = (wgt[:, None] * delta).sum(0)
            if c["positions"] == "refine":
                num, den = [], []
                for ax in (0, 1):
                    u = sm.read(obj, ax) * w[0]
                    num.append((u.conj() * delta[:, 0]).real.sum((1, 2)))
                    den.append(_sq(u).sum((1, 2)))
                offs = _position_step(offs, fr, _position_directions(
                    (torch.stack(num, 1), torch.stack(den, 1)), 1e-6 * m.scale))
            obj = obj + d_obj
            probe = probe + d_probe / len(fr)
    return obj[None, None], probe, offs


def _lsqml(c, m, io, objects, probe, offs):
    ns, nmode, n, moved = c["slices"], c["modes"], c["n"], c["positions"] == "refine"
    obj = [o[0].clone() for o in objects]
    frames = list(range(c["frames"]))
    a_far = torch.full((c["frames"],), 0.5, dtype=torch.float64, device=probe.device)
    pre = None
    for ep in range(c["passes"]):
        illum = m.add(torch.zeros_like(obj[0].real), frames,
                      _sq(probe).sum(0).expand(c["frames"], -1, -1).contiguous())
        if pre is None:
            pre = illum * (torch.nan_to_num(io).sum((1, 2)).max() / (4 * n * n * m.scale))
        pre = (pre + illum) / 2
        for fr in _batches(c["frames"], min(c["batch"], c["frames"]), 7, ep):
            wins = [m.read(o, fr)[:, None] for o in obj]
            q = m.q
            w = probe[None]
            if moved:
                rp = m.ramps(offs[fr])[:, None]
                w = torch.fft.ifft2(torch.fft.fft2(probe)[None] * rp)
                dy, dx = offs[fr, 0, None, None], offs[fr, 1, None, None]
                ph = m.curv * (dy * (dy - 2 * m.d[None, :, None]) + dx * (dx - 2 * m.d[None, None]))
                q = (m.q * torch.polar(torch.ones_like(ph), ph))[:, None]
            inc = [w.expand(len(fr), -1, -1, -1)]
            for s in range(ns - 1):
                inc.append(m.gap(inc[-1] * wins[s]))
            psi = inc[-1] * wins[-1] * q
            far = m.forward(psi)
            ic, y = _sq(far).sum(1), io[fr]
            masked = torch.isnan(y)
            y = torch.nan_to_num(y)
            keep = (~masked).double()
            if c["cost"] == "poisson":
                af = a_far[fr]
                for _ in range(2):
                    prev = af.mean()
                    xi = (1 - y / (ic + 1e-5)) * keep
                    num = (xi * (ic - y / (1 - prev * xi))).sum((1, 2))
                    den = (xi * xi * ic).sum((1, 2))
                    af = (0.5 * prev + 0.5 * torch.where(den > 0, num / den, 0 * num)).clamp(0, 1)
                a_far[fr] = af
                fac = (1 - y / (ic + 1e-6)) * keep
            else:
                af = torch.full((len(fr),), 0.5, dtype=torch.float64, device=probe.device)
                fac = 2 * (1 - torch.sqrt(y) / (torch.sqrt(ic) + 1e-9)) * keep
            chi = m.back(far * (1 - af[:, None, None] * fac)[:, None]) - psi
            qs = [torch.ones_like(m.q)] * (ns - 1) + [q]
            chis = [chi]
            for s in range(ns - 2, -1, -1):
                chis.insert(0, m.gap(chis[0] * (qs[s + 1] * wins[s + 1]).conj(), True))
            d_obj = []
            for s in range(ns):
                t = (chis[s] * (qs[s] * inc[s]).conj()).sum(1)
                d_obj.append(m.add(torch.zeros_like(obj[s]), fr, t)
                             / torch.sqrt(pre * pre + (0.1 * pre.max()) ** 2))
            d = (qs[0] * wins[0]).conj() * chis[0]
            if moved:
                d = torch.fft.ifft2(torch.fft.fft2(d) * rp.conj())
            d_probe = d.mean(0)
            lam = 1.2e-7 * m.scale / (n * n) * nmode * n * n
            # the joint 2x2 system of slice 0 and the probe
            q0 = m.q if ns == 1 else 1.0
            u = inc[0] * m.read(d_obj[0], fr)[:, None] * (qs[0] if ns == 1 else 1.0)
            v = d_probe[None] * wins[0] * q0
            a11, a22 = _sq(u).sum((1, 2, 3)) + lam, _sq(v).sum((1, 2, 3)) + lam
            a12 = (u * v.conj()).sum((1, 2, 3))
            b1 = (u.conj() * chis[0]).real.sum((1, 2, 3))
            b2 = (v.conj() * chis[0]).real.sum((1, 2, 3))
            a11, a22 = a11 + 0.1 * a11.mean(), a22 + 0.1 * a22.mean()
            det = a11 * a22 - _sq(a12)
            a_obj = [0.9 * ((a22 * b1 - a12.real * b2) / det).clamp(min=0) / (ns * nmode)]
            a_probe = 0.9 * ((a11 * b2 - a12.real * b1) / det).clamp(min=0)
            for s in range(1, ns):
                u = inc[s] * m.read(d_obj[s], fr)[:, None] * qs[s]
                a_obj.append((0.45 * (u.conj() * chis[s]).real.sum((1, 2, 3))
                              / _sq(u).sum((1, 2, 3)) / (ns * nmode)).clamp(min=0))
            new_offs = offs
            if moved:
                s = ns // 2
                spec = torch.fft.fft2(wins[s][:, 0])
                wq = (inc[s] * qs[s])[:, 0]
                num, den = [], []
                for ff in (m.f[:, None], m.f[None]):
                    g = torch.fft.ifft2(spec * (2j * math.pi * ff)) * wq
                    num.append((g.conj() * chis[s][:, 0]).real.sum((1, 2)))
                    den.append(_sq(g).sum((1, 2)))
                new_offs = _position_step(offs, fr, _position_directions(
                    (torch.stack(num, 1), torch.stack(den, 1)), 1e-6 * m.scale))
            for s in range(ns):
                v = a_obj[s].sort()[0]
                k = int(math.ceil(len(v) * 0.1 / 2 - 0.5))
                obj[s] = obj[s] + v[k:len(v) - k].mean() * d_obj[s]
            probe = probe + a_probe.mean() * d_probe
            offs = new_offs
    return torch.stack(obj)[:, None], probe, offs


def _no_ramp(c, m, obj, probe):
    """The shared linear phase of object and probe taken out, by the probe spectrum's centre."""
    n, side = c["n"], m.side
    v = torch.fft.fftshift(_sq(torch.fft.fft2(torch.fft.ifftshift(probe, dim=(-2, -1)))).sum(0))
    k = torch.arange(n, device=v.device, dtype=torch.float64)
    dy = (v * k[:, None]).sum() / v.sum() - n // 2
    dx = (v * k[None]).sum() / v.sum() - n // 2

    def ramp(a, size, sign):
        t = sign * 2 * math.pi * (torch.arange(size, device=v.device, dtype=torch.float64)
                                  - size // 2) / n
        ph = dy * t[:, None] + dx * t[None]
        return a * torch.polar(torch.ones_like(ph), ph)
    return ramp(obj, side, 1.0), ramp(probe, n, -1.0)


def _chunks(c, size=64):
    return [list(range(s, min(c["frames"], s + size))) for s in range(0, c["frames"], size)]


def _blend(old, num, norm, inertia):
    reg = norm.amax() * inertia
    return (num + old * reg) / (norm + reg).clamp(min=1e-12)


def _project(c, m, io, obj, probe, offs):
    obj = obj[0, 0].clone()
    alg = c["alg"]
    psi = torch.zeros((c["frames"], c["modes"], c["n"], c["n"]), dtype=torch.complex128,
                      device=obj.device)

    def sums(do_obj, do_probe):
        on, od = torch.zeros_like(obj), torch.zeros_like(obj.real)
        pn, pd = torch.zeros_like(probe), torch.zeros_like(probe.real)
        for fr in _chunks(c):
            if do_obj:
                m.add(on, fr, (psi[fr] * (m.q * probe).conj()).sum(1))
                m.add(od, fr, _sq(probe).sum(0).expand(len(fr), -1, -1).contiguous())
            if do_probe:
                win = m.read(obj, fr)
                pn += (psi[fr] * (m.q * win).conj()[:, None]).sum(0)
                pd += _sq(win).sum(0)
        return on, od, pn, pd

    for cyc in range(c["passes"]):
        for fr in _chunks(c):
            po = probe * m.q * m.read(obj, fr)[:, None]
            if alg == "ap" or cyc == 0:
                it = po
            elif alg == "dm":
                it = po * 1.98 - psi[fr] * 0.98
            else:
                it = psi[fr] * 0.55 + (po * 2 - iterate[fr]) * 0.45
            out = m.back(_amplitude(io[fr], m.forward(it), 0, 1e-12))
            if alg == "dm" and cyc > 0:
                out = out + (po - it) * 0.98
            if alg == "raar":
                if cyc == 0 and fr[0] == 0:
                    iterate = torch.empty_like(psi)
                iterate[fr] = it
            psi[fr] = out
        if alg == "ap":
            on, od, pn, pd = sums(True, True)
            obj, probe = _blend(obj, on, od, 0.01), _blend(probe, pn, pd, 0.01)
        else:
            on, od, _, _ = sums(True, False)
            obj = _blend(obj, on, od, 0.01)
            _, _, pn, pd = sums(False, True)
            probe = _blend(probe, pn, pd, 0.001)
    obj, probe = _no_ramp(c, m, obj, probe)
    return obj[None, None], probe, offs


def _ml(c, m, io, obj, probe, offs):
    obj = obj[0, 0].clone()

    def field(o, p, fr):
        return m.forward(p * m.q * m.read(o, fr)[:, None])

    calc = sum((_sq(field(obj, probe, fr)).sum(1) * (~torch.isnan(io[fr]))).sum()
               for fr in _chunks(c))
    s = torch.sqrt(torch.nan_to_num(io).sum() / calc)
    os_, ps = obj.abs().sum(), probe.abs().sum()
    probe, obj = probe * torch.sqrt(os_ / ps * s), obj * torch.sqrt(ps / os_ * s)
    last, do, dp = None, torch.zeros_like(obj), torch.zeros_like(probe)
    for _ in range(c["passes"]):
        go, gp = torch.zeros_like(obj), torch.zeros_like(probe)
        for fr in _chunks(c):
            far = field(obj, probe, fr)
            r = 2 * (1 - io[fr] / _sq(far).sum(1).clamp(min=1e-12))
            g = m.back(far * torch.nan_to_num(r)[:, None])
            m.add(go, fr, (g * (m.q * probe).conj()).sum(1))
            if c["probe"]:
                gp += (g * (m.q * m.read(obj, fr)).conj()[:, None]).sum(0)
        beta = 0.0
        if last is not None:
            num = sum((a.conj() * (a - b)).real.sum() for a, b in zip((go, gp), last))
            b = float(num / sum(_sq(b).sum() for b in last))
            beta = b if math.isfinite(b) and b >= 0 else 0.0
        do, dp = do * beta - go, dp * beta - gp
        num = den = 0.0
        for fr in _chunks(c, 32):
            po, b = field(obj, probe, fr), field(do, dp, fr)
            a = field(do, probe, fr) + field(obj, dp, fr)
            calc = _sq(po).sum(1).clamp(min=1e-32)
            r = (po.conj() * a).real.sum(1)
            s = (_sq(a) + 2 * (po.conj() * b).real).sum(1)
            y = io[fr]
            d = 1 - y / calc
            num += float(torch.nan_to_num(-2 * r * d).sum())
            den += float(torch.nan_to_num(2 * s * d + y * (2 * r / calc) ** 2).sum())
        obj, probe = obj + do * (num / den), probe + dp * (num / den)
        last = (go, gp)
    obj, probe = _no_ramp(c, m, obj, probe)
    return obj[None, None], probe, offs


def _grad(c, m, io, objects, probe):
    o = objects.detach().clone().requires_grad_(True)
    p = probe.detach().clone().requires_grad_(True)
    total = 0.0
    for fr in _chunks(c):
        ic = _sq(m.forward(m.exit_waves(list(o), p, fr, None))).sum(1)
        y = io[fr]
        keep = ~torch.isnan(y)
        y, ic = y[keep], ic[keep]
        pos = y > 0
        if c["cost"] == "poisson":
            one = torch.ones_like(y)
            log = torch.where(pos, y * (torch.log(torch.where(pos, y, one))
                                        - torch.log(torch.where(pos, ic, one))), 0 * y)
            loss = (ic - torch.where(pos, y, 0 * y) + log).sum()
        else:
            loss = ((torch.sqrt(ic) - torch.sqrt(y)) ** 2).sum()
        loss.backward()
        total += float(loss.detach())
    return dict(loss=torch.tensor(total, dtype=torch.float64), objects=o.grad, probe=p.grad)


def exact(case, seed):
    c = dict(_BASE, **case)
    d = _inputs(c, seed)
    m = d["model"]
    io = m.observed(d["counts"])
    dt = torch.complex64 if c["dtype"] == "c64" else torch.complex128
    if c["alg"] == "grad":  # the call's inputs are the tensors in the case's precision
        return _grad(c, m, io, d["obj"].to(dt).to(torch.complex128),
                     d["probe"].to(dt).to(torch.complex128))
    offs = torch.from_numpy(d["offs"]).cuda()
    f = {"rpie": _rpie, "lsqml": _lsqml, "ml": _ml}.get(c["alg"], _project)
    obj, probe, offs = f(c, m, io, d["obj"], d["probe"], offs)
    out = dict(objects=obj.cpu().numpy(), probe=probe.cpu().numpy())
    if c["positions"] == "refine":
        out["position"] = offs.cpu().numpy()
    return out
