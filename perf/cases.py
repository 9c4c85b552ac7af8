"""What a user of this framework has it compute, as cases that can be timed and compared.

A case is one whole call through the public interface (``spintrack.Particle``,
``Particle.batch``, ``adjoint.ForwardRun``): the ensemble is seeded and advanced through its
output times, and everything the program gets back is returned.  Sizes, cells, species and
integrator settings are those of this repository's workloads (``spintrack.configs``), tests and
benchmark.

Paths
  loop      the drop-in loop of mainAnalysis: runSimulation + snapshot to the host per interval
  run       the persistent form: one ``run`` over all output times, snapshot blocks on the GPU
  sweep     ``Particle.batch`` over field configurations with per-particle stop times, then the
            per-particle phase analysis of its blocks
  dressing  neutrons and He-3 co-tracked in one batch with a pulse along y
  adjoint   checkpointed forward run, then the gradient of a phase loss
  spectral  integratorType 6: the run's summed covariance spectrum and the Bloch vector
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spin-tracking_amd"))
import spintrack as st  # noqa: E402
from spintrack import adjoint as st_adjoint  # noqa: E402
from spintrack import configs  # noqa: E402

FAST, EXACT = st.VARIANT_FAST, st.VARIANT_EXACT
# integratorType: 0 DOP853, 1 RK45, 2 MagnusCFET, 3 RK45 quaternion, -1 trajectory only


def listed():
    return [
        # the smallest run a program makes: one output interval of a few dozen particles through
        # the drop-in loop (a check of a parameter file, a unit test)
        dict(name="loop_neutron_64", path="loop", species="neutron", n=64, tf=0.05, intervals=1,
             integrator=0, variant="exact", diffuse=0.0),
        # the default ensemble of the params grammar, 1000 particles, drop-in loop, default variant
        dict(name="loop_neutron_1000", path="loop", species="neutron", n=1000, tf=0.2, intervals=4,
             integrator=0, variant="exact", diffuse=0.0),
        # gas collisions, diffuse walls, an odd count, drop-in loop
        dict(name="loop_he3_2047", path="loop", species="he3", n=2047, tf=0.15, intervals=3,
             integrator=0, variant="fast", diffuse=0.05),
        # one configuration's ensemble of a field sweep, run by itself
        dict(name="run_he3_16384", path="run", species="he3", n=16384, tf=0.2, intervals=2,
             integrator=0, variant="fast", diffuse=0.05),
        # the benchmark's ensemble, one of its output intervals
        dict(name="run_he3_1M", path="run", species="he3", n=1048576, tf=0.5, intervals=1,
             integrator=0, variant="fast", diffuse=0.05),
        # the reference's published neutron runs: MagnusCFET, 65,536 neutrons, gravity, specular
        # walls, default variant
        dict(name="run_magnus_65536", path="run", species="neutron", n=65536, tf=4.0, intervals=2,
             integrator=2, variant="exact", diffuse=0.0),
        # the same integrator at the persistent loop's default variant, a small ensemble
        dict(name="run_magnus_4096", path="run", species="neutron", n=4096, tf=2.0, intervals=2,
             integrator=2, variant="fast", diffuse=0.0),
        # integratorType 1
        dict(name="run_rk45_8192", path="run", species="neutron", n=8192, tf=0.002, intervals=2,
             integrator=1, variant="fast", diffuse=0.0),
        # the reference's energy-conservation runs: trajectories only, diffuse walls
        dict(name="run_trajectory_262144", path="run", species="neutron", n=262144, tf=5.0, intervals=2,
             integrator=-1, variant="exact", diffuse=1.0),
        # field sweep in one launch, phases analysed on the GPU
        dict(name="sweep_32x2048", path="sweep", n_cfg=32, n=2048, tf=2.0, intervals=2, variant="fast"),
        # spin dressing, two species together
        dict(name="dressing_2x8192", path="dressing", n=8192, tf=0.05, intervals=2, variant="fast"),
        # a gradient step on the field coefficients
        dict(name="adjoint_8192", path="adjoint", n=8192, tf=2.0, intervals=8, variant="fast", diffuse=0.01),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for: 64 .. 524,288 particles, every
    integrator and variant above, durations so that a case stays below the largest listed one."""
    path = rng.choice(["loop", "loop", "run", "run", "run", "run", "sweep", "dressing", "adjoint", "spectral"])
    variant = rng.choice(["fast", "exact"])
    intervals = rng.randint(1, 4)
    if path == "loop" or path == "run":
        species = rng.choice(["neutron", "he3"])
        integrator = rng.choice([0, 0, 0, 2, 2, 3, 1, -1])
        n = _log_int(rng, 64, 65536) if path == "loop" else 2 * _log_int(rng, 32, 262144)
        # simulated particle-seconds a case may take: about half the largest listed case's time
        budget = {0: 1e5, 1: 1e2, 2: 1.5e5, 3: 1e5, -1: 5e5}[integrator] / (1 if species == "he3" else 0.7)
        tf = min({0: 0.4, 1: 0.002, 2: 4.0, 3: 2.0, -1: 5.0}[integrator] * (0.1 if species == "he3" else 1.0),
                 budget / n) * rng.uniform(0.5, 1.0)
        if integrator == 1:
            species, variant = "neutron", "fast"
        return dict(path=path, species=species, n=n, tf=tf, intervals=intervals, integrator=integrator,
                    variant=variant, diffuse=rng.choice([0.0, 0.05]) if species == "neutron" else 0.05)
    if path == "sweep":
        n_cfg = rng.randint(2, 64)
        n = 2 * _log_int(rng, 32, 131072 // n_cfg)
        return dict(path=path, n_cfg=n_cfg, n=n, tf=rng.uniform(0.5, 2.0), intervals=intervals, variant="fast")
    if path == "dressing":
        return dict(path=path, n=_log_int(rng, 64, 16384), tf=rng.uniform(0.01, 0.04), intervals=intervals,
                    variant=variant)
    if path == "adjoint":
        return dict(path=path, n=_log_int(rng, 64, 16384), tf=rng.uniform(0.5, 2.0), intervals=rng.randint(4, 8),
                    variant="fast", diffuse=rng.choice([0.0, 0.01]))
    return dict(path=path, n=_log_int(rng, 256, 65536), tf=rng.uniform(0.02, 0.1), intervals=intervals,
                variant="fast")


# ---------------------------------------------------------------------------------------------
# what the program has in hand: the options, the handle and the output buffer
# ---------------------------------------------------------------------------------------------
def _seed(seed):
    # particle i draws from stream seed + i: distinct ensembles need distant seeds
    return (int(seed) * 1000003 + 17) & 0x3FFFFFFF


def _options(case, seed):
    """Options block(s) of the case and its per-particle stop times (sweep only)."""
    out = case["tf"] / case["intervals"]
    s = _seed(seed)
    if case["path"] == "sweep":
        # particles stop between a tenth of the span and its end
        return configs.batched_sweep(n_cfg=case["n_cfg"], n_per=case["n"], seed=s, tf=case["tf"], ioutInt=out,
                                     dur=(0.1 * case["tf"], case["tf"]))
    if case["path"] == "dressing":
        return configs.dressing_cotracked(n=case["n"], tf=case["tf"], ioutInt=out, seed=s), None
    if case["path"] == "adjoint":
        return [configs.adjoint_case(n=case["n"], tf=case["tf"], ioutInt=out, diffuse=case["diffuse"], seed=s)], None
    if case["path"] == "spectral":
        # the benchmark's spectral drive: 3e-5 T at 1 kHz, samples every 1e-4 s
        o = configs.he3_thermal(n=case["n"], tf=case["tf"], ioutInt=out, seed=s, integrator=6)
        st.set_fields(o, a=3e-5, w=2.0 * math.pi * 1000.0, h=1e-4)
        return [o], None
    if case["species"] == "he3":
        o = configs.he3_thermal(n=case["n"], tf=case["tf"], ioutInt=out, seed=s, integrator=case["integrator"])
    else:
        o = configs.neutron_cell(n=case["n"], tf=case["tf"], ioutInt=out, seed=s)
        # spins transverse to B0, so that they precess
        st.set_fields(o, integratorType=case["integrator"], yi=(0.0, 1.0, 0.0))
    st.set_fields(o, diffuse=case["diffuse"])
    return [o], None


def _times(case):
    return np.array([(i + 1.0) * (case["tf"] / case["intervals"]) for i in range(case["intervals"])])


def prepare(case, seed):
    opts, stop_at = _options(case, seed)
    variant = FAST if case["variant"] == "fast" else EXACT
    times = _times(case)
    if case["path"] == "adjoint":
        return dict(path="adjoint", fwd=st_adjoint.ForwardRun(opts[0], variant=variant))
    if case["path"] in ("sweep", "dressing"):
        p = st.Particle.batch(opts, pulse_axis=1 if case["path"] == "dressing" else 2, variant=variant)
        if stop_at is not None:
            p.set_stop_times(stop_at)
    else:
        # large ensembles bound the record buffer (the default takes up to half the card)
        p = st.Particle(opts[0], variant=variant, seg_buffer_mb=40960 if case["n"] > 131072 else 0)
    p.initParticles()   # seeds the ensemble and allocates what the handle keeps
    blocks = None
    if case["path"] not in ("loop", "spectral"):
        blocks = torch.empty(p.block_bytes() * len(times), dtype=torch.uint8, device="cuda")
    p.synchronize()
    return dict(path=case["path"], p=p, n=p.n, times=times, blocks=blocks)


_FIELDS = (("t", 0, 8, 1, torch.float64), ("pos", 8, 24, 3, torch.float64), ("v", 32, 24, 3, torch.float64),
           ("S", 56, 24, 3, torch.float64), ("failure", 80, 4, 1, torch.int32), ("n_coll", 84, 8, 1, torch.int64),
           ("n_bounce", 92, 8, 1, torch.int64), ("n_steps", 100, 8, 1, torch.int64))


def _block_views(buf, n, k):
    """The eight arrays of snapshot block k (even n: every array is aligned)."""
    base = 108 * n * k
    out = {}
    for name, off, size, width, dtype in _FIELDS:
        a = buf[base + off * n: base + (off + size) * n].view(dtype)
        out["%d.%s" % (k, name)] = a.view(n, 3) if width == 3 else a
    return out


def run(state):
    if state["path"] == "adjoint":
        f = state["fwd"]
        means = f.run()
        _, g = st_adjoint.phase_loss(means, f.times, f.opt.t0)
        return dict(means=means, grad=f.gradient(g))
    p, n, times = state["p"], state["n"], state["times"]
    p.initParticles()
    out = {}
    if state["path"] == "loop":
        for k, t in enumerate(times):
            p.runSimulation(t)
            s = p.snapshot()
            for name in st.particle.SNAPSHOT_FIELDS:
                a = s[name]
                out["%d.%s" % (k, name)] = a.view("<f8").reshape(n, 3) if a.dtype == st.COORDS else a
        return out
    if state["path"] == "spectral":
        for t in times:
            p.runSimulation(t)
        return dict(variance=p.spectrum()["raw"], b_end=p.floquetResults())
    p.run(times, state["blocks"].data_ptr())
    for k in range(len(times)):
        out.update(_block_views(state["blocks"], n, k))
    if state["path"] == "sweep":
        out["phase"] = p.phase_stats(state["blocks"].data_ptr(), len(times))
    return out


# ---------------------------------------------------------------------------------------------
# work: particle-seconds times what one of them cannot do without
# ---------------------------------------------------------------------------------------------
# per particle-second: integrator trials and trajectory segments (counted on these ensembles),
# and the operations of one trial of each integrator and of one event
_RATES = {("neutron", 0): (2760.0, 72.0), ("he3", 0): (3060.0, 1260.0), ("neutron", 1): (6.9e5, 90.0),
          ("neutron", 2): (157.0, 68.0), ("he3", 2): (1300.0, 1260.0), ("neutron", 3): (557.0, 68.0),
          ("he3", 3): (2000.0, 1260.0), ("neutron", -1): (0.0, 68.0), ("he3", -1): (0.0, 1260.0),
          ("dressing", 0): (58400.0, 1570.0)}
_TRIAL_FLOPS = {0: 1410.0, 1: 650.0, 2: 1520.0, 3: 1000.0, -1: 0.0}
_EVENT_FLOPS = 75.0


def work(case):
    n = case["n"] * case.get("n_cfg", 2 if case["path"] == "dressing" else 1)
    # the 38 state fields written once, the snapshot blocks written once
    by = n * (38 * 8.0 + 108.0 * case["intervals"])
    if case["path"] == "spectral":
        # 17 filters of three axes per sample, a sample every 1e-4 s
        return dict(bytes=n * 38 * 8.0, flops=n * case["tf"] * (1255.0 * _EVENT_FLOPS + 1e4 * 617.0))
    integ = case.get("integrator", 0)
    species = {"sweep": "neutron", "adjoint": "neutron", "dressing": "dressing"}.get(case["path"], case.get("species"))
    trials, segs = _RATES[(species, integ)]
    seconds = n * case["tf"] * (0.55 if case["path"] == "sweep" else 1.0)
    fl = seconds * (trials * _TRIAL_FLOPS[integ] + segs * _EVENT_FLOPS)
    return dict(bytes=by, flops=2.0 * fl if case["path"] == "adjoint" else fl)


# ---------------------------------------------------------------------------------------------
# exact: the same ensembles in plain torch, 64 bits
# ---------------------------------------------------------------------------------------------
_M53 = (1 << 53) - 1


def _s64(v):
    return v - (1 << 64) if v >= 1 << 63 else v


def _lsr(a, k):
    return (a >> k) & ((1 << (64 - k)) - 1)


class _Streams:
    """One random stream per particle: splitmix64 seeding, the reference's xoshiro variant
    (src/particle.cpp:33-119), polar-method normals with a cached spare."""

    def __init__(self, seed, device):
        st_ = seed & 0xFFFFFFFF
        halves = []
        for _ in range(2):
            st_ = st_ + _s64(0x9E3779B97F4A7C15)
            r = (st_ ^ _lsr(st_, 30)) * _s64(0xBF58476D1CE4E5B9)
            r = (r ^ _lsr(r, 27)) * _s64(0x94D049BB133111EB)
            r = r ^ _lsr(r, 31)
            halves += [r & 0xFFFFFFFF, _lsr(r, 32)]
        self.x, self.y, self.z, self.w = halves
        self.spare = torch.zeros(len(seed), dtype=torch.float64, device=device)
        self.has = torch.zeros(len(seed), dtype=torch.bool, device=device)
        every = torch.arange(len(seed), device=device)
        for _ in range(3):
            self.uniform(every)

    def uniform(self, i):
        x, y, z, w = self.x[i], self.y[i], self.z[i], self.w[i]
        r = x + z
        t = y << 17
        z = z ^ x
        w = w ^ y
        y = y ^ z
        x = x ^ w
        z = z ^ t
        w = (z << 45) | _lsr(z, 19)
        self.x[i], self.y[i], self.z[i], self.w[i] = x, y, z, w
        return (_lsr(r, 11) & _M53).double() * 2.0 ** -53

    def expo(self, i, tc):
        return -tc * torch.log(1.0 - self.uniform(i))

    def normal(self, i):
        out = self.spare[i].clone()
        had = self.has[i].clone()
        self.has[i] = False
        left = i[~had]
        at = (~had).nonzero().flatten()
        while len(left):
            u = self.uniform(left) * 2.0 + -1.0
            v = self.uniform(left) * 2.0 + -1.0
            s = u * u + v * v
            ok = (s < 1.0) & (s != 0.0)
            f = torch.sqrt(-2.0 * torch.log(s[ok]) / s[ok])
            self.spare[left[ok]] = v[ok] * f
            self.has[left[ok]] = True
            out[at[ok]] = u[ok] * f
            left, at = left[~ok], at[~ok]
        return out


def _cross(a, b):
    return torch.stack([a[..., 1] * b[..., 2] - a[..., 2] * b[..., 1], a[..., 2] * b[..., 0] - a[..., 0] * b[..., 2],
                        a[..., 0] * b[..., 1] - a[..., 1] * b[..., 0]], -1)


def _qmul(a, b):
    aw, av, bw, bv = a[..., :1], a[..., 1:], b[..., :1], b[..., 1:]
    return torch.cat([aw * bw - (av * bv).sum(-1, keepdim=True), aw * bv + bw * av + _cross(av, bv)], -1)


class _Fields:
    """gamma*B of one particle each: B0 + G r + v x E / c^2 + a cos(w t) along one axis."""

    def __init__(self, opts, counts, axis, device):
        def per(values):
            a = torch.tensor(np.array(values, dtype=np.float64), device=device)
            return a.repeat_interleave(torch.tensor(counts, device=device), 0)
        self.gamma = per([o.gamma for o in opts])
        self.B0 = per([[*o.B0] for o in opts])
        self.E = per([[*o.E] for o in opts])
        self.G = per([[[*o.Gx], [*o.Gy], [*o.Gz]] for o in opts])
        self.a, self.w = per([o.a for o in opts]), per([o.w for o in opts])
        self.axis = axis
        self.pulse = any(o.a != 0.0 for o in opts)
        self.w_max = max(o.w for o in opts) if self.pulse else 0.0

    def turn(self, S, t0, p0, v0, ay, dt):
        """S after a segment of length dt: sixth-order Magnus steps on S' = S x gamma*B, all
        steps of all particles at once, their rotations multiplied pairwise."""
        rate = float(self.gamma.abs().max()) * float((self.B0.norm(dim=-1) + self.a.abs()).max())
        longest = float(dt.max())
        m = 1 << max(2, math.ceil(math.log2(max(1.0, longest * max(rate / 0.25, self.w_max / 0.2)))))
        rows = max(1, (1 << 24) // m)
        return torch.cat([self._turn(S[i:i + rows], t0[i:i + rows], p0[i:i + rows], v0[i:i + rows], ay,
                                     dt[i:i + rows], m, slice(i, i + rows)) for i in range(0, len(S), rows)])

    def _turn(self, S, t0, p0, v0, ay, dt, m, at):
        h = (dt / m)[:, None]
        k = torch.arange(m, dtype=torch.float64, device=S.device)[None, :]
        root = math.sqrt(15.0) / 10.0
        acc = torch.zeros(3, dtype=torch.float64, device=S.device)
        acc[1] = ay
        samples = []
        for c in (0.5 - root, 0.5, 0.5 + root):
            tau = ((k + c) * h)[..., None]
            r = p0[:, None] + tau * (v0[:, None] + 0.5 * tau * acc)
            v = v0[:, None] + tau * acc
            B = self.B0[at][:, None] + sum(self.G[at][:, None, :, j] * r[..., None, j] for j in range(3))
            B = B + _cross(v, self.E[at][:, None].expand_as(v)) / 299792458.0 ** 2
            if self.pulse:
                t = t0[:, None] + tau[..., 0]
                B[..., self.axis] += self.a[at][:, None] * torch.cos(self.w[at][:, None] * t)
            samples.append(-self.gamma[at][:, None, None] * B)
        h = h[..., None]
        a1 = h * samples[1]
        a2 = math.sqrt(15.0) / 3.0 * h * (samples[2] - samples[0])
        a3 = 10.0 / 3.0 * h * (samples[2] - 2.0 * samples[1] + samples[0])
        c1 = _cross(a1, a2)
        c2 = _cross(a1, 2.0 * a3 + c1) / -60.0
        om = a1 + a3 / 12.0 + _cross(-20.0 * a1 - a3 + c1, a2 + c2) / 240.0
        half = 0.5 * om.norm(dim=-1, keepdim=True)
        q = torch.cat([torch.cos(half), 0.5 * om * torch.sinc(half / math.pi)], -1)
        while q.shape[1] > 1:
            q = _qmul(q[:, 1::2], q[:, 0::2])   # the later step acts after the earlier one
        q = q[:, 0]
        t = 2.0 * _cross(q[:, 1:], S)
        return S + q[:, :1] * t + _cross(q[:, 1:], t)


def _sgn(v):
    return torch.where(v < 0, -1.0, 1.0).double()


def _trajectories(opts, times, stop_at, axis, spin):
    """The ensemble at each output time: the event loop of src/particle.cpp:712-837 over all
    particles at once, one event each per pass."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    counts = [int(o.numParticles) for o in opts]
    n = sum(counts)
    o = opts[0]
    seeds = torch.cat([torch.arange(c, device=dev) + int(q.seed) for q, c in zip(opts, counts)])

    def per(values):
        return torch.tensor(np.array(values, dtype=np.float64), device=dev).repeat_interleave(torch.tensor(counts, device=dev), 0)
    rng = _Streams(seeds, dev)
    every = torch.arange(n, device=dev)
    L = torch.tensor([*o.L], dtype=torch.float64, device=dev)
    kt, tc, diffuse, V = (per([getattr(q, f) for q in opts]) for f in ("sqrtKT_m", "tc", "diffuse", "V"))
    pos = torch.stack([rng.uniform(every) * L[c] - L[c] / 2.0 for c in range(3)], -1)
    gas = rng.expo(every, tc) if o.gas_coll else torch.full((n,), 1.7976931348623157e308, dtype=torch.float64, device=dev)
    v = torch.stack([rng.normal(every) for _ in range(3)], -1)
    v = v * kt[:, None] if o.dist == b"M" else V[:, None] * v / torch.sqrt(v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1] + v[:, 2] * v[:, 2])[:, None]
    S = per([[*q.yi] for q in opts])
    F = _Fields(opts, counts, axis, dev)
    t = torch.full((n,), float(o.t0), dtype=torch.float64, device=dev)
    g = -9.81
    stop = torch.full((n,), math.inf, dtype=torch.float64, device=dev) if stop_at is None else torch.tensor(stop_at, device=dev)
    prev, out = float(o.t0), []
    inf6 = torch.tensor(1e6, dtype=torch.float64, device=dev)
    for target in times:
        tf = torch.minimum(stop, torch.full_like(stop, float(target)))
        busy = prev < stop
        while bool(busy.any()):
            d = _sgn(v) * L / 2.0 - pos
            dt = d / v
            y2 = v[:, 1] * v[:, 1]
            # under gravity: falling to the floor, over the apex to the floor, or up to the ceiling
            fall = _sgn(v[:, 1]) <= 0.0
            top = -0.5 * y2 / g + pos[:, 1] >= 0.5 * L[1]
            t1 = -v[:, 1] / g
            high = pos[:, 1] + v[:, 1] * t1 + 0.5 * g * t1 * t1
            arg = torch.where(fall, -2.0 * g * (pos[:, 1] + L[1] * 0.5) + y2,
                              torch.where(top, y2 - 2.0 * g * (pos[:, 1] - 0.5 * L[1]), (-0.5 * L[1] - high) * 2.0 / g))
            root = torch.sqrt(arg)
            both = torch.minimum((-(root + v[:, 1]) / g).abs(), ((root - v[:, 1]) / g).abs())
            dty = torch.where(fall | top, both, t1 + root)
            dtx, dtz = dt[:, 0], dt[:, 2]
            bx = (dtx < 1e-16) | dtx.isnan()
            by = ~bx & ((dty < 1e-16) | dty.isnan())
            bz = ~bx & ~by & ((dtz < 1e-16) | dtz.isnan())
            walls = torch.stack([torch.where(bx, inf6, dtx), torch.where(by, inf6, dty), torch.where(bz, inf6, dtz)], -1)
            tb, wall = walls.min(-1)
            tgas = gas - t
            is_gas = tgas < tb
            tcol = torch.where(is_gas, tgas, tb)
            end = tf - t <= o.maxPosStep
            tnone = torch.where(end, tf - t, torch.full_like(t, o.maxPosStep))
            hit = tcol <= tnone
            step = torch.where(hit, tcol, tnone)
            done = end & (~hit | (tcol == tnone))
            step = torch.where(busy, step, torch.zeros_like(step))
            if spin:
                S = torch.where(busy[:, None], F.turn(S, t, pos, v, g, step), S)
            dd = step[:, None]
            new = pos + v * dd
            new[:, 1] = (pos[:, 1] + v[:, 1] * step) + ((0.5 * g) * step) * step
            nv = v.clone()
            nv[:, 1] = v[:, 1] + g * step
            pos = torch.where(busy[:, None], new, pos)
            v = torch.where(busy[:, None], nv, v)
            t = torch.where(busy, t + step, t)
            # walls: snap, then mirror or re-emit
            w = (busy & hit & ~is_gas).nonzero().flatten()
            c = wall[w]
            pos[w, c] = _sgn(pos[w, c]) * L[c] * 0.5
            speed = torch.sqrt(v[:, 0] * v[:, 0] + v[:, 1] * v[:, 1] + v[:, 2] * v[:, 2])
            rough = torch.zeros_like(w, dtype=torch.bool)
            can = diffuse[w] > 1.17549435082228750797e-38
            if bool(can.any()):
                rough[can] = rng.uniform(w[can]) < diffuse[w[can]]
            m, cm = w[~rough], c[~rough]
            v[m, cm] = v[m, cm] * -1.0
            r, cr = w[rough], c[rough]
            if len(r):
                phi = torch.acos(torch.sqrt(rng.uniform(r)))
                theta = rng.uniform(r) * 2.0 * math.pi
                vel = speed[r]
                n1 = vel * torch.sin(phi) * torch.cos(theta)
                n2 = vel * torch.sin(phi) * torch.sin(theta)
                along = -1.0 * _sgn(v[r, cr]) * vel * torch.cos(phi)
                v[r] = torch.stack([torch.where(cr == 0, along, n1),
                                    torch.where(cr == 0, -n1, torch.where(cr == 1, along, n2)),
                                    torch.where(cr == 2, along, n2)], -1)
            gi = (busy & hit & is_gas).nonzero().flatten()
            if len(gi):
                gas[gi] += rng.expo(gi, tc[gi])
                v[gi] = torch.stack([rng.normal(gi) for _ in range(3)], -1) * kt[gi][:, None]
            busy = busy & ~done
        prev = float(target)
        out.append(dict(t=t.clone(), pos=pos.clone(), v=v.clone(), S=S.clone()))
    return out


def _passes(case):
    """Passes of the event loop above: events of the busiest particles, about twice the mean."""
    he3 = case["path"] in ("dressing",) or case.get("species") == "he3"
    per_s = {"dressing": 2600.0}.get(case["path"], 1500.0 if he3 else 260.0)
    return per_s * case["tf"] + 20 * case["intervals"]


def exact(case, seed):
    if case["path"] == "spectral":
        return None   # the Floquet frequencies of the drive come from the library
    n = case["n"] * case.get("n_cfg", 2 if case["path"] == "dressing" else 1)
    turns = {"dressing": 64.0}.get(case["path"], 8.0 if case.get("species") == "he3" else 32.0)
    spin = case.get("integrator", 0) >= 0
    # ~4 ms of launches per pass, and the memory its tensors go through
    if n > 65536 or _passes(case) * (4e-3 + n * (3e3 + (turns * 2e3 if spin else 0.0)) / 2e12) > 18.0:
        return None
    opts, stop_at = _options(case, seed)
    snaps = _trajectories(opts, _times(case), stop_at, 1 if case["path"] == "dressing" else 2, spin)
    if case["path"] == "adjoint":
        return dict(means=torch.stack([s["S"].mean(0) for s in snaps]).cpu().numpy(), grad=None)
    out = {}
    for k, s in enumerate(snaps):
        for name, *_ in _FIELDS:
            out["%d.%s" % (k, name)] = s[name].cpu().numpy() if name in s else None
    if case["path"] == "sweep":
        out["phase"] = None
    return out
