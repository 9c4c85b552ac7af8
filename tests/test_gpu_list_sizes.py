"""One ensemble at every size that selects another kernel.  A particle's
stream depends on its index alone, so a run of n particles is the start of a
longer one, and every kernel form gives the same bits.  On 1,024 SIMDs:

    n         spin kernel (integratorTypes 0, 1, fast 2)     k_kin
    4,099     four lanes per particle,  8 particles a wave    8 a wave
    8,195     the same,                16 a wave (ragged)    16 a wave
    32,767    the same, two waves per SIMD                   32 a wave
    40,001    one lane per particle (fast DOP853: k_spin_lone) 64 a wave
    65,601    one lane per particle, a second wave per SIMD    64 a wave
"""
import functools

import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu

SIZES = (4099, 8195, 32767, 40001)
LARGE = 65601


def options(kind, integ, extra, n, seed=11):
    if kind == "dressing":
        o = configs.dressing(n=n, species="he3", tf=0.004, ioutInt=0.002, seed=seed)
    elif kind == "he3":
        o = configs.he3_thermal(n=n, tf=0.01, ioutInt=0.005, seed=seed)
    else:
        o = configs.neutron_cell(n=n, tf=0.03, ioutInt=0.015, seed=seed)
        st.set_fields(o, yi=(0.0, 1.0, 0.0))
    if integ == 1:
        st.set_fields(o, integratorType=1, rtol=1e-9, tf=o.tf / 20.0, ioutInt=o.ioutInt / 20.0)
    if integ == 2:
        st.set_fields(o, integratorType=2, rtol=1e-6)
    return st.set_fields(o, **dict(extra))


def run(p, times):
    """state, counters and snapshot blocks of a run of one chunk"""
    p.initParticles()
    p.kernel_timing(True)
    bb = p.block_bytes()
    buf = _lib.DeviceBuffer(bb * len(times))
    p.run(times, buf.ptr)
    raw = p.copy_to_host(buf.ptr, bb * len(times))
    buf.free()
    assert p.kernel_times()["kin_launches"] == 1     # the list is never shorter than the ensemble
    blocks = [raw[k * bb:(k + 1) * bb].view(st.snapshot_block_dtype(p.n))[0] for k in range(len(times))]
    return p.get_state(), p.particle_counters(), blocks


def plain(kind, variant, integ, extra, n):
    o = options(kind, integ, extra, n)
    with st.Particle(o, variant=variant, pulse_axis=1 if kind == "dressing" else 2, chunk_records=256) as p:
        return run(p, list(st.output_times(o)))


large = functools.lru_cache(maxsize=1)(lambda *a: plain(*a, LARGE))


def same(small, whole, n):
    (s, c, b), (ws, wc, wb) = small, whole
    for name in s.dtype.names:
        assert s[name][:n].tobytes() == ws[name][:n].tobytes(), name
    for name in c:
        assert np.array_equal(c[name][:n], wc[name][:n]), name
    for k in range(len(b)):
        for name in b[k].dtype.names:
            assert b[k][name][:n].tobytes() == wb[k][name][:n].tobytes(), (k, name)


EXACT, FAST = st.VARIANT_EXACT, st.VARIANT_FAST
BETA = (("beta", 0.04),)
KEEP = (("keepStepSize", True),)
NMAX = (("nmax", 4),)
ONE = (("nmax", 1),)
HMIN = (("hmin", 5e-4),)            # rejected first steps fall below it
CASES = [(kind, v, integ, ()) for integ in (0, 1) for kind in ("neutron", "he3", "dressing") for v in (EXACT, FAST)]
CASES += [(kind, FAST, 2, ()) for kind in ("neutron", "he3", "dressing")]
CASES += [(kind, v, 0, BETA) for kind in ("neutron", "dressing") for v in (EXACT, FAST)]
CASES += [("he3", v, 0, e) for e in (KEEP, NMAX, (("fixedStepSize", True), ("h", 2e-4), ("hmin", 2e-4)))
          for v in (EXACT, FAST)]
CASES += [("neutron", v, 1, e) for e in (KEEP, NMAX, HMIN, (("fixedStepSize", True), ("h", 2e-5), ("hmin", 2e-5)))
          for v in (EXACT, FAST)]
CASES += [("neutron", FAST, 2, ONE)]        # (its segments take few trials)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("case", range(len(CASES)))
def test_every_list_size_gives_the_same_bits(case, n):
    print(f"[list sizes] {CASES[case]} n={n}", flush=True)
    same(plain(*CASES[case], n), large(*CASES[case]), n)
    if CASES[case][3] in (NMAX, ONE, HMIN):
        assert np.any(large(*CASES[case])[0]["failure"] < 0)


# the batched one-lane kernels past 65,536 particles, two waves per SIMD
@pytest.mark.parametrize("variant", [EXACT, FAST])
@pytest.mark.parametrize("kind", ["he3", "dressing"])
def test_batched_past_a_wave_per_simd(kind, variant):
    n = 4099
    print(f"[list sizes] batched {kind} variant={variant}", flush=True)
    cfgs = [options(kind, 0, (), n), options(kind, 0, (), 62000, seed=5000)]
    with st.Particle.batch(cfgs, variant=variant, pulse_axis=1 if kind == "dressing" else 2, chunk_records=256) as b:
        whole = run(b, list(st.output_times(cfgs[0])))
    same(plain(kind, variant, 0, (), n), whole, n)


# overflow pages with several particles in a k_kin wave: 16 (9,000) and 32 (17,000)
@pytest.mark.parametrize("kind,n,mb", [("neutron", 9000, 62), ("he3", 17000, 117)])
def test_overflow_pages_with_full_waves(kind, n, mb):
    print(f"[list sizes] overflow pages {kind} n={n}", flush=True)
    o = (configs.neutron_cell(n=n, tf=2.0, ioutInt=0.5) if kind == "neutron" else
         configs.he3_thermal(n=n, tf=0.1, ioutInt=0.025))
    times = list(st.output_times(o))

    def go(**kw):
        with st.Particle(o, variant=FAST, **kw) as p:
            p.initParticles()
            p.run(times)
            return p.get_state(), p.particle_counters()

    s, c = go(seg_buffer_mb=mb)             # depth 112 and a pool of a quarter as many records
    s_deep, c_deep = go(chunk_records=1024)
    assert np.mean(c_deep["segments"] > 112) > 0.25
    for name in s.dtype.names:
        assert s[name].tobytes() == s_deep[name].tobytes(), name
    for name in c:
        assert np.array_equal(c[name], c_deep[name]), name
