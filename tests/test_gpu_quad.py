"""Four lanes per particle against one (csrc/st_quad.h): a small ensemble runs
on the quad kernels, and the same particles as one configuration of a batch
too large for them run on the one-lane kernels.  Both form every value by the
same operations, so states, counters and snapshots are equal bit for bit."""
import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu

FILLER = 33000      # with it, the batch is past the quad kernels' 32,768


def options(kind, n, seed, integ=0):
    if kind == "dressing":
        o = configs.dressing(n=n, species="he3", tf=0.008, ioutInt=0.004, seed=seed)
    elif kind == "he3":
        o = configs.he3_thermal(n=n, tf=0.02, ioutInt=0.01, seed=seed)
    else:
        o = configs.neutron_cell(n=n, tf=0.06, ioutInt=0.03, seed=seed)
        st.set_fields(o, yi=(0.0, 1.0, 0.0))
    if integ == 1:      # RK45: far more steps per second at a loose tolerance already
        st.set_fields(o, integratorType=1, rtol=1e-9, tf=o.tf / 20.0, ioutInt=o.ioutInt / 20.0)
    if integ == 2:      # MagnusCFET: steps of tens of radians on the neutrons' smooth field
        st.set_fields(o, integratorType=2, rtol=1e-6)
    return o


def run(p, times):
    p.initParticles()
    bb = p.block_bytes()
    buf = _lib.DeviceBuffer(bb * len(times))
    p.run(times, buf.ptr)
    raw = p.copy_to_host(buf.ptr, bb * len(times))
    buf.free()
    return p.get_state(), p.particle_counters(), raw, bb


# 1; a ragged wave; one particle past one per SIMD (two per wave)
@pytest.mark.parametrize("n", [1, 17, 1025])
@pytest.mark.parametrize("kind,variant", [("he3", st.VARIANT_FAST), ("dressing", st.VARIANT_FAST),
                                          ("neutron", st.VARIANT_FAST), ("he3", st.VARIANT_EXACT),
                                          ("dressing", st.VARIANT_EXACT), ("neutron", st.VARIANT_EXACT)])
@pytest.mark.parametrize("integ", [0, 1])
def test_quad_equals_one_lane(kind, variant, n, integ):
    print(f"[quad] {kind} variant={variant} n={n} integratorType={integ}", flush=True)
    axis = 1 if kind == "dressing" else 2
    small, filler = options(kind, n, 11, integ), options(kind, FILLER, 5000, integ)
    times = list(st.output_times(small))
    with st.Particle(small, variant=variant, pulse_axis=axis) as p:
        state, cnt, raw, bb = run(p, times)
    with st.Particle.batch([small, filler], variant=variant, pulse_axis=axis, chunk_records=64) as b:
        bstate, bcnt, braw, bbb = run(b, times)
    for name in state.dtype.names:
        assert state[name].tobytes() == bstate[:n][name].tobytes(), name
    for name, v in cnt.items():
        assert np.array_equal(v, bcnt[name][:n]), name
    for k in range(len(times)):
        x = raw[k * bb:(k + 1) * bb].view(st.snapshot_block_dtype(n))[0]
        y = braw[k * bbb:(k + 1) * bbb].view(st.snapshot_block_dtype(n + FILLER))[0]
        for name in x.dtype.names:
            assert x[name].tobytes() == y[name][:n].tobytes(), (k, name)


# MagnusCFET has quads in its fast variant only
@pytest.mark.parametrize("n", [1, 17, 1025])
@pytest.mark.parametrize("kind", ["he3", "dressing", "neutron"])
def test_magnus_quad_equals_one_lane(kind, n):
    test_quad_equals_one_lane(kind, st.VARIANT_FAST, n, 2)


# the walk back (k_adj_quad against k_adj): gradients of one configuration
@pytest.mark.parametrize("kind,n", [("neutron", 1), ("neutron", 70), ("dressing", 17)])
def test_quad_adjoint_equals_one_lane(kind, n):
    print(f"[quad adjoint] {kind} n={n}", flush=True)
    axis = 1 if kind == "dressing" else 2
    small, filler = options(kind, n, 11), options(kind, FILLER, 5000)
    times = list(st.output_times(small))
    seeds = np.linspace(-1.0, 1.0, 3 * len(times)).reshape(1, len(times), 3)

    def gradient(p, s):
        p.set_checkpointing(True)
        p.initParticles()
        buf = _lib.DeviceBuffer(p.block_bytes() * len(times))
        p.run(times, buf.ptr)
        g = p.adjoint(buf.ptr, s)
        buf.free()
        return g

    with st.Particle(small, variant=st.VARIANT_FAST, pulse_axis=axis, chunk_records=8) as p:
        g = gradient(p, seeds)
    with st.Particle.batch([small, filler], variant=st.VARIANT_FAST, pulse_axis=axis, chunk_records=8) as b:
        gb = gradient(b, np.concatenate([seeds, seeds]))
    assert np.all(np.isfinite(g)) and np.any(g != 0.0)
    assert g[0].tobytes() == gb[0].tobytes()
