"""The adjoint's walk back at every list size: four lanes per particle with
several particles in a wave (k_adj_quad, up to 32,768 particles) and one lane
per particle (k_adj), batched and plain.  The gradient's sums run over blocks
whose number follows the largest configuration, so batches of equal
configurations are compared, bit for bit."""
import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu


def options(kind, n, seed, beta=0.0):
    if kind == "dressing":
        o = configs.dressing(n=n, species="he3", tf=0.008, ioutInt=0.004, seed=seed)
    else:
        o = configs.adjoint_case(n=n, tf=0.06, ioutInt=0.03, seed=seed)
    return st.set_fields(o, beta=beta)


def gradient(cfgs):
    """(configurations, 15); cfgs: one Options (a plain handle) or a list"""
    first = cfgs[0] if isinstance(cfgs, list) else cfgs
    axis = 1 if first.a else 2
    times = list(st.output_times(first))
    count = len(cfgs) if isinstance(cfgs, list) else 1
    seeds = np.tile(np.linspace(-1.0, 1.0, 3 * len(times)).reshape(1, len(times), 3), (count, 1, 1))
    kw = dict(variant=st.VARIANT_FAST, pulse_axis=axis, chunk_records=16)
    with (st.Particle.batch(cfgs, **kw) if isinstance(cfgs, list) else st.Particle(cfgs, **kw)) as p:
        p.set_checkpointing(True)
        p.initParticles()
        buf = _lib.DeviceBuffer(p.block_bytes() * len(times))
        p.run(times, buf.ptr)
        g = p.adjoint(buf.ptr, seeds)
        buf.free()
    assert np.all(np.isfinite(g)) and np.all(np.any(g != 0.0, axis=1))
    return g


# 2,050 particles: four in a wave; 24,585: sixteen.  With 33 and 5
# configurations the same ones run on one lane each.
@pytest.mark.parametrize("beta", [0.0, 0.04])
@pytest.mark.parametrize("kind", ["neutron", "dressing"])
@pytest.mark.parametrize("n,few,many", [(1025, 2, 33), (8195, 3, 5)])
def test_full_waves_equal_one_lane(kind, n, few, many, beta):
    print(f"[adjoint sizes] {kind} n={n} x {few} and {many} beta={beta}", flush=True)
    cfgs = [options(kind, n, 11 + n * c, beta) for c in range(many)]
    assert gradient(cfgs[:few]).tobytes() == gradient(cfgs)[:few].tobytes()


# one lane per particle: a plain handle against the batched form
@pytest.mark.parametrize("kind", ["neutron", "dressing"])
def test_plain_one_lane_equals_batched(kind):
    print(f"[adjoint sizes] {kind} plain", flush=True)
    big, other = options(kind, 33001, 11), options(kind, 17, 90000)
    assert gradient(big)[0].tobytes() == gradient([big, other])[0].tobytes()


# The controller's general form (beta != 0) takes other steps to the same
# gradient: steps of 1e-12 each, some hundreds of them, of sums that cancel by
# less than two digits.
@pytest.mark.parametrize("kind", ["neutron", "dressing"])
def test_beta_changes_steps_only(kind):
    print(f"[adjoint sizes] {kind} beta", flush=True)
    g, gb = gradient(options(kind, 300, 11))[0], gradient(options(kind, 300, 11, 0.04))[0]
    for part in (slice(0, 9), slice(9, 12), slice(12, 15)):
        assert np.abs(g[part] - gb[part]).max() <= 1e-8 * np.abs(g[part]).max()
    assert g.tobytes() != gb.tobytes()
