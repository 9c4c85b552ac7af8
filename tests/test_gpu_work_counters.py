"""st_work_counters is the sum of the particles' counters, whichever kernels ran
and however many workgroups they had (each adds to one of several copies)."""
import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu


# four lanes per particle; one (64 or more workgroups each); the fused engine
@pytest.mark.parametrize("engine,n", [(_lib.ENGINE_PIPELINE, 1), (_lib.ENGINE_PIPELINE, 5000),
                                      (_lib.ENGINE_PIPELINE, 70001), (_lib.ENGINE_FUSED, 70001)])
def test_work_counters_are_the_particles_sums(engine, n):
    print(f"[work counters] engine={engine} n={n}", flush=True)
    o = configs.he3_thermal(n=n, tf=0.004, ioutInt=0.002)
    with st.Particle(o, variant=st.VARIANT_FAST, engine=engine) as p:
        p.initParticles()
        for t in st.output_times(o):
            p.runSimulation(t)
        w, c, steps = p.work_counters(), p.particle_counters(), p.snapshot()["n_steps"]
        assert w["accepted"] == c["accepted"].sum() > 0
        assert w["rejected"] == c["rejected"].sum()
        assert w["segments"] == c["segments"].sum() >= n
        if engine == _lib.ENGINE_PIPELINE:
            assert w["events"] == steps.astype(np.int64).sum()
        p.initParticles()       # a new ensemble starts from zero
        assert all(v == 0 for v in p.work_counters().values())
