"""The spin kernels' copy of a batched handle's physics: up to 64
configurations in LDS, the table in memory above.  Lists past 32,768 particles
(one lane per particle), each configuration with its own field, against plain
handles of the first and last configuration.  Batched and plain runs form the
same operations, so the comparison is bit for bit."""
import numpy as np
import pytest

import spintrack as st
from spintrack import configs

pytestmark = pytest.mark.gpu


def options(c, n, integ):
    o = configs.he3_thermal(n=n, tf=0.01, ioutInt=0.005, seed=1000 * c + 7, integrator=integ)
    st.set_fields(o, B0=(0.0, 0.0, 3.0e-6 * (1.0 + 0.01 * c)))
    return o


@pytest.mark.parametrize("integ", [0, 2])
# (the last: past one wave per SIMD, 65,536, against plain lists below it)
@pytest.mark.parametrize("n_cfg,n", [(64, 514), (65, 509), (2, 33000)])
def test_table_in_lds_and_in_memory(n_cfg, n, integ):
    print(f"[batch table] {n_cfg} x {n} integratorType={integ}", flush=True)
    opts = [options(c, n, integ) for c in range(n_cfg)]
    times = [0.005, 0.01]
    with st.Particle.batch(opts, variant=st.VARIANT_FAST) as b:
        b.initParticles()
        b.run(times)
        bstate = b.get_state()
    for c in (0, n_cfg - 1):
        with st.Particle(opts[c], variant=st.VARIANT_FAST) as p:
            p.initParticles()
            p.run(times)
            state = p.get_state()
        for name in state.dtype.names:
            assert state[name].tobytes() == bstate[c * n:(c + 1) * n][name].tobytes(), (c, name)
