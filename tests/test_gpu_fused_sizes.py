"""The fused engine at every size that selects another kernel: exact RK45 in
one launch has a form of its own up to 65,536 particles on 1,024 SIMDs.  A run
of n particles is the start of a longer one, and of the same run with one
launch per output time, bit for bit."""
import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu


def final(n, integ, variant, persistent):
    o = configs.dressing(n=n, species="he3", tf=0.0004, ioutInt=0.0002, seed=7)
    st.set_fields(o, integratorType=integ, rtol=1e-9 if integ == 1 else 1e-12)
    times = list(st.output_times(o))
    with st.Particle(o, variant=variant, engine=_lib.ENGINE_FUSED, pulse_axis=1) as p:
        p.initParticles()
        if persistent:
            p.run(times)
        else:
            for t in times:
                p.runSimulation(t)
        return p.get_state(), p.particle_counters()


@pytest.mark.parametrize("variant", [st.VARIANT_EXACT, st.VARIANT_FAST])
@pytest.mark.parametrize("integ", [0, 1])
def test_fused_sizes_give_the_same_bits(integ, variant):
    print(f"[fused sizes] integratorType={integ} variant={variant}", flush=True)
    whole, counts = final(65601, integ, variant, True)
    for n, persistent in ((1, True), (300, True), (65536, True), (300, False)):
        s, c = final(n, integ, variant, persistent)
        for name in s.dtype.names:
            assert s[name].tobytes() == whole[name][:n].tobytes(), (n, persistent, name)
        for name in c:
            assert np.array_equal(c[name], counts[name][:n]), (n, persistent, name)
