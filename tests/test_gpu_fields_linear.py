"""Edited field hooks that keep both traits (tests/fields/linear_hooks.h): the
exact variant evaluates them as written for every ensemble, whichever kernel
its size selects.  The graph-captured chunk loop runs one lane per particle at
every size, so a small ensemble of the host loop is compared with it bit for
bit."""
import os

import pytest

import spintrack as st
from spintrack import configs

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB_LINEAR = os.path.join(ROOT, "spin-tracking_amd", "libspintrack_fieldlin.so")


def final_state(integ, pulse, library, graph_chunks):
    o = configs.neutron_cell(n=64, tf=0.02, ioutInt=0.01, seed=5)
    # gradient fields of B0's size, so that their rounding reaches the spins
    st.set_fields(o, B0=(1e-7, 2e-7, -1e-7), Gx=(3e-5, -2e-5, 1e-5), Gy=(-1e-5, 2e-5, 3e-5),
                  Gz=(2e-5, 1e-5, -2e-5), yi=(0.0, 0.6, 0.8), integratorType=integ)
    if integ == 1:
        st.set_fields(o, rtol=1e-9, tf=0.004, ioutInt=0.002)
    if pulse:
        st.set_fields(o, a=1e-6, w=300.0)
    with st.Particle(o, variant=st.VARIANT_EXACT, pulse_axis=1, library=library, chunk_records=16,
                     graph_chunks=graph_chunks) as p:
        p.initParticles()
        p.run(st.output_times(o))
        return p.get_state()


@pytest.mark.parametrize("pulse", [False, True])
@pytest.mark.parametrize("integ", [0, 1])
def test_small_ensembles_evaluate_the_hooks(integ, pulse):
    print(f"[linear hooks] integratorType={integ} pulse={pulse}", flush=True)
    small = final_state(integ, pulse, LIB_LINEAR, 0)
    assert small.tobytes() == final_state(integ, pulse, LIB_LINEAR, 2).tobytes()
    # the summation order shows in the spins, so the comparison can tell
    assert small["S"].tobytes() != final_state(integ, pulse, None, 0)["S"].tobytes()
