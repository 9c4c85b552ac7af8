"""The Lund-stabilised step-size controller of DOP853 (the reference's `beta`
option, 0 by default; in the loop of src/integrator.cpp:128-247) against the oracle, in both
variants, on the kernels with four lanes per particle and with one."""
import pytest

import spintrack as st
from spintrack import configs
from test_gpu_parity import compare, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [st.VARIANT_EXACT, st.VARIANT_FAST])
@pytest.mark.parametrize("kind", ["neutron", "dressing"])
def test_beta_matches_oracle(oracle, kind, variant):
    print(f"[beta] {kind} variant={variant}", flush=True)
    axis = 1 if kind == "dressing" else 2
    if kind == "dressing":
        o = configs.dressing(n=128, species="n", tf=0.02, ioutInt=0.00624)
        st.set_fields(o, gas_coll=False, diffuse=0.0)
    else:
        o = configs.neutron_cell(n=128, tf=0.2, ioutInt=0.1)
        st.set_fields(o, yi=(0.0, 0.6, 0.8))
    st.set_fields(o, beta=0.04)
    targets = st.output_times(o)
    E = run_oracle(oracle, o, targets, pulse_axis=axis)
    for graph in (0, 2):        # the captured loop: one lane per particle
        with st.Particle(o, variant=variant, pulse_axis=axis, graph_chunks=graph, chunk_records=64) as p:
            p.initParticles()
            p.run(targets)
            print(f"  graph_chunks={graph}:", compare(oracle, p.snapshot(), p.get_state(), p.particle_counters(), E),
                  flush=True)
