"""Snapshot blocks of particles whose spin integration fails inside an output
interval (st_run): every block holds the stopped particle, and nothing is
written past the last block.  The buffer is followed by as many guard blocks
as a particle has intervals left, so a write past the end would land in them.
"""
import numpy as np
import pytest

import spintrack as st
from spintrack import _lib, configs

pytestmark = pytest.mark.gpu


# four lanes per particle, and one (lists above 32,768 particles)
@pytest.mark.parametrize("n", [70, 33000])
@pytest.mark.parametrize("variant", [st.VARIANT_EXACT, st.VARIANT_FAST])
def test_blocks_after_a_failure(n, variant):
    print(f"[failure blocks] n={n} variant={variant}", flush=True)
    o = configs.neutron_cell(n=n, tf=0.03, ioutInt=0.01, seed=3)
    # nearly every particle has a segment of more than four trials, in the
    # first interval or a later one
    st.set_fields(o, nmax=4)
    times = [0.01, 0.02, 0.03]
    with st.Particle(o, variant=variant, chunk_records=64) as p:
        p.initParticles()
        bb = p.block_bytes()
        buf = _lib.DeviceBuffer(2 * len(times) * bb)
        for k in range(2 * len(times)):     # the seeded ensemble in every block
            p.snapshot_block_device(buf.ptr + k * bb)
        guard = p.copy_to_host(buf.ptr + len(times) * bb, len(times) * bb)
        p.run(times, buf.ptr)
        raw = p.copy_to_host(buf.ptr, 2 * len(times) * bb)
        state = p.get_state()
        buf.free()
    assert raw[len(times) * bb:].tobytes() == guard.tobytes()
    assert np.mean(state["failure"] == -1) > 0.9
    failed = np.zeros(n, bool)
    for k in range(len(times)):
        b = raw[k * bb:(k + 1) * bb].view(st.snapshot_block_dtype(n))[0]
        now = b["failure"] == -1
        assert not np.any(failed & ~now)    # a failure stays for every later block
        failed = now
        for field in (b["t"][:, None], st.xyz(b["S"]), st.xyz(b["pos"])):
            assert np.array_equal(np.isnan(field).any(axis=1), now)
            assert np.array_equal(np.isnan(field).all(axis=1), now)
    assert np.array_equal(state["failure"] == -1, failed)
