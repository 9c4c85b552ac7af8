"""Which field hooks the exact variant's four-lane kernels may stand in for
(fields_by_component, csrc/st_device.h): hooks whose every component is formed
by the default hooks' operations, however they are written, and no others,
whatever the traits say.  Built for the host by hipcc with the library's
optimisation level; no GPU is used.
"""
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = "/opt/rocm/bin/hipcc"
FIELDS = os.path.join(ROOT, "tests", "fields")

HEAD = """
#define ST_FIELDS_GRAD_LINEAR 1
#define ST_FIELDS_PULSE_COS_AXIS 1
"""
PULSE = """
ST_FIELD_FN void st_field_pulse(double t, double a, double w, int axis, double B[3]) {
    for (int i = 0; i < 3; ++i) B[i] = i == axis ? a * cos(w * t) : 0.0;
}
"""
GRAD = """
ST_FIELD_FN void st_field_grad(const double r[3], const double G[9], double B[3]) {
    for (int i = 0; i < 3; ++i) {
        double s = G[3 * i] * r[0];
        for (int j = 1; j < 3; ++j) s += G[3 * i + j] * r[j];
        B[i] = s;
    }
}
"""


def row(i, expr):
    """the default gradient with component i replaced"""
    return GRAD.replace("}\n}\n", "}\n    B[%d] = %s;\n}\n" % (i, expr))


CASES = {
    "default": (None, True),
    # the same operations, written as loops
    "loops": (HEAD + GRAD + PULSE, True),
    "linear_hooks.h": (os.path.join(FIELDS, "linear_hooks.h"), False),
    "quadratic_hooks.h": (os.path.join(FIELDS, "quadratic_hooks.h"), False),
    # edits that left the traits at 1
    "one term more": (HEAD + row(2, "B[2] + 1e-9 * r[0] * r[0]") + PULSE, False),
    "symmetric G": (HEAD + row(1, "r[0] * G[1] + r[1] * G[4] + r[2] * G[5]") + PULSE, False),
    "one region": (HEAD + row(0, "r[2] > 0.1 ? 0.0 : B[0]") + PULSE, False),
    "rotating pulse": (HEAD + GRAD + PULSE.replace(": 0.0", ": a * sin(w * t)"), False),
    "pulse of -0": (HEAD + GRAD + PULSE.replace(": 0.0", ": -0.0"), False),
}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("name", list(CASES))
def test_hooks_are_recognised(tmp_path, name):
    hooks, expected = CASES[name]
    flags = []
    if hooks is not None:
        path = hooks
        if not os.path.exists(hooks):
            path = str(tmp_path / "hooks.h")
            with open(path, "w") as f:
                f.write(hooks)
        flags = [f'-DST_FIELDS_FILE="{path}"']
    exe = str(tmp_path / "host_fields")
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O3", "-std=c++17", "-ffp-contract=off", "-w", *flags,
                    os.path.join(ROOT, "tests", "host_fields_main.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True)
    assert r.stdout.strip() == ("1" if expected else "0")
