"""The step policy of a launch (steps, tri_quarters, refill_below) is that of its own trace kind: the
path tracer's shadow rays, whose parameters start as a copy of the closest-hit launch's, included."""
import os
import re
import subprocess

import pytest

from luisacompute_amd import build

PROGRAM = r"""
#include "lc_hip_internal.h"
#include <cstdio>
using namespace lchip;
int main() {
    TraceConfig closest, any;
    closest.steps = 11; closest.tri_quarters = 1; closest.refill_below = 13;
    any.steps = 21; any.tri_quarters = 4; any.refill_below = 23;
    TraceParams C{};
    set_step_policy(C, closest);
    TraceParams A = C;
    set_step_policy(A, any);
    QueryParams Q{};
    set_step_policy(Q, any);
    std::printf("%d %u %u %d %u %u %d %u %u\n", C.steps, C.tri_quarters, C.refill_below, A.steps, A.tri_quarters,
                A.refill_below, Q.steps, Q.tri_quarters, Q.refill_below);
}
"""


def test_policy_comes_whole_from_one_configuration(tmp_path):
    src, exe = tmp_path / "policy.cpp", tmp_path / "policy"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", build.CSRC, "-I",
                    os.path.join(build.ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert out.split() == "11 1 13 21 4 23 21 4 23".split()


@pytest.mark.parametrize("name", ("runtime.cpp", "pathtracer.hip"))
def test_every_launch_takes_its_policy_whole(name):
    """Each caller of trace_launch / query_launch sets the policy with set_step_policy, for the
    configuration whose grid it launches, and no field of it by itself."""
    text = open(os.path.join(build.CSRC, name)).read()
    assert not re.findall(r"\b[A-Z]\.(?:steps|tri_quarters|refill_below)\s*=", text)
    launches = re.findall(r"(?:trace|query)_launch\((\w), ", text)
    policies = re.findall(r"set_step_policy\((\w), (\w+)\)", text)
    assert [p for p, _ in policies] == launches
    if name == "pathtracer.hip":
        assert policies == [("P", "cc"), ("A", "ca")]
