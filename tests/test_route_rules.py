"""Which kernels a pass takes: the host rules of fft_launch.hpp,
fft_two_launch.hpp and exec.hpp, evaluated on the CPU by
tests/cpp/route_rules.cpp."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    hipcc = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
    exe = str(tmp_path_factory.mktemp("rules") / "route_rules")
    subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-O0", "-w",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    os.path.join(HERE, "cpp", "route_rules.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return dict(line.split(" ", 1) for line in out.splitlines())


def test_measured_c2c_choice_leaves_the_fused_passes(rules):
    """A C2C tile that MEASURE preferred (s4v >= -2, not forced) does not move
    the axis's multiply and derivative off the mixed-radix kernels; a choice
    made by hand does."""
    for s4v in (-2, 0):
        for mode in ("mult", "deriv"):
            assert rules[f"mix512_f64_{mode}_{s4v}_0"] == "1"
            assert rules[f"mix512_f64_{mode}_{s4v}_1"] == "0"
        for prec in ("f32", "f64"):
            assert rules[f"mix512_{prec}_c2c_{s4v}_0"] == "0"
    for prec in ("f32", "f64"):
        assert rules[f"mix512_{prec}_c2c_-1_0"] == "1"
    # (the FP32 fused passes of 512 points stay with the two-level tiles)
    assert rules["mix512_f32_mult_-1_0"] == "0"


def test_measure_times_the_passes_of_the_transform(rules):
    """Where pass 2 is the plain x pass (N1 = 32 or 64) it is timed and takes
    a choice without leaving the two-pass form; a plan on pass 2's own
    kernels times nothing and leaves the form for a choice; one without a
    two-pass form times y and x."""
    for key in ("f32_1_2048x64x512", "f64_1_512x32x256", "f32_2_1024x64x64"):
        assert rules["tune_" + key] == "two 1 1 0 axes 0", key
    # (64 rows of 512 points in two blocks of 32: M = 2)
    for key in ("f64_2_512x64x512", "f32_1_512x512x512"):
        assert rules["tune_" + key] == "two 1 0 0 axes", key
    assert rules["tune_f64_1_512x512x500"] == "two 0 0 0 axes 1 0"
