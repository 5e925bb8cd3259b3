"""Which kernels a pass takes: the host rules of fft_launch.hpp,
fft_two_launch.hpp and exec.hpp, evaluated on the CPU by
tests/cpp/route_rules.cpp."""
import os
import re
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


def test_large_pass_1_tiles_need_blocks(rules):
    """Tiles of 128 KiB and more, and of 512-point lines, run in two passes
    from as many x planes as the tile has complex rows."""
    def rows(prec, n0, n1, n2):
        return tuple(int(v) for v in rules[f"rows_{prec}_{n0}x{n1}x{n2}"].split())
    for prec in ("f32", "f64"):
        for n0 in (1, 15, 31, 32, 512):  # small tiles: any number of planes
            assert rows(prec, n0, 64, 32) == (64, 64)
        # real rows of 512 points: 16 (32 rows) and 32 (64 rows) blocks
        assert rows(prec, 15, 32, 512)[0] == 0 and rows(prec, 16, 32, 512)[0] == 32
        assert rows(prec, 31, 64, 512)[0] == 0 and rows(prec, 32, 64, 512)[0] == 64
        assert rows(prec, 31, 32, 512)[1] == 0 and rows(prec, 32, 32, 512)[1] == 32
        assert rows(prec, 512, 128, 512)[0] == 64
    # 256 points: FP32 r2c tiles of 64 rows are 64 KiB, FP64 ones 128 KiB
    assert rows("f32", 1, 64, 256) == (64, 0)
    assert rows("f64", 31, 64, 256) == (0, 0) and rows("f64", 32, 64, 256) == (64, 0)
    assert rows("f32", 63, 64, 256) == (64, 0) and rows("f32", 64, 64, 256) == (64, 64)
    assert rows("f64", 1, 64, 128) == (64, 0) and rows("f64", 64, 64, 128) == (64, 64)
    # FP64 complex rows of 512 points: 32 at a time, two blocks a plane
    assert rows("f64", 32, 64, 512)[1] == 32


def test_large_passes_of_short_power_of_two_lines(rules):
    """The mixed-radix kernels take power-of-two z and C2C passes up to the
    bytes from which the wider tiles are faster, and fused strided passes of
    any size.  Entries: log2 of the most points (27: any), 0 never."""
    c2c, r2c, c2r, deriv, mult = rules["modes"].split()
    n = (16, 32, 64, 128, 256, 512, 1024)

    def row(prec, kind, mode, odd=0):
        return tuple(int(rules[f"most_{prec}_{v}_{kind}{mode}_{odd}"]) for v in n)
    for odd in (0, 1):
        for mode in (r2c, c2r):
            assert row("f32", "z", mode, odd) == (19, 21, 23, 25, 0, 0, 0)
            assert row("f64", "z", mode, odd) == (19, 21, 23, 24, 0, 0, 0)
            # a pencil share's column blocks
            assert row("f32", "z", mode, 2) == (19, 21, 23, 23, 0, 0, 0)
            assert row("f64", "z", mode, 2) == (19, 21, 22, 22, 0, 0, 0)
        assert row("f32", "z", deriv, odd) == (20, 22, 24, 25, 27, 27, 0)
        assert row("f64", "z", deriv, odd) == (20, 22, 24, 24, 0, 0, 0)
        assert row("f32", "z", c2c, odd) == (21, 23, 24, 24, 0, 0, 0)
        assert row("f64", "z", c2c, odd) == (21, 23, 24, 24, 0, 0, 0)
        assert row("f32", "s", deriv, odd) == (27, 27, 27, 27, 27, 0, 0)
        for mode in (mult, deriv):
            assert row("f64", "s", mode, odd) == (27, 27, 27, 27, 27, 27, 0)
    assert row("f32", "s", c2c, 0) == (19, 21, 23, 24, 26, 27, 0)
    assert row("f32", "s", c2c, 1) == (19, 21, 23, 24, 26, 27, 0)
    assert row("f64", "s", c2c, 0) == (20, 22, 24, 24, 25, 27, 0)
    assert row("f64", "s", c2c, 1) == (19, 21, 23, 24, 25, 27, 0)


def test_every_mixed_radix_kernel_is_reached(rules):
    """The library holds the kernels of the list's lengths that a pass can
    be sent to, and no others."""
    import accfft_amd as af
    nm = shutil.which("nm")
    if nm is None or not os.path.exists(af.LIB_PATH):
        pytest.skip("needs nm and the built library")
    syms = subprocess.run([nm, "-C", af.LIB_PATH], check=True, capture_output=True, text=True).stdout
    have = {(k, t, int(n), m) for k, t, n, m in re.findall(
        r" afft::mix_([sz])_kernel<(float|double), (\d+), (\d)>", syms)}
    lists = open(os.path.join(HERE, "..", "accfft_amd", "csrc", "fft_mix_list.hpp")).read()
    lengths = [int(v) for v in re.findall(r"X\((\d+)\)", lists.split("#define AFFT_MIX_EACH")[0])]
    c2c, r2c, c2r, deriv, mult = rules["modes"].split()
    want = set()
    for t, prec in (("float", "f32"), ("double", "f64")):
        for n in lengths:
            for kind, modes in (("s", (c2c, mult, deriv)), ("z", (c2c, r2c, c2r, deriv))):
                for m in modes:
                    if n & (n - 1) or int(rules[f"most_{prec}_{n}_{kind}{m}_0"]):
                        want.add((kind, t, n, m))
    assert have == want


def test_pass_2_tiles_are_whole(rules):
    """Every plan's pass 2 has a whole number of tiles (the kernel has no
    guard, its launcher refuses others), and its 32-bit byte offsets reach
    the whole grid."""
    most = 0
    for prec in ("f32", "f64"):
        for n0 in (32, 64, 128, 256, 512):
            for m in (2, 4, 8):
                plans, left, span = map(int, rules[f"pass2_{prec}_{n0}_{m}"].split())
                assert plans > 0 and left == 0 and span < 2 ** 32
                most = max(most, span)
    assert most == 512 * 512 * 257 * 16  # the 512^3 half spectrum in FP64
