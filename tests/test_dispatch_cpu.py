"""The dispatch rules of the library on the CPU: a small program with the rules'
own headers answers for given sizes, so a change of a rule that sends a size
elsewhere is seen without a GPU.

Viscosity chunks: a launch of the viscosity kernel halves its chunks of levels
only while the halved chunks still run at once, which is what it gains by
(times in us on an MI355X: 128 x 128 x 96 FP64 with the surface model 24.7 with
8 levels per block, 27.8 with 4).

Transforms by lane groups: the plans that the GPU tests of tests/test_gpu_rowfft.py name
for their grids, so that a change of the rule cannot take them off the narrow
groups unseen, and the lengths without a plan.

Argument buffers of a batch: the first substep of a step records fewer launches
than the others (12 members FP32: 46,848 bytes of arguments, then up to 66,960), and
a buffer that was made for it holds the others too; one that grows in the middle
of a step waits for the GPU.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("rules") / "dispatch_rules")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-O1", "-std=c++17",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "microhh_amd", "csrc"), "-x", "hip",
                    os.path.join(ROOT, "tests", "dispatch_rules.cpp"), "-o", exe], check=True)

    def ask(*lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
        return r.stdout.split("\n")[:len(lines)]
    return ask


@pytest.mark.parametrize("itot,jtot,ktot,fp64,limits,sfc,mason,levels", [
    (128, 128, 96, 1, 0, 1, 1, 8), (150, 100, 75, 1, 0, 1, 1, 8), (96, 96, 64, 1, 0, 1, 1, 4),
    (90, 75, 61, 1, 0, 1, 0, 4), (32, 32, 32, 1, 0, 1, 1, 2),
    (128, 128, 96, 1, 0, 0, 0, 4), (192, 144, 64, 1, 0, 0, 0, 8), (200, 160, 20, 1, 0, 0, 0, 4),
    (128, 128, 96, 1, 1, 0, 0, 8), (256, 160, 24, 0, 0, 1, 1, 4), (150, 100, 75, 0, 0, 1, 1, 4),
    (320, 256, 12, 0, 0, 1, 1, 4), (160, 128, 80, 0, 0, 0, 0, 4), (32, 32, 32, 0, 0, 0, 0, 2),
    (512, 512, 256, 1, 0, 0, 0, 64)])
def test_viscosity_chunks(rules, itot, jtot, ktot, fp64, limits, sfc, mason, levels):
    tiles = ((itot + 63) // 64) * ((jtot + 3) // 4)
    assert rules(f"visc {tiles} {ktot} {fp64} {limits} {sfc} {mason}") == [str(levels)]


@pytest.mark.parametrize("first,largest", [(46848, 66960), (4 * 46848, 4 * 66960), (1, 65536)])
def test_batch_arguments_fit_what_a_step_needs(rules, first, largest):
    assert int(rules(f"batch {first}")[0]) >= largest


def test_plans_of_the_gpu_tests(rules):
    from tests.test_gpu_rowfft import FALLBACK, NARROW, NARROW32
    for itot, jtot, ktot, x, y in NARROW + NARROW32:
        got = rules(f"row {itot} {(jtot + 1) // 2 * ktot}", f"row {jtot} {(itot // 2 + 1) * ktot}")
        for want, answer in zip((x, y), got):
            if want == "none":
                assert answer == "none"
            else:
                lanes, values, arith = answer.split()
                assert f"{lanes} {arith}" == want, (itot, jtot, ktot)
    for itot, jtot, ktot in FALLBACK:
        assert "none" in rules(f"row {itot} 100", f"row {jtot} 100")


def test_lengths_without_a_plan(rules):
    def rest(n):
        for q in (2, 3, 5, 7, 11, 13):
            while n % q == 0:
                n //= q
        return n
    smooth = [n for n in range(1, 2049) if rest(n) == 1]
    none = [n for n, a in zip(smooth, rules(*[f"row {n} 1000" for n in smooth])) if a == "none"]
    assert none[:2] == [1, 1050] and len([n for n in smooth if n > 1024]) == 105 and len(none) == 1 + 55
