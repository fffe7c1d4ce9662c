"""The tiling of tests/test_tiling.py as the library plans it: the halo of tb_halo
(kernels.h), and starts and origins even in x too.  (That test's own figures, a halo
of 2K + 4 and no alignment in x, are no variant's any more.)"""
import os
import re
import shutil
import subprocess

import pytest

from tests.test_tiling import CSRC, DRIVER, variants

OURS = DRIVER.replace("2 * K + 4", "HALO").replace("check(EX, H, 1, nmax)", "check(EX, H, 2, nmax)")


def _halo():
    m = re.search(r"tb_halo\(int k\) \{ return (.*?); \}", open(os.path.join(CSRC, "kernels.h")).read())
    return m.group(1).replace("k", "K")


def _run(dir_, include, args):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    src, exe = dir_ / "t.cpp", dir_ / "t"
    src.write_text(OURS.replace("HALO", _halo()))
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", str(include), str(src), "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)] + args, capture_output=True, text=True, timeout=120)


def test_the_planner_calls_match():
    assert OURS.count("HALO") == 1 and OURS.count("check(EX, H, 2, nmax)") == 1
    api = open(os.path.join(CSRC, "api.hip")).read()
    calls = re.findall(r"plan_axis\((.*?), v\.(e[xy]), H, (\d)\)", api)
    assert len(calls) == 4 and all(q == "2" for _, _, q in calls)
    assert len(re.findall(r"const int H = tb_halo\(v\.k\);", api)) == 2


def test_axis_tiling_invariants_with_the_variants_halo(tmp_path):
    r = _run(tmp_path, CSRC, ["2100"] + [str(x) for kxy in variants() for x in kxy])
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("old,new", [("e0 = E - q - H", "e0 = E - H"),
                                     ("const int o = E - 2 * H", "const int o = E - 2 * H + 2"),
                                     ("start - H}", "start - H + 2}")])
def test_a_wrong_planner_is_caught(tmp_path, old, new):
    text = open(os.path.join(CSRC, "tiling.h")).read()
    assert old in text
    (tmp_path / "tiling.h").write_text(text.replace(old, new))
    r = _run(tmp_path, tmp_path, ["700", "6", "96", "96"])
    assert r.returncode != 0 and "FAIL" in r.stdout
