"""The bounds that the network's two gradient buffers are sized with, each by itself
(tests/test_nn_sizes.py compares both needs with the larger of them): a layer's
weight partials with dw_partials, its bias partials with bias_partials."""
import os
import subprocess

import pytest

from tests.test_nn_sizes import CSRC, DRIVER
from tests import test_nn_sizes

OURS = (DRIVER.replace("const int64_t bound = grad_partials(c[0], c[1], cap);",
                       "const int64_t dw = dw_partials(c[0], c[1], cap), db = bias_partials(c[1], cap);")
        .replace("ch * c[1] * 9 * c[0] > bound", "ch * c[1] * 9 * c[0] > dw")
        .replace("bias_blocks(npix) * c[1] > bound", "bias_blocks(npix) * c[1] > db"))


def _run(monkeypatch, include, out_dir, dense):
    monkeypatch.setattr(test_nn_sizes, "DRIVER", OURS)
    exe = test_nn_sizes._build(include, out_dir)
    return subprocess.run([exe, dense], capture_output=True, text=True, timeout=300)


def test_each_buffer_holds_the_partials_of_every_smaller_batch(tmp_path, monkeypatch):
    assert "grad_partials" not in OURS and "> dw)" in OURS and "> db)" in OURS
    r = _run(monkeypatch, CSRC, tmp_path, "3000000")
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr


@pytest.mark.parametrize("old,new,what", [
    ("std::max<int64_t>(257,", "std::max<int64_t>(256,", "FAIL dw"),
    ("(npix + 127) / 128, 257) * cout", "(npix + 127) / 128, 255) * cout", "FAIL bias"),
    ("(npix + 127) / 128, 257) * cout", "(npix + 255) / 256, 257) * cout", "FAIL bias")])
def test_a_bound_that_is_too_small_is_caught(tmp_path, monkeypatch, old, new, what):
    text = open(os.path.join(CSRC, "nn_sizes.h")).read()
    assert old in text
    (tmp_path / "nn_sizes.h").write_text(text.replace(old, new))
    r = _run(monkeypatch, tmp_path, tmp_path, "300000")
    assert r.returncode != 0 and what in r.stdout
