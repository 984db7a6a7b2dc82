"""Device sources run on the CPU, thread by thread (tests/cpp/emulate), under AddressSanitizer.

The runtime-length pass takes every length without a compile-time tile in every form (complex, real
sides, Hermitian load, partial store, fused product, split-axis twiddle, cosine and sine modes); its
index arithmetic, radix plans and LDS layouts are checked against direct transforms for all orders
of both sides, with arrays and LDS that end where the pass may last touch them.  The fused two-axis
pass likewise over many plane shapes, and the fused phases of a batch over the work lists of one.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "heffte_amd", "csrc")
CLANG = "/opt/rocm/llvm/bin/clang++" if os.path.exists("/opt/rocm/llvm/bin/clang++") else shutil.which("clang++")
SHARES = 8


def build(tmp_path_factory, name, sources):
    out = str(tmp_path_factory.mktemp("emulate") / name)
    cmd = [CLANG, "-std=c++17", "-O1", "-fsanitize=address", "-Wno-pass-failed", "-I", os.path.join(HERE, "cpp", "emulate"),
           "-I", os.path.join(HERE, "cpp"), "-I", CSRC, os.path.join(HERE, "cpp", name + ".cpp")] + \
        [os.path.join(CSRC, s) for s in sources] + ["-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return out


@pytest.mark.skipif(CLANG is None, reason="clang++ not found")
@pytest.mark.parametrize("name", ["emulate_generic", "emulate_plane", "emulate_batch"])
def test_kernel(tmp_path_factory, name):
    exe = build(tmp_path_factory, name, ["hmi_generic_plan.cpp"])
    runs = [subprocess.Popen([exe, str(i), str(SHARES)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
            for i in range(SHARES)]
    for p in runs:
        text = p.communicate(timeout=600)[0]
        assert p.returncode == 0 and "FAIL" not in text and "\nok " in "\n" + text, text[-2000:]
