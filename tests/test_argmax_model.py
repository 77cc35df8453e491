"""The arg-max that every top-k and top-m selection is built on, on the host:
tests/host/argmax_model.cpp compiles select_key and argmax_take from the
kernels' header and runs the lanes' exchange steps over finite, infinite and
NaN values."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_selection_is_one_order_for_every_lane(tmp_path):
    exe = str(tmp_path / "argmax_model")
    r = subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "spider-web-moe_amd", "csrc"),
                        os.path.join(HERE, "host", "argmax_model.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:]
    assert "selections agree" in r.stdout
