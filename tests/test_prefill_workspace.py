"""The workspace an engine sizes for its prefill's batched products (gemv_mfma_workspace_upto) holds every
launch of at most that many rows, whichever kernel its plan picks: a launch that did not fit would allocate
inside a captured graph.  Plans only (host code), on the CPU."""
import os
import subprocess

import pytest

from edgeforge_amd import build as hipbuild

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_prefill_workspace_holds_every_launch(tmp_path):
    if not os.path.exists(hipbuild.LIB):
        pytest.skip("libedgeforge_hip.so not built")
    exe, lib = str(tmp_path / "prefill_workspace"), os.path.dirname(hipbuild.LIB)
    r = subprocess.run([hipbuild.HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1",
                        f"-I{hipbuild.CSRC}", os.path.join(ROOT, "tests", "cpp", "prefill_workspace.hip"), "-o", exe,
                        f"-L{lib}", "-ledgeforge_hip", f"-Wl,-rpath,{lib}"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
