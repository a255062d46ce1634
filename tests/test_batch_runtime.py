"""Which processes advance a batch by one graph (no compute calls: CPU only)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("steps,available", [
    (["from macau_amd import _lib; _lib.lib()"], 1),
    (["import torch", "from macau_amd import _lib; _lib.lib()"], 0),   # one runtime, PyTorch's
    (["from macau_amd import _lib; _lib.lib()", "import torch"], 0)])  # two runtimes
def test_one_graph_only_under_the_library_s_own_runtime(steps, available):
    code = "\n".join(steps + ["print('available', _lib.lib().macau_batch_graph_available())"])
    if any("torch" in s for s in steps):
        # a PyTorch without a HIP runtime of its own changes nothing
        probe = "import torch; print(torch.version.hip or '')"
        hip = subprocess.run([sys.executable, "-c", probe], capture_output=True, text=True, timeout=300)
        if hip.returncode or not hip.stdout.strip():
            pytest.skip("no PyTorch for ROCm")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr
    assert out.stdout.split()[-2:] == ["available", str(available)]
