"""The library's own staging, launches and error exits on a HIP runtime answered on the host (no GPU, kernels
do not run): tests/host_hip/checks.py in a process that loads that build."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "gemma-embed-swift_amd", "_build", "libgemmaembed_host_hip.so")


def test_on_the_host_hip_runtime():
    assert os.path.exists(LIB), f"{LIB} is not built (make -C gemma-embed-swift_amd host_hip)"
    r = subprocess.run([sys.executable, "-m", "pytest", "-q", "-p", "no:cacheprovider", "tests/host_hip/checks.py"],
                       cwd=ROOT, env=dict(os.environ, GE_LIBRARY=LIB), capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, (r.stdout + r.stderr)[-6000:]
