"""How comp_amd.host reaches the library, without a GPU: what importing it needs of torch, and which
library its calls go to."""

import os
import subprocess
import sys
import types

from comp_amd import _abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_imports_on_a_torch_without_gpu_support():
    """Such a torch has neither of torch._C's device and stream functions; the host-side calls need none of them."""
    code = (
        "import torch\n"
        "for name in ('_cuda_getCurrentRawStream', '_cuda_getDevice'):\n"
        "    delattr(torch._C, name)\n"
        "from comp_amd import host\n"
        "wq, ws = host.split('q4_0', bytes(range(18)) * 4, 2, 64)\n"
        "assert wq.shape == (2, 32) and ws.shape == (2, 2)\n"
    )
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True,
                       env=dict(os.environ, PYTHONPATH=os.pathsep.join((ROOT, os.path.join(ROOT, "oracle")))))  # fmt: skip
    assert r.returncode == 0, r.stderr


def test_calls_go_to_the_library_that_is_loaded_now(monkeypatch):
    """A library loaded in place of another one (a rebuild in one process) is the one that is called."""
    got = []
    for i in (1, 2):
        monkeypatch.setattr(_abi, "_lib", types.SimpleNamespace(komp_quant_q8_0=lambda *a, i=i: got.append(i) or 0))
        _abi.call("komp_quant_q8_0")
        assert _abi.entry("komp_quant_q8_0")() == 0
    assert got == [1, 1, 2, 2]
