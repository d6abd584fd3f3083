"""How comp_amd.host reaches the library, without a GPU: what importing it needs of torch, which
library its calls go to, what they hand over and return, and on which device and stream they launch."""

import contextlib
import os
import subprocess
import sys
import types

import torch

from comp_amd import _abi, host

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
        monkeypatch.setattr(host, "_current_device", lambda: -1)
        monkeypatch.setattr(host, "_raw_stream", lambda dev: None)
        host._launch("komp_quant_q8_0", torch.zeros(1))
    assert got == [1, 1, 2, 2]


class DeviceLike(torch.Tensor):
    """A tensor subclass that says it is on a device (its memory is the host's; nothing launches)."""

    is_cuda = True


def test_outputs_are_plain_tensors_whatever_the_inputs_type(monkeypatch):
    """As torch.empty gives them: a subclass of the input's would run its own code on every later use of a plane."""
    monkeypatch.setattr(host, "_launch", lambda name, *a: None)
    monkeypatch.setattr(host, "_check_gemv", lambda *a: (2, 4))
    monkeypatch.setattr(host, "_weights_fit", lambda *a: True)
    like = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype).as_subclass(DeviceLike)  # noqa: E731
    x, w = like(2, 1024), like(8, 512, dtype=torch.uint8)
    q = (*host.quantize("q4_0", x), *host.quantize("tq2_0", x, bsums=True))
    xq, xd = like(2, 1024, dtype=torch.int8), like(2, 32)
    y = [f("q4_0", w, w, xq, xd, 8, 1024)[0] for f in (host.gemv, host.gemm)] + [host.gemv_f32("q4_0", w, w, x, 8, 1024)[0]]
    assert [type(t) for t in (*q, *y)] == [torch.Tensor] * 8
    assert [(t.shape, t.dtype) for t in y] == [((2, 8), torch.float32)] * 3
    assert [(tuple(t.shape), t.dtype) for t in q] == [
        ((2, 1024), torch.int8), ((2, 32), torch.float32),
        ((2, 1024), torch.int8), ((2, 4), torch.float32), ((2, 64), torch.int16)]  # fmt: skip


class OnDeviceOne(DeviceLike):
    def get_device(self):
        return 1


def test_launches_pass_the_tensors_devices_current_stream(monkeypatch):
    """The stream is the last argument, and the device is switched for the call alone, if it is another one."""
    log, current = [], [0]

    @contextlib.contextmanager
    def switched(dev):
        before, current[0] = current[0], dev
        log.append(("switch", dev))
        yield
        current[0] = before

    class Library:
        def __getattr__(self, name):
            return lambda *a: log.append((name, current[0], a[-1])) or 0

    monkeypatch.setattr(_abi, "_lib", Library())
    monkeypatch.setattr(host, "_raw_stream", lambda dev: 1000 + dev)
    monkeypatch.setattr(host, "_current_device", lambda: current[0])
    monkeypatch.setattr(torch.cuda, "device", switched)
    monkeypatch.setattr(host, "_weights_fit", lambda *a: True)
    like = lambda t: t.as_subclass(OnDeviceOne)  # noqa: E731
    w, ws = like(torch.zeros((8, 512), dtype=torch.uint8)), like(torch.zeros((8, 32), dtype=torch.int16))
    x, xq, xd = like(torch.zeros((2, 1024))), like(torch.zeros((2, 1024), dtype=torch.int8)), like(torch.zeros((2, 32)))
    monkeypatch.setattr(host, "_Tensor", OnDeviceOne)  # as plain tensors, so that the device stays the fake one
    for call, name in (
        (lambda: host.quantize("q4_0", x), "komp_quant_q8_0"),
        (lambda: host.gemv("q4_0", w, ws, xq, xd, 8, 1024), "komp_q4_0_gemv"),
        (lambda: host.gemm("q4_0", w, ws, xq, xd, 8, 1024), "komp_q4_0_gemm"),
        (lambda: host.gemv_f32("q4_0", w, ws, x, 8, 1024), "komp_q4_0_gemv_f32"),
    ):
        for at in (0, 1):
            current[0] = at
            log.clear()
            call()
            assert log == ([("switch", 1)] if at == 0 else []) + [(name, 1, 1001)] and current[0] == at
