"""The launching calls' short checks accept what the full checks accept and refuse, with their errors, what those refuse;
and the launches run on the caller's current stream."""

import numpy as np
import pytest
import torch

from comp_amd import _abi, host
from oracle import oracle as O
from tests.checks import outputs_ok

pytestmark = pytest.mark.gpu


def setup(fmt="q4_0", n=40, k=1024, m=2, pad=0):
    W, x = O.problem(fmt, n, k, m, 5)
    wq, ws = host.split(fmt, W, n, k)
    rq, rd, _ = O.quantize(fmt, x)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    t = dict(wq=d(np.pad(wq, ((0, 0), (0, pad)))), ws=d(ws), x=d(x), xq=d(rq), xd=d(rd))
    return t, (ws, rd, *O.gemv(fmt, wq, ws, rq, rd, n, k)), n, k


BAD = {
    "wq": [lambda t: t.cpu(), lambda t: t.to(torch.int8), lambda t: t[:, :-16], lambda t: t[:-1], lambda t: t.T.contiguous().T,
           lambda t: t[None]],
    "ws": [lambda t: t.cpu(), lambda t: t.to(torch.int32), lambda t: t[:, :-1], lambda t: t.T.contiguous().T],
    "x": [lambda t: t.cpu(), lambda t: t.half(), lambda t: t[:, :-32], lambda t: t[None]],
    "xq": [lambda t: t.cpu(), lambda t: t.to(torch.uint8), lambda t: t[:, :-32], lambda t: t.T.contiguous().T],
    "xd": [lambda t: t.cpu(), lambda t: t.double(), lambda t: t[:, :-1], lambda t: t.T.contiguous().T],
}


@pytest.mark.parametrize("name", sorted(BAD))
def test_refused_tensors_stay_refused(name):
    t, _, n, k = setup()
    for i, spoil in enumerate(BAD[name]):
        b = dict(t, **{name: spoil(t[name])})
        print(name, i, flush=True)
        with pytest.raises(_abi.KompArgumentError):
            if name in ("xq", "xd"):
                host.gemv("q4_0", b["wq"], b["ws"], b["xq"], b["xd"], n, k, mode=2)
            else:
                host.gemv_f32("q4_0", b["wq"], b["ws"], b["x"], n, k)
        if name in ("wq", "ws"):
            with pytest.raises(_abi.KompArgumentError):
                host.gemm("q4_0", b["wq"], b["ws"], b["xq"], b["xd"], n, k)
    with pytest.raises(TypeError):
        host.gemv_f32("q4_0", t["wq"].cpu().numpy(), t["ws"], t["x"], n, k)
    with pytest.raises(_abi.KompArgumentError):
        host.gemv_f32_into("q4_0", t["wq"], t["ws"], t["x"], torch.empty((2, n + 1), device="cuda"), n, k)


@pytest.mark.parametrize("fmt", ["q4_0", "tq2_0"])
def test_accepted_forms_on_another_stream(fmt):
    t, (ws, rd, r, rs), n, k = setup(fmt, pad=32)  # padded weight rows
    x = t["x"].T.contiguous().T  # any strides: the call makes its own copy
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y, _ = host.gemv_f32(fmt, t["wq"], t["ws"], x, n, k)
        xq, xd = host.quantize(fmt, x)
        y2, _ = host.gemv(fmt, t["wq"], t["ws"], xq, xd, n, k, block_n=None, mode=2)
    s.synchronize()
    assert torch.equal(xq, t["xq"]) and torch.equal(xd, t["xd"])
    for v in (y, y2):
        assert outputs_ok(fmt, v.cpu().numpy(), ws, rd, rs, r)


@pytest.mark.parametrize("entry", ["quantize", "gemv", "gemm", "gemv_f32", "split"])
def test_captured_launches_are_on_the_capturing_stream(entry):
    """Each entry captured on a stream that is not the default one: the replays compute from inputs written after the
    capture, so the launch is in the graph and not on some other stream."""
    t, _, n, k = setup()
    x2 = torch.randn_like(t["x"])
    blocks = torch.randint(0, 256, (n * (k // 32) * 18,), dtype=torch.uint8, device="cuda")
    xq, xd = torch.empty_like(t["xq"]), torch.empty_like(t["xd"])
    y = torch.empty((t["x"].shape[0], n), device="cuda")
    wq, ws = torch.empty_like(t["wq"]), torch.empty_like(t["ws"])
    call, outs = {
        "quantize": (lambda: host.quantize_into("q4_0", t["x"], xq, xd), (xq, xd)),
        "gemv": (lambda: host.gemv_into("q4_0", t["wq"], t["ws"], t["xq"], t["xd"], y, n, k), (y,)),
        "gemm": (lambda: host.gemm_into("q4_0", t["wq"], t["ws"], t["xq"], t["xd"], y, n, k), (y,)),
        "gemv_f32": (lambda: host.gemv_f32_into("q4_0", t["wq"], t["ws"], t["x"], y, n, k), (y,)),
        "split": (lambda: host.split_into("q4_0", blocks, wq, ws, n, k), (wq, ws)),
    }[entry]
    call()  # loads the kernel
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call()
    torch.cuda.synchronize()
    for i in range(3):
        t["x"].copy_(x2 * (i + 1))
        q2, d2 = host.quantize("q4_0", t["x"])
        t["xq"].copy_(q2)
        t["xd"].copy_(d2)
        blocks.add_(1)
        call()
        want = [o.clone() for o in outs]
        for o in outs:
            o.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want)) and any(bool(o.any()) for o in outs)
