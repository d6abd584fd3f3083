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
