"""GEMMs over weight planes that are views: the last columns of a wider plane (a layer split along K), whose last row ends
where the storage ends.  Nothing past a row's own blocks is read there, and the result is the packed plane's."""

import pytest
import torch

from comp_amd import host
from oracle import oracle as O
from tests.test_gpu_gemm import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["q4_0", "tq2_0", "q8_0", "iq4_nl", "q4_k"])
@pytest.mark.parametrize("blocks", [3, 5, 22, 23])  # the last K step partial, of the short rows' kernel and of the tile
@pytest.mark.parametrize("m", [4, 20, 70])
def test_last_columns_of_a_wider_plane(fmt, blocks, m):
    n, k = 37, blocks * O.FORMATS[fmt]["block"]
    W, x = O.problem(fmt, n, k, m, 17)
    wq, ws = (dev(a) for a in host.split(fmt, W, n, k))
    xq, xd = host.quantize(fmt, dev(x))
    want, s = host.gemm(fmt, wq, ws, xq, xd, n, k, store_s=True)
    print(f"gemm of a view {fmt} n={n} k={k} m={m} {host.gemm_plan(fmt, m, n, k)}", flush=True)
    row = wq.shape[1]
    wide = torch.full((n, row + 64), 0x77, dtype=torch.uint8, device="cuda")
    view = wide[:, 64:]
    view.copy_(wq)
    assert view.data_ptr() + (n - 1) * view.stride(0) + row == wide.data_ptr() + wide.numel()
    got, s2 = host.gemm(fmt, view, ws, xq, xd, n, k, store_s=True)
    assert torch.equal(got, want) and torch.equal(s, s2)
