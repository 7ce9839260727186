"""route_topk over its whole range of widths and counts: the order rule (NaN first, value
descending, index ascending) against a stable sort, the same bits from every kernel, and the
routing-weight gradient with repeated and dropped selections at any width."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _hip():
    from rte_amd import _lib

    if not _lib.device_ready():
        pytest.fail("HIP backend not ready (library or gfx950 device missing)")
    yield


def _order(lg, k):
    """ids of the k best per row: NaN before numbers, larger first, lower index first."""
    key = torch.where(lg.isnan(), torch.full_like(lg, float("inf")), lg).double() + 0.0
    key = torch.where(lg.isnan(), torch.full_like(key, float("inf")), key.clamp(max=1e300))
    return key.sort(dim=1, descending=True, stable=True).indices[:, :k].int()


# widths on both sides of one and two logits per lane and of the lanes-per-row limits, counts on both sides
# of each of them: C 1000 takes 64, 32, 16 and 8 lanes a row over these T
@pytest.mark.parametrize("C,k", [(1, 1), (3, 2), (31, 4), (32, 1), (33, 3), (64, 16), (65, 5), (65, 16), (100, 8),
                                 (128, 12), (129, 1), (129, 16), (256, 16), (257, 9), (512, 8), (1000, 1), (1000, 16),
                                 (1024, 3)])
@pytest.mark.parametrize("T", [1, 37, 2050, 5000, 12000, 16400])
def test_order_and_agreement(C, k, T):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(C * 17 + k)
    lg = torch.randn(T, C, generator=g)
    lg = torch.where(torch.rand(T, C, generator=g) < 0.3, (lg * 2).round() / 2, lg)  # ties
    lg[::5] = torch.where(torch.rand(lg[::5].shape, generator=g) < 0.05, torch.tensor(float("nan")), lg[::5])
    lg[1::7, : C // 2] = float("-inf")
    lg[2::11, C // 3] = 3.4e38
    ids, w = H.route_topk(lg.to(DEV), k)
    assert torch.equal(ids.cpu(), _order(lg, k))
    n = min(T, 30)  # few rows take another kernel at some widths: the same bits
    ids_n, w_n = H.route_topk(lg[:n].to(DEV), k)
    assert torch.equal(ids_n, ids[:n])
    assert torch.equal(w_n.view(torch.int32), w[:n].view(torch.int32)) or torch.allclose(w_n, w[:n], rtol=0, atol=0,
                                                                                         equal_nan=True)


@pytest.mark.parametrize("T,C,k", [(1, 1, 1), (5, 7, 3), (35, 63, 5), (70, 64, 16), (18, 65, 16),
                                   (130, 256, 16), (33, 1025, 16), (9, 4098, 4)])
def test_route_bwd_rows(T, C, k):
    from rte_amd import _lib

    g = torch.Generator().manual_seed(C)
    ids = torch.randint(0, C, (T, k), generator=g, dtype=torch.int32)  # repeats among them
    w = torch.rand(T, k, generator=g)
    slot = torch.randperm(T * k, generator=g).to(torch.int32).view(T, k)
    slot[torch.rand(T, k, generator=g) < 0.2] = -1
    dw = torch.randn(T * k, generator=g)
    dev = [t.to(DEV) for t in (ids, w, dw, slot)]
    out = torch.full((T, C), 7.0, device=DEV, dtype=torch.bfloat16)
    out32 = torch.full((T, C), 7.0, device=DEV)
    _lib.call("rte_route_bwd", dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(), dev[3].data_ptr(), T, C, k,
              out.data_ptr(), out32.data_ptr(), _lib.stream_ptr())
    d = torch.where(slot >= 0, dw[slot.long().clamp(min=0)], torch.zeros(()))
    s = (w.double() * d.double()).sum(1, keepdim=True)
    want = torch.zeros(T, C, dtype=torch.float64)
    for j in range(k):  # the last selection of a cluster writes it
        want[torch.arange(T), ids[:, j].long()] = (w[:, j:j + 1].double() * (d[:, j:j + 1].double() - s))[:, 0]
    # a difference of sums of k products: k 2^-23 of their magnitude
    assert (out32.cpu().double() - want).abs().max() <= k * 2**-22 * float((w * d).abs().max() + s.abs().max())
    assert torch.equal(out, out32.to(torch.bfloat16))
