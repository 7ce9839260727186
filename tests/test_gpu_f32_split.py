"""Split reductions of the fp32 GEMM (weight gradients over many tokens): k ranges cut over several
workgroups, their partials added in order, against float64.  Tolerance: an fp32 sum of K products is
off by about sqrt(K) 2^-24 of the row norms (Frobenius, factor 8)."""

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


def _rel(got, ref):
    return float((got.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("M,N,K,b_t", [(32, 256, 8192, 1), (33, 37, 1023, 1), (64, 64, 512, 1), (130, 70, 2049, 0),
                                       (17, 9, 511, 1)])  # the last one is not split
def test_dense(M, N, K, b_t):
    from rte_amd.kernels import f32_ops as F

    g = torch.Generator(device=DEV).manual_seed(K)
    A = torch.randn(K, M, device=DEV, generator=g)
    B = torch.randn((K, N) if b_t else (N, K), device=DEV, generator=g)
    C0 = torch.randn(M, N, device=DEV, generator=g)
    ref = 0.5 * A.double().t() @ (B.double() if b_t else B.double().t()) - 2.0 * C0.double()
    outs = []
    for _ in range(2):
        C = C0.clone()
        F.gemm(A, M, 1, B, B.shape[1], b_t, C, N, M, N, K, alpha=0.5, beta=-2.0)
        outs.append(C)
    assert _rel(outs[0], ref) <= 8 * K**0.5 * 2**-24
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("counts", [[0, 256, 257, 1, 1000, 0, 512], [3000], [5, 0, 7], [40] * 130])
def test_grouped(counts):
    """Groups of one chunk, of several, empty ones, and more groups than one wave looks at."""
    from rte_amd.kernels import f32_ops as F

    g = torch.Generator(device=DEV).manual_seed(len(counts))
    G, M, N, T = len(counts), 36, 72, 500
    P = sum(counts)
    goff = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    x = torch.randn(T, N, device=DEV, generator=g)
    dy = torch.randn(P, M, device=DEV, generator=g)
    tok = torch.randint(0, T, (P,), device=DEV, generator=g, dtype=torch.int32)
    sc = torch.rand(P, device=DEV, generator=g)
    rows = torch.randperm(G * M, device=DEV, generator=g).to(torch.int32)
    outs = []
    for _ in range(2):
        C = torch.full((G * M, N), 3.0, device=DEV)
        F.gemm_grouped(2, goff, G, dy, M, 1, x, N, 1, C, N, M, N, P, b_rows=tok, b_scale=sc, c_rows=rows,
                       c_rows_gstride=M)
        outs.append(C)
    grp = torch.repeat_interleave(torch.arange(G), torch.tensor(counts)).to(DEV)
    ref = torch.zeros(G, M, N, dtype=torch.float64, device=DEV)
    ref.index_add_(0, grp, dy.double()[:, :, None] * (x.double()[tok.long()] * sc.double()[:, None])[:, None, :])
    want = torch.empty(G * M, N, dtype=torch.float64, device=DEV)
    want[rows.long()] = ref.view(G * M, N)
    assert _rel(outs[0], want) <= 8 * max(counts)**0.5 * 2**-24
    assert torch.equal(outs[0], outs[1])
