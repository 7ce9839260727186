"""Routed pools of 64- and 96-neuron clusters on the grouped products: few rows per cluster, empty
clusters, ragged tiles and clusters cut into several reduction chunks, against float64 under the
kernel's own routing.  Tolerance: the stored bf16 activations (up, gate, z, dug, pair rows) each round by
2^-9 at most; a few of them meet in every output."""

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


def _ref(x, wr, wug, wd, ids, k):
    T, C, F = x.shape[0], wr.shape[0], wd.shape[1]
    n = F // C
    w = (x @ wr.t()).gather(1, ids).softmax(dim=-1)
    y = torch.zeros_like(x)
    for c in range(C):
        tok, j = (ids == c).nonzero(as_tuple=True)
        if tok.numel():
            up = x[tok] @ wug[c * n:(c + 1) * n].t()
            gate = x[tok] @ wug[F + c * n:F + (c + 1) * n].t()
            z = (up * torch.nn.functional.silu(gate)) @ wd[:, c * n:(c + 1) * n].t()
            y = y.index_add(0, tok, w[tok, j].unsqueeze(1) * z)
    return y


@pytest.mark.parametrize("T,d,C,n,k,skew", [
    (3, 128, 8, 64, 2, False),       # clusters of no or one row
    (130, 192, 4, 64, 3, False),
    (4100, 256, 4, 64, 2, True),     # a dominant cluster: several chunks
    (300, 1024, 16, 64, 4, False),
    (513, 128, 6, 96, 2, True),      # wider clusters: the general products
    (2049, 1024, 12, 64, 1, True),
])
def test_pool(T, d, C, n, k, skew):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(T + d)
    F = C * n
    x = torch.randn(T, d, generator=g)
    wr = torch.randn(C, d, generator=g) * 0.05
    if skew:
        x[:, 0] = 4.0
        wr[:, 0] = torch.linspace(1.0, -1.0, C)
    wug, wd = torch.randn(2 * F, d, generator=g) * d**-0.5, torch.randn(d, F, generator=g) * n**-0.5
    dy = torch.randn(T, d, generator=g)
    args = [x.to(DEV).to(torch.bfloat16).requires_grad_(), *[t.to(DEV).requires_grad_() for t in (wr, wug, wd)]]
    out, ids, _ = H.routed_cluster_pool_swiglu(*args, k)
    grads = torch.autograd.grad(out, args, dy.to(DEV))
    again = torch.autograd.grad(H.routed_cluster_pool_swiglu(*args, k)[0], args, dy.to(DEV))
    ref_args = [t.detach().to(torch.bfloat16).double().requires_grad_() for t in args]
    ref = _ref(*ref_args, ids.long(), k)
    want = torch.autograd.grad(ref, ref_args, dy.to(DEV).double())
    for a, b in zip((out, *grads), (ref, *want)):
        a, b = a.detach().double(), b.detach()
        assert float((a - b).norm() / b.norm().clamp_min(1e-30)) <= 5 * 2**-9
    assert all(torch.equal(a, b) for a, b in zip(grads, again))
