"""The on-chip SVD FFN where its loop over 32-row tiles changes shape: one tile, every remainder of the
three-stage rotation, a last tile that is partly empty, one and several splits, both ranks."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as TF

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("r", [64, 128])
@pytest.mark.parametrize("T,F", [(8, 128), (40, 128), (104, 256), (136, 384), (160, 128), (8200, 128), (33000, 256),
                                 (264, 8320)])
def test_against_float64(T, F, r):
    from rte_amd.kernels import hip_ops as H

    d = 64
    assert H.svd_ffn_fused_supported(T, d, F, r)
    g = torch.Generator().manual_seed(T + F + r)

    def rnd(*shape, scale):
        return (torch.randn(*shape, generator=g) * scale).bfloat16()

    w = [rnd(d, 2 * r, scale=d ** -0.5), rnd(2 * F, r, scale=r ** -0.5), rnd(F, r, scale=F ** -0.5),
         rnd(d, r, scale=r ** -0.5)]
    x, dy = rnd(T, d, scale=1.0), rnd(T, d, scale=1.0)
    print(f"svd_ffn T={T} F={F} r={r}", flush=True)
    tx, tw = x.to(DEV).requires_grad_(), [t.float().to(DEV).requires_grad_() for t in w]
    y = H.svd_ffn(tx, *tw)
    y.backward(dy.to(DEV).to(y.dtype))
    rx, rw = x.double().requires_grad_(), [t.double().requires_grad_() for t in w]
    a = rx @ rw[0]
    u, gt = a[:, :r] @ rw[1][:F].t(), a[:, r:] @ rw[1][F:].t()
    ref = ((u * TF.silu(gt)) @ rw[2]) @ rw[3].t()
    ref.backward(dy.double())
    # each result passes at most six roundings to bf16 (a, z or du / dg, b or db, da, the stored
    # result, and g's share through silu'), each of relative size 2^-9 and independent
    for name, got, want in zip(("y", "dx", "dus_ug", "dv_ug", "dv_dn", "dus_dn"), [y, tx.grad, *[t.grad for t in tw]],
                               [ref, rx.grad, *[t.grad for t in rw]]):
        err = (got.detach().double().cpu() - want.detach()).norm() / want.detach().norm()
        assert err <= 6 * 2.0 ** -9, f"{name}: {float(err):.2e}"
