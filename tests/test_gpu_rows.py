"""The pools' pair products, where a group's weight stays in LDS and its rows stream past: row counts on both
sides of the rule that takes them, empty groups and groups that end inside a block of 32, column remainders,
k 64 and 128 in both weight layouts, rows scattered to another order."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("n", [32, 64, 128])
@pytest.mark.parametrize("P,G,d", [(4095, 7, 256), (4096, 7, 128), (4500, 300, 264), (20000, 3, 1000), (9000, 40, 512)])
def test_pair_products(P, G, n, d):
    from rte_amd import _lib

    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(P + G + n + d)
    T = P // 4

    def rnd(*shape, scale):
        return (torch.randn(*shape, device=DEV, generator=g) * scale).bfloat16()

    x, dout = rnd(T, d, scale=1.0), rnd(T, d, scale=1.0)
    wug, wd = rnd(2 * G * n, d, scale=d ** -0.5), rnd(d, G * n, scale=n ** -0.5)
    cl = (torch.rand(P, device=DEV, generator=g) ** 2 * G).long().clamp(max=G - 1)
    cl = torch.where(cl == G // 2, torch.zeros_like(cl), cl).sort().values          # an empty group
    off = torch.zeros(G + 1, dtype=torch.int32, device=DEV)
    off[1:] = torch.bincount(cl, minlength=G).cumsum(0).int()
    pair = torch.randperm(P, device=DEV, generator=g).int()
    tok = (pair // 4).clamp(max=T - 1).int()
    ws = torch.rand(P, device=DEV, generator=g)
    new = lambda *s, dt=torch.bfloat16: torch.empty(*s, dtype=dt, device=DEV)
    ug, zw, y, dug, dx = new(P, 2 * n), new(P, n), new(P, d), new(P, 2 * n), new(P, d)
    dws, dwug, dwd = new(P, dt=torch.float32), new(2 * G * n, d, dt=torch.float32), new(d, G * n, dt=torch.float32)
    nb = lib.rte_grouped_swiglu_bwd_workspace_bytes(P, G, n, d)
    buf = new(max(nb, 256), dt=torch.uint8)
    st = torch.cuda.current_stream().cuda_stream
    q = lambda t: t.data_ptr()
    print(f"pair products P={P} G={G} n={n} d={d}", flush=True)
    _lib.call("rte_grouped_swiglu_fwd", q(x), T, d, q(off), G, n, P, q(tok), q(pair), q(ws), q(wug), q(wd), G * n,
              q(ug), q(zw), q(y), st)
    _lib.call("rte_grouped_swiglu_bwd", q(dout), q(x), T, d, q(off), G, n, P, q(tok), q(pair), q(ws), q(wug), q(wd),
              G * n, q(ug), q(zw), q(dug), q(dws), q(dx), q(dwug), q(dwd), 0, 0.0, q(buf), nb, st)
    torch.cuda.synchronize()
    pair, cl = pair.long().cpu(), cl.cpu()
    zw, dug, wd, wug, y, dx = [t.double().cpu() for t in (zw, dug, wd, wug, y, dx)]
    assert bool(torch.isfinite(y).all()) and bool(torch.isfinite(dx).all())
    for c in range(G):
        rows = (cl == c).nonzero().flatten()
        if rows.numel() == 0:
            continue
        w2 = wd[:, c * n:(c + 1) * n].t()
        # dug holds 32 up, 32 gate columns in turn; wug the up rows, then the gate rows
        at = torch.arange(2 * n)
        r = c * 2 * n + at
        w1 = wug[(r // 64) * 32 + r % 32 + torch.where(r % 64 < 32, 0, G * n)]
        for got, a, w in ((y, zw, w2), (dx, dug, w1)):
            want, mag = a[rows] @ w, a[rows].abs() @ w.abs()
            # one rounding to bf16 and at most 2 n + 1 of the sums in fp32
            bound = 2.0 ** -8 * want.abs() + (2 * n + 1) * 2.0 ** -23 * mag + 1e-37
            assert bool(((got[pair[rows]] - want).abs() <= bound).all()), f"group {c}"
