"""segment_reduce_rows where its sort and its sums change shape: pair counts on both sides of the
sort-block and chunk limits, one key to the largest key count, row widths that do not fill a column
slab, ids repeated inside a wave, keys out of range, rows in bf16 and fp32."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("P,V,d,div", [
    (4097, 1, 8, 1),                 # first count past the one-launch path, a single key
    ((1 << 18) - 1, 33, 136, 2),     # short chunks, just below the limit
    (1 << 18, 33, 136, 2),           # long chunks
    (1 << 19, 32768, 128, 128),      # short sort blocks, the largest key count
    ((1 << 19) + 4097, 1000, 264, 128),  # long sort blocks, a last block of one pair
    (5000, 1025, 2048, 1),           # widest rows, few pairs
    (5000, 32768, 264, 1),           # far fewer pairs than keys
])
def test_sums_against_float64(P, V, d, div, f32):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(P + V)
    keys = torch.randint(-2, V + 2, (P,), generator=g)
    keys[: P // 4] = V // 2                      # one key with many chunks
    keys[P // 2: P // 2 + P // 8] //= 3          # repeats inside a wave
    rows = torch.randn((P + div - 1) // div, d, generator=g).to(torch.float32 if f32 else torch.bfloat16)
    w = torch.randn(P, generator=g)
    kd, rd, wd = keys.to(DEV), rows.to(DEV), w.to(DEV)
    print(f"segment_reduce P={P} V={V} d={d} div={div} f32={f32}", flush=True)
    got = H.segment_reduce_rows(kd, V, rd, w=wd, row_div=div)
    assert torch.equal(got, H.segment_reduce_rows(kd, V, rd, w=wd, row_div=div))
    ok = (keys >= 0) & (keys < V)
    want, mag = torch.zeros(V, d, dtype=torch.float64), torch.zeros(V, d, dtype=torch.float64)
    at = ok.nonzero().flatten()
    for part in at.split(1 << 16):
        x = rows[part // div].double() * w[part].double()[:, None]
        want.index_add_(0, keys[part], x)
        mag.index_add_(0, keys[part], x.abs())
    # one rounding per product and addition: a chunk of at most 128 pairs, then the chunks of a key
    # in turn (at least 64 pairs each), then the sum with what was there
    n = torch.bincount(keys[ok], minlength=V).double()[:, None]
    bound = (128 + n / 64 + 3) * 2.0 ** -24 * mag
    assert bool(((got.cpu().double() - want).abs() <= bound).all())
    acc = torch.ones_like(got)
    H.segment_reduce_rows(kd, V, rd, w=wd, row_div=div, out=acc, accumulate=True)
    assert bool(((acc.cpu().double() - want - 1.0).abs() <= bound + 2.0 ** -23 * (1.0 + want.abs())).all())


def test_no_key_in_range():
    from rte_amd.kernels import hip_ops as H

    keys = torch.full((5000,), -1, device=DEV)
    keys[::2] = 2000
    rows = torch.randn(5000, 520, device=DEV)
    print("segment_reduce without a valid key", flush=True)
    assert not bool(H.segment_reduce_rows(keys, 2000, rows).any())
    acc = torch.ones(2000, 520, device=DEV)
    H.segment_reduce_rows(keys, 2000, rows, out=acc, accumulate=True)
    assert bool((acc == 1).all())
