"""The register-pipelined tile GEMM (csrc/gemm_tile.hip) at the sizes where it can go wrong: tile
edges, odd numbers of k tiles, ragged layout-T reductions (rows past the end come back as zeros),
split reductions, and its epilogues (residual / beta / alpha, bf16 and fp32 output, SwiGLU forward
and backward), against float64 on the CPU.

Tolerances: bf16 operands are exact in float64; an fp32 sum of K products is off by at most about
sqrt(K) 2^-24 of the row norms (Frobenius, factor 8 for the worst draw), a bf16 output by 2^-9."""

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
    return float((got.double().cpu() - ref).norm() / ref.norm())


def _mat(rows, cols, g):
    return torch.randn(rows, cols, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("lay,M,N,K", [
    ("nn", 65, 72, 128),        # the general kernel
    ("nn", 3079, 2104, 128),    # one k tile per stage, ragged tile edges
    ("nn", 7, 520, 512),        # few rows, short reduction: unsplit
    ("nn", 129, 136, 192),      # three k tiles: short k and few outputs, the general kernel
    ("nn", 3080, 2104, 192),    # the same k over enough outputs: three k tiles in two stages
    ("nn", 130, 136, 320),      # five k tiles in two stages
    ("nn", 300, 200, 576),
    ("nn", 4096, 4160, 320),    # 256 x 256 tiles with ragged columns, odd tile count
    ("nt", 257, 264, 448),
    ("nt", 1000, 512, 4096),    # split reduction over activation rows
    ("tt", 136, 128, 129),      # ragged reductions: one row past, most of a tile missing, long
    ("tt", 72, 264, 200),
    ("tt", 512, 520, 8191),     # split, the last chunk ragged
    ("tt", 4096, 4352, 1000),   # 256 x 256 tiles, ragged reduction
    ("tt", 96, 96, 127),        # below the kernel's shortest reduction: the general kernel
])
@pytest.mark.parametrize("f32", [True, False])
def test_layouts(lay, M, N, K, f32):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(M * 31 + N * 7 + K)
    a = _mat(K, M, g) if lay[0] == "t" else _mat(M, K, g)
    b = _mat(K, N, g) if lay[1] == "t" else _mat(N, K, g)
    ref = (a.double().t() if lay[0] == "t" else a.double()) @ (b.double() if lay[1] == "t" else b.double().t())
    got = H.gemm(a.to(DEV), b.to(DEV), a_t=lay[0] == "t", b_t=lay[1] == "t", out_f32=f32)
    tol = 8 * K**0.5 * 2**-24 if f32 else 2**-9
    assert _rel(got, ref) <= tol
    again = H.gemm(a.to(DEV), b.to(DEV), a_t=lay[0] == "t", b_t=lay[1] == "t", out_f32=f32)
    assert torch.equal(got, again)


@pytest.mark.parametrize("M,K", [(200, 256), (1000, 4096)])  # unsplit, split
def test_epilogue_terms(M, K):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(3)
    N = 136
    a, b = _mat(M, K, g), _mat(N, K, g)
    r, c = torch.randn(M, N, generator=g), torch.randn(M, N, generator=g)
    ref = 0.5 * (a.double() @ b.double().t()) + r.double() - 2.0 * c.double()
    got = H.gemm(a.to(DEV), b.to(DEV), alpha=0.5, resid=r.to(DEV), out=c.to(DEV), beta=-2.0, out_f32=True)
    assert _rel(got, ref) <= 8 * K**0.5 * 2**-24


def _fresh():
    """Every stream's workspace is given back: the next call asks for its own."""
    from rte_amd.kernels import hip_ops as H

    torch.cuda.synchronize()
    H._WS.clear()


def test_rows_do_not_depend_on_their_company():
    """An activation row's product has the same bits alone, in a small call and in a larger one
    (unsplit k: any sizes; a split k: those of one bucket, 1 / 1.4142 to 1.4142 times a power of two),
    with the workspace each call asks for."""
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(5)
    for N, K, sizes in ((520, 512, (64, 1088, 8192)), (520, 2048, (1024, 1088)), (512, 1024, (91, 96, 127, 128, 176)),
                        (512, 2048, (91, 96, 112, 128, 181)), (512, 2048, (363, 400, 511, 512, 724)),
                        (512, 8192, (65, 80, 90))):
        a, b = _mat(max(sizes), K, g).to(DEV), _mat(N, K, g).to(DEV)
        outs = []
        for m in sizes:
            _fresh()
            outs.append(H.gemm(a[:m].contiguous(), b, out_f32=True)[:min(sizes)])
        for m, o in zip(sizes, outs):
            assert torch.equal(o, outs[0]), (N, K, m)


@pytest.mark.parametrize("lay,M,N,K", [
    ("nn", 65, 512, 8192), ("nn", 100, 512, 1024), ("nn", 200, 512, 4096), ("nn", 96, 512, 2048),
    ("nt", 96, 512, 4096),         # the dense SwiGLU's input gradient of 96 tokens
    ("tt", 6144, 1024, 16384),     # its weight gradient: partials past 64 MiB
    ("tt", 1024, 3072, 8192), ("tt", 512, 512, 8192),
])
def test_splits_come_from_the_shape(lay, M, N, K):
    """The same product has the same bits with the workspace it asks for, with a longer one, and
    through the stream's workspace before and after a larger user has grown it."""
    from rte_amd import _lib
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    at, bt = lay[0] == "t", lay[1] == "t"
    a = torch.randn((K, M) if at else (M, K), device=DEV, generator=g).to(torch.bfloat16)
    b = torch.randn((K, N) if bt else (N, K), device=DEV, generator=g).to(torch.bfloat16)
    need = _lib.load().rte_gemm_workspace_bytes(M, N, K)
    outs = []
    for nbytes in (need, need + (512 << 20)):
        ws, out = torch.empty(nbytes, dtype=torch.uint8, device=DEV), torch.empty(M, N, device=DEV)
        _lib.call("rte_gemm_bf16", a.data_ptr(), a.shape[1], int(at), None, b.data_ptr(), b.shape[1], int(bt), None,
                  out.data_ptr(), N, 1, M, N, K, 1.0, 0.0, None, 0, ws.data_ptr(), nbytes, _lib.stream_ptr())
        outs.append(out)
    _fresh()
    outs.append(H.gemm(a, b, a_t=at, b_t=bt, out_f32=True))
    H.workspace(512 << 20, torch.device(DEV))
    outs.append(H.gemm(a, b, a_t=at, b_t=bt, out_f32=True))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


@pytest.mark.parametrize("d,hd,batches", [
    (128, 32, (1, 3, 40)), (256, 64, (1, 2, 17)),  # 33 rows on tiles, more on the general kernel
    (512, 64, (1, 4, 16, 40)),                     # tiles, general, general, tiles
])
def test_qkv_rope_by_rows(d, hd, batches):
    """QKV + RoPE of short k against float64, and a sample's rows the same bits in every batch."""
    from rte_amd import _lib

    g = torch.Generator().manual_seed(d)
    S, H = 33, d // hd
    x, w = _mat(max(batches) * S, d, g), _mat(3 * d, d, g)
    ang = torch.rand(S, hd // 2, generator=g).repeat_interleave(2, dim=1) * 6.0
    cos, sin = ang.cos().contiguous(), ang.sin().contiguous()
    xd, wd, cd, sd = (t.to(DEV) for t in (x, w, cos, sin))
    firsts = []
    for B in batches:
        out = torch.empty(3, B, H, S, hd, device=DEV, dtype=torch.bfloat16)
        need = _lib.load().rte_gemm_workspace_bytes(B * S, 3 * d, d)
        ws = torch.empty(max(need, 16), dtype=torch.uint8, device=DEV)
        _lib.call("rte_qkv_rope_fwd", xd.data_ptr(), wd.data_ptr(), cd.data_ptr(), sd.data_ptr(), B, S, H, hd,
                  out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), ws.data_ptr(), need, _lib.stream_ptr())
        firsts.append(out[:, 0])
        y = (x[:B * S].double() @ w.double().t()).view(B, S, 3, H, hd).permute(2, 0, 3, 1, 4)
        turned = torch.stack([-y[..., 1::2], y[..., 0::2]], dim=-1).flatten(-2)
        ref = torch.cat([y[:2] * cos.double() + turned[:2] * sin.double(), y[2:]])
        assert _rel(out, ref) <= 2**-9
    assert all(torch.equal(f, firsts[0]) for f in firsts[1:])


@pytest.mark.parametrize("T,d,F", [(5, 128, 32), (70, 192, 96), (300, 256, 1056), (2048, 512, 2048)])
def test_dense_swiglu(T, d, F):
    from rte_amd.kernels import hip_ops as H

    g = torch.Generator().manual_seed(T)
    x, dy = _mat(T, d, g), _mat(T, d, g)
    wug, wd = (torch.randn(2 * F, d, generator=g) * d**-0.5), (torch.randn(d, F, generator=g) * F**-0.5)
    args = [t.to(DEV).requires_grad_() for t in (x, wug, wd)]
    y = H.dense_swiglu(*args)
    grads = torch.autograd.grad(y, args, dy.float().to(DEV))
    ref_args = [t.to(torch.bfloat16).double().requires_grad_() for t in (x, wug, wd)]
    up, gate = (ref_args[0] @ ref_args[1].t()).chunk(2, dim=-1)
    ref = (up * torch.nn.functional.silu(gate)) @ ref_args[2].t()
    ref_grads = torch.autograd.grad(ref, ref_args, dy.double())
    # up, gate, z, dz, dug are each kept in bf16 (2^-9 relative at most, 2^-10 rms): a few of them meet
    for got, want in zip((y, *grads), (ref, *ref_grads)):
        assert _rel(got, want.detach()) <= 4 * 2**-9
