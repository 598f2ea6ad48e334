"""The small-problem and any-alignment GEMM kernels (sh_gemm_small.hip, the late-fold 64 x 64 tile) on the GPU: every variant
forced (SH_GEMM_SMALL) against the tile table (SH_GEMM_SMALL=-2) at tile and slice edges, and odd operands against float64.

Every unsplit call (splits = 1) is one chain of 16-k blocks per output and stores the table's bits; with the split left to the
library (splits = 0) the variants that sum K in up to four ranges differ by the fp32 summation order only, so their fp16 outputs
differ by at most one rounding each (2^-11 relative, more only through a cancelling z_old or residual, which is added to the
rounded product): the difference's norm is held to 2^-11 of the result's."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import codes, to_dev, to_np
from softhier_mlir_amd import data, shops

pytestmark = pytest.mark.gpu
A = shops.addr
RANGES32, RANGES64, ANY64, ANY128, DMA, DMA2 = range(6)


def _f32(*shape):
    import torch
    return torch.empty(shape, dtype=torch.float32, device="cuda")


@pytest.mark.parametrize("wt", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (33, 40, 64), (50, 720, 720), (130, 200, 136), (257, 96, 768), (65, 32, 2048)])
def test_variants_against_the_table(lib, gpu, monkeypatch, M, N, K, wt):
    import torch
    P = N // 32 if N % 32 == 0 else 0
    x, w = data.normal((M, K), 11), data.normal((K, N), 12, std=1 / np.sqrt(K))
    X, W = to_dev(x), to_dev(np.ascontiguousarray(w.T) if wt else w)
    B16, R, Z0 = to_dev(data.normal((1, N), 13)), to_dev(data.normal((M, N), 14)), to_dev(data.normal((M, N + 8), 15))
    B32 = torch.from_numpy(data.normal((1, N), 16).astype(np.float32)).cuda()
    C = torch.from_numpy(data.normal((1, N), 17).astype(np.float32)).cuda()
    ST = torch.from_numpy(np.abs(data.normal((M, 2), 18).astype(np.float32)) + 0.5).cuda()
    PARTS = torch.from_numpy(np.abs(data.normal((M, max(1, K // 32), 2), 19).astype(np.float32)) + 0.5).cuda()
    FP32, GELU = shops.SH_BIAS_FP32, shops.SH_ACT_GELU
    epis = {"plain": (lambda s, n: shops.epi(splits=n), None), "gelu": (lambda s, n: shops.epi(bias=A(B16), act=GELU, splits=n), None),
            "res": (lambda s, n: shops.epi(bias=A(B16), residual=A(R), ldr=N, splits=n), None),
            "b32_acc": (lambda s, n: shops.epi(bias=A(B32), bias_fmt=FP32, residual=A(R), ldr=N, splits=n), shops.cfg(accumulate=1))}
    if K % 64 == 0:
        epis["fold"] = (lambda s, n: shops.epi(bias=A(B32), bias_fmt=FP32, act=GELU, ln_stats=A(ST), ln_c=A(C), splits=n), None)
        epis["fold_parts"] = (lambda s, n: shops.epi(bias=A(B32), bias_fmt=FP32, ln_stats=A(PARTS), ln_c=A(C), ln_parts=K // 32,
                                                     ln_eps=1e-6, splits=n), None)
        if P:
            epis["stats"] = (lambda s, n: shops.epi(bias=A(B16), residual=A(R), ldr=N, stats_out=A(s), splits=n), None)
    fn = lib.sh_gemm_ex_wt if wt else lib.sh_gemm_ex
    for name, (mk, cfg) in epis.items():
        outs = {}
        for v, n in [(-2, 1)] + [(v, n) for v in (RANGES32, RANGES64, ANY64, ANY128, DMA, DMA2, -1) for n in (1, 0)]:
            monkeypatch.setenv("SH_GEMM_SMALL", str(v))
            Z, S = Z0.clone(), _f32(M, max(P, 1), 2).zero_()
            assert fn(A(X), A(W), A(Z), M, N, K, K, K if wt else N, N + 8, cfg, mk(S, n)) == 0, (name, v, n, shops.last_error())
            outs[v, n] = (codes(Z), to_np(Z)[:, :N].astype(np.float64), to_np(S))
        ref = outs[-2, 1]
        for v, (c, z, s) in outs.items():
            assert np.array_equal(c[:, N:], codes(Z0)[:, N:]), (name, v, "wrote outside the view")
            # (the table takes W^T with K % 64 != 0, and K < 64, in another order)
            if v[1] == 1 and K >= 64 and not (wt and K % 64):
                assert np.array_equal(c, ref[0]), (name, v)
                assert np.array_equal(s, ref[2]) or name != "stats", (name, v)
            assert np.linalg.norm(z - ref[1]) <= 2.0 ** -11 * np.linalg.norm(ref[1]), (name, v)
            if name == "stats":                            # the partials of what this variant stored
                zb = z.reshape(M, P, 32)
                mag = np.abs(zb).sum(2)
                assert np.all(np.abs(s[..., 0] - zb.sum(2)) <= 32 * 2.0 ** -24 * mag), v
                m2 = ((zb - zb.mean(2, keepdims=True)) ** 2).sum(2)
                assert np.all(np.abs(s[..., 1] - m2) <= 64 * 2.0 ** -24 * (m2 + mag ** 2 / 32)), v


@pytest.mark.parametrize("wt", [False, True])
@pytest.mark.parametrize("M,N,K,px,pw,pz,off", [(70, 45, 37, 1, 3, 2, 1), (33, 9, 12, 0, 0, 0, 0), (100, 100, 588, 0, 0, 0, 0),
                                                (257, 131, 77, 3, 1, 5, 1), (1, 333, 64, 0, 1, 0, 0), (64, 1001, 199, 0, 0, 0, 1)])
def test_odd_operands_against_float64(lib, gpu, monkeypatch, M, N, K, px, pw, pz, off, wt):
    """Odd sizes, leading dims and bases, the operands' buffers ending with their last element; nothing outside the output
    view changes. fp32 sums of at most 588 products and three fp16 roundings: 4 x 2^-11 of the result's norm."""
    import torch
    rows, cols = (N, K) if wt else (K, N)
    ldx, ldw, ldz = K + px, cols + pw, N + pz
    g = torch.Generator(device="cuda").manual_seed(3)
    rn = lambda n, s=1.0: (torch.randn(n, generator=g, device="cuda") * s).half()   # noqa: E731
    xb, wb, zb0 = rn((M - 1) * ldx + K + off), rn((rows - 1) * ldw + cols + off, K ** -0.5), rn(M * ldz + off)
    b, r = rn(N + 1), rn(M * N)
    view = lambda t, n, c, ld: torch.as_strided(t, (n, c), (ld, 1), off)             # noqa: E731
    x, w = view(xb, M, K, ldx).double(), view(wb, rows, cols, ldw).double()
    prod = x @ (w.t().contiguous() if wt else w)
    fn = lib.sh_gemm_ex_wt if wt else lib.sh_gemm_ex
    outside = torch.ones_like(zb0, dtype=torch.bool)
    view(outside, M, N, ldz).fill_(False)
    for name, mk, cfg, want in (("plain", lambda n: shops.epi(splits=n), None, prod),
                                ("res", lambda n: shops.epi(bias=A(b, 1), residual=A(r), ldr=N, splits=n), None,
                                 prod + b[1:].double() + r.view(M, N).double()),
                                ("acc", lambda n: shops.epi(splits=n), shops.cfg(accumulate=1), prod + view(zb0, M, N, ldz).double())):
        for v in [(v, n) for v in (RANGES32, RANGES64, ANY64, ANY128, -1) for n in (1, 0)]:
            monkeypatch.setenv("SH_GEMM_SMALL", str(v[0]))
            e = mk(v[1])
            zb = zb0.clone()
            assert fn(A(xb, off), A(wb, off), A(zb, off), M, N, K, ldx, ldw, ldz, cfg, e) == 0, (name, v, shops.last_error())
            err = (view(zb, M, N, ldz).double() - want).norm() / want.norm()
            assert err <= 4 * 2.0 ** -11, (name, v, float(err))
            assert torch.equal(zb.view(torch.int16)[outside], zb0.view(torch.int16)[outside]), (name, v)


@pytest.mark.parametrize("N,K,off", [(768, 768, 0), (768, 3072, 0), (2304, 768, 0), (960, 960, 0), (64, 64, 0), (720, 2056, 0), (504, 136, 0),
                                     (717, 589, 0), (768, 768, 1), (100, 3001, 0)])
def test_an_unsplit_product_is_one_chain(lib, gpu, N, K, off):
    """splits = 1: a row's bits depend neither on the rows beside it (one sequence alone or in a batch), whichever kernel its
    problem size takes, nor on the epilogue (the fold with mu = 0, r = 1, c = d = 0 and a zero residual add nothing)."""
    import torch
    M = 4096
    g = torch.Generator(device="cuda").manual_seed(7)
    xb = torch.randn(M * K + off, generator=g, device="cuda").half()
    W = (torch.randn(K, N, generator=g, device="cuda") * K ** -0.5).half()
    R, P = torch.zeros(M, N, device="cuda", dtype=torch.float16), N // 32
    outs = {}
    for m in (1, 33, 50, 256, 588, 1024, M):
        Z = torch.empty(m, N, device="cuda", dtype=torch.float16)
        assert lib.sh_gemm_ex(A(xb, off), A(W), A(Z), m, N, K, K, N, N, None, shops.epi()) == 0, shops.last_error()
        outs[m] = codes(Z)
    for m in outs:
        assert np.array_equal(outs[m], outs[M][:m]), m
    z = outs[M].view(np.float16)
    if off or K % 8 or N % 8:
        return
    ST = torch.tensor([0.0, 1.0], device="cuda").repeat(M, 1).contiguous()
    Z32 = torch.zeros(N, device="cuda")
    for m in (50, 256, 588, 1024):
        epis = {"res": (shops.epi(residual=A(R), ldr=N), None)}
        if K % 64 == 0:
            epis["fold"] = (shops.epi(bias=A(Z32), bias_fmt=shops.SH_BIAS_FP32, ln_stats=A(ST), ln_c=A(Z32)), None)
        if N % 32 == 0:
            S = _f32(m, P, 2)
            epis["stats"] = (shops.epi(residual=A(R), ldr=N, stats_out=A(S)), None)
        for name, (e, cfg) in epis.items():
            Z = torch.empty(m, N, device="cuda", dtype=torch.float16)
            assert lib.sh_gemm_ex(A(xb), A(W), A(Z), m, N, K, K, N, N, cfg, e) == 0, (name, shops.last_error())
            assert np.array_equal(to_np(Z), z[:m]), (name, m)          # (values: -0 + 0 is +0)


def test_a_forced_split_count_reaches_small_problems(lib, gpu, monkeypatch):
    """SH_GEMM_SPLITS sets the split of a call that leaves it to the library: the bits of the same request."""
    import torch
    M, N, K = 256, 512, 1536
    X, W = to_dev(data.normal((M, K), 21)), to_dev(data.normal((K, N), 22, std=1 / np.sqrt(K)))
    z = {}
    for name, splits, env in (("asked", 3, None), ("forced", 0, "3"), ("free", 0, None)):
        monkeypatch.setenv("SH_GEMM_SPLITS", env) if env else monkeypatch.delenv("SH_GEMM_SPLITS", raising=False)
        Z = torch.empty(M, N, device="cuda", dtype=torch.float16)
        assert lib.sh_gemm_ex(A(X), A(W), A(Z), M, N, K, K, N, N, None, shops.epi(splits=splits)) == 0, shops.last_error()
        z[name] = codes(Z)
    assert np.array_equal(z["asked"], z["forced"])
    assert not np.array_equal(z["free"], z["forced"])                  # (four or eight ranges without it)
