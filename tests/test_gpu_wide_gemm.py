"""bf16 projections of many rows on the wide-tile kernel (16x16x32 MFMA, tiles up to 256 x 256), every tile pinned in turn:
against float32 products and, bit for bit, against the 64 x 64 kernel, whose products it adds in the same order."""
import numpy as np
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, F32 = pkg.VLA_DT_BF16, pkg.VLA_DT_F32
SMALL = 4   # VLA_GEMM_TILE of the 64 x 64 tiles
WIDE = range(16, 22)  # of the wide tiles


def rnd(gen, *shape, scale=1.0):
    return (torch.randn(*shape, generator=gen) * scale).to(torch.bfloat16).cuda()


def every_tile(tune, run):
    tune.set("VLA_GEMM_TILE", SMALL)
    want = run()
    for tile in WIDE:
        tune.set("VLA_GEMM_TILE", tile)
        for g, w in zip(run(), want):
            assert torch.equal(g, w), tile
    return want


def close(got, want):
    """bf16 outputs of fp32 sums: one rounding (2^-8 of the value) beside sums that differ by 1e-5 of the largest"""
    got, want = got.float(), want.float()
    return bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max()).all())


# one row; ragged rows and columns around the tiles' edges; K of one partial tile, of fewer tiles than a ring holds, of a
# partial last tile in either half (720 = 11 x 64 + 16, 1072 = 16 x 64 + 48), of whole tiles
@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (193, 200, 48), (257, 520, 128), (385, 333, 720), (400, 264, 1072), (520, 576, 512)])
def test_linear(tune, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x, W, res = rnd(g, M, K), rnd(g, N, K, scale=0.05), rnd(g, M, N)
    b, gate = torch.randn(N, generator=g).cuda(), torch.randn(N, generator=g).cuda()

    def run():
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, BF16, F32, M, N, K)
        yb = res.clone()  # in place: the residual is the output
        pkg.call("vla_linear", x, W, b, yb, yb, BF16, BF16, M, N, K)
        ya, yg = torch.zeros_like(res), torch.zeros_like(res)
        pkg.call("vla_linear_act", x, W, b, res, ya, BF16, BF16, M, N, K, pkg.VLA_ACT_GELU)
        pkg.call("vla_linear_gated", x, W, None, gate, res, yg, BF16, BF16, M, N, K)
        return y, yb, ya, yg

    y, yb, ya, yg = every_tile(tune, run)
    lin = x.double() @ W.double().T
    assert ((y - lin).abs().max() / lin.abs().max()).item() < 1e-5
    assert close(yb, lin + b + res)
    assert close(ya, torch.nn.functional.gelu(lin + b, approximate="tanh") + res)
    assert close(yg, lin * gate + res)


def test_values_past_a_partial_k_tile_are_not_multiplied(tune):
    """K = 80: the second k tile holds 16 of 64 k.  Infinities in a row must reach that row alone."""
    M, N, K = 130, 64, 80
    g = torch.Generator().manual_seed(3)
    x, W = rnd(g, M, K), rnd(g, N, K)
    x[5, K - 3] = float("inf")

    def run():
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, BF16, F32, M, N, K)
        return (y,)

    y, = every_tile(tune, run)
    assert torch.isfinite(y[torch.arange(M) != 5]).all() and torch.isinf(y[5]).all()


@pytest.mark.parametrize("M,I,K,eps", [(200, 96, 720, 1e-5), (130, 288, 64, -1.0), (385, 160, 528, 1e-6)])
def test_gated(tune, M, I, K, eps):
    g = torch.Generator().manual_seed(M)
    x, W = rnd(g, M, K, scale=2.0), rnd(g, 2 * I, K, scale=0.05)
    b = torch.randn(2 * I, generator=g).cuda()

    def run():
        y, yf = torch.zeros(M, I, dtype=torch.bfloat16, device="cuda"), torch.zeros(M, I, device="cuda")
        pkg.call("vla_glu_linear", x, W, b, y, BF16, BF16, M, I, K, pkg.VLA_ACT_SILU, eps)
        pkg.call("vla_glu_linear", x, W, None, yf, BF16, F32, M, I, K, pkg.VLA_ACT_SILU, eps)
        return y, yf

    y, yf = every_tile(tune, run)
    xd = x.double()
    if eps >= 0:
        xd = xd * torch.rsqrt((xd * xd).mean(1, keepdim=True) + eps)
    lin = xd @ W.double().T
    glu = lambda v: torch.nn.functional.silu(v[:, :I]) * v[:, I:]
    assert close(y, glu(lin + b))
    assert ((yf - glu(lin)).abs().max() / glu(lin).abs().max()).item() < 1e-5


@pytest.mark.parametrize("norm", ["none", "rms", "layer"])
@pytest.mark.parametrize("B,S,Hq,Hkv,D,K,rope,kv", [(5, 51, 8, 1, 256, 208, True, True), (4, 50, 15, 5, 64, 720, True, True),
                                                    (7, 49, 8, 8, 48, 96, False, True), (3, 50, 5, 5, 64, 720, True, False)])
def test_qkv(tune, B, S, Hq, Hkv, D, K, rope, kv, norm):
    g = torch.Generator().manual_seed(S + D)
    M, P, nk = B * S, 9, Hkv if kv else 0
    N, T = (Hq + 2 * nk) * D, (P + S + 63) // 64 * 64
    x, W = rnd(g, M, K, scale=2.0) + 0.5, rnd(g, N, K, scale=0.05)
    b, cs = torch.randn(N, generator=g).cuda(), W.float().sum(1)
    ang = torch.rand(S, D // 2, generator=g).cuda() * 6
    cos, sin = (ang.cos(), ang.sin()) if rope else (None, None)
    kv_args = (Hq, Hkv, int(kv), int(kv), D, cos, sin)

    def run():
        q = torch.zeros(M, Hq * D, dtype=torch.bfloat16, device="cuda")
        kc, vc = torch.zeros(B, Hkv, T, D, dtype=torch.bfloat16, device="cuda"), torch.zeros(B, Hkv, D, T, dtype=torch.bfloat16, device="cuda")
        head = {"none": ("vla_attn_qkv_rope", x, W, b), "rms": ("vla_rmsnorm_attn_qkv_rope", x, W, b),
                "layer": ("vla_layernorm_attn_qkv_rope", x, W, cs, b)}[norm]
        pkg.call(*head, BF16, M, K, S, *kv_args, q, kc, vc, T, P, *(() if norm == "none" else (1e-5,)))
        return q, kc, vc

    q, kc, vc = every_tile(tune, run)
    xd = x.double()
    if norm == "rms":
        xd = xd * torch.rsqrt((xd * xd).mean(1, keepdim=True) + 1e-5)
    if norm == "layer":
        xd = (xd - xd.mean(1, keepdim=True)) * torch.rsqrt(xd.var(1, unbiased=False, keepdim=True) + 1e-5)
    y = (xd @ W.double().T + b).view(B, S, Hq + 2 * nk, D)
    if rope:
        c, s = cos.double()[None, :, None], sin.double()[None, :, None]
        lo, hi = y[..., :D // 2].clone(), y[..., D // 2:].clone()
        rot = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
        y = torch.cat([rot[:, :, :Hq + nk], y[:, :, Hq + nk:]], 2)
    tol = lambda got, want: bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max()).all())
    assert tol(q.view(B, S, Hq, D), y[:, :, :Hq])
    if kv:
        assert tol(kc[:, :, P:P + S], y[:, :, Hq:Hq + Hkv].transpose(1, 2))
        assert tol(vc[:, :, :, P:P + S], y[:, :, Hq + Hkv:].permute(0, 2, 3, 1))
        assert not kc[:, :, :P].any() and not kc[:, :, P + S:].any() and not vc[..., :P].any() and not vc[..., P + S:].any()
