"""fp32 projections of few rows on narrow tiles (16x16x4 MFMA, K shared out over wavefronts and accumulators), both numbers of
rows in turn, against float64 products.  A sum of K products in fp32 is off by at most about sqrt(K) 2^-24 of its terms' norm;
1e-6 of the largest output covers K up to 2052."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, F32 = pkg.VLA_DT_BF16, pkg.VLA_DT_F32
TOL = 1e-6


def off(got, want):
    return ((got.double() - want).abs().max() / want.abs().max()).item()


def each_plan(tune):
    for plan in (1, 3):
        tune.set("VLA_GEMM_ROWS_PLAN", plan)
        yield plan


# rows and columns around the 16, 32 and 64 row tiles and the 16 columns; K of less than one 16-k group, of a partial one, of
# a partial stage (128 k), of fewer stages than the ring holds, of many
@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (16, 37, 52), (33, 200, 128), (50, 720, 960), (65, 96, 388), (64, 1601, 720), (130, 64, 2052)])
def test_linear(tune, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x, W = torch.randn(M, K, generator=g).cuda(), (torch.randn(N, K, generator=g) / K ** 0.5).cuda()
    b, gate, res = torch.randn(N, generator=g).cuda(), torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).cuda()
    lin = x.double() @ W.double().T
    for plan in each_plan(tune):
        y, ya, yg = (torch.zeros(M, N, device="cuda") for _ in range(3))
        yr, yb = res.clone(), torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
        room = torch.zeros(M * N + 1, device="cuda")  # an output four bytes off a 16-byte boundary
        pkg.call("vla_linear", x, W, None, None, y, F32, F32, M, N, K)
        pkg.call("vla_linear", x, W, b, yr, yr, F32, F32, M, N, K)  # in place: the residual is the output
        pkg.call("vla_linear_act", x, W, b, res, ya, F32, F32, M, N, K, pkg.VLA_ACT_SILU)
        pkg.call("vla_linear_gated", x, W, None, gate, res, yg, F32, F32, M, N, K)
        pkg.call("vla_linear", x, W, b, res.to(torch.bfloat16), yb, F32, BF16, M, N, K)
        pkg.call("vla_linear", x, W, None, None, room[1:], F32, F32, M, N, K)
        assert off(y, lin) < TOL and off(yr, lin + b + res) < TOL, plan
        assert off(ya, torch.nn.functional.silu(lin + b) + res) < TOL and off(yg, lin * gate + res) < TOL, plan
        assert off(yb, lin + b + res.to(torch.bfloat16)) < 2.0 ** -8, plan
        assert torch.equal(room[1:].view(M, N), y) and room[0] == 0, plan


def test_values_past_the_last_stage_are_not_multiplied(tune):
    """K = 132: the second stage holds 4 of 128 k.  An infinity in a row must reach that row alone."""
    M, N, K = 40, 48, 132
    g = torch.Generator().manual_seed(3)
    x, W = torch.randn(M, K, generator=g).cuda(), torch.randn(N, K, generator=g).cuda()
    x[5, K - 1] = float("inf")
    for plan in each_plan(tune):
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, F32, F32, M, N, K)
        assert torch.isfinite(y[torch.arange(M) != 5]).all() and torch.isinf(y[5]).all(), plan


@pytest.mark.parametrize("M,I,K", [(50, 2048, 720), (17, 32, 84), (65, 96, 256)])
def test_gated(tune, M, I, K):
    g = torch.Generator().manual_seed(M)
    x, W, b = torch.randn(M, K, generator=g).cuda(), (torch.randn(2 * I, K, generator=g) / K ** 0.5).cuda(), torch.randn(2 * I, generator=g).cuda()
    lin = x.double() @ W.double().T + b
    for plan in each_plan(tune):
        y, yb = torch.zeros(M, I, device="cuda"), torch.zeros(M, I, dtype=torch.bfloat16, device="cuda")
        pkg.call("vla_glu_linear", x, W, b, y, F32, F32, M, I, K, pkg.VLA_ACT_SILU, -1.0)
        pkg.call("vla_glu_linear", x, W, b, yb, F32, BF16, M, I, K, pkg.VLA_ACT_SILU, -1.0)
        want = torch.nn.functional.silu(lin[:, :I]) * lin[:, I:]
        assert off(y, want) < TOL and off(yb, want) < 2.0 ** -8, plan


@pytest.mark.parametrize("B,S,Hq,Hkv,D,K,rope,kv", [(1, 50, 15, 5, 64, 720, True, True), (2, 9, 4, 2, 64, 84, True, False), (1, 17, 4, 4, 48, 256, False, True), (3, 5, 8, 8, 40, 100, False, True),
                                                    (1, 51, 8, 1, 256, 320, True, True)])
def test_qkv(tune, B, S, Hq, Hkv, D, K, rope, kv):
    g = torch.Generator().manual_seed(S + D)
    M, P, nk = B * S, 9, Hkv if kv else 0
    N, T = (Hq + 2 * nk) * D, (P + S + 63) // 64 * 64
    x, W, b = torch.randn(M, K, generator=g).cuda(), (torch.randn(N, K, generator=g) / K ** 0.5).cuda(), torch.randn(N, generator=g).cuda()
    ang = torch.rand(S, D // 2, generator=g).cuda() * 6
    cos, sin = (ang.cos(), ang.sin()) if rope else (None, None)
    y = (x.double() @ W.double().T + b).view(B, S, Hq + 2 * nk, D)
    if rope:
        c, s = cos.double()[None, :, None], sin.double()[None, :, None]
        lo, hi = y[..., :D // 2].clone(), y[..., D // 2:].clone()
        y = torch.cat([torch.cat([lo * c - hi * s, hi * c + lo * s], -1)[:, :, :Hq + nk], y[:, :, Hq + nk:]], 2)
    for plan in each_plan(tune):
        q, kc, vc = torch.zeros(M, Hq * D, device="cuda"), torch.zeros(B, Hkv, T, D, device="cuda"), torch.zeros(B, Hkv, D, T, device="cuda")
        pkg.call("vla_attn_qkv_rope", x, W, b, F32, M, K, S, Hq, Hkv, int(kv), int(kv), D, cos, sin, q, kc, vc, T, P)
        assert off(q.view(B, S, Hq, D), y[:, :, :Hq]) < TOL, plan
        if kv:
            assert off(kc[:, :, P:P + S], y[:, :, Hq:Hq + Hkv].transpose(1, 2)) < TOL, plan
            assert off(vc[:, :, :, P:P + S], y[:, :, Hq + Hkv:].permute(0, 2, 3, 1)) < TOL, plan
            assert not kc[:, :, :P].any() and not kc[:, :, P + S:].any() and not vc[..., :P].any() and not vc[..., P + S:].any(), plan


@pytest.mark.parametrize("M,N,K,heads", [(50, 720, 960, None), (33, 2816, 1024, None), (51, 2560, 2048, None), (48, 8192, 720, None), (64, 8192, 2048, None), (17, 8192, 1024, None),
                                         (16, 36864, 720, None), (32, 40960, 256, None), (51, 20480, 1024, None),
                                         (51, 2560, 1024, (8, 1, 256)), (51, 2560, 2048, (8, 1, 256)), (50, 2880, 720, (15, 15, 64)), (64, 3072, 1024, (16, 16, 64))])
def test_default_tiles_add_in_short_sums(M, N, K, heads):
    """Plain and QKV products of up to 64 rows: 64 partial sums of n = K / 64 products each, added in pairs.  An
    addition is off by a 0.24 (2^-24)^2 share of its result's square (uniform rounding errors, values spread over a binade),
    a partial sum's square grows with its length: n / 2 + 6 times that in all.  Four times as long sums are off by 1.5 to 1.7 times as much."""
    g = torch.Generator().manual_seed(N + K)
    x, W = torch.randn(M, K, generator=g).cuda(), (torch.randn(N, K, generator=g) / K ** 0.5).cuda()
    if heads:
        Hq, Hkv, D = heads
        q, kc, vc = torch.zeros(M, Hq * D, device="cuda"), torch.zeros(1, Hkv, 64, D, device="cuda"), torch.zeros(1, Hkv, D, 64, device="cuda")
        pkg.call("vla_attn_qkv_rope", x, W, None, F32, M, K, M, Hq, Hkv, 1, 1, D, None, None, q, kc, vc, 64, 0)
        y = torch.cat([q, kc[0, :, :M].transpose(0, 1).reshape(M, -1), vc[0, :, :, :M].permute(2, 0, 1).reshape(M, -1)], 1)
    else:
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, F32, F32, M, N, K)
    want = x.double() @ W.double().T
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err < 2.0 ** -24 * (0.24 * (K / 128 + 6)) ** 0.5, err


@pytest.mark.parametrize("arch,batch", [("smolvla", 1), ("smolvla", 3), ("smolvla", 11), ("pi0", 1)])
def test_norms_inside_the_projection_launches(tmp_path, monkeypatch, arch, batch):
    """An fp32 model with its RMSNorms inside the projections (few rows) against the same model with norms as launches of
    their own: a norm inside rounds x w once and scales the sum, one apart rounds x rstd and times w; 1e-5 of the largest
    output as for the models themselves.  Batch 3 mixes both (the gated projection has too many tiles), from batch 11 on
    every projection of the suffix is the tiled one."""
    import os

    import numpy as np
    from test_gpu_chunk import ckpt, ffi, make_obs

    cfg = ckpt.smolvla_config(2, "f32", suffix_mask=1) if arch == "smolvla" else dict(ckpt.pi0_config(1), dtype="f32")
    cfg = dict(cfg, ffn_dim=1024)
    path = os.path.join(str(tmp_path), "m.vlaw")
    ckpt.write_synthetic(path, cfg, ckpt.synth_weights(cfg, seed=77))
    r = np.random.default_rng(5)
    obs = [make_obs(cfg, r, n_views=2) for _ in range(batch)]
    out = []
    for apart in (False, True):
        if apart:
            monkeypatch.setenv("VLA_NO_NORM_FUSION", "1")
        m = ffi.Model(path)
        out.append(np.asarray(m.predict_batch(obs), np.float64))
        m.close()
    assert np.abs(out[0] - out[1]).max() / np.abs(out[1]).max() < 1e-5
    assert not np.array_equal(out[0], out[1])  # the two are different launches (the final norm's too)
