"""bf16 attention of 48- and 64-wide heads: a launch of few workgroups takes a wavefront per 64-key tile, a larger one the tiled
kernel that walks the tiles.  Which one depends on the batch, so both have to give the same bits."""
import os

import numpy as np
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

from vla_cpp_amd import checkpoint as ckpt  # noqa: E402
from vla_cpp_amd import ffi  # noqa: E402

BF16 = pkg.VLA_DT_BF16


def inputs(B, S, Hq, Hkv, D, n_keys, t_max, size, seed=0):
    g = torch.Generator().manual_seed(1000 * n_keys + S + seed)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    k = torch.full((B, Hkv, t_max, D), float("nan"), dtype=torch.bfloat16, device="cuda")  # stale cache contents
    vt = torch.full((B, Hkv, D, t_max), float("nan"), dtype=torch.bfloat16, device="cuda")
    k[:, :, :n_keys], vt[..., :n_keys] = rnd(B, Hkv, n_keys, D), rnd(B, Hkv, D, n_keys)
    return rnd(B, S, Hq, D) * size, k, vt


def attend(q, k, vt, n_keys, kind, n_prefix, pad, given):
    (B, S, Hq, D), Hkv, t_max = q.shape, k.shape[1], k.shape[2]
    out = torch.full((B, S, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    pkg.call("vla_attn_prefix_suffix", q, k, vt, out, BF16, B, S, Hq, Hkv, D, t_max, n_keys, D ** -0.5, kind, n_prefix, pad[0], pad[1], given)
    return out


# ragged last row tile, one row; one tile of a single key, two tiles (one key slice of 64-wide heads), three (two slices), a partial
# last tile and a cache row that ends in it, five tiles (room for two workgroups a CU) and six, ten (the most)
@pytest.mark.parametrize("D", [48, 64])
@pytest.mark.parametrize("B,S,Hq,Hkv,n_keys,t_max", [(1, 50, 15, 5, 291, 320), (3, 7, 4, 2, 33, 40), (1, 17, 9, 3, 1, 8), (2, 40, 3, 3, 100, 104), (1, 49, 6, 6, 129, 136),
                                                     (1, 33, 8, 1, 320, 320), (2, 64, 2, 2, 321, 384), (1, 1, 40, 1, 640, 640), (9, 16, 2, 1, 600, 640)])
@pytest.mark.parametrize("mask", ["none", "causal", "state", "padded", "given"])
@pytest.mark.parametrize("size", [1.0, 24.0])  # larger scores: the running maximum is renewed tile after tile
def test_has_the_tiled_kernels_bits(tune, D, B, S, Hq, Hkv, n_keys, t_max, mask, size):
    tune.set("VLA_ATTN_DIRECT_ROWS", 0)  # few rows take a kernel of their own otherwise
    q, k, vt = inputs(B, S, Hq, Hkv, D, n_keys, t_max, size)
    kind, n_prefix, pad, given = pkg.VLA_MASK_NONE, max(0, n_keys - S), (0, 0), None
    if mask == "causal":
        kind = pkg.VLA_MASK_CAUSAL_SUFFIX
    elif mask == "state":
        kind = pkg.VLA_MASK_PI0_STATE
    elif mask == "padded":  # whole tiles without a visible key among them
        n_prefix, pad = n_keys, (n_keys // 5, 3 * n_keys // 4)
    elif mask == "given":
        g = torch.Generator().manual_seed(n_keys)
        given = 10 * torch.randn(S, n_keys, generator=g)
        given[torch.rand(S, n_keys, generator=g) < 0.3] = float("-inf")
        given[0] = float("-inf")  # a row without a key: zeros
        given[S // 2, : n_keys // 2] = torch.finfo(torch.float32).min
        given = given.cuda()
    out = {}
    for rows in (0, 1):
        tune.set("VLA_ATTN_ROWS", rows)
        out[rows] = attend(q, k, vt, n_keys, kind, n_prefix, pad, given)
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("D,S,Hq,Hkv,n_keys,t_max,B", [(64, 50, 15, 5, 291, 320, 32), (64, 50, 15, 5, 241, 256, 24), (48, 49, 32, 32, 291, 320, 16)])
def test_an_observation_has_the_same_bits_alone_and_in_any_batch(D, S, Hq, Hkv, n_keys, t_max, B):
    """Default dispatch, on both sides of the rule."""
    q, k, vt = inputs(B, S, Hq, Hkv, D, n_keys, t_max, 1.0, seed=B)
    args = (n_keys, pkg.VLA_MASK_CAUSAL_SUFFIX, n_keys - S, (0, 0), None)
    whole = attend(q, k, vt, *args)
    for b in (0, 1, B - 1):
        assert torch.equal(attend(q[b:b + 1], k[b:b + 1], vt[b:b + 1], *args)[0], whole[b]), b
    for n in (2, 5, 8, 9, 11, 15):
        assert torch.equal(attend(q[:n], k[:n], vt[:n], *args), whole[:n]), n


@pytest.mark.parametrize("D", [48, 64])
def test_infinities_in_keys_and_values(tune, D):
    """An infinite key element (in the last piece, which 48-wide keys repeat in LDS) gives an infinite score, and what the output
    is then is the tiled kernel's answer too."""
    tune.set("VLA_ATTN_DIRECT_ROWS", 0)
    q, k, vt = inputs(1, 20, 4, 2, D, 150, 192, 1.0)
    q[:, :, 0], q[:, :, 1] = q[:, :, 0].abs(), -q[:, :, 1].abs()
    k[0, 0, 70, D - 1] = float("-inf")
    k[0, 1, 149, 3] = float("inf")
    vt[0, 1, D - 1, 5] = float("inf")
    out = {}
    for rows in (0, 1):
        tune.set("VLA_ATTN_ROWS", rows)
        out[rows] = attend(q, k, vt, 150, pkg.VLA_MASK_NONE, 150, (0, 0), None)
    a, b = (torch.where(torch.isnan(o), torch.zeros_like(o), o) for o in (out[0], out[1]))
    assert torch.equal(a, b) and torch.equal(torch.isnan(out[0]), torch.isnan(out[1]))
    assert torch.isfinite(out[1][0, :, 0]).all()


def test_an_action_chunk_has_the_same_bits_alone_and_in_a_served_batch(tmp_path):
    """The same through the model handle: SmolVLA's chunk of an observation alone and among 16 and 32."""
    cfg = dict(ckpt.smolvla_config(n_layers=4, dtype="bf16", suffix_mask=1), ffn_dim=2048)
    path = os.path.join(str(tmp_path), "batch.vlaw")
    ckpt.write_synthetic(path, cfg, ckpt.synth_weights(cfg, seed=77))
    r = np.random.default_rng(77)
    obs = [dict(img_emb=r.standard_normal((3 * cfg["n_img"], cfg["hidden"])).astype(np.float32) / np.float32(np.sqrt(cfg["hidden"])), n_views=3,
                lang=r.integers(0, cfg["vocab"], cfg["n_lang"]).astype(np.int32), state=r.standard_normal(cfg["max_state_dim"]).astype(np.float32),
                noise=r.standard_normal((50, cfg["max_action_dim"])).astype(np.float32)) for _ in range(32)]
    m = ffi.Model(path)
    alone = [m.predict(obs[i]).reshape(50, -1) for i in (0, 7, 15)]
    for n in (16, 32):
        got = m.predict_batch(obs[:n]).reshape(n, 50, -1)
        for i, want in zip((0, 7, 15), alone):
            assert np.array_equal(got[i], want), (n, i)
    m.close()
