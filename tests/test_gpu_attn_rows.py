"""Attention of 48- and 64-wide heads with the key blocks shared out over a workgroup's wavefronts (pinned with VLA_ATTN_ROWS=1; bf16:
32 rows a workgroup, up to ten 64-key tiles, fp32: 16 rows), against float64."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, F32 = pkg.VLA_DT_BF16, pkg.VLA_DT_F32


def reference(q, k, v, scale, bias):
    """q [B, S, Hq, D]; k, v [B, Hkv, T, D] in float64; bias [S, T] of 0 and -inf or any value"""
    g = q.shape[2] // k.shape[1]
    s = torch.einsum("bshd,bhtd->bhst", q, k.repeat_interleave(g, 1)) * scale + bias
    m = s.amax(-1, keepdim=True)
    p = torch.exp(s - torch.where(torch.isinf(m), torch.zeros_like(m), m))
    l = p.sum(-1, keepdim=True)
    p = torch.where(l > 0, p / l, torch.zeros_like(p))
    return torch.einsum("bhst,bhtd->bshd", p, v.repeat_interleave(g, 1))


# row tiles with a ragged last one; key blocks: one of a single key, a partial last one, as many as wavefronts, more than those
# (fp32 10 of 32 keys; bf16 keys past its ten tiles take the tiled kernel), a cache row that ends inside the last block (t_max = 40, 104)
@pytest.mark.parametrize("D", [48, 64])
@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("B,S,Hq,Hkv,n_keys,t_max", [(1, 50, 15, 5, 227, 256), (2, 50, 15, 5, 291, 320), (3, 7, 4, 2, 33, 40), (1, 17, 9, 3, 1, 8), (1, 40, 3, 3, 100, 104),
                                                     (1, 33, 8, 1, 512, 512), (9, 16, 2, 1, 600, 640), (1, 1, 40, 1, 1000, 1024)])
@pytest.mark.parametrize("mask", ["none", "causal", "state", "padded", "given"])
def test_against_float64(tune, D, dtype, B, S, Hq, Hkv, n_keys, t_max, mask):
    tune.set("VLA_ATTN_ROWS", 1)
    tune.set("VLA_ATTN_DIRECT_ROWS", 0)  # few rows take a kernel of their own otherwise
    dt = torch.bfloat16 if dtype == BF16 else torch.float32
    g = torch.Generator().manual_seed(n_keys + S)
    q = torch.randn(B, S, Hq, D, generator=g).to(dt).cuda()
    k = torch.full((B, Hkv, t_max, D), float("nan"), dtype=dt, device="cuda")  # stale cache contents
    vt = torch.full((B, Hkv, D, t_max), float("nan"), dtype=dt, device="cuda")
    k[:, :, :n_keys] = torch.randn(B, Hkv, n_keys, D, generator=g).to(dt).cuda()
    vt[..., :n_keys] = torch.randn(B, Hkv, D, n_keys, generator=g).to(dt).cuda()
    n_prefix = max(0, n_keys - S)
    kind, pad, given = pkg.VLA_MASK_NONE, (0, 0), None
    bias = torch.zeros(S, n_keys, dtype=torch.float64, device="cuda")
    key, row = torch.arange(n_keys, device="cuda")[None], torch.arange(S, device="cuda")[:, None]
    if mask == "causal":
        kind = pkg.VLA_MASK_CAUSAL_SUFFIX
        bias[key > n_prefix + row] = float("-inf")
    elif mask == "state":
        kind = pkg.VLA_MASK_PI0_STATE
        bias[(row == 0) & (key > n_prefix)] = float("-inf")
    elif mask == "padded":
        pad = (n_keys // 4, n_keys // 2)
        n_prefix = n_keys
        bias[((key >= pad[0]) & (key < pad[1])).expand(S, -1)] = float("-inf")
    elif mask == "given":
        given = torch.randn(S, n_keys, generator=g).cuda()
        given[torch.rand(S, n_keys, generator=g).cuda() < 0.3] = float("-inf")
        given[0] = float("-inf")  # a row without a key: zeros
        bias = given.double()
    out = torch.full((B, S, Hq, D), float("nan"), dtype=dt, device="cuda")
    pkg.call("vla_attn_prefix_suffix", q, k, vt, out, dtype, B, S, Hq, Hkv, D, t_max, n_keys, D ** -0.5, kind, n_prefix, pad[0], pad[1], given)
    want = reference(q.double(), k[:, :, :n_keys].double(), vt[..., :n_keys].double().transpose(2, 3), D ** -0.5, bias)
    err = (out.double() - want).abs().max().item() / max(want.abs().max().item(), 1e-30)
    # bf16: probabilities and the output rounded to 2^-8 each.  fp32: a score of size 8 summed from 64 products is off by up to
    # 8 sqrt(64) 2^-24 = 4e-6, and its probability by that share of itself
    assert err < (2.0 ** -7 if dtype == BF16 else 4e-6), err
    first = out.clone()
    pkg.call("vla_attn_prefix_suffix", q, k, vt, out, dtype, B, S, Hq, Hkv, D, t_max, n_keys, D ** -0.5, kind, n_prefix, pad[0], pad[1], given)
    assert torch.equal(first, out)


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_an_infinity_in_the_last_piece_of_a_48_wide_key(tune, dtype):
    """K rows are kept 64 wide in LDS, the last piece repeated: an infinite key element gives an infinite score (probability
    one here), not a NaN from beside the head."""
    tune.set("VLA_ATTN_ROWS", 1)
    tune.set("VLA_ATTN_DIRECT_ROWS", 0)
    dt = torch.bfloat16 if dtype == BF16 else torch.float32
    q, k, vt = torch.ones(1, 20, 2, 48), torch.zeros(1, 2, 64, 48), torch.zeros(1, 2, 48, 64)
    k[0, 0, 3, 47] = float("-inf")  # that key is never seen by head 0
    vt[0, :, :, 3], vt[0, :, :, :3] = 5.0, 1.0
    q, k, vt = (t.to(dt).cuda() for t in (q, k, vt))
    out = torch.empty_like(q)
    pkg.call("vla_attn_prefix_suffix", q, k, vt, out, dtype, 1, 20, 2, 2, 48, 64, 4, 48 ** -0.5, pkg.VLA_MASK_NONE, 4, 0, 0, None)
    assert torch.equal(out[:, :, 0], torch.ones_like(out[:, :, 0])) and torch.equal(out[:, :, 1], torch.full_like(out[:, :, 1], 2.0))
