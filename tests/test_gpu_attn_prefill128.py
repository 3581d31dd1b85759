"""bf16 attention of 128-wide heads with more workgroups than the chip has CUs: tiles straight into LDS, two workgroups a CU.  Every
observation has the bits that it has alone, on the kernel that stages tiles in registers (which test_gpu_kernels.py compares with the oracle)."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

D = 128


# rows per kv head 4 S: three and four row tiles per workgroup, ragged last ones; keys: less than a tile, one, one more, a ragged last tile whose cache
# row ends in it, several tiles; kv heads that do and do not fill the XCDs evenly
@pytest.mark.parametrize("B,S,Hq,Hkv,n_keys,t_max", [(53, 20, 20, 5, 20, 24), (33, 24, 32, 8, 64, 64), (90, 31, 12, 3, 65, 72), (11, 150, 20, 5, 150, 152),
                                                     (7, 301, 20, 5, 583, 584)])
@pytest.mark.parametrize("mask", ["none", "causal", "padded", "given"])
@pytest.mark.parametrize("dtype", [pkg.VLA_DT_BF16, pkg.VLA_DT_BF16_P2])
def test_many_workgroups(tune, B, S, Hq, Hkv, n_keys, t_max, mask, dtype):
    g = torch.Generator().manual_seed(1000 * n_keys + S)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    k = torch.full((B, Hkv, t_max, D), float("nan"), dtype=torch.bfloat16, device="cuda")  # stale cache contents
    vt = torch.full((B, Hkv, D, t_max), float("nan"), dtype=torch.bfloat16, device="cuda")
    k[:, :, :n_keys], vt[..., :n_keys] = rnd(B, Hkv, n_keys, D), rnd(B, Hkv, D, n_keys)
    q = rnd(B, S, Hq, D) * 4
    kind, n_prefix, pad, given = pkg.VLA_MASK_NONE, max(0, n_keys - S), (0, 0), None
    if mask == "causal":
        kind = pkg.VLA_MASK_CAUSAL_SUFFIX
    elif mask == "padded":  # whole tiles without a visible key among them
        n_prefix, pad = n_keys, (n_keys // 5, 3 * n_keys // 4 + 1)
    elif mask == "given":
        given = torch.randn(S, n_keys, generator=g)
        given[torch.rand(S, n_keys, generator=g) < 0.3] = float("-inf")
        given = given.cuda()
    assert (B * Hkv) * ((Hq // Hkv * S + 127) // 128) > 256 >= Hkv * ((Hq // Hkv * S + 127) // 128)

    def run(b0, b1, shift=0):
        n = b1 - b0
        kk, vv = k[b0:b1], vt[b0:b1]
        if shift:  # caches that 16-byte accesses would not hit aligned
            kk, vv = (torch.empty(x.numel() + shift, dtype=x.dtype, device="cuda")[shift:].view(x.shape).copy_(x) for x in (kk, vv))
        o = torch.full((n, S, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
        pkg.call("vla_attn_prefix_suffix", q[b0:b1], kk, vv, o, dtype, n, S, Hq, Hkv, D, t_max, n_keys, D ** -0.5, kind, n_prefix, pad[0], pad[1], given)
        return o

    every = run(0, B)
    assert torch.isfinite(every).all()
    for b in (0, B // 2, B - 1):
        assert torch.equal(run(b, b + 1)[0], every[b])
    assert torch.equal(run(0, B, 4), every)  # eight bytes off
    tune.set("VLA_ATTN_DL", 0)  # the kernel that stages tiles in registers, on the same launch
    assert torch.equal(run(0, B), every)
