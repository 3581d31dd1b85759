"""bf16 attention of 256-wide heads on workgroups of 16 or 32 rows whose wavefronts walk 64-key units of their own (attn_wide_kernel)."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, D = pkg.VLA_DT_BF16, 256


def reference(q, k, vt, n_keys, kind, n_prefix, pad, given):
    """float64; a row without a visible key gives zeros"""
    B, S, Hq, _ = q.shape
    grp = Hq // k.shape[1]
    kk = k[:, :, :n_keys].double().cpu().repeat_interleave(grp, 1)
    vv = vt[..., :n_keys].double().cpu().repeat_interleave(grp, 1).transpose(2, 3).contiguous()
    qq = q.double().cpu().transpose(1, 2).contiguous()
    s = torch.matmul(qq, kk.transpose(2, 3).contiguous()) * D ** -0.5
    key, row = torch.arange(n_keys)[None, :], torch.arange(S)[:, None]
    see = torch.ones(S, n_keys, dtype=torch.bool)
    if kind == pkg.VLA_MASK_CAUSAL_SUFFIX:
        see &= key < n_prefix + row + 1
    elif kind == pkg.VLA_MASK_PI0_STATE:
        see &= (row != 0) | (key < n_prefix + 1)
    see &= ~((key >= pad[0]) & (key < min(pad[1], n_prefix)))
    s = s.masked_fill(~see, float("-inf")) if given is None else s + given.double().cpu()
    p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
    return torch.matmul(p, vv).transpose(1, 2)


def error(got, want):
    return ((got.double().cpu() - want).norm() / want.norm()).item()


# rows: one, a block, one more, 32, ragged; keys: one, a unit, one more, a wavefront's second unit (257), partial units whose cache row
# ends in them (t_max no multiple of 64), several slices, several heads and observations; forced: more than one round of workgroups
@pytest.mark.parametrize("B,S,Hq,Hkv,n_keys,t_max,forced", [
    (1, 1, 1, 1, 1, 8, False), (1, 16, 1, 1, 64, 64, False), (2, 17, 2, 2, 65, 72, False), (1, 32, 1, 1, 128, 128, False),
    (3, 11, 6, 2, 257, 264, False), (1, 51, 8, 1, 842, 848, False), (2, 50, 8, 1, 955, 1024, False), (16, 50, 8, 1, 330, 336, False),
    (8, 51, 8, 1, 523, 528, False), (5, 3, 4, 4, 200, 200, False), (40, 50, 8, 1, 130, 136, True), (1, 1, 8, 1, 1990, 2000, False)])
@pytest.mark.parametrize("mask", ["none", "causal", "state", "padded", "given"])
@pytest.mark.parametrize("size", [1.0, 16.0])  # larger scores: the running maximum is renewed unit after unit
def test_attention_of_256_wide_heads(tune, B, S, Hq, Hkv, n_keys, t_max, forced, mask, size):
    """No further from float64 than the tiled kernel is: both round probabilities and outputs to bf16 (2^-9 each); the two
    roundings differ from kernel to kernel, hence a tenth, and 1e-4 where a norm of few values is their whole sum."""
    g = torch.Generator().manual_seed(1000 * n_keys + S)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    k = torch.full((B, Hkv, t_max, D), float("nan"), dtype=torch.bfloat16, device="cuda")  # stale cache contents
    vt = torch.full((B, Hkv, D, t_max), float("nan"), dtype=torch.bfloat16, device="cuda")
    k[:, :, :n_keys], vt[..., :n_keys] = rnd(B, Hkv, n_keys, D), rnd(B, Hkv, D, n_keys)
    q = rnd(B, S, Hq, D) * size
    kind, n_prefix, pad = pkg.VLA_MASK_NONE, max(0, n_keys - S), (0, 0)
    if mask == "causal":
        kind = pkg.VLA_MASK_CAUSAL_SUFFIX
    elif mask == "state":
        kind = pkg.VLA_MASK_PI0_STATE
    elif mask == "padded":  # whole units without a visible key among them; one key: none at all
        n_prefix, pad = n_keys, (n_keys // 5, 3 * n_keys // 4 + 1)
    given = None
    if mask == "given":
        given = 10 * torch.randn(S, n_keys, generator=g)
        given[torch.rand(S, n_keys, generator=g) < 0.3] = float("-inf")
        given[0] = float("-inf")  # a row without a key: zeros
        given[S // 2, : n_keys // 2] = -1e38  # beside any other key nothing
        given = given.cuda()
    want = reference(q, k, vt, n_keys, kind, n_prefix, pad, given)
    out = {}
    for rows in ("0", "1" if forced else "-1"):
        tune.set("VLA_ATTN_ROWS", rows)
        o = torch.full((B, S, Hq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
        pkg.call("vla_attn_prefix_suffix", q, k, vt, o, BF16, B, S, Hq, Hkv, D, t_max, n_keys, D ** -0.5, kind, n_prefix, pad[0], pad[1], given)
        out[rows] = o
    tiled, new = out.values()
    if want.norm() == 0:
        assert torch.equal(new, torch.zeros_like(new))
        return
    assert error(tiled, want) < 2 ** -8
    assert error(new, want) <= 1.1 * error(tiled, want) + 1e-4
    assert error(new, want) < 2 ** -8


@pytest.mark.parametrize("B,n_keys", [(1, 955), (5, 842), (8, 955), (16, 842)])  # four key slices, none, none, workgroups of 32 rows
@pytest.mark.parametrize("size", [0.25, 4.0])  # rows of many alike and of few dominating probabilities
def test_error_is_no_larger_than_the_tiled_kernels(tune, B, n_keys, size):
    """Over 100,000 rounded outputs and more the ratio of the two errors is known to 2 / sqrt(100,000), about half a per cent."""
    S, Hq = 50, 8
    g = torch.Generator().manual_seed(B + n_keys)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    k, vt, q = rnd(B, 1, 960, D), rnd(B, 1, D, 960), rnd(B, S, Hq, D) * size
    want = reference(q, k, vt, n_keys, pkg.VLA_MASK_NONE, 0, (0, 0), None)
    out = []
    for rows in ("0", "-1"):
        tune.set("VLA_ATTN_ROWS", rows)
        out.append(torch.empty_like(q))
        pkg.call("vla_attn_prefix_suffix", q, k, vt, out[-1], BF16, B, S, Hq, 1, D, 960, n_keys, D ** -0.5, pkg.VLA_MASK_NONE, 0, 0, 0, None)
    tiled, new = out
    assert not torch.equal(tiled, new)  # two kernels
    assert error(new, want) <= 1.006 * error(tiled, want)


def test_fp32_partials_pin_the_tiled_kernel(tune):
    """VLA_ATTN_PART_F32 says in what format the tiled kernel's key slices travel: alone it gives the bits that it gives with that kernel
    pinned, and they are those neither of fp16 partials nor of the kernel that this launch takes by itself."""
    B, S, Hq, n_keys = 1, 51, 8, 867
    g = torch.Generator().manual_seed(9)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    q, k, vt = rnd(B, S, Hq, D), rnd(B, 1, 896, D), rnd(B, 1, D, 896)

    def run(**env):
        tune.clear("VLA_ATTN_PART_F32", "VLA_ATTN_ROWS")
        for key, value in env.items():
            tune.set("VLA_ATTN_" + key, value)
        o = torch.empty_like(q)
        pkg.call("vla_attn_prefix_suffix", q, k, vt, o, BF16, B, S, Hq, 1, D, 896, n_keys, D ** -0.5, pkg.VLA_MASK_NONE, 0, 0, 0, None)
        return o

    f32 = run(PART_F32=1)
    assert torch.equal(f32, run(PART_F32=1, ROWS=0))
    assert not torch.equal(f32, run(ROWS=0)) and not torch.equal(f32, run())
