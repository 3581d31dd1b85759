"""Activations of bf16 projections: bf16 outputs take short forms (a division in seven instructions, GELU as a sigmoid), fp32 outputs the
exact ones; every kernel of the projections, over the whole range of bf16 inputs, infinities and NaN among them."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, F32 = pkg.VLA_DT_BF16, pkg.VLA_DT_F32


def ref(x, act):
    if act == pkg.VLA_ACT_RELU:
        return torch.where(x > 0, x, torch.zeros_like(x))
    u = x if act == pkg.VLA_ACT_SILU else 2 * 0.7978845608028654 * x * (1 + 0.044715 * x * x)
    return x / (1 + torch.exp(-u))


@pytest.mark.parametrize("act", [pkg.VLA_ACT_SILU, pkg.VLA_ACT_GELU, pkg.VLA_ACT_RELU])
@pytest.mark.parametrize("rows,env", [(48, {}), (4096, {}), (4096, {"VLA_GEMM_DL": 0})])
def test_every_bf16_value(tune, act, rows, env):
    for k, v in env.items():
        tune.set(k, v)
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    x = torch.cat([x[torch.isfinite(x)], x[~torch.isfinite(x)][::8]])  # every finite value, some NaN and both infinities
    x = torch.cat([x, torch.tensor([float("inf"), float("-inf")], device="cuda", dtype=torch.bfloat16)])
    if rows < 512:  # the few-row kernel: every 37th value and the last ones
        x = torch.cat([x[::37], x[-64:]])
    for lo in range(0, x.numel(), rows):  # one value per row, the other k zero
        v = x[lo:lo + rows]
        A = torch.zeros(v.numel(), 64, dtype=torch.bfloat16, device="cuda")
        A[:, 0] = v
        W = torch.ones(8, 64, dtype=torch.bfloat16, device="cuda")
        y, yf = torch.zeros(v.numel(), 8, dtype=torch.bfloat16, device="cuda"), torch.zeros(v.numel(), 8, device="cuda")
        pkg.call("vla_linear_act", A, W, None, None, y, BF16, BF16, v.numel(), 8, 64, act)
        pkg.call("vla_linear_act", A, W, None, None, yf, BF16, F32, v.numel(), 8, 64, act)
        want = ref(v.double(), act)[:, None].expand(-1, 8)
        nan, size = torch.isnan(want), torch.nan_to_num(v.double()).abs()[:, None]
        if act != pkg.VLA_ACT_RELU:
            assert torch.equal(torch.isnan(y.float()), nan) and torch.equal(torch.isnan(yf), nan)
        # one bf16 rounding (half an ulp of 8 significant bits, 2^-8 of the value); the exponential of an argument of size u is off by u 2^-23,
        # at most 1e-5 of the value here; an exponential past the largest number is infinite, the value zero, an error of up to |x| 2^-126
        ok = (y.double() - want).abs() <= (2.0 ** -8 + 1e-5) * want.abs() + 2.0 ** -126 * (1 + size)
        assert bool((ok | nan | torch.isinf(want)).all())
        # fp32: tanh form, half an ulp of 1 in 1 + tanh times x
        okf = (yf.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * size
        assert bool((okf | nan | torch.isinf(want)).all())


@pytest.mark.parametrize("rows,env", [(48, {}), (4096, {}), (4096, {"VLA_GEMM_DL": 0})])
def test_silu_of_bf16_outputs_is_the_exact_form_rounded(tune, rows, env):
    """The short form against the exact one (fp32 output), over every exponent from 2^-120 on, where e^-x overflows among them, and
    densely around one."""
    for k, v in env.items():
        tune.set(k, v)
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    x = x[torch.isinf(x) | (torch.isfinite(x) & (x.float().abs() > 2.0 ** -120))]
    if rows < 512:
        x = torch.cat([x[::37], x[(x.float() < -86) & (x.float() > -90)]])
    for lo in range(0, x.numel(), rows):
        v = x[lo:lo + rows]
        A = torch.zeros(v.numel(), 64, dtype=torch.bfloat16, device="cuda")
        A[:, 0] = v
        A[:, 1] = torch.where(torch.isfinite(v) & (v.float().abs() < 1e30), v, torch.zeros_like(v))
        W = torch.zeros(16, 64, dtype=torch.bfloat16, device="cuda")
        W[:, 0] = 1.0
        W[1:, 1] = torch.linspace(-0.01, 0.01, 15).to(torch.bfloat16)  # values between the bf16 ones
        y, yf = torch.zeros(v.numel(), 16, dtype=torch.bfloat16, device="cuda"), torch.zeros(v.numel(), 16, device="cuda")
        pkg.call("vla_linear_act", A, W, None, None, y, BF16, BF16, v.numel(), 16, 64, pkg.VLA_ACT_SILU)
        pkg.call("vla_linear_act", A, W, None, None, yf, BF16, F32, v.numel(), 16, 64, pkg.VLA_ACT_SILU)
        want = yf.to(torch.bfloat16)
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(y), nan)
        assert torch.equal(y[~nan].view(torch.int16), want[~nan].view(torch.int16)), (y[~nan] != want[~nan]).nonzero()[:4]
