"""Plain bf16 projections on the wide-tile kernel's tiles of 32- and 48-column wavefronts, every tile pinned in turn: against float64
products and, bit for bit, against the 64 x 64 kernel, whose products they add in the same order."""
import pytest
import torch

from util import pkg

pytestmark = pytest.mark.gpu

BF16, F32 = pkg.VLA_DT_BF16, pkg.VLA_DT_F32
SMALL = 4                  # VLA_GEMM_TILE of the 64 x 64 tiles
PLAIN = range(22, 25)      # 96 x 96, 128 x 96, 96 x 64


# one row; rows, columns and K at and around the tiles' edges: columns that end in the first 32 or the last 16 of a 48-column
# wavefront, an N that four but not eight divides, K of one partial tile, of as many tiles as a ring holds, of more with a partial last one
@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (95, 40, 48), (96, 96, 192), (97, 100, 208), (128, 184, 320), (129, 333, 336), (193, 720, 960), (500, 392, 1072)])
def test_plain_tiles(tune, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x, W, res = (torch.randn(*s, generator=g).to(torch.bfloat16).cuda() for s in ((M, K), (N, K), (M, N)))
    b, gate, res_f = torch.randn(N, generator=g).cuda(), torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).cuda()

    def run():
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, BF16, F32, M, N, K)
        yf = res_f.clone()  # in place: the residual is the output
        pkg.call("vla_linear", x, W, b, yf, yf, BF16, F32, M, N, K)
        yb = res.clone()
        pkg.call("vla_linear", x, W, b, yb, yb, BF16, BF16, M, N, K)
        ya, yg = torch.zeros_like(res), torch.zeros_like(res)
        pkg.call("vla_linear_act", x, W, b, res, ya, BF16, BF16, M, N, K, pkg.VLA_ACT_GELU)
        pkg.call("vla_linear_gated", x, W, None, gate, res, yg, BF16, BF16, M, N, K)
        return y, yf, yb, ya, yg

    tune.set("VLA_GEMM_TILE", SMALL)
    want = run()
    for tile in PLAIN:
        tune.set("VLA_GEMM_TILE", tile)
        for got, w in zip(run(), want):
            assert torch.equal(got, w), tile
    lin = x.double() @ W.double().T
    # fp32 sums of K exact products: K 2^-24 of their absolute sum at most
    bound = K * 2.0 ** -24 * (x.double().abs() @ W.double().abs().T)
    assert ((want[0] - lin).abs() <= bound).all()
    # one more rounding of the sum with bias and residual to fp32, then to bf16
    out = lin + b + res.double()
    assert ((want[2] - out).abs() <= bound + 2.0 ** -8 * out.abs() + 2.0 ** -22 * (lin.abs() + b.abs() + res.double().abs())).all()


def test_an_infinite_row_reaches_that_row_alone(tune):
    """K = 80: the second k tile holds 16 of 64 k, the rest of it is read from valid addresses and not multiplied."""
    M, N, K = 200, 104, 80
    g = torch.Generator().manual_seed(3)
    x, W = (torch.randn(*s, generator=g).to(torch.bfloat16).cuda() for s in ((M, K), (N, K)))
    x[5, K - 3] = float("inf")
    for tile in PLAIN:
        tune.set("VLA_GEMM_TILE", tile)
        y = torch.zeros(M, N, device="cuda")
        pkg.call("vla_linear", x, W, None, None, y, BF16, F32, M, N, K)
        assert torch.isfinite(y[torch.arange(M) != 5]).all() and not torch.isfinite(y[5]).any(), tile
