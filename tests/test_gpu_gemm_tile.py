"""The tiled GEMM for more than 64 token rows (csrc/gemm_tile.hip) where it can go wrong: the edges of
its tiles in rows and columns, each tile shape its cost estimate picks, strided rows, every epilogue.

Up to 256 rows it adds the partial sums the 64-row kernel adds, so it is compared with that kernel bit
for bit; above, each output is one chain of fp32 products, within half a bf16 ulp plus the fp32 order
slack of the exact product (as tests/test_gpu_gemm.py derives it).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, pkg
from test_gpu_gemm import _bits, _exact, _order_slack, _rand, _ulp_bf16
from oracle import bf16

pytestmark = pytest.mark.gpu
gemm = pkg("gemm")


# Tiles of 64, 128 and 256 rows and 64, 128 and 256 columns; one row more than a tile, one less; K from one
# stage pair up, with 1, 2 and 4 partial sums; columns that are no multiple of 16 or of a lane's 4.
@pytest.mark.parametrize("m,k,n", [(65, 128, 40), (129, 256, 100), (127, 2048, 4096), (256, 6144, 64),
                                   (193, 2304, 2048), (256, 1024, 12_288)])
@pytest.mark.parametrize("epi", ["store", "silu", "add", "partial"])
def test_up_to_256_rows_equal_64_row_slices(m: int, k: int, n: int, epi: str) -> None:
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    x = _rand(g, m, k + 24)[:, :k]  # strided rows
    w = _rand(g, 2 * n if epi == "silu" else n, k, std=0.02)
    weights = [w] if epi == "silu" and n % 16 else [w, gemm.pack_weight(w)]
    for wt in weights:
        announce("tile", m, k, n, epi, type(wt).__name__)
        if epi == "partial":
            splits = gemm.partial_splits(n, k)
            got = torch.full((splits, m, n), float("nan"), device="cuda")
            gemm.linear_partial(x, wt, got)
            for r0 in range(0, m, 64):
                want = torch.full((splits, min(64, m - r0), n), float("nan"), device="cuda")
                gemm.linear_partial(x[r0:r0 + 64], wt, want)
                torch.cuda.synchronize()
                assert torch.equal(got[:, r0:r0 + 64], want), r0
            continue
        if epi == "add":
            r = _rand(g, m, n)
            got = gemm.linear_add_(r.clone(), x, wt)
            want = torch.cat([gemm.linear_add_(r[r0:r0 + 64].clone(), x[r0:r0 + 64], wt) for r0 in range(0, m, 64)])
        else:
            fn = gemm.linear if epi == "store" else gemm.linear_silu_mul
            got, want = fn(x, wt), torch.cat([fn(x[r0:r0 + 64], wt) for r0 in range(0, m, 64)])
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_silu_of_every_bf16_value() -> None:
    """One-hot token rows and weights holding every bf16 gate value, infinities and NaN among them (up rows 1): the
    tiled kernel's SiLU gives the bits of the 64-row kernel's expf and correctly rounded divide."""
    values = torch.arange(65_536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).cuda()
    w = torch.zeros(2 * values.numel(), 128, dtype=torch.bfloat16, device="cuda")
    w[:values.numel(), 0], w[values.numel():, 0] = values, 1.0
    x = torch.zeros(72, 128, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = 1.0
    announce("silu of every value")
    got, want = gemm.linear_silu_mul(x, w), gemm.linear_silu_mul(x[:64], w)
    torch.cuda.synchronize()
    assert torch.equal(got[:64].view(torch.int16), want.view(torch.int16))
    assert torch.equal(got[71].view(torch.int16), want[0].view(torch.int16))


# Rows of NaN with payloads and signs of their own, of infinities and of their differences: the NaN outputs have the
# canonical bits of the 64-row kernel, in whole column groups and in a last one of two columns.
@pytest.mark.parametrize("m", [64, 72, 300])
@pytest.mark.parametrize("n", [1024, 42])
@pytest.mark.parametrize("epi", ["store", "silu", "add"])
def test_nan_outputs_are_canonical(m: int, n: int, epi: str) -> None:
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x, w, r = _rand(g, m, 256), _rand(g, 2 * n if epi == "silu" else n, 256, std=0.02), _rand(g, m, n)
    odd = torch.tensor([0x7F81, -0x7F, 0x7FC1, -0x3B, 0x7F80, -0x80], dtype=torch.int16).view(torch.bfloat16).cuda()
    w[:30:5, 3], w[33, 200], r[5, 30:36], r[m - 1, 9] = odd, float("inf"), odd, odd[1]
    x[7, 11], x[m - 2, 17] = odd[3], float("inf")

    def fn(x: torch.Tensor, r: torch.Tensor) -> torch.Tensor:
        y = torch.empty(r.shape[0], n + 2, dtype=torch.bfloat16, device="cuda")[:, :n] if n == 42 else torch.empty_like(r)
        if epi == "add":
            return gemm.linear_add_(y.copy_(r), x, w)
        return (gemm.linear if epi == "store" else gemm.linear_silu_mul)(x, w, out=y)

    announce("nan", m, n, epi)
    got, want = fn(x, r), torch.cat([fn(x[i:i + 64], r[i:i + 64]) for i in range(0, m, 64)])
    torch.cuda.synchronize()
    assert torch.equal(got.isnan(), want.isnan()) and bool(got.isnan().any())
    assert bool((got.contiguous().view(torch.int16)[got.isnan()] == 0x7FC0).all())
    if m <= 256:
        assert torch.equal(got.contiguous().view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,k,n", [(257, 128, 40), (300, 2048, 4096), (513, 384, 1000), (1025, 1024, 12_288)])
@pytest.mark.parametrize("epi", ["store", "silu", "add"])
def test_tall_rows_match_exact_products(m: int, k: int, n: int, epi: str) -> None:
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    x = _rand(g, m, k + 8)[:, :k]
    w = _rand(g, 2 * n if epi == "silu" else n, k, std=0.02)
    r = _rand(g, m, n)
    rows = np.r_[0:16, 120:136, m - 16:m]  # of the first tile, a tile edge, the last tile
    exact = _exact(x[rows], w)
    slack = _ulp_bf16(exact) + _order_slack(x[rows], w)
    for wt in ([w] if epi == "silu" and n % 16 else [w, gemm.pack_weight(w)]):
        announce("tall", m, k, n, epi, type(wt).__name__)
        out = {"store": lambda: gemm.linear(x, wt), "silu": lambda: gemm.linear_silu_mul(x, wt),
               "add": lambda: gemm.linear_add_(r.clone(), x, wt)}[epi]()
        torch.cuda.synchronize()
        assert bool(torch.isfinite(out).all())
        got = bf16.to_f32(_bits(out[rows])).astype(np.float64)
        if epi == "store":
            assert (np.abs(got - exact) <= slack).all()
        elif epi == "add":
            want = bf16.round_f32(exact.astype(np.float32)).astype(np.float64) + bf16.to_f32(_bits(r[rows]))
            assert (np.abs(got - want) <= slack + _ulp_bf16(want)).all()
        else:
            # |d silu / d gate| <= 1.1; each of gate, up, silu and the product rounds once.
            gate, up = exact[:, :n], exact[:, n:]
            silu = gate / (1.0 + np.exp(-gate))
            bound = (1.1 * slack[:, :n] + _ulp_bf16(silu)) * (np.abs(up) + slack[:, n:]) + slack[:, n:] * np.abs(silu)
            assert (np.abs(got - silu * up) <= bound + _ulp_bf16(silu * up)).all()
