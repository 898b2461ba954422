"""Prefill attention where a row's maximum rises from tile to tile, so that what was summed before it is rescaled
(by neither 0 nor 1), against a float64 softmax.

Tolerance: the largest probability of a row is exactly 1, so beside the output's bf16 rounding (2^-8 of it) only the
other keys' probabilities are rounded (2^-8 of their share of |v|); 1e-5 for the fp32 exponentials and sums.
"""

from __future__ import annotations

import pytest
import torch

from conftest import announce, pkg

pytestmark = pytest.mark.gpu
attention = pkg("attention")

# Key positions (one in each of four 64-key tiles) and their first components; all other keys score far below.
RISING = {5: 0.0, 100: 5.0, 170: 7.25, 250: 8.5}


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("h,kv", [(8, 8), (2, 1)])
def test_largest_probability_is_not_rounded(h: int, kv: int, causal: bool) -> None:
    n = 300
    g = torch.Generator().manual_seed(7)
    q, k = torch.zeros(n, h, 128), torch.zeros(n, kv, 128)
    # Row i, head j: log2-domain scores of 0.7 to 1.0 per unit of the key's first component.
    q[:, :, 0] = (0.7 + 0.3 * torch.rand(n, h, generator=g)) * 128 ** 0.5 / 1.4426950408889634
    k[:, :, 0] = -100.0
    for at, value in RISING.items():
        k[at, :, 0] = value
    q, k = q.bfloat16(), k.bfloat16()
    v = torch.randn(n, kv, 128, generator=g).bfloat16()
    announce("varlen rising maxima", h, kv, causal)
    out = attention.varlen(q.cuda(), k.cuda(), v.cuda(), torch.tensor([0, n], dtype=torch.int32).cuda(), n,
                           causal=causal)
    torch.cuda.synchronize()
    rows = torch.arange(5 if causal else 0, n)  # from the first row that sees one of the keys
    for head in range(h):
        kd, vd = k[:, head // (h // kv)].double(), v[:, head // (h // kv)].double()
        scores = q[rows, head].double() @ kd.t() * 128 ** -0.5
        if causal:
            scores.masked_fill_(torch.arange(n)[None] > rows[:, None], float("-inf"))
        p = torch.softmax(scores, -1)
        want = p @ vd
        p.scatter_(1, p.argmax(-1, keepdim=True), 0.0)
        bound = 2.0 ** -8 * (want.abs() + p @ vd.abs()) + 1e-5
        err = (out[rows, head].double().cpu() - want).abs()
        assert bool((err <= bound).all()), (head, (err / bound).max().item())
