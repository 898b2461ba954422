"""The LM head for 33 to 256 token rows (csrc/lm_head_wide.hip) where its vocab tiles and its epilogue can go wrong:
1 to 9 tiles of 32 rows per workgroup (whole and half groups, groups whose last waves have nothing to load), vocab
sizes that end inside a tile, and logits that are NaN or infinite, in whole tiles and in the last one.

Tolerance: the logit's bf16 rounding (2^-8 of it) and K fp32 roundings of partial sums no larger than sum |x w|
(K 2^-24 of it).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, pkg
from oracle import lm_head as oracle_lm_head
from test_gpu_gemm import _bits, _rand

pytestmark = pytest.mark.gpu
gemm = pkg("gemm")
lm_head = pkg("lm_head")

K = 512
CUS = 256  # workgroups: one per CU, a balanced range of tiles each


def _run(hidden: torch.Tensor, packed, n: int) -> tuple[torch.Tensor, torch.Tensor]:
    logits = torch.full((hidden.shape[0], n), float("nan"), dtype=torch.bfloat16, device="cuda")
    pred, _ = lm_head.lm_head_argmax(hidden, packed, return_logits=True, logits=logits)
    ids, _ = lm_head.lm_head_argmax(hidden, packed)
    torch.cuda.synchronize()
    assert torch.equal(pred, ids)
    assert np.array_equal(pred.cpu().numpy(), oracle_lm_head.argmax(_bits(logits)))
    return logits, pred


@pytest.mark.parametrize("vocab", [100, 32 * CUS, 32 * CUS + 1, 2 * 32 * CUS, 3 * 32 * CUS + 40, 4 * 32 * CUS, 32_000,
                                   5 * 32 * CUS - 8, 6 * 32 * CUS + 16, 8 * 32 * CUS, 9 * 32 * CUS + 17])
@pytest.mark.parametrize("rows", [33, 128, 200])
def test_tiles_per_workgroup(rows: int, vocab: int) -> None:
    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    hidden, weight = _rand(g, rows, K), _rand(g, vocab, K, std=0.02)
    top = (hidden[rows - 1].float() * 0.05).to(torch.bfloat16)
    weight[vocab - 1] = top  # the last row's largest logit
    announce("lm head tiles", rows, vocab)
    logits, pred = _run(hidden, gemm.pack_weight(weight), vocab)
    assert int(pred[rows - 1]) == vocab - 1
    exact = hidden.double() @ weight.double().t()
    bound = 2.0 ** -8 * exact.abs() + K * 2.0 ** -24 * (hidden.double().abs() @ weight.double().abs().t())
    assert bool(((logits.double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("rows", [40, 128, 256])
@pytest.mark.parametrize("vocab", [32_000, 3 * 32 * CUS + 40])
def test_nan_and_infinite_logits(rows: int, vocab: int) -> None:
    """NaN rows of every sign and payload, infinities and their differences: the first NaN wins, NaN is canonical."""
    g = torch.Generator(device="cuda").manual_seed(rows + vocab + 1)
    hidden, weight = _rand(g, rows, K), _rand(g, vocab, K, std=0.02)
    odd = torch.tensor([0x7F81, -0x7F, 0x7FC1, -0x3B], dtype=torch.int16).view(torch.bfloat16).cuda()
    hidden[:, 5:8] = 0.0
    hidden[0::7, 5], hidden[1::7, 6], hidden[2::7, 7] = 1.0, -1.0, 1.0
    hidden[3, 100] = odd[1]  # a row of NaN
    weight[vocab - 3, 5], weight[70, 6] = float("inf"), float("inf")  # +inf for some rows, -inf for others
    weight[[9000, 41, vocab - 1, 15_000], 7] = odd  # 0 x NaN: NaN for every row
    announce("lm head nan", rows, vocab)
    logits, pred = _run(hidden, gemm.pack_weight(weight), vocab)
    nan = logits.isnan()
    want = torch.zeros_like(nan)
    want[:, [41, 9000, 15_000, vocab - 1]] = True
    want[3] = True
    want[hidden[:, 5] == 0, vocab - 3] = True  # 0 x inf
    want[hidden[:, 6] == 0, 70] = True
    assert torch.equal(nan, want)
    assert bool((logits.view(torch.int16)[nan] == 0x7FC0).all())
    assert bool((pred == torch.where(torch.arange(rows, device="cuda") == 3, 0, 41)).all())
    weight[[9000, 41, vocab - 1, 15_000], 7], hidden[3, 100] = 0.0, 0.0
    weight[vocab - 3, 5], weight[70, 6] = 3e38, -3e38  # logits that overflow to infinity in bf16 or are largest
    hidden[0::7, 5] = 4.0
    logits, pred = _run(hidden, gemm.pack_weight(weight), vocab)
    assert not bool(logits.isnan().any()) and bool(torch.isinf(logits[0::7, vocab - 3]).all())
    assert bool((pred[0::7] == vocab - 3).all())
