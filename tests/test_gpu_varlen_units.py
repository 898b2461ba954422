"""Bidirectional prefill deals its (sequence, kv head) pairs to the XCDs, whole or cut into 2, 4 or 8 parts of
query tiles (kv heads no multiple of 8, few pairs): every part count, with fewer query tiles than parts, one
more and several per part, empty sequences, and many short ones, against the oracle."""

from __future__ import annotations

import pytest
import torch

from conftest import announce
from test_gpu_varlen import _case, attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV", [(8, 1), (6, 3), (4, 2), (12, 12), (8, 8)])
def test_bidirectional_units(H: int, KV: int) -> None:
    rows = 256 // (H // KV)  # positions per query tile
    _case([rows - 1, 0, 2 * rows + 1, 1], H, KV, False, seed=30 + KV)
    if KV <= 3:
        _case([9 * rows // 2], H, KV, False, seed=40 + KV)


@pytest.mark.parametrize("lens,H,KV", [([30] * 300, 5, 5), ([600] * 7, 12, 6), ([77] * 64, 8, 1), ([90] * 9, 8, 1)])
def test_bidirectional_many_short_sequences(lens: list[int], H: int, KV: int) -> None:
    """Several rounds of 8 pairs: whole ones, and parts with fewer query tiles than there are parts."""
    _case(lens, H, KV, False, seed=50 + KV)


def test_bidirectional_a_million_one_token_sequences() -> None:
    """One key each: the output is v.  Eight workgroups a sequence would be more threads than a launch holds."""
    n = 1_050_000
    g = torch.Generator(device="cuda").manual_seed(60)
    q, k, v = (torch.randn(n, 1, 128, generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    announce("varlen a million one-token sequences")
    out = attention.varlen(q, k, v, torch.arange(n + 1, dtype=torch.int32, device="cuda"), 1, causal=False)
    torch.cuda.synchronize()
    assert torch.equal(out, v)
