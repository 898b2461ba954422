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


@pytest.mark.parametrize("causal", [True, False])
def test_rows_past_32_bit_offsets(causal: bool) -> None:
    """270,000 kv heads: 63 rows of a key tile are more than 2^32 bytes.  A few heads against float64, with a tile cut by
    the sequence's end; tolerance: bf16 rounding of the output and of the probabilities (2^-8 of each)."""
    n, kv = 65, 270_000
    g = torch.Generator(device="cuda").manual_seed(61)
    q, k, v = (torch.empty(n, kv, 128, dtype=torch.bfloat16, device="cuda").normal_(generator=g) for _ in range(3))
    announce("varlen wide rows", n, kv, causal)
    out = attention.varlen(q, k, v, torch.tensor([0, n], dtype=torch.int32, device="cuda"), n, causal=causal)
    torch.cuda.synchronize()
    for head in (0, 1, 135_000, kv - 1):
        qd, kd, vd = (t[:, head].double() for t in (q, k, v))
        scores = qd @ kd.t() * 128 ** -0.5
        if causal:
            scores.masked_fill_(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
        p = torch.softmax(scores, -1)
        want = p @ vd
        err = (out[:, head].double() - want).abs()
        assert bool((err <= 2.0 ** -8 * (want.abs() + p @ vd.abs()) + 1e-5).all()), head
