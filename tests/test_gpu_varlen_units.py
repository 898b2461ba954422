"""Bidirectional prefill deals its (sequence, kv head) pairs to the XCDs, cut into 1, 2, 4 or 8 parts of
query tiles when the kv heads do not divide by 8: every part count, with fewer query tiles than parts,
one more and several per part, and empty sequences, against the oracle."""

from __future__ import annotations

import pytest

from test_gpu_varlen import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV", [(8, 1), (6, 3), (4, 2), (12, 12), (8, 8)])
def test_bidirectional_units(H: int, KV: int) -> None:
    rows = 256 // (H // KV)  # positions per query tile
    _case([rows - 1, 0, 2 * rows + 1, 1], H, KV, False, seed=30 + KV)
    if KV <= 3:
        _case([9 * rows // 2], H, KV, False, seed=40 + KV)
