"""Argument checks of the GEMM wrappers that come before any device call."""

from __future__ import annotations

import pytest
import torch

from conftest import pkg

gemm = pkg("gemm")


@pytest.mark.parametrize("m", [0, 3])
def test_packed_output_needs_a_packed_weight(m: int) -> None:
    x, w = torch.zeros(m, 128, dtype=torch.bfloat16), torch.zeros(128, 128, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="packed w"):
        gemm._run(x, w, 128, gemm.EPI_STORE, gemm.packed_rows(m, 128, "cpu"), torch.device("cpu"))


def test_no_rows_is_no_call() -> None:
    x, w = torch.zeros(0, 128, dtype=torch.bfloat16), torch.zeros(128, 128, dtype=torch.bfloat16)
    gemm._run(x, w, 128, gemm.EPI_STORE, torch.zeros(0, 128, dtype=torch.bfloat16), torch.device("cpu"))
