"""The build's check of the generated code around loads into LDS (``dma_faults``): what it accepts and refuses."""

from __future__ import annotations

import pytest

from conftest import pkg

LOAD = "\ts_mov_b32 m0, s2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 v1, s[10:11]{} ; comment\n"


def faults(asm: str) -> list[str]:
    return pkg("build").dma_faults(asm)


@pytest.mark.parametrize("before", [
    "", "\ts_add_u32 s10, s10, s4\n\ts_addc_u32 s11, s11, 0\n",  # scalar writes need no wait
    "\tv_readfirstlane_b32 s10, v3\n\ts_nop 2\n",  # 3 + 2 wait states of the block's own
    "\tv_readfirstlane_b32 s10, v3\n\ts_add_u32 s4, s4, 1\n\ts_add_u32 s4, s4, 1\n\ts_add_u32 s4, s4, 1\n",
    "\tv_readlane_b32 s12, v218, 4\n", "\tv_cmp_eq_u32_e64 s[12:13], 0, v0\n",  # other registers
    "\tv_add_u32_e32 v2, s10, v1\n",  # reads it
    "\tv_readlane_b32 s11, v218, 4\n\ts_branch .LBB0_9\n.LBB0_1:\n",  # not on the way here
])
def test_accepts(before: str) -> None:
    assert faults(before + LOAD.format("")) == [] and faults(before + LOAD.format(" nt")) == []


@pytest.mark.parametrize("before", [
    "\tv_readfirstlane_b32 s10, v3\n", "\tv_readfirstlane_b32 s11, v3\n\ts_nop 1\n", "\tv_readlane_b32 s11, v218, 4\n",
    "\tv_cmp_eq_u32_e64 s[10:11], 0, v0\n", "\tv_add_co_u32_e64 v2, s[10:11], v3, v4\n",
    "\tv_mad_u64_u32 v[2:3], s[10:11], v4, v5, v[6:7]\n",
    "\tv_readlane_b32 s11, v218, 4\n.LBB0_1:\n",  # falls through a label
    "\tv_readlane_b32 s11, v218, 4\n\ts_cbranch_scc1 .LBB0_2\n\ts_nop 7\n\ts_endpgm\n.LBB0_2:\n",  # branches here
])
def test_refuses_a_vector_write_of_the_base(before: str) -> None:
    assert len(faults(before + LOAD.format(""))) == 1


def test_refuses_other_uses_of_m0() -> None:
    assert len(faults(LOAD.format("") + "\ts_mov_b32 m0, s3\n\tv_movrels_b32 v1, v2\n")) == 1
    assert len(faults(LOAD.format("") + "\ts_add_u32 s4, m0, 4\n")) == 1
    assert len(faults("\tglobal_load_lds_dwordx4 v1, s[10:11]\n")) == 1  # m0 as someone else left it
    assert len(faults(LOAD.format("").replace("s[10:11]", "vcc"))) == 1  # a base the check does not follow
