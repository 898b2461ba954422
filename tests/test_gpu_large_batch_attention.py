"""Paged attention of large batches, where every context is one workgroup's work (256 (context, kv-head group)
units and more): mixed, equal, rising, falling, empty and one-key contexts, contexts longer than ``max_seq_len``,
sharp scores; every head grouping, both page sizes, verify and decode widths -- against a float64 softmax over the
gathered keys, and the fused launch against the separate q/k norm + RoPE + store and attention calls bit for bit.
A context's result depends on neither its neighbours' lengths nor the workspace.  Tolerance: the outputs' bf16
rounding (2^-8) and the bf16 rounding of the probabilities (2^-8 of a convex combination of |v|).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, pkg

pytestmark = pytest.mark.gpu
attention = pkg("attention")
kernels = pkg("kernels")

D = 128


def _batch(lens: list[int], bs: int, kv: int, g: torch.Generator):
    pages = [-(-max(n, 1) // bs) for n in lens]
    order = np.random.default_rng(len(lens)).permutation(sum(pages)).astype(np.int32)
    table = np.zeros((len(lens), max(pages)), dtype=np.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = order[at:at + n]
        at += n
    shape = (sum(pages), bs, kv, D)
    kc = torch.randn(shape, generator=g, device="cuda").clamp(-6, 6).to(torch.bfloat16)
    vc = torch.randn(shape, generator=g, device="cuda").clamp(-6, 6).to(torch.bfloat16)
    return kc, vc, torch.from_numpy(table).cuda(), torch.tensor(lens, dtype=torch.int32, device="cuda")


def _check(out: torch.Tensor, q: torch.Tensor, kc, vc, table, lens: list[int]) -> None:
    """Every row of every context; a token before its context's first key (fewer keys than tokens) sees none: zeros."""
    _, s, h, _ = q.shape
    kv, bs = kc.shape[2], kc.shape[1]
    for b, n in enumerate(lens):
        pos = n - s + torch.arange(s, device="cuda")
        assert bool((out[b, pos < 0] == 0).all()), (b, n)
        if n == 0:
            continue
        at = torch.arange(n, device="cuda")
        slot = table[b].long()[at // bs] * bs + at % bs
        k, v = (c.view(-1, kv, D)[slot].double().repeat_interleave(h // kv, 1) for c in (kc, vc))
        scores = q[b].double().permute(1, 0, 2).contiguous() @ k.permute(1, 2, 0).contiguous() * D ** -0.5
        scores.masked_fill_(at[None, :] > pos[:, None], float("-inf"))
        p = torch.softmax(scores, -1).nan_to_num(0.0)
        want = (p @ v.permute(1, 0, 2).contiguous()).permute(1, 0, 2)
        mass = (p @ v.abs().permute(1, 0, 2).contiguous()).permute(1, 0, 2)
        err = (out[b].double() - want).abs()
        assert bool((err <= 2.0 ** -8 * want.abs() + 2.0 ** -8 * mass + 1e-5).all()), (b, n, err.max().item())


def _extend(q: torch.Tensor, kc, vc, lens_t, table, **kw) -> torch.Tensor:
    out = torch.full_like(q, float("nan"))
    attention.paged_extend(q, kc, vc, lens_t, table, out=out, **kw)
    torch.cuda.synchronize()
    return out


def _sequences(s: int, h: int, kv: int) -> int:
    """A batch of just over 256 units: head groups of two kv heads while their rows fit, else one."""
    groups = kv // 2 if kv % 2 == 0 and 2 * s * (h // kv + 2) <= 32 else kv
    return -(-256 // groups) + 6


MIXED = [1, 3000, 32, 33, 0, 700, 4096, 2, 1024, 513] + [64 + 37 * i for i in range(60)]


@pytest.mark.parametrize("s,h,kv,bs", [(1, 16, 8, 256), (1, 16, 8, 16), (4, 16, 8, 16), (8, 16, 8, 256), (1, 16, 4, 16),
                                       (1, 32, 4, 16), (2, 8, 8, 256), (3, 5, 5, 16), (1, 128, 8, 16)])
def test_mixed_contexts(s: int, h: int, kv: int, bs: int) -> None:
    g = torch.Generator(device="cuda").manual_seed(s * 100 + h + kv)
    lens = (MIXED * 4)[: _sequences(s, h, kv)]
    kc, vc, table, lens_t = _batch(lens, bs, kv, g)
    q = torch.randn(len(lens), s, h, D, generator=g, device="cuda").to(torch.bfloat16)
    announce("large batch", s, h, kv, bs, len(lens))
    _check(_extend(q, kc, vc, lens_t, table), q, kc, vc, table, lens)


@pytest.mark.parametrize("lens", [[1024] * 64, [1056] * 100, [16] * 63 + [8000], [600] * 110 + [1100], [1025] * 60 + [1] * 59,
                                  list(range(0, 2600, 40)), list(range(5080, 0, -40)), [33] * 129, [0] * 70,
                                  [7, 0, 3000, 64] * 48 + [65], [5] * 256 + [300]], ids=lambda l: f"{len(l)}x{l[0]}-{l[-1]}")
def test_equal_long_and_short_contexts(lens: list[int]) -> None:
    """One round of workgroups and several; lengths alike, one far longer, rising, falling, empty."""
    g = torch.Generator(device="cuda").manual_seed(len(lens))
    kc, vc, table, lens_t = _batch(lens, 16, 8, g)
    q = torch.randn(len(lens), 1, 16, D, generator=g, device="cuda").to(torch.bfloat16)
    announce("large batch lengths", lens[0], lens[-1], len(lens))
    _check(_extend(q, kc, vc, lens_t, table), q, kc, vc, table, lens)


@pytest.mark.parametrize("s", [1, 4])
def test_sharp_scores_and_clamped_contexts(s: int) -> None:
    g = torch.Generator(device="cuda").manual_seed(90 + s)
    lens = (MIXED * 2)[:70]
    kc, vc, table, lens_t = _batch(lens, 16, 8, g)
    q = (12 * torch.randn(len(lens), s, 16, D, generator=g, device="cuda")).to(torch.bfloat16)
    announce("large batch sharp", s)
    _check(_extend(q, kc, vc, lens_t, table), q, kc, vc, table, lens)
    _check(_extend(q, kc, vc, lens_t, table, max_seq_len=1000), q, kc, vc, table, [min(n, 1000) for n in lens])


@pytest.mark.parametrize("batch", [64, 96])
def test_a_context_does_not_depend_on_its_neighbours(batch: int) -> None:
    """Bit for bit, and nothing is written to the workspace."""
    g = torch.Generator(device="cuda").manual_seed(batch)
    lens = (MIXED * 2)[:batch]
    kc, vc, table, lens_t = _batch([4096] * batch, 256, 8, g)
    q = torch.randn(batch, 1, 16, D, generator=g, device="cuda").to(torch.bfloat16)
    workspace = torch.full((attention.workspace_bytes(batch, 8, 4096),), 0xAB, dtype=torch.uint8, device="cuda")
    lens_t = torch.tensor(lens, dtype=torch.int32, device="cuda")
    announce("large batch neighbours", batch)
    full = _extend(q, kc, vc, lens_t, table, workspace=workspace)
    other = lens_t.clone()
    other[10:] = other[10:].flip(0) // 3 + 1
    got = _extend(q, kc, vc, other, table, workspace=workspace)
    assert torch.equal(got[:10].view(torch.int16), full[:10].view(torch.int16))
    assert bool((workspace == 0xAB).all())


@pytest.mark.parametrize("s,h,kv", [(1, 16, 8), (4, 16, 8), (8, 16, 8), (3, 8, 8)])
def test_fused_equals_separate_calls(s: int, h: int, kv: int) -> None:
    """Contexts of at least s keys; output and both caches."""
    g = torch.Generator(device="cuda").manual_seed(s)
    lens = [max(n, s) for n in (MIXED * 4)[: _sequences(s, h, kv)]]
    kc, vc, table, lens_t = _batch(lens, 16, kv, g)
    n = len(lens) * s
    qkv = torch.randn(n, (h + 2 * kv) * D, generator=g, device="cuda").to(torch.bfloat16)
    qw, kw = ((0.5 + torch.rand(D, generator=g, device="cuda")).to(torch.bfloat16) for _ in range(2))
    angles = torch.rand(max(lens), D // 2, generator=g, device="cuda") * 6.28
    cos, sin = angles.cos().to(torch.bfloat16), angles.sin().to(torch.bfloat16)
    pos = (lens_t.long()[:, None] - s + torch.arange(s, device="cuda")).reshape(-1)
    slots = table.long().gather(1, pos.view(-1, s) // 16).view(-1) * 16 + pos % 16
    k2, v2 = kc.clone(), vc.clone()
    announce("large batch fused", s, h, kv)
    q, _, _ = kernels.qk_norm_rope_store(qkv, qw, kw, cos[pos].contiguous(), sin[pos].contiguous(), 1e-6, k2, v2, slots,
                                         h, kv, D, need_kv=False)
    want = attention.paged_extend(q.view(len(lens), s, h, D), k2, v2, lens_t, table)
    got = attention.qk_norm_rope_paged_extend(qkv, qw, kw, cos, sin, pos, 1e-6, kc, vc, slots, lens_t, table, h)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    assert torch.equal(kc.view(torch.int16), k2.view(torch.int16)) and torch.equal(vc, v2)
