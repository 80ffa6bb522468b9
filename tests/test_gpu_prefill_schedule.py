"""Causal prefill over the forms of its workgroup schedule: units cut to an XCD's share of the heads, calls dealt to
the XCDs, and grids of 257-512 workgroups, whose first 32 per XCD are taken in reverse."""
import pytest
import torch

import fused_attn
from helpers import TOL, announce, max_err, randn
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hkv,n", [
    (1, 32, 8, 1030),  # 8-head units would be cut: 288 workgroups, reversed
    (2, 12, 4, 300),   # 24 heads: units of 3
    (1, 12, 4, 700),   # dealt: 12 heads, 72 workgroups
    (1, 28, 4, 1300),  # dealt and reversed: 308 workgroups
    (3, 3, 1, 130),    # dealt: 9 heads
    (5, 20, 5, 333),   # 100 heads: units of 12, 300 workgroups
    (1, 4, 1, 2200),   # fewer heads than XCDs
    (4, 33, 11, 500),  # 132 heads, 528 workgroups: not reversed
])
@pytest.mark.parametrize("d", [64, 128])
def test_causal_schedules(b, hq, hkv, n, d):
    announce(f"prefill schedule b={b} hq={hq} hkv={hkv} n={n} d={d}")
    torch.manual_seed(0)
    q = randn(b, hq, n, d, dtype=torch.bfloat16)
    k, v = (randn(b, hkv, n, d, dtype=torch.bfloat16) for _ in range(2))
    out = fused_attn.attention(q, k, v, causal=True)
    assert max_err(out, orc.attention(q.cpu(), k.cpu(), v.cpu(), causal=True)) <= TOL[torch.bfloat16]
