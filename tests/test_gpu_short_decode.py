"""Decode steps against contexts below the long-context threshold that split-K serves: both sides of the rule,
against the oracle and the prefill kernel."""
import pytest
import torch

import fused_attn
from fused_attn import _hip, ops
from helpers import TOL, announce, max_err, randn
from oracle import attention_oracle as orc

CASES = [  # b, hq, hkv, nq, nk, d -> kernel family
    ((2, 8, 2, 1, 511, 128), "fwd"), ((2, 8, 2, 1, 512, 128), "splitk"), ((2, 8, 2, 8, 700, 64), "splitk"),
    ((2, 8, 2, 9, 700, 64), "fwd"), ((2, 8, 2, 1, 1000, 256), "fwd"), ((9, 8, 2, 1, 1000, 256), "splitk"),
    ((17, 32, 8, 1, 191, 128), "fwd"), ((17, 32, 8, 3, 192, 128), "splitk"), ((16, 8, 8, 4, 600, 64), "fwd"),
    ((16, 8, 8, 5, 600, 64), "fwd"), ((17, 8, 8, 1, 600, 64), "fwd"),
    # the context from which each of these is faster grows with the queries, at D=64 and where few heads share a
    # kv-head (us: prefill kernel and split-K)
    ((8, 8, 8, 4, 640, 64), "fwd"), ((8, 8, 8, 4, 641, 64), "splitk"), ((16, 8, 8, 1, 1280, 128), "fwd"),
    ((2, 32, 8, 1, 640, 64), "fwd"),  # 10.1 and 11.1
    ((32, 32, 8, 8, 384, 64), "fwd"),  # 19.1 and 31.9
    ((16, 32, 8, 8, 640, 128), "fwd"), ((16, 32, 8, 8, 1280, 128), "splitk"),
    ((32, 16, 8, 8, 1600, 128), "fwd"),  # 46.1 and 53.7
    ((64, 16, 8, 4, 192, 64), "fwd"),  # 12.7 and 20.8
    ((16, 16, 8, 8, 1000, 256), "fwd"),  # 35.0 and 40.5
    ((32, 64, 8, 2, 255, 64), "fwd"), ((32, 64, 8, 2, 256, 64), "splitk"),
]


@pytest.mark.parametrize("shape,family", CASES)
def test_rule(shape, family):
    b, hq, hkv, nq, nk, d = shape
    q, k = torch.empty(b, hq, nq, d, dtype=torch.bfloat16), torch.empty(b, hkv, nk, d, dtype=torch.bfloat16)
    assert ops._hip_kernel_for(q, k) == family
    assert ops._hip_kernel_for(q.float(), k.float()) == "fwd"


def test_malformed_calls_reach_the_checks():
    q, k = torch.empty(2, 8, 1, 64, dtype=torch.bfloat16), torch.empty(2, 3, 600, 64, dtype=torch.bfloat16)
    for bad in (k, k[:, :0], k[0]):
        assert ops._hip_kernel_for(q, bad) == "fwd"


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [s for s, family in CASES if family == "splitk"])
def test_matches_oracle_and_prefill_kernel(shape, dtype, causal):
    announce(f"short decode {shape} {dtype} causal={causal}")
    b, hq, hkv, nq, nk, d = shape
    torch.manual_seed(0)
    q = randn(b, nq, hq, d, dtype=dtype).transpose(1, 2)
    k, v = (randn(b, nk, hkv, d, dtype=dtype).transpose(1, 2) for _ in range(2))
    out = fused_attn.attention(q, k, v, causal=causal)
    assert max_err(out, orc.attention(q.cpu(), k.cpu(), v.cpu(), causal=causal)) <= TOL[dtype]
    assert max_err(out, _hip.fwd(q, k, v, causal=causal)) <= TOL[dtype]
    one = k[:1]  # a shared cache: batch 1 against q's
    out = fused_attn.attention(q, one, one, causal=causal)
    assert max_err(out, orc.attention(q.cpu(), one.cpu().expand(b, -1, -1, -1), one.cpu().expand(b, -1, -1, -1),
                                      causal=causal)) <= TOL[dtype]
