"""D=64 and D=32 prefill in grids beyond two workgroups per CU, which take 64-key tiles: edges of the tiles and of the
row blocks, causal or not.  Varlen grids, which are laid out for the longest sequence, keep 128-key tiles."""
import pytest
import torch

import fused_attn
from fused_attn import _hip
from helpers import TOL, announce, max_err, randn
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nq,nk", [(1, 1), (31, 63), (64, 64), (65, 129), (128, 191), (129, 65), (257, 257)])
def test_large_grids(nq, nk, causal, d, dtype):
    announce(f"short tile nq={nq} nk={nk} causal={causal} d={d} {dtype}")
    torch.manual_seed(0)
    b, h = 33, 16  # 528 heads: beyond 512 workgroups at any length
    q = randn(b, nq, h, d, dtype=dtype).transpose(1, 2)
    k, v = (randn(b, h // 4, nk, d, dtype=dtype) for _ in range(2))
    out = fused_attn.attention(q, k, v, causal=causal)
    assert max_err(out, orc.attention(q.cpu(), k.cpu(), v.cpu(), causal=causal)) <= TOL[dtype]


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_varlen(d, causal):
    announce(f"short tile varlen d={d} causal={causal}")
    torch.manual_seed(0)
    lens = [0, 1, 63, 64, 65, 128, 300, 513] * 5
    q, cu, mx = fused_attn.pack_varlen([randn(n, 16, d, dtype=torch.bfloat16) for n in lens])
    k, _, _ = fused_attn.pack_varlen([randn(n, 4, d, dtype=torch.bfloat16) for n in lens])
    v, _, _ = fused_attn.pack_varlen([randn(n, 4, d, dtype=torch.bfloat16) for n in lens])
    out = fused_attn.attention_varlen(q, k, v, cu, cu, mx, mx, causal=causal)
    ref = orc.attention_varlen(q.cpu(), k.cpu(), v.cpu(), cu.cpu(), cu.cpu(), causal=causal)
    assert max_err(out, ref) <= TOL[torch.bfloat16]


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_varlen_sequence_equals_the_sequence_alone(d, causal):
    """Alone, a sequence's grid stays below 512 workgroups: the same tiles in the same order, so the same bits."""
    announce(f"varlen tile d={d} causal={causal}")
    torch.manual_seed(0)
    lens = [300, 1, 129, 512, 64, 400, 257, 33]
    q, cu, mx = fused_attn.pack_varlen([randn(n, 32, d, dtype=torch.float16) for n in lens])
    k, _, _ = fused_attn.pack_varlen([randn(n, 8, d, dtype=torch.float16) for n in lens])
    v, _, _ = fused_attn.pack_varlen([randn(n, 8, d, dtype=torch.float16) for n in lens])
    out = fused_attn.attention_varlen(q, k, v, cu, cu, mx, mx, causal=causal)
    for i, n in enumerate(lens):
        t = slice(int(cu[i]), int(cu[i]) + n)
        one = _hip.fwd(*(x[t].transpose(0, 1)[None] for x in (q, k, v)), causal=causal)
        assert torch.equal(out[t].transpose(0, 1)[None], one), n
