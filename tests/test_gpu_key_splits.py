"""Prefill calls with few row blocks against many keys: each block's key tiles are cut over several
workgroups, whose fp32 partials a second kernel merges.  Against the fp32 oracle, at the edges of the
cut: ragged key tiles, row blocks with fewer tiles than splits, rows without keys, both output layouts."""
import pytest
import torch

from fused_attn import _hip
from helpers import TOL, announce, close, max_err, randn
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu


def _workspace(q, k, causal):
    p = _hip.make_params(q, k, k, q, causal, 1.0)
    return _hip.load_library().fa_attention_fwd_workspace_bytes(p)


# (b, hq, hkv, nq, nk, d, causal, splits, [B, N, H, D] views)
CASES = [
    (1, 4, 1, 70, 3000, 128, True, 8, False),  # 4-wave blocks, one row block
    (1, 4, 1, 300, 4097, 128, True, 16, True),  # 8-wave blocks, the last tile holds one key
    (2, 4, 2, 129, 2047, 128, False, 8, False),
    (1, 2, 1, 1200, 1100, 128, True, 4, False),  # n_q > n_k: first rows see no key, first blocks few tiles
    (1, 4, 4, 65, 5000, 64, True, 8, True),
    (1, 3, 1, 64, 2500, 256, True, 16, False),
    (1, 4, 2, 200, 6001, 32, False, 8, False),
    (1, 2, 2, 100, 6100, 16, True, 8, True),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,nq,nk,d,causal,splits,views", CASES)
def test_key_splits_match_oracle(b, hq, hkv, nq, nk, d, causal, splits, views, dtype):
    announce(f"key splits b={b} hq={hq} hkv={hkv} nq={nq} nk={nk} d={d} causal={causal} {dtype}")
    gen = torch.Generator(device="cuda").manual_seed(9)
    q = randn(b, hq, nq, d, dtype=dtype, gen=gen)
    k = randn(b, hkv, nk, d, dtype=dtype, gen=gen)
    v = randn(b, hkv, nk, d, dtype=dtype, gen=gen)
    if views:
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    assert _workspace(q, k, causal) == splits * b * hq * nq * (d + 2) * 4
    out, lse = _hip.fwd(q, k, v, causal=causal, return_lse=True)
    want, want_lse = orc.attention(q.cpu(), k.cpu(), v.cpu(), causal=causal), orc.lse(q.cpu(), k.cpu(), causal=causal)
    assert max_err(out, want) <= TOL[dtype]
    torch.testing.assert_close(lse.cpu(), want_lse, atol=5e-3, rtol=1e-3)  # P is rounded to 16 bits: 2^-9 relative in l
    again = _hip.fwd(q, k, v, causal=causal)
    assert torch.equal(again, out)
    # a caller's output with 8-byte strides (rows of d + 4 elements) takes the same merge
    wide = torch.zeros(b, hq, nq, d + 4, dtype=dtype, device="cuda")
    _hip.fwd(q, k, v, causal=causal, out=wide[..., :d])
    assert torch.equal(wide[..., :d], out) and not wide[..., d:].any()


def test_workspace_too_small_is_an_error():
    q, k = randn(1, 4, 70, 128, dtype=torch.bfloat16), randn(1, 1, 3000, 128, dtype=torch.bfloat16)
    p = _hip.make_params(q, k, k, torch.empty_like(q), True, 1.0)
    lib = _hip.load_library()
    need = lib.fa_attention_fwd_workspace_bytes(p)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    assert lib.fa_attention_fwd_ws(p, ws.data_ptr(), need - 1, None) == 3  # FA_ERR_WORKSPACE
    assert lib.fa_attention_fwd_ws(p, None, 0, None) == 3


@pytest.mark.parametrize("b,hq,hkv,nq,nk,d,causal,splits,views", CASES)
def test_result_does_not_depend_on_the_workspace(b, hq, hkv, nq, nk, d, causal, splits, views):
    """Every partial that the merge reads was written: a workspace of NaN changes nothing."""
    announce(f"key splits, NaN workspace b={b} hq={hq} nq={nq} nk={nk} d={d} causal={causal}")
    gen = torch.Generator(device="cuda").manual_seed(10)
    q, k, v = (randn(b, h, n, d, dtype=torch.bfloat16, gen=gen) for h, n in ((hq, nq), (hkv, nk), (hkv, nk)))
    want, want_lse = _hip.fwd(q, k, v, causal=causal, return_lse=True)
    out, lse = torch.empty_like(q), torch.empty(b, hq, nq, device="cuda")
    p = _hip.make_params(q, k, v, out, causal, d ** -0.5, lse=lse)
    lib = _hip.load_library()
    need = lib.fa_attention_fwd_workspace_bytes(p)
    ws = torch.full((need // 4 + 64,), float("nan"), device="cuda")
    assert lib.fa_attention_fwd_ws(p, ws.data_ptr(), need, _hip._stream(q)) == 0
    assert torch.equal(out, want) and torch.equal(lse, want_lse)
    assert ws[need // 4:].isnan().all()


@pytest.mark.parametrize("scale", [-0.2, 0.0, 3.0])
def test_scales(scale):
    announce(f"key splits scale={scale}")
    gen = torch.Generator(device="cuda").manual_seed(11)
    q, k, v = (randn(1, h, n, 128, dtype=torch.float16, gen=gen) for h, n in ((4, 70), (1, 3000), (1, 3000)))
    out = _hip.fwd(q, k, v, causal=True, scale=scale)
    assert close(out, orc.attention(q.cpu(), k.cpu(), v.cpu(), causal=True, scale=scale), TOL[torch.float16])


@pytest.mark.parametrize("d,nq", [(128, 70), (128, 300), (64, 65), (256, 64)])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_infinities_and_nan(value, where, d, nq):
    """One such value in one split: the rows and columns that it reaches are those of the unsplit kernel and of 64-bit
    softmax (the oracle gives a row of NaN scores zeros, as the reference does), and the others keep their values."""
    announce(f"key splits {value} in {where} d={d} nq={nq}")
    gen = torch.Generator(device="cuda").manual_seed(12)
    q, k, v = (randn(1, h, n, d, dtype=torch.bfloat16, gen=gen) for h, n in ((4, nq), (2, 3000), (2, 3000)))
    (k if where == "k" else v)[0, 1, 1700, 5] = value
    assert _workspace(q, k, False) > 0
    out = _hip.fwd(q, k, v)
    unsplit = torch.empty_like(q)
    p = _hip.make_params(q, k, v, unsplit, False, d ** -0.5)
    assert _hip.load_library().fa_attention_fwd(p, _hip._stream(q)) == 0
    kd, vd = (x.cpu().double().repeat_interleave(2, 1) for x in (k, v))
    want = (torch.softmax(q.cpu().double() @ kd.transpose(-1, -2) / d ** 0.5, -1) @ vd).float().to("cuda")
    for other in (unsplit.float(), want):
        assert torch.equal(out.isnan(), other.isnan()) and torch.equal(out.isinf(), other.isinf())
    seen = want.isfinite()
    assert seen[:, :2].all() and not seen.all()
    assert torch.equal(out[want.isinf()].float(), want[want.isinf()])
    assert max_err(out[seen], want[seen]) <= TOL[torch.bfloat16]
