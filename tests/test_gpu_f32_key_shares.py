"""fp32 prefill of small grids, where the waves of a 32-query workgroup share out the key tiles: edges of the
32-row blocks, of the 32-key tiles and of the waves' shares, beside the plain kernel's larger grids."""
import pytest
import torch

from fused_attn.triton_fwd import attention_triton
from helpers import announce, randn

pytestmark = pytest.mark.gpu


def _reference(q, k, v, causal, scale):
    """64-bit attention on the CPU: (o, lse)."""
    group, (nq, nk) = q.shape[1] // k.shape[1], (q.shape[2], k.shape[2])
    qd, kd, vd = q.cpu().double(), *(x.cpu().double().repeat_interleave(group, 1) for x in (k, v))
    s = qd @ kd.transpose(-1, -2) * scale
    if causal:
        s = s.masked_fill(torch.arange(nk)[None] > torch.arange(nq)[:, None] + (nk - nq), -torch.inf)
    return torch.softmax(s, -1).nan_to_num(nan=0.0) @ vd, torch.logsumexp(s, -1)


def _check(b, hq, hkv, nq, nk, d, causal, transposed=False, scale=None):
    torch.manual_seed(0)
    if transposed:
        q, k, v = (randn(b, n, h, d, dtype=torch.float32).transpose(1, 2) for n, h in ((nq, hq), (nk, hkv), (nk, hkv)))
    else:
        q, k, v = (randn(b, h, n, d, dtype=torch.float32) for n, h in ((nq, hq), (nk, hkv), (nk, hkv)))
    out, lse = attention_triton(q, k, v, causal=causal, scale=scale, return_lse=True)
    ref, want = _reference(q, k, v, causal, d ** -0.5 if scale is None else scale)
    # sums of at most 600 products of N(0, 1) values in fp32: 600 * 2^-24 of a value of a few units
    assert (out.cpu().double() - ref).abs().max() <= 1e-4
    seen = torch.isfinite(want)
    assert torch.equal(torch.isfinite(lse.cpu()), seen)
    assert (lse.cpu().double() - want)[seen].abs().max() <= 1e-4 if seen.any() else True


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("nq,nk", [(1, 1), (31, 33), (32, 32), (33, 97), (64, 128), (65, 129), (1, 600), (100, 257), (160, 40)])
def test_small_grids(nq, nk, d, causal):
    announce(f"fp32 key shares nq={nq} nk={nk} d={d} causal={causal}")
    _check(2, 4, 2, nq, nk, d, causal)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,n", [(16, 16, 128), (3, 8, 255)])  # the plain kernel, and on the other side of the rule
def test_both_sides_of_the_rule(b, h, n, causal):
    announce(f"fp32 key shares b={b} h={h} n={n} causal={causal}")
    _check(b, h, h, n, n, 64, causal, transposed=True)


@pytest.mark.parametrize("scale", [-0.2, 0.0])
def test_scales(scale):
    announce(f"fp32 key shares scale={scale}")
    _check(2, 4, 2, 65, 129, 64, True, scale=scale)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("where", ["k", "v"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_infinities_and_nan(value, where, d):
    """One such value in one wave's share: it reaches the rows and columns that it reaches in 64 bits."""
    announce(f"fp32 key shares {value} in {where} d={d}")
    torch.manual_seed(0)
    q, k, v = (randn(1, h, n, d, dtype=torch.float32) for h, n in ((4, 70), (2, 300), (2, 300)))
    (k if where == "k" else v)[0, 1, 170, 5] = value
    out = attention_triton(q, k, v)
    s = q.cpu().double() @ k.cpu().double().repeat_interleave(2, 1).transpose(-1, -2) / d ** 0.5
    want = torch.softmax(s, -1) @ v.cpu().double().repeat_interleave(2, 1)
    out = out.cpu().double()
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    seen = want.isfinite()
    assert seen[:, :2].all() and not seen.all()
    assert torch.equal(out[want.isinf()], want[want.isinf()])
    assert (out[seen] - want[seen]).abs().max() <= 1e-4
