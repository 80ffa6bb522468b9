"""Ragged paged decode: lengths at the edges of partitions, grids that are no multiple of the XCD count, and
partitions past a sequence's end, which the kernel leaves unwritten."""
import math

import pytest
import torch

import fused_attn
from fused_attn import _hip
from fused_attn.paged import default_paged_split_len
from helpers import TOL, announce, max_err, randn
from oracle import attention_oracle as orc

LENS = [0, 127, 128, 129, 1000, 1, 384]


@pytest.mark.gpu
@pytest.mark.parametrize("nq", [1, 5, 20])  # 1, 2 and 4 waves; 20 queries of 4 heads also make one row block,
@pytest.mark.parametrize("group", [4, 7])  # of 7 heads two
@pytest.mark.parametrize("hkv", [1, 3])
def test_unwritten_partitions_are_not_read(nq, group, hkv):
    """The workspace starts as NaN: the merge must take only the partitions below each sequence's end."""
    announce(f"paged ragged nq={nq} group={group} hkv={hkv}")
    torch.manual_seed(0)
    b, n, d, split_len = len(LENS), max(LENS), 128, 128
    q = randn(b, hkv * group, nq, d, dtype=torch.bfloat16)
    k, v = (randn(b, hkv, n, d, dtype=torch.bfloat16) for _ in range(2))
    kc, vc, bt, sl = fused_attn.paged_from_dense(k, v, 32, seqlens=LENS)
    words = _hip.workspace_bytes(b, hkv * group, nq, d, -(-n // split_len)) // 4
    ws = torch.full((words + 4,), math.nan, dtype=torch.float32, device="cuda")
    out, lse = _hip.paged_decode(q, kc, vc, bt, sl, n, causal=True, split_len=split_len, workspace=ws, return_lse=True)
    ref = orc.attention_paged(q, kc, vc, bt, sl, causal=True)
    assert not torch.isnan(out).any() and not torch.isnan(lse).any()
    assert max_err(out, ref) <= TOL[torch.bfloat16]
    assert torch.all(out[0] == 0) and torch.all(torch.isneginf(lse[0]))


@pytest.mark.gpu
def test_fp8_two_partitions_per_workgroup():
    """FP8 pools in a grid of 16384 workgroups or more: a workgroup takes two partitions, of which a sequence
    may end in the first."""
    announce("paged ragged fp8, two partitions per workgroup")
    torch.manual_seed(0)
    lens = [64 * i + (i % 3) for i in range(64)]
    b, hkv, n, d = len(lens), 8, 4096, 64
    k, v = (randn(b, hkv, n, d, dtype=torch.bfloat16) for _ in range(2))
    k8, ks = fused_attn.quantize_kv_fp8(k)
    v8, vs = fused_attn.quantize_kv_fp8(v)
    q = randn(b, 16, 1, d, dtype=torch.bfloat16)
    kc, vc, ksc, vsc, bt, sl = fused_attn.paged.paged_from_dense_fp8(k8, ks, v8, vs, 64, seqlens=lens)
    words = _hip.workspace_bytes(b, 16, 1, d, n // 64) // 4
    ws = torch.full((words + 4,), math.nan, dtype=torch.float32, device="cuda")
    out = _hip.paged_decode(q, kc, vc, bt, sl, n, split_len=64, workspace=ws, k_scale=ksc, v_scale=vsc)
    assert not torch.isnan(out).any() and torch.all(out[0] == 0)
    for i in (1, 2, 17, 63):
        one = fused_attn.attention_fp8(q[i:i + 1], k8[i:i + 1, :, :lens[i]].contiguous(),
                                       ks[i:i + 1, :, :-(-lens[i] // 64)].contiguous(), v8[i:i + 1, :, :lens[i]].contiguous(),
                                       vs[i:i + 1, :, :-(-lens[i] // 64)].contiguous(), split_len=64)
        assert max_err(out[i:i + 1], one.float().cpu()) <= TOL[torch.bfloat16]


@pytest.mark.parametrize("row_bytes", [256, 512])
@pytest.mark.parametrize("n", [0, 1, 600, 8192, 1 << 20])
@pytest.mark.parametrize("b,hkv,group,nq", [(1, 1, 1, 1), (16, 4, 4, 1), (48, 8, 4, 1), (100, 8, 4, 4), (300, 32, 8, 16)])
def test_default_partitions(b, hkv, group, nq, n, row_bytes):
    """The longest power of two whose grid reaches its target: 2048 workgroups (1152 above 256-byte rows) down to 512
    keys, 1000 below."""
    keys = default_paged_split_len(nq, n, b, hkv, group, row_bytes)
    large = 2048 if row_bytes == 256 else 1152

    def workgroups(length):
        return b * hkv * -(-group * nq // 128) * -(-n // length)

    assert 128 <= keys <= 4096 and keys & (keys - 1) == 0
    assert keys == 128 or workgroups(keys) >= (large if keys > 512 else 1000)
    assert keys == 4096 or workgroups(2 * keys) < (large if keys >= 512 else 1000)


@pytest.mark.parametrize("args,keys", [
    ((1, 8192, 48, 8, 4, 256), 1024), ((1, 2000, 100, 8, 4, 256), 512), ((1, 4096, 16, 4, 4, 256), 256),
    ((1, 2000, 100, 8, 4, 512), 1024),
    ((1, 4096, 64, 8, 4, 256), 1024), ((4, 16384, 32, 4, 8, 256), 1024), ((1, 32768, 32, 8, 4, 256), 4096),
    # rows of fewer than 256 bytes: the dense policy
    ((8, 8192, 48, 8, 4, 128), 1408), ((16, 4000, 24, 8, 8, 64), 384), ((1, 3000, 4, 32, 4, 128), 192),
])
def test_default_partitions_as_measured(args, keys):
    assert default_paged_split_len(*args) == keys


def test_default_partitions_of_a_malformed_head_dim():
    """A head dim of 0 reaches the checks of the call itself."""
    assert default_paged_split_len(1, 1000, 2, 2, 4, 0) == 128
