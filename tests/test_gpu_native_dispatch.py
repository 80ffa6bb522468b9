"""The native dispatcher kernels of fused_attn::attention: same choice of kernel as the Python kernel, same results,
and every call that they do not take reaches the Python kernel."""
import os
import random
import threading

import pytest
import torch

import fused_attn
from fused_attn import _hip, ops
from helpers import announce, randn


def test_route_equals_the_python_rule():
    assert _hip._native is not None, "libfused_attn_torch.so is not built"
    rng = random.Random(0)
    edges = [1, 2, 15, 16, 17, 31, 32, 33, 128, 191, 192, 511, 512, 513, 2047, 2048, 2049, 5000, 32768, 100000]
    for _ in range(20000):
        b, hkv, group = rng.choice([1, 2, 3, 16, 64, 300]), rng.choice([1, 2, 8, 32]), rng.choice([1, 2, 4, 7, 8])
        nq, nk, d = rng.choice(edges[:9]), rng.choice(edges), rng.choice([16, 32, 64, 128, 256])
        dtype = rng.choice([torch.float16, torch.bfloat16, torch.float32])
        q = torch.empty(b, hkv * group, nq, d, dtype=dtype, device="meta")
        k = torch.empty(b, hkv, nk, d, dtype=dtype, device="meta")
        want = ops.default_split_len(nq, nk, b, hkv, group) if ops._hip_kernel_for(q, k) == "splitk" else 0
        assert _hip._native.fa_torch_route(dtype != torch.float32, b, hkv * group, hkv, nq, nk, d) == want


@pytest.mark.parametrize("name,value", [("fa_torch_built_for", '"2.9.9+rocm7.0 0123"'), ("fa_torch_abi_version", "5"),
                                        ("fa_torch_params_size", "8"), ("fa_torch_register", "0"), (None, None)])
def test_a_library_built_for_another_torch_is_not_registered(name, value, tmp_path, monkeypatch):
    """A library that says it was built for another torch, ABI or parameter block (or one that says nothing: name None)
    is left out with a warning, before it registers anything."""
    import ctypes
    import subprocess

    has = {"fa_torch_built_for": f'"{torch.__version__} {torch.version.git_version}"', "fa_torch_abi_version": str(_hip.ABI_VERSION),
           "fa_torch_params_size": str(ctypes.sizeof(_hip.FwdParams)), "fa_torch_register": "1"}
    types = {"fa_torch_built_for": "const char*", "fa_torch_params_size": "unsigned long"}
    lines = [] if name is None else [f"{types.get(n, 'int')} {n}(void) {{ {'registered++;' if n.endswith('register') else ''} return {value if n == name else v}; }}"
                                     for n, v in has.items()]
    (tmp_path / "other.c").write_text("int registered;\n" + "\n".join(lines))
    subprocess.run(["cc", "-shared", "-fPIC", str(tmp_path / "other.c"), "-o", str(tmp_path / _hip.TORCH_LIB_NAME)], check=True)
    monkeypatch.setattr(_hip, "__file__", str(tmp_path / "_hip.py"))
    monkeypatch.setattr(_hip, "_native", None)
    with pytest.warns(UserWarning, match="slower Python path"):
        _hip.load_native()
    assert _hip._native is None
    registered = ctypes.c_int.in_dll(ctypes.CDLL(str(tmp_path / _hip.TORCH_LIB_NAME)), "registered").value
    assert registered == (name == "fa_torch_register")


def test_forced_backend_is_read_beside_threads_that_set_variables(monkeypatch):
    """The environment is read under the GIL, as the Python kernel reads it: threads may assign variables meanwhile."""
    forced = _hip._native.fa_torch_backend_forced  # (a ctypes call: without the GIL until the function takes it)
    monkeypatch.delenv("FUSED_ATTN_BACKEND", raising=False)
    assert not forced()
    for value in ("splitk", "bogus"):
        monkeypatch.setenv("FUSED_ATTN_BACKEND", value)
        assert forced()
    monkeypatch.setenv("FUSED_ATTN_BACKEND", "")
    assert not forced()
    stop = threading.Event()
    names = [f"FUSED_ATTN_TEST_{i}" for i in range(500)]

    def assign():
        while not stop.is_set():
            for n in names:  # growing the table moves it
                os.environ[n] = "x" * 100
            for n in names:
                del os.environ[n]

    thread = threading.Thread(target=assign)
    thread.start()
    try:
        assert not any(forced() for _ in range(3000))
    finally:
        stop.set()
        thread.join()


@pytest.fixture
def python_calls(monkeypatch):
    """Calls that reached the Python kernel, after one that let the device be found."""
    q = randn(1, 2, 8, 64, dtype=torch.float16)
    fused_attn.attention(q, q, q)
    calls = []
    for name in ("fwd", "splitk"):
        real = getattr(_hip, name)
        monkeypatch.setattr(_hip, name, lambda *a, _real=real, **kw: calls.append(1) or _real(*a, **kw))
    return calls


def _python(q, k, v, causal=False, scale=None):
    return ops.attention._init_fn(q, k, v, causal, scale)


def _qkv(b, hq, hkv, nq, nk, d, dtype, bnhd=False):
    if bnhd:
        return [randn(b, n, h, d, dtype=dtype).transpose(1, 2) for n, h in ((nq, hq), (nk, hkv), (nk, hkv))]
    return [randn(b, h, n, d, dtype=dtype) for n, h in ((nq, hq), (nk, hkv), (nk, hkv))]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("bnhd", [False, True])
def test_taken_calls_equal_the_python_kernel(dtype, d, bnhd, python_calls):
    announce(f"native dispatch {dtype} d={d} bnhd={bnhd}")
    torch.manual_seed(0)
    for nq, nk, causal, scale in ((1, 600, True, None), (37, 37, True, 0.3), (3, 2100, False, -0.1), (130, 70, True, 0), (64, 9000, True, None)):
        q, k, v = _qkv(2, 8, 2, nq, nk, d, dtype, bnhd)
        out = fused_attn.attention(q, k, v, causal=causal, scale=scale)
        assert not python_calls, "the native kernel should have taken this call"
        assert out.is_contiguous() and out.dtype == dtype
        assert torch.equal(out, _python(q, k, v, causal, scale))
        python_calls.clear()
    one = k[:1]  # a shared cache
    assert torch.equal(fused_attn.attention(q, one, one), _python(q, one, one))


@pytest.mark.gpu
def test_calls_that_need_preparation_go_on(python_calls, monkeypatch):
    announce("native dispatch: calls handed on")
    q, k, v = _qkv(1, 4, 2, 33, 65, 64, torch.bfloat16)
    shifted = torch.empty(q.numel() + 1, device="cuda", dtype=q.dtype)[1:].view(q.shape).copy_(q)  # 2-byte aligned
    strided = torch.empty(*q.shape[:3], 128, device="cuda", dtype=q.dtype)[..., ::2].copy_(q)
    want = fused_attn.attention(q, k, v)
    for x in (shifted, strided):
        n = len(python_calls)
        assert torch.equal(fused_attn.attention(x, k, v), want) and len(python_calls) == n + 1
    assert fused_attn.attention(q[:, :, :0], k, v).shape == (1, 4, 0, 64)
    monkeypatch.setenv("FUSED_ATTN_BACKEND", "splitk")
    n = len(python_calls)
    fused_attn.attention(q, k, v)
    assert len(python_calls) == n + 1
    monkeypatch.setenv("FUSED_ATTN_BACKEND", "bogus")
    with pytest.raises(ValueError):
        fused_attn.attention(q, k, v)
    monkeypatch.delenv("FUSED_ATTN_BACKEND")
    for bad in ((q, k.half(), v), (q, k, v[:, :, :-1]), (q, k.cpu(), v), (q[:, :3], k, v), (q[..., :32], k, v),
                (q.repeat(2, 1, 1, 1), k.repeat(3, 1, 1, 1), v.repeat(3, 1, 1, 1)), (q[0], k[0], v[0])):
        with pytest.raises(Exception) as native:
            fused_attn.attention(*bad)
        with pytest.raises(Exception) as python:
            _python(*bad)
        assert type(native.value) is type(python.value) and str(native.value) == str(python.value)


@pytest.mark.gpu
def test_autograd_and_tracing(python_calls):
    announce("native dispatch: autograd and tracing")
    q, k, v = _qkv(1, 4, 2, 33, 65, 64, torch.bfloat16)
    want = fused_attn.attention(q, k, v, causal=True)
    out = fused_attn.attention(q.clone().requires_grad_(), k, v, causal=True)
    assert out.requires_grad and torch.equal(out, want)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        out.sum().backward()
    with torch.no_grad():
        assert not fused_attn.attention(q.clone().requires_grad_(), k, v, causal=True).requires_grad
    with torch.inference_mode():
        assert torch.equal(fused_attn.attention(q, k, v, causal=True), want)
    torch.library.opcheck(fused_attn.attention, (q, k, v, True, None))
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode() as mode:
        f = fused_attn.attention(*(mode.from_tensor(x) for x in (q, k, v)))
    assert f.shape == q.shape and f.device == q.device
    from torch.utils._python_dispatch import TorchDispatchMode

    seen = []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Seen():
        assert torch.equal(fused_attn.attention(q, k, v, causal=True), want)
    assert "fused_attn.attention.default" in seen


@pytest.mark.gpu
def test_streams_threads_and_graphs(python_calls):
    announce("native dispatch: streams, threads and graphs")
    q, k, v = _qkv(2, 8, 2, 1, 3000, 128, torch.bfloat16)
    want = fused_attn.attention(q, k, v, causal=True)
    torch.cuda.synchronize()
    got = [None] * 4

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(20):
                got[i] = fused_attn.attention(q, k, v, causal=True)
        s.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert all(torch.equal(g, want) for g in got)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fused_attn.attention(q, k, v, causal=True)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(fused_attn.attention(q, k, v, causal=True), want)
    assert not python_calls
