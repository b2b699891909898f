"""The direct calls (csrc/host.cpp) against the Python wrappers they stand in
for: the same results for every form of argument, and NotImplemented wherever
the wrapper has to do the work."""
import threading
import warnings

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import omni_int8 as oi
from omni_int8 import _lib, convrot, f16


class NoDirect:
    """Every direct call refused: the Python wrappers alone."""

    def __getattr__(self, name):
        return lambda *a: NotImplemented


def calls(device):
    g = torch.Generator().manual_seed(3)
    x = torch.randn((24, 512), generator=g).half().to(device)
    w = torch.randint(-127, 128, (96, 512), generator=g, dtype=torch.int8).to(device)
    scale = torch.rand(96, generator=g).to(device)
    zero = torch.randint(-3, 4, (96,), generator=g, dtype=torch.int32).to(device)
    bias = torch.randn(96, generator=g).to(device)
    q = torch.randint(0, 256, (96, 256), generator=g, dtype=torch.uint8).to(device)
    gs = torch.rand((96, 4), generator=g).bfloat16().to(device)
    wf = torch.randn((96, 512), generator=g).half().to(device)
    big = torch.randn((256, 4096), generator=g).half().to(device)
    wbig = (torch.randn((4096, 4096), generator=g) * 0.02).half().to(device)
    packed = oi.pack_i8(w)
    layer = convrot.Int8Linear(512, 96, packed, scale, zero)
    layer32 = convrot.Int8Linear(512, 96, packed, scale, zero, torch.float32)
    return {
        "try": lambda: oi.try_int8_gemm(x, packed, scale, zero),
        "try f32": lambda: oi.try_int8_gemm(x.float(), packed, scale, zero),
        "try bf16 strided": lambda: oi.try_int8_gemm(x.t().contiguous().t().bfloat16(), packed, scale, zero.long()),
        "try grad": lambda: oi.try_int8_gemm(x.float().requires_grad_(), packed, torch.nn.Parameter(scale), zero),
        "try None": lambda: oi.try_int8_gemm(x, packed[:-1], scale, zero),
        "quantize": lambda: oi.quantize_rows(x),
        "quantize strided": lambda: oi.quantize_rows(x[:, 8:264]),
        "quantize columns": lambda: oi.quantize_rows(x[:, ::2]),
        "gemm": lambda: oi.w8a8_gemm(w[:24], bias[:24], zero[:24], w, scale, zero, bias, torch.float16),
        "gemm plain": lambda: oi.w8a8_gemm(w[:24], bias[:24], None, w, scale),
        "gemm dump": lambda: oi.w8a8_gemm(w[:24], bias[:24], None, w, scale, acc_dump=True),
        "gemm words": lambda: oi.w8a8_gemm(w[:24], bias[:24], None, packed, scale),
        "w8a16": lambda: oi.w8a16_linear(x, w, scale.half()),
        "w8a16 bias 3d": lambda: oi.w8a16_linear(x.reshape(4, 6, 512), w, scale.half(), bias.half()),
        "w8a16 vector": lambda: oi.w8a16_linear(x[0], w, scale.half()),
        "w8a16 strided": lambda: oi.w8a16_linear(x[::2], w[:, :].t().contiguous().t(), scale.half()),
        "w4a16": lambda: oi.w4a16_linear(x, q, gs),
        "w4a16 bias": lambda: oi.w4a16_linear(x[:3], q, gs.reshape(-1), bias.half(), 128),
        "f16 gemv": lambda: f16.depth_try_linear(x, wf.t()),
        "f16 gemv copy": lambda: f16.depth_try_linear(x[:, None], wf.t().contiguous()),
        "f16 None": lambda: f16.depth_try_linear(big, wbig.t()),
        "f16 gemm": lambda: f16.tensorops_try_linear(big, wbig.t()),
        "convrot": lambda: layer(x),
        "convrot f32": lambda: layer32(x.float().reshape(2, 12, 512)),
        "convrot bf16": lambda: layer(x.bfloat16()),
    }


def flat(v):
    return list(v) if isinstance(v, tuple) else [v]


def same(a, b):
    for u, v in zip(flat(a), flat(b), strict=True):
        if u is None or v is None:
            assert u is None and v is None
            continue
        assert (u.shape, u.dtype, u.stride(), u.requires_grad) == (v.shape, v.dtype, v.stride(), v.requires_grad)
        assert torch.equal(u.contiguous().view(torch.uint8), v.contiguous().view(torch.uint8))


@pytest.mark.gpu
def test_direct_calls_equal_the_wrappers(monkeypatch):
    every = calls("cuda")
    got = {k: f() for k, f in every.items()}
    monkeypatch.setattr(_lib, "_host", NoDirect())
    for k, f in every.items():
        same(got[k], f())


@pytest.mark.gpu
def test_direct_calls_refuse_what_is_not_plain():
    h = _lib.host()
    x = torch.randn((4, 512), device="cuda").half()
    w = torch.zeros((96, 512), dtype=torch.int8, device="cuda")
    s = torch.ones(96, dtype=torch.float16, device="cuda")
    assert h.w8a16_linear(x, w, s, None) is not NotImplemented

    class Sub(torch.Tensor):
        pass

    for bad in ((x.as_subclass(Sub), w, s, None), (x.cpu(), w, s, None), (x, w.cpu(), s, None), (x[:0], w, s, None),
                (x, w, s[:95], None), (x, w[:, :256], s, None), (x.float(), w, s, None), (x, w, None, None),
                (x, w, s, s.float()), (x.to_sparse(), w, s, None), (x, w, s), (1, w, s, None)):
        assert h.w8a16_linear(*bad) is NotImplemented
    seen = []

    class FunctionMode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class DispatchMode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    for mode in (FunctionMode, DispatchMode):
        seen.clear()
        with mode():
            assert h.w8a16_linear(x, w, s, None) is NotImplemented
            oi.w8a16_linear(x, w, s)
        assert seen


@pytest.mark.gpu
def test_direct_calls_from_threads_and_streams():
    every = calls("cuda")
    want = {k: f() for k, f in every.items()}
    torch.cuda.synchronize()
    errors = []

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(3):
                    got = {k: f() for k, f in every.items()}
                torch.cuda.current_stream().synchronize()
            for k in got:
                same(got[k], want[k])
        except Exception as e:  # noqa: BLE001
            errors.append(repr(e))

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


@pytest.mark.parametrize("content", [None, b"not a shared object"])
def test_calls_work_without_the_module(content, tmp_path, monkeypatch):
    # The library alone is enough, as it was before the direct calls: a module
    # that is missing or does not load is said once, and the wrappers do the work.
    path = tmp_path / "_host.so"
    if content:
        path.write_bytes(content)
    monkeypatch.setattr(_lib, "HOST_PATH", str(path))
    monkeypatch.setattr(_lib, "_host", None)
    x, w = torch.zeros((2, 64)).half(), torch.zeros((64, 8)).half()
    with pytest.warns(RuntimeWarning, match="does not load"):
        assert f16.depth_try_linear(x, w) is None  # host tensors
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert f16.depth_try_linear(x, w) is None
        with pytest.raises(oi.OmniError):
            oi.quantize_rows(x)
    assert all(getattr(_lib.host(), name)() is NotImplemented for name in _lib.HOST_CALLS)


@pytest.mark.gpu
def test_calls_run_without_the_module(tmp_path, monkeypatch):
    every = calls("cuda")
    want = {k: f() for k, f in every.items()}
    monkeypatch.setattr(_lib, "HOST_PATH", str(tmp_path / "_host.so"))
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.warns(RuntimeWarning, match="does not load"):
        got = {k: f() for k, f in every.items()}
    for k in every:
        same(got[k], want[k])


def test_direct_calls_leave_host_tensors_to_the_wrapper():
    h = _lib.host()
    x, w = torch.zeros((2, 64)).half(), torch.zeros((8, 64), dtype=torch.int8)
    one, z = torch.ones(8), torch.zeros(8, dtype=torch.int32)
    assert h.try_int8_gemm(x, oi.pack_i8(w), one, z) is NotImplemented
    assert h.convrot_linear(x, oi.pack_i8(w), one, z, True) is NotImplemented
    assert h.quantize_rows(x) is NotImplemented
    assert h.w8a8_gemm(w, one, None, w, one, None, None, False) is NotImplemented
    assert h.w8a16_linear(x, w, one.half(), None) is NotImplemented
    assert h.w4a16_linear(x, w[:, :32].to(torch.uint8), one.bfloat16(), None, 64) is NotImplemented
    assert h.f16_linear(False, x, w.half().t()) is NotImplemented
    with pytest.raises(oi.OmniError):
        oi.w8a16_linear(x, w, one.half())
    with pytest.raises(ValueError):
        h.bind({})
