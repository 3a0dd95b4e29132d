"""The native call of kernel objects (csrc/host_call.cpp): the same results as the adapter's own code, and what it does not
settle (a stream of the caller's, a wrong operand, a subclass, a mode) is the adapter's to carry out or to refuse."""

import threading

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import tilelang_amd as tl
from tilelang_amd.w4linear import W4A16Linear

pytestmark = pytest.mark.gpu


def _mxfp4(cuda, M, N, K, bias):
    gen = torch.Generator(device=cuda).manual_seed(M + N)
    return (torch.randn((M, K), generator=gen, device=cuda).bfloat16(),
            torch.randint(0, 256, (N, K // 2), generator=gen, device=cuda, dtype=torch.uint8),
            torch.randint(119, 128, (N, K // 32), generator=gen, device=cuda, dtype=torch.uint8),
            torch.randn((M, N), generator=gen, device=cuda).bfloat16() if bias else None)


def _python(kernel, *inputs):
    native, kernel._native = kernel._native, None
    try:
        return kernel(*inputs)
    finally:
        kernel._native = native


@pytest.mark.parametrize("M,N,K,bias", [(1, 264, 192, True), (3, 264, 512, False), (96, 2048, 8192, True), (200, 520, 256, True)])
def test_same_results(cuda, M, N, K, bias):
    args = _mxfp4(cuda, M, N, K, bias)
    kernel = tl.matmul_bf16_mxfp4(M, N, K, with_bias=bias, weight_format="e2m1", scale_bias=127)
    want = _python(kernel, *args)
    assert torch.equal(kernel(*args), want)
    assert kernel._native(*args) is not NotImplemented
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        on_side = kernel(*args)
    side.synchronize()
    named = kernel(*args, stream=side.cuda_stream)
    side.synchronize()
    assert torch.equal(on_side, want) and torch.equal(named, want)
    results = [None] * 4

    def work(i):
        for _ in range(20):
            results[i] = kernel(*args)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    torch.cuda.synchronize()
    assert all(torch.equal(r, want) for r in results)


def test_unsettled_calls(cuda):
    kernel = tl.matmul_bf16_mxfp4(3, 264, 512, weight_format="e2m1", scale_bias=127)
    a, b, s, bias = _mxfp4(cuda, 3, 264, 512, True)
    want = kernel(a, b, s, bias)
    assert kernel._native(a, b, s, bias) is not NotImplemented
    for wrong, message in (((a.float(), b, s, bias), "dtype mismatch for parameter A"), ((a, b[:-1], s, bias), "shape mismatch for parameter B"),
                           ((a, b, s.cpu(), bias), "device mismatch for parameter Scale"),
                           ((a, b, s, torch.empty((3, 528), dtype=torch.bfloat16, device=cuda)[:, ::2]), "stride mismatch for parameter Bias"),
                           ((a, b, s), "Expected 5 inputs, got 4")):
        with pytest.raises(ValueError, match=message):
            kernel(*wrong)

    class Sub(torch.Tensor):
        pass

    assert kernel._native(a.as_subclass(Sub), b, s, bias) is NotImplemented
    assert torch.equal(kernel(a.as_subclass(Sub), b.view(torch.int8), s, bias), want)
    seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        assert torch.equal(kernel(a, b, s, bias), want)
    assert torch.ops.aten.empty.memory_format in seen


@pytest.mark.parametrize("zeros", [False, True])
def test_w4a16_layer(cuda, zeros):
    K, N = 512, 264
    layer = W4A16Linear(K, N, with_zeros=zeros, bias=True).to(cuda)
    layer.load_float_weight(torch.randn((N, K)), torch.randn(N))
    x = torch.randn((2, 3, K), device=cuda).half()
    out = layer(x)
    assert out.shape == (2, 3, N)
    kernel = layer._get_kernel(6)
    ref = torch.empty((6, N), dtype=torch.float16, device=cuda)
    _python(kernel, x.reshape(6, K), layer.qweight, layer.scales, *([layer.zeros] if zeros else []), ref)
    assert torch.equal(out.reshape(6, N), ref + layer.bias) and torch.equal(layer(x.reshape(6, K)), out.reshape(6, N))
    assert layer(x[0, 0]).shape == (N,) and torch.equal(layer(x.float()), out)
    with pytest.raises(RuntimeError):
        layer(torch.zeros((2, 2 * K), dtype=torch.float16, device=cuda))
    qweight = layer.qweight
    del layer.qweight
    layer.qweight = torch.nn.Parameter(qweight, requires_grad=False)
    assert torch.equal(layer(x), out)
