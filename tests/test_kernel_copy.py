"""Copies of kernel objects, and of the layers that keep them: a model is deep-copied whole, called before or not."""

import copy

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib
from tilelang_amd.bitlinear import BitLinear
from tilelang_amd.w4linear import W4A16Linear

native = pytest.mark.skipif(_lib.host_call() is None, reason="the native call is not built")


def _mxfp4_args(device="cpu"):
    return (torch.zeros((3, 512), dtype=torch.bfloat16, device=device), torch.zeros((264, 256), dtype=torch.uint8, device=device),
            torch.zeros((264, 16), dtype=torch.uint8, device=device), None)


@pytest.mark.parametrize("bound", [False, pytest.param(True, marks=native)])
@pytest.mark.parametrize("make_copy", [copy.copy, copy.deepcopy])
def test_kernel_object(bound, make_copy):
    kernel = tl.matmul_bf16_mxfp4(3, 264, 512, weight_format="e2m1", scale_bias=127)
    if bound:  # what the first call does
        kernel._native = kernel._bind(kernel.result_idx)
        kernel._native_new[4] = kernel._bind([4])
        assert kernel._native is not None
    other = make_copy(kernel)
    assert other.params == kernel.params and other.result_idx == kernel.result_idx
    # a call that is refused gets as far as the operands' check, in the copy as in the original
    for k in (kernel, other):
        with pytest.raises(ValueError, match="device mismatch for parameter A"):
            k(*_mxfp4_args())


def test_kernel_object_without_native_call():
    kernel = tl.bitnet_activation_quant(2, 256)
    other = copy.deepcopy(kernel)
    with pytest.raises(ValueError, match="device mismatch for parameter x"):
        other(torch.zeros((2, 256), dtype=torch.float16))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["w4a16", "bitlinear"])
def test_layer(cuda, kind):
    layer = (W4A16Linear(512, 264, bias=True) if kind == "w4a16" else BitLinear(512, 264)).to(cuda)
    gen = torch.Generator().manual_seed(1)
    weight = torch.randn((264, 512), generator=gen)
    if kind == "w4a16":
        layer.load_float_weight(weight, torch.randn(264, generator=gen))
    else:
        layer.load_float_weight(weight)
    x = torch.randn((3, 512), generator=gen).to(cuda).half()
    want = layer(x)
    other = copy.deepcopy(layer)
    layer.qweight.zero_()  # the copy has weights of its own
    assert torch.equal(other(x), want) and not torch.equal(layer(x), want)
    assert torch.equal(copy.deepcopy(other)(x), want)
