"""MXFP4 x bf16 at a decode batch where K is an odd number of 64 k and too long for one slice of the register-resident kernel:
the last chunk of the last slice is half empty.  Operands are small integers and powers of two: every sum is exact."""

import pytest
import torch

import tilelang_amd as tl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (3, 130, 6208), (16, 515, 7232), (20, 64, 8128),                  # two slices, seven or eight chunks a wave without them
    (1, 1001, 8256), (2, 130, 8256), (8, 4100, 8256), (16, 33, 12352),  # two slices, three; one and two rows: dot products
    (1, 130, 9728), (2, 65, 12288), (1, 40, 18432), (2, 33, 18240),   # whole ones: dot products in chunks of three steps
    (1, 40, 32832), (5, 64, 24640),                                   # beyond the dot-product kernel; five slices
])
def test_half_chunk(cuda, fmt, with_bias, M, N, K):
    gen = torch.Generator(device=cuda).manual_seed(K + N)

    def ints(lo, hi, *shape, dtype):
        return torch.randint(lo, hi + 1, shape, generator=gen, device=cuda).to(dtype)

    A = ints(-2, 2, M, K, dtype=torch.bfloat16)
    B = ints(0, 255, N, K // 2, dtype=torch.uint8)
    S = ints(125, 127, N, K // 32, dtype=torch.uint8)
    bias = ints(-3, 3, M, N, dtype=torch.bfloat16)
    C = tl.matmul_bf16_mxfp4(M, N, K, with_bias=with_bias, weight_format=fmt, scale_bias=127)(A, B, S, bias)
    code = torch.stack((B & 15, B >> 4), dim=-1).reshape(N, K).int()
    if fmt == "e2m1":
        values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=cuda)
        W = torch.cat((values, -values))[code]
    else:
        value = torch.exp2(((code >> 1) & 3).double() - 1) * (1 + (code & 1).double() / 2)
        W = torch.where(code > 7, -value, value)
    W = W * torch.exp2(S.double() - 127).repeat_interleave(32, dim=1)
    ref = A.double() @ W.t()
    assert torch.equal(C, (ref + bias.double() if with_bias else ref).bfloat16())
