"""K over the waves of a workgroup (dq_gemm_kwaves.h) at the edges of its walk: fewer chunks of K than waves, a chunk in part,
rows of scales that are no multiple of a window, ragged rows and columns, each of its forms.  Operands are small integers and
powers of two, so that every product and every fp32 sum is exact and the result is one rounding of the float64 product."""

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib

pytestmark = pytest.mark.gpu


def _ints(gen, lo, hi, *shape, dtype, device):
    return torch.randint(lo, hi + 1, shape, generator=gen, device=device).to(dtype)


def _nibbles(packed):
    b = packed.view(torch.uint8)
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1)


@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("decode", [0, 1])
@pytest.mark.parametrize("M,N,K", [
    (2, 2264, 1024), (3, 33, 128), (5, 97, 384), (16, 300, 2176),      # 16 rows; one to nine chunks of 256 k
    (17, 130, 256), (31, 1001, 1920), (32, 8200, 640),                 # 32 rows
    (33, 9000, 896), (48, 16400, 768), (64, 20003, 512), (61, 24700, 640),  # 32, 48 and 64 rows by 64 columns
    (65, 500, 2048), (129, 300, 1152), (200, 3001, 2304),              # passes
])
def test_int8_int4(cuda, M, N, K, decode, transposed):
    gen = torch.Generator(device=cuda).manual_seed(M + K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    C = torch.full((N + 1, M) if transposed else (M + 1, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, decode, 0, int(transposed),
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    codes = _nibbles(B).short()
    W = (torch.where(codes > 7, codes - 16, codes) if decode else codes).double()
    ref = (W @ A.double().t()) if transposed else (A.double() @ W.t())
    assert torch.equal(C[:-1], ref.int()) and bool((C[-1] == -7).all())


@pytest.mark.parametrize("M,N,K", [
    (3, 2100, 13824), (14, 2168, 6720), (17, 130, 512), (20, 1001, 576),  # the least K; a chunk in part
    (32, 8200, 2880), (33, 9000, 1088), (48, 16400, 768), (64, 20003, 832), (64, 3000, 2112),
    (101, 2000, 4800), (254, 1030, 1344),                                # passes (K % 128 == 64)
    (81, 2004, 1024), (95, 2760, 2304), (327, 1036, 1792), (204, 2912, 3328),  # in place of the cut over workgroups
])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
def test_mxfp4(cuda, fmt, with_bias, M, N, K):
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -2, 2, M, K, dtype=torch.bfloat16, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    S = _ints(gen, 125, 127, N, K // 32, dtype=torch.uint8, device=cuda)
    bias = _ints(gen, -3, 3, M, N, dtype=torch.bfloat16, device=cuda)
    C = tl.matmul_bf16_mxfp4(M, N, K, with_bias=with_bias, weight_format=fmt, scale_bias=127)(A, B, S, bias)
    code = _nibbles(B).int()
    if fmt == "e2m1":
        values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=cuda)
        W = torch.cat((values, -values))[code]
    else:
        value = torch.exp2(((code >> 1) & 3).double() - 1) * (1 + (code & 1).double() / 2)
        W = torch.where(code > 7, -value, value)
    W = W * torch.exp2(S.double() - 127).repeat_interleave(32, dim=1)
    ref = A.double() @ W.t()
    assert torch.equal(C, (ref + bias.double() if with_bias else ref).bfloat16())


def test_mxfp4_infinite_scale_stays_in_its_row(cuda):
    """K = 832 ends in a chunk of which a quarter is there: what the lanes hold of the rest (the next row's codes, some byte of
    the window) meets zeros with a finite scale, so one row's largest block exponents leave the others alone and are
    infinities or NaN exactly where the float64 product has them."""
    M, N, K = 40, 300, 832
    gen = torch.Generator(device=cuda).manual_seed(1)
    A = _ints(gen, 1, 2, M, K, dtype=torch.bfloat16, device=cuda)
    B = torch.full((N, K // 2), 0x22, dtype=torch.uint8, device=cuda)  # every weight 1.0
    S = torch.full((N, K // 32), 127, dtype=torch.uint8, device=cuda)
    S[7, -1] = 254
    S[8] = 0
    C = tl.matmul_bf16_mxfp4(M, N, K, weight_format="e2m1", scale_bias=127)(A, B, S, torch.zeros((M, N), dtype=torch.bfloat16, device=cuda))
    W = torch.exp2(S.double() - 127).repeat_interleave(32, dim=1)
    W[7, -32:] = 2.0 ** 127
    ref = (A.double() @ W.t()).float().bfloat16()
    keep = [n for n in range(N) if n != 8]  # (2 ** -127 is subnormal)
    assert torch.equal(C[:, keep], ref[:, keep])


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("M,N,K,group", [
    (3, 130, 1152, 128), (8, 1001, 3968, 64), (16, 515, 640, 64),        # nine groups: a window and one
    (24, 6712, 1408, 128), (33, 9000, 1152, 128), (48, 16400, 896, 64), (64, 20003, 1152, 128),
    (88, 700, 3712, 64), (200, 300, 1920, 128),
    (20, 300, 2176, 32),                                                 # a window a chunk
    (20, 300, 640, 128),                                                 # less than a window of groups: not this kernel's
])
def test_uint4(cuda, M, N, K, group, zeros):
    gen = torch.Generator(device=cuda).manual_seed(K + group)
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    B = _ints(gen, -128, 127, N, K // 2, dtype=torch.int8, device=cuda)
    S = torch.exp2(_ints(gen, -3, 0, N, K // group, dtype=torch.float16, device=cuda))
    Z = _ints(gen, 5, 11, N, K // group, dtype=torch.float16, device=cuda)
    kern = tl.matmul_w4a16(M, N, K, group_size=group, source_format="uint" if zeros else "int", with_zeros=zeros)
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    kern(A, B, S, *([Z] if zeros else []), C)
    zero = Z.double().repeat_interleave(group, dim=1) if zeros else 8.0
    W = (_nibbles(B).double() - zero) * S.double().repeat_interleave(group, dim=1)
    assert torch.equal(C, (A.double() @ W.t()).half())


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("convention", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [
    (5, 130, 384), (16, 1001, 2688), (9, 3248, 640),                     # K % 256 == 128, a chunk of 512 k in part
    (17, 300, 256), (32, 2000, 2048), (33, 9000, 768), (48, 16400, 512), (64, 20000, 1280),
    (145, 8296, 1024), (200, 700, 2560), (130, 515, 1152),
])
def test_int8_int2(cuda, M, N, K, convention, interleaved):
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    codes = _ints(gen, 0, 3, N, K // 16, 4, 4, dtype=torch.uint8, device=cuda)
    if interleaved:  # element e of a word at bit 8 (e % 4) + 2 (e / 4)
        packed = sum(codes[:, :, j] << (2 * j) for j in range(4))
    else:  # at bit 2 e
        packed = sum(codes[:, :, :, j] << (2 * j) for j in range(4))
    B = packed.reshape(N, K // 4).contiguous()
    C = torch.full((M, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint2(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, convention, int(interleaved), None,
                                                1.0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    c = codes.reshape(N, K).double()
    W = c if convention == 0 else (c - 2 if convention == 1 else torch.where(c > 1, c - 4, c))
    assert torch.equal(C, (A.double() @ W.t()).int())
