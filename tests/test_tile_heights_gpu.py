"""The direct-to-LDS GEMM (dq_gemm_core.h) on tiles of 96 and of 192 rows, where those fill their rounds of workgroups best: odd
and even counts of k-blocks, on four waves and on eight, ragged last tiles, groups of every kind.  Every case names the tile's rows
and asks the library whether it would take them.  Operands are small integers and powers of two, so that every product and every
fp32 sum is exact and the result is one rounding of the float64 product."""

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib

pytestmark = pytest.mark.gpu

# (rows of the tile, M, N): one row beyond a block of 32, one short of a tile, rows of C off 32 bytes
SHAPES = [(192, 1089, 10700), (192, 1151, 10752), (96, 280, 20000), (96, 257, 20002), (96, 288, 21504), (128, 481, 12544)]


def _rows(operands, M, N, K, group=0, mode=0):
    return _lib.load_library().dq_tile_rows(operands, M, N, K, group, mode)


def _ints(gen, lo, hi, *shape, dtype, device):
    return torch.randint(lo, hi + 1, shape, generator=gen, device=device).to(dtype)


def _nibbles(packed):
    b = packed.view(torch.uint8)
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1)


@pytest.mark.parametrize("rows,M,N", SHAPES)
@pytest.mark.parametrize("K,group,zeros", [
    (192, 64, True), (320, 64, False), (384, 128, True), (512, 32, False), (1024, 128, True),   # four waves
    (1152, 128, True), (1280, 64, False), (1536, 512, True),                                     # eight on tiles of 96 rows
])
def test_uint4(cuda, rows, M, N, K, group, zeros):
    assert _rows(_lib.OPERANDS_F16_UINT4, M, N, K, group, 5 if zeros else 3) == rows
    gen = torch.Generator(device=cuda).manual_seed(K + M)
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    B = _ints(gen, -128, 127, N, K // 2, dtype=torch.int8, device=cuda)
    S = torch.exp2(_ints(gen, -4, 0, N, K // group, dtype=torch.float16, device=cuda))
    Z = _ints(gen, 5, 11, N, K // group, dtype=torch.float16, device=cuda)
    C = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=cuda)
    rc = _lib.get_library().call_dequant_gemm_w4_fp16(A.data_ptr(), B.data_ptr(), S.data_ptr(), Z.data_ptr() if zeros else None, C.data_ptr(),
                                                      M, N, K, group, 5 if zeros else 3, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    zero = Z.double().repeat_interleave(group, dim=1) if zeros else 8.0
    W = (_nibbles(B).double() - zero) * S.double().repeat_interleave(group, dim=1)
    assert torch.equal(C[:M], (A.double() @ W.t()).half()) and bool(torch.isnan(C[M]).all())


# (the rule takes 96 rows for the first shapes at a shorter K)
@pytest.mark.parametrize("rows,M,N,K", [(rows, M, N, K) for rows, M, N in SHAPES for K in ((1088, 1280, 1344) if rows == 192 else (128, 192, 1088, 1280))])
@pytest.mark.parametrize("with_bias", [False, True])
def test_mxfp4(cuda, rows, M, N, K, with_bias):
    assert _rows(_lib.OPERANDS_BF16_MXFP4, M, N, K) == rows
    gen = torch.Generator(device=cuda).manual_seed(K + M)
    A = _ints(gen, -2, 2, M, K, dtype=torch.bfloat16, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    S = _ints(gen, 124, 127, N, K // 32, dtype=torch.uint8, device=cuda)
    bias = _ints(gen, -3, 3, M, N, dtype=torch.bfloat16, device=cuda)
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=cuda)
    rc = _lib.get_library().call_dequant_gemm_bf16_mxfp4(A.data_ptr(), B.data_ptr(), S.data_ptr(), bias.data_ptr() if with_bias else None,
                                                         C.data_ptr(), M, N, K, 32, 0, 127, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=cuda)
    W = torch.cat((values, -values))[_nibbles(B).int()] * torch.exp2(S.double() - 127).repeat_interleave(32, dim=1)
    ref = A.double() @ W.t()
    assert torch.equal(C, (ref + bias.double() if with_bias else ref).bfloat16())


@pytest.mark.parametrize("M,N", [(280, 20000), (1089, 10700)])
def test_mxfp4_rows_keep_their_bits(cuda, M, N):
    """Uncut, a row's products are added in one order whatever the tile: real-valued operands, against a call of 80 rows."""
    K = 1280
    assert _rows(_lib.OPERANDS_BF16_MXFP4, M, N, K) in (96, 192)
    gen = torch.Generator(device=cuda).manual_seed(M)
    A = torch.randn((M, K), generator=gen, device=cuda).bfloat16()
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    S = _ints(gen, 119, 127, N, K // 32, dtype=torch.uint8, device=cuda)
    out = []
    for a in (A, A[M - 80:].contiguous()):
        C = torch.empty((a.shape[0], N), dtype=torch.bfloat16, device=cuda)
        rc = _lib.get_library().call_dequant_gemm_bf16_mxfp4(a.data_ptr(), B.data_ptr(), S.data_ptr(), None, C.data_ptr(), a.shape[0], N, K,
                                                             32, 0, 127, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _lib.last_error()
        out.append(C)
    assert torch.equal(out[0][M - 80:].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("M,N", [(1089, 10700), (1151, 10752), (1092, 10700)])
@pytest.mark.parametrize("K", [256, 384, 1152])
@pytest.mark.parametrize("transposed", [True, False])
def test_int8_int4(cuda, M, N, K, transposed):
    """No tiles of these heights for it: 256 rows."""
    assert _rows(_lib.OPERANDS_INT8_INT4, M, N, K) == 256
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    C = torch.full((N, M) if transposed else (M, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 1, 0, int(transposed),
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    codes = _nibbles(B).short()
    W = torch.where(codes > 7, codes - 16, codes).double()
    assert torch.equal(C, ((W @ A.double().t()) if transposed else (A.double() @ W.t())).int())


# four waves to K = 1024, eight beyond, an even and an odd count of k-blocks each; 192 rows at a longer K only
@pytest.mark.parametrize("rows,M,N,K", [(rows, M, N, K) for rows, M, N in SHAPES for K in ((3328, 3456) if rows == 192 else (256, 1024, 1152, 1280, 1536))]
                         + [(96, 1089, 10700, 384), (96, 1151, 10752, 640), (192, 1151, 10748, 3456)])
def test_bitnet(cuda, rows, M, N, K):
    assert _rows(_lib.OPERANDS_INT8_INT2, M, N, K) == rows
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    codes = _ints(gen, 0, 3, N, K // 4, 4, dtype=torch.uint8, device=cuda)  # code e of a byte at bit 2 e
    B = codes[..., 0] | (codes[..., 1] << 2) | (codes[..., 2] << 4) | (codes[..., 3] << 6)
    C = torch.full((M, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint2(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 1, 0, None, 1.0, 0,
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    assert torch.equal(C, (A.double() @ (codes.reshape(N, K).double() - 2).t()).int())
