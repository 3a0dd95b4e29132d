"""The direct-to-LDS GEMM (dq_gemm_core.h) where K is an odd number of k-blocks or of scale groups: the walk ends on an even
tile, and every other row of scales starts in the middle of a dword.  Operands are small integers and powers of two, so that
every product and every fp32 sum is exact and the result is one rounding of the float64 product."""

import numpy as np
import pytest
import torch

import tilelang_amd as tl
from oracle import dq_oracle as orc
from tilelang_amd import _lib

pytestmark = pytest.mark.gpu

# many tiles and few; ragged last tiles of odd widths (with an odd count of groups such a call is staged through registers)
TALL, HALF = (2570, 5131), (1100, 3503)


def _rows(operands, M, N, K, group=0, mode=0):
    """The rows of the direct-to-LDS kernel's tiles that the call runs on."""
    return _lib.load_library().dq_tile_rows(operands, M, N, K, group, mode)


def _ints(gen, lo, hi, *shape, dtype, device):
    return torch.randint(lo, hi + 1, shape, generator=gen, device=device).to(dtype)


def _nibbles(packed):
    b = packed.view(torch.uint8)
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1)


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("M,N", [TALL, HALF, (1100, 3504)])
@pytest.mark.parametrize("K,group", [
    (192, 64), (320, 64), (448, 64),     # odd tiles and odd groups; the slot of dword 0 is due again from the seventh tile on
    (576, 64), (832, 64), (1088, 64),
    (384, 128), (640, 128), (1152, 128), (1408, 128),  # odd groups, even tiles (eight waves beyond K = 1024)
    (768, 256), (1792, 256), (3584, 512),
    (320, 32), (224 * 3 - 32, 32),
])
def test_uint4(cuda, M, N, K, group, zeros):
    _uint4(cuda, M, N, K, group, zeros)


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("rows,M,N,K,group", [
    (128, 1020, 8190, 192, 64), (128, 1020, 8190, 448, 64), (128, 1020, 8190, 1088, 64), (128, 2041, 4090, 384, 128),
    (128, 1020, 8190, 1152, 128), (128, 1020, 8190, 1792, 256), (128, 1020, 8190, 320, 32), (128, 1020, 8185, 320, 32),
    (256, 2570, 5132, 640, 64), (256, 2570, 5132, 832, 64), (256, 2570, 5132, 1152, 128), (256, 3050, 5100, 1792, 256), (256, 3050, 5100, 1088, 64),
    (192, 2050, 5132, 192, 64), (192, 2050, 5132, 1152, 128), (96, 257, 20002, 448, 64), (96, 257, 20002, 1408, 128),
])
def test_uint4_on_tiles(cuda, rows, M, N, K, group, zeros):
    assert _rows(_lib.OPERANDS_F16_UINT4, M, N, K, group, 5 if zeros else 3) == rows
    _uint4(cuda, M, N, K, group, zeros)


def _uint4(cuda, M, N, K, group, zeros):
    gen = torch.Generator(device=cuda).manual_seed(K + group)
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    B = _ints(gen, -128, 127, N, K // 2, dtype=torch.int8, device=cuda)
    S = torch.exp2(_ints(gen, -4, 0, N, K // group, dtype=torch.float16, device=cuda))
    Z = _ints(gen, 5, 11, N, K // group, dtype=torch.float16, device=cuda)
    C = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=cuda)
    mode = 5 if zeros else 3
    rc = _lib.get_library().call_dequant_gemm_w4_fp16(A.data_ptr(), B.data_ptr(), S.data_ptr(), Z.data_ptr() if zeros else None,
                                                      C.data_ptr(), M, N, K, group, mode, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    zero = Z.double().repeat_interleave(group, dim=1) if zeros else 8.0
    W = (_nibbles(B).double() - zero) * S.double().repeat_interleave(group, dim=1)
    assert torch.equal(C[:M], (A.double() @ W.t()).half()) and bool(torch.isnan(C[M]).all())


@pytest.mark.parametrize("M,N", [TALL, HALF])
@pytest.mark.parametrize("K", [192, 320, 448, 576, 1088])
@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
def test_mxfp4(cuda, M, N, K, fmt):
    _mxfp4(cuda, M, N, K, fmt)


@pytest.mark.parametrize("rows,M,N,K", [
    (128, 1020, 8190, 192), (128, 1020, 8190, 448), (128, 2041, 4090, 1088), (128, 2570, 5132, 576),
    (256, 3050, 5100, 1088), (256, 3050, 5100, 1344), (256, 2570, 5132, 1600),  # B by pairs of tiles: the last pair is half
    (192, 2050, 5132, 1088), (96, 1100, 3504, 1088), (96, 257, 20002, 448),
])
@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
def test_mxfp4_on_tiles(cuda, rows, M, N, K, fmt):
    assert _rows(_lib.OPERANDS_BF16_MXFP4, M, N, K) == rows
    _mxfp4(cuda, M, N, K, fmt)


def _mxfp4(cuda, M, N, K, fmt):
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -2, 2, M, K, dtype=torch.bfloat16, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    S = _ints(gen, 124, 127, N, K // 32, dtype=torch.uint8, device=cuda)
    kern = tl.matmul_bf16_mxfp4(M, N, K, weight_format=fmt, scale_bias=127)
    C = kern(A, B, S, torch.zeros((M, N), dtype=torch.bfloat16, device=cuda))
    code = _nibbles(B).int()
    if fmt == "e2m1":
        values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=cuda)
        W = torch.cat((values, -values))[code]
    else:  # bits (s << 15) | ((E + 126) << 7) | (m << 6)
        value = torch.exp2(((code >> 1) & 3).double() - 1) * (1 + (code & 1).double() / 2)
        W = torch.where(code > 7, -value, value)
    W = W * torch.exp2(S.double() - 127).repeat_interleave(32, dim=1)
    assert torch.equal(C, (A.double() @ W.t()).bfloat16())


@pytest.mark.parametrize("M,N", [TALL, HALF, (1020, 8190), (1017, 8191)])
@pytest.mark.parametrize("K", [384, 640, 896, 1408])
@pytest.mark.parametrize("transposed", [True, False])
def test_int8_int4(cuda, M, N, K, transposed):
    assert _rows(_lib.OPERANDS_INT8_INT4, M, N, K) == {TALL: 256, HALF: 0}.get((M, N), 128)
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    C = torch.full((N, M) if transposed else (M, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 1, 0, int(transposed),
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    codes = _nibbles(B).short()
    W = torch.where(codes > 7, codes - 16, codes).double()
    ref = (W @ A.double().t()) if transposed else (A.double() @ W.t())
    assert torch.equal(C, ref.int())


@pytest.mark.parametrize("M,N", [TALL, (2050, 5131), HALF])
@pytest.mark.parametrize("K", [384, 640, 1152, 1408])
def test_bitnet(cuda, M, N, K):
    _bitnet(cuda, M, N, K)


@pytest.mark.parametrize("rows,M,N,K", [
    (128, 2570, 5131, 384), (128, 2570, 8190, 640), (128, 1020, 8185, 1152), (128, 2041, 4090, 1408), (128, 1020, 8190, 2432),
    (256, 2040, 6141, 4480), (192, 1089, 10703, 3456), (96, 2050, 5131, 384), (96, 1281, 4073, 1152),
])
def test_bitnet_on_tiles(cuda, rows, M, N, K):
    assert _rows(_lib.OPERANDS_INT8_INT2, M, N, K) == rows
    _bitnet(cuda, M, N, K)


def _bitnet(cuda, M, N, K):
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    codes = _ints(gen, 0, 3, N, K // 4, 4, dtype=torch.uint8, device=cuda)  # code e of a byte at bit 2 e
    B = codes[..., 0] | (codes[..., 1] << 2) | (codes[..., 2] << 4) | (codes[..., 3] << 6)
    C = torch.full((M, N), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint2(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 1, 0, None, 1.0, 0,
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    W = codes.reshape(N, K).double() - 2
    assert torch.equal(C, (A.double() @ W.t()).int())


@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("K,split", [(384, 2), (640, 2), (576, 3), (512, 2)])  # the last: an even count
def test_fp16_fp4_slices(cuda, K, split, transposed):
    """An even number of k-blocks in all and an odd one in each equal slice."""
    M, N = HALF[0], 3504
    rng = np.random.default_rng(K)
    A = rng.integers(-2, 3, size=(M, K)).astype(np.float16)
    B = rng.integers(0, 256, size=(N, K // 2), dtype=np.uint8) & 0x33  # magnitudes to 1.5
    out = tl.matmul_fp16_fp4(M, N, K, split=split, transposed_output=transposed)(torch.from_numpy(A).to(cuda), torch.from_numpy(B).to(cuda))
    ref = orc.ref_fp16xfp4_splitk(A, B, split)
    np.testing.assert_array_equal(out.cpu().numpy(), ref.T if transposed else ref)
