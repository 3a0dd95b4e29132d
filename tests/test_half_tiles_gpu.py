"""The 128 x 256 tile of the direct-to-LDS GEMM (dq_gemm_core.h) at the edges of its walk over K and of the matrix, and the
stores of rows that are no whole cache lines.  Operands are small integers and powers of two, so that every product and every
fp32 sum is exact and the result is one rounding of the float64 product, whatever order the kernel adds in."""

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib, quantize

pytestmark = pytest.mark.gpu

# What the rule leaves on tiles of 128 rows, whatever K: 256 of them, or some hundreds
ON_128 = ((1020, 8190), (2041, 4090), (2570, 8190), (1367, 13198))


def _on_128(operands, M, N, K, group=0, mode=0):
    return (M, N) not in ON_128 or _lib.load_library().dq_tile_rows(operands, M, N, K, group, mode) == 128


def _ints(gen, lo, hi, *shape, dtype, device):
    return torch.randint(lo, hi + 1, shape, generator=gen, device=device).to(dtype)


def _nibbles(packed):
    b = packed.view(torch.uint8)
    return torch.stack((b & 15, b >> 4), dim=-1).reshape(b.shape[0], -1)


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("M,N,K,group", [
    (1025, 3076, 384, 64),    # up to K = 1024 four waves; one row and four columns in the last tiles
    (1100, 3500, 256, 128),
    (1100, 3500, 640, 64),
    (1100, 3500, 1024, 128),  # a dword of scales every other stage
    (1025, 3076, 1152, 64),   # nine stages of 128 k on eight waves, a dword of scales each
    (1100, 3500, 1280, 128),  # every other
    (1100, 3500, 3072, 512),  # every eighth
    (1100, 3500, 1536, 32),   # one per 64 k: four waves
    (1100, 3500, 512, 32),
    (897, 4104, 1024, 256),   # rows of C that are no whole lines
    (897, 4104, 1280, 256),
    (2600, 6200, 2048, 256), (2600, 6200, 2304, 256),  # more than 512 tiles: four waves to K = 2048, eight beyond
    (1020, 8190, 384, 64), (1020, 8190, 256, 128), (1020, 8190, 1024, 128), (2041, 4090, 640, 64),  # as above, on tiles of 128 rows
    (1020, 8190, 1152, 64), (1020, 8190, 1280, 128), (2041, 4090, 3072, 512), (1020, 8190, 1536, 32), (1020, 8190, 512, 32),
    (1367, 13198, 2048, 256), (1367, 13198, 2304, 256),
])
def test_uint4(cuda, M, N, K, group, zeros):
    assert _on_128(_lib.OPERANDS_F16_UINT4, M, N, K, group, 5 if zeros else 3)
    gen = torch.Generator(device=cuda).manual_seed(K + group)
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    B = _ints(gen, -128, 127, N, K // 2, dtype=torch.int8, device=cuda)
    S = torch.exp2(_ints(gen, -4, 0, N, K // group, dtype=torch.float16, device=cuda))
    Z = _ints(gen, 5, 11, N, K // group, dtype=torch.float16, device=cuda)
    kern = tl.matmul_w4a16(M, N, K, group_size=group, source_format="uint" if zeros else "int", with_zeros=zeros)
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    kern(A, B, S, *([Z] if zeros else []), C)
    zero = Z.double().repeat_interleave(group, dim=1) if zeros else 8.0
    W = (_nibbles(B).double() - zero) * S.double().repeat_interleave(group, dim=1)
    assert torch.equal(C, (A.double() @ W.t()).half())


@pytest.mark.parametrize("K", [384, 640, 256, 1152, 1280])
def test_fp4(cuda, K):
    M, N = 1100, 3500
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -2, 2, M, K, dtype=torch.bfloat16, device=cuda)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=cuda)
    rc = _lib.get_library().call_dequant_gemm_bf16_fp4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 0,
                                                       torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    values = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=cuda)
    W = torch.cat((values, -values))[_nibbles(B).int()]
    assert torch.equal(C, (A.double() @ W.t()).bfloat16())


@pytest.mark.parametrize("M,N,K", [(1100, 3500, 640), (1100, 3500, 128), (2600, 6200, 384), (1020, 8190, 640), (2570, 8190, 384)])
def test_mxfp4_rows_keep_their_bits(cuda, M, N, K):
    """Uncut, a row's products are added in one order whatever tile the call runs on: the rows of a large product against
    a call of 80 of them (real-valued operands, so that another order would show)."""
    assert _on_128(_lib.OPERANDS_BF16_MXFP4, M, N, K)
    gen = torch.Generator(device=cuda).manual_seed(N + K)
    A = torch.randn((M, K), generator=gen, device=cuda).bfloat16()
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    S = _ints(gen, 119, 127, N, K // 32, dtype=torch.uint8, device=cuda)
    out = []
    for a in (A, A[M - 80:].contiguous()):
        C = torch.empty((a.shape[0], N), dtype=torch.bfloat16, device=cuda)
        rc = _lib.get_library().call_dequant_gemm_bf16_mxfp4(a.data_ptr(), B.data_ptr(), S.data_ptr(), None, C.data_ptr(),
                                                             a.shape[0], N, K, 32, 0, 127, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _lib.last_error()
        out.append(C)
    assert torch.equal(out[0][M - 80:].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("M,N,K", [
    (1000, 3500, 768),   # 128 x 256; columns of Ct that are no whole lines
    (1001, 3500, 256),   # and no multiple of 16 bytes: stored by elements; two k-blocks
    (1002, 3333, 512),
    (1002, 3333, 1152),  # 128 x 256 on eight waves
    (1001, 3500, 1280),
    (1024, 3500, 1024),
    (999, 11008, 512),   # 256 x 256
    (2600, 6200, 384),   # 525 tiles of 128 x 256: more than 320 and no multiple of eight are dealt to the XCDs in runs too
    (3300, 9970, 256),   # 507 of 256 x 256
    (1100, 2490, 384),   # 351 of 128 x 64, register-staged
    (131, 200, 384),     # register-staged
    (36, 130, 256),
])
@pytest.mark.parametrize("transposed", [True, False])
def test_int8_int4(cuda, M, N, K, transposed):
    gen = torch.Generator(device=cuda).manual_seed(M)
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


# a transposed column by blocks of 32 rows (up to 47 rows left in a wave's 64), one row short of that and one beyond it
@pytest.mark.parametrize("M", [1, 31, 33, 47, 49, 63, 65, 111, 113, 129])
def test_transposed_rows_off_16_bytes(cuda, M):
    N, K = 203, 256
    gen = torch.Generator(device=cuda).manual_seed(M)
    B = _ints(gen, 0, 255, N, K // 2, dtype=torch.uint8, device=cuda)
    stream = torch.cuda.current_stream().cuda_stream
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    C = torch.full((N + 1, M), -7, dtype=torch.int32, device=cuda)
    rc = _lib.get_library().call_gemm_int8xint4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 0, 0, 1, stream)
    assert rc == 0, _lib.last_error()
    assert torch.equal(C[:N], (_nibbles(B).double() @ A.double().t()).int()) and bool((C[N:] == -7).all())
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    C = torch.full((N + 1, M), float("nan"), dtype=torch.float16, device=cuda)
    rc = _lib.get_library().call_dequant_gemm_fp16_fp4(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, 1, stream)
    assert rc == 0, _lib.last_error()
    code = _nibbles(B).int()
    value = torch.exp2(((code >> 1) & 3).double() - 1) * (1 + (code & 1).double() / 2)  # bits (E + 14) << 10 | m << 9
    W = torch.where(code > 7, -value, value)
    assert torch.equal(C[:N], (W @ A.double().t()).half()) and bool(torch.isnan(C[N:]).all())


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("fragments", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (1300, 4000, 768), (1300, 4000, 512), (1281, 4072, 1280), (1300, 4000, 1536),  # four waves; eight on five stages, on six
    (1800, 7000, 1024), (1800, 7000, 1280),  # 224 tiles of 256 rows, 420 of 128: the second to K = 1024, the first beyond
    (1300, 7000, 768), (1300, 6000, 256), (2050, 7690, 512), (2050, 7690, 2304),  # 308, 264, 527 tiles: two workgroups per CU; rounds of four waves; of eight
    (1020, 8190, 768), (2041, 4090, 512), (1020, 8190, 1280), (2041, 4090, 1536), (2570, 8190, 512), (2570, 8190, 2304),  # tiles of 128 rows
])
def test_bitnet(cuda, M, N, K, fragments, interleaved):
    assert _on_128(_lib.OPERANDS_INT8_INT2, M, N, K)
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = _ints(gen, -128, 127, M, K, dtype=torch.int8, device=cuda)
    codes = _ints(gen, 1, 3, N, K // 16, 4, 4, dtype=torch.uint8, device=cuda)  # element e of a word at bit 8 (e % 4) + 2 (e / 4)
    if interleaved:
        packed = sum(codes[:, :, j] << (2 * j) for j in range(4))
    else:  # code e of a word at bit 2 e
        packed = sum(codes[:, :, :, j] << (2 * j) for j in range(4))
    packed = packed.reshape(N, K // 4).view(torch.int8)
    s_a = torch.exp2(_ints(gen, -1, 2, M, dtype=torch.float32, device=cuda))
    B = quantize.prepack_i2_fragments(packed) if fragments else packed
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    layout = int(interleaved) | (2 if fragments else 0)
    rc = _lib.get_library().call_gemm_int8xint2(A.data_ptr(), B.data_ptr(), out.data_ptr(), M, N, K, 1, layout, s_a.data_ptr(), 4.0,
                                                1, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    W = codes.reshape(N, K).double() - 2
    ref = (A.double() @ W.t()) / s_a.double()[:, None] / 4.0
    assert torch.equal(out, ref.half())
