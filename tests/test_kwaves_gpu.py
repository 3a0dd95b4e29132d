"""K over the waves of a workgroup (dq_gemm_kwaves.h) at the edges of its walk: fewer chunks of K than waves, a chunk in part,
rows of scales that are no multiple of a window, ragged rows and columns, each of its forms, which every case names (0 .. 4: 16, 32,
32, 48, 64 rows by 32, 32, 64, 64, 64 columns).  Operands are small integers and powers of two, so that every product and every
fp32 sum is exact and the result is one rounding of the float64 product."""

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


def _form(operands, M, N, K, group=0, mode=0):
    return _lib.load_library().dq_kwaves_form(operands, M, N, K, group, mode, 1)


@pytest.mark.parametrize("transposed", [True, False])
@pytest.mark.parametrize("decode", [0, 1])
@pytest.mark.parametrize("M,N,K,form", [
    (2, 2264, 1024, 0), (3, 33, 128, 0), (5, 97, 384, 0), (16, 300, 2176, 0),  # one to nine chunks of 256 k
    (17, 130, 256, 1), (31, 1001, 1920, 1), (32, 8200, 640, 2),
    (33, 9000, 896, 3), (48, 16400, 768, 3), (64, 20003, 512, 2), (61, 24700, 640, 4), (63, 12920, 1152, 4),
    (65, 500, 2048, 1), (129, 300, 1152, 1), (200, 3001, 2304, 3), (121, 6920, 1152, 4), (222, 1728, 384, 2),  # passes
])
def test_int8_int4(cuda, M, N, K, form, decode, transposed):
    assert transposed is False and M <= 4 or _form(_lib.OPERANDS_INT8_INT4, M, N, K) == form  # (row-major, to 4 rows: dot products)
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


@pytest.mark.parametrize("M,N,K,form", [
    (3, 2100, 13824, 0), (14, 2168, 6720, 0), (7, 5159, 512, 0), (7, 5159, 576, 0), (34, 18690, 512, 2),  # the least K; a chunk in part
    (32, 8200, 2880, 2), (33, 9000, 1088, 3), (48, 16400, 768, 3), (64, 20003, 832, 2), (64, 3000, 2112, 1), (62, 8421, 1280, 4),
    (101, 2000, 4800, 1), (254, 1030, 1344, 2), (159, 4619, 1088, 4),    # passes (K % 128 == 64)
    (81, 2004, 1024, 1), (95, 2760, 2304, 2), (327, 1036, 1792, 1), (204, 2912, 3328, 3),  # in place of the cut over workgroups
])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
def test_mxfp4(cuda, fmt, with_bias, M, N, K, form):
    assert _form(_lib.OPERANDS_BF16_MXFP4, M, N, K) == form
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
    M, N, K = 60, 2999, 832
    assert _form(_lib.OPERANDS_BF16_MXFP4, M, N, K) >= 0
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


# W4A16: w of the codes, the scales and the zero points, by mode (enum dq_w4_mode)
UINT4_MODES = {
    0: lambda q, s, z: q, 1: lambda q, s, z: torch.where(q > 7, q - 16, q), 2: lambda q, s, z: q - 8,
    3: lambda q, s, z: (q - 8) * s, 4: lambda q, s, z: q * s, 5: lambda q, s, z: (q - z) * s, 6: lambda q, s, z: q * s - z,
    7: lambda q, s, z: (q - z) * s,
}


def _uint4(cuda, M, N, K, group, mode, layout, variant):
    """(C, the float64 product rounded): an exact result whatever the order of the sums."""
    gen = torch.Generator(device=cuda).manual_seed(K + group)
    A = _ints(gen, -2, 2, M, K, dtype=torch.float16, device=cuda)
    codes = _ints(gen, 0, 15, N, K // 8, 8, dtype=torch.int32, device=cuda)
    # element e of a 32-bit word: nibble e, or interleaved nibble e / 2 of half e % 2
    places = [4 * (e // 2) + 16 * (e % 2) for e in range(8)] if layout else [4 * e for e in range(8)]
    B = sum(codes[..., e].long() << places[e] for e in range(8)).to(torch.int32).view(torch.int8).reshape(N, K // 2).contiguous()
    S = torch.exp2(_ints(gen, -3, 0, N, K // group, dtype=torch.float16, device=cuda))
    Z = _ints(gen, 5, 11, N, K // group, dtype=torch.float16, device=cuda)
    C = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=cuda)
    rc = _lib.get_library().call_dequantize_gemv_w4a16(A.data_ptr(), B.data_ptr(), S.data_ptr() if mode >= 3 else None,
                                                       Z.data_ptr() if mode >= 5 else None, C.data_ptr(), M, N, K, group, mode, layout,
                                                       variant, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    assert bool(torch.isnan(C[M]).all())
    grow = [t.double().repeat_interleave(group, dim=1) for t in (S, Z)]
    return C[:M], (A.double() @ UINT4_MODES[mode](codes.reshape(N, K).double(), *grow).t()).half()


@pytest.mark.parametrize("form", range(5))
@pytest.mark.parametrize("M,N,K,group", [
    (3, 130, 1152, 128), (8, 1001, 3968, 64), (16, 515, 640, 64),        # nine groups: a window and one
    (24, 671, 1408, 128), (33, 900, 1152, 128), (48, 1640, 896, 64), (65, 2003, 1152, 128),
    (58, 2528, 3840, 128), (13, 622, 7424, 128), (9, 130, 2048, 256),    # K % 256 == 0
    (20, 300, 2176, 32), (40, 97, 256, 32),                              # a window a chunk
    (17, 75, 8192, 1024), (5, 33, 32768, 4096),                          # one of many
    (200, 300, 1920, 128),                                               # passes
])
def test_uint4_forms(cuda, M, N, K, group, form):
    for mode in (3, 5):
        got, ref = _uint4(cuda, M, N, K, group, mode, 0, 80 + form)
        assert torch.equal(got, ref)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("mode", sorted(UINT4_MODES))
def test_uint4_modes(cuda, mode, layout):
    for form in (0, 3):
        got, ref = _uint4(cuda, 50, 201, 1152, 128, mode, layout, 80 + form)
        assert torch.equal(got, ref)


@pytest.mark.parametrize("M,N,K,group,form", [
    (8, 1001, 3968, 64, 0), (3, 130, 8320, 64, 0), (24, 6712, 1408, 128, 1), (48, 16400, 896, 64, 3), (64, 20003, 1152, 128, 4),
    (88, 700, 3712, 64, 1), (200, 300, 1920, 128, 1), (58, 2528, 3840, 128, 1), (7, 6952, 2816, 128, 0), (20, 300, 2176, 32, 1),
    (3, 130, 1152, 128, -1), (20, 300, 640, 128, -1),                    # dot products; less than a window of groups
])
def test_uint4_by_choice(cuda, M, N, K, group, form):
    assert _form(_lib.OPERANDS_F16_UINT4, M, N, K, group, 5) == form
    got, ref = _uint4(cuda, M, N, K, group, 5, 0, -1)
    assert torch.equal(got, ref)


def test_uint4_form_refused(cuda):
    """Less than a window of groups, one group per row."""
    for K, group in ((640, 128), (1152, 1152)):
        with pytest.raises(AssertionError, match="K over the waves does not cover"):
            _uint4(cuda, 20, 300, K, group, 3, 0, 80)


@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("convention", [0, 1, 2])
@pytest.mark.parametrize("M,N,K,form", [
    (5, 130, 384, 0), (16, 1001, 2688, 0), (9, 3248, 640, 0),            # K % 256 == 128, a chunk of 512 k in part
    (17, 300, 256, 1), (33, 9000, 768, 3), (48, 16400, 512, 2), (64, 20000, 1280, 2), (28, 21660, 1152, 2),
    (145, 8296, 1024, 2), (200, 700, 2560, 1), (130, 515, 1152, 1), (93, 7271, 1280, 3), (192, 8715, 1280, 4),
])
def test_int8_int2(cuda, M, N, K, form, convention, interleaved):
    assert _form(_lib.OPERANDS_INT8_INT2, M, N, K) == form
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
