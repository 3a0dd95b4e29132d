"""W4A16 on the tiled GEMM with K cut over workgroups: slices of unequal length, one tile height and the other, the workspace
that the library asks for.  Operands are small integers and powers of two, so that every product and every fp32 sum is exact and
the result is one rounding of the float64 product, whatever the slices."""

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib

pytestmark = pytest.mark.gpu


def _operands(cuda, M, N, K, group, seed):
    gen = torch.Generator(device=cuda).manual_seed(seed)

    def ints(lo, hi, *shape, dtype):
        return torch.randint(lo, hi + 1, shape, generator=gen, device=cuda).to(dtype)

    A = ints(-2, 2, M, K, dtype=torch.float16)
    B = ints(-128, 127, N, K // 2, dtype=torch.int8)
    S = torch.exp2(ints(-4, -1, N, K // group, dtype=torch.float16))
    Z = ints(5, 11, N, K // group, dtype=torch.float16)
    b = B.view(torch.uint8)
    codes = torch.stack((b & 15, b >> 4), dim=-1).reshape(N, K).double()
    return A, B, S, Z, codes


def _ref(A, S, Z, codes, group, zeros):
    zero = Z.double().repeat_interleave(group, dim=1) if zeros else 8.0
    return (A.double() @ ((codes - zero) * S.double().repeat_interleave(group, dim=1)).t()).half()


@pytest.mark.parametrize("zeros", [True, False])
@pytest.mark.parametrize("M,N,K,group,split", [
    (65, 260, 512, 64, 2),        # 96 rows; two slices of 256 k: eight waves have too few stages
    (96, 1028, 2304, 64, 3),      # slices of 768 k
    (97, 516, 2560, 128, 4),      # 128 rows; slices of 512 and 768 k
    (190, 1000, 4096, 128, 5),    # two tiles of 96
    (257, 700, 3072, 256, 2),     # three of 96
    (129, 2052, 8192, 1024, 3),   # units of 2048 k
    (130, 258, 1024, 32, 4),      # a dword of scales per 64 k: four waves
    (200, 5, 1536, 128, 6),       # one column block in part
])
def test_named_slices(cuda, M, N, K, group, split, zeros):
    A, B, S, Z, codes = _operands(cuda, M, N, K, group, K + M)
    room = split * M * N * 4
    around = torch.full((256 + room + 256,), 255, dtype=torch.uint8, device=cuda)
    ws = around[256:256 + room]
    C = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=cuda)
    rc = _lib.get_library().call_dequantize_gemv_w4a16_ws(A.data_ptr(), B.data_ptr(), S.data_ptr(), Z.data_ptr() if zeros else None, C.data_ptr(),
                                                          ws.data_ptr(), room, M, N, K, group, 5 if zeros else 3, 0, 50 + split,
                                                          torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    assert torch.equal(C[:M], _ref(A, S, Z, codes, group, zeros)) and bool(torch.isnan(C[M]).all())
    assert bool((around[:256] == 255).all()) and bool((around[256 + room:] == 255).all())
    assert bool(torch.isfinite(ws.view(torch.float32)).all())


@pytest.mark.parametrize("M,N,K,group,zeros", [(200, 5004, 10752, 128, True), (700, 1648, 8960, 64, False), (90, 5528, 7936, 128, False)])
def test_default(cuda, M, N, K, group, zeros):
    """Shapes that the library cuts by itself, through the kernel object, which brings the workspace."""
    room = int(_lib.load_library().dq_w4a16_workspace_bytes(M, N, K, group, 5 if zeros else 3))
    assert room and room % (M * N * 4) == 0
    A, B, S, Z, codes = _operands(cuda, M, N, K, group, 7)
    kern = tl.dequantize_gemv(M, N, K, group_size=group, source_format="uint" if zeros else "int", with_scaling=True, with_zeros=zeros)
    assert [p.shape for p in kern.params if p.name == "Workspace"] == [(room,)]
    C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    kern(A, B, S, *([Z] if zeros else []), C)
    assert torch.equal(C, _ref(A, S, Z, codes, group, zeros))
    # and it is the tiled GEMM that is cut: the same bits as the slices named
    ws = torch.empty(room, dtype=torch.uint8, device=cuda)
    A = torch.randn(A.shape, device=cuda).half()
    out = []
    for variant in (-1, 50 + room // (M * N * 4)):
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        rc = _lib.get_library().call_dequantize_gemv_w4a16_ws(A.data_ptr(), B.data_ptr(), S.data_ptr(), Z.data_ptr() if zeros else None, C.data_ptr(),
                                                              ws.data_ptr(), room, M, N, K, group, 5 if zeros else 3, 0, variant,
                                                              torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _lib.last_error()
        out.append(C)
    assert torch.equal(out[0], out[1])


def test_less_room_than_asked_for(cuda):
    """A smaller workspace lowers the count, none at all leaves the call uncut."""
    M, N, K, group = 90, 5528, 7936, 128
    lib = _lib.get_library()
    full = int(lib.dq_w4a16_workspace_bytes(M, N, K, group, 3))
    assert full >= 3 * M * N * 4
    A, B, S, Z, codes = _operands(cuda, M, N, K, group, 9)
    ref = _ref(A, S, Z, codes, group, False)
    ws = torch.empty(full, dtype=torch.uint8, device=cuda)
    for room, used in ((full, full), (2 * M * N * 4 + 16, 2 * M * N * 4), (16, None), (0, None)):
        ws.fill_(255)
        C = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
        rc = lib.call_dequantize_gemv_w4a16_ws(A.data_ptr(), B.data_ptr(), S.data_ptr(), None, C.data_ptr(), ws.data_ptr() if room else None, room,
                                               M, N, K, group, 3, 0, -1, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _lib.last_error()
        assert torch.equal(C, ref)
        assert bool((ws[used or 0:] == 255).all())
