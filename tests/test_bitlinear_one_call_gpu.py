"""call_bitlinear_fp16 (quantiser and GEMM in one call, at a decode batch in one kernel) against the two calls it stands for,
bit for bit, and the quantiser's rounding where its cheap form does not apply."""

import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import _lib, quantize
from tilelang_amd.bitlinear import activation_quant_reference

pytestmark = pytest.mark.gpu


def _activations(gen, M, K, cuda):
    x = torch.randn((M, K), generator=gen, device=cuda) * torch.rand((M, 1), generator=gen, device=cuda) * 20
    x = x.half()
    x[0, :16] = torch.tensor([0.5, -0.5, 1.5, 2.5, -2.5, 0.0, 1e-4, -1e-4] * 2, dtype=torch.float16, device=cuda)
    if M > 1:
        x[1] = 0  # the clamp of the largest magnitude decides the scale
    if M > 2:
        x[2] = torch.randint(-127, 128, (K,), generator=gen, device=cuda).half() / 2  # products half way between whole numbers
        x[2, 5] = 63.5
    return x


def _both(x, B, M, N, K, layout, cuda):
    lib, stream = _lib.get_library(), torch.cuda.current_stream().cuda_stream
    q, s = tl.bitnet_activation_quant(M, K)(x)
    two = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    assert lib.call_gemm_int8xint2(q.data_ptr(), B.data_ptr(), two.data_ptr(), M, N, K, 1, layout, s.data_ptr(), 3.0, 1, stream) == 0, _lib.last_error()
    room = int(lib.dq_bitlinear_workspace_bytes(M, N, K, layout))
    around = torch.full((room + 512,), 77, dtype=torch.uint8, device=cuda)
    one = torch.full((M, N), float("nan"), dtype=torch.float16, device=cuda)
    assert lib.call_bitlinear_fp16(x.data_ptr(), B.data_ptr(), one.data_ptr(), around[256:].data_ptr() if room else None, room, M, N, K,
                                   layout, 3.0, stream) == 0, _lib.last_error()
    assert bool((around[:256] == 77).all()) and bool((around[256 + room:] == 77).all())
    return q, s, two, one, room


@pytest.mark.parametrize("layout", [0, 1, 3])  # plain, interleaved, interleaved in the operand order
@pytest.mark.parametrize("M,N,K,one_kernel", [
    (1, 33, 256, True), (1, 4100, 4096, True), (1, 72, 16384, True), (1, 40, 32768, None),  # dot products
    (2, 4096, 2048, True), (2, 70, 16384, True), (2, 48, 18432, False),
    (3, 4099, 4096, True), (4, 136, 12288, True), (4, 16, 16384, True),                     # two pairs of rows resident
    (5, 1001, 256, True), (8, 8200, 4096, True), (7, 520, 10240, True), (8, 260, 11008, False),
    (9, 130, 2048, True), (16, 4112, 1792, True), (16, 128, 2304, False),
    (17, 300, 2048, False), (200, 512, 2048, False), (1, 130, 384, None), (3, 130, 384, False),
])
def test_one_call(cuda, M, N, K, one_kernel, layout):
    gen = torch.Generator(device=cuda).manual_seed(M * K + N)
    x = _activations(gen, M, K, cuda)
    B = torch.randint(-128, 128, (N, K // 4), generator=gen, device=cuda, dtype=torch.int8)
    if layout & 2:
        if M > 16 and K % 2048:
            pytest.skip("no kernel for this order")
        B = quantize.prepack_i2_fragments(B)
    lib = _lib.get_library()
    if (layout & 2) and K % 2048 and not lib.dq_bitlinear_workspace_bytes(M, N, K, layout) == 0:
        pytest.skip("no kernel for this order")
    q, s, two, one, room = _both(x, B, M, N, K, layout, cuda)
    assert torch.equal(one.view(torch.int16), two.view(torch.int16))
    if one_kernel is not None:
        assert (room == 0) == one_kernel
    rq, rs = activation_quant_reference(x.cpu())
    assert torch.equal(q.cpu(), rq) and torch.equal(s.cpu(), rs.reshape(-1))


@pytest.mark.parametrize("layout", [1, 3])
@pytest.mark.parametrize("M,K", [(1, 4096), (2, 4096), (4, 2048), (8, 4096), (16, 2048), (40, 2048)])
def test_infinities_and_nan(cuda, M, K, layout):
    """A row with an infinity has a scale of zero, NaN is no largest magnitude, and NaN products go to -128: the same in every
    path, and the other rows untouched."""
    N = 264
    gen = torch.Generator(device=cuda).manual_seed(M)
    clean = _activations(gen, M, K, cuda)
    B = torch.randint(-128, 128, (N, K // 4), generator=gen, device=cuda, dtype=torch.int8)
    if layout & 2:
        B = quantize.prepack_i2_fragments(B)
    for value in (float("inf"), float("-inf"), float("nan")):
        x = clean.clone()
        x[M // 2, K - 3] = value
        q, s, two, one, _ = _both(x, B, M, N, K, layout, cuda)
        # 0 / 0 of a zero scale: NaN on both sides
        assert torch.equal(torch.isnan(one), torch.isnan(two)) and torch.equal(one.nan_to_num(), two.nan_to_num())
        row = x[M // 2].float()
        amax = row.nan_to_num(nan=0.0, posinf=float("inf"), neginf=float("-inf")).abs().max().clamp(min=1e-5)
        scale = amax.reciprocal() * 127
        want = (row * scale).round().nan_to_num(nan=-128.0).clamp(-128, 127).to(torch.int8)
        assert torch.equal(q[M // 2], want) and float(s[M // 2]) == float(scale)
        for m in range(M):
            if m != M // 2:
                cq, cs = activation_quant_reference(clean[m:m + 1].cpu())
                assert torch.equal(q[m].cpu(), cq[0]) and float(s[m]) == float(cs)


def test_refusals(cuda):
    lib = _lib.get_library()
    M, N, K = 40, 64, 2048
    x = torch.zeros((M, K), dtype=torch.float16, device=cuda)
    B = torch.zeros((N, K // 4), dtype=torch.int8, device=cuda)
    C = torch.zeros((M, N), dtype=torch.float16, device=cuda)
    room = int(lib.dq_bitlinear_workspace_bytes(M, N, K, 1))
    ws = torch.zeros(room + 16, dtype=torch.uint8, device=cuda)
    assert room >= M * K + 4 * M and lib.dq_bitlinear_workspace_bytes(0, N, K, 1) == 0
    for workspace, size, layout, s_w, message in (
            (None, 0, 1, 1.0, "non-NULL"), (ws.data_ptr(), room - 1, 1, 1.0, "bytes"), (ws.data_ptr() + 8, room, 1, 1.0, "16-byte aligned"),
            (ws.data_ptr(), room, 1, 0.0, "s_w"), (ws.data_ptr(), room, 8, 1.0, "layout")):
        rc = lib.call_bitlinear_fp16(x.data_ptr(), B.data_ptr(), C.data_ptr(), workspace, size, M, N, K, layout, s_w, 0)
        assert rc == -1 and message in _lib.last_error()
