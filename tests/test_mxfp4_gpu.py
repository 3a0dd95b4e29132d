"""GPU parity of the MXFP4 x bf16 GEMM (through the C-ABI) against the CPU oracle.

bf16 outputs within rtol=1e-2, atol=1e-2 of ``A.float() @ (decode(B) * 2**(Scale - bias)).float().T -> bf16``
(the dequantised operand is exact in bf16, the only rounding is the fp32 accumulation and the final cast).
"""

import numpy as np
import pytest
import torch

import tilelang_amd as tl
from tilelang_amd import workloads
from oracle import dq_oracle as orc

pytestmark = pytest.mark.gpu
RTOL = ATOL = 1e-2


def _dev(x, cuda):
    return torch.from_numpy(np.ascontiguousarray(x)).to(cuda)


def _check(cuda, M, N, K, fmt, scale_bias, seed=0, with_bias=False, exp_range=(-8, 0)):
    d = workloads.mxfp4(M, N, K, seed=seed, scale_exp_range=exp_range, scale_bias=scale_bias)
    B = d["B"]
    if fmt == "twiddling":
        B = orc.twiddle_pack_fp4(orc.unpack_u4(B))
    kern = tl.matmul_bf16_mxfp4(M, N, K, weight_format=fmt, scale_bias=scale_bias, with_bias=with_bias)
    A = _dev(d["A"], cuda).view(torch.bfloat16)
    rng = np.random.default_rng(seed + 1)
    bias_bits = orc.f32_to_bf16_bits(rng.standard_normal((M, N), dtype=np.float32) * 4)
    Bias = _dev(bias_bits, cuda).view(torch.bfloat16)
    C = kern(A, _dev(B, cuda), _dev(d["Scale"], cuda), Bias)
    torch.cuda.synchronize()
    ref_bits = orc.ref_mxfp4(d["A"], B, d["Scale"], bias_bits if with_bias else None, fmt=fmt, scale_bias=scale_bias)
    ref = orc.bf16_bits_to_f32(ref_bits)
    got = C.float().cpu().numpy()
    assert got.shape == (M, N) and np.isfinite(got).all()
    np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL)
    return got


@pytest.mark.parametrize("fmt", ["e2m1", "twiddling", "simple"])
@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (64, 64, 64), (128, 512, 128)])
def test_reference_test_shapes(cuda, fmt, M, N, K):
    """Shapes of testing/python/amd/test_tilelang_mxfp4_gfx950.py:111-222, but over all 16 codes
    and, like the reference programs, the raw unbiased exponent (2**Scale, Scale in 0..2)."""
    _check(cuda, M, N, K, fmt, scale_bias=0, exp_range=(0, 2))


@pytest.mark.parametrize("fmt", ["e2m1", "twiddling", "simple"])
def test_e8m0_scales(cuda, fmt):
    _check(cuda, 512, 768, 512, fmt, scale_bias=127)


@pytest.mark.parametrize("M,N,K", [(1, 256, 64), (100, 300, 192), (257, 255, 128), (300, 520, 320)])
def test_ragged_shapes(cuda, M, N, K):
    _check(cuda, M, N, K, "e2m1", scale_bias=127)


@pytest.mark.parametrize("fmt", ["e2m1", "twiddling", "simple"])
@pytest.mark.parametrize("with_bias", [False, True])
def test_many_tiles(cuda, fmt, with_bias):
    """Enough 256 x 256 tiles for the direct-to-LDS kernel (ragged edges, K of 2 and of 5 tiles), and the
    128 x 128 tile choice below it."""
    _check(cuda, 3581, 3589, 128, fmt, scale_bias=127, with_bias=with_bias)
    _check(cuda, 3584, 3584, 320, fmt, scale_bias=0, with_bias=with_bias, exp_range=(0, 4))
    _check(cuda, 1500, 2000, 192, fmt, scale_bias=127, with_bias=with_bias)
    # too few 256 x 256 tiles, 96 of 128 x 256: the direct-to-LDS kernel on its half-height tile (ragged both ways)
    _check(cuda, 1500, 2000, 256, fmt, scale_bias=127, with_bias=with_bias)
    _check(cuda, 1025, 3000, 384, fmt, scale_bias=127, with_bias=with_bias)
    if not with_bias:  # direct-to-LDS kernel with 4, 6 and 10 K tiles: prologue pair, steady pairs, tail
        for K in (256, 384, 640):
            _check(cuda, 3584, 3600, K, fmt, scale_bias=127)


@pytest.mark.parametrize("fmt", ["e2m1", "twiddling", "simple"])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 256, 128), (5, 300, 1024), (16, 1001, 2048), (8, 4100, 2176), (3, 64, 8192),
                                   (16, 9000, 5120), (17, 515, 1280), (40, 130, 4096), (64, 8200, 768), (12, 33, 6144),
                                   # K % 128 == 64: the last chunk of 128 k is half empty (2880: a hidden size in use)
                                   (4, 300, 2880), (16, 5763, 2880), (8, 100, 192), (20, 513, 4160), (3, 2880, 64),
                                   # K beyond 8192: slices of at most 6144 k, running sums in LDS between them
                                   (8, 300, 14336), (16, 4500, 8320), (5, 130, 28672), (24, 64, 12288),
                                   # K % 256 == 0: whole pairs of chunks per wave, runs of unequal length (7168 = 28 pairs, 256 = 1)
                                   (9, 700, 7168), (16, 130, 256), (2, 48, 3584),
                                   # one row up to K = 8192: the dot-product kernel (whole rows per wave, lanes beyond a row's end idle)
                                   (1, 300, 1024), (1, 1001, 2880), (1, 4100, 8192), (1, 513, 5120), (1, 5, 64), (1, 9000, 7168), (1, 31, 4160),
                                   # two rows: the same with the activations in LDS
                                   (2, 4100, 8192), (2, 1001, 5120), (2, 515, 1024), (2, 9000, 7168), (2, 7, 64),
                                   # one and two rows beyond K = 8192: chunks of four steps, activations padded to whole chunks in LDS
                                   (1, 300, 14336), (2, 1001, 16384), (1, 64, 28672), (2, 130, 8320), (1, 4100, 12288), (2, 33, 32768),
                                   (1, 40, 40960)])
def test_decode_batches(cuda, fmt, with_bias, M, N, K):
    """Decode batches with K a multiple of 64 (of 128 beyond 8192): the kernel that keeps the activations in registers
    and streams weights and scale bytes once per 16 rows.  Ragged N (last block of 16 weight rows, N % 4 != 0), K slices of unequal
    length over the eight waves (2176 = 17 chunks, 1280 = 10, 128 = 1), the eight-chunk form with parked activations
    (8192), passes of 16 rows (17, 40, 64), every format, with and without bias."""
    _check(cuda, M, N, K, fmt, scale_bias=127, seed=M + K, with_bias=with_bias)


def test_decode_batch_full_size_and_deterministic(cuda):
    """N = K = 8192 at 16 rows against the oracle, twice: the partial sums of the eight K slices are added in a
    fixed order."""
    a = _check(cuda, 16, 8192, 8192, "e2m1", scale_bias=127, seed=4)
    b = _check(cuda, 16, 8192, 8192, "e2m1", scale_bias=127, seed=4)
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("fmt", ["e2m1", "simple"])
def test_bias(cuda, fmt):
    _check(cuda, 384, 512, 256, fmt, scale_bias=127, with_bias=True)


def test_weight_values_exact(cuda):
    """A = identity picks single weights: C[i, n] must equal decode(B)[n, i] * 2**e exactly (bf16)."""
    N, K = 512, 256
    for fmt in ("e2m1", "twiddling", "simple"):
        d = workloads.mxfp4(K, N, K, seed=7, scale_bias=127)
        B = d["B"]
        # every byte value appears
        B[0, :] = np.arange(K // 2, dtype=np.uint8)
        B[1, :] = np.arange(K // 2, dtype=np.uint8)[::-1] + 128
        Bp = orc.twiddle_pack_fp4(orc.unpack_u4(B)) if fmt == "twiddling" else B
        eye = orc.f32_to_bf16_bits(np.eye(K, dtype=np.float32))
        kern = tl.matmul_bf16_mxfp4(K, N, K, weight_format=fmt, scale_bias=127)
        C = kern(_dev(eye, cuda).view(torch.bfloat16), _dev(Bp, cuda), _dev(d["Scale"], cuda),
                 torch.empty((K, N), dtype=torch.bfloat16, device=cuda))
        torch.cuda.synchronize()
        W = orc.mxfp4_dequant(Bp, d["Scale"], fmt, 32, 127)  # [N, K] float32, exact
        got = C.float().cpu().numpy()
        np.testing.assert_array_equal(got, W.T + np.float32(0.0))


def test_full_size_properties(cuda):
    """Benchmark configuration 4 (M=4096, N=K=8192), checked without a full CPU matmul: a sample of
    rows and columns against the oracle, and linearity in A."""
    M, N, K = 4096, 8192, 8192
    d = workloads.mxfp4(M, N, K, seed=0, scale_bias=127)
    kern = tl.matmul_bf16_mxfp4(M, N, K, weight_format="e2m1", scale_bias=127)
    A = _dev(d["A"], cuda).view(torch.bfloat16)
    B, S = _dev(d["B"], cuda), _dev(d["Scale"], cuda)
    bias = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
    C = kern(A, B, S, bias)
    torch.cuda.synchronize()
    rng = np.random.default_rng(1)
    rows = rng.choice(M, 48, replace=False)
    cols = rng.choice(N, 64, replace=False)
    Af = orc.bf16_bits_to_f32(d["A"][rows])
    W = orc.mxfp4_dequant(d["B"][cols], d["Scale"][cols], "e2m1", 32, 127)
    ref = orc.bf16_bits_to_f32(orc.f32_to_bf16_bits(Af @ W.T))
    got = C[torch.from_numpy(rows).to(cuda)][:, torch.from_numpy(cols).to(cuda)].float().cpu().numpy()
    np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL)
    # whole-matrix check against a row sample: rows of C computed by an independent call on A[rows] (80 rows: the tiled
    # kernel again, whose sums do not depend on where in the matrix a row lies; up to 64 rows the decode kernel would
    # take the call and add the same products in another order)
    rows = rng.choice(M, 80, replace=False)
    kern_small = tl.matmul_bf16_mxfp4(len(rows), N, K, weight_format="e2m1", scale_bias=127)
    C_rows = kern_small(A[torch.from_numpy(rows).to(cuda)].contiguous(), B, S, bias[: len(rows)].contiguous())
    torch.cuda.synchronize()
    assert torch.equal(C_rows, C[torch.from_numpy(rows).to(cuda)])
    # and the decode kernel on 16 of those rows: within rounding of the same values
    kern_dec = tl.matmul_bf16_mxfp4(16, N, K, weight_format="e2m1", scale_bias=127)
    C_dec = kern_dec(A[torch.from_numpy(rows[:16]).to(cuda)].contiguous(), B, S, bias[:16].contiguous())
    torch.cuda.synchronize()
    np.testing.assert_allclose(C_dec.float().cpu().numpy(), C_rows[:16].float().cpu().numpy(), rtol=RTOL, atol=ATOL)
    # linearity: C(2A) == 2 C(A) exactly (power-of-two scaling commutes with every rounding)
    C2 = kern((A.float() * 2).to(torch.bfloat16), B, S, bias)
    torch.cuda.synchronize()
    assert torch.equal(C2.float(), C.float() * 2)


# ---- bf16 x fp4 without block scales (the example with kernel(A, qB)) ------------------------------------------------

@pytest.mark.parametrize("fast_dequant", [True, False])
@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (100, 300, 192), (512, 1024, 2048), (1500, 2000, 256)])
def test_unscaled_bf16_fp4(cuda, fast_dequant, M, N, K):
    """examples/dequantize_gemm/example_dequant_gemm_bf16_fp4_hopper.py: main(256, 256, 256, fast_dequant) against
    ref_program_twiddling / ref_program_simple, here the oracle's restatement of them (block exponent 0)."""
    fmt = "twiddling" if fast_dequant else "simple"
    d = workloads.mxfp4(M, N, K, seed=11, scale_exp_range=(0, 0), scale_bias=0)
    B = orc.twiddle_pack_fp4(orc.unpack_u4(d["B"])) if fast_dequant else d["B"]
    kern = tl.matmul_bf16_fp4(M, N, K, "bfloat16", "bfloat16", "float32", num_bits=4, fast_dequant=fast_dequant,
                              block_M=256, block_N=128, block_K=128, num_stages=2, threads=256, split=1)
    C = kern(_dev(d["A"], cuda).view(torch.bfloat16), _dev(B, cuda))
    torch.cuda.synchronize()
    zero_scale = np.zeros((N, K // 32), np.uint8)
    ref = orc.bf16_bits_to_f32(orc.ref_mxfp4(d["A"], B, zero_scale, None, fmt=fmt, scale_bias=0))
    got = C.float().cpu().numpy()
    assert got.shape == (M, N) and np.isfinite(got).all()
    np.testing.assert_allclose(got, ref, rtol=RTOL, atol=ATOL)


def test_unscaled_bf16_fp4_reads_back_the_reference_vectors(cuda):
    """A = identity makes the GEMM return the dequantised operand itself, exactly: against what the reference's own
    torch_convert_bit_twiddling (all 65 536 byte pairs) and torch_convert (all 256 bytes) produce
    (tests/golden/reference_vectors.npz, written by tests/golden/make_vectors.py)."""
    import os

    v = np.load(os.path.join(os.path.dirname(__file__), "golden", "reference_vectors.npz"))
    for fast, qB, want_bits in ((True, v["twiddling_in"], v["twiddling_out_bits"]), (False, v["convert_in"], v["convert_out_bits"])):
        N, K = qB.shape[0], qB.shape[1] * 2
        kern = tl.matmul_bf16_fp4(K, N, K, fast_dequant=fast)
        eye = torch.eye(K, dtype=torch.bfloat16, device=cuda)
        C = kern(eye, _dev(qB, cuda))
        torch.cuda.synchronize()
        got = C.float().cpu().numpy().T  # [N, K]
        np.testing.assert_array_equal(got, orc.bf16_bits_to_f32(want_bits))


def _cut_call(A, B, S, bias, C, ws, room, M, N, K, fmt, split):
    from tilelang_amd import _lib, kernels

    return _lib.get_library().call_dequant_gemm_bf16_mxfp4_ws(
        A.data_ptr(), B.data_ptr(), S.data_ptr(), None if bias is None else bias.data_ptr(), C.data_ptr(),
        None if ws is None else ws.data_ptr(), room, M, N, K, 32, kernels._FP4_FORMATS[fmt], 127, split,
        torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("fmt", ["e2m1", "twiddling", "simple"])
@pytest.mark.parametrize("M,N,K,split,with_bias,cut", [
    (17, 256, 256, 2, False, True),     # one unit of 128 k per slice: the pipeline's shortest walk
    (129, 260, 1152, 2, True, True),    # ragged edges, slices of four and five units
    (40, 1028, 1664, 12, True, True),   # slices of one and two units
    (8, 262, 512, 4, True, True),       # rows of the partial sums that start off 16 bytes: stored by elements
    (100, 1027, 1152, 3, True, True),   # and off 8 bytes: the sum kernel's quadruples straddle rows
    (300, 516, 384, 8, False, False),   # more slices asked for than units: the kernel is not cut
    (7, 262, 512, 4, True, False),      # M * N no multiple of four: not cut
    (257, 1284, 1024, 3, False, True),
])
def test_k_slices(cuda, fmt, M, N, K, split, with_bias, cut):
    """K cut over workgroups, through the C-ABI with the slice count named; and a workspace with room for one slice
    fewer.  Same tolerance as the uncut kernel: the fp32 sums are only grouped otherwise.  The workspace says whether the
    call was cut: its slices' sums, added in order with the bias and rounded once, are the result, and nothing around
    them is written; an uncut call writes none of it."""
    from tilelang_amd import _lib

    d = workloads.mxfp4(M, N, K, seed=3, scale_bias=127)
    B = orc.twiddle_pack_fp4(orc.unpack_u4(d["B"])) if fmt == "twiddling" else d["B"]
    bias_bits = orc.f32_to_bf16_bits(np.random.default_rng(4).standard_normal((M, N), dtype=np.float32) * 4)
    A, Bd, S = _dev(d["A"], cuda), _dev(B, cuda), _dev(d["Scale"], cuda)
    bias = _dev(bias_bits, cuda) if with_bias else None
    ref = orc.bf16_bits_to_f32(orc.ref_mxfp4(d["A"], B, d["Scale"], bias_bits if with_bias else None, fmt=fmt, scale_bias=127))
    guard = 1024
    for slices in (split, split - 1):
        room = slices * M * N * 4
        around = torch.full((guard + room + guard,), 255, dtype=torch.uint8, device=cuda)  # NaN wherever a sum were left out
        ws = around[guard:guard + room]
        C = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
        assert _cut_call(A, Bd, S, bias, C, ws, room, M, N, K, fmt, split) == 0, _lib.last_error()
        torch.cuda.synchronize()
        np.testing.assert_allclose(C.float().cpu().numpy(), ref, rtol=RTOL, atol=ATOL)
        assert bool((around[:guard] == 255).all()) and bool((around[guard + room:] == 255).all())
        if not cut or slices < 2:
            assert bool((ws == 255).all())
            continue
        parts = ws.view(torch.float32).view(slices, M, N)
        total = parts[0].clone()
        for z in range(1, slices):
            total += parts[z]
        if with_bias:
            total += bias.view(torch.bfloat16).float()
        assert bool(torch.isfinite(parts).all())
        assert torch.equal(total.to(torch.bfloat16).view(torch.int16), C.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(81, 4096, 4096), (96, 8192, 8192), (200, 4104, 4224), (100, 8190, 4096)])
def test_k_slices_by_default(cuda, M, N, K):
    """Shapes that the default cuts: through the kernel object, which brings the workspace."""
    assert any(p.name == "Workspace" for p in tl.matmul_bf16_mxfp4(M, N, K, weight_format="e2m1", scale_bias=127).params)
    _check(cuda, M, N, K, "e2m1", scale_bias=127, with_bias=True)


@pytest.mark.parametrize("M,N,K,cut", [(166, 5818, 3072, ("e2m1", "twiddling")), (256, 4096, 8192, ("e2m1", "twiddling", "simple"))])
def test_default_cut_by_format(cuda, M, N, K, cut):
    """The "simple" format, whose decoder is the longest, is cut where that is faster with it and not with the others."""
    from tilelang_amd import _lib

    room = int(_lib.load_library().dq_mxfp4_workspace_bytes(M, N, K))
    assert room
    d = workloads.mxfp4(M, N, K, seed=7, scale_bias=127)
    A, B, S = (_dev(d[k], cuda) for k in ("A", "B", "Scale"))
    C = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
    ws = torch.empty(room, dtype=torch.uint8, device=cuda)
    for fmt in ("e2m1", "twiddling", "simple"):
        ws.fill_(255)
        assert _cut_call(A, B, S, None, C, ws, room, M, N, K, fmt, 0) == 0, _lib.last_error()
        torch.cuda.synchronize()
        assert bool((ws == 255).all()) == (fmt not in cut)


def test_k_slice_workspace_through_c_abi(cuda):
    """The library's own choice with its full room, with less, with none: fewer slices and in the end the plain entry
    point's bits; what is refused."""
    from tilelang_amd import _lib

    lib = _lib.get_library()
    M, N, K = 200, 1028, 8192
    d = workloads.mxfp4(M, N, K, seed=6, scale_bias=127)
    A, B, S = (_dev(d[k], cuda) for k in ("A", "B", "Scale"))
    full = int(lib.dq_mxfp4_workspace_bytes(M, N, K))
    assert full >= 4 * M * N * 4
    ws = torch.empty(full + 16, dtype=torch.uint8, device=cuda)
    C = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
    plain = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
    rc = lib.call_dequant_gemm_bf16_mxfp4(A.data_ptr(), B.data_ptr(), S.data_ptr(), None, plain.data_ptr(), M, N, K, 32, 0, 127,
                                          torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    ref = orc.bf16_bits_to_f32(orc.ref_mxfp4(d["A"], d["B"], d["Scale"], None, fmt="e2m1", scale_bias=127))
    for room, slices in ((full, full // (M * N * 4)), (3 * M * N * 4 + 8, 3), (2 * M * N * 4, 2), (M * N * 4, 1), (8, 1), (0, 1)):
        ws.fill_(255)
        C.fill_(float("nan"))
        assert _cut_call(A, B, S, None, C, ws if room else None, room, M, N, K, "e2m1", 0) == 0, _lib.last_error()
        torch.cuda.synchronize()
        used = slices * M * N * 4 if slices > 1 else 0
        assert bool((ws[used:] == 255).all()) and bool(torch.isfinite(ws[:used].view(torch.float32)).all())
        np.testing.assert_allclose(C.float().cpu().numpy(), ref, rtol=RTOL, atol=ATOL)
        if slices == 1:
            assert torch.equal(C.view(torch.int16), plain.view(torch.int16))
    for workspace, room, split, message in ((None, full, 0, "Workspace is expected to have non-NULL data pointer"),
                                            (ws[4:], full, 0, "16-byte aligned"), (ws, full, -1, "split must be in 0..16"),
                                            (ws, full, 17, "split must be in 0..16")):
        assert _cut_call(A, B, S, None, C, workspace, room, M, N, K, "e2m1", split) == -1
        assert message in _lib.last_error()


@pytest.mark.parametrize("offset", [1, 2, 3])
@pytest.mark.parametrize("M,N,K,split", [
    (96, 4100, 1024, 2),   # would be cut
    (1500, 2000, 256, 0),  # 96 tiles of 128 x 256
    (4096, 3072, 128, 0),  # 192 tiles of 256 x 256
])
def test_scales_that_start_at_any_byte(cuda, M, N, K, split, offset):
    """Scale is bytes and need not start at a multiple of four: the kernels that fetch it by dwords leave such a call to
    the one that reads bytes, with the bits of the aligned, uncut call."""
    from tilelang_amd import _lib

    d = workloads.mxfp4(M, N, K, seed=5, scale_bias=127)
    A, B, S = (_dev(d[k], cuda) for k in ("A", "B", "Scale"))
    shifted = torch.zeros(S.numel() + 4, dtype=torch.uint8, device=cuda)[offset:offset + S.numel()]
    shifted.copy_(S.reshape(-1))
    ws = torch.full((2 * M * N * 4,), 255, dtype=torch.uint8, device=cuda)
    results = []
    for scale, slices in ((S, 1), (shifted, split)):
        C = torch.empty((M, N), dtype=torch.bfloat16, device=cuda)
        assert _cut_call(A, B, scale, None, C, ws, ws.numel(), M, N, K, "e2m1", slices) == 0, _lib.last_error()
        results.append(C)
    torch.cuda.synchronize()
    assert bool((ws == 255).all())  # neither call was cut
    assert torch.equal(results[0].view(torch.int16), results[1].view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(64, 20000, 1280), (30, 20000, 768), (254, 2176, 6336), (95, 6000, 2304)])
def test_one_slice_asked_for_keeps_the_bits_of_a_large_product(cuda, M, N, K):
    """split = 1: the rows of a call on the tiled GEMM have the bits that they have in a product of many rows, also where the
    library's choice would run K over the waves of a workgroup (real-valued operands, so that another order would show)."""
    from tilelang_amd import _lib

    assert _lib.load_library().dq_kwaves_form(1, M, N, K, 0, 0, 1) >= 0
    gen = torch.Generator(device=cuda).manual_seed(K)
    A = torch.randn((1100, K), generator=gen, device=cuda).bfloat16()
    B = torch.randint(0, 256, (N, K // 2), generator=gen, device=cuda).to(torch.uint8)
    S = torch.randint(119, 128, (N, K // 32), generator=gen, device=cuda).to(torch.uint8)
    out = []
    for rows in (1100, M):
        C = torch.empty((rows, N), dtype=torch.bfloat16, device=cuda)
        assert _cut_call(A, B, S, None, C, None, 0, rows, N, K, "e2m1", 1) == 0, _lib.last_error()
        out.append(C)
    assert torch.equal(out[0][:M].view(torch.int16), out[1].view(torch.int16))
