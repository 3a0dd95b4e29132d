"""The library's choice between its kernels, asked of the host code: no GPU.  Where two kernels were timed against each other,
the shapes are some of those measured, with the times that decided (us)."""

import random

import pytest

import tilelang_amd as tl
from tilelang_amd import _lib

UINT4, MXFP4, INT4, INT2, FP4 = _lib.OPERANDS_F16_UINT4, _lib.OPERANDS_BF16_MXFP4, _lib.OPERANDS_INT8_INT4, _lib.OPERANDS_INT8_INT2, _lib.OPERANDS_FP4
SCALE, ZEROS = 3, 5


def form(operands, M, N, K, group=0, mode=0, room=1):
    return _lib.load_library().dq_kwaves_form(operands, M, N, K, group, mode, room)


@pytest.mark.parametrize("operands", [MXFP4, INT4, INT2, UINT4])
def test_a_launch_that_fills_the_chip_is_counted_as_it_runs(operands):
    """Two passes of 32 rows over 8192 weight rows, 64 each, are 256 workgroups, one per CU.  Counted as more, they came after
    one pass of 64 rows, on half of the CUs."""
    assert form(operands, 64, 8192, 8192 if operands == MXFP4 else 4096 + 128, 128, SCALE) == 2


@pytest.mark.parametrize("M,N,K,register_resident,over_waves", [
    (29, 1184, 8192, 9.6, 13.6), (32, 720, 5888, 8.1, 11.6), (56, 632, 4096, 6.0, 8.6), (4, 16384, 2048, 7.3, 8.6),
    (8, 13632, 2048, 9.2, 10.2), (95, 312, 1728, 4.2, 5.2), (77, 448, 5056, 10.4, 12.8),
    (64, 8192, 8192, 49, 20), (14, 2168, 13760, 22, 14), (23, 8376, 2816, 14.5, 9.9), (101, 4336, 4800, 39, 17),
    (106, 14536, 2048, 18.7, 14.3), (404, 3592, 3072, 23.0, 18.1), (202, 6272, 3072, 20.7, 16.9),  # K shared out evenly
])
def test_mxfp4_against_its_neighbours(M, N, K, register_resident, over_waves):
    assert (form(MXFP4, M, N, K) >= 0) == (over_waves < register_resident)


@pytest.mark.parametrize("M,N,K,neighbour,over_waves", [
    (27, 20384, 3840, 10.3, 13.2), (18, 17864, 1792, 7.2, 8.7), (37, 3560, 2048, 5.0, 5.8),   # register-resident
    (322, 4872, 256, 6.9, 10.4), (1251, 2160, 128, 6.0, 12.4), (70, 21400, 256, 8.3, 10.0), (483, 3800, 256, 6.9, 10.4),  # tiles
    (20, 3000, 3200, 17, 7.7), (39, 6544, 12288, 39.7, 14.6), (33, 20592, 3328, 22.3, 14.0), (196, 3960, 1280, 9.5, 7.5),
    (117, 2592, 2048, 6.7, 5.3), (350, 2872, 2048, 11.1, 8.9), (332, 5400, 6144, 34.8, 21.6), (97, 15752, 6528, 32.8, 24.0),  # K shared out evenly
    (1099, 2168, 11776, 67, 49), (1104, 2552, 7680, 43, 36), (3038, 176, 16384, 30, 55), (2876, 184, 16384, 30, 53),  # activations that no L2 holds
])
def test_int8_int2_against_its_neighbours(M, N, K, neighbour, over_waves):
    assert (form(INT2, M, N, K) >= 0) == (over_waves < neighbour)


@pytest.mark.parametrize("M,N,K,tiles,over_waves", [
    (35, 14608, 256, 5.0, 5.8), (34, 10472, 256, 4.8, 5.5), (48, 11960, 256, 4.7, 5.4), (46, 9352, 384, 5.7, 5.9),
    (64, 8192, 8192, 27, 13), (41, 11736, 640, 6.7, 6.3), (22, 13640, 256, 4.6, 4.5), (128, 8192, 8192, 28, 19),
])
def test_int8_int4_against_the_tiles(M, N, K, tiles, over_waves):
    assert (form(INT4, M, N, K) >= 0) == (over_waves < tiles)



def test_activations_that_no_l2_holds_are_read_by_sets_of_64_weight_rows():
    """50 us on sets of 32 (form 1), which read them five times an XCD, and 32 on sets of 64."""
    assert form(INT2, 776, 1136, 13056) == 4 and form(INT2, 776, 1136, 2304 + 128) != 4


def tile_rows(operands, M, N, K, group=0, mode=0):
    return _lib.load_library().dq_tile_rows(operands, M, N, K, group, mode)


@pytest.mark.parametrize("operands,M,N,K,staged,direct", [
    (INT4, 273, 8087, 640, 11.7, 15.3), (INT4, 1088, 2631, 1152, 15.7, 18.9), (INT4, 385, 6825, 1408, 17.1, 20.4),
    (FP4, 409, 5890, 320, 9.7, 11.7), (FP4, 3446, 810, 320, 12.2, 14.2), (MXFP4, 110, 24823, 320, 12.1, 16.0),
    (INT2, 317, 17954, 640, 21.4, 26.8), (INT2, 2236, 2645, 640, 21.8, 26.3), (INT2, 254, 25530, 896, 24.8, 28.5),
])
def test_an_odd_count_of_k_blocks_stays_register_staged(operands, M, N, K, staged, direct):
    assert staged < direct and tile_rows(operands, M, N, K) == 0
    # an even count is the direct-to-LDS kernel's, and so is a long K
    assert tile_rows(operands, M, N, K + (64 if operands in (MXFP4, FP4) else 128)) and tile_rows(operands, M, N, 4224)


@pytest.mark.parametrize("M,N,K", [(461, 25216, 3072), (860, 20736, 3072), (201, 17152, 4864), (213, 17856, 2304)])
def test_uint4_groups_of_32_with_zeros_are_not_on_tiles_of_96_rows(M, N, K):
    """104 us on tiles of 128 rows and 152 on 96 (the first), 149 and 213, 74 and 88, 37 and 44."""
    assert tile_rows(UINT4, M, N, K, 32, ZEROS) in (128, 192)


def test_a_call_that_brings_no_room_runs_as_with_it():
    """Over the range of the layers: where K goes over the waves of a workgroup with room, it does so without."""
    rng, seen = random.Random(0), 0
    for _ in range(4000):
        M, N, K = rng.randint(2, 400), rng.randint(64, 3600) * 8, rng.randint(2, 100) * 128
        group, mode = rng.choice(((128, SCALE), (128, ZEROS), (64, ZEROS), (1024, SCALE), (128, 0)))
        if K % group == 0 and form(UINT4, M, N, K, group, mode, 1) >= 0:
            seen += 1
            assert form(UINT4, M, N, K, group, mode, 0) >= 0, (M, N, K, group, mode)
    assert seen > 300


def _room(kernel):
    return [p.shape[0] for p in kernel.params if p.name == "Workspace"]


@pytest.mark.parametrize("M,N,K,over_waves", [(58, 2528, 3840, True), (90, 2528, 4096, True), (16, 4096, 14336, False), (202, 8928, 10752, False)])
def test_uint4_kernel_objects_bring_room_only_where_sums_are_written(M, N, K, over_waves):
    lib = _lib.load_library()
    asked = lib.dq_w4a16_workspace_bytes(M, N, K, 128, SCALE)
    room = _room(tl.dequantize_gemv(M, N, K, group_size=128, source_format="int", with_scaling=True))
    assert asked and room == ([] if over_waves else [asked]) and (form(UINT4, M, N, K, 128, SCALE) >= 0) == over_waves


@pytest.mark.parametrize("M,N,K,over_waves", [(101, 1696, 3456, True), (204, 2912, 3328, True), (96, 8192, 8192, False), (600, 4096, 8192, False)])
def test_mxfp4_kernel_objects_bring_sums_room_only_where_sums_are_written(M, N, K, over_waves):
    asked = _lib.load_library().dq_mxfp4_workspace_bytes(M, N, K)
    assert _room(tl.matmul_bf16_mxfp4(M, N, K)) == [16 if over_waves else asked] and (form(MXFP4, M, N, K) >= 0) == over_waves


@pytest.mark.parametrize("M,N,K", [(170, 15548, 2048), (546, 5024, 2176), (380, 8036, 2432)])
def test_simple_mxfp4_kernel_objects_keep_room_for_the_sums(M, N, K):
    """The "simple" format is cut here, which e2m1 is not: with less than two slices' room the call would run uncut."""
    asked = _lib.load_library().dq_mxfp4_workspace_bytes(M, N, K)
    assert form(MXFP4, M, N, K) >= 0 and _room(tl.matmul_bf16_mxfp4(M, N, K, weight_format="e2m1")) == [16]
    assert _room(tl.matmul_bf16_mxfp4(M, N, K, weight_format="simple")) == [asked] and asked >= 2 * 4 * M * N


@pytest.mark.parametrize("M,N,K,streamed,cut", [(93, 38384, 28160, 501, 679), (135, 16832, 25600, 367, 489), (138, 19706, 14080, 224, 287),
                                              (156, 10674, 18432, 104, 136), (146, 9408, 26880, 139, 166)])
def test_uint4_groups_of_32_are_cut_into_less_than_a_round(M, N, K, streamed, cut):
    room = _lib.load_library().dq_w4a16_workspace_bytes
    tiles = -(-M // 96) * -(-N // 256)
    assert streamed < cut and room(M, N, K, 32, ZEROS) // (4 * M * N) * tiles <= 192 < room(M, N, K, 128, ZEROS) // (4 * M * N) * tiles


@pytest.mark.parametrize("operands,M,N,K,tiles,over_waves", [
    (INT4, 3859, 256, 22272, 60, 98), (INT4, 4024, 256, 7168, 23, 35), (INT4, 2019, 592, 15616, 44, 64), (INT4, 1309, 752, 8960, 29, 42),
    (INT2, 3998, 512, 23040, 68, 111), (INT2, 4037, 192, 20992, 56, 88), (INT2, 1245, 601, 27136, 70, 108), (MXFP4, 2416, 448, 3072, 21, 26),
    (INT4, 847, 614, 6144, 22, 14), (INT2, 843, 413, 6912, 22, 12),
])
def test_many_rows_against_the_tiles(operands, M, N, K, tiles, over_waves):
    assert (form(operands, M, N, K) >= 0) == (over_waves < tiles)


@pytest.mark.parametrize("M,N,K,rows128,rows96", [(101, 31779, 256, 14.8, 18.5), (122, 32242, 512, 17.4, 20.1), (112, 32150, 896, 23.6, 27.1),
                                                 (122, 25464, 4928, 69.9, 58.6), (110, 25840, 2496, 35.7, 30.8), (126, 26648, 9280, 131, 117)])
def test_tiles_of_96_rows_in_place_of_half_as_many_of_128(M, N, K, rows128, rows96):
    assert tile_rows(MXFP4, M, N, K) == (128 if rows128 < rows96 else 96)
