"""Error behaviour of the C ABI (include/mllm_hip_qlinear.h): null pointers, unknown enums, shapes the kernels do not
take and misaligned pointers are rejected with the documented negative code BEFORE any device call, so these run
without a GPU.  The pointers below are made-up addresses: a rejected call never reads them.

The reference asserts the same preconditions on the CPU path (mllm/backends/cpu/ops/LinearOp.cpp: K a multiple of the
block size; mllm/backends/cpu/kernels/common/ggml/matmul_ggml.cpp: type pairs it has kernels for)."""
import ctypes as C

import pytest

from mllm_amd import _lib

P = 0x7F0000100000        # "device pointer", aligned to 1 MiB
ODD = P + 2               # breaks every alignment requirement above 2 bytes
BADARG, SHAPE, ALIGN = -1, -2, -3
Q4_0, Q8_0, Q4_K, Q6_K = 0, 1, 2, 3
F32, BF16, IMAGE = 0, 1, 2


def _part(packed=P, bias=None, y=P, N=64):
    return (_lib.GemvPart * 1)(_lib.GemvPart(packed, bias, y, N))


# name -> (valid argument list, [(argument index, bad value, expected code)])
def _cases():
    part = _part()
    cases = {
        "mllm_hip_q_prepack": ([Q4_0, P, 0, P, 64, 64, None],
                               [(0, 7, BADARG), (1, None, BADARG), (3, None, BADARG), (2, 5, BADARG), (5, 48, SHAPE), (4, 0, BADARG)]),
        "mllm_hip_linear_q_gemv": ([Q4_0, P, P, F32, None, P, 1, 64, 64, 0, None],
                                   [(0, 9, BADARG), (1, None, BADARG), (2, None, BADARG), (5, None, BADARG), (3, 5, BADARG),
                                    (6, 0, SHAPE), (8, 48, SHAPE), (9, 3, BADARG), (2, ODD, ALIGN)]),
        "mllm_hip_linear_q_gemv_multi": ([Q4_0, 1, part, P, F32, 1, 64, 0, None],
                                         [(1, 0, BADARG), (1, 5, BADARG), (2, None, BADARG), (3, None, BADARG), (5, 0, SHAPE),
                                          (6, 40, SHAPE), (3, ODD, ALIGN)]),
        "mllm_hip_linear_q_gemv_multi_ws": ([Q8_0, 1, part, P, BF16, 4, 64, 0, P, None],
                                            [(3, None, BADARG), (6, 40, SHAPE), (8, ODD, ALIGN)]),
        # the workspace of stated size: one smaller than the image of eight rows is refused
        "mllm_hip_linear_q_gemv_multi_wsn": ([Q8_0, 1, part, P, BF16, 4, 64, 0, P, 8 * 2 * 40, None],
                                             [(3, None, BADARG), (4, IMAGE, BADARG), (6, 40, SHAPE), (8, ODD, ALIGN),
                                              (9, 8 * 2 * 40 - 1, SHAPE)]),
        # the variant that allocates nothing: rows longer than its static array hold are refused
        "mllm_hip_linear_q_gemv_multi_static": ([Q8_0, 1, part, P, BF16, 4, 64, 0, None],
                                                [(3, None, BADARG), (4, IMAGE, BADARG), (6, 32768 + 32, SHAPE), (6, 40, SHAPE)]),
        "mllm_hip_linear_q": ([Q4_0, P, P, F32, None, P, 16, 64, 64, 0, P, None],
                              [(1, None, BADARG), (2, None, BADARG), (5, None, BADARG), (10, None, BADARG), (8, 50, SHAPE),
                               (6, 0, BADARG)]),
        "mllm_hip_linear_q_gemm": ([Q4_0, P, P, F32, None, P, 16, 64, 64, 0, P, None],
                                   [(0, Q4_K, BADARG), (1, None, BADARG), (2, None, BADARG), (5, None, BADARG), (10, None, BADARG),
                                    (8, 50, SHAPE)]),
        "mllm_hip_linear_q_gemm_short": ([Q8_0, P, P, BF16, None, P, 16, 64, 64, 0, P, None],
                                         [(1, None, BADARG), (5, None, BADARG), (10, None, BADARG), (8, 50, SHAPE), (6, -1, BADARG)]),
        "mllm_hip_q_gemm_prepack": ([Q4_0, P, 0, P, 64, 64, None], [(1, None, BADARG), (3, None, BADARG), (5, 48, SHAPE)]),
        "mllm_hip_quantize_q8_0": ([P, F32, P, P, 4, 64, None], [(0, None, BADARG), (2, None, BADARG), (3, None, BADARG), (5, 48, SHAPE),
                                                                 (1, 4, BADARG)]),
        "mllm_hip_quantize_weight_blocks": ([Q4_0, P, P, 0, 8, 64, None], [(1, None, BADARG), (2, None, BADARG), (5, 33, SHAPE),
                                                                           (0, 5, BADARG)]),
        "mllm_hip_q_dequantize": ([Q8_0, P, P, 8, 64, None], [(1, None, BADARG), (2, None, BADARG), (4, 31, SHAPE)]),
        "mllm_hip_mlp_gate_up_q": ([Q4_0, P, P, P, F32, P, None, 1, 64, 64, 0, None],
                                   [(1, None, BADARG), (2, None, BADARG), (3, None, BADARG), (7, 0, SHAPE), (7, 9, SHAPE),
                                    (8, 48, SHAPE), (9, 48, SHAPE), (0, Q6_K, BADARG)]),
        "mllm_hip_moe_ffn_q": ([Q4_0, P, P, P, P, F32, P, P, P, 4, 64, 64, 8, 2, 0, P, None],
                               [(1, None, BADARG), (4, None, BADARG), (6, None, BADARG), (7, None, BADARG), (8, None, BADARG),
                                (15, None, BADARG), (10, 48, SHAPE), (11, 48, SHAPE), (12, 0, BADARG), (13, 0, BADARG), (12, 3073, SHAPE)]),
        "mllm_hip_moe_ffn_q_gemm": ([Q4_0, P, P, P, P, F32, P, P, P, 4, 64, 64, 8, 2, 0, P, None],
                                    [(2, None, BADARG), (3, None, BADARG), (15, None, BADARG), (10, 48, SHAPE), (11, 48, SHAPE),
                                     (4, ODD, ALIGN), (0, Q4_K, BADARG), (12, 3073, SHAPE)]),
        # the routing pass keeps five int arrays of E entries in 64 KB of LDS
        "mllm_hip_moe_route": ([P, 4, 8, 2, None, None, None, P, None], [(0, None, BADARG), (7, None, BADARG), (2, 3073, SHAPE), (2, 0, BADARG)]),
        "mllm_hip_moe_ffn_kq": ([Q4_K, P, P, P, P, F32, P, P, P, 4, 256, 256, 8, 2, P, None],
                                [(0, Q4_0, BADARG), (1, None, BADARG), (3, None, BADARG), (4, None, BADARG), (6, None, BADARG),
                                 (14, None, BADARG), (10, 128, SHAPE), (11, 320, SHAPE), (9, 40000, SHAPE), (4, ODD, ALIGN)]),
        "mllm_hip_moe_ffn_kq2": ([Q4_K, Q6_K, P, P, P, P, F32, P, P, P, 4, 256, 256, 8, 2, P, None],
                                 [(0, Q4_0, BADARG), (1, Q8_0, BADARG), (2, None, BADARG), (5, None, BADARG), (11, 128, SHAPE),
                                  (12, 320, SHAPE), (10, 40000, SHAPE), (5, ODD, ALIGN)]),
        "mllm_hip_kq_quantize_weight_blocks": ([Q6_K, P, P, 0, 8, 256, None], [(0, Q8_0, BADARG), (1, None, BADARG), (2, None, BADARG),
                                                                              (3, 7, BADARG), (5, 128, SHAPE), (4, 0, BADARG)]),
        "mllm_hip_kq_prepack": ([Q4_K, P, 0, P, 8, 256, None], [(0, Q4_0, BADARG), (1, None, BADARG), (3, None, BADARG), (5, 128, SHAPE)]),
        "mllm_hip_linear_kq": ([Q6_K, P, P, F32, None, P, 1, 8, 256, P, None],
                               [(0, Q8_0, BADARG), (1, None, BADARG), (2, None, BADARG), (5, None, BADARG), (9, ODD, ALIGN),
                                (8, 320, SHAPE), (6, 0, BADARG)]),
        # the workspace of stated size: one smaller than the Q8_K image of eight rows is refused
        "mllm_hip_linear_kq_multi_ws": ([Q4_K, 1, part, P, BF16, 4, 256, P, 8 * 256 + 8 * 36, None],
                                        [(0, Q4_0, BADARG), (1, 0, BADARG), (1, 5, BADARG), (2, None, BADARG), (3, None, BADARG),
                                         (4, IMAGE, BADARG), (5, 0, BADARG), (6, 320, SHAPE), (7, ODD, ALIGN), (8, 8 * 256 + 8 * 36 - 1, BADARG)]),
        "mllm_hip_kq_set_rows_shape": ([0, 0], [(0, 1, BADARG), (1, 1, BADARG), (0, -1, BADARG)]),
        "mllm_hip_kq_rows_shape": ([Q4_K, 5, 64, 4096, 0], [(0, Q4_0, 0), (1, 2, 0), (1, 9, 0), (2, 0, 0), (3, 320, 0), (3, 16128, 0), (4, -1, 0)]),
        "mllm_hip_kq_set_slice_meeting": ([-1, 0], [(0, 2, BADARG), (0, -2, BADARG), (1, 9, BADARG), (1, -1, BADARG)]),
        # switches for comparison runs: anything but 0 and 1 is refused and leaves the setting alone
        "mllm_hip_w8a8_set_decode": ([1], [(0, 2, BADARG), (0, -1, BADARG)]),
        "mllm_hip_w8a8_set_decode_mfma_from": ([5], [(0, 0, BADARG), (0, 34, BADARG)]),
        "mllm_hip_w4a16_set_decode": ([1], [(0, 2, BADARG), (0, -1, BADARG)]),
        "mllm_hip_w4a16_set_decode_mfma_from": ([2], [(0, 0, BADARG), (0, 34, BADARG)]),
        "mllm_hip_q_gemm_set_form": ([0], [(0, 13, BADARG), (0, -1, BADARG)]),
        "mllm_hip_w8a8_packed_form": ([64, 64, 64], [(0, 0, 0), (1, -1, 0), (2, 0, 0)]),
        "mllm_hip_w8a8_packed_halves": ([64, 64, 64], [(0, 0, 0), (1, -1, 0), (2, 0, 0)]),
        "mllm_hip_w4a16_packed_form": ([64, 64, 64], [(0, 0, 0), (1, -1, 0), (2, 0, 0)]),
        "mllm_hip_w4a16_packed_eight": ([64, 64, 64], [(0, 0, 0), (1, -1, 0), (2, 0, 0)]),
        "mllm_hip_q_gemm_form": ([Q4_0, 64, 64, 256, 1], [(0, 5, 0), (1, 0, 0), (2, 0, 0), (3, -1, 0)]),
        "mllm_hip_q_gemm_eight": ([Q4_0, 64, 64, 256, 1], [(0, 5, 0), (1, 0, 0), (2, 0, 0), (3, -1, 0)]),
        "mllm_hip_moe_gate_set_form": ([1], [(0, 2, BADARG), (0, -1, BADARG)]),
        "mllm_hip_kq_gemm_prepack": ([Q4_K, P, 0, P, 8, 256, None], [(0, Q8_0, BADARG), (1, None, BADARG), (5, 96, SHAPE)]),
        "mllm_hip_linear_kq_gemm": ([Q4_K, P, P, F32, None, P, 16, 8, 256, P, None],
                                    [(0, Q4_0, BADARG), (1, None, BADARG), (5, None, BADARG), (9, None, BADARG), (8, 100, SHAPE)]),
        "mllm_hip_linear_kq_gemm_short": ([Q6_K, P, P, BF16, None, P, 16, 8, 256, P, None],
                                          [(0, Q4_0, BADARG), (2, None, BADARG), (9, None, BADARG), (8, 100, SHAPE)]),
        "mllm_hip_quantize_q8_K": ([P, F32, P, P, P, 2, 256, None], [(0, None, BADARG), (2, None, BADARG), (3, None, BADARG),
                                                                     (4, None, BADARG), (6, 64, SHAPE)]),
        "mllm_hip_per_token_quant_int8": ([P, BF16, P, P, 4, 64, None], [(0, None, BADARG), (2, None, BADARG), (3, None, BADARG),
                                                                        (1, 7, BADARG), (4, 0, BADARG)]),
        "mllm_hip_w8a8_gemm": ([P, P, P, P, None, P, None, 16, 64, 64, None],
                               [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (3, None, BADARG), (5, None, BADARG),
                                (7, 0, BADARG), (9, 40, SHAPE), (0, ODD, ALIGN)]),
        "mllm_hip_w8a8_linear": ([P, BF16, P, P, None, P, 16, 64, 64, P, None],
                                 [(0, None, BADARG), (2, None, BADARG), (3, None, BADARG), (5, None, BADARG), (9, None, BADARG),
                                  (1, 9, BADARG), (8, 40, SHAPE)]),
        "mllm_hip_w8a8_linear_packed": ([P, BF16, P, P, None, P, 16, 64, 64, P, None],
                                        [(0, None, BADARG), (2, None, BADARG), (3, None, BADARG), (5, None, BADARG), (9, None, BADARG)]),
        "mllm_hip_w4a16_gemm": ([P, P, P, P, None, P, 16, 64, 256, 128, None],
                                [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (5, None, BADARG), (9, 100, SHAPE),
                                 (8, 200, SHAPE)]),
        "mllm_hip_w4a16_from_awq": ([P, P, P, 64, 256, 128, P, P, P, None],
                                    [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (6, None, BADARG), (7, None, BADARG),
                                     (8, None, BADARG), (3, 60, SHAPE), (4, 100, SHAPE), (5, 96, SHAPE), (6, ODD, ALIGN)]),
        "mllm_hip_w4a16_gemm_packed": ([P, P, None, P, 16, 64, 256, 128, None],
                                       [(0, None, BADARG), (1, None, BADARG), (3, None, BADARG), (7, 100, SHAPE)]),
        "mllm_hip_rmsnorm": ([P, F32, P, P, 1, 64, C.c_float(1e-6), 0, None, 0, None],
                             [(0, None, BADARG), (2, None, BADARG), (1, 3, BADARG), (4, 0, BADARG)]),
        "mllm_hip_silu_mul": ([P, P, P, F32, 1, 64, None, 0, None], [(0, None, BADARG), (1, None, BADARG), (3, 3, BADARG), (4, 0, BADARG)]),
        "mllm_hip_add": ([P, P, P, F32, 1, 64, None, 0, None], [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG)]),
        "mllm_hip_softmax": ([P, P, 2, 16, None], [(0, None, BADARG), (1, None, BADARG), (2, 0, BADARG)]),
        "mllm_hip_topk": ([P, P, P, 2, 16, 4, 1, 1, None], [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (5, 0, SHAPE),
                                                            (5, 17, SHAPE)]),
        "mllm_hip_matmul_batched": ([P, P, P, 0, 2, 4, 4, 4, 16, 16, 16, 0, 0, None],
                                    [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (3, 2, BADARG), (3, 7, BADARG),
                                     (4, 0, BADARG), (5, 0, BADARG), (8, -1, BADARG), (10, 8, SHAPE), (0, P + 2, ALIGN)]),
        "mllm_hip_matmul_set_tile": ([0], [(0, 32, BADARG), (0, -1, BADARG)]),
        "mllm_hip_matmul_f32": ([P, P, P, 4, 4, 4, 0, 0, None], [(0, None, BADARG), (1, None, BADARG), (2, None, BADARG), (3, 0, BADARG)]),
    }
    return cases


_CASES = _cases()
_PARAMS = [(name, idx, bad, code) for name, (_, bads) in _CASES.items() for (idx, bad, code) in bads]


@pytest.mark.parametrize("name,idx,bad,code", _PARAMS, ids=["%s-arg%d-%s" % (n, i, b) for n, i, b, _ in _PARAMS])
def test_entry_point_rejects_bad_argument(name, idx, bad, code):
    L = _lib.lib()
    args = list(_CASES[name][0])
    args[idx] = bad
    rc = getattr(L, name)(*args)
    assert rc == code, "%s with argument %d = %r returned %d, expected %d" % (name, idx, bad, rc, code)


@pytest.mark.parametrize("wtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("N", [128, 2048, 4096])
def test_long_rows_of_few_channels_take_two_slices_per_wave(wtype, N):
    """three to six rows of 13 to 16 K slices, one tile per workgroup: a wave per slice was 3 to 17 % slower than two slices per wave"""
    shape = _lib.lib().mllm_hip_kq_rows_shape
    for K, waves in ((6144, 12), (6400, 7), (6656, 7), (7168, 7), (7680, 8), (8192, 8), (8448, 9)):
        assert [shape(wtype, M, N, K, 0) - 16 for M in (3, 4, 6)] == [waves] * 3
    assert shape(wtype, 8, N, 8192, 0) == 16 + 16 and shape(wtype, 3, 4112, 8192, 0) == 2 * 16 + 8


@pytest.mark.parametrize("wtype", [Q4_K, Q6_K])
def test_rows_that_take_two_slices_per_wave_are_quantized_once(wtype):
    """three and four rows of 13 to 16 slices were up to 13 % slower where every workgroup quantizes them (four items per thread with a wave per slice)"""
    image = _lib.lib().mllm_hip_kq_rows_image
    for N in (80, 2560, 4096):
        assert [image(wtype, M, N, K) for K in (6400, 6656, 7168, 8192) for M in (3, 4, 6)] == [1] * 12
        assert [image(wtype, M, N, K) for K in (1024, 2560, 4096) for M in (3, 4)] == [0] * 6
    assert image(wtype, 5, 2560, 4096) == 1 and image(wtype, 4, 2048, 6144) == 0 and image(wtype, 2, 2560, 4096) == 0 and image(wtype, 5, 2560, 9728) == 1


def test_moe_tiles_of_long_rows_spread_their_slices_over_waves():
    """one wave per tile walked all of K: 4 to 21 % slower than a workgroup per slice with eight experts of 3584 or 4096 elements"""
    shape = lambda *a: divmod(_lib.lib().mllm_hip_kq_rows_shape(*a), 16)  # noqa: E731
    for wtype in (Q4_K, Q6_K):
        assert shape(wtype, 8, 512, 3584, 10) == (2, 4) and shape(wtype, 8, 512, 3584, 5) == (1, 4)
        assert shape(wtype, 8, 2048, 2048, 5) == (2, 2) and shape(wtype, 8, 16, 1536, 9) == (1, 2)
        assert shape(wtype, 8, 2048, 768, 100) == (4, 1) and shape(wtype, 8, 1536, 2048, 129) == (4, 1)
    assert shape(Q4_K, 8, 2 * 768, 4096, 10) == (4, 2) and shape(Q6_K, 8, 2 * 768, 4096, 10) == (2, 4)


def test_moe_pairs_take_two_tiles_per_wave_where_that_is_faster():
    """from 2048 workgroups of all parts on, and for rows of three super-blocks: longer ones were up to 5 % slower with two (1536 and 2048 workgroups of 1024
    and 1536 elements), and so were three (1536 workgroups)"""
    tiles = _lib.lib().mllm_hip_kq_moe_pair_tiles
    for parts, N in ((1, 2048), (2, 1024)):
        assert [tiles(parts, N, 768, slots) for slots in (16, 48, 63, 64, 128)] == [1, 1, 1, 2, 2]
        assert [tiles(parts, N, K, 64) for K in (512, 1024, 1280, 1536, 1792)] == [0, 1, 1, 1, 0]
    assert tiles(1, 1024, 768, 127) == 1 and tiles(1, 1024, 768, 128) == 2 and tiles(0, 2048, 768, 64) == 0 and tiles(1, 2048, 768, 15) == 0


def test_softmax_is_cut_into_pieces_only_where_that_is_not_slower():
    """193 to 256 rows, one whole round of workgroups, stay a workgroup per row up to 50 000 elements"""
    room = _lib.lib().mllm_hip_softmax_workspace_bytes
    for rows, ln, pieces in ((1, 40960, 0), (1, 40961, 11), (192, 40968, 11), (193, 46120, 0), (256, 50000, 0), (256, 50001, 13), (257, 40968, 11),
                             (512, 40968, 11), (513, 151936, 0)):
        assert room(rows, ln) == rows * pieces * 8, (rows, ln)


@pytest.mark.parametrize("M,N,K,form", [(1811, 264, 1280, 4), (381, 1480, 1664, 4), (3409, 1176, 704, 7), (1117, 872, 1344, 4), (169, 4592, 1216, 4),
                                        (2048, 6144, 2048, 8), (93, 2560, 9728, 1), (20, 1968, 192, 1)])
def test_w8a8_takes_a_form_that_measures_fast(M, N, K, form):
    """shapes at which a choice by tiles and K steps alone took 13 to 26 % longer than this form (the first five), and where it took it"""
    L = _lib.lib()
    assert L.mllm_hip_w8a8_packed_form(M, N, K) == form
    assert [L.mllm_hip_w8a8_packed_form(t, N, K) for t in (1, 4)] == [9, 9] and len({L.mllm_hip_w8a8_packed_form(t, N, K) for t in (5, 17, 32)}) == 1


@pytest.mark.parametrize("M,N,K,form", [(1155, 1912, 4288, 4), (338, 5456, 4928, 4), (998, 2488, 3904, 4), (927, 1032, 9728, 3), (270, 3232, 7040, 3), (1204, 803, 6592, 3)])
def test_w8a8_keeps_the_form_that_halves_of_larger_tiles_do_not_beat(M, N, K, form):
    """shapes at which a gain of halves of K in the choice took larger tiles, 8 to 22 % slower"""
    assert _lib.lib().mllm_hip_w8a8_packed_form(M, N, K) == form


def test_w8a8_runs_halves_of_k_where_they_are_faster():
    """from six (64 x 128) and ten (128 x 128) blocks of 128 on, up to 256 tiles; with fewer blocks halves took up to 1.07 and 1.12 of the time"""
    L = _lib.lib()
    for M, N, block, form in ((99, 16384, 6, 4), (128, 12288, 6, 4), (728, 5064, 10, 5), (488, 8184, 10, 5)):
        for blocks, halves in ((block - 1, 0), (block, 1)):
            assert (L.mllm_hip_w8a8_packed_form(M, N, 128 * blocks), L.mllm_hip_w8a8_packed_halves(M, N, 128 * blocks)) == (form, halves)
    assert (L.mllm_hip_w8a8_packed_form(128, 16512, 768), L.mllm_hip_w8a8_packed_halves(128, 16512, 768)) == (4, 0)  # 258 tiles
    for N, blocks, halves in ((24576, 23, 1), (24584, 23, 0), (24584, 24, 1)):  # one tile of rows and more than 192 of channels
        assert (L.mllm_hip_w8a8_packed_form(33, N, 128 * blocks), L.mllm_hip_w8a8_packed_halves(33, N, 128 * blocks)) == (4, halves)
    assert L.mllm_hip_w8a8_packed_halves(4, 4096, 4096) == 0 and L.mllm_hip_w8a8_packed_halves(2048, 6144, 2048) == 0


@pytest.mark.parametrize("M,N,K,form", [(3500, 456, 1280, 8), (4580, 576, 512, 8), (5226, 376, 2688, 8), (738, 2720, 384, 8), (2048, 9728, 2560, 6), (93, 2048, 6144, 2),
                                        (64, 9728, 128, 10), (1, 1440, 512, 10), (65, 9728, 128, 8), (64, 9728, 576, 4)])
def test_w4a16_takes_a_form_that_measures_fast(M, N, K, form):
    """shapes at which a choice without tiles of 64 rows took 23 to 33 % longer (the first four), few K blocks, and a long prompt; the tokens of
    a decode step take one form however many there are"""
    L = _lib.lib()
    assert L.mllm_hip_w4a16_packed_form(M, N, K) == form
    assert len({L.mllm_hip_w4a16_packed_form(t, N, K) for t in (1, 5, 9, 32)}) == 1


@pytest.mark.parametrize("M,N,K,form", [(778, 1915, 1792, 3), (296, 4756, 1664, 3), (177, 7068, 1280, 4), (458, 4129, 4480, 3), (258, 6832, 5120, 3), (526, 3808, 8448, 3),
                                        (297, 5525, 3328, 4), (184, 8764, 3712, 4), (1064, 1283, 7936, 8)])
def test_w4a16_keeps_the_form_that_halves_of_larger_tiles_do_not_beat(M, N, K, form):
    """shapes at which halves of K of larger tiles took 9 to 25 % longer (rows that are no multiple of 16 bytes) and 6 to 8 % (the two whose rows are), and at which
    they are the faster ones all the same"""
    assert _lib.lib().mllm_hip_w4a16_packed_form(M, N, K) == form


def test_w4a16_runs_eight_waves_where_they_are_faster():
    """from as many blocks of K on as pay for the meeting of the sums: 64 x 64 with six blocks took 1.02 of the time by eight, with four 1.06"""
    L = _lib.lib()
    take = lambda M, N, K: (L.mllm_hip_w4a16_packed_form(M, N, K), L.mllm_hip_w4a16_packed_eight(M, N, K))  # noqa: E731
    for M, N, K, form in ((211, 2832, 448, 4), (1009, 624, 448, 4), (745, 4632, 448, 5), (1146, 6816, 512, 6), (138, 9376, 512, 8), (604, 2880, 512, 8)):
        assert take(M, N, K - 64) == (form, 0) and take(M, N, K) == (form, 1)
    assert take(8, 4096, 4096)[1] == 0 and take(2048, 9728, 2560) == (6, 0)


@pytest.mark.parametrize("shape,side", [((42, 157, 721, 1301, 0, 0), 64), ((9, 3206, 145, 1475, 0, 0), 64), ((19, 161, 1610, 1070, 1, 0), 64), ((50, 162, 589, 813, 1, 0), 64),
                                        ((18, 1578, 99, 33, 0, 1), 64), ((17, 382, 515, 35, 0, 1), 64), ((8, 3108, 128, 777, 0, 0), 128), ((8, 504, 504, 128, 0, 0), 0)])
def test_matmul_takes_a_form_that_measures_fast(shape, side):
    """edges of large tiles (8 to 15 % slower than small ones at the first four) and K that fills a step of the fp32 instructions by a thirty-second (18 and 20 %)"""
    assert _lib.lib().mllm_hip_matmul_split_side(*shape) == side


def test_topk_is_cut_into_pieces_only_where_that_is_faster():
    """rows without whole vectors of up to 8192 elements stay one workgroup's work while that is one round of workgroups"""
    room = _lib.lib().mllm_hip_topk_workspace_bytes
    for rows, ln, k, pieces in ((8, 4096, 50, 0), (8, 4097, 50, 0), (1, 8191, 1, 0), (256, 5001, 128, 0), (257, 4097, 50, 2), (8, 4100, 50, 2), (8, 8192, 50, 2),
                                (8, 8193, 50, 3), (8, 151936, 128, 38), (512, 151936, 20, 38), (513, 151936, 20, 0), (8, 151936, 129, 0)):
        assert room(rows, ln, k) == rows * pieces * k * 8, (rows, ln, k)


@pytest.mark.parametrize("wtype,M,N,K,forms", [
    (Q6_K, 54, 6144, 2048, (2,)), (Q6_K, 138, 2288, 1536, (2,)), (Q4_K, 394, 2560, 9728, (10,)), (Q4_0, 415, 5640, 8768, (9,)),
    (Q6_K, 316, 8880, 7424, (6, 8)), (Q4_0, 1956, 760, 4832, (8, 9, 10)), (Q6_K, 114, 2560, 9728, (2,)), (Q6_K, 130, 3544, 5632, (3,)),
    (Q8_0, 135, 3856, 5760, (3,)), (Q4_0, 256, 2560, 9728, (3,)), (Q4_0, 41, 8504, 9600, (11,)), (Q4_K, 33, 8376, 8448, (11,)),
    (Q4_0, 1287, 712, 8160, (11,)), (Q4_0, 1028, 728, 8224, (12,)), (Q4_0, 1287, 712, 8192, (3,))])
def test_q_gemm_takes_a_form_that_measures_fast(wtype, M, N, K, forms):
    """shapes at which a choice by rows, columns and K steps alone was 10 to 23 % slower than the forms here (measured, all twelve), and at which ranges by
    a margin over 64 x 64 tiles took 3 to 29 % longer or, at two of one tile of rows, those tiles 10 %; rows near 16 KB apart that straddle cache lines (42 and
    31 %) and one that does not"""
    assert _lib.lib().mllm_hip_q_gemm_form(wtype, M, N, K, 1) in forms
    assert _lib.lib().mllm_hip_q_gemm_form(wtype, M, N, K, 0) <= 5  # no room for partial results: no ranges


@pytest.mark.parametrize("wtype,M,N,K,form,eight", [
    (Q8_0, 984, 816, 7040, 12, 0), (Q6_K, 99, 8480, 5376, 11, 0), (Q8_0, 162, 3888, 17472, 12, 1), (Q6_K, 394, 2560, 9728, 10, 1), (Q4_K, 1466, 752, 6912, 11, 1),
    (Q4_0, 180, 3120, 7680, 3, 1), (Q6_K, 138, 2288, 1536, 2, 1), (Q4_0, 2048, 9728, 2560, 5, 0)])
def test_q_gemm_runs_eight_waves_where_they_are_faster(wtype, M, N, K, form, eight):
    """the first two: byte codes in ranges of fourteen and twelve blocks on nearly every CU, 4 and 2 % slower by eight"""
    L = _lib.lib()
    assert (L.mllm_hip_q_gemm_form(wtype, M, N, K, 1), L.mllm_hip_q_gemm_eight(wtype, M, N, K, 1)) == (form, eight)


@pytest.mark.parametrize("M,N,K", [(200, 2560, 9728), (200, 2558, 9728), (70, 260, 160), (200, 1024, 640), (512, 512, 65536)])
def test_q_gemm_has_room_for_the_ranges_of_each_format(M, N, K):
    """partial results of the larger of a call's two formats, 64 MB at most; none where no format takes ranges or N % 4"""
    L = _lib.lib()
    up = lambda b: (b + 255) // 256 * 256
    for types, room, plain in (((Q4_0, Q8_0), L.mllm_hip_linear_q_gemm_short_workspace_bytes, up(L.mllm_hip_linear_q_gemm_workspace_bytes(M, K))),
                               ((Q4_K, Q6_K), L.mllm_hip_linear_kq_gemm_short_workspace_bytes, L.mllm_hip_linear_kq_gemm_workspace_bytes(M, K))):
        if K % 256 and Q4_K in types:
            continue
        z = max(max(1, L.mllm_hip_q_gemm_form(t, M, N, K, 1) - 4) for t in types)
        partial = room(M, N, K) - plain - 256
        assert partial == (up(z * M * N * 4) if z > 1 else 0) and partial <= 64 << 20
        assert N % 4 == 0 or z == 1


def test_size_helpers_return_zero_for_shapes_they_do_not_take():
    L = _lib.lib()
    assert L.mllm_hip_q_packed_bytes(Q4_0, 64, 48) == 0
    assert L.mllm_hip_q_packed_bytes(5, 64, 64) == 0
    assert L.mllm_hip_kq_packed_bytes(Q4_K, 8, 128) == 0
    assert L.mllm_hip_kq_packed_bytes(Q4_0, 8, 256) == 0
    assert L.mllm_hip_q_gemm_packed_bytes(Q4_0, 0, 64) == 0
    assert L.mllm_hip_kq_gemm_packed_bytes(Q8_0, 8, 256) == 0
    assert L.mllm_hip_gemv_workspace_bytes(0, 64) == 0
    assert L.mllm_hip_gemv_workspace_bytes(1, 48) == 0
    assert L.mllm_hip_moe_workspace_bytes(4, 48, 64, 8, 2) == 0
    assert L.mllm_hip_moe_gemm_workspace_bytes(4, 64, 64, 0, 2) == 0
    assert L.mllm_hip_w4a16_packed_bytes(64, 256, 100) == 0
    assert L.mllm_hip_moe_kq_workspace_bytes(4, 128, 256, 8, 2) == 0
    assert L.mllm_hip_kq_workspace_bytes_n(4, 128, 64) == 0
    # no kernel leaves partial sums there: the image alone, whatever the channels
    for k, n in ((256, 64), (4096, 64), (4096, 0), (9728, 9728)):
        assert L.mllm_hip_kq_workspace_bytes_n(4, k, n) == L.mllm_hip_kq_workspace_bytes(4, k) > 8 * k
