"""GPU parity of the W4A16 path: dequantized weight table bit-exact; GEMM output rel-L2 <= 1e-3 against the oracle
(the oracle sums in float64, the matrix cores in fp32, and both round once to bf16)."""
import numpy as np
import pytest
import torch

from mllm_amd import _lib, qlinear as ql, synth
from oracle import oracle as orc
from gpu_util import announce, bf16_dev, rel_l2, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def _same_values(got_bits, want_bits):
    """bf16 tables equal as numbers; bit patterns may differ only in the sign of a zero (a zero scale: the kernel forms
    fma(q, s, -zp*s) = +0 where the closed form (q - zp) * 0 carries the sign of q - zp)."""
    g, w = synth.bf16_bits_to_fp32(got_bits), synth.bf16_bits_to_fp32(want_bits)
    neq = got_bits != want_bits
    return np.array_equal(g, w) and bool(((g == 0) & (w == 0))[neq].all())


def _dev(qw, s, zp):
    return to_dev(qw), torch.from_numpy(s.view(np.float16).copy()).cuda(), to_dev(zp)


def test_dequant_table_exhaustive():
    """every (q, zp) pair against a spread of scales"""
    s_bits = np.float16([0.01, 0.0123, 1.0, 3.14e-3, 6.1e-5, 2.5, 0.0, 1e-7]).view(np.uint16)
    rows = [(zp, si) for zp in range(16) for si in range(len(s_bits))]
    N, K = len(rows), 256
    q = np.tile(np.arange(16, dtype=np.uint8), (N, 16))
    z = np.array([[r[0], 15 - r[0]] for r in rows], dtype=np.uint8)
    s = np.array([[s_bits[r[1]], s_bits[(r[1] + 3) % len(s_bits)]] for r in rows], dtype=np.uint16)
    announce("w4a16 dequant table")
    got = _bits(ql.w4a16_dequantize(*_dev(synth.pack_nibbles(q), s, synth.pack_nibbles(z))))
    assert _same_values(got, orc.w4a16_dequant(synth.pack_nibbles(q), s, synth.pack_nibbles(z)))


def test_dequant_every_code_and_zero_point():
    """all 256 pairs of a code and a zero point with scales from the smallest denormal to the largest number of fp16, bit for bit, in both
    layouts: a nibble is converted as a number of 2^-9 times its value, the scale as 2^9 times its own"""
    scales = np.array([0x0001, 0x03ff, 0x0400, 0x1234, 0x3555, 0x3c00, 0x7bff, 0x9555, 0xfbff], np.uint16)
    N, K, group = 16 * len(scales), 64, 64
    q = np.tile(np.arange(16, dtype=np.uint8), (N, K // 16))
    z = np.tile(np.arange(16, dtype=np.uint8)[:, None], (len(scales), 1))
    qw, zp = synth.pack_nibbles(q), synth.pack_nibbles(z)
    s = np.repeat(scales, 16)[:, None].copy()
    want = orc.w4a16_dequant(qw, s, zp, group)
    announce("w4a16 every code and zero point")
    args = _dev(qw, s, zp)
    assert _same_values(_bits(ql.w4a16_dequantize(*args, group)), want)
    assert _same_values(_bits(ql.w4a16_dequantize_packed(ql.w4a16_prepack(*args, group), N, K, group)), want)


def test_dequant_full_size_bit_exact():
    rng = synth.rng_for(2)
    qw, s, zp, _, _ = synth.make_w4a16(rng, 9728, 2560)
    announce("w4a16 dequant full")
    got = _bits(ql.w4a16_dequantize(*_dev(qw, s, zp)))
    assert np.array_equal(got, orc.w4a16_dequant(qw, s, zp))


@pytest.mark.parametrize("M,N,K,group", [(1, 64, 128, 128), (9, 24, 384, 128), (130, 200, 512, 128), (64, 96, 256, 64),
                                         (257, 193, 1024, 256), (33, 128, 2560, 128)])
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_gemm_vs_oracle(M, N, K, group, tile):
    rng = synth.rng_for(2, M + N + K + group)
    qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
    a_bits, _ = synth.make_x_bf16(rng, M, K)
    bias = synth.fp32_to_bf16_bits((rng.standard_normal(N) * 0.1).astype(np.float32))
    L = _lib.lib()
    try:
        assert L.mllm_hip_w4a16_set_tuning(tile) == 0
        announce("w4a16 gemm", M, N, K, group, "tile", tile)
        d = _dev(qw, s, zp)
        c = _bits(ql.w4a16_gemm(bf16_dev(a_bits), *d, None, group))
        cb = _bits(ql.w4a16_gemm(bf16_dev(a_bits), *d, bf16_dev(bias), group))
    finally:
        L.mllm_hip_w4a16_set_tuning(0)
    want = orc.w4a16_gemm(a_bits, qw, s, zp, None, group)
    wantb = orc.w4a16_gemm(a_bits, qw, s, zp, bias, group)
    assert rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) <= TOL
    assert rel_l2(synth.bf16_bits_to_fp32(cb), synth.bf16_bits_to_fp32(wantb)) <= TOL
    # almost every element identical, the rest one bf16 ulp apart (different summation order before the single rounding)
    diff = np.abs(c.astype(np.int32) - want.astype(np.int32))
    assert diff.max() <= 1 or rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) < 1e-4
    assert (diff == 0).mean() > 0.97


# whatever form a shape takes: ragged edges, a K that is not a multiple of the 128-element K step, and groups of 64 / 128 / 256
PACKED_SHAPES = [(1, 64, 128, 128), (9, 24, 384, 128), (130, 200, 512, 128), (64, 96, 256, 64), (257, 193, 1024, 256),
                 (33, 128, 2560, 128), (70, 100, 192, 64), (1536, 6144, 256, 128), (512, 9216, 128, 128),
                 (1024, 3072, 128, 64)]


@pytest.mark.parametrize("M,N,K,group", PACKED_SHAPES)
def test_gemm_packed_vs_oracle(M, N, K, group):
    rng = synth.rng_for(2, 3 * M + N + K + group)
    qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
    a_bits, _ = synth.make_x_bf16(rng, M, K)
    bias = synth.fp32_to_bf16_bits((rng.standard_normal(N) * 0.1).astype(np.float32))
    announce("w4a16 packed gemm", M, N, K, group)
    packed = ql.w4a16_prepack(*_dev(qw, s, zp), group)
    table = _bits(ql.w4a16_dequantize_packed(packed, N, K, group))
    assert _same_values(table, orc.w4a16_dequant(qw, s, zp, group))
    c = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, None, group))
    cb = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, bf16_dev(bias), group))
    want = orc.w4a16_gemm(a_bits, qw, s, zp, None, group)
    wantb = orc.w4a16_gemm(a_bits, qw, s, zp, bias, group)
    assert rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) <= TOL
    assert rel_l2(synth.bf16_bits_to_fp32(cb), synth.bf16_bits_to_fp32(wantb)) <= TOL
    diff = np.abs(c.astype(np.int32) - want.astype(np.int32))
    assert diff.max() <= 1 or rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) < 1e-4
    assert (diff == 0).mean() > 0.97


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 13, 16, 27, 32])
def test_decode_gemv_packed_vs_oracle_and_tiles(M):
    """a few tokens take the forms whose waves split K of a 32-row tile (one piece of eight rows of it up to eight tokens): the oracle
    within the GEMM's tolerance, nearly every output the tile kernels' bits; ragged N, K not a multiple of 128, groups of 64 / 128 / 256,
    bias"""
    L = _lib.lib()
    for N, K, group in ((9728, 2560, 128), (2560, 9728, 128), (77, 192, 64), (200, 1024, 256), (33, 4096 + 64, 64)):
        rng = synth.rng_for(2, 900 + 3 * M + N + K + group)
        qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
        a_bits, _ = synth.make_x_bf16(rng, M, K)
        bias = synth.fp32_to_bf16_bits((rng.standard_normal(N) * 0.1).astype(np.float32))
        announce("w4a16 decode gemv", M, N, K, group)
        packed = ql.w4a16_prepack(*_dev(qw, s, zp), group)
        c = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, None, group))
        cb = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, bf16_dev(bias), group))
        want = orc.w4a16_gemm(a_bits, qw, s, zp, None, group)
        wantb = orc.w4a16_gemm(a_bits, qw, s, zp, bias, group)
        assert rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) <= TOL
        assert rel_l2(synth.bf16_bits_to_fp32(cb), synth.bf16_bits_to_fp32(wantb)) <= TOL
        assert L.mllm_hip_w4a16_set_decode(0) == 0
        try:
            ct = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, bf16_dev(bias), group))
        finally:
            assert L.mllm_hip_w4a16_set_decode(1) == 0
        diff = np.abs(cb.astype(np.int32) - ct.astype(np.int32))
        assert diff.max() <= 1 or rel_l2(synth.bf16_bits_to_fp32(cb), synth.bf16_bits_to_fp32(ct)) < 1e-4
        assert (diff == 0).mean() > 0.95
    assert L.mllm_hip_w4a16_set_decode(2) == -1
    # (checks its argument and selects nothing: every token count is on the matrix cores)
    assert [L.mllm_hip_w4a16_set_decode_mfma_from(t) for t in (1, 33, 0, 34)] == [0, 0, -1, -1]


@pytest.mark.parametrize("M", [1, 5, 8])
def test_one_piece_of_eight_rows_gives_the_bits_of_the_whole_tile(M):
    """up to eight tokens load and sum one piece of a 32-row tile; 9 and 32 tokens take the same form with all four (the costs depend on
    the tiles only).  16 waves, 8 waves, 8 waves on 64 channels and 4 waves (K up to 512), ragged N, N % 4 != 0, one K block and K blocks that do not divide;
    rows past the batch of NaN and infinities must not reach it"""
    for N, K, group in ((40, 64, 64), (1030, 448, 64), (77, 512, 128), (77, 576, 64), (1030, 1984, 64), (33, 8192, 128), (8195, 128, 64), (8202, 2048, 128), (40_001, 64, 64)):
        rng = synth.rng_for(2, 1700 + M + N + K)
        qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
        a_bits, _ = synth.make_x_bf16(rng, 32, K)
        a_bits[9:] = np.resize(np.array([0x7fc0, 0x7f80, 0xff80], np.uint16), a_bits[9:].shape)
        bias = bf16_dev(synth.fp32_to_bf16_bits((rng.standard_normal(N) * 0.1).astype(np.float32)))
        announce("w4a16 eight rows", M, N, K, group)
        packed = ql.w4a16_prepack(*_dev(qw, s, zp), group)
        got, nine, all32 = (_bits(ql.w4a16_gemm_packed(bf16_dev(a_bits[:m]), packed, N, bias, group)) for m in (M, 9, 32))
        assert np.array_equal(got, nine[:M]) and np.array_equal(got, all32[:M])


# a ragged last tile of rows and channels, N % 4 != 0 (element stores), K of one block and of an odd number; 128x256 with a
# short last round of half-height tiles (612 tiles; 16 + tile: whole ones)
@pytest.mark.parametrize("M,N,K,group", [(200, 800, 384, 128), (131, 390, 64, 64), (65, 1030, 448, 64), (2070, 9100, 128, 128)])
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 16 + 1, 16 + 5])
def test_gemm_packed_every_tile(tile, M, N, K, group):
    rng = synth.rng_for(2, 77 + tile + M - 200)
    qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
    a_bits, _ = synth.make_x_bf16(rng, M, K)
    L = _lib.lib()
    packed = ql.w4a16_prepack(*_dev(qw, s, zp), group)
    try:
        assert L.mllm_hip_w4a16_packed_set_tuning(tile) == 0
        announce("w4a16 packed gemm tile", tile)
        c = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, None, group))
    finally:
        L.mllm_hip_w4a16_packed_set_tuning(0)
    want = orc.w4a16_gemm(a_bits, qw, s, zp, None, group)
    assert rel_l2(synth.bf16_bits_to_fp32(c), synth.bf16_bits_to_fp32(want)) <= TOL


def test_full_size_prefill():
    """A bf16 [2048,2560], W uint4 [9728,2560] g128: a row sample against the oracle, plus linearity on all rows:
    GEMM(2*A) == 2*GEMM(A) exactly (scaling by two commutes with every rounding)."""
    rng = synth.rng_for(2)
    M, N, K = 2048, 9728, 2560
    qw, s, zp, _, _ = synth.make_w4a16(rng, N, K)
    a_bits, a = synth.make_x_bf16(rng, M, K)
    announce("w4a16 full size")
    d = _dev(qw, s, zp)
    c = ql.w4a16_gemm(bf16_dev(a_bits), *d)
    cb = _bits(c)
    rows = np.sort(rng.choice(M, 32, replace=False))
    want = orc.w4a16_gemm(a_bits[rows], qw, s, zp)
    r = rel_l2(synth.bf16_bits_to_fp32(cb[rows]), synth.bf16_bits_to_fp32(want))
    assert r <= TOL, r
    a2 = synth.fp32_to_bf16_bits(a * 2)
    c2 = ql.w4a16_gemm(bf16_dev(a2), *d)
    assert torch.equal(c2.float(), c.float() * 2)
    # (this shape runs 512 full tiles and 192 half-height tiles in the packed kernel's schedule)
    # the prepacked-weight path: table bit-exact, same row sample, same linearity, and close to the plain path everywhere
    packed = ql.w4a16_prepack(*d)
    assert np.array_equal(_bits(ql.w4a16_dequantize_packed(packed, N, K)), orc.w4a16_dequant(qw, s, zp))
    cp = ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N)
    r = rel_l2(synth.bf16_bits_to_fp32(_bits(cp)[rows]), synth.bf16_bits_to_fp32(want))
    assert r <= TOL, r
    assert torch.equal(ql.w4a16_gemm_packed(bf16_dev(a2), packed, N).float(), cp.float() * 2)
    assert rel_l2(cp.float().cpu().numpy(), c.float().cpu().numpy()) <= 1e-4
    # zero-point equal to every code -> exact zeros
    z_un = rng.integers(0, 16, (64, K // 128), dtype=np.uint8)
    qz = np.repeat(z_un, 128, axis=1)
    dz = _dev(synth.pack_nibbles(qz), s[:64].copy(), synth.pack_nibbles(z_un))
    c0 = ql.w4a16_gemm(bf16_dev(a_bits[:128]), *dz)
    assert (c0.float() == 0).all()


def test_argument_errors():
    L = _lib.lib()
    t = torch.zeros(4096, dtype=torch.uint8, device="cuda")
    g = L.mllm_hip_w4a16_gemm
    p = t.data_ptr()
    assert g(p, p, p, p, None, p, 8, 8, 128, 100, None) == -2     # group not a multiple of 64
    assert g(p, p, p, p, None, p, 8, 8, 192, 128, None) == -2     # K not a multiple of the group
    assert g(None, p, p, p, None, p, 8, 8, 128, 128, None) == -1
    assert g(p, p + 1, p, p, None, p, 8, 8, 128, 128, None) == -3
    assert L.mllm_hip_w4a16_set_tuning(-1) == -1


@pytest.mark.parametrize("N,K,group", [(8, 128, 128), (24, 384, 128), (200, 512, 64), (72, 1000, 200), (9728, 2560, 128)])
def test_awq_checkpoint_unpack_bit_exact_and_gemm(N, K, group):
    """AWQ int32 tensors -> row-major tensors byte for byte (against the known codes and against the oracle's unpack of the
    same dwords), then the packed GEMM on them against the oracle."""
    rng = synth.rng_for(2, N + K + group + 5)
    qweight, qzeros, scales, q, z, s = synth.make_awq(rng, N, K, group)
    announce("w4a16 from awq N=%d K=%d group=%d" % (N, K, group))
    qw_d, s_d, z_d = ql.w4a16_from_awq(torch.from_numpy(qweight).cuda(), torch.from_numpy(qzeros).cuda(),
                                       torch.from_numpy(scales.view(np.float16).copy()).cuda(), group)
    torch.cuda.synchronize()
    assert np.array_equal(qw_d.cpu().numpy(), synth.pack_nibbles(q))
    assert np.array_equal(z_d.cpu().numpy(), synth.pack_nibbles(z))
    assert np.array_equal(_bits(s_d), s)
    oq, osb, oz = orc.awq_unpack(qweight, qzeros, scales)
    assert np.array_equal(qw_d.cpu().numpy(), oq) and np.array_equal(z_d.cpu().numpy(), oz) and np.array_equal(_bits(s_d), osb)
    if group % 64 or N > 1000:
        return
    M = 37
    a_bits, _ = synth.make_x_bf16(rng, M, K)
    packed = ql.w4a16_prepack(qw_d, s_d, z_d, group)
    got = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, None, group))
    want = orc.w4a16_gemm(a_bits, oq, osb, oz, None, group)
    assert rel_l2(synth.bf16_bits_to_fp32(got), synth.bf16_bits_to_fp32(want)) <= TOL


@pytest.mark.parametrize("M", [2, 31, 33, 64, 97, 300])
def test_waves_that_split_k(M):
    """the forms whose waves share a tile and split K: ragged ends, fewer K blocks than waves, K blocks that do not divide among the waves,
    N not a multiple of 4 (element stores) and of 64, a group per K block and fewer"""
    _waves_cases((M, *s) for s in ((40, 64, 64), (193, 1088, 64), (1030, 2560, 128), (4100, 768, 256), (256, 6208, 64)))


def test_waves_that_split_k_of_larger_tiles():
    """tiles of 32x64, of 64x64 and of 64x128 (halves of K): ragged rows and channels, N % 4 != 0, K blocks that do not divide"""
    shapes = ((65, 3002, 576, 64), (45, 4101, 704, 64), (131, 4101, 576, 64), (97, 6002, 640, 128), (193, 6002, 576, 64), (300, 4101, 704, 64))
    assert [_lib.lib().mllm_hip_w4a16_packed_form(*s[:3]) for s in shapes] == [3, 3, 4, 4, 8, 8]
    _waves_cases(shapes)


def test_waves_that_split_k_of_64x64_tiles_by_eight_and_four_waves():
    """256 such tiles (eight waves) and 510 (four), ragged rows and channels, K blocks that do not divide among the waves, and six blocks (four)"""
    shapes = {(119, 8134, 1216, 64): 1, (322, 5380, 576, 64): 0, (66, 5457, 448, 64): 1, (65, 6419, 384, 64): 0}
    L = _lib.lib()
    assert {s: L.mllm_hip_w4a16_packed_eight(*s[:3]) for s in shapes} == shapes and {L.mllm_hip_w4a16_packed_form(*s[:3]) for s in shapes} == {4}
    _waves_cases(shapes)


def test_halves_of_k():
    """tiles of 128x128, 64x128, 128x256 and 64x384 that have a CU to themselves, by eight waves with half of K each: ragged rows and channels, N % 8 != 0
    (element stores), 64x128 and 64x384 with an odd number of K steps (the second half has one less; K is padded to two steps of the others); one past 256 tiles and
    one of six blocks, by four"""
    shapes = {(643, 4110, 576, 64): (5, 1), (643, 3856, 640, 64): (5, 1), (226, 4113, 576, 64): (8, 1), (225, 4104, 640, 128): (8, 1), (257, 3592, 576, 64): (8, 1),
              (97, 8220, 512, 64): (8, 1), (771, 7952, 576, 64): (6, 1), (642, 9729, 512, 64): (6, 1), (515, 8256, 1152, 64): (9, 1), (524, 8211, 1152, 64): (9, 1),
              (393, 9994, 1280, 128): (9, 1), (451, 4110, 576, 64): (8, 0), (769, 9194, 384, 64): (6, 0)}
    L = _lib.lib()
    assert {s: (L.mllm_hip_w4a16_packed_form(*s[:3]), L.mllm_hip_w4a16_packed_eight(*s[:3])) for s in shapes} == shapes
    _waves_cases(shapes)


def _waves_cases(shapes):
    for M, N, K, group in shapes:
        rng = synth.rng_for(2, 1300 + 3 * M + N + K + group)
        qw, s, zp, _, _ = synth.make_w4a16(rng, N, K, group)
        a_bits, _ = synth.make_x_bf16(rng, M, K)
        bias = synth.fp32_to_bf16_bits((rng.standard_normal(N) * 0.1).astype(np.float32))
        announce("w4a16 waves split K", M, N, K, group)
        packed = ql.w4a16_prepack(*_dev(qw, s, zp), group)
        got = _bits(ql.w4a16_gemm_packed(bf16_dev(a_bits), packed, N, bf16_dev(bias), group))
        want = orc.w4a16_gemm(a_bits, qw, s, zp, bias, group)
        assert rel_l2(synth.bf16_bits_to_fp32(got), synth.bf16_bits_to_fp32(want)) <= TOL
        assert (got == want).mean() > 0.95  # the rest one bf16 step apart: a sum in another order next to a rounding edge
