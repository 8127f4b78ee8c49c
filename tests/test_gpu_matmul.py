"""GPU parity of the MatMul slot (activation x activation, mllm/backends/cpu/ops/MatMulOp.cpp:19-90).

fp32: exact products summed in fp32 on the matrix cores, against a float64 sum of the same products; the bound is a few
ulp of fp32 per sqrt(K) (rel-L2 <= 2e-6 written below).  bf16 / fp16: exact products, fp32 sums, one rounding; compared with
the float64 result rounded the same way (rel-L2 <= 1e-3, the bound the quantized Linears use)."""
import numpy as np
import pytest
import torch

from mllm_amd import _lib, qlinear as ql, synth
from gpu_util import announce, rel_l2

pytestmark = pytest.mark.gpu


def _ref(a, b, ta, tb):
    a64 = a.astype(np.float64)
    b64 = b.astype(np.float64)
    if ta:
        a64 = np.swapaxes(a64, -1, -2)
    if tb:
        b64 = np.swapaxes(b64, -1, -2)
    return a64 @ b64


SHAPES = [(1, 1, 1, 1), (1, 70, 130, 96), (3, 33, 65, 31), (2, 128, 128, 128), (5, 1, 257, 64), (2, 200, 7, 40),
          (4, 129, 131, 250), (1, 64, 64, 2049),
          # up to four rows against [K][N] (a decode token's probabilities x values): the GEMV form when not transposed
          (32, 1, 128, 1024), (3, 2, 136, 300), (2, 4, 1024, 257), (1, 3, 2052, 512), (5, 1, 8, 4096)]


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", SHAPES)
def test_matmul_fp32(batch, M, N, K, ta, tb):
    rng = synth.rng_for(6, batch + M + N + K + 2 * ta + tb)
    a = rng.standard_normal((batch, K, M) if ta else (batch, M, K)).astype(np.float32)
    b = rng.standard_normal((batch, N, K) if tb else (batch, K, N)).astype(np.float32)
    announce("matmul fp32 %s ta=%d tb=%d" % ((batch, M, N, K), ta, tb))
    c = ql.matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), ta, tb).cpu().numpy()
    assert c.shape == (batch, M, N)
    assert rel_l2(c, _ref(a, b, ta, tb)) <= 2e-6


def test_matmul_fp32_integers_are_exact_and_batches_do_not_mix():
    """small integers: every product and partial sum is exact in fp32, so the result must equal the integer product; each
    batch entry carries a different multiplier so that a wrong stride shows"""
    rng = synth.rng_for(6, 1)
    batch, M, N, K = 6, 96, 160, 72
    a = rng.integers(-8, 9, (batch, M, K)).astype(np.float32) * (1 + np.arange(batch, dtype=np.float32))[:, None, None]
    b = rng.integers(-8, 9, (batch, N, K)).astype(np.float32)
    announce("matmul fp32 exact")
    c = ql.matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), False, True).cpu().numpy()
    assert np.array_equal(c, _ref(a, b, False, True).astype(np.float32))
    # one right-hand matrix for the whole batch
    c1 = ql.matmul(torch.from_numpy(a).cuda(), torch.from_numpy(b[2]).cuda(), False, True).cpu().numpy()
    assert np.array_equal(c1, _ref(a, b[2][None], False, True).astype(np.float32))


def test_matmul_unaligned_views_take_the_element_path():
    """operands that start 4 bytes into an allocation, and odd leading dimensions"""
    rng = synth.rng_for(6, 2)
    M, N, K = 50, 40, 37
    a = rng.standard_normal(M * K + 1).astype(np.float32)
    b = rng.standard_normal(N * K + 1).astype(np.float32)
    ad, bd = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    announce("matmul fp32 unaligned")
    c = ql.matmul(ad[1:].view(M, K), bd[1:].view(N, K), False, True).cpu().numpy()
    assert rel_l2(c, _ref(a[1:].reshape(M, K), b[1:].reshape(N, K), False, True)) <= 2e-6


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", [(1, 70, 130, 96), (3, 33, 65, 31), (2, 256, 128, 128), (16, 128, 256, 64), (2, 9, 200, 1000),
                                          (32, 1, 128, 1024), (3, 2, 136, 300), (2, 4, 1024, 264), (1, 3, 4104, 512)])
def test_matmul_16_bit(batch, M, N, K, ta, tb, dtype):
    rng = synth.rng_for(6, 1000 + batch + M + N + K + 2 * ta + tb)
    td = torch.bfloat16 if dtype == "bf16" else torch.float16
    a = torch.from_numpy(rng.standard_normal((batch, K, M) if ta else (batch, M, K)).astype(np.float32)).to(td)
    b = torch.from_numpy(rng.standard_normal((batch, N, K) if tb else (batch, K, N)).astype(np.float32)).to(td)
    announce("matmul %s %s ta=%d tb=%d" % (dtype, (batch, M, N, K), ta, tb))
    c = ql.matmul(a.cuda(), b.cuda(), ta, tb).cpu()
    want = torch.from_numpy(_ref(a.float().numpy(), b.float().numpy(), ta, tb)).to(td)
    assert rel_l2(c.float().numpy(), want.float().numpy()) <= 1e-3
    # and against the unrounded float64 result: no worse than one rounding of the result type
    assert rel_l2(c.float().numpy(), _ref(a.float().numpy(), b.float().numpy(), ta, tb)) <= (3e-3 if dtype == "bf16" else 4e-4)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("batch,M,N,K,ta,tb", [
    # tiles (the larger one for the first shape in 16 bits), rows past the end repeated, K steps that end behind K, [K][rows] operands
    # whose rows are or are not a multiple of a vector, fewer rows than a vector
    (1, 2050, 2174, 257, False, True), (33, 513, 387, 290, False, False), (1, 2177, 2049, 288, True, True), (3, 65, 63, 33, False, False),
    (2, 3, 2, 64, True, False), (2, 66, 68, 96, True, False), (2, 5, 3, 31, False, False), (1, 64, 7, 320, True, False),
    # up to four rows: dot products (one and four rows of B per group, groups of 4 to 64 lanes, several pieces per lane), values
    (1, 4, 5, 8, False, True), (1, 1, 63, 2056, False, True), (40, 4, 401, 128, False, True), (7, 2, 1030, 264, False, True),
    (1, 3, 64, 2048, False, True), (9, 3, 520, 1027, False, False), (1, 4, 8, 259, False, False)])
def test_matmul_forms_at_their_edges(batch, M, N, K, ta, tb, dtype):
    """fp32: products of integers up to 8 and their sums (<= 64 K < 2^24) are exact, so the result is the integer product; 16 bits:
    the same sums, rounded once to the result type"""
    rng = synth.rng_for(6, 2000 + batch + M + N + K)
    td = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    a = rng.integers(-8, 9, (batch, K, M) if ta else (batch, M, K)).astype(np.float32)
    b = rng.integers(-8, 9, (batch, N, K) if tb else (batch, K, N)).astype(np.float32)
    announce("matmul %s %s ta=%d tb=%d" % (dtype, (batch, M, N, K), ta, tb))
    c = ql.matmul(torch.from_numpy(a).to(td).cuda(), torch.from_numpy(b).to(td).cuda(), ta, tb).cpu()
    a, b = torch.from_numpy(a), torch.from_numpy(b)
    want = torch.matmul(a.transpose(1, 2).contiguous() if ta else a, b.transpose(1, 2).contiguous() if tb else b).to(td)
    assert torch.equal(c, want)


@pytest.mark.parametrize("side", [64, 128])
@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", [(3, 130, 262, 37), (2, 257, 129, 160), (1, 128, 256, 31), (2, 66, 68, 290), (2, 7, 5, 33), (5, 300, 132, 64),
                                         (1, 770, 642, 163), (1, 768, 644, 1024)])
def test_matmul_on_each_tile(batch, M, N, K, ta, tb, dtype, side):
    """either tile in every order: ragged and whole tiles, rows that are and are not a multiple of a vector, K steps that end behind K, K
    of one step and less; exact as above"""
    rng = synth.rng_for(6, 4000 + batch + M + N + K)
    td = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    a = torch.from_numpy(rng.integers(-8, 9, (batch, K, M) if ta else (batch, M, K)).astype(np.float32))
    b = torch.from_numpy(rng.integers(-8, 9, (batch, N, K) if tb else (batch, K, N)).astype(np.float32))
    announce("matmul tile %d %s %s ta=%d tb=%d" % (side, dtype, (batch, M, N, K), ta, tb))
    try:
        assert _lib.lib().mllm_hip_matmul_set_tile(side) == 0
        c = ql.matmul(a.to(td).cuda(), b.to(td).cuda(), ta, tb).cpu()
    finally:
        assert _lib.lib().mllm_hip_matmul_set_tile(0) == 0
    want = torch.matmul(a.transpose(1, 2).contiguous() if ta else a, b.transpose(1, 2).contiguous() if tb else b).to(td)
    assert torch.equal(c, want)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", [(16, 16, 16, 16), (1000, 8, 8, 8), (1, 300, 132, 40), (3, 68, 60, 24), (2, 64, 128, 504), (5, 12, 8, 56)])
def test_short_matmuls_of_whole_vectors(batch, M, N, K, ta, tb, dtype):
    """K steps that end behind K with every vector inside or outside it, rows that end inside a tile: exact as above"""
    rng = synth.rng_for(6, 3000 + batch + M + N + K)
    td = torch.float32 if dtype == "fp32" else torch.bfloat16
    a = torch.from_numpy(rng.integers(-8, 9, (batch, K, M) if ta else (batch, M, K)).astype(np.float32))
    b = torch.from_numpy(rng.integers(-8, 9, (batch, N, K) if tb else (batch, K, N)).astype(np.float32))
    announce("matmul of whole vectors %s %s ta=%d tb=%d" % (dtype, (batch, M, N, K), ta, tb))
    c = ql.matmul(a.to(td).cuda(), b.to(td).cuda(), ta, tb).cpu()
    want = torch.matmul(a.transpose(1, 2).contiguous() if ta else a, b.transpose(1, 2).contiguous() if tb else b).to(td)
    assert torch.equal(c, want)


@pytest.mark.parametrize("dtype", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", [(4, 70, 7, 18), (1, 65, 130, 1), (2, 5, 3, 32), (3, 67, 129, 31), (2, 130, 66, 5), (100, 12, 520, 132),
                                         (101, 31, 513, 37), (40, 32, 1280, 64), (90, 5, 577, 33)])
def test_matmul_of_one_k_step_and_of_few_rows_by_many(batch, M, N, K, ta, tb, dtype):
    """one K step loaded element by element; up to 32 rows x [N][K] over 800 tiles and more (fp32: rows past the end left out), the last K
    step ending behind K: exact as above, and an infinity in the last row and a NaN at the last k stay in their own row and column"""
    rng = synth.rng_for(6, 6000 + batch + M + N + K)
    td = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}[dtype]
    a = torch.from_numpy(rng.integers(1, 9, (batch, M, K)).astype(np.float32))
    b = torch.from_numpy(rng.integers(-8, 9, (batch, N, K)).astype(np.float32))
    b[:, 0], b[:, N - 1] = 1., 2.
    b[:, 1, K - 1], a[:, M - 1, 0] = float("nan"), float("inf")
    want = torch.matmul(a, b.transpose(1, 2).contiguous())
    assert want[:, :M - 1].isfinite().sum() == batch * (M - 1) * (N - 1) and want[:, M - 1, N - 1].isinf().all()
    announce("matmul one step / narrow %s %s ta=%d tb=%d" % (dtype, (batch, M, N, K), ta, tb))
    ad, bd = a.transpose(1, 2).contiguous() if ta else a, b if tb else b.transpose(1, 2).contiguous()
    c = ql.matmul(ad.to(td).cuda(), bd.to(td).cuda(), ta, tb).cpu()
    want = want.to(td)
    assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c.nan_to_num(nan=0.), want.nan_to_num(nan=0.))


@pytest.mark.parametrize("side", [0, 64, 128])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(70, 130, 37), (129, 66, 64), (5, 133, 100)])
def test_matmul_keeps_infinities_and_nan_in_their_rows(M, N, K, ta, tb, dtype, side):
    """a row past the end repeats the last one, and what lies past K is zero on both sides: an infinity or a NaN reaches the results of its
    own row and column alone, also from the last row and the last k"""
    rng = synth.rng_for(6, 5000 + M + N + K)
    td = torch.float32 if dtype == "fp32" else torch.bfloat16
    a = torch.from_numpy(rng.integers(1, 9, (M, K)).astype(np.float32))
    b = torch.from_numpy(rng.integers(1, 9, (N, K)).astype(np.float32))
    a[M - 1, K - 1], a[0, 0], b[N - 1, K - 2], b[1, 0] = float("inf"), float("nan"), float("-inf"), float("inf")
    want = torch.matmul(a, b.t().contiguous()).to(td)
    ad, bd = a.t().contiguous() if ta else a, b if tb else b.t().contiguous()
    announce("matmul of infinities %s %s ta=%d tb=%d tile %d" % (dtype, (M, N, K), ta, tb, side))
    try:
        assert _lib.lib().mllm_hip_matmul_set_tile(side) == 0
        c = ql.matmul(ad.to(td).cuda(), bd.to(td).cuda(), ta, tb).cpu()
    finally:
        assert _lib.lib().mllm_hip_matmul_set_tile(0) == 0
    assert want[0].isnan().all() and want[M - 1, N - 1].isnan() and want[M - 1, 0].isinf() and want.isfinite().sum() == (M - 2) * (N - 2)
    assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c.nan_to_num(nan=0.), want.nan_to_num(nan=0.))


def _split(side, a, b, ta, tb):
    try:
        assert _lib.lib().mllm_hip_matmul_set_split(side) == 0
        return ql.matmul(a.cuda(), b.cuda(), ta, tb).cpu()
    finally:
        assert _lib.lib().mllm_hip_matmul_set_split(0) == 0


@pytest.mark.parametrize("side", [64, 128])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch,M,N,K", [(1, 5, 7, 16), (3, 65, 63, 17), (2, 64, 128, 32), (2, 129, 127, 47), (3, 128, 64, 48), (1, 257, 130, 63), (5, 70, 129, 31),
                                         (1, 200, 333, 1000)])
def test_matmul_fp32_from_bf16_parts(batch, M, N, K, ta, tb, side):
    """one to four K steps (all stages of the loop's start and end), last steps of one to sixteen k, ragged and whole tiles, in every order.  A
    product of floats has 48 bits and three bf16 parts hold a float exactly: integers below 2^12 by powers of two are exact, a one-hot
    operand returns the other one bit for bit, and random floats are within the bound of the fp32 instructions"""
    rng = synth.rng_for(6, 8000 + batch + M + N + K)
    put = lambda a, b: (torch.from_numpy(np.ascontiguousarray(np.swapaxes(a, 1, 2) if ta else a)), torch.from_numpy(np.ascontiguousarray(b if tb else np.swapaxes(b, 1, 2))))  # noqa: E731
    announce("matmul from parts %s ta=%d tb=%d side %d" % ((batch, M, N, K), ta, tb, side))
    a = (rng.integers(-4095, 4096, (batch, M, K)) * 2.0 ** rng.integers(-20, 20, (batch, M, 1))).astype(np.float32)
    b = rng.integers(-1, 2, (batch, N, K)).astype(np.float32)
    want = a.astype(np.float64) @ np.swapaxes(b, 1, 2)
    assert np.array_equal(_split(side, *put(a, b), ta, tb).numpy(), want.astype(np.float32))
    a = rng.standard_normal((batch, M, K)).astype(np.float32)
    pick = rng.integers(0, K, (batch, N))
    b = (np.arange(K) == pick[..., None]).astype(np.float32)
    assert np.array_equal(_split(side, *put(a, b), ta, tb).numpy(), np.take_along_axis(a, pick[:, None, :].repeat(M, 1), 2))
    b = rng.standard_normal((batch, N, K)).astype(np.float32)
    assert rel_l2(_split(side, *put(a, b), ta, tb).numpy(), a.astype(np.float64) @ np.swapaxes(b.astype(np.float64), 1, 2)) <= 2e-6


@pytest.mark.parametrize("side", [64, 128])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("K", [16, 61, 160])
def test_matmul_from_bf16_parts_single_products(K, ta, tb, side):
    """diag(d) B: every result is one product of two 24-bit significands, rounded once by fp32 instructions.  The parts but x0 y0 are at most 2^-7 of
    it; their seven instructions lose less than an ulp of that each, 2^-30 of the product or 2^-6 of its ulp: within 0.5 + 7 / 64 ulp"""
    rng = synth.rng_for(6, 8500 + K)
    some = lambda *s: ((rng.integers(1 << 23, 1 << 24, s) * rng.choice([-1, 1], s)) * 2.0 ** rng.integers(-33, -13, s)).astype(np.float32)  # noqa: E731
    hard = np.float32(1 + 2.0 ** -8 - 2.0 ** -16 + 2.0 ** -17 - 2.0 ** -23)  # its square loses 2^-24 without x1 y2 and x2 y1
    d, b = some(K), some(K, 150)
    d[0], b[0] = hard, hard * 2.0 ** rng.integers(-9, 9, 150).astype(np.float32)
    a = np.diag(d)
    announce("matmul from parts of single products %d ta=%d tb=%d side %d" % (K, ta, tb, side))
    c = _split(side, torch.from_numpy(a), torch.from_numpy(np.ascontiguousarray(b.T) if tb else b), ta, tb).numpy()
    want = d[:, None].astype(np.float64) * b
    ulps = np.abs(c - want) / np.exp2(np.floor(np.log2(np.abs(want))) - 23)
    assert ulps.max() <= 0.5 + 7 / 64, ulps.max()


@pytest.mark.parametrize("side", [64, 128])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(70, 130, 37), (129, 66, 64), (5, 133, 100)])
def test_matmul_from_bf16_parts_outside_their_range(M, N, K, ta, tb, side):
    """infinities, NaN, floats that round to an infinity in bf16, sums that overflow, elements whose parts are below the smallest bf16 number and
    operands of any size: fp32 instructions multiply them again, and no other row or column is infinite or NaN"""
    rng = synth.rng_for(6, 9000 + M + N + K)
    a = torch.from_numpy(rng.integers(1, 9, (M, K)).astype(np.float32))
    b = torch.from_numpy(rng.integers(1, 9, (N, K)).astype(np.float32))
    a[M - 1, K - 1], a[0, 0], b[N - 1, K - 2], b[1, 0] = float("inf"), float("nan"), float("-inf"), float("inf")
    order = lambda a, b: (a.t().contiguous() if ta else a, b if tb else b.t().contiguous())  # noqa: E731
    announce("matmul from parts of infinities %s ta=%d tb=%d side %d" % ((M, N, K), ta, tb, side))
    c, want = _split(side, *order(a, b), ta, tb), torch.matmul(a, b.t().contiguous())
    assert want.isfinite().sum() == (M - 2) * (N - 2)
    assert torch.equal(c.isnan(), want.isnan()) and torch.equal(c.nan_to_num(nan=0.), want.nan_to_num(nan=0.))
    for scale in (2.0 ** -120, 2.0 ** -104, 2.0 ** 60, 2.0 ** 107):  # a row of A; integers times a power of two: exact (sums below 2^12 2 100 2^107 < 2^127)
        a = torch.from_numpy(rng.integers(1, 1 << 12, (M, K)).astype(np.float32))
        b = torch.from_numpy(rng.integers(-2, 3, (N, K)).astype(np.float32))
        a[M // 2] *= scale
        assert torch.equal(_split(side, *order(a, b), ta, tb), torch.matmul(a.double(), b.double().t().contiguous()).float())
    for few in (False, True):  # elements below the smallest part, everywhere or one of an operand of zeros: the sums of the parts are zero
        def pair(small, other):
            x = torch.from_numpy(rng.integers(1, 1 << 9, (small, K)).astype(np.float32)) * 2.0 ** -143
            if few:
                x *= torch.arange(small * K).reshape(small, K) == (small - 1) * K + K // 2
            return x, torch.from_numpy(rng.integers(-2, 3, (other, K)).astype(np.float32)) * 2.0 ** 20
        for a, b in (pair(M, N), pair(N, M)[::-1]):
            want = torch.matmul(a.double(), b.double().t().contiguous()).float()
            assert torch.equal(_split(-1, *order(a, b), ta, tb), want) and torch.equal(_split(side, *order(a, b), ta, tb), want)
    a = torch.full((M, K), 3.3961775e38)  # below the largest float, an infinity in bf16
    b = torch.zeros((N, K))
    b[:, 0] = 1.
    assert torch.equal(_split(side, *order(a, b), ta, tb), a[:, :1].expand(M, N))


@pytest.mark.parametrize("side", [64, 128])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(70, 130, 37), (129, 66, 64), (200, 133, 100)])
def test_matmul_from_bf16_parts_depends_on_one_row_and_one_column(M, N, K, ta, tb, side):
    """random floats with a row of A, then a column of B, out of the parts' range or of zeros: its results are those of the fp32 instructions,
    every other result keeps its bits"""
    g = torch.Generator().manual_seed(M + N + K)
    a, b = torch.randn((M, K), generator=g), torch.randn((N, K), generator=g)
    run = lambda side, a, b: _split(side, a.t().contiguous() if ta else a, b if tb else b.t().contiguous(), ta, tb)  # noqa: E731
    announce("matmul from parts beside rows out of their range %s ta=%d tb=%d side %d" % ((M, N, K), ta, tb, side))
    plain = run(side, a, b)
    bits = lambda t: t.contiguous().view(torch.int32)  # noqa: E731
    for value in (float("nan"), float("inf"), 2. ** 31, 2. ** 100, 2. ** -80, 2. ** -140, 0., "one NaN", "one infinity", "one large", "zeros and one small"):
        for rows, of_b in ((M, False), (N, True)):
            x, at = (b if of_b else a).clone(), rows - 2
            if isinstance(value, float):
                x[at] *= value
            else:
                if value == "zeros and one small":
                    x[at] = 0.
                x[at, K // 2] = {"one NaN": float("nan"), "one infinity": -float("inf"), "one large": 2. ** 40, "zeros and one small": 2. ** -141}[value]
            got, want = (run(s, *((a, x) if of_b else (x, b))) for s in (side, -1))
            if of_b:
                got, want, rest = got.t(), want.t(), plain.t()
            else:
                rest = plain
            keep = torch.arange(rows) != at
            assert torch.equal(bits(got[keep]), bits(rest[keep])), (value, of_b)
            assert torch.equal(got[at].nan_to_num(nan=7.), want[at].nan_to_num(nan=7.)), (value, of_b)


def test_matmul_takes_the_bf16_parts_where_they_are_faster():
    """host-only query of the rule.  us, fp32 instructions / parts on small / large tiles: 8 x 504 x 504 x 128 9.4 / 9.5 / 12.2, 8 x 1308 x 327 x 64 11.2 /
    10.8 / 16.1, 4 x 2060 x 515 x 64 12.1 / 12.4 / 16.2, 59 x 397 x 1677 x 24 45.4 / 57.0 / 63.5, 8 x 1024 x 128 x 1024 26 / 30 / 53"""
    side = _lib.lib().mllm_hip_matmul_split_side
    for shape in ((8, 504, 504, 128), (8, 1308, 327, 64), (4, 2060, 515, 64)):
        assert side(*shape, 0, 0) != 128
    for shape in ((59, 397, 1677, 24), (8, 1024, 128, 1024), (8, 500, 500, 128), (1, 5, 4096, 2048), (8, 64, 64, 2048)):
        assert side(*shape, 0, 0) == 0
    assert side(8, 4096, 1024, 128, 0, 1) == 64 and side(1, 2048, 2048, 2048, 0, 0) == 128


def _graph_time(call, n=20):
    """median of seven replays of n calls, in us per call"""
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(n):
            call()
    times = []
    for _ in range(9):
        first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        first.record()
        graph.replay()
        last.record()
        torch.cuda.synchronize()
        times.append(first.elapsed_time(last) * 1e3 / n)
    return sorted(times[2:])[3]


def test_matmul_of_zeros_takes_no_longer():
    """a zero row of the probabilities, cache rows not yet filled, a zero column of the values, and sums of zero without a zero row: their tiles were
    searched for small elements a load at a time, 130 to 148 us where the dense product takes 42.  Bounds with room for other noise"""
    g = torch.Generator(device="cuda").manual_seed(4)
    p, v = torch.rand((8, 3108, 777), device="cuda", generator=g), torch.randn((8, 777, 128), device="cuda", generator=g)
    out = torch.empty((8, 3108, 128), device="cuda")
    assert _lib.lib().mllm_hip_matmul_split_side(8, 3108, 128, 777, 0, 0)
    announce("matmul of zeros")
    time = lambda a, b: _graph_time(lambda: ql.matmul(a, b, out=out))  # noqa: E731
    dense = time(p, v)
    row, cache, column = p.clone(), p.clone(), v.clone()
    row[:, 50], cache[:, :, 600:], column[:, :, 5] = 0, 0, 0
    unfilled = v.clone()
    unfilled[:, 600:] = 0
    for a, b in ((row, v), (cache, unfilled), (p, column)):
        assert time(a, b) <= 1.4 * dense
    row[:, 50, :400] = 1.
    column[:, :400, 5], column[:, 400:, 5] = 0, 1.
    assert (row @ column)[:, 50, 5].eq(0).all() and time(row, column) <= 1.5 * dense


def test_matmul_beside_a_nan_row_takes_one_more_product():
    """the second product of a tile, for a row or column out of the parts' range: 1.7 times the dense time, 2.3 without loads ahead (4.9 with a search
    for small elements before it)"""
    g = torch.Generator(device="cuda").manual_seed(4)
    p, v = torch.rand((8, 3108, 777), device="cuda", generator=g), torch.randn((8, 777, 128), device="cuda", generator=g)
    out = torch.empty((8, 3108, 128), device="cuda")
    announce("matmul beside a NaN row")
    dense = _graph_time(lambda: ql.matmul(p, v, out=out))
    p[:, 50] = float("nan")
    assert _graph_time(lambda: ql.matmul(p, v, out=out)) <= 2.2 * dense


def test_matmul_of_attention_sizes_takes_the_bf16_parts():
    side = _lib.lib().mllm_hip_matmul_split_side
    assert side(8, 3108, 777, 128, 0, 1) == 64 and side(8, 3108, 128, 777, 0, 0) == 128 and side(8, 1000, 520, 128, 0, 1) == 64
    assert side(8, 64, 64, 64, 0, 1) == 0 and side(1, 1 << 15, 1 << 15, 128, 0, 1) == 0 and side(8, 3108, 777, 15, 0, 1) == 0
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = torch.randn((8, 1000, 128), device="cuda", generator=g), torch.randn((8, 520, 128), device="cuda", generator=g)
    announce("matmul of 8 x 1000 x 520 x 128")
    c = ql.matmul(a, b, transpose_b=True)
    want = torch.matmul(a.double(), b.double().transpose(1, 2).contiguous())
    err = lambda c: float((c.double() - want).norm() / want.norm())  # noqa: E731
    assert side(8, 1000, 520, 128, 0, 1) and err(c) <= err(_split(-1, a, b, False, True).cuda()) <= 3e-7


def test_matmul_batches_beyond_a_grid_dimension():
    """more workgroups than a grid dimension's 32 bits of work-items hold (2^24 of 256 threads, 2^22 of 1024), once per kernel: tiles,
    dot products, values; small integers, exact"""
    n = (1 << 24) + 3
    g = torch.Generator(device="cuda").manual_seed(5)
    ints = lambda *shape, top=8, dtype=torch.float32: torch.randint(0, top, shape, device="cuda", generator=g, dtype=torch.int8).to(dtype)  # noqa: E731
    a, b = ints(n, 1, 1), ints(n, 1, 1)
    announce("matmul of 2^24 + 3 products")
    assert torch.equal(ql.matmul(a, b), a * b)
    a, b = ints(n, 1, 4), ints(n, 1, 4)
    announce("matmul of 2^24 + 3 dot products")
    assert torch.equal(ql.matmul(a, b, False, True), (a * b).sum(-1, keepdim=True))
    del a, b
    n = (1 << 22) + 3
    a, b = ints(n, 1, 256, top=2, dtype=torch.bfloat16), ints(256, 8, top=2, dtype=torch.bfloat16)  # sums up to 256: exact in bf16
    announce("matmul of 2^22 + 3 value products")
    c = ql.matmul(a, b)
    for i in range(0, n, 1 << 20):
        assert torch.equal(c[i:i + (1 << 20), 0].float(), torch.mm(a[i:i + (1 << 20), 0].float(), b.float()))
