"""GPU parity of the W8A8 path: per-token int8 activation quantization (bit-exact), int32 accumulators (bit-exact) and the
scaled bf16 output (the epilogue is the same three fp32 operations as the oracle's, so it is compared bit for bit; the
stated bar is rel-L2 <= 1e-3)."""
import numpy as np
import pytest
import torch

from mllm_amd import _lib, qlinear as ql, synth
from oracle import oracle as orc
from gpu_util import announce, bf16_dev, rel_l2, to_dev

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


def test_per_token_quant_bit_exact_special_rows():
    rng = synth.rng_for(3, 1)
    a_bits, _, _ = synth.make_w8a8(rng, 40, 8, 512)
    x = synth.bf16_bits_to_fp32(a_bits)
    x[5] = 0                                                              # all-zero row -> absmax clamps to 1e-10
    x[6, :] = np.float32(0.25) * np.arange(512, dtype=np.float32)         # many exact ties after scaling
    x[7, 3] = 1e4                                                         # huge outlier
    announce("per-token quant special rows")
    for dev_x in (to_dev(x), bf16_dev(synth.fp32_to_bf16_bits(x))):
        xf = x if dev_x.dtype == torch.float32 else synth.bf16_bits_to_fp32(synth.fp32_to_bf16_bits(x))
        q, s = ql.per_token_quant_int8(dev_x)
        wq, wsc = orc.per_token_quant_int8(xf)
        assert np.array_equal(q.cpu().numpy(), wq)
        assert np.array_equal(s.cpu().numpy().view(np.uint32), wsc.view(np.uint32))


def _codes_by_division(x):
    """numpy, one IEEE division per element: the maximum passes over NaN, the code of NaN is -128"""
    amax = np.fmax(np.nanmax(np.abs(x), axis=1, initial=0.0), np.float32(1e-10)).astype(np.float32)
    scale = amax / np.float32(127.0)
    with np.errstate(invalid="ignore"):
        q = np.rint(x / scale[:, None])
    return np.where(np.isnan(q), -128.0, np.clip(q, -128.0, 127.0)).astype(np.int8), scale


def _hard_rows(rows, K):
    """rows with NaN, infinities, zeros, tiny and largest magnitudes, and rows of every code's half-way points (scale * (n + 1/2), one ulp below and above,
    both signs) under scales of random significands"""
    rng = synth.rng_for(3, 77 + K)
    x = rng.standard_normal((rows, K)).astype(np.float32)
    x[0, K // 2], x[0, 0] = np.nan, -np.nan
    x[1, 1], x[1, K - 1], x[1, 5] = np.inf, -np.inf, np.nan
    x[2] = 0.0
    x[3] *= np.float32(1e-38)
    x[4] = np.where(np.arange(K) % 3, -3.4028235e38, 1e36).astype(np.float32)
    x[5] *= np.float32(2.0 ** -42)
    x[6] = np.nan
    x[7] = np.float32(-1e-10) * (np.arange(K) % 255).astype(np.float32) / 254
    half = np.arange(127, dtype=np.float64) + 0.5
    for r in range(8, rows):
        amax = np.float32((1 + rng.random()) * 2.0 ** int(rng.integers(-30, 100)))
        mid = (half * float(amax / np.float32(127.0))).astype(np.float32)
        mid = np.concatenate([mid, np.nextafter(mid, np.float32(0)), np.nextafter(mid, np.float32(np.inf))])
        mid = np.concatenate([mid, -mid])
        mid = mid[np.abs(mid) <= amax][:K - 1]
        x[r] = 0.0
        x[r, :mid.size], x[r, K - 1] = mid, amax
    return x


@pytest.mark.parametrize("K", [768, 2816, 9728])
def test_per_token_codes_are_those_of_a_division(K):
    """the rows above through the launch that quantizes (a row in registers, and read twice) and through the Linear of one to four tokens, whose one-hot
    weights return the codes times the scales"""
    x = _hard_rows(48, K)
    for xd in (to_dev(x), to_dev(x).bfloat16()):
        xf = xd.float().cpu().numpy()
        want, scale = _codes_by_division(xf)
        announce("per-token codes beside a division", K, str(xd.dtype))
        q, s = ql.per_token_quant_int8(xd)
        assert np.array_equal(s.cpu().numpy().view(np.uint32), scale.view(np.uint32))
        assert np.array_equal(q.cpu().numpy(), want)
        if K > 768:
            continue
        W = ql.w8a8_prepack(torch.eye(K, dtype=torch.int8, device="cuda"))
        one = torch.ones(K, device="cuda")
        with np.errstate(invalid="ignore", over="ignore"):
            f = torch.from_numpy(want.astype(np.float32) * (np.float32(1.0) * scale[:, None]))
        for M in (1, 2, 3, 4):
            for r in range(0, 48, M):
                y = ql.w8a8_linear_packed(xd[r:r + M].contiguous(), W, K, one).float().cpu()
                w = f[r:r + M].bfloat16().float()
                assert torch.equal(y.nan_to_num(nan=3e38), w.nan_to_num(nan=3e38)), (M, r)


@pytest.mark.parametrize("M,K", [(2048, 2048), (7, 100), (3, 8), (5, 6144 + 24)])
def test_per_token_quant_bit_exact(M, K):
    rng = synth.rng_for(3, M + K)
    a_bits, _, _ = synth.make_w8a8(rng, M, 8, K)
    announce("per-token quant", M, K)
    q, s = ql.per_token_quant_int8(bf16_dev(a_bits))
    wq, wsc = orc.per_token_quant_int8(synth.bf16_bits_to_fp32(a_bits))
    assert np.array_equal(q.cpu().numpy(), wq)
    assert np.array_equal(s.cpu().numpy().view(np.uint32), wsc.view(np.uint32))


# the shapes the reference's own int8 GEMM test uses (mllm-kernel/tests/test_int8_scaled_mm_cutlass.py:123-132)
REF_SHAPES = [(1, 64, 32), (1, 2048, 2048), (8, 128, 64), (16, 6144, 2048), (32, 2048, 2048), (93, 6144, 2048),
              (128, 2048, 6144)]


@pytest.mark.parametrize("M,N,K", REF_SHAPES + [(300, 200, 48), (257, 193, 80)])
@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4])
def test_gemm_bit_exact(M, N, K, tile):
    rng = synth.rng_for(3, M * 7 + N + K)
    xq = rng.integers(-127, 128, (M, K), dtype=np.int8)
    W = rng.integers(-127, 128, (N, K), dtype=np.int8)
    xs = ((rng.random(M) + 0.01) * 0.01).astype(np.float32)
    ws = ((rng.random(N) + 0.01) * 0.01).astype(np.float32)
    bias = (rng.standard_normal(N) * 0.01).astype(np.float32)
    L = _lib.lib()
    try:
        assert L.mllm_hip_w8a8_set_tuning(tile) == 0
        announce("w8a8 gemm", M, N, K, "tile", tile)
        y, acc = ql.w8a8_gemm(to_dev(xq), to_dev(xs), to_dev(W), to_dev(ws), None, want_acc=True)
        yb = ql.w8a8_gemm(to_dev(xq), to_dev(xs), to_dev(W), to_dev(ws), to_dev(bias))
    finally:
        L.mllm_hip_w8a8_set_tuning(0)
    wacc, wy = orc.w8a8_gemm(xq, xs, W, ws, None)
    _, wyb = orc.w8a8_gemm(xq, xs, W, ws, bias)
    assert np.array_equal(acc.cpu().numpy(), wacc)
    assert np.array_equal(_bits(y), wy)
    assert np.array_equal(_bits(yb), wyb)
    assert rel_l2(synth.bf16_bits_to_fp32(_bits(y)), synth.bf16_bits_to_fp32(wy)) <= 1e-3


def _pack_reference(W):
    """The packed layout restated with numpy: block (nb, kb) of 32 rows x 32 bytes, lane l = (row l%32, half l/32)."""
    N, K = W.shape
    Np, Kp = (N + 31) // 32 * 32, (K + 127) // 128 * 128
    Wp = np.zeros((Np, Kp), dtype=np.int8)
    Wp[:N, :K] = W
    # [nb][row][kb][half][16] -> [nb][kb][half][row][16]
    return Wp.reshape(Np // 32, 32, Kp // 32, 2, 16).transpose(0, 2, 3, 1, 4).reshape(-1)


# whatever form a shape takes (waves that split K, tiles of 64x128), ragged edges
PACKED_SHAPES = REF_SHAPES + [(300, 200, 48), (257, 193, 80), (1536, 6144, 256), (512, 9216, 128), (1024, 3072, 128),
                              (200, 800, 144)]


@pytest.mark.parametrize("M,N,K", PACKED_SHAPES)
def test_gemm_packed_bit_exact(M, N, K):
    rng = synth.rng_for(3, M * 11 + N + K)
    xq = rng.integers(-127, 128, (M, K), dtype=np.int8)
    W = rng.integers(-127, 128, (N, K), dtype=np.int8)
    xs = ((rng.random(M) + 0.01) * 0.01).astype(np.float32)
    ws = ((rng.random(N) + 0.01) * 0.01).astype(np.float32)
    bias = (rng.standard_normal(N) * 0.01).astype(np.float32)
    announce("w8a8 packed gemm", M, N, K)
    Wp = ql.w8a8_prepack(to_dev(W))
    assert np.array_equal(Wp.cpu().numpy().view(np.int8), _pack_reference(W))
    y, acc = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), None, want_acc=True)
    y1 = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), None)      # bf16 only: the fast store path
    yb = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), to_dev(bias))
    wacc, wy = orc.w8a8_gemm(xq, xs, W, ws, None)
    _, wyb = orc.w8a8_gemm(xq, xs, W, ws, bias)
    assert np.array_equal(acc.cpu().numpy(), wacc)
    assert np.array_equal(_bits(y), wy)
    assert np.array_equal(_bits(y1), wy)
    assert np.array_equal(_bits(yb), wyb)


@pytest.mark.parametrize("M,N,K", [(131, 200, 144), (257, 193, 80), (65, 1030, 16), (70, 392, 272), (33, 776, 1040), (300, 385, 384)])
@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5])
def test_gemm_packed_every_tile_bit_exact(tile, M, N, K):
    """each tile of the weights-from-global kernel at ragged rows and channels (N % 8 == 0: whole stores that the buffer's bound cuts; else
    by elements), one K step and an odd number of them; with and without the accumulators, with bias: the oracle's bits"""
    rng = synth.rng_for(3, 400 + M * 11 + N + K)
    xq = rng.integers(-127, 128, (M, K), dtype=np.int8)
    W = rng.integers(-127, 128, (N, K), dtype=np.int8)
    xs = ((rng.random(M) + 0.01) * 0.01).astype(np.float32)
    ws = ((rng.random(N) + 0.01) * 0.01).astype(np.float32)
    bias = (rng.standard_normal(N) * 0.01).astype(np.float32)
    announce("w8a8 packed tile", tile, M, N, K)
    Wp = ql.w8a8_prepack(to_dev(W))
    wacc, wy = orc.w8a8_gemm(xq, xs, W, ws, None)
    _, wyb = orc.w8a8_gemm(xq, xs, W, ws, bias)
    L = _lib.lib()
    try:
        assert L.mllm_hip_w8a8_nsplit_set_tuning(tile) == 0
        y, acc = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), None, want_acc=True)
        y1 = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), None)
        yb = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), to_dev(bias))
    finally:
        assert L.mllm_hip_w8a8_nsplit_set_tuning(0) == 0
    assert np.array_equal(acc.cpu().numpy(), wacc)
    assert np.array_equal(_bits(y), wy) and np.array_equal(_bits(y1), wy) and np.array_equal(_bits(yb), wyb)


@pytest.mark.parametrize("M,mfma_from", [(1, 5), (2, 5), (3, 5), (5, 33), (8, 33), (1, 1), (2, 2), (3, 2), (5, 5), (8, 5), (13, 5), (16, 5),
                                         (27, 5), (32, 5)])
def test_decode_gemv_packed_bit_exact(M, mfma_from):
    """up to 32 tokens take the GEMV kernels (a block row of the packed matrix per workgroup; dot instructions, or the matrix
    cores from `mfma_from` tokens): the oracle's bits, and the tile kernels' bits; ragged N and K (zero padding of the packed
    layout), rows long enough to pass through LDS in several runs, bias"""
    L = _lib.lib()
    assert L.mllm_hip_w8a8_set_decode_mfma_from(mfma_from) == 0
    try:
        _decode_gemv_cases(L, M)
    finally:
        assert L.mllm_hip_w8a8_set_decode_mfma_from(5) == 0
    assert L.mllm_hip_w8a8_set_decode_mfma_from(0) == -1 and L.mllm_hip_w8a8_set_decode_mfma_from(34) == -1


def _decode_gemv_cases(L, M):
    for N, K in ((9728, 2560), (2560, 9728), (77, 48), (200, 144), (33, 4096 + 16)):
        rng = synth.rng_for(3, 700 + M * 11 + N + K)
        xq = rng.integers(-127, 128, (M, K), dtype=np.int8)
        W = rng.integers(-127, 128, (N, K), dtype=np.int8)
        xs = ((rng.random(M) + 0.01) * 0.01).astype(np.float32)
        ws = ((rng.random(N) + 0.01) * 0.01).astype(np.float32)
        bias = (rng.standard_normal(N) * 0.01).astype(np.float32)
        announce("w8a8 decode gemv", M, N, K)
        Wp = ql.w8a8_prepack(to_dev(W))
        y, acc = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), None, want_acc=True)
        yb = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), to_dev(bias))
        wacc, wy = orc.w8a8_gemm(xq, xs, W, ws, None)
        _, wyb = orc.w8a8_gemm(xq, xs, W, ws, bias)
        assert np.array_equal(acc.cpu().numpy(), wacc)
        assert np.array_equal(_bits(y), wy) and np.array_equal(_bits(yb), wyb)
        assert L.mllm_hip_w8a8_set_decode(0) == 0
        try:
            yt = ql.w8a8_gemm_packed(to_dev(xq), to_dev(xs), Wp, N, to_dev(ws), to_dev(bias))
        finally:
            assert L.mllm_hip_w8a8_set_decode(1) == 0
        assert np.array_equal(_bits(yt), wyb)
    assert L.mllm_hip_w8a8_set_decode(2) == -1


def test_full_size_prefill():
    """A bf16 [2048,2048] with outliers, W int8 [6144,2048]: quantization bit-exact on every row; accumulators checked on a
    row sample against the oracle and on ALL rows through the column-sum identity
    sum_n acc[m][n] = sum_k xq[m][k] * (sum_n W[n][k])."""
    rng = synth.rng_for(3)
    M, N, K = 2048, 6144, 2048
    a_bits, W, ws = synth.make_w8a8(rng, M, N, K)
    announce("w8a8 full size")
    xd = bf16_dev(a_bits)
    Wd, wsd = to_dev(W), to_dev(ws)
    q, s = ql.per_token_quant_int8(xd)
    wq, wsc = orc.per_token_quant_int8(synth.bf16_bits_to_fp32(a_bits))
    assert np.array_equal(q.cpu().numpy(), wq) and np.array_equal(s.cpu().numpy(), wsc)
    y, acc = ql.w8a8_gemm(q, s, Wd, wsd, None, want_acc=True)
    acc = acc.cpu().numpy()
    colsum = W.astype(np.int64).sum(axis=0)
    assert np.array_equal(acc.astype(np.int64).sum(axis=1), wq.astype(np.int64) @ colsum)
    rows = np.sort(rng.choice(M, 48, replace=False))
    wacc, wy = orc.w8a8_gemm(wq[rows], wsc[rows], W, ws, None)
    assert np.array_equal(acc[rows], wacc)
    assert np.array_equal(_bits(y)[rows], wy)
    # the fused entry point (quantize + GEMM) gives the same bits
    y2 = ql.w8a8_linear(xd, Wd, wsd)
    assert torch.equal(y2.view(torch.int16), y.view(torch.int16))
    # and so does the prepacked-weight path, on every element
    Wp = ql.w8a8_prepack(Wd)
    y3, acc3 = ql.w8a8_gemm_packed(q, s, Wp, N, wsd, None, want_acc=True)
    assert np.array_equal(acc3.cpu().numpy(), acc)
    y4 = ql.w8a8_linear_packed(xd, Wp, N, wsd)
    assert torch.equal(y3.view(torch.int16), y.view(torch.int16))
    assert torch.equal(y4.view(torch.int16), y.view(torch.int16))


def test_argument_errors():
    L = _lib.lib()
    t = torch.zeros(64 * 64, dtype=torch.int8, device="cuda")
    f = torch.zeros(64, device="cuda")
    o = torch.zeros(64 * 64, dtype=torch.bfloat16, device="cuda")
    g = L.mllm_hip_w8a8_gemm
    assert g(t.data_ptr(), f.data_ptr(), t.data_ptr(), f.data_ptr(), None, o.data_ptr(), None, 64, 64, 40, None) == -2
    assert g(None, f.data_ptr(), t.data_ptr(), f.data_ptr(), None, o.data_ptr(), None, 64, 64, 64, None) == -1
    assert g(t.data_ptr(), f.data_ptr(), t.data_ptr(), f.data_ptr(), None, None, None, 64, 64, 64, None) == -1
    assert g(t.data_ptr() + 1, f.data_ptr(), t.data_ptr(), f.data_ptr(), None, o.data_ptr(), None, 8, 8, 64, None) == -3
    assert L.mllm_hip_per_token_quant_int8(None, 1, t.data_ptr(), f.data_ptr(), 4, 64, None) == -1
    assert L.mllm_hip_w8a8_set_tuning(9) == -1
    assert L.mllm_hip_w8a8_prepack(t.data_ptr(), 64, 40, o.data_ptr(), None) == -2
    assert L.mllm_hip_w8a8_prepack(None, 64, 64, o.data_ptr(), None) == -1
    assert L.mllm_hip_w8a8_packed_bytes(33, 130) == 64 * 256


@pytest.mark.parametrize("M", [5, 31, 33, 64, 97, 300])
def test_waves_that_split_k(M):
    """tiles of 32x32 whose waves split K (at most of these shapes; else 32x64, or 64x128 and whole K): ragged ends, fewer K blocks than waves,
    K blocks that do not divide among the waves, N not a multiple of 4 (element stores) and of 64; same bits as the
    oracle"""
    _waves_cases(((M, N, K) for N, K in ((40, 64), (40, 144), (193, 1104), (1030, 2560), (4100, 784), (256, 6160))))


def test_waves_that_split_k_of_larger_tiles():
    """tiles of 32x64 and of 64x64: ragged ends, N % 4 != 0, K blocks that do not divide"""
    small, large = ((70, 4100, 784), (33, 6002, 1104), (300, 1030, 2560), (31, 9001, 2560)), ((97, 4101, 2560), (65, 6002, 2560), (33, 9001, 2560), (120, 4101, 2576))
    assert [_lib.lib().mllm_hip_w8a8_packed_form(*s) for s in small + large] == [2] * 4 + [3] * 4
    _waves_cases(small + large)


def test_halves_of_k():
    """tiles of 64x128 and 128x128 that have a CU to themselves, by eight waves with half of K each: ragged rows and channels, an odd number of K
    steps (the second half has one less), N % 8 != 0 (element stores); beside them, by four, too few blocks of K and more than 256 tiles"""
    shapes = {(99, 4116, 704): (4, 1), (98, 4172, 640): (4, 0), (129, 3288, 704): (4, 1), (105, 4128, 640): (4, 0), (451, 4110, 640): (4, 0),
              (66, 5589, 832): (4, 1), (65, 5608, 832): (4, 1), (193, 8405, 768): (4, 0),
              (834, 3869, 1216): (5, 1), (833, 3872, 1216): (5, 1), (900, 3723, 1088): (5, 0), (841, 3984, 1088): (5, 0), (838, 4100, 704): (5, 0),
              (323, 8603, 1344): (5, 1), (327, 8592, 1344): (5, 1), (1163, 6408, 1216): (5, 0)}
    L = _lib.lib()
    assert {s: (L.mllm_hip_w8a8_packed_form(*s), L.mllm_hip_w8a8_packed_halves(*s)) for s in shapes} == shapes
    _waves_cases(shapes)


def _waves_cases(shapes):
    L = _lib.lib()
    for M, N, K in shapes:
        rng = synth.rng_for(3, 1300 + 3 * M + N + K)
        a_bits, W, w_scale = synth.make_w8a8(rng, M, N, K)
        bias = (rng.standard_normal(N) * 0.1).astype(np.float32)
        announce("w8a8 waves split K", M, N, K)
        q, s = ql.per_token_quant_int8(bf16_dev(a_bits))
        packed = ql.w8a8_prepack(to_dev(W))
        y, acc = ql.w8a8_gemm_packed(q, s, packed, N, to_dev(w_scale), to_dev(bias), want_acc=True)
        want = (q.cpu().numpy().astype(np.float64) @ W.astype(np.float64).T).astype(np.int64)  # exact
        assert np.array_equal(acc.cpu().numpy(), want)
        assert L.mllm_hip_w8a8_set_decode(0) == 0
        try:
            yt = ql.w8a8_gemm_packed(q, s, packed, N, to_dev(w_scale), to_dev(bias))
        finally:
            assert L.mllm_hip_w8a8_set_decode(1) == 0
        assert torch.equal(y.view(torch.int16), yt.view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (2, 33, 144), (3, 65, 1008), (4, 31, 1024), (1, 96, 8208), (2, 40, 16400), (4, 10240, 528),
                                   (3, 10272, 272), (4, 8, 38656), (4, 8, 38672)])
def test_linear_that_quantizes_beside_its_sums(M, N, K):
    """one to four tokens, quantized by every workgroup (the last four sizes: the most workgroups and one more, the longest tokens that LDS
    takes and one past them): the bits of quantizing in a launch of its own, with a row of zeros, one with a NaN, one with an infinity, one
    of ties, a tiny one, results over the tokens, fp32 and bf16"""
    rng = synth.rng_for(3, M * 5 + N + K)
    W = rng.integers(-127, 128, (N, K), dtype=np.int8)
    ws = to_dev(((rng.random(N) + 0.01) * 0.01).astype(np.float32))
    bias = to_dev((rng.standard_normal(N) * 0.01).astype(np.float32))
    Wp = ql.w8a8_prepack(to_dev(W))
    base = rng.standard_normal((M, K)).astype(np.float32)
    forms = {"plain": base.copy()}
    for name in ("zero", "nan", "inf", "ties", "tiny"):
        x = base.copy()
        if name == "zero": x[0] = 0
        if name == "nan": x[M - 1, K // 2] = np.nan
        if name == "inf": x[0, 0], x[0, K - 1] = -np.inf, np.inf
        if name == "ties": x[M - 1] = np.arange(K) % 255 * 0.5 - 63.5
        if name == "tiny": x[0] *= np.float32(1e-38)
        forms[name] = x
    for name, x in forms.items():
        for xd in (to_dev(x), to_dev(x).bfloat16()):
            announce("W8A8 Linear of few tokens", M, N, K, name, str(xd.dtype))
            q, s = ql.per_token_quant_int8(xd)
            for b in (None, bias):
                want = _bits(ql.w8a8_gemm_packed(q, s, Wp, N, ws, b))
                assert np.array_equal(_bits(ql.w8a8_linear_packed(xd, Wp, N, ws, b)), want)
            if N <= K:
                L, over = _lib.lib(), xd.clone()
                scratch = torch.empty(L.mllm_hip_w8a8_workspace_bytes(M, K), dtype=torch.uint8, device="cuda")
                torch.cuda.synchronize()
                assert L.mllm_hip_w8a8_linear_packed(over.data_ptr(), ql.F32 if xd.dtype == torch.float32 else ql.BF16, Wp.data_ptr(),
                                                     ws.data_ptr(), None, over.data_ptr(), M, N, K, scratch.data_ptr(), None) == 0
                torch.cuda.synchronize()
                assert np.array_equal(over.view(torch.int16).flatten()[:M * N].cpu().numpy().view(np.uint16).reshape(M, N),
                                      _bits(ql.w8a8_gemm_packed(q, s, Wp, N, ws, None)))
