"""GPU parity of the Q4_K / Q6_K Linear against the CPU oracle (which is pinned bit for bit against the compiled reference
kernels in tests/test_oracle_vs_reference.py).

Bars: Q8_K activation codes, scales and sums of 16, and dequantized weights bit-exact; fp32 outputs rel-L2 <= 1e-3 (the
integer part is exact, the fp32 accumulation order differs from the CPU's eight lanes; measured about 1e-7)."""
import numpy as np
import pytest
import torch

from mllm_amd import _lib, qlinear as ql, synth
from oracle import oracle as orc
from gpu_util import announce, bf16_dev, rel_l2, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-3


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_q8_K_quantization_bit_exact(dtype):
    rng = synth.rng_for(7, 1)
    M, K = 7, 2560
    if dtype == "bf16":
        bits, xf = synth.make_x_bf16(rng, M, K)
        x = bf16_dev(bits)
    else:
        xf = synth.make_x_fp32(rng, M, K) * 3
        xf[1, 256:512] = 0                       # an all-zero super-block
        xf[2, :256] = 0.1
        xf[2, 9], xf[2, 200] = -4.5, 4.5         # equal magnitudes, opposite signs: the first one decides
        xf[3, 512:768] = 0.25
        xf[3, 767] = -0.25                       # the LAST element differs in sign only
        xf[4, :256] = 0.1
        xf[4, 16], xf[4, 17] = 5.0, -5.0         # the tie inside one lane's eight elements, positive first
        xf[5, :256] = 0.1
        xf[5, 18], xf[5, 21] = -5.0, 5.0         # ... negative first
        xf[6, 256:512] = 0.1
        xf[6, 256 + 128], xf[6, 256 + 255] = 6.0, -6.0  # the tie across the two 16-lane rows of an odd super-block
        x = to_dev(xf)
    announce("q8_K quantization", dtype)
    q, d, bs = ql.quantize_q8_K(x)
    oq, od, obs = orc.quantize_rows_q8_K(xf)
    assert np.array_equal(q.cpu().numpy(), oq)
    assert np.array_equal(d.cpu().numpy().view(np.uint32), od.view(np.uint32))
    assert np.array_equal(bs.cpu().numpy(), obs)


def test_q8_K_quantization_signs_and_magnitudes():
    """super-blocks of every magnitude (also past the range of the reciprocal's estimate), of one sign, of zeros of both
    signs, with the largest magnitude in two places of either sign: in one lane's eight elements, in two lanes, in the two halves of sixteen
    lanes, next to a block that has no such pair"""
    rng = synth.rng_for(7, 2)
    x = rng.standard_normal((24, 512)).astype(np.float32)
    # from 128 / max_float = 3.8e-37 on: below it the scale 128 / amax is infinite and the reference's codes are no numbers
    x[:16] *= np.float32(10.0) ** np.array([-36, -34, -30, -25, -20, -19.2, -19, -10, -1, 5, 10, 19, 19.3, 20, 30, 37.5], np.float32)[:, None]
    x[16] = -np.abs(x[16])
    x[17] = np.abs(x[17])
    x[18, ::2], x[18, 1::2] = 0.0, -0.0
    for r, (a, b) in zip(range(19, 24), ((3, 5), (8, 250), (127, 128), (0, 255), (40, 41))):
        x[r, a], x[r, b] = 7.5, -7.5
        x[r, 256 + b], x[r, 256 + a] = (7.5, -7.5) if r % 2 else (9.5, -3.0)
    want = orc.quantize_rows_q8_K(x)
    announce("q8_K signs and magnitudes")
    for got, w in zip(ql.quantize_q8_K(to_dev(x)), want):
        got = got.cpu().numpy()
        assert np.array_equal(got.view(np.uint32) if got.dtype == np.float32 else got, w.view(np.uint32) if w.dtype == np.float32 else w)


@pytest.mark.parametrize("wtype", [2, 3])
def test_prepack_and_dequantize_bit_exact(wtype):
    rng = synth.rng_for(7, 10 + wtype)
    N, K = 37, 1280
    W = synth.make_weight(rng, wtype, N, K)
    announce("kq dequantize", wtype)
    w = ql.PackedKWeight(wtype, torch.from_numpy(W))
    assert np.array_equal(w.dequantize().cpu().numpy().view(np.uint32), orc.dequantize_k(W, wtype, orc.SCALE_IEEE).view(np.uint32))
    # blocks written by the x86 build: the fp16 fields hold the pattern as a NUMBER
    Wx = W.copy()
    for off in ((0, 2) if wtype == 2 else (208,)):
        pat = W[:, :, off:off + 2].copy().view(np.uint16).astype(np.float32)
        Wx[:, :, off:off + 2] = pat.astype(np.float16).view(np.uint16).reshape(N, -1, 1).view(np.uint8)
    wx = ql.PackedKWeight(wtype, torch.from_numpy(Wx), weight_scale_mode=ql.SCALE_X86_REF)
    assert np.array_equal(wx.dequantize().cpu().numpy().view(np.uint32), orc.dequantize_k(W, wtype, orc.SCALE_X86_REF).view(np.uint32))


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M,N,K", [(1, 256, 2560), (2, 100, 256), (3, 77, 768), (4, 512, 2048), (8, 130, 9728), (5, 31, 512),
                                   (11, 64, 1024), (20, 48, 2560)])
def test_linear_kq(wtype, M, N, K):
    rng = synth.rng_for(7, 100 + wtype * 1000 + M * 13 + N)
    W = synth.make_weight(rng, wtype, N, K)
    w = ql.PackedKWeight(wtype, torch.from_numpy(W))
    bias = rng.standard_normal(N).astype(np.float32)
    xf = synth.make_x_fp32(rng, M, K)
    announce("linear kq", wtype, M, N, K)
    y = ql.linear_kq(w, to_dev(xf)).cpu().numpy()
    assert rel_l2(y, orc.linear_kq(xf, W, wtype, None, orc.SCALE_X86_REF)) < 2e-6
    yb = ql.linear_kq(w, to_dev(xf), to_dev(bias)).cpu().numpy()
    assert rel_l2(yb, orc.linear_kq(xf, W, wtype, bias, orc.SCALE_X86_REF)) < 2e-6
    bits, xb = synth.make_x_bf16(rng, M, K)
    y2 = ql.linear_kq(w, bf16_dev(bits))
    assert rel_l2(y2.cpu().numpy(), orc.linear_kq(xb, W, wtype, None, orc.SCALE_X86_REF)) < 2e-6
    # with a workspace (x quantized once by its own kernel): the same bits
    ws = ql.kq_workspace(M, K)
    assert torch.equal(ql.linear_kq(w, to_dev(xf), to_dev(bias), workspace=ws), torch.from_numpy(yb).cuda())
    assert torch.equal(ql.linear_kq(w, bf16_dev(bits), workspace=ws), y2)


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M", [1, 4, 8, 13])
def test_linear_kq_multi_equals_single(wtype, M):
    """sibling projections in one launch: per part the bits of the single launch"""
    rng = synth.rng_for(7, 300 + wtype * 10 + M)
    K = 1280
    Ns = [96, 33, 200, 8]
    Ws = [synth.make_weight(rng, wtype, n, K) for n in Ns]
    ws = [ql.PackedKWeight(wtype, torch.from_numpy(W)) for W in Ws]
    biases = [to_dev(rng.standard_normal(n).astype(np.float32)) if i % 2 == 0 else None for i, n in enumerate(Ns)]
    x = to_dev(synth.make_x_fp32(rng, M, K))
    announce("kq multi", wtype, M)
    wsp = ql.kq_workspace(M, K)
    for nparts in (2, 4):
        outs = ql.linear_kq_multi(ws[:nparts], x, biases[:nparts], workspace=wsp if M % 2 else None)
        for w, b, o in zip(ws, biases, outs):
            assert torch.equal(o, ql.linear_kq(w, x, b))


@pytest.mark.parametrize("wtype", [2, 3])
def test_linear_kq_exact_cases(wtype):
    """unit scales and integer activations that quantize to themselves: every product is an integer below 2^24, so the
    result must equal the integer matrix product exactly"""
    rng = synth.rng_for(7, 50 + wtype)
    N, K, M = 64, 512, 4
    W = synth.make_weight(rng, wtype, N, K)
    if wtype == 2:
        W[:, :, 0:2] = np.array([0x00, 0x3c], np.uint8)
        W[:, :, 2:4] = np.array([0x00, 0x3c], np.uint8)
    else:
        W[:, :, 208:210] = np.array([0x00, 0x3c], np.uint8)
        W[:, :, 192:208] = rng.integers(-3, 4, size=(N, K // 256, 16)).astype(np.int8).view(np.uint8)
    x = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
    x[:, ::256] = -128.0  # max = -128 -> iscale = 1, d = 1: codes equal the values
    wd = orc.dequantize_k(W, wtype, orc.SCALE_IEEE).astype(np.float64)
    want = x.astype(np.float64) @ wd.T
    assert np.abs(want).max() < 2 ** 24
    announce("linear kq exact", wtype)
    y = ql.linear_kq(ql.PackedKWeight(wtype, torch.from_numpy(W)), to_dev(x)).cpu().numpy()
    assert np.array_equal(y.astype(np.float64), want)


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M,N,K", [(9, 100, 256), (64, 257, 768), (130, 512, 2560), (33, 31, 512), (300, 96, 9728), (512, 300, 1024)])
def test_linear_kq_gemm(wtype, M, N, K):
    """many rows on the matrix cores (fp16 operands with folded scales) against the oracle's integer / fp32 arithmetic"""
    rng = synth.rng_for(7, 700 + wtype * 1000 + M * 13 + N)
    W = synth.make_weight(rng, wtype, N, K)
    wg = ql.PackedKWeight(wtype, torch.from_numpy(W), layout="gemm")
    bias = rng.standard_normal(N).astype(np.float32)
    xf = synth.make_x_fp32(rng, M, K)
    announce("linear kq gemm", wtype, M, N, K)
    want = orc.linear_kq(xf, W, wtype, bias, orc.SCALE_X86_REF)
    y = ql.linear_kq_gemm(wg, to_dev(xf), to_dev(bias)).cpu().numpy()
    err = rel_l2(y, want)
    print("rel-L2 %.2e" % err)
    assert err < TOL
    bits, xb = synth.make_x_bf16(rng, M, K)
    y2 = ql.linear_kq_gemm(wg, bf16_dev(bits)).cpu().numpy()
    assert rel_l2(y2, orc.linear_kq(xb, W, wtype, None, orc.SCALE_X86_REF)) < TOL
    ys = ql.linear_kq_gemm(wg, to_dev(xf), to_dev(bias), short=True).cpu().numpy()  # K ranges as separate workgroups
    assert rel_l2(ys, y) < 2e-6
    # and against the GEMV path (the reference arithmetic itself) on the same device
    yv = ql.linear_kq(ql.PackedKWeight(wtype, torch.from_numpy(W)), to_dev(xf), to_dev(bias)).cpu().numpy()
    assert rel_l2(y, yv) < TOL


@pytest.mark.parametrize("wtype", [2, 3])
def test_linear_kq_gemm_exact_cases(wtype):
    """unit scales, small integer sub-block scales and integer activations that quantize to themselves: every operand is
    an integer that fp16 holds exactly and every partial sum stays below 2^24, so the result must equal the integer
    matrix product exactly (a misplaced code, scale or offset in the packed layout cannot pass)"""
    rng = synth.rng_for(7, 60 + wtype)
    N, K, M = 70, 768, 37
    W = synth.make_weight(rng, wtype, N, K)
    if wtype == 2:
        W[:, :, 0:2] = np.array([0x00, 0x3c], np.uint8)
        W[:, :, 2:4] = np.array([0x00, 0x3c], np.uint8)
    else:
        W[:, :, 208:210] = np.array([0x00, 0x3c], np.uint8)
        W[:, :, 192:208] = rng.integers(-3, 4, size=(N, K // 256, 16)).astype(np.int8).view(np.uint8)
    x = rng.integers(-3, 4, size=(M, K)).astype(np.float32)
    x[:, ::256] = -128.0  # max = -128 -> iscale = 1, d = 1: codes equal the values
    wd = orc.dequantize_k(W, wtype, orc.SCALE_IEEE).astype(np.float64)
    assert np.abs(wd).max() <= 2048
    want = x.astype(np.float64) @ wd.T
    assert (np.abs(x).astype(np.float64) @ np.abs(wd).T).max() < 2 ** 24
    announce("linear kq gemm exact", wtype)
    y = ql.linear_kq_gemm(ql.PackedKWeight(wtype, torch.from_numpy(W), layout="gemm"), to_dev(x)).cpu().numpy()
    assert np.array_equal(y.astype(np.float64), want)


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M", [3, 4, 5, 8, 11])
def test_matrix_core_and_dot4_kernels_agree(wtype, M):
    """three to eight rows: the matrix-core kernels (default) and the dot4 kernel are independent implementations of the same
    arithmetic (exact integer sums, fp32 scaling in another order)"""
    rng = synth.rng_for(7, 900 + M + 100 * wtype)
    L = _lib.lib()
    for N, K in ((9728, 2560), (2560, 9728), (77, 768), (130, 4096 + 256), (33, 256)):
        W = synth.make_weight(rng, wtype, N, K)
        w = ql.PackedKWeight(wtype, torch.from_numpy(W))
        bias = to_dev(rng.standard_normal(N).astype(np.float32))
        xf = synth.make_x_fp32(rng, M, K)
        xd = to_dev(xf)
        announce("kq both kernels", wtype, M, N, K)
        assert L.mllm_hip_kq_set_path(2) == 0  # the matrix-core kernel also where the default keeps the dot4 kernel
        try:
            y0 = ql.linear_kq(w, xd, bias)
            assert torch.equal(y0, ql.linear_kq(w, xd, bias, workspace=ql.kq_workspace(M, K)))
            assert L.mllm_hip_kq_set_path(1) == 0
            y1 = ql.linear_kq(w, xd, bias)
        finally:
            assert L.mllm_hip_kq_set_path(0) == 0
        yd = ql.linear_kq(w, xd, bias)  # whatever the default picks per group of eight rows: one of the two, bit for bit
        for lo in range(0, M, 8):
            assert torch.equal(yd[lo:lo + 8], y0[lo:lo + 8]) or torch.equal(yd[lo:lo + 8], y1[lo:lo + 8])
        assert rel_l2(y0.cpu().numpy(), y1.cpu().numpy()) < 2e-6
        assert rel_l2(y0.cpu().numpy(), orc.linear_kq(xf, W, wtype, bias.cpu().numpy(), orc.SCALE_X86_REF)) < 2e-6
    assert L.mllm_hip_kq_set_path(3) == -1


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M", [3, 4, 7, 8, 19])
def test_rows_give_the_same_bits_in_every_launch_shape(wtype, M):
    """the K slices of a tile meet in LDS in slice order: the same bits with any number of tiles per workgroup and of waves per tile
    (fewer than slices, as many, more), and with the quantized image in a workspace or without one.  Ragged N, several parts, bias, fp32
    and bf16 activations, the workspace used again and again, room beyond the image."""
    rng = synth.rng_for(7, 1300 + M + 50 * wtype)
    L = _lib.lib()
    for Ns, K in (((2560,), 9728), ((2560,), 4096), ((77, 130), 4096 + 256), ((33, 16, 50, 200), 3072), ((700, 90), 2560), ((40,), 256)):
        ws = [ql.PackedKWeight(wtype, torch.from_numpy(synth.make_weight(rng, wtype, N, K))) for N in Ns]
        biases = [to_dev(rng.standard_normal(N).astype(np.float32)) if i % 2 == 0 else None for i, N in enumerate(Ns)]
        xf = synth.make_x_fp32(rng, M, K)
        room = torch.empty(ql.kq_workspace(M, K).numel() + 1000, dtype=torch.uint8, device="cuda")
        for x in (to_dev(xf), to_dev(xf).to(torch.bfloat16)):
            announce("kq rows in every shape", wtype, M, Ns, K, x.dtype)
            want = ql.linear_kq_multi(ws, x, biases)
            try:
                for tiles, waves in ((0, 0), (1, 1), (1, 2), (1, 5), (1, 16), (2, 3), (2, 8), (3, 1), (4, 4), (5, 2), (8, 1), (8, 2)):
                    assert L.mllm_hip_kq_set_rows_shape(tiles, waves) == 0
                    for workspace in (None, room):
                        got = ql.linear_kq_multi(ws, x, biases, workspace=workspace)
                        assert all(torch.equal(a, c) for a, c in zip(want, got)), (tiles, waves, workspace is None)
            finally:
                assert L.mllm_hip_kq_set_rows_shape(0, 0) == 0
    # a workspace smaller than the image is an error, stated size or not
    p = ws[0].ptr
    part = (_lib.GemvPart * 1)(_lib.GemvPart(p, None, want[0].data_ptr(), 40))
    assert L.mllm_hip_linear_kq_multi_ws(wtype, 1, part, x.data_ptr(), ql._xdtype(x), M, 256, room.data_ptr(), 16, None) == -1
    # (checks its arguments and selects nothing)
    assert [L.mllm_hip_kq_set_slice_meeting(*v) for v in ((-1, 0), (1, 8), (2, 0), (0, 9))] == [0, 0, -1, -1]


@pytest.mark.parametrize("wtype", [2, 3])
@pytest.mark.parametrize("M,Ns,K", [(3, (1, 16, 17), 256), (4, (15,), 768), (8, (33,), 1024), (5, (4097, 33), 1280), (8, (16 * 1400 + 3,), 512), (6, (40,), 15872), (6, (90,), 6912),
                                    (7, (9, 70), 16128)])
def test_rows_kernel_edges(wtype, M, Ns, K):
    """three to eight rows: part and odd tiles of 16 channels, one to many tiles per workgroup, odd numbers of super-blocks, more waves
    than slices, the longest rows whose codes fit the LDS and the first that do not, with a workspace and without"""
    rng = synth.rng_for(7, 1700 + M + 50 * wtype)
    Ws = [synth.make_weight(rng, wtype, N, K) for N in Ns]
    ws = [ql.PackedKWeight(wtype, torch.from_numpy(W)) for W in Ws]
    xf = synth.make_x_fp32(rng, M, K)
    announce("kq rows", wtype, M, Ns, K)
    ys = ql.linear_kq_multi(ws, to_dev(xf))
    yw = ql.linear_kq_multi(ws, to_dev(xf), workspace=ql.kq_workspace(M, K))
    for W, y, y2 in zip(Ws, ys, yw):
        assert torch.equal(y, y2)
        assert rel_l2(y.cpu().numpy(), orc.linear_kq(xf, W, wtype, None, orc.SCALE_X86_REF)) < 2e-6


@pytest.mark.parametrize("wtype,H,I,T,E,k,shared,same_as", [
    # pairs one by one, pairs in groups of four (Q6_K, three to six super-blocks; gate / up, down or both), at the edges of that rule
    (2, 768, 1024, 16, 64, 2, 19, 1), (3, 2048, 768, 8, 64, 2, 0, 1), (3, 1024, 512, 11, 64, 2, 9, 1), (3, 1024, 2048, 4, 64, 4, 5, 1),
    ((2, 3), 2048, 768, 32, 256, 2, 21, 1), ((2, 3), 2048, 768, 63, 256, 1, 13, 1), ((3, 2), 768, 1024, 32, 256, 2, 21, 1), ((3, 3), 768, 1024, 31, 256, 2, 9, 1),  # (two tiles per wave, one)
    ((2, 3), 2048, 768, 9, 64, 3, 19, 1), ((2, 3), 2048, 1536, 31, 256, 4, 124, 1), ((3, 2), 1536, 1024, 15, 64, 2, 30, 1), (3, 1280, 1280, 13, 128, 2, 13, 1),
    # less than one pair per expert, with the sums of the sorted tiles
    (3, 256, 512, 20, 256, 8, 9, 2), ((2, 3), 512, 256, 17, 64, 3, 0, 2), ((3, 2), 1792, 256, 31, 128, 4, 124, 2)])
def test_moe_pairs_that_find_their_expert_group(wtype, H, I, T, E, k, shared, same_as):
    """MoE pairs whose workgroups find the pairs that share an expert give the bits of the form they stand in for: one GEMV row per
    pair (1) or the sorted tiles (2).  shared = how many slots name expert 3, so that some experts have one, exactly a group's,
    one more and many pairs; invalid ids among them; against the oracle"""
    wtype, wdown = wtype if isinstance(wtype, tuple) else (wtype, wtype)
    rng = synth.rng_for(9, 7300 + wtype + 5 * wdown + T + H + I + E)
    L = _lib.lib()
    Wg, Wu, Wd = (synth.make_weight(rng, wt, E * n, K).reshape(E, n, K // 256, -1) for wt, n, K in ((wtype, I, H), (wtype, I, H), (wdown, H, I)))
    g, u, d = (ql.PackedKExperts(wt, torch.from_numpy(W)) for wt, W in ((wtype, Wg), (wtype, Wu), (wdown, Wd)))
    ids = rng.integers(0, E, size=(T, k)).astype(np.int32)
    ids.reshape(-1)[:shared] = 3
    ids[T - 1, k - 1], ids[0, k - 1] = -1, E
    w = rng.random((T, k)).astype(np.float32)
    xf = synth.make_x_fp32(rng, T, H)
    bits, xb = synth.make_x_bf16(rng, T, H)
    announce("moe groups", wtype, wdown, H, I, T, E, k, shared)
    run = lambda: [ql.moe_ffn_kq(g, u, d, x, to_dev(ids), to_dev(w)) for x in (to_dev(xf), bf16_dev(bits))]  # noqa: E731
    y = run()
    assert L.mllm_hip_moe_kq_set_path(same_as) == 0
    try:
        y1 = run()
    finally:
        assert L.mllm_hip_moe_kq_set_path(0) == 0
    assert torch.equal(y[0], y1[0]) and torch.equal(y[1], y1[1])
    assert rel_l2(y[0].cpu().numpy(), orc.moe_ffn_kq(xf, ids, w, Wg, Wu, Wd, wtype, wtype_down=wdown)) < 1e-3


def _fma(a, b, c):
    """fp32 fma: the product is exact in 64 bits, the sum rounded there first (a tie of the second rounding: once in 2^29)"""
    a, b, c = (np.asarray(v, np.float64) for v in (a, b, c))
    return (a * b + c).astype(np.float32)


def _moe_tile_sums(x, W, wtype):
    """codes [M, K] x W [N, K/256, block] in the fp32 order of the MoE tiles (kquant_rows.h): every sub-block of 32 (Q6_K: unit of
    16) scaled on its own, a chain per lane group over a slice, lane groups pairwise, slices in order"""
    codes, d, _ = orc.quantize_rows_q8_K(x)
    (M, K), N = codes.shape, W.shape[0]
    nsb, f32 = K // 256, np.float32
    half = lambda a: np.ascontiguousarray(a).view(np.float16).astype(f32)[..., 0]  # noqa: E731
    if wtype == 2:
        sc12, qs, dw, dmin = W[:, :, 4:16].astype(np.int32), W[:, :, 16:144].reshape(N, nsb, 4, 32), half(W[:, :, 0:2]), half(W[:, :, 2:4])
        q = np.stack([qs & 15, qs >> 4], axis=3).reshape(N, nsb, 8, 32).astype(np.int32)
        lo, hi = sc12[:, :, 0:4], sc12[:, :, 4:8]
        sc = np.concatenate([lo & 63, (sc12[:, :, 8:] & 15) | ((lo >> 6) << 4)], axis=2)
        mn = np.concatenate([hi & 63, (sc12[:, :, 8:] >> 4) | ((hi >> 6) << 4)], axis=2)
        size, groups, steps = 32, 2, [(4 * j + h, 2) for j in range(2) for h in range(2)]  # sub-block of group 0, step to the next group's
    else:
        l, h = W[:, :, :128].reshape(N, nsb, 2, 2, 32).astype(np.int32), W[:, :, 128:192].reshape(N, nsb, 2, 32).astype(np.int32)
        sc, dw = W[:, :, 192:208].view(np.int8).astype(np.int32), half(W[:, :, 208:210])
        q = np.stack([(l[:, :, :, 0] & 15) | (h & 3) << 4, (l[:, :, :, 1] & 15) | (h >> 2 & 3) << 4, (l[:, :, :, 0] >> 4) | (h >> 4 & 3) << 4,
                      (l[:, :, :, 1] >> 4) | (h >> 6) << 4], axis=3).reshape(N, nsb, 16, 16) - 32
        size, groups, steps = 16, 4, [(8 * j + 4 * h, 1) for j in range(2) for h in range(2)]
    c = codes.astype(np.int32).reshape(M, nsb, 256 // size, size)
    D, X = np.einsum("nbse,mbse->bsmn", q, c), c.sum(-1)
    slices = 1
    while slices < 8 and nsb > 5 * slices:
        slices *= 2
    per, total = -(-nsb // slices), None
    for s in range(0, nsb, per):
        acc = [np.zeros((M, N), f32) for _ in range(groups)]
        for b in range(s, min(nsb, s + per)):
            dx = d[:, b, None]
            for first, stride in steps:
                for i in range(groups):
                    k = first + stride * i
                    acc[i] = _fma((dw[:, b] * sc[:, b, k].astype(f32)) * dx, D[b, k], acc[i])
                    if wtype == 2:
                        acc[i] = _fma(-((dmin[:, b] * mn[:, b, k].astype(f32)) * dx), X[:, b, k, None], acc[i])
        v = acc[0] + acc[1] if groups == 2 else (acc[0] + acc[1]) + (acc[2] + acc[3])
        total = v if total is None else total + v
    return total


@pytest.mark.parametrize("wtype,wdown,E,H,I", [(2, 2, 8, 2816, 512), (3, 3, 8, 2816, 512), (2, 3, 40, 1536, 512), (3, 2, 40, 512, 1536), (2, 3, 8, 512, 3584),
                                               (3, 2, 8, 4096, 256), (3, 2, 8, 512, 2048), (3, 2, 40, 4096, 512)])
def test_moe_tiles_keep_the_order_of_their_sums(wtype, wdown, E, H, I):
    """eight-row tiles (three pairs per expert and less), sorted (8 experts) and found by the workgroups (40), slices one after another and
    spread over waves: bit for bit the stated fp32 order, through SiLU, the second quantization and the weighted sum (one pair per token)"""
    T, rng = 24, synth.rng_for(9, 7500 + wtype + 5 * wdown + E)
    Wg, Wu, Wd = (synth.make_weight(rng, wt, E * n, K).reshape(E, n, K // 256, -1) for wt, n, K in ((wtype, I, H), (wtype, I, H), (wdown, H, I)))
    g, u, d = (ql.PackedKExperts(wt, torch.from_numpy(W)) for wt, W in ((wtype, Wg), (wtype, Wu), (wdown, Wd)))
    ids, w, x = rng.integers(0, E, size=(T, 1)).astype(np.int32), rng.random((T, 1)).astype(np.float32), synth.make_x_fp32(rng, T, H)
    announce("moe tile order", wtype, wdown, E, H, I)
    y = ql.moe_ffn_kq(g, u, d, to_dev(x), to_dev(ids), to_dev(w)).cpu().numpy()
    want = np.empty_like(y)
    for e in np.unique(ids):
        rows = np.nonzero(ids[:, 0] == e)[0]
        h = ql.silu_mul(to_dev(_moe_tile_sums(x[rows], Wg[e], wtype)), to_dev(_moe_tile_sums(x[rows], Wu[e], wtype))).cpu().numpy()
        want[rows] = _moe_tile_sums(h, Wd[e], wdown) * w[rows]
    assert np.array_equal(y, want)


@pytest.mark.parametrize("wtype", [2, 3])
def test_units_in_flight_do_not_change_the_bits(wtype):
    """one or two rows: a lane adds its units in the same order whether the row is requested whole before the quantization of
    x (the default for Q4_K rows of up to 96 / 128 units) or trip by trip (mllm_hip_kq_set_tuning with units in flight)"""
    rng = synth.rng_for(7, 1500 + wtype)
    L = _lib.lib()
    for M in (1, 2):
        for N, K in ((1000, 2560), (300, 4096), (70, 768), (2560, 2560 + 512)):
            w = ql.PackedKWeight(wtype, torch.from_numpy(synth.make_weight(rng, wtype, N, K)))
            x = to_dev(synth.make_x_fp32(rng, M, K)).to(torch.bfloat16)
            announce("kq units in flight", wtype, M, N, K)
            want = ql.linear_kq(w, x)
            try:
                for u in (1, 2, 4):
                    assert L.mllm_hip_kq_set_tuning(0, 0, u) == 0
                    assert torch.equal(want, ql.linear_kq(w, x)), u
            finally:
                assert L.mllm_hip_kq_set_tuning(0, 0, 0) == 0


@pytest.mark.parametrize("M,N,K", [(1, 300, 5120), (1, 300, 5376), (2, 70, 7936), (2, 70, 8192), (1, 33, 10240), (1, 33, 10496), (2, 130, 14592), (1, 130, 18944)])
def test_whole_trips_ahead_do_not_change_the_bits(M, N, K):
    """long Q4_K rows in the large workgroups: a second set of registers for the next trip, either side of the lengths that keep the ring, against
    the ring (the units in flight stated)"""
    rng = synth.rng_for(7, 1700 + N + K)
    L = _lib.lib()
    w = ql.PackedKWeight(2, torch.from_numpy(synth.make_weight(rng, 2, N, K)))
    x = to_dev(synth.make_x_fp32(rng, M, K))
    announce("kq trips ahead", M, N, K)
    want = ql.linear_kq(w, x)
    assert torch.isfinite(want).all() and want.abs().max() > 0
    try:
        assert L.mllm_hip_kq_set_tuning(0, 0, 4) == 0
        assert torch.equal(want, ql.linear_kq(w, x))
    finally:
        assert L.mllm_hip_kq_set_tuning(0, 0, 0) == 0


def _graph_time(call, n=24):
    """median of nine replays of call(0) .. call(n - 1), in us per call"""
    call(0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for i in range(n):
            call(i)
    times = []
    for _ in range(11):
        first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        first.record()
        graph.replay()
        last.record()
        torch.cuda.synchronize()
        times.append(first.elapsed_time(last) * 1e3 / n)
    return sorted(times[2:])[4]


def test_long_q4_k_rows_are_requested_a_trip_ahead():
    """1552 x 7936, one row, weights that no cache of an XCD holds: 6.8 us, by the ring 8.1.  A bound with room for other noise"""
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(1)
    ws = [ql.PackedKWeight.synthetic(2, 1552, 7936, g) for _ in range(8)]
    x, y = torch.randn((1, 7936), device="cuda", generator=g), torch.empty((1, 1552), device="cuda")
    announce("kq trips ahead, time")
    ahead = _graph_time(lambda i: ql.linear_kq(ws[i % 8], x, out=y))
    try:
        assert L.mllm_hip_kq_set_tuning(0, 0, 4) == 0
        assert ahead <= 0.93 * _graph_time(lambda i: ql.linear_kq(ws[i % 8], x, out=y))
    finally:
        assert L.mllm_hip_kq_set_tuning(0, 0, 0) == 0


@pytest.mark.parametrize("wtype,H", [(2, 512), (2, 768), (2, 1024), (2, 1280), (2, 2048), (2, 2304), (2, 2560), (2, 3072), (3, 1024), (3, 1280), (3, 2048), (3, 2304), (3, 4096)])
def test_units_in_flight_of_expert_pairs_do_not_change_the_bits(wtype, H):
    """a token's experts, a GEMV row per pair with sixteen lanes: rows whose units fit one or two per lane, Q4_K four at a time and beyond that a whole trip ahead,
    Q6_K the ring of two, the last trip partly filled among them, against one unit at a time (mllm_hip_kq_set_tuning).  Eight pairs of 768 rows: more workgroups
    than the form for few rows takes"""
    I, E, k = 768, 8, 8
    rng = synth.rng_for(9, 7900 + wtype + H)
    L = _lib.lib()
    Wg, Wu = (synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1) for _ in range(2))
    Wd = synth.make_weight(rng, wtype, E * H, I).reshape(E, H, I // 256, -1)
    g, u, d = (ql.PackedKExperts(wtype, torch.from_numpy(W)) for W in (Wg, Wu, Wd))
    ids, w = synth.make_moe_routing(rng, 1, E, k)
    ids, w, x = to_dev(ids), to_dev(w), to_dev(synth.make_x_fp32(rng, 1, H))
    announce("moe k-quant pairs, units in flight", wtype, H, I)
    try:
        assert L.mllm_hip_moe_kq_set_path(1) == 0  # (eight pairs of eight experts of Q6_K are tiles otherwise)
        want = ql.moe_ffn_kq(g, u, d, x, ids, w)
        assert torch.isfinite(want).all() and want.abs().max() > 0
        assert L.mllm_hip_kq_set_tuning(0, 0, 1) == 0
        assert torch.equal(want, ql.moe_ffn_kq(g, u, d, x, ids, w))
    finally:
        assert L.mllm_hip_kq_set_tuning(0, 0, 0) == 0 and L.mllm_hip_moe_kq_set_path(0) == 0


def test_expert_pairs_of_long_q4_k_rows_are_requested_a_trip_ahead():
    """eight experts of 2560 x 3072, one token of all eight: 30.9 us, four units at a time by the ring 34.0.  A bound with room for other noise"""
    L = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(1)
    g, u, d = (ql.PackedKExperts.synthetic(2, 8, n, k, gen) for n, k in ((3072, 2560), (3072, 2560), (2560, 3072)))
    ids, w = synth.make_moe_routing(synth.rng_for(9, 1), 1, 8, 8)
    ids, w, x = to_dev(ids), to_dev(w), torch.randn((1, 2560), device="cuda", generator=gen)
    y, ws = torch.empty_like(x), torch.empty(L.mllm_hip_moe_kq_workspace_bytes(1, 2560, 3072, 8, 8), dtype=torch.uint8, device="cuda")
    call = lambda i: ql.moe_ffn_kq(g, u, d, x, ids, w, workspace=ws, out=y)  # noqa: E731
    announce("moe k-quant pairs, time")
    ahead = _graph_time(call)
    try:
        assert L.mllm_hip_kq_set_tuning(0, 0, 4) == 0
        assert ahead <= 0.96 * _graph_time(call)
    finally:
        assert L.mllm_hip_kq_set_tuning(0, 0, 0) == 0


def test_argument_checks():
    L = _lib.lib()
    buf = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    p = buf.data_ptr()
    assert L.mllm_hip_kq_packed_bytes(2, 4, 100) == 0
    assert L.mllm_hip_kq_packed_bytes(0, 4, 256) == 0
    assert L.mllm_hip_linear_kq(2, p, p, 0, None, p, 1, 4, 100, None, None) == -2
    assert L.mllm_hip_linear_kq(1, p, p, 0, None, p, 1, 4, 256, None, None) == -1
    assert L.mllm_hip_linear_kq(2, p + 16, p, 0, None, p, 1, 4, 256, None, None) == -3
    assert L.mllm_hip_kq_prepack(3, None, 0, p, 4, 256, None) == -1
    assert L.mllm_hip_quantize_q8_K(p, 0, p, p, p, 1, 100, None) == -2
    assert L.mllm_hip_kq_gemm_packed_bytes(2, 4, 100) == 0
    assert L.mllm_hip_kq_gemm_packed_bytes(1, 4, 256) == 0
    assert L.mllm_hip_kq_gemm_packed_bytes(2, 33, 256) == 64 * 256 // 2 + 64 * 4 * 8
    assert L.mllm_hip_linear_kq_gemm(2, p, p, 0, None, p, 16, 4, 100, p, None) == -2
    assert L.mllm_hip_linear_kq_gemm(0, p, p, 0, None, p, 16, 4, 256, p, None) == -1
    assert L.mllm_hip_linear_kq_gemm(2, p, p, 0, None, p, 16, 4, 256, None, None) == -1


@pytest.mark.parametrize("name,wtype", [("q4_k", 2), ("q6_k", 3)])
def test_golden_kquant(golden_dir, name, wtype):
    """against what the compiled reference produced on blocks written by its own offline quantizers"""
    import os
    g = np.load(os.path.join(golden_dir, "kquant_kat.npz"))
    announce("golden kquant", name)
    w = ql.PackedKWeight(wtype, torch.from_numpy(g[f"{name}_W"]))
    assert np.array_equal(w.dequantize().cpu().numpy().view(np.uint32), g[f"{name}_deq"].view(np.uint32))
    for M in (1, 3, 8):
        y = ql.linear_kq(w, to_dev(g[f"{name}_x{M}"]), to_dev(g[f"{name}_bias"])).cpu().numpy()
        assert rel_l2(y, g[f"{name}_y{M}"]) < 1e-5
    q, d, bs = ql.quantize_q8_K(to_dev(g["q8k_x"]))
    assert np.array_equal(q.cpu().numpy(), g["q8k_q"]) and np.array_equal(d.cpu().numpy().view(np.uint32), g["q8k_d"].view(np.uint32))
    assert np.array_equal(bs.cpu().numpy(), g["q8k_bsums"])


@pytest.mark.parametrize("wtype,T,H,I,E,k", [(2, 1, 2048, 768, 16, 8), (3, 1, 2048, 768, 16, 8), (2, 5, 512, 256, 6, 3), (3, 9, 256, 512, 4, 2),
                                            (2, 8, 2048, 768, 128, 8)])
def test_moe_ffn_with_k_quant_experts(wtype, T, H, I, E, k):
    """Q4_K / Q6_K experts (Qwen3-30B-A3B dimensions included): every (token, expert) pair one K-quant GEMV row, SiLU and product,
    down GEMV, weighted sum in slot order, against the oracle's composition of the same Linears; slots with an expert id
    outside [0, E) add nothing; permuting tokens permutes outputs bit for bit; bf16 activations"""
    rng = synth.rng_for(9, 7000 + wtype + T + H + I + E)
    Wg = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wu = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wd = synth.make_weight(rng, wtype, E * H, I).reshape(E, H, I // 256, -1)
    ids, w = synth.make_moe_routing(rng, T, E, k)
    g, u, d = (ql.PackedKExperts(wtype, torch.from_numpy(W)) for W in (Wg, Wu, Wd))
    x = synth.make_x_fp32(rng, T, H)
    announce("moe k-quant", wtype, T, H, I, E, k)
    y = ql.moe_ffn_kq(g, u, d, to_dev(x), to_dev(ids), to_dev(w)).cpu().numpy()
    want = orc.moe_ffn_kq(x, ids, w, Wg, Wu, Wd, wtype)
    assert rel_l2(y, want) < 1e-3, rel_l2(y, want)
    perm = rng.permutation(T)
    y2 = ql.moe_ffn_kq(g, u, d, to_dev(x[perm]), to_dev(ids[perm]), to_dev(w[perm])).cpu().numpy()
    assert np.array_equal(y2, y[perm])
    bad = ids.copy()
    bad[0, 0] = E + 3
    if k > 1:
        bad[T - 1, k - 1] = -1
    y3 = ql.moe_ffn_kq(g, u, d, to_dev(x), to_dev(bad), to_dev(w)).cpu().numpy()
    assert rel_l2(y3, orc.moe_ffn_kq(x, bad, w, Wg, Wu, Wd, wtype)) < 1e-3
    bits, xb = synth.make_x_bf16(rng, T, H)
    y4 = ql.moe_ffn_kq(g, u, d, bf16_dev(bits), to_dev(ids), to_dev(w)).cpu().numpy()
    assert rel_l2(y4, orc.moe_ffn_kq(xb, ids, w, Wg, Wu, Wd, wtype)) < 1e-3


@pytest.mark.parametrize("wtype,T,H,I,E,k", [(2, 40, 512, 256, 6, 3), (3, 33, 256, 512, 4, 2), (2, 96, 2048, 768, 16, 4),
                                            (3, 64, 2048, 768, 8, 2), (2, 9, 256, 256, 3, 1)])
def test_moe_ffn_k_quant_grouped_form_equals_the_pair_form(wtype, T, H, I, E, k):
    """Many pairs per expert: the pairs sorted by expert run as tiles of eight rows on the matrix-core kernels (x and h
    quantized to Q8_K once, tiles gather their rows).  Same arithmetic as one GEMV row per pair (exact integer sums, fp32
    scaling in another order): the two forms agree to 1e-5, both meet the oracle; invalid expert ids add nothing; a permutation
    of the tokens permutes the outputs bit for bit; bf16 activations."""
    rng = synth.rng_for(9, 7100 + wtype + T + H + I + E)
    L = _lib.lib()
    Wg = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wu = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wd = synth.make_weight(rng, wtype, E * H, I).reshape(E, H, I // 256, -1)
    ids, w = synth.make_moe_routing(rng, T, E, k)
    ids[1, 0] = E + 2          # an expert id out of range
    if k > 1:
        ids[T - 1, k - 1] = -1
    g, u, d = (ql.PackedKExperts(wtype, torch.from_numpy(W)) for W in (Wg, Wu, Wd))
    x = synth.make_x_fp32(rng, T, H)
    announce("moe k-quant grouped", wtype, T, H, I, E, k)
    outs = {}
    for path in (1, 2):
        assert L.mllm_hip_moe_kq_set_path(path) == 0
        try:
            outs[path] = ql.moe_ffn_kq(g, u, d, to_dev(x), to_dev(ids), to_dev(w)).cpu().numpy()
            if path == 2:
                perm = rng.permutation(T)
                y2 = ql.moe_ffn_kq(g, u, d, to_dev(x[perm]), to_dev(ids[perm]), to_dev(w[perm])).cpu().numpy()
                bits, xb = synth.make_x_bf16(rng, T, H)
                y4 = ql.moe_ffn_kq(g, u, d, bf16_dev(bits), to_dev(ids), to_dev(w)).cpu().numpy()
        finally:
            assert L.mllm_hip_moe_kq_set_path(0) == 0
    want = orc.moe_ffn_kq(x, ids, w, Wg, Wu, Wd, wtype)
    assert rel_l2(outs[2], want) < 1e-3, rel_l2(outs[2], want)
    assert rel_l2(outs[2], outs[1]) < 1e-5, rel_l2(outs[2], outs[1])
    assert np.array_equal(y2, outs[2][perm])
    assert rel_l2(y4, orc.moe_ffn_kq(xb, ids, w, Wg, Wu, Wd, wtype)) < 1e-3
    assert L.mllm_hip_moe_kq_set_path(4) == -1


@pytest.mark.parametrize("wtype,T,H,I,E,k", [(2, 40, 512, 256, 6, 3), (2, 96, 2048, 768, 16, 4), (2, 200, 1024, 512, 5, 2),
                                            (2, 33, 256, 256, 1, 1), (2, 70, 768, 2048, 9, 4), (2, 300, 256, 512, 64, 8),
                                            (3, 40, 512, 256, 6, 3), (3, 96, 2048, 768, 16, 4), (3, 33, 256, 256, 1, 1),
                                            (3, 70, 768, 2048, 9, 4), ((2, 3), 96, 2048, 768, 16, 4), ((2, 3), 200, 512, 256, 5, 2),
                                            ((3, 2), 64, 256, 512, 4, 2)])
def test_moe_ffn_k_quant_tiles_of_32_rows(wtype, T, H, I, E, k):
    """Four pairs per expert and more: tiles of 32 expert-sorted rows, the weights as the second operand of 32 x 32 matrix
    instructions, integer sub-block sums scaled in int32 (experts with one row, 32, 33 rows, none at all; channel counts that
    end inside a workgroup's 128 or 256).  Same integers as one GEMV row per pair, fp32 scaling in another order: the forms
    agree row by row (see below) and meet the oracle; invalid expert ids add nothing; a permutation of the tokens permutes the outputs bit
    for bit; bf16 activations.  Q6_K: groups of 16 elements on 32 x 32 x 16 instructions, the offset of 32 through the sums
    of 16.  A pair of formats: gate / up in the first, down in the second (the shipped recipe is Q4_K / Q6_K)."""
    wtype, wdown = wtype if isinstance(wtype, tuple) else (wtype, wtype)
    rng = synth.rng_for(9, 7300 + wtype + 5 * wdown + T + H + I + E)
    L = _lib.lib()
    Wg = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wu = synth.make_weight(rng, wtype, E * I, H).reshape(E, I, H // 256, -1)
    Wd = synth.make_weight(rng, wdown, E * H, I).reshape(E, H, I // 256, -1)
    ids, w = synth.make_moe_routing(rng, T, E, k)
    if E > 2:
        ids[1, 0] = E + 2          # an expert id out of range
        if k > 1:
            ids[T - 1, k - 1] = -1
    g, u = (ql.PackedKExperts(wtype, torch.from_numpy(W)) for W in (Wg, Wu))
    d = ql.PackedKExperts(wdown, torch.from_numpy(Wd))
    x = synth.make_x_fp32(rng, T, H)
    announce("moe k-quant tiles of 32 rows", wtype, T, H, I, E, k)
    outs = {}
    for path in (1, 3):
        assert L.mllm_hip_moe_kq_set_path(path) == 0
        try:
            outs[path] = ql.moe_ffn_kq(g, u, d, to_dev(x), to_dev(ids), to_dev(w)).cpu().numpy()
            if path == 3:
                perm = rng.permutation(T)
                y2 = ql.moe_ffn_kq(g, u, d, to_dev(x[perm]), to_dev(ids[perm]), to_dev(w[perm])).cpu().numpy()
                bits, xb = synth.make_x_bf16(rng, T, H)
                y4 = ql.moe_ffn_kq(g, u, d, bf16_dev(bits), to_dev(ids), to_dev(w)).cpu().numpy()
        finally:
            assert L.mllm_hip_moe_kq_set_path(0) == 0
    want = orc.moe_ffn_kq(x, ids, w, Wg, Wu, Wd, wtype, wtype_down=wdown)
    assert rel_l2(outs[3], want) < 1e-3, rel_l2(outs[3], want)
    # row by row against the pair form: the same integers, fp32 sums in another order (about 2e-7); where the last bit of an h
    # value decides a Q8_K code, that one row of the down projection moves by a code step (a few 1e-4 of the row)
    rows = np.linalg.norm(outs[3] - outs[1], axis=1) / np.maximum(np.linalg.norm(outs[1], axis=1), 1e-30)
    assert np.median(rows) < 1e-6 and (rows > 1e-5).mean() <= 0.05 and rel_l2(outs[3], outs[1]) < 2e-4, (np.median(rows), rows.max())
    assert np.array_equal(y2, outs[3][perm])
    assert rel_l2(y4, orc.moe_ffn_kq(xb, ids, w, Wg, Wu, Wd, wtype, wtype_down=wdown)) < 1e-3


def _x86_field_to_pattern(field):
    """what a read on x86 makes of a stored fp16 field: the half-precision number, as an integer"""
    return field.view(np.float16).astype(np.float32).astype(np.uint16)


@pytest.mark.parametrize("wtype", [2, 3])
def test_offline_k_quant_quantizers_byte_exact(wtype, golden_dir):
    """mllm_hip_kq_quantize_weight_blocks against the oracle (pinned byte for byte to the compiled reference quantizers) in both
    storage modes, against the fixture the compiled reference wrote, and through the library's own Linear."""
    import os
    rng = synth.rng_for(7, 300 + wtype)
    N, K = 48, 1024
    w = (rng.standard_normal((N, K)) * 0.04).astype(np.float32)
    w[0, :256] = 0.0
    w[1, :32], w[1, 32:64] = 0.3, -0.3
    w[2, :256] = np.abs(w[2, :256])
    w[3, :512] *= 80
    w[4, :16] = 0.0
    w[5, :256] = np.float32(1e-3) * rng.integers(-8, 8, 256)
    w[6, 0], w[6, 5] = 0.9, -0.9
    w[7, :] = 1e-20                                      # below the all-zero threshold of the Q6_K search, not of the Q4_K one
    announce("offline k-quant quantizer", wtype)
    for mode, omode in ((ql.SCALE_X86_REF, orc.SCALE_X86_REF), (ql.SCALE_IEEE, orc.SCALE_IEEE)):
        got = ql.kq_quantize_weight_blocks(to_dev(w), wtype, mode).cpu().numpy()
        want = orc.quantize_weight_rows_k(w, wtype, omode)
        assert np.array_equal(got, want), (mode, np.argwhere(got != want)[:5])
    # the fixture of the compiled reference: codes and sub-block scales byte for byte, the fp16 fields as an x86 read decodes them
    g = np.load(os.path.join(golden_dir, "kquant_quantizer_kat.npz"))
    ref = g["q4_k_blocks" if wtype == 2 else "q6_k_blocks"]
    gb = ql.kq_quantize_weight_blocks(to_dev(g["w"]), wtype, ql.SCALE_X86_REF).cpu().numpy()
    body = np.ones(gb.shape[2], bool)
    for a, b in ([(0, 2), (2, 4)] if wtype == 2 else [(208, 210)]):
        body[a:b] = False
        assert np.array_equal(_x86_field_to_pattern(gb[:, :, a:b].copy().view(np.uint16)[:, :, 0]), ref[:, :, a:b].copy().view(np.uint16)[:, :, 0])
    assert np.array_equal(gb[:, :, body], ref[:, :, body])
    # quantize -> prepack -> Linear on the GPU equals the oracle's Linear on the oracle's blocks
    blocks = ql.kq_quantize_weight_blocks(to_dev(w), wtype, ql.SCALE_IEEE)
    pw = ql.PackedKWeight(wtype, blocks)
    x = synth.make_x_fp32(rng, 3, K)
    y = ql.linear_kq(pw, to_dev(x)).cpu().numpy()
    assert rel_l2(y, orc.linear_kq(x, orc.quantize_weight_rows_k(w, wtype, orc.SCALE_IEEE), wtype, None, orc.SCALE_IEEE)) < 2e-6
    # and the blocks reproduce the weights to the format's resolution
    deq = pw.dequantize().cpu().numpy()
    assert np.abs(deq - w).max() <= (0.08 if wtype == 2 else 0.05) * np.abs(w).max()
    L = _lib.lib()
    p = blocks.data_ptr()
    assert L.mllm_hip_kq_quantize_weight_blocks(wtype, None, p, 0, 4, 256, None) == -1
    assert L.mllm_hip_kq_quantize_weight_blocks(0, p, p, 0, 4, 256, None) == -1
    assert L.mllm_hip_kq_quantize_weight_blocks(wtype, p, p, 2, 4, 256, None) == -1
    assert L.mllm_hip_kq_quantize_weight_blocks(wtype, p, p, 0, 4, 128, None) == -2
    assert L.mllm_hip_kq_quantize_weight_blocks(wtype, p + 4, p, 0, 4, 256, None) == -3
