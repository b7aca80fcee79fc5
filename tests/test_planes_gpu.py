"""fp32 activations on FP4-KM weights with E2M1 values (two fp16 planes where the products are halves, three
bf16 terms on E8M0 scales), half weights and Q4 weights (two planes) on the MI355X against the oracle, at
the edges of the tiles and of the table's scales.

Bar: the reference test's tolerance (max|diff| <= 1e-4 * max(1, peak)); infinities and NaNs where the
oracle has them.
"""
import numpy as np
import pytest

from parity import ref_check

pytestmark = pytest.mark.gpu

SHAPES = [(1, 128, 16), (16, 256, 128), (17, 384, 130), (33, 1280, 129), (48, 1024, 264), (64, 2048, 127), (65, 640, 300),
          (130, 1152, 520)]


def fp4_case(M, K, N, scales, seed):
    from bybylang_amd import synth
    g = synth.rng(seed)
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    t = np.zeros(272, np.float32)
    t[:16] = synth.E2M1
    i = np.arange(256)
    with np.errstate(over="ignore"):
        t[16:] = np.ldexp(np.float32(1), i - 127) if scales != "ref" else (1 + i % 13) / 64
    sb = {"ref": g.integers(0, 256, (N, K // 32)), "mx": g.integers(104, 141, (N, K // 32)),
          "edge": g.integers(100, 150, (N, K // 32)), "one": g.integers(120, 130, (N, K // 32))}[scales].astype(np.uint8)
    if scales == "one":
        sb[N // 2, (K // 32) // 2] = 150  # one scale past the halves
    x = synth.activations(g, M, K, np.float32)
    return x, np.concatenate([synth.fp4km_pack(codes).reshape(-1), sb.reshape(-1)]), t


def run_fp4(hip, x, blob, t, M, K, N, mirror):
    """With a host copy of the table the host chooses the route, without one the device does."""
    import ctypes as C
    from bybylang_amd import _abi
    y = hip.DeviceBuffer(M * N * 4)
    lut = hip.DeviceBuffer.from_array(t)
    p = C.c_void_p()
    if mirror:
        _abi.check(_abi.load().byhip_session_upload(t.ctypes.data, t.size, C.byref(p)))
    bd, xd = hip.DeviceBuffer.from_array(blob), hip.DeviceBuffer.from_array(x.reshape(-1))
    _abi.check(_abi.load().byhip_fp4km_tile_gemm(xd.ptr, hip.F32, bd.ptr, bd.nbytes, N * (K // 2), p.value or lut.ptr, 272, 0,
                                                 y.ptr, hip.F32, M, K, N))
    out = y.read(np.float32)
    if mirror:
        _abi.check(_abi.load().byhip_session_free(p))
    return out


@pytest.mark.parametrize("mirror", [True, False])
@pytest.mark.parametrize("scales", ["ref", "mx", "edge", "one"])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_fp4km_planes(hip, oracle, M, K, N, scales, mirror):
    x, blob, t = fp4_case(M, K, N, scales, M + K + N)
    want = oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t, x)
    ref_check(run_fp4(hip, x, blob, t, M, K, N, mirror), want)


@pytest.mark.parametrize("splits", [2, 3])
def test_fp4km_planes_split_k(hip, oracle, monkeypatch, splits):
    M, K, N = 70, 1408, 200
    x, blob, t = fp4_case(M, K, N, "one", 5)
    monkeypatch.setenv("BYHIP_Q4_SPLIT", str(splits))
    want = oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t, x)
    ref_check(run_fp4(hip, x, blob, t, M, K, N, True), want)


def test_fp4km_planes_other_table_and_nonfinite(hip, oracle):
    """A table that is not E2M1, the same table through both choices of the route, and scales and
    activations that are not finite: finite where the oracle is, with its infinities and NaNs."""
    M, K, N = 20, 256, 130
    x, blob, t = fp4_case(M, K, N, "mx", 9)
    t2 = t.copy()
    t2[1] = 0.75
    want = oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t2, x)
    for mirror in (True, False):
        ref_check(run_fp4(hip, x, blob, t2, M, K, N, mirror), want)
    sb = blob[N * (K // 2):].reshape(N, K // 32)
    sb[3, 1] = 255                  # infinite scale: NaN where a code is 0 or signs differ
    x[5, 40] = np.inf               # an infinite activation
    x[6, 7] = np.nan
    want = np.asarray(oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t, x)).reshape(-1)
    for mirror in (True, False):
        got = run_fp4(hip, x, blob, t, M, K, N, mirror)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isinf(got), np.isinf(want))
        fin = np.isfinite(want)
        assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
        ref_check(got[fin], want[fin])


def test_planes_in_row_blocks(hip, oracle):
    """More rows than the scratch holds planes for: the rows go in blocks."""
    M, K, N = 1200, 4096, 48        # 19.7 MB of planes against half of 32 MB
    x, blob, t = fp4_case(M, K, N, "ref", 11)
    got = run_fp4(hip, x, blob, t, M, K, N, True).reshape(M, N)
    for r in (0, 959, 960, 1023, 1024, 1199):
        want = oracle.tile_gemm(0, 1, K, N, N * (K // 2), 0, blob, t, x[r])
        ref_check(got[r], want)


@pytest.mark.parametrize("M,K,N", [(1, 64, 16), (16, 192, 128), (20, 320, 130), (40, 1088, 129), (64, 640, 264), (130, 1152, 520)])
def test_f16_planes(hip, oracle, M, K, N):
    from bybylang_amd import synth
    g = synth.rng(M + K)
    x = synth.activations(g, M, K, np.float32) * np.float32(300.0)
    w = (g.standard_normal((N, K)) * 0.05).astype(np.float16)
    want = oracle.tile_gemm(1, M, K, N, 0, 0, w.view(np.uint8).reshape(-1), None, x)
    y = hip.DeviceBuffer(M * N * 4)
    hip.f16_tile_gemm(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, hip.DeviceBuffer.from_array(w.reshape(-1)), y, hip.F32,
                      M, K, N)
    ref_check(y.read(np.float32), want)


@pytest.mark.parametrize("M,K,N", [(1, 4096, 257), (32, 448, 127), (33, 2112, 128), (65, 256, 640), (128, 1536, 300), (300, 64, 8200), (257, 320, 8193)])
def test_f16_tiles(hip, oracle, M, K, N):
    """Half weights at the edges of the 32-, 64- and 128-row tiles, fewer sub-steps than buffers, and with K
    split; one row's infinity and one weight's NaN stay in their row and column."""
    from bybylang_amd import synth
    g = synth.rng(M + K + N)
    x = synth.activations(g, M, K, np.float32)
    w = (g.standard_normal((N, K)) * 0.05).astype(np.float16)
    run = lambda: hip.f16_tile_gemm(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, hip.DeviceBuffer.from_array(w.reshape(-1)), y, hip.F32,
                                    M, K, N)
    y = hip.DeviceBuffer(M * N * 4)
    run()
    want = np.asarray(oracle.tile_gemm(1, M, K, N, 0, 0, w.view(np.uint8).reshape(-1), None, x)).reshape(M, N)
    ref_check(y.read(np.float32), want)
    x[M - 1, K - 1] = np.inf
    w[N - 1, 0] = np.nan
    run()
    got = y.read(np.float32).reshape(M, N)
    assert np.isnan(got[:, N - 1]).all()
    assert not np.isfinite(got[M - 1]).any()
    if M > 1:
        ref_check(got[:M - 1, :N - 1], want[:M - 1, :N - 1])


@pytest.mark.parametrize("scales", ["ref", "mx", "edge"])
@pytest.mark.parametrize("K,N", [(32, 1), (96, 9), (2048, 65), (2080, 16), (4096, 130), (6176, 7), (8224, 24), (15360, 17), (15392, 17)])
def test_fp4km_decode_row(hip, oracle, K, N, scales):
    """One row at each count of groups per lane, past the decode GEMV's K, and with inf and NaN."""
    x, blob, t = fp4_case(1, K, N, scales, K + N)
    for mirror in (True, False):
        want = oracle.tile_gemm(0, 1, K, N, N * (K // 2), 0, blob, t, x)
        ref_check(run_fp4(hip, x, blob, t, 1, K, N, mirror), want)
    if scales == "mx":
        blob[N * (K // 2) + K // 32 - 1] = 255  # row 0's last group: an infinite scale
        want = np.asarray(oracle.tile_gemm(0, 1, K, N, N * (K // 2), 0, blob, t, x)).reshape(-1)
        got = run_fp4(hip, x, blob, t, 1, K, N, True)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ref_check(got[np.isfinite(want)], want[np.isfinite(want)])
        x[0, K - 1] = np.inf
        want = np.asarray(oracle.tile_gemm(0, 1, K, N, N * (K // 2), 0, blob, t, x)).reshape(-1)
        got = run_fp4(hip, x, blob, t, 1, K, N, True)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert np.array_equal(np.isinf(got), np.isinf(want))


@pytest.mark.parametrize("zeros", ["one", "group"])
@pytest.mark.parametrize("splits", [0, 2])
@pytest.mark.parametrize("M,K,N,group", [(1, 64, 16, 32), (16, 192, 130, 64), (17, 256, 127, 0), (40, 1344, 264, 32), (64, 1024, 129, 128),
                                         (65, 576, 72, 192), (130, 640, 300, 32)])
def test_q4_planes(hip, oracle, monkeypatch, M, K, N, group, zeros, splits):
    """The prefill copy's weights through the planes, activations over a wide range; every output type."""
    from bybylang_amd import synth
    g = synth.rng(M + K + N)
    wq, sc, ze, _ = synth.q4_weights(g, N, K, group or K)
    if zeros == "group":
        ze = g.integers(0, 16, ze.size).astype(np.float32)
    x = (synth.activations(g, M, K, np.float32) * 10.0 ** g.uniform(-8, 6, (M, 1))).astype(np.float32)
    gpr = K // group if group else 1
    monkeypatch.setenv("BYHIP_Q4_PLANES", "1")
    monkeypatch.setenv("BYHIP_Q4_ROUTE", "2")
    if splits:
        monkeypatch.setenv("BYHIP_Q4_SPLIT", str(splits))
    w = hip.Q4Weights(wq, sc, ze, K, N, group, gpr)
    xd = hip.DeviceBuffer.from_array(x.reshape(-1))
    want = oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, gpr)
    outs = {}
    for yt, nbytes in ((hip.F32, 4), (hip.BF16, 2)):
        y = hip.DeviceBuffer(M * N * nbytes)
        hip.q4_matmul(xd, hip.F32, w, y, yt, M)
        outs[yt] = y.read(hip.np_dtype(yt)).reshape(M, N)
    for m in range(M):  # row by row: each at its own magnitude
        scale = max(1e-30, float(np.max(np.abs(want[m]))))
        ref_check(outs[hip.F32][m] / scale, want[m] / scale)
    from parity import f32_to_bf16_rne
    assert np.array_equal(outs[hip.BF16], (f32_to_bf16_rne(outs[hip.F32]).view(np.uint32) >> 16).astype(np.uint16))


@pytest.mark.parametrize("fmt", ["f16", "fp4km"])
@pytest.mark.parametrize("K", [4194304 - 128, 4194304])
def test_rows_longer_than_the_scratch(hip, fmt, K):
    """Rows whose planes do not fit the scratch (from K = 4,194,304 on) run on the other kernels. Whole numbers
    few enough for exact sums."""
    from bybylang_amd import synth
    M, N = 2, 3
    g = synth.rng(K)
    x = np.zeros((M, K), np.float32)
    x[:, :: K // 512] = g.integers(-8, 9, size=x[:, :: K // 512].shape)
    x[:, K - 1] = 5
    y = hip.DeviceBuffer(M * N * 4)
    if fmt == "f16":
        w = g.integers(-4, 5, size=(N, K)).astype(np.float16)
        hip.f16_tile_gemm(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, hip.DeviceBuffer.from_array(w.reshape(-1)), y, hip.F32, M, K, N)
    else:
        codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
        t = np.concatenate([synth.E2M1, np.full(256, 2.0)]).astype(np.float32)
        w = 2 * np.asarray(synth.E2M1)[codes]
        blob = np.concatenate([synth.fp4km_pack(codes).reshape(-1), np.zeros(N * (K // 32), np.uint8)])
        hip.fp4km_tile_gemm(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, hip.DeviceBuffer.from_array(blob), N * (K // 2),
                            hip.DeviceBuffer.from_array(t), 0, y, hip.F32, M, K, N)
    k = np.nonzero(x.any(axis=0))[0]
    assert np.array_equal(y.read(np.float32).reshape(M, N), x[:, k].astype(np.float64) @ w[:, k].astype(np.float64).T)


@pytest.mark.parametrize("scales", ["ref", "one"])
@pytest.mark.parametrize("K", [2304, 4224])
@pytest.mark.parametrize("M", [16, 32, 48, 64, 128])
def test_fp4km_long_k(hip, oracle, monkeypatch, M, K, scales):
    """All of K in one block, at each tile height: 18 and 33 steps, so that the loop over eight sub-steps runs
    twice and more, its scale bytes are handed over each time, and a guarded tail follows."""
    N = 130
    x, blob, t = fp4_case(M, K, N, scales, M + K)
    monkeypatch.setenv("BYHIP_Q4_SPLIT", "1")
    ref_check(run_fp4(hip, x, blob, t, M, K, N, True), oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t, x))


@pytest.mark.parametrize("M,K,N", [(33, 256, 16400), (49, 1088, 9000), (67, 64, 8320), (331, 896, 5696), (392, 576, 2368), (391, 1024, 5000),
                                   (448, 384, 3776), (70, 4096, 8256), (361, 8192, 2100)])
@pytest.mark.parametrize("zeros", ["one", "group"])
def test_q4_tile_heights(hip, oracle, monkeypatch, M, K, N, zeros):
    """Calls that the times of the blocks' rounds give to tiles of 32, 48 and 64 rows, whole and with K split: rows at
    the tiles' edges against the oracle."""
    from bybylang_amd import synth
    g = synth.rng(M + K)
    wq, sc, ze, _ = synth.q4_weights(g, N, K, 32)
    if zeros == "group":
        ze = g.integers(0, 16, ze.size).astype(np.float32)
    monkeypatch.setenv("BYHIP_Q4_PLANES", "1")
    x = synth.activations(g, M, K, np.float32)
    y = hip.DeviceBuffer(M * N * 4)
    hip.q4_matmul(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, hip.Q4Weights(wq, sc, ze, K, N, 32, K // 32), y, hip.F32, M)
    rows = sorted({0, 31, 32, min(47, M - 1), min(48, M - 1), min(64, M - 1), M - 1})
    want = oracle.matmul_q4(x[rows].reshape(-1), wq, sc, ze, len(rows), K, N, 32, K // 32)
    ref_check(y.read(np.float32).reshape(M, N)[rows], np.asarray(want).reshape(len(rows), N))


@pytest.mark.parametrize("fmt", ["f16", "q4"])
@pytest.mark.parametrize("M", [257, 292, 293, 600])
def test_rows_about_what_the_scratch_holds(hip, oracle, monkeypatch, fmt, M):
    """K = 14336, where half the scratch holds the planes of 292 rows: all of them in one pass, also where
    that is no whole number of 64-row tiles, or in blocks."""
    from bybylang_amd import synth
    K, N = 14336, 24
    g = synth.rng(M)
    x = synth.activations(g, M, K, np.float32)
    y = hip.DeviceBuffer(M * N * 4)
    xd = hip.DeviceBuffer.from_array(x.reshape(-1))
    rows = sorted({0, 63, 64, 127, 128, 191, 192, 255, 256, M // 2, M - 65, M - 1})
    if fmt == "f16":
        w = (g.standard_normal((N, K)) * 0.05).astype(np.float16)
        hip.f16_tile_gemm(xd, hip.F32, hip.DeviceBuffer.from_array(w.reshape(-1)), y, hip.F32, M, K, N)
        want = oracle.tile_gemm(1, len(rows), K, N, 0, 0, w.view(np.uint8).reshape(-1), None, x[rows])
    else:
        wq, sc, ze, _ = synth.q4_weights(g, N, K, 32)
        monkeypatch.setenv("BYHIP_Q4_PLANES", "1")
        hip.q4_matmul(xd, hip.F32, hip.Q4Weights(wq, sc, ze, K, N, 32, K // 32), y, hip.F32, M)
        want = oracle.matmul_q4(x[rows].reshape(-1), wq, sc, ze, len(rows), K, N, 32, K // 32)
    ref_check(y.read(np.float32).reshape(M, N)[rows], np.asarray(want).reshape(len(rows), N))
