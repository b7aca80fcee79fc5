"""FP4-KM with fp32 activations: the reference forms value * scale in fp32 and multiplies the fp32
activation with it (cpu_vm.c:583-628), so every bit of an activation counts, whatever its size beside its
neighbours', and no product leaves fp32's range that the reference's does not.

Bar: against the result in 64 bits, the roundings of an fp32 sum. Each of the K products and additions
may round once (2^-24 of what it holds), in any order at most |error| <= K 2^-24 sum |x w|, and sums
formed as trees or chains of a few dozen stay far below: 64 2^-24 sum |x w| (3.8e-6) is the bar.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BAR = 64 * 2.0 ** -24


def mx_table():
    from bybylang_amd import synth
    t = np.zeros(272, np.float32)
    t[:16] = synth.E2M1
    with np.errstate(over="ignore"):
        t[16:] = np.ldexp(np.float32(1), np.arange(256) - 127)
    return t


def run(hip, x, codes, sb, t):
    from bybylang_amd import synth
    M, K = x.shape
    N = codes.shape[0]
    blob = np.concatenate([synth.fp4km_pack(codes).reshape(-1), sb.astype(np.uint8).reshape(-1)])
    y = hip.DeviceBuffer(M * N * 4)
    hip.fp4km_tile_gemm(hip.DeviceBuffer.from_array(np.ascontiguousarray(x, np.float32).reshape(-1)), hip.F32,
                        hip.DeviceBuffer.from_array(blob), N * (K // 2), hip.DeviceBuffer.from_array(t), 0, y, hip.F32, M, K, N)
    return y.read(np.float32).reshape(M, N)


def exact(x, codes, sb, t):
    """(x . W^T, |x| . |W|^T) in 64 bits, the weights rounded to fp32 as the reference forms them."""
    with np.errstate(over="ignore", invalid="ignore"):
        w = (t[codes] * np.repeat(t[16 + sb.astype(np.int64)], 32, axis=1)).astype(np.float64)
        return x.astype(np.float64) @ w.T, np.abs(x.astype(np.float64)) @ np.abs(w).T


def check(got, x, codes, sb, t):
    want, size = exact(x, codes, sb, t)
    assert np.all(np.isfinite(want)) and np.all(np.isfinite(got))
    err = np.abs(got - want) / np.maximum(size, 2.0 ** -126)
    assert err.max() <= BAR, f"{err.max():.3g} of sum |x w| at {np.unravel_index(err.argmax(), err.shape)}"


@pytest.mark.parametrize("M", [1, 2, 17, 70])
@pytest.mark.parametrize("lead", [-10, -20, -30])
def test_small_activations_beside_large_ones(hip, M, lead):
    """The first activations of each 32-value group are 2^-lead times the others, and their codes zero:
    the results are sums of the small ones alone."""
    from bybylang_amd import synth
    g = synth.rng(100 * M - lead)
    K, N = 512, 40
    x = synth.activations(g, M, K, np.float32)
    codes = g.integers(1, 8, size=(N, K), dtype=np.uint8) | (g.integers(0, 2, size=(N, K), dtype=np.uint8) << 3)
    big = np.arange(K) % 32 < 3
    x[:, ~big] *= np.float32(2.0 ** lead)
    codes[:, big] = 0
    sb = g.integers(120, 130, size=(N, K // 32))
    check(run(hip, x, codes, sb, mx_table()), x, codes, sb, mx_table())


@pytest.mark.parametrize("M", [1, 2, 17, 70])
@pytest.mark.parametrize("spread,byte", [(8, 127), (26, 113), (60, 127)])
def test_groups_of_small_activations_on_large_weights(hip, M, spread, byte):
    """Group i of a row holds activations of about 2^-e, e up to `spread`, each column's scale there is 2^(e +
    byte - 127): every group counts alike. (26, 113) keeps every product within fp16's range."""
    from bybylang_amd import synth
    g = synth.rng(7 * M + spread)
    K, N = 1024, 70
    e = g.integers(0, spread + 1, size=K // 32)
    x = synth.activations(g, M, K, np.float32) * np.repeat(2.0 ** -e, 32).astype(np.float32)
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    sb = np.broadcast_to(byte + e, (N, K // 32)) + g.integers(-1, 2, size=(N, K // 32))
    check(run(hip, x, codes, sb, mx_table()), x, codes, sb, mx_table())


@pytest.mark.parametrize("M", [1, 5, 40])
@pytest.mark.parametrize("size,byte", [(1.5 * 2.0 ** 126, 117), (2.0 ** 120, 100), (2.0 ** 126, 60), (2.0 ** -126, 180), (2.0 ** -140, 230)])
def test_activations_at_the_ends_of_fp32(hip, M, size, byte):
    """Activations up to 1.5 2^126, whose sums with codes alone pass 2^128, on scales that bring them back,
    and subnormal ones on large scales."""
    from bybylang_amd import synth
    g = synth.rng(M + byte)
    K, N = 256, 33
    x = (g.uniform(0.5, 1.0, (M, K)) * size).astype(np.float32)
    codes = g.integers(1, 8, size=(N, K), dtype=np.uint8)
    codes[:, :4] = 7
    sb = np.full((N, K // 32), byte)
    check(run(hip, x, codes, sb, mx_table()), x, codes, sb, mx_table())


@pytest.mark.parametrize("table", ["mx", "other"])
@pytest.mark.parametrize("M", [1, 40])
def test_products_that_overflow_or_vanish(hip, oracle, M, table):
    """Scale entries of 2^126 and 2^127 (value * scale overflows for the larger codes), infinity, zero and
    subnormals, and a huge activation beside them: infinities and NaNs where the reference has them.
    The activations on the largest scales are about 2^-8, so that no finite sum passes 2^128 in any
    order of its additions."""
    from bybylang_amd import synth
    g = synth.rng(900 + M)
    K, N = 256, 64
    t = mx_table()
    if table == "other":
        t[16 + 10] = 0.0
        t[16 + 11] = 2.0 ** -149
        t[16 + 12] = 3 * 2.0 ** -149
    x = synth.activations(g, M, K, np.float32)
    x[:, 64:96] *= np.float32(2.0 ** -8)
    x[:, 5] = 2.0 ** 127
    x[:, 70] = 0.0
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    sb = np.full((N, K // 32), 100)
    sb[:, 0] = np.array([10, 11, 12, 0, 1, 90])[np.arange(N) % 6]
    sb[:32, 2] = np.array([253, 254, 255, 252])[np.arange(32) % 4]
    got = run(hip, x, codes, sb, t)
    blob = np.concatenate([synth.fp4km_pack(codes).reshape(-1), sb.astype(np.uint8).reshape(-1)])
    want = np.asarray(oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, blob, t, x.reshape(-1))).reshape(M, N)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    fin = np.isfinite(want)
    _, size = exact(x, codes, sb, t)
    assert np.all(np.abs(got[fin] - want[fin]) <= 2 * BAR * size[fin])


@pytest.mark.parametrize("K,N", [(32, 3), (2080, 33), (4096, 130), (15360, 9)])
@pytest.mark.parametrize("recorded", [False, True])
def test_one_row_takes_any_table(hip, oracle, recorded, K, N):
    """One row on E2M1 with E8M0 scales, on values that are not E2M1's, on scales that are not halves: the
    same recording follows the table the buffer holds at each replay."""
    from bybylang_amd import _abi, synth
    from bybylang_amd import gpubackend as gb
    g = synth.rng(K + N)
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    sb = g.integers(118, 136, size=(N, K // 32), dtype=np.uint8)
    x = synth.activations(g, 1, K, np.float32)
    mx = mx_table()
    values = mx.copy()
    values[:16] = g.standard_normal(16)
    scales = mx.copy()
    scales[16:] = np.exp(g.normal(0, 2, 256))
    minus = mx.copy()
    minus[8] = 0.0  # E2M1 but for the sign of its second zero
    if not recorded:
        for t in (mx, values, scales, minus):
            check(run(hip, x, codes, sb, t), x, codes, sb, t)
        return
    blob = np.concatenate([synth.fp4km_pack(codes).reshape(-1), sb.reshape(-1)])
    words = np.zeros((blob.size + 3) // 4, np.float32)
    words.view(np.uint8)[: blob.size] = blob
    assert gb.sessionBegin(gb.gbHip)
    hx, hw, ht = (gb.sessionUpload(gb.gbHip, v) for v in (x.reshape(-1), words, mx))
    ho = gb.sessionAllocScratch(gb.gbHip, N)
    assert gb.sessionEnd(gb.gbHip)
    assert gb.sessionBeginRecording(gb.gbHip)
    assert gb.sessionFp4GemmTensorCore(gb.gbHip, hx, hw, ht, ho, 1, K, N)
    assert gb.sessionEnd(gb.gbHip), gb.sessionGetLastError(gb.gbHip)
    rid = gb.sessionLastRecording(gb.gbHip)
    for t in (mx, values, scales, minus, mx):
        _abi.check(_abi.load().byhip_upload(ht.hipHandle, 0, t.ctypes.data, t.nbytes))
        assert gb.sessionReplay(gb.gbHip, rid, 1), gb.sessionGetLastError(gb.gbHip)
        check(np.asarray(gb.sessionRead(gb.gbHip, ho, N)).reshape(1, N), x, codes, sb, t)
    gb.sessionFreeRecording(gb.gbHip, rid)
    for h in (hx, hw, ht, ho):
        gb.sessionFree(gb.gbHip, h)


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("M,K,N", [(2, 128, 1), (16, 2432, 129), (17, 2176, 128), (40, 1152, 200), (63, 640, 127), (64, 2304, 130), (65, 4224, 40), (129, 256, 300)])
def test_three_term_tiles(hip, monkeypatch, M, K, N, splits):
    """E8M0 tables at the edges of the 16- to 64-row tiles, even and odd steps per K group, one to 17 of them,
    and K split: the scales up to byte 252, one zero-filled group with byte 0."""
    from bybylang_amd import synth
    g = synth.rng(M + K + N)
    if splits:
        monkeypatch.setenv("BYHIP_Q4_SPLIT", str(splits))
    x = synth.activations(g, M, K, np.float32)
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    sb = g.integers(120, 134, size=(N, K // 32))
    codes[N // 2, 32:64] = 0
    sb[N // 2, 1] = 0
    x[:, :4] *= np.float32(2.0 ** -8)  # no sum of the last column's passes 2^128 in any order
    codes[N - 1, :] = 0     # a column whose only weights are at the ends of the scales
    codes[N - 1, :4] = [1, 7, 9, 15]
    sb[N - 1, 0] = 252 if M % 2 else 1
    check(run(hip, x, codes, sb, mx_table()), x, codes, sb, mx_table())


@pytest.mark.parametrize("M,K,N", [(2, 128, 40), (40, 1152, 130), (130, 640, 72), (1000, 4096, 2120), (1024, 4096, 40)])
def test_recorded_rows_follow_the_table(hip, M, K, N):
    """A recording of more than one row queues every route and runs the one for the table the buffer holds at each
    replay: E8M0 scales, scales whose products are halves, other values with halves, any values. K = 4096: 1023
    rows' planes fit the scratch."""
    from bybylang_amd import _abi, synth
    from bybylang_amd import gpubackend as gb
    g = synth.rng(M + N)
    codes = g.integers(0, 16, size=(N, K), dtype=np.uint8)
    sb = g.integers(118, 136, size=(N, K // 32), dtype=np.uint8)
    x = synth.activations(g, M, K, np.float32)
    mx = mx_table()
    halves = mx.copy()
    halves[16:] = (1 + np.arange(256) % 13) / 64
    values = halves.copy()
    values[1] = 0.75
    other = mx.copy()
    other[:16] = g.standard_normal(16)
    blob = np.concatenate([synth.fp4km_pack(codes).reshape(-1), sb.reshape(-1)])
    words = np.zeros((blob.size + 3) // 4, np.float32)
    words.view(np.uint8)[: blob.size] = blob
    assert gb.sessionBegin(gb.gbHip)
    hx, hw, ht = (gb.sessionUpload(gb.gbHip, v) for v in (x.reshape(-1), words, mx))
    ho = gb.sessionAllocScratch(gb.gbHip, M * N)
    assert gb.sessionEnd(gb.gbHip)
    assert gb.sessionBeginRecording(gb.gbHip)
    assert gb.sessionFp4GemmTensorCore(gb.gbHip, hx, hw, ht, ho, M, K, N)
    assert gb.sessionEnd(gb.gbHip), gb.sessionGetLastError(gb.gbHip)
    rid = gb.sessionLastRecording(gb.gbHip)
    for t in (mx, halves, other, values, mx, values, halves):
        _abi.check(_abi.load().byhip_upload(ht.hipHandle, 0, t.ctypes.data, t.nbytes))
        assert gb.sessionReplay(gb.gbHip, rid, 1), gb.sessionGetLastError(gb.gbHip)
        check(np.asarray(gb.sessionRead(gb.gbHip, ho, M * N)).reshape(M, N), x, codes, sb, t)
    gb.sessionFreeRecording(gb.gbHip, rid)
    for h in (hx, hw, ht, ho):
        gb.sessionFree(gb.gbHip, h)
