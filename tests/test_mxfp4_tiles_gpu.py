"""The MXFP4 GEMM's tile sizes on the MI355X against the oracle, at the edges of tiles, steps and splits.

Bar: fp32 outputs within 1e-5 of the peak (products and scales are exact, only the order of the fp32
sums differs); fp16 and bf16 outputs are the fp32 ones rounded.
"""
import numpy as np
import pytest

from parity import bf16_bits_to_f32, f32_to_bf16_rne, max_abs_rel

pytestmark = pytest.mark.gpu


def operands(M, K, N, seed, nan=False):
    from bybylang_amd import synth
    g = synth.rng(seed)
    xb, xc, xe = synth.mxfp4_operand(g, M, K)
    wb, wc, we = synth.mxfp4_operand(g, N, K)
    if nan:  # a NaN scale in the first group of a row: the row before it reads nothing past its end
        xe[M // 2, 0] = 255
        we[N // 2, 0] = 255
        xb[M * (K // 2):] = xe.reshape(-1)
        wb[N * (K // 2):] = we.reshape(-1)
    return xb, synth.mx_decode(xc, xe), wb, xe, we


@pytest.mark.parametrize("mid", ["", "0", "1", "2", "3", "4"])
@pytest.mark.parametrize("M,K,N", [(1, 128, 16), (16, 256, 127), (17, 384, 130), (47, 640, 264), (64, 1152, 128), (65, 3200, 100),
                                   (130, 512, 300), (33, 4224, 24)])
def test_mxfp4_tiles(hip, oracle, monkeypatch, M, K, N, mid):
    """The default choice, the large tiles and each smaller tile, each output type; split K for the
    longer rows (the default splits them)."""
    from bybylang_amd import synth
    xb, xf, wb, _, _ = operands(M, K, N, M + K)
    if mid:
        monkeypatch.setenv("BYHIP_MX_MID", mid)
    want = np.asarray(oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, wb, synth.mx_table(), xf)).reshape(M, N)
    x, w = hip.DeviceBuffer.from_array(xb), hip.DeviceBuffer.from_array(wb)
    outs = {}
    for yt, nbytes in ((hip.F32, 4), (hip.F16, 2), (hip.BF16, 2)):
        y = hip.DeviceBuffer(M * N * nbytes)
        hip.mxfp4_gemm(x, w, y, yt, M, K, N)
        outs[yt] = y.read(hip.np_dtype(yt)).reshape(M, N)
    assert max_abs_rel(outs[hip.F32], want) < 1e-5
    assert np.array_equal(outs[hip.F16].view(np.uint16), outs[hip.F32].astype(np.float16).view(np.uint16))
    assert np.array_equal(bf16_bits_to_f32(outs[hip.BF16]), f32_to_bf16_rne(outs[hip.F32]))


@pytest.mark.parametrize("M,K,N", [(20, 128, 40), (20, 384, 130), (50, 640, 40)])
def test_mxfp4_nan_scales_stay_in_their_rows(hip, M, K, N):
    xb, _, wb, xe, we = operands(M, K, N, 7, nan=True)
    y = hip.DeviceBuffer(M * N * 4)
    hip.mxfp4_gemm(hip.DeviceBuffer.from_array(xb), hip.DeviceBuffer.from_array(wb), y, hip.F32, M, K, N)
    got = np.isnan(y.read(np.float32).reshape(M, N))
    want = np.zeros((M, N), bool)
    want[M // 2, :] = True
    want[:, N // 2] = True
    assert np.array_equal(got, want)


@pytest.mark.parametrize("mid", ["1", "2", "3", "4"])
@pytest.mark.parametrize("K", [3072, 3200, 5888, 6272])
def test_mxfp4_small_tiles_long_k(hip, oracle, monkeypatch, K, mid):
    """12, 13, 23 and 25 pairs of steps in one block: the loop over 12 pairs run once and twice, then a tail,
    with even and odd counts of steps."""
    from bybylang_amd import synth
    M, N = 16 * int(mid) - 3, 130
    xb, xf, wb, _, _ = operands(M, K, N, M + K)
    monkeypatch.setenv("BYHIP_MX_MID", mid)
    monkeypatch.setenv("BYHIP_MX_SPLIT", "1")
    want = np.asarray(oracle.tile_gemm(0, M, K, N, N * (K // 2), 0, wb, synth.mx_table(), xf)).reshape(M, N)
    y = hip.DeviceBuffer(M * N * 4)
    hip.mxfp4_gemm(hip.DeviceBuffer.from_array(xb), hip.DeviceBuffer.from_array(wb), y, hip.F32, M, K, N)
    assert max_abs_rel(y.read(np.float32).reshape(M, N), want) < 1e-5
