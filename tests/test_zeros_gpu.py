"""Q4 weights with a zero point per group on the MI355X against the oracle.

Whole-number zeros travel in the prefill copy, so the wide and the tall tile take such weights;
others stay on the general kernels. Bars as in test_q4_gpu.py: fp32 activations within the
reference's tolerance (the weights stay exact), fp16 activations above the decode rows within the
fp32-accumulate tier (each weight rounded once to fp16).
"""
import numpy as np
import pytest

from parity import TIER_F32_ACC, ref_check, tier_check

pytestmark = pytest.mark.gpu


def case(seed, M, K, N, group, zeros):
    from bybylang_amd import synth
    g = synth.rng(seed)
    wq, sc, _, _ = synth.q4_weights(g, N, K, group or K)
    ng = sc.size
    ze = {"codes": g.integers(0, 16, ng), "wide": g.integers(-1024, 1025, ng),
          "past": g.integers(-1200, 1201, ng), "halves": g.integers(0, 31, ng) / 2}[zeros].astype(np.float32)
    if zeros == "wide":
        ze[:2] = [-1024, 1024]
    # |x| stays small where the zeros are large, so that the oracle's fp32 sums keep the tolerance
    x = synth.activations(g, M, K, np.float16)
    return x, wq, sc, ze


@pytest.mark.parametrize("x_dtype", ["F32", "F16"])
@pytest.mark.parametrize("zeros", ["codes", "wide", "past", "halves"])
@pytest.mark.parametrize("M,K,N,group", [(2, 192, 40, 32), (8, 1344, 264, 64), (9, 512, 136, 128), (32, 1024, 72, 0),
                                         (33, 384, 130, 96), (130, 768, 520, 32)])
def test_zero_per_group(hip, oracle, monkeypatch, M, K, N, group, zeros, x_dtype):
    x, wq, sc, ze = case(M + K, M, K, N, group, zeros)
    gpr = K // group if group else 1
    w = hip.Q4Weights(wq, sc, ze, K, N, group, gpr)
    assert not w.info()["zero_uniform"]
    xd = hip.DeviceBuffer.from_array(x.astype(np.float32 if x_dtype == "F32" else np.float16).reshape(-1))
    want = oracle.matmul_q4(x.astype(np.float32).reshape(-1), wq, sc, ze, M, K, N, group, gpr)
    for tile in (0, 2, 3):  # the default route, the 128 x 256 tile, the wide tile
        if tile:
            monkeypatch.setenv("BYHIP_Q4_PREFILL", str(tile))
        yd = hip.DeviceBuffer(M * N * 4)
        hip.q4_matmul(xd, getattr(hip, x_dtype), w, yd, hip.F32, M)
        got = yd.read(np.float32)
        if x_dtype == "F32":
            ref_check(got, want)
        else:
            tier_check(got, want, TIER_F32_ACC)


def test_zero_per_group_equal_zeros_match_one_zero(hip):
    """The same weights with one zero for all and with that zero in all groups but an unused one
    (a column of zero scales) give the same bits on the tall and the wide tile."""
    from bybylang_amd import synth
    M, K, N = 130, 512, 520
    x, wq, sc, _ = case(3, M, K, N, 32, "codes")
    sc[: K // 32] = 0.0
    one = np.full(sc.size, 8.0, np.float32)
    per = one.copy()
    per[: K // 32] = 3.0
    xd = hip.DeviceBuffer.from_array(x.reshape(-1))
    outs = []
    for ze in (one, per):
        w = hip.Q4Weights(wq, sc, ze, K, N, 32, K // 32)
        yd = hip.DeviceBuffer(M * N * 4)
        hip.q4_matmul(xd, hip.F16, w, yd, hip.F32, M)
        outs.append(yd.read(np.float32).view(np.uint32))
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("M,K,N", [(251, 512, 8320), (65, 8192, 16400)])
def test_tiles_past_one_round(hip, oracle, monkeypatch, M, K, N):
    """The wide tile with a few tiles more than CUs, unsplit (short K) and split (long K) by default: the
    first and last rows against the oracle, every row against the same tile with K split three ways,
    which differs by the order of the fp32 sums only."""
    x, wq, sc, ze = case(M + K, M, K, N, 32, "codes")
    w = hip.Q4Weights(wq, sc, ze, K, N, 32, K // 32)
    xd = hip.DeviceBuffer.from_array(x.reshape(-1))
    outs = []
    monkeypatch.setenv("BYHIP_Q4_PREFILL", "3")
    for split in (None, "3"):
        if split:
            monkeypatch.setenv("BYHIP_Q4_SPLIT", split)
        yd = hip.DeviceBuffer(M * N * 4)
        hip.q4_matmul(xd, hip.F16, w, yd, hip.F32, M)
        outs.append(yd.read(np.float32).reshape(M, N))
    ref_check(outs[0], outs[1])
    rows = [0, M - 1]
    want = oracle.matmul_q4(x[rows].astype(np.float32).reshape(-1), wq, sc, ze, 2, K, N, 32, K // 32)
    tier_check(outs[0][rows].reshape(-1), np.asarray(want).reshape(-1), TIER_F32_ACC)
