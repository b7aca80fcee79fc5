"""The pipelined fp32 GEMM for Q4 weights with fp32 scales (micro-VM slots, weights outside fp16's
range) on the MI355X against the oracle, at the edges of its tiles, steps and splits.

Bar: the reference test's tolerance; the arithmetic is fp32 as in the reference.
"""
import numpy as np
import pytest

from oracle_lib import OP_Q4_COOP_GEMM, q4_blob, shape_op_program
from parity import ref_check

pytestmark = pytest.mark.gpu


def slots(seed, M, K, N, group, spread):
    from bybylang_amd import synth
    g = synth.rng(seed)
    ng = K // group
    wq, _, _, _ = synth.q4_weights(g, N, K, group)
    sc = (g.standard_normal(N * ng) * 0.02).astype(np.float32)
    if spread:
        sc *= (10.0 ** g.uniform(-6, 6, N * ng)).astype(np.float32)
    ze = (8 + g.standard_normal(N * ng)).astype(np.float32)
    return synth.activations(g, M, K, np.float32), wq, sc, ze


@pytest.mark.parametrize("spread", [False, True])
@pytest.mark.parametrize("M,K,N,group", [(3, 128, 16, 32), (8, 256, 130, 64), (16, 640, 127, 128), (17, 1024, 40, 32), (48, 384, 300, 32),
                                         (64, 2048, 128, 256), (65, 512, 136, 512), (130, 896, 72, 128)])
@pytest.mark.parametrize("splits", [0, 3])
def test_f32_q4_program(hip, oracle, monkeypatch, M, K, N, group, spread, splits):
    x, wq, sc, ze = slots(M + K, M, K, N, group, spread)
    if splits:
        monkeypatch.setenv("BYHIP_Q4_SPLIT", str(splits))
    by, fl = q4_blob(wq, sc, ze, K, N, K // group)
    mem = hip.DeviceBuffer(M * N * 4)
    hip.program_dispatch(shape_op_program(OP_Q4_COOP_GEMM, M, K, N, group, K // group), mem, hip.DeviceBuffer.from_array(by),
                         hip.DeviceBuffer.from_array(fl), hip.DeviceBuffer.from_array(x.reshape(-1)))
    want = oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, K // group)
    ref_check(mem.read(np.float32), want)


@pytest.mark.parametrize("M,K,N,group,zeros", [(5, 256, 40, 0, "one"), (20, 1152, 130, 32, "one"), (40, 512, 100, 0, "group")])
def test_f32_q4_resident(hip, oracle, M, K, N, group, zeros):
    """Resident weights outside fp16's range: one zero for all, or one per group; one group per row."""
    x, wq, sc, ze = slots(M, M, K, N, group or K, True)
    if zeros == "one":
        ze[:] = 7.5
    w = hip.Q4Weights(wq, sc, ze, K, N, group, K // group if group else 1)
    assert not w.info()["f16_safe"]
    y = hip.DeviceBuffer(M * N * 4)
    hip.q4_matmul(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, w, y, hip.F32, M)
    want = oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, K // group if group else 1)
    ref_check(y.read(np.float32), want)


@pytest.mark.parametrize("zeros", ["one", "group"])
@pytest.mark.parametrize("M,K,N,group", [(3, 896, 16, 32), (9, 1024, 130, 128), (16, 1152, 600, 64), (11, 2176, 40, 0), (16, 4096, 72, 256),
                                         (5, 4224, 1000, 32)])
def test_f32_q4_columns(hip, oracle, M, K, N, group, zeros):
    """Up to 16 rows on few columns, K split over a block's eight waves: waves without a step, one step
    for each, one more for the first, up to five for some."""
    x, wq, sc, ze = slots(M + N, M, K, N, group or K, True)
    if zeros == "one":
        ze[:] = 7.5
    gpr = K // group if group else 1
    w = hip.Q4Weights(wq, sc, ze, K, N, group, gpr)
    assert not w.info()["f16_safe"]
    y = hip.DeviceBuffer(M * N * 4)
    hip.q4_matmul(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, w, y, hip.F32, M)
    ref_check(y.read(np.float32), oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, gpr))


@pytest.mark.parametrize("M,K", [(13, 2176), (30, 1152), (48, 1280), (60, 2304)])
def test_f32_q4_unsplit(hip, oracle, monkeypatch, M, K):
    """All of K in one block of 16 to 64 rows: several rounds of the three buffers, and each remainder."""
    N, group = 130, 64
    x, wq, sc, ze = slots(M, M, K, N, group, True)
    monkeypatch.setenv("BYHIP_Q4_SPLIT", "1")
    w = hip.Q4Weights(wq, sc, ze, K, N, group, K // group)
    y = hip.DeviceBuffer(M * N * 4)
    hip.q4_matmul(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, w, y, hip.F32, M)
    ref_check(y.read(np.float32), oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, K // group))


@pytest.mark.parametrize("M,K,N", [(3, 1024, 4104), (3, 2048, 4097), (4, 1024, 4104), (4, 2048, 4100), (3, 4096, 8200), (3, 4096, 8192), (4, 4096, 4104)])
def test_few_rows_on_many_columns(hip, oracle, M, K, N):
    """Three and four rows with more columns than one 16-column block per CU, on either side of the GEMV's lines."""
    group = 64
    x, wq, sc, ze = slots(K + M, M, K, N, group, True)
    w = hip.Q4Weights(wq, sc, ze, K, N, group, K // group)
    y = hip.DeviceBuffer(M * N * 4)
    hip.q4_matmul(hip.DeviceBuffer.from_array(x.reshape(-1)), hip.F32, w, y, hip.F32, M)
    ref_check(y.read(np.float32), oracle.matmul_q4(x.reshape(-1), wq, sc, ze, M, K, N, group, K // group))
