"""The streaming GEMM's waves of 64 rows x 64 columns (Q4_0, Q8_0, IQ4_NL; one product or a gate/up
pair), against the CPU oracle and the 32-row waves, through the C ABI.

Bar: MUL_MAT's own (rel_err <= 1e-3 of the floored reference): an exact integer dot per block with
float32 sums (~1e-6).  Against 32-row waves on one K slice: the same sums in the same order, so the
same bits."""
import numpy as np
import pytest

from arcint_amd import qmm, synth
from conftest import rel_err
from test_gpu_parity import TOL, Scope, be, glu_case, say, sc  # noqa: F401  (fixtures)

BLOCKS = [qmm.Q4_0, qmm.Q8_0, qmm.IQ4_NL]


def product(be, sc, qtype, M, K, N, B, seed):
    """weights shared by B batches of N columns; dst rows and columns padded with 7"""
    w = sc.weights(qtype, synth.weights(qtype, M, K, seed=seed), (K, M))
    x = sc.f32(synth.activations(B * N, K, seed=seed + 1).reshape(B, N, K)).view((K, N, B), (4, 4 * K, 4 * K * N, 4 * K * N * B))
    full = sc.f32(np.full((B, N + 1, M + 3), 7.0, np.float32))
    nb1 = 4 * (M + 3)
    be.mul_mat(w, x, full.view((M, N, B), (4, nb1, nb1 * (N + 1), nb1 * (N + 1) * B)))
    be.synchronize()
    return be.get_f32(full).reshape(B, N + 1, M + 3)


# rows: one of a tile, a whole tile, one past a work-group's four; columns: one past a tile, a pair,
# an odd number of tiles; K: one block past a group, one group, several
@pytest.mark.gpu
@pytest.mark.parametrize("qtype", BLOCKS)
@pytest.mark.parametrize("M,K,N,B", [(1, 288, 33, 1), (64, 256, 64, 1), (257, 1280, 97, 1), (450, 800, 161, 3)])
def test_wide_product(be, sc, monkeypatch, qtype, M, K, N, B):
    say("wide", qtype, M, K, N, B)
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    out = []
    for env in ({"QMM_GEMM3_WIDE": "1"}, {"QMM_GEMM3_WIDE": "0", "QMM_GEMM3_KQ": "0", "QMM_GEMM3_TAIL": "0"}):
        with monkeypatch.context() as mp:
            for k, v in env.items():
                mp.setenv(k, v)
            out.append(product(be, sc, qtype, M, K, N, B, 601))
            assert be.last_path() == "gemm-stream"
    assert np.all(out[0][:, N:, :] == 7.0) and np.all(out[0][:, :, M:] == 7.0)     # nothing written past the view
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("qtype,op", [(qmm.Q4_0, qmm.GLU_SWIGLU), (qmm.Q8_0, qmm.GLU_GEGLU), (qmm.IQ4_NL, qmm.GLU_REGLU)])
def test_wide_pair(be, sc, orc, monkeypatch, qtype, op):
    monkeypatch.setenv("QMM_GEMM3_WIDE", "1")
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    for (M, K, N, seed) in [(33, 256, 64, 611), (200, 768, 33, 614), (450, 1280, 97, 617)]:
        say("wide pair", qtype, M, K, N)
        got, ref = glu_case(be, sc, orc, qtype, qtype, M, K, N, op, seed=seed)
        assert be.last_path() == "glu-gemm-stream"
        assert rel_err(got, ref) <= TOL, (M, K, N)


# a pair over batches that share weights, dst columns and batches padded, columns of src1 at a stride: against the
# 32-row waves (the same sums in the same order), rows and columns past a tile
@pytest.mark.gpu
@pytest.mark.parametrize("qtype", BLOCKS)
def test_wide_pair_strides_and_batches(be, sc, monkeypatch, qtype):
    K, M, N, B = 544, 97, 75, 4
    say("wide pair strides", qtype)
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    w = [sc.weights(qtype, synth.weights(qtype, 2 * M, K, seed=631 + i), (K, M, 2)) for i in range(2)]
    x = sc.f32(synth.activations(B * 2 * N, K, seed=633).reshape(B, 2 * N, K)).view((K, N, B), (4, 8 * K, 8 * K * N, 8 * K * N * B))
    out = []
    for env in ({"QMM_GEMM3_WIDE": "1"}, {"QMM_GEMM3_WIDE": "0", "QMM_GEMM3_PAIR": "0"}):
        with monkeypatch.context() as mp:
            for k, v in env.items():
                mp.setenv(k, v)
            full = sc.f32(np.full((B, N + 3, M + 5), 7.0, np.float32))
            nb1 = 4 * (M + 5)
            be.mul_mat_glu(w[0], w[1], x, full.view((M, N, B), (4, nb1, nb1 * (N + 3), nb1 * (N + 3) * B)), qmm.GLU_SWIGLU)
            be.synchronize()
            assert be.last_path() == "glu-gemm-stream"
            out.append(be.get_f32(full).reshape(B, N + 3, M + 5))
    assert np.all(out[0][:, N:, :] == 7.0) and np.all(out[0][:, :, M:] == 7.0)     # nothing written past the view
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


# the launch rule: 64-row waves from about a round of 512 work-groups on, not where most of a further
# round would be empty (r rounds of 128 row tiles x 64-column pairs), and not for the other types
@pytest.mark.parametrize("qtype,N,wide", [(qmm.Q4_0, 64, False), (qmm.Q4_0, 768, False), (qmm.Q4_0, 1024, True),
                                          (qmm.Q4_0, 1088, False), (qmm.Q4_0, 1536, True), (qmm.Q4_0, 2048, True),
                                          (qmm.Q8_0, 1536, True), (qmm.Q8_0, 1088, False), (qmm.IQ4_NL, 896, False),
                                          (qmm.IQ4_NL, 1024, True), (qmm.Q4_K, 1024, False)])
def test_wide_rule(qtype, N, wide):
    fake = qmm.Buffer(ptr=0x1000, size=1 << 44)
    info = qmm.describe_mul_mat(qmm.Tensor(fake, qtype, (4096, 8192)), qmm.Tensor(fake, qmm.F32, (4096, N)),
                                qmm.Tensor(fake, qmm.F32, (8192, N)))
    pairs = -(-N // 64)
    if wide:
        assert (info["threads"], info["workgroups"], info["lds_bytes"]) == (256, 32 * pairs, 37 * 1024)
    else:
        assert (info["threads"], info["workgroups"]) != (256, 32 * pairs)


# short K, where the stores decide (op us, 64-row / 32-row waves)
@pytest.mark.parametrize("qtype,M,K,N,wide", [(qmm.Q4_0, 13756, 768, 836, False),        # 44 / 38
                                              (qmm.Q4_0, 39216, 512, 1961, False),       # 150 / 144
                                              (qmm.Q4_0, 31219, 544, 360, False),        # 42 / 36
                                              (qmm.IQ4_NL, 16884, 896, 669, False),      # 53 / 50
                                              (qmm.Q8_0, 12838, 512, 790, False),        # 34 / 31
                                              (qmm.Q8_0, 12222, 544, 1329, True),        # 51 / 55
                                              (qmm.Q8_0, 16384, 4096, 512, True),        # 97 / 121
                                              (qmm.Q4_0, 4096, 11008, 2048, True)])      # 247 / 275
def test_wide_rule_short_k(qtype, M, K, N, wide):
    fake = qmm.Buffer(ptr=0x1000, size=1 << 44)
    info = qmm.describe_mul_mat(qmm.Tensor(fake, qtype, (K, M)), qmm.Tensor(fake, qmm.F32, (K, N)),
                                qmm.Tensor(fake, qmm.F32, (M, N)))
    groups = -(-M // 256) * -(-N // 64)
    assert ((info["threads"], info["lds_bytes"]) == (256, 37 * 1024) and info["workgroups"] == -(-groups // 8) * 8) == wide
