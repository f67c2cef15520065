"""The streaming GEMM's launch shape by estimated time (one product, K from 8192 on, below one round of
4-wave blocks): the choice, and the blocks in pieces along K that it takes, against the CPU oracle.

Bar: MUL_MAT's own (rel_err <= 1e-3 of the floored reference): an exact integer dot per block with
float32 sums (~1e-6)."""
import numpy as np
import pytest

import oracle
from arcint_amd import qmm, synth
from conftest import rel_err
from test_gpu_parity import TOL, Scope, be, say, sc  # noqa: F401  (fixtures)

TYPES = [qmm.Q4_0, qmm.Q8_0, qmm.IQ4_NL, qmm.Q4_K, qmm.Q5_K, qmm.Q6_K, qmm.IQ4_XS]


def describe(qtype, K, M, N):
    fake = qmm.Buffer(ptr=0x1000, size=1 << 44)
    return qmm.describe_mul_mat(qmm.Tensor(fake, qtype, (K, M)), qmm.Tensor(fake, qmm.F32, (K, N)),
                                qmm.Tensor(fake, qmm.F32, (M, N)))


# GEMV or GEMM by the smaller estimate, and the GEMM's work-groups: 4-wave blocks in four pieces along K
# (64 row tiles' halves in fours x column pairs x 4), or 12 waves over four K slices
@pytest.mark.parametrize("qtype,K,M,N,path,wg", [
    (qmm.Q8_0, 14336, 4096, 40, "gemv-mfma", None), (qmm.Q8_0, 14336, 4096, 128, "gemm-stream", (256, 256)),
    (qmm.Q8_0, 14304, 11861, 36, "gemm-stream", None), (qmm.IQ4_XS, 14336, 4096, 128, "gemm-stream", (256, 256)),
    (qmm.Q4_K, 17408, 5120, 64, "gemv-mfma", None), (qmm.Q5_K, 17408, 5120, 40, "gemm-stream", (256, 160)),
    (qmm.Q4_K, 17408, 5120, 256, "gemm-stream", (768, 216)),
    (qmm.Q8_0, 8160, 4096, 128, "gemm-stream", None),             # 32 groups: by time
    (qmm.Q8_0, 7936, 4096, 40, "gemv-mfma", None)])               # 31: by rounds
def test_longk_rule(qtype, K, M, N, path, wg):
    info = describe(qtype, K, M, N)
    assert info["path"] == path
    if wg:
        assert (info["threads"], info["workgroups"]) == wg


# rows: one of a tile, past a block's 128, ragged; columns: one tile, one past a pair, an odd number of
# tiles; K: the first group count that pieces take, and one whose last piece is shorter
@pytest.mark.gpu
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("M,K,N", [(1, 8192, 17), (130, 8448, 65), (450, 8960, 97)])
def test_longk_product(be, sc, monkeypatch, qtype, M, K, N):
    say("longk", qtype, M, K, N)
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    raw, x = synth.weights(qtype, M, K, seed=701), synth.activations(N, K, seed=702)
    w, xt = sc.weights(qtype, raw, (K, M)), sc.f32(x)
    full = sc.f32(np.full((N + 1, M + 3), 7.0, np.float32))       # dst rows padded with 7
    for _ in range(2):                                            # (the tree slots are left as they were)
        be.mul_mat(w, xt, full.view((M, N), (4, 4 * (M + 3), 4 * (M + 3) * (N + 1), 4 * (M + 3) * (N + 1))))
        be.synchronize()
        assert be.last_path() == "gemm-stream"
        got = be.get_f32(full).reshape(N + 1, M + 3)
        assert np.all(got[N:] == 7.0) and np.all(got[:, M:] == 7.0)
        assert rel_err(got[:N, :M], oracle.mul_mat(qtype, raw, M, K, x)) <= TOL
