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


# without exchange slots the path is still the described one: the GEMV where it is chosen by time, the GEMM
# in whole blocks elsewhere
@pytest.mark.gpu
@pytest.mark.parametrize("qtype,M,K,N", [(qmm.Q8_0, 4096, 14336, 40), (qmm.Q8_0, 4096, 14336, 128), (qmm.Q5_K, 722, 8704, 308),
                                         (qmm.IQ4_XS, 4096, 14336, 77)])
def test_longk_noalloc(be, sc, qtype, M, K, N):
    say("longk noalloc", qtype, M, K, N)
    raw, x = synth.weights(qtype, M, K, seed=711), synth.activations(N, K, seed=712)
    w, xt, ya, yb = sc.weights(qtype, raw, (K, M)), sc.f32(x), sc.empty_f32((M, N)), sc.empty_f32((M, N))
    path = describe(qtype, K, M, N)["path"]
    be.mul_mat_noalloc(w, xt, yb)
    assert be.last_path() == path
    be.mul_mat(w, xt, ya)
    assert be.last_path() == path
    be.synchronize()
    got = be.get_f32(yb).reshape(N, M)
    assert rel_err(got, be.get_f32(ya).reshape(N, M)) <= TOL
    rows = 64
    assert rel_err(got[:, :rows], oracle.mul_mat(qtype, raw[:raw.size // M * rows], rows, K, x)) <= TOL


# a capture by a context without exchange slots, after the op ran once: the eager call's path on the eager
# call's scratch, whichever it is; replays with eager work between them
@pytest.mark.gpu
@pytest.mark.parametrize("qtype,M,K,N,path", [(qmm.Q8_0, 4096, 14336, 40, "gemv-mfma"), (qmm.Q8_0, 4096, 14336, 128, "gemm-stream")])
def test_longk_captured_without_slots(monkeypatch, qtype, M, K, N, path):
    say("longk captured cold", qtype, M, K, N)
    with qmm.Backend(0) as be:
        s = Scope(be)
        raw = synth.weights(qtype, M, K, seed=721)
        w, xs = s.weights(qtype, raw, (K, M)), [synth.activations(N, K, seed=722 + i) for i in range(3)]
        x, y, z = s.f32(xs[0]), s.empty_f32((M, N)), s.empty_f32((M, N))
        monkeypatch.setenv("QMM_GEMM3_TAIL", "0" if path == "gemm-stream" else "1")    # (whole blocks: no slots grown)
        be.mul_mat(w, x, y)
        be.synchronize()
        monkeypatch.setenv("QMM_GEMM3_TAIL", "1")
        be.capture_begin()
        be.mul_mat(w, x, y)
        g = be.capture_end()
        assert be.last_path() == path
        for v in xs:
            be.set_tensor(x, v.view(np.uint8).ravel())
            be.graph_launch(g)
            be.mul_mat_noalloc(w, x, z)                               # (whole blocks too)
            be.synchronize()
            assert be.last_path() == path
            if path == "gemm-stream":                                 # (the GEMV's K slices meet in any order)
                assert np.array_equal(be.get_f32(y).view(np.uint32), be.get_f32(z).view(np.uint32))
            assert rel_err(be.get_f32(y).reshape(N, M), be.get_f32(z).reshape(N, M)) <= TOL
            assert rel_err(be.get_f32(y).reshape(N, M)[:, :64], oracle.mul_mat(qtype, raw[:raw.size // M * 64], 64, K, v)) <= TOL
        g.free()
        s.close()
