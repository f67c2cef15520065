"""The dense gate/up + GLU pair on the streaming GEMM (gate and up waves side by side in a work-group,
their sums meeting in LDS, the GLU at the store), against the CPU oracle, through the C ABI.

Bar: MUL_MAT's own (rel_err <= 1e-3 of the floored reference): each product is an exact integer dot per
block with float32 sums (~1e-6), and an activation of slope at most 1.13 leaves that order."""
import numpy as np
import pytest

from arcint_amd import qmm, synth
from conftest import rel_err
from test_gpu_parity import TOL, TYPES, Scope, be, glu_case, say, sc  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


# each launch shape (U waves x K slices, forced by index) on ragged shapes: rows not a whole number of
# a block's row halves, an odd number of column tiles, a last tile of one column, K slices of unequal
# length, a single group of K
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("shape", range(5))
def test_pair_shapes(be, sc, orc, monkeypatch, qtype, shape):
    monkeypatch.setenv("QMM_GEMM3_PAIR", str(shape))
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    for (M, K, N, seed) in [(200, 768, 33, 501), (70, 256, 64, 504), (450, 1280, 97, 507), (330, 4352, 80, 510)]:
        say("pair", qtype, shape, M, K, N)
        got, ref = glu_case(be, sc, orc, qtype, qtype, M, K, N, qmm.GLU_SWIGLU, seed=seed)
        assert be.last_path() == "glu-gemm-stream"
        assert rel_err(got, ref) <= TOL, (M, K, N)


# the blocks past a whole number per CU in 2 and 3 pieces along K whose (gate, up) sums meet as
# 64-bit exchanges: 29 row blocks x 9 column pairs = 261 blocks of 4 waves; the same bits on a
# second call (every slot is left empty; a + b = b + a), every GLU
@pytest.mark.parametrize("qtype,K,op", [(qmm.Q4_K, 1024, qmm.GLU_SWIGLU), (qmm.Q6_K, 1536, qmm.GLU_GEGLU),
                                        (qmm.Q4_0, 1024, qmm.GLU_REGLU), (qmm.IQ4_XS, 2048, qmm.GLU_GEGLU_QUICK),
                                        (qmm.Q5_K, 1536, qmm.GLU_GEGLU_ERF)])
def test_pair_tail_pieces(be, sc, orc, monkeypatch, qtype, K, op):
    monkeypatch.setenv("QMM_GEMM3_PAIR", "3")
    monkeypatch.setenv("QMM_GEMM3_TAIL", "3" if K == 1536 else "2")
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    say("pair-tail", qtype, K, op)
    got, ref = glu_case(be, sc, orc, qtype, qtype, 1850, K, 561, op, seed=521)
    assert be.last_path() == "glu-gemm-stream"
    assert rel_err(got, ref) <= TOL
    again, _ = glu_case(be, sc, orc, qtype, qtype, 1850, K, 561, op, seed=521)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))


# against the general path (two products and a GLU launch): broadcast weights over batches, a dst
# with padded columns and batches, columns of src1 at a stride
@pytest.mark.parametrize("qtype", [qmm.Q4_K, qmm.Q8_0])
def test_pair_strides_and_batches(be, sc, orc, monkeypatch, qtype):
    K, M, N, B = 512, 96, 45, 4
    say("pair strides", qtype)
    wg = sc.weights(qtype, synth.weights(qtype, 2 * M, K, seed=531), (K, M, 2))
    wu = sc.weights(qtype, synth.weights(qtype, 2 * M, K, seed=532), (K, M, 2))
    x = sc.f32(synth.activations(B * 2 * N, K, seed=533).reshape(B, 2 * N, K)).view((K, N, B), (4, 8 * K, 8 * K * N, 8 * K * N * B))
    out = []
    for env in ({"QMM_GEMM_MIN_COLS": "16"}, {"QMM_GEMM_MIN_COLS": "16", "QMM_GEMM3": "0"}):
        with monkeypatch.context() as mp:
            for k, v in env.items():
                mp.setenv(k, v)
            full = sc.f32(np.full((B, N + 3, M + 5), 7.0, np.float32))
            nb1 = 4 * (M + 5)
            y = full.view((M, N, B), (4, nb1, nb1 * (N + 3), nb1 * (N + 3) * B))
            be.mul_mat_glu(wg, wu, x, y, qmm.GLU_SWIGLU)
            be.synchronize()
            out.append((be.last_path(), be.get_f32(full).reshape(B, N + 3, M + 5)))
    assert [p for p, _ in out] == ["glu-gemm-stream", "glu-gemm-mfma"]
    a, b = out[0][1], out[1][1]
    assert np.all(a[:, N:, :] == 7.0) and np.all(a[:, :, M:] == 7.0)     # nothing written past the view
    assert rel_err(a[:, :N, :M].reshape(-1, M), b[:, :N, :M].reshape(-1, M)) <= TOL


# GEMV or GEMM by the smaller estimate: pairs that measured 12-45 % apart (op us, GEMV / GEMM)
@pytest.mark.parametrize("qtype,M,K,N,path", [
    (qmm.Q8_0, 2048, 1024, 40, "glu-fused-gemv-mfma"),            # 13.0 / 16.4
    (qmm.Q8_0, 4096, 4096, 48, "glu-fused-gemv-mfma"),            # 24.4 / 33.3
    (qmm.Q8_0, 512, 2048, 200, "glu-fused-gemv-mfma"),            # 16.4 / 23.2
    (qmm.Q8_0, 2048, 2048, 256, "glu-gemm-stream"),               # 29.6 / 23.3
    (qmm.Q4_0, 512, 2048, 200, "glu-fused-gemv-mfma"),            # 16.8 / 19.8
    (qmm.Q4_0, 4096, 2048, 128, "glu-gemm-stream"),               # 29.9 / 19.9
    (qmm.Q4_K, 512, 2048, 160, "glu-fused-gemv-mfma"),            # 15.8 / 19.6
    (qmm.Q4_K, 4096, 2048, 128, "glu-gemm-stream"),               # 29.0 / 19.9
    (qmm.Q5_K, 2048, 1024, 48, "glu-gemm-stream"),                # 23.7 / 15.9
    (qmm.Q6_K, 512, 2048, 160, "glu-fused-gemv-mfma"),            # 16.6 / 19.7
    (qmm.Q6_K, 2048, 2048, 200, "glu-gemm-stream"),               # 31.5 / 20.1
    (qmm.IQ4_XS, 1024, 1024, 96, "glu-fused-gemv-mfma"),          # 13.9 / 16.5
    (qmm.IQ4_XS, 4096, 2048, 128, "glu-gemm-stream"),             # 29.4 / 21.6
    (qmm.IQ4_NL, 512, 2048, 160, "glu-fused-gemv-mfma"),          # 16.6 / 21.6
    (qmm.IQ4_NL, 2048, 2048, 200, "glu-gemm-stream")])            # 28.2 / 22.3
def test_pair_rule(be, sc, orc, qtype, M, K, N, path):
    say("pair rule", qtype, M, K, N)
    got, ref = glu_case(be, sc, orc, qtype, qtype, M, K, N, qmm.GLU_SWIGLU, seed=541)
    assert be.last_path() == path
    assert rel_err(got, ref) <= TOL


def test_pair_captured_without_slots(orc, monkeypatch):
    """a pair whose launch has tail pieces, captured by a context that has no exchange slots: the blocks run
    whole, in every replay, with eager work between them"""
    say("pair captured cold")
    monkeypatch.setenv("QMM_GEMM3_PAIR", "3")
    monkeypatch.setenv("QMM_GEMM3_TAIL", "0")
    monkeypatch.setenv("QMM_GEMM_MIN_COLS", "16")
    q, M, K, N = qmm.Q4_K, 1850, 1024, 561                        # 256 + 5 blocks
    with qmm.Backend(0) as be:
        s = Scope(be)
        w = [s.weights(q, synth.weights(q, M, K, seed=551 + i), (K, M)) for i in range(2)]
        xs = [synth.activations(N, K, seed=555 + i) for i in range(3)]
        x, y, z = s.f32(xs[0]), s.empty_f32((M, N)), s.empty_f32((M, N))
        be.mul_mat_glu(w[0], w[1], x, y, qmm.GLU_SWIGLU)          # (whole: scratch for the activations, no slots)
        be.synchronize()
        monkeypatch.setenv("QMM_GEMM3_TAIL", "2")
        be.capture_begin()
        be.mul_mat_glu(w[0], w[1], x, y, qmm.GLU_SWIGLU)
        g = be.capture_end()
        monkeypatch.setenv("QMM_GEMM3_TAIL", "0")
        for v in xs:
            be.set_tensor(x, v.view(np.uint8).ravel())
            be.graph_launch(g)
            be.mul_mat_glu(w[0], w[1], x, z, qmm.GLU_SWIGLU)      # eager, whole blocks: the same sums
            be.synchronize()
            assert np.array_equal(be.get_f32(y).view(np.uint32), be.get_f32(z).view(np.uint32))
        g.free()
        s.close()
