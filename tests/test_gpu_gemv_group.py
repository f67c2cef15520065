"""One-column MUL_MAT nodes of a graph in one launch (k_gemv_fq1), and the one-product form, through the C
ABI: against the CPU oracle, and bit for bit against the nodes run one by one (the same sums in the
same order).

Bar against the oracle: MUL_MAT's own (rel_err <= 1e-3)."""
import numpy as np
import pytest

from arcint_amd import qmm, synth
from conftest import rel_err
from test_gpu_parity import TOL, TYPES, Scope, be, say, sc  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

# rows x K: a partial tile, one row, one wave's worth of K past a work-group's, the longest K not first
SHAPES = [(300, 2304), (1, 2560), (130, 5120), (64, 1280), (100, 2304), (65, 2304), (128, 2304), (200, 2304), (70, 2304)]


def build(be, sc, qtype, shapes, seed):
    xs, nodes, refs = {}, [], []
    for i, (M, K) in enumerate(shapes):
        if K not in xs:
            x = synth.activations(1, K, seed + K)
            xs[K] = (x, sc.f32(x))
        raw = synth.weights(qtype, M, K, seed + i)
        y = sc.f32(np.full((1, M), 3.0, np.float32))
        nodes.append((qmm.OP_MUL_MAT, sc.weights(qtype, raw, (K, M)), xs[K][1], None, y))
        refs.append((raw, M, K, xs[K][0]))
    return nodes, refs


@pytest.mark.parametrize("qtype", TYPES)
def test_group_matches_single(be, sc, orc, monkeypatch, qtype):
    """nine products (one more than a launch takes) of unequal rows and K"""
    say("group", qtype)
    nodes, refs = build(be, sc, qtype, SHAPES, 601)
    out = []
    for env in ("1", "0"):
        monkeypatch.setenv("QMM_GEMV_GROUP", env)
        for _ in range(2):                                   # (the slots empty again after each)
            be.graph_compute(nodes)
        be.synchronize()
        assert be.last_path() == "gemv-fq"
        out.append([be.get_f32(n[4]).copy() for n in nodes])
        for n in nodes:
            be.set_tensor(n[4], np.zeros(n[4].ne[0], np.float32))
    for i, (raw, M, K, x) in enumerate(refs):
        assert rel_err(out[0][i].reshape(1, M), orc.mul_mat(qtype, raw, M, K, x)) <= TOL, (M, K)
        assert np.array_equal(out[0][i].view(np.uint32), out[1][i].view(np.uint32)), (M, K)


def test_group_keeps_order(be, sc, orc):
    """a node that reads what an earlier one writes, one that writes an earlier one's dst or input, and
    a node of another type end a run: the results are those of the nodes in order"""
    say("group order")
    q, K, M = qmm.Q4_K, 2304, 2304
    raws = [synth.weights(q, M, K, 640 + i) for i in range(4)]
    w = [sc.weights(q, r, (K, M)) for r in raws]
    r6 = synth.weights(qmm.Q6_K, 96, K, 650)
    w6 = sc.weights(qmm.Q6_K, r6, (K, 96))
    x0 = synth.activations(1, K, 651)
    x, a, b, y6 = sc.f32(x0), sc.f32(np.zeros((1, M))), sc.f32(np.zeros((1, M))), sc.f32(np.zeros((1, 96)))
    mm = qmm.OP_MUL_MAT
    # a = w0 x; b = w1 a (reads a); a = w2 x (writes a, which b's node read); y6 = w6 b; x = w3 b (writes x)
    be.graph_compute([(mm, w[0], x, None, a), (mm, w[1], a, None, b), (mm, w[2], x, None, a), (mm, w6, b, None, y6),
                      (mm, w[3], b, None, x)])
    be.synchronize()
    ra = orc.mul_mat(q, raws[0], M, K, x0)
    rb = orc.mul_mat(q, raws[1], M, K, np.ascontiguousarray(ra, np.float32))
    assert rel_err(be.get_f32(a).reshape(1, M), orc.mul_mat(q, raws[2], M, K, x0)) <= TOL
    got_b = be.get_f32(b).reshape(1, M)
    # (a's last bit may move a code of w1's activations: one step of 1/127 of its super-block's largest)
    assert rel_err(got_b, rb) <= 2e-2
    assert rel_err(be.get_f32(y6).reshape(1, 96), orc.mul_mat(qmm.Q6_K, r6, 96, K, got_b)) <= TOL
    assert rel_err(be.get_f32(x).reshape(1, M), orc.mul_mat(q, raws[3], M, K, got_b)) <= TOL




def test_group_captured(be, sc, orc):
    """the run inside a captured graph, replayed on new inputs with eager work between"""
    say("group captured")
    q, K = qmm.Q5_K, 2304
    nodes, refs = build(be, sc, q, [(300, K), (130, K), (70, K)], 661)
    be.graph_compute(nodes)
    be.synchronize()
    be.capture_begin()
    be.graph_compute(nodes)
    g = be.capture_end()
    for r in range(3):
        x = synth.activations(1, K, 670 + r)
        be.set_tensor(nodes[0][2], x.view(np.uint8).ravel())
        be.graph_launch(g)
        be.synchronize()
        got = [be.get_f32(n[4]).copy() for n in nodes]
        be.graph_compute(nodes)
        be.synchronize()
        for (raw, M, _, _), v, n in zip(refs, got, nodes):
            assert rel_err(v.reshape(1, M), orc.mul_mat(q, raw, M, K, x)) <= TOL
            assert np.array_equal(v.view(np.uint32), be.get_f32(n[4]).view(np.uint32))
    g.free()


# K of 3 to 8 groups whole in one work-group (every order of sums that differs from the split plan's), and
# 14336 x 4096's one-slice plan of 16 waves (Q6_K's stays split): a run keeps each node's own plan
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("shapes", [[(70, 768), (130, 768)], [(512, 1536), (64, 1536), (100, 1536)],
                                    [(512, 2048), (256, 2048), (300, 2304), (100, 2048)], [(14336, 4096)] * 2])
def test_group_keeps_each_plans_sums(be, sc, orc, monkeypatch, qtype, shapes):
    say("group one-slice", qtype, shapes)
    nodes, refs = build(be, sc, qtype, shapes, 681)
    out = []
    for env in ("1", "0"):
        monkeypatch.setenv("QMM_GEMV_GROUP", env)
        for n in nodes:
            be.set_tensor(n[4], np.zeros(n[4].ne[0], np.float32))
        be.graph_compute(nodes)
        be.synchronize()
        out.append([be.get_f32(n[4]).copy() for n in nodes])
    for i, (raw, M, K, x) in enumerate(refs):
        assert np.array_equal(out[0][i].view(np.uint32), out[1][i].view(np.uint32)), (M, K)
        if M < 1000:
            assert rel_err(out[0][i].reshape(1, M), orc.mul_mat(qtype, raw, M, K, x)) <= TOL, (M, K)
