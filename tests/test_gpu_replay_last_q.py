"""The intermediates of the last q after a replayed iteration, with a call for
another q in between: they are those of the replay's last q, under that q's
number.  A q computed by itself runs the same sums: equal bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def plan(ggpu, synth, nk, nao, NQ, seed):
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, 1, 50.0, tau, seed)
    k = ggpu.GwKernel(nao, 1, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)), solver="cholesky")
    k.load_integrals(synth.make_integrals(nk, NQ, nao, seed + 1))
    return k, G


def check(k, G, last):
    got = [k.last_polarization(w) for w in range(3)]
    assert [iq for iq, _ in got] == [last] * 3
    for w in range(3):
        assert np.array_equal(got[w][1], k.polarization(G, last, w))


@pytest.mark.parametrize("nk,share,last", [(3, (0, 1), 2), (19, (0, 1), 18), (19, (1, 4), 17)])
def test_last_q_of_a_replayed_iteration(ggpu, synth, nk, share, last):
    k, G = plan(ggpu, synth, nk, 2, 3, 91)
    k.set_q_share(*share)
    k.set_graph(True)
    print(f"nk={nk} share={share}", flush=True)
    for _ in range(3):
        S = k.solve(G)
        assert np.isfinite(S).all()
        check(k, G, last)
        k.polarization(G, 0, 1)
    assert k.graph_captures() == 1


def test_last_q_of_a_replayed_batch(ggpu, synth):
    ks, Gs = zip(*[plan(ggpu, synth, nk, 2, 3, 95) for nk in (2, 5)])
    Gd = [ggpu.DeviceArray.from_numpy(G) for G in Gs]
    Sd = [ggpu.DeviceArray.empty_like(g) for g in Gd]
    b = ggpu.GwBatch(list(ks), [g.ptr for g in Gd], [s.ptr for s in Sd])
    for _ in range(3):
        b.run()
        for k, G, last in zip(ks, Gs, (1, 4)):
            check(k, G, last)
            k.polarization(G, 0, 1)
