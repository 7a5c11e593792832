"""The Dyson buffers of a plan follow its share of the q: their memory is given
back, the last q's intermediates are kept, and the partial Sigma of the shares
is the same whatever share the plan had before.

Equal bits: each q runs the same sums in every share."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["lu", "cholesky"])
def test_dyson_buffers_follow_the_share(ggpu, synth, solver):
    nk, nao, NQ = 8, 2, 300
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, 1, 50.0, tau, 101)
    V = synth.make_integrals(nk, NQ, nao, 102, sigma=0.05)

    def plan():
        k = ggpu.GwKernel(nao, 1, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)), solver=solver)
        k.load_integrals(V)
        return k

    k = plan()
    k.solve(G)
    before = [k.last_polarization(w) for w in range(3)]
    free = ggpu.device_memory()[0]
    k.set_q_share(3, nk)
    # all slots of P0(Omega) and of the factor but one: as many as 1 GiB holds (six)
    slot = 2 * 16 * k.nw_b * NQ * NQ
    given_back = ggpu.device_memory()[0] - free
    print(f"{solver}: given back {given_back / 1e6:.0f} MB", flush=True)
    assert given_back > 0.9 * ((1 << 30) // slot - 1) * slot
    for w in range(3):
        iq, P = k.last_polarization(w)
        assert iq == before[w][0] and np.array_equal(P, before[w][1])
    part = k.solve(G)
    assert np.array_equal(k.last_polarization(1)[1], k.polarization(G, 3, 1))
    fresh = plan()
    fresh.set_q_share(3, nk)
    assert np.array_equal(fresh.solve(G), part)
    k.set_q_share(1, 3)
    wider = k.solve(G)
    fresh.set_q_share(1, 3)
    assert np.array_equal(fresh.solve(G), wider)


def test_replays_follow_a_changed_share(ggpu, synth):
    """A plan's graph and a batch's are captured again on the new buffers."""
    nk, nao, NQ = 8, 2, 3
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, 1, 50.0, tau, 111)
    V = synth.make_integrals(nk, NQ, nao, 112)

    def plan(rank, size):
        k = ggpu.GwKernel(nao, 1, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)))
        k.load_integrals(V)
        k.set_q_share(rank, size)
        return k

    want = {s: plan(*s).solve(G) for s in [(0, 1), (2, 8), (1, 3)]}
    single, ks = plan(0, 1), [plan(0, 1), plan(2, 8)]
    single.set_graph(True)
    Gd = ggpu.DeviceArray.from_numpy(G)
    Sd = [ggpu.DeviceArray.empty_like(Gd) for _ in ks]
    batch = ggpu.GwBatch(ks, [Gd.ptr] * 2, [s.ptr for s in Sd])
    for a, b in [((0, 1), (2, 8)), ((2, 8), (1, 3)), ((0, 1), (0, 1)), ((1, 3), (2, 8))]:
        print(f"shares {a} {b}", flush=True)
        single.set_q_share(*a)
        ks[0].set_q_share(*a)
        ks[1].set_q_share(*b)
        for _ in range(3):
            assert np.array_equal(single.solve(G), want[a])
            batch.run()
            assert np.array_equal(Sd[0].numpy(), want[a]) and np.array_equal(Sd[1].numpy(), want[b])
