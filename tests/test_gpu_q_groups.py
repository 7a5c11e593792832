"""GW iterations whose q are solved in several groups of Dyson equations, against
the oracle and against one q at a time.

Tolerance: Sigma sums some 1e3 products of six chained contractions in 64 bits
around a Dyson solve of condition below 10: 1e-12 of its maximum, held to 1e-11.
A q computed by itself runs the same sums: equal bits."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["lu", "cholesky"])
@pytest.mark.parametrize("nk,share", [(2, (0, 1)), (10, (0, 1)), (19, (0, 1)), (19, (1, 2)), (3, (2, 3))])
def test_groups_of_q(ggpu, synth, oracle, nk, share, solver):
    nao, NQ, ns, mesh = 2, 3, 1, (nk, 1, 1)
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    sym = ggpu.mesh_symmetry_none(mesh)
    G, _ = synth.make_green(nk, nao, ns, 50.0, tau, 41)
    V = synth.make_integrals(nk, NQ, nao, 42)
    k = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, sym, solver=solver)
    k.load_integrals(V)
    S = np.zeros((tau.size, ns, nk, nao, nao), complex)
    for rank in range(share[1]):
        k.set_q_share((share[0] + rank) % share[1], share[1])
        S = S + k.solve(G)
    last = [k.last_polarization(w) for w in range(3)]
    mine = list(range((share[0] + share[1] - 1) % share[1], nk, share[1]))
    assert all(iq == mine[-1] for iq, _ in last)
    for w in range(3):
        assert np.array_equal(last[w][1], k.polarization(G, mine[-1], w))
    ref = oracle.gw_solve(G, V, oracle.symmetry_none(mesh, nao, NQ), T_wt, T_tw, solver=solver)
    err = max_abs(S, ref)
    print(f"nk={nk} share={share} {solver}: max-abs {err:.2e} of {np.abs(ref).max():.2e}", flush=True)
    assert err < 1e-11 * np.abs(ref).max()
