"""P(Omega) = (1 - P0)^-1 P0 against the oracle over the sizes where the factorisation
and solve kernels change: one block of 32 and less, remainders of one column or
row, panels of up to 64, 256 and 512 rows and longer ones, both solvers, and
for LU an indefinite 1 - P0 whose rows are interchanged.

Tolerance: a backward stable solve errs by at most about NQ eps cond of the largest
element, the sums in P0 by a few hundred eps, which the solve amplifies by
cond as well; cond is that of the oracle's 1 - P0."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,definite", [("lu", False), ("lu", True), ("cholesky", True)])
@pytest.mark.parametrize("nao,NQ", [(3, 5), (5, 31), (4, 32), (5, 33), (8, 64), (9, 65), (6, 97), (9, 154),
                                    (9, 256), (9, 257), (6, 512), (6, 513)])
def test_dyson_against_oracle(ggpu, synth, oracle, nao, NQ, solver, definite):
    mesh, ns = (1, 1, 1), 1
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(1, nao, ns, 50.0, tau, 31)
    V = synth.make_integrals(1, NQ, nao, 32)
    osym = oracle.symmetry_none(mesh, nao, NQ)
    if not definite:
        G[tau.size // 2:] *= -1.0
    P0w = oracle.tau_to_omega(oracle.gw_p0(oracle.g_full(G, osym), V, osym, 0, ns, tau.size), T_wt)
    P0w = np.stack([oracle.herm(p) for p in P0w])
    lam = max(np.abs(np.linalg.eigvalsh(p)).max() for p in P0w)
    V = V * np.sqrt(3.0 / lam)
    P0w = P0w * (3.0 / lam)
    A = np.eye(NQ) - P0w
    ref = np.linalg.solve(A, P0w)
    cond = max(np.linalg.cond(a) for a in A)
    k = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none(mesh), solver=solver)
    k.load_integrals(V)
    Pw = k.polarization(G, 0, 1)
    err, tol = max_abs(Pw, ref), cond * (NQ + 200) * np.finfo(float).eps * np.abs(ref).max()
    print(f"nao={nao} NQ={NQ} {solver} definite={definite}: cond {cond:.2g} max-abs {err:.2e} (tolerance {tol:.2e})",
          flush=True)
    assert err < tol
