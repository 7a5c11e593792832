"""The FP64 GEMM kernel's tiles through the GW chain: extents around every
tile edge, K tails of every remainder, the forced tiles, and operands whose
strides need 64-bit offsets.

Tolerance: a sum of n products carries at most about n * 2^-53 of the sum of
their magnitudes; the longest sums here (nao^2 * NQ ~ 1e6 terms, through P0,
the Dyson solve and Sigma) stay below 1e-10 of the largest |Sigma|."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu

SIZES = [(1, 3), (5, 16), (15, 33), (17, 48), (26, 65), (33, 47), (49, 64), (64, 81), (72, 97), (81, 60), (97, 113),
         (113, 49)]


@pytest.mark.parametrize("nao,NQ", SIZES)
def test_gw_fp64_tile_edges(ggpu, synth, oracle, nao, NQ):
    mesh, ns = (1, 1, 1), 2
    sym = ggpu.mesh_symmetry_none(mesh)
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(sym.nk, nao, ns, 50.0, tau, 11)
    V = synth.make_integrals(sym.nk, NQ, nao, 12, sigma=0.5 / np.sqrt(nao * nao))
    print(f"FP64 tiles nao={nao} NQ={NQ}", flush=True)
    kern = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, sym, solver="cholesky")
    kern.load_integrals(V)
    S = kern.solve(G)
    ref = oracle.gw_solve(G, V, oracle.symmetry_none(mesh, nao, NQ), T_wt, T_tw, solver="cholesky")
    assert max_abs(S, ref) < 1e-10 * np.abs(ref).max()
    for variant in (8, 16, 83):
        v = [-1] * len(ggpu.SITES)
        for s in ("p0_gv", "p0_gvh", "p0_contract", "sig_vg", "sig_py", "sig_contract"):
            v[ggpu.SITES.index(s)] = variant
        kern.set_variants(v)
        assert np.array_equal(kern.solve(G), S), variant


def test_p0_with_64_bit_offsets(ggpu):
    """P0 contraction with a row stride of nao^2 = 2.4 M elements (a tile of
    B then spans more than 4 GiB), two auxiliary functions, four tau points."""
    nao, NQ, nts = 1560, 2, 4
    rng = np.random.default_rng(3)
    sym = ggpu.mesh_symmetry_none((1, 1, 1))
    G = (rng.normal(size=(nts, 1, 1, nao, nao)) + 1j * rng.normal(size=(nts, 1, 1, nao, nao))) / nao
    V = (rng.normal(size=(1, NQ, nao, nao)) + 1j * rng.normal(size=(1, NQ, nao, nao))) / nao
    print("P0 with 64-bit offsets, nao=1560", flush=True)
    kern = ggpu.GwKernel(nao, 1, NQ, np.ones((3, 2)), np.ones((4, 3)), sym, work_bytes=1 << 30)
    kern.load_integrals(V)
    P0 = kern.polarization(G, 0, 0)
    ref = np.empty((NQ, NQ), complex)
    for a in range(NQ):
        X = G[-1, 0, 0] @ V[0, a] @ G[0, 0, 0]          # G(beta) V^a G(0)
        for b in range(NQ):
            ref[a, b] = -2.0 * np.sum(X * np.conj(V[0, b]))
    assert max_abs(P0[0], ref) < 1e-10 * np.abs(ref).max()
