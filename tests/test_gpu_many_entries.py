"""Split-bf16 products of many (k, spin) entries sent as one launch, under the
variants that split their operands once: the number of batches, entries x tau,
passes 65535, the limit of the split kernel's grid.

Every split-bf16 variant sums in the same steps: equal bits.  Against the oracle
the operands carry 16 bits (2^-17 = 8e-6 each, three chained products and a sum
over 300 k of random sign), held to 1e-3 of the largest |Sigma|."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu


def test_presplit_tiles_take_any_number_of_batches(ggpu, synth):
    nk, ns, nao, NQ = 300, 2, 2, 3
    tau, T_wt, T_tw = synth.load_ir(100.0, 1e4)
    assert nk * ns * tau.size > 65535
    G, _ = synth.make_green(nk, nao, ns, 100.0, tau, 71)
    V = synth.make_integrals(nk, NQ, nao, 72)
    k = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)), precision="bf16x3",
                      solver="cholesky")
    k.load_integrals(V)
    k.set_q_share(7, nk)                 # one q of the 300
    Sig = k.solve(G)
    assert np.isfinite(Sig).all() and np.abs(Sig).max() > 0
    for v in (10, 11, 12, 13):
        print(f"{nk * ns} entries x {tau.size} tau, variant {v}", flush=True)
        table = [-1] * len(ggpu.SITES)
        for s in ("p0_gv", "p0_gvh", "p0_contract", "sig_vg", "sig_py", "sig_contract"):
            table[ggpu.SITES.index(s)] = v
        k.set_variants(table)
        assert np.array_equal(k.solve(G), Sig)
    k64 = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)), solver="cholesky")
    k64.load_integrals(V)
    k64.set_q_share(7, nk)
    ref = k64.solve(G)
    err = max_abs(Sig, ref) / np.abs(ref).max()
    print(f"against FP64: {err:.1e}", flush=True)
    assert err < 1e-3
