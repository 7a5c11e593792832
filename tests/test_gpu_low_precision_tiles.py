"""Every launch variant of the FP32 and split-bf16 products gives the same
bits: the sums run over k in the same steps whatever the tile, loader or
address width.  Sizes around the edges of the tiles and of the k steps (k tails
of 1 to 31, one and several steps), with every layout and conjugation of the
chain.  The split-bf16 reference is variant 0 (64 x 64, 64-bit addresses, bounds
checked per element); FP32's tiles share one loader, so the result is also
held against FP64.

Tolerance against FP64: three chained sums of up to nao^2 = 4225 terms, 65
rounding errors deep if they are random: 65 x 3 x 6e-8 = 1.2e-5 of the largest
element; 1e-4 leaves a factor of eight for the largest of all elements."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REFERENCE = {"bf16x3": 0, "fp32": 8}
VARIANTS = {"bf16x3": [-1, 1, 4, 5, 6, 7, 8, 9, 10, 13], "fp32": [-1, 16, 83]}


@pytest.mark.parametrize("precision", sorted(VARIANTS))
@pytest.mark.parametrize("nao,NQ,mesh", [(1, 3, (1, 1, 1)), (5, 31, (2, 1, 1)), (8, 32, (1, 1, 1)), (17, 65, (2, 1, 1)),
                                         (26, 97, (2, 1, 1)), (32, 100, (1, 1, 1)), (33, 129, (1, 1, 1)),
                                         (41, 130, (1, 1, 1)), (52, 161, (1, 1, 1)), (65, 200, (1, 1, 1))])
def test_variants_give_the_same_bits(ggpu, synth, nao, NQ, mesh, precision):
    nk, ns = int(np.prod(mesh)), 2
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, ns, 50.0, tau, 41)
    V = synth.make_integrals(nk, NQ, nao, 42)
    sym = ggpu.mesh_symmetry_none(mesh)
    k = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, sym, precision=precision)
    k.load_integrals(V)
    sites = ["p0_gv", "p0_gvh", "p0_contract", "sig_vg", "sig_py", "sig_contract"]
    table = lambda v: [v if s in sites else -1 for s in ggpu.SITES]
    k.set_variants(table(REFERENCE[precision]))
    P0, Sig = k.polarization(G, 0, 0), k.solve(G)
    assert np.isfinite(Sig).all() and np.abs(Sig).max() > 0
    for v in VARIANTS[precision]:
        print(f"{precision} nao={nao} NQ={NQ} variant {v}", flush=True)
        k.set_variants(table(v))
        assert np.array_equal(k.polarization(G, 0, 0), P0)
        assert np.array_equal(k.solve(G), Sig)
    if precision == "fp32":
        k64 = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, sym)
        k64.load_integrals(V)
        ref = k64.solve(G)
        err = np.abs(Sig - ref).max() / np.abs(ref).max()
        print(f"against FP64: {err:.1e}", flush=True)
        assert err < 1e-4
