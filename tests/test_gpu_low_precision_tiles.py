"""Every launch variant of the split-bf16 products gives the same bits: the
sums run over k in the same steps whatever the tile, loader or address width.
Sizes around the edges of the tiles and of the 32 k per step (k tails of 1 to
31, one and several k steps), with every layout and conjugation of the chain.
Variant 0 (64 x 64, 64-bit addresses, bounds checked per element) is the
reference; its accuracy is what the parity tests check."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VARIANTS = {"bf16x3": [-1, 1, 4, 5, 6, 7, 8, 9, 10, 13]}


@pytest.mark.parametrize("precision", sorted(VARIANTS))
@pytest.mark.parametrize("nao,NQ,mesh", [(1, 3, (1, 1, 1)), (5, 31, (2, 1, 1)), (8, 32, (1, 1, 1)), (17, 65, (2, 1, 1)),
                                         (26, 97, (2, 1, 1)), (32, 100, (1, 1, 1)), (33, 129, (1, 1, 1)),
                                         (52, 161, (1, 1, 1)), (65, 200, (1, 1, 1))])
def test_variants_give_the_same_bits(ggpu, synth, nao, NQ, mesh, precision):
    nk, ns = int(np.prod(mesh)), 2
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, ns, 50.0, tau, 41)
    V = synth.make_integrals(nk, NQ, nao, 42)
    k = ggpu.GwKernel(nao, ns, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none(mesh), precision=precision)
    k.load_integrals(V)
    sites = ["p0_gv", "p0_gvh", "p0_contract", "sig_vg", "sig_py", "sig_contract"]
    table = lambda v: [v if s in sites else -1 for s in ggpu.SITES]
    k.set_variants(table(0))
    P0, Sig = k.polarization(G, 0, 0), k.solve(G)
    assert np.isfinite(Sig).all() and np.abs(Sig).max() > 0
    for v in VARIANTS[precision]:
        print(f"{precision} nao={nao} NQ={NQ} variant {v}", flush=True)
        k.set_variants(table(v))
        assert np.array_equal(k.polarization(G, 0, 0), P0)
        assert np.array_equal(k.solve(G), Sig)
