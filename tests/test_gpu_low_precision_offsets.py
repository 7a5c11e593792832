"""The P0 contraction in reduced precision with a row stride of nao^2 = 4.2 M
elements: a tile of B then spans more than 4 GiB, which FP32 runs with 64-bit
offsets and split-bf16 on its tile with 64-bit addresses.  Two auxiliary functions,
four tau points.

Tolerance: a sum of n = 4.2 M products of random sign in FP32 is off by about
sqrt(n) 2^-24 = 1.2e-4 of its size, the splits and the two products before it by 1e-5;
1e-3 leaves a factor of eight.  An offset that wraps reads other elements: an
error of the size of the result."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
def test_p0_with_64_bit_offsets(ggpu, precision):
    nao, NQ, nts = 2050, 2, 4
    rng = np.random.default_rng(3)
    sym = ggpu.mesh_symmetry_none((1, 1, 1))
    G = (rng.normal(size=(nts, 1, 1, nao, nao)) + 1j * rng.normal(size=(nts, 1, 1, nao, nao))) / nao
    V = (rng.normal(size=(1, NQ, nao, nao)) + 1j * rng.normal(size=(1, NQ, nao, nao))) / nao
    print(f"P0 with 64-bit offsets, {precision}, nao={nao}", flush=True)
    kern = ggpu.GwKernel(nao, 1, NQ, np.ones((3, 2)), np.ones((4, 3)), sym, precision=precision, work_bytes=1 << 30)
    kern.load_integrals(V)
    P0 = kern.polarization(G, 0, 0)
    ref = np.empty((NQ, NQ), complex)
    for a in range(NQ):
        X = G[-1, 0, 0] @ V[0, a] @ G[0, 0, 0]          # G(beta) V^a G(0)
        for b in range(NQ):
            ref[a, b] = -2.0 * np.sum(X * np.conj(V[0, b]))
    assert max_abs(P0[0], ref) < 1e-3 * np.abs(ref).max()
