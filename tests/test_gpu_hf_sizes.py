"""HF (K, J, Ewald and the energy) against the oracle over the sizes where its
kernels change: 16-row blocks and their remainders, one and many auxiliary
functions, pairs that are stored transposed or conjugated (time reversal),
every residence, spins and the two-component form.

Tolerance: each element of F is a sum of at most nk NQ nao^2 products, so
1e-12 of the largest |F| leaves more than three digits above its rounding."""
import numpy as np
import pytest

from conftest import max_abs

pytestmark = pytest.mark.gpu


def time_reversal_tables(mesh, nso, NQ):
    """k and -k related by time reversal, pairs reduced accordingly."""
    import gw_oracle as oracle
    sym = oracle.symmetry_none(mesh, nso, NQ)
    n = np.array(mesh)
    nk = sym.nk
    i = np.arange(nk)
    xyz = np.stack([i // (n[1] * n[2]), (i // n[2]) % n[1], i % n[2]], axis=1)
    m = (-xyz) % n
    minus = (m[:, 0] * n[1] + m[:, 1]) * n[2] + m[:, 2]
    rep = np.minimum(i, minus)
    r2f = np.unique(rep)
    sym.ink = sym.inq = len(r2f)
    sym.k_full_to_reduced = sym.q_full_to_reduced = np.searchsorted(r2f, rep).astype(np.int64)
    sym.k_reduced_to_full = sym.q_reduced_to_full = r2f.astype(np.int64)
    sym.k_tr_conj = sym.q_tr_conj = (i > minus).astype(np.int64)
    sym.k_stars = sym.q_stars = [np.nonzero(rep == r)[0] for r in r2f]
    npair = nk * (nk + 1) // 2
    conj, trans, pos = np.arange(npair), np.arange(npair), np.full(npair, -1)
    stored = 0
    for a in range(nk):
        for b in range(a + 1):
            p, x, y = a * (a + 1) // 2 + b, minus[a], minus[b]
            o = x * (x + 1) // 2 + y if x >= y else y * (y + 1) // 2 + x
            if o < p:
                (conj if x >= y else trans)[p] = o
            else:
                pos[p] = stored
                stored += 1
    sym.conj_kpair, sym.trans_kpair, sym.irre_pos, sym.num_kpair_stored = conj, trans, pos, stored
    return sym


def system(oracle, mesh, nao, NQ, ns, tr, x2c, seed=5):
    rng = np.random.default_rng(seed)
    nso = 2 * nao if x2c else nao
    sym = time_reversal_tables(mesh, nso, NQ) if tr else oracle.symmetry_none(mesh, nso, NQ)
    z = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)
    V = z(sym.num_kpair_stored, NQ, nao, nao) / nao
    D = z(ns, sym.ink, nso, nso) / nso
    D = D + np.conj(np.swapaxes(D, -1, -2))
    S = np.eye(nso) + 0.05 * (lambda x: x + np.conj(np.swapaxes(x, -1, -2)))(z(ns, sym.ink, nso, nso) / nso)
    return sym, V, D, S


CASES = [  # mesh, nao, NQ, ns, time reversal, two-component, residence
    ((1, 1, 1), 1, 1, 1, False, False, "device"),
    ((2, 1, 1), 5, 3, 2, False, False, "device"),
    ((3, 1, 1), 15, 70, 2, True, False, "device"),
    ((3, 2, 1), 16, 9, 1, True, False, "host"),
    ((2, 2, 1), 17, 65, 1, False, False, "device"),
    ((3, 1, 1), 26, 40, 2, True, False, "device"),
    ((2, 1, 1), 31, 33, 1, False, True, "device"),
    ((2, 1, 1), 32, 20, 2, False, False, "host"),
    ((3, 1, 1), 33, 50, 2, True, False, "device"),
    ((2, 1, 1), 47, 37, 1, False, False, "device"),
    ((2, 1, 1), 49, 20, 2, False, False, "device"),
    ((3, 1, 1), 57, 21, 1, True, False, "device"),
    ((2, 1, 1), 58, 21, 2, False, False, "device"),
    ((1, 1, 1), 70, 300, 1, False, True, "device"),
]


@pytest.mark.parametrize("mesh,nao,NQ,ns,tr,x2c,where", CASES)
def test_hf_sizes(ggpu, oracle, mesh, nao, NQ, ns, tr, x2c, where):
    sym, V, D, S = system(oracle, mesh, nao, NQ, ns, tr, x2c)
    print(f"HF mesh={mesh} nao={nao} NQ={NQ} ns={ns} tr={tr} x2c={x2c} {where}", flush=True)
    if x2c:
        ref = oracle.hf_solve_x2c(D, V, sym, S, 0.3)
        refK = oracle.hf_exchange_x2c(D, V, sym)
    else:
        ref = oracle.hf_solve(D, V, sym, ns, S, 0.3)
        refK = oracle.hf_exchange(D, V, sym, ns)
    k = ggpu.HfKernel(nao, ns, NQ, sym, madelung=0.3, S_k=S, nso=D.shape[-1], integrals=where)
    k.load_integrals(V)
    scale = max(np.abs(ref).max(), np.abs(refK).max())
    for _ in range(2):                                   # the second pass finds used buffers
        F = k.solve(D)
        assert max_abs(F, ref) < 1e-12 * scale
        e = oracle.hf_energy(D, ref, sym)
        assert abs(k.energy() - e) < 1e-12 * D.size * scale
    assert max_abs(k.exchange(D), refK) < 1e-12 * scale
    k.set_k_share(1, 2)
    part = k.solve(D)
    rows = np.arange(sym.ink) % 2 == 1
    assert np.array_equal(part[:, rows], F[:, rows]) and not part[:, ~rows].any()
