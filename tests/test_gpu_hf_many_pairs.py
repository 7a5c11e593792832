"""The fused HF exchange where a workgroup sums several pairs (64 k points and
more): the next pair's V and D, its transpose and conjugation, a last chunk of fewer
pairs, staged batches, and more k than one launch's partial sums hold.

Tolerance: as in the test of the HF sizes, 1e-12 of the largest |F|."""
import numpy as np
import pytest

from conftest import max_abs
from test_gpu_hf_sizes import system

pytestmark = pytest.mark.gpu

CASES = [  # nk (odd: two pairs per chunk leave one), nao, NQ, ns, time reversal, residence
    (113, 5, 1, 2, False, "device"),
    (67, 17, 3, 2, False, "host"),
    (67, 33, 2, 1, True, "device"),
    (67, 48, 1, 1, True, "host"),
    (67, 49, 1, 2, False, "device"),      # 22 Mi elements of partial sums: several launches of 16 Mi
]


@pytest.mark.parametrize("nk,nao,NQ,ns,tr,where", CASES)
def test_hf_many_pairs(ggpu, oracle, nk, nao, NQ, ns, tr, where):
    sym, V, D, S = system(oracle, (nk, 1, 1), nao, NQ, ns, tr, False)
    print(f"HF nk={nk} nao={nao} NQ={NQ} ns={ns} tr={tr} {where}", flush=True)
    ref = oracle.hf_solve(D, V, sym, ns, S, 0.3)
    scale = np.abs(ref).max()
    k = ggpu.HfKernel(nao, ns, NQ, sym, madelung=0.3, S_k=S, integrals=where)
    k.load_integrals(V)
    for _ in range(2):
        F = k.solve(D)
        assert max_abs(F, ref) < 1e-12 * scale
    K = k.exchange(D)
    if where == "device":                 # the static scratch holds 4 Mi elements
        Dd = ggpu.DeviceArray.from_numpy(D)
        Kd = ggpu.DeviceArray.empty_like(Dd)
        assert ggpu.lib().ggpu_hf_exchange_device_noalloc(k._h, Dd.ptr, Kd.ptr) == 0
        assert np.array_equal(Kd.numpy(), K)
    k.set_k_share(1, 3)
    part = k.solve(D)
    rows = np.arange(sym.ink) % 3 == 1
    assert np.array_equal(part[:, rows], F[:, rows]) and not part[:, ~rows].any()
