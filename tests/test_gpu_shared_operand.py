"""Split-bf16 products of many (pair, spin) entries in one launch, under the
variants that split one V once for all its tau: the A-stationary tile (9) must
run, and the pre-split tiles (10 .. 13) must split V once per entry, not once per
entry and tau.  Which kernels run, and on which grid, is read from torch's
trace in a process of its own, in which torch is imported before the library
(the other order leaves torch without a GPU).

All split-bf16 variants sum in the same steps: the bits are those of variant 0
(64 x 64, bounds checked per element)."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 3), (2, 13, 40), (3, 26, 97), (2, 32, 33), (2, 33, 65), (3, 52, 61), (1, 64, 30)]   # nk, nao, NQ
SITE_ID = {"p0_gvh": 2, "sig_vg": 4}
NS = 2


def test_one_v_for_all_tau(tmp_path):
    subprocess.run([sys.executable, "-u", os.path.abspath(__file__), str(tmp_path)], check=True, timeout=110)


def traced(path, call):
    """(result, [(kernel name, grid)]) of one call."""
    import torch
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        out = call()
        torch.cuda.synchronize()
    p.export_chrome_trace(path)
    with open(path) as f:
        events = json.load(f)["traceEvents"]
    return out, [(e["name"], tuple(e["args"]["grid"])) for e in events if e.get("cat") == "kernel"]


def check(ggpu, synth, np, folder, nk, nao, NQ):
    tau, T_wt, T_tw = synth.load_ir(50.0, 1e3)
    G, _ = synth.make_green(nk, nao, NS, 50.0, tau, 81)
    k = ggpu.GwKernel(nao, NS, NQ, T_wt, T_tw, ggpu.mesh_symmetry_none((nk, 1, 1)), precision="bf16x3",
                      solver="cholesky")
    k.load_integrals(synth.make_integrals(nk, NQ, nao, 82))
    k.set_q_share(0, nk)

    def force(v):
        print(f"nk={nk} nao={nao} NQ={NQ} variant {v}", flush=True)
        table = [-1] * len(ggpu.SITES)
        for s in SITE_ID:
            table[ggpu.SITES.index(s)] = v
        k.set_variants(table)

    force(0)
    ref = k.solve(G)
    assert np.isfinite(ref).all() and np.abs(ref).max() > 0
    for v in (9, 10, 13):
        force(v)
        Sig, kernels = traced(os.path.join(folder, f"{nao}_{v}.json"), lambda: k.solve(G))
        assert np.array_equal(Sig, ref)
        if v == 9:
            for site in SITE_ID.values():
                assert any("astat_kernel" in n and n.split(">(")[0].endswith(f", {site}") for n, _ in kernels), kernels
            continue
        # matrices split: V of every entry at both sites, G of every entry at tau < nts / 2 and at all tau
        entries, nts = nk * NS, tau.size
        splits = sorted(g[2] for n, g in kernels if "fb_split_kernel" in n)
        assert splits == sorted([entries, entries * (nts // 2), entries, entries * nts]), splits
    k.close()


if __name__ == "__main__":
    import numpy as np
    import torch

    torch.zeros(1, device="cuda")
    import conftest
    package = conftest.load_package()
    import green_gpu_amd.synth as inputs
    for size in SIZES:
        check(package, inputs, np, sys.argv[1], *size)
