"""The kernels and grids of a split-bf16 product Y1[t] = V G(t) of many (pair, spin)
entries in one launch, from a host-only build of the dispatch that launches
nothing: the A-stationary tile (variant 9) runs wherever it is forced and applies,
and the pre-split tiles (10 .. 13) split V once per entry, not once per entry and
tau, on grids within the device's limits."""
import os
import re
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "green-gpu_amd", "csrc")
TILE_COLUMNS = {10: 128, 11: 128, 12: 128, 13: 192}
GiB = 1 << 30


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("launches") / "split_bf16_launches")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-std=c++17", "-O1", "--offload-arch=gfx950",
                    "--offload-host-only", "-w", "-I", CSRC, "-x", "hip",
                    os.path.join(HERE, "launches", "split_bf16_launches.hip"), "-no-hip-rt", "-o", exe], check=True)
    return exe


def launches(program, *args):
    """[(kernel, (x, y, z))] of VARIANT M N K NB0 NB1 WORKSPACE_BYTES."""
    r = subprocess.run([program] + [str(a) for a in args], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    return [(line.split()[0], tuple(int(x) for x in line.split()[1:])) for line in r.stdout.splitlines()]


SIZES = [  # nao, NQ, tau, entries
    (1, 3, 2, 2), (13, 40, 31, 4), (26, 97, 62, 16), (32, 33, 31, 1), (33, 65, 55, 6), (52, 61, 62, 7), (64, 30, 110, 2)]


@pytest.mark.parametrize("nao,NQ,nts,entries", SIZES)
def test_a_stationary_tile_runs_where_it_is_forced(program, nao, NQ, nts, entries):
    (name, grid), = launches(program, 9, NQ * nao, nao, nao, nts, entries, GiB)
    assert "gemm_bf16x3_astat_kernel" in name
    tiles = -(-NQ * nao // 64) * -(-nao // 64)
    # every entry's tau in runs of at most 16
    runs = grid[0] / (tiles * entries)
    assert runs == int(runs) and -(-nts // 16) <= runs <= nts and grid[1:] == (1, 1)


def test_a_stationary_tile_gives_way_to_its_own_size(program):
    for size in [(66, 40, 31, 4), (13, 40, 1, 4)]:          # K > 64; one tau
        nao, NQ, nts, entries = size
        (name, _), = launches(program, 9, NQ * nao, nao, nao, nts, entries, GiB)
        assert "gemm_bf16x3_big_kernel" in name and "Li2ELi2E" in name


@pytest.mark.parametrize("variant", sorted(TILE_COLUMNS))
@pytest.mark.parametrize("nao,NQ,nts,entries,workspace",
                         [s + (100 * GiB,) for s in SIZES] + [(2, 3, 110, 600, 100 * GiB), (2, 3, 62, 1058, 100 * GiB),
                                                              (33, 65, 55, 6, 12 << 20), (33, 65, 55, 6, 4 << 20)])
def test_presplit_tiles_split_v_once(program, variant, nao, NQ, nts, entries, workspace):
    k_blocks, M, N = -(-nao // 32), NQ * nao, nao
    rows_v = -(-M // 128) * 8
    rows_g = -(-N // TILE_COLUMNS[variant]) * (TILE_COLUMNS[variant] // 16)
    out = launches(program, variant, M, N, nao, nts, entries, workspace)
    assert len(out) % 3 == 0
    v = g = batches = 0
    parts_of_one_entry = set()
    for (sv, gv), (sg, gg), (mm, gm) in zip(out[::3], out[1::3], out[2::3]):
        assert "fb_split_kernel" in sv and "fb_split_kernel" in sg and "gemm_bf16x3_frag_kernel" in mm
        assert gv[1] == rows_v and gg[1] == rows_g and max(gv[2], gg[2], gv[1], gg[1]) <= 65535
        assert (gv[2] * rows_v + gg[2] * rows_g) * k_blocks * 4096 <= workspace
        v, g = v + gv[2], g + gg[2]
        batches += gm[0] // (rows_v // 8 * (rows_g * 16 // TILE_COLUMNS[variant]))
        parts_of_one_entry.add(gg[2] < nts)
    assert g == batches == nts * entries
    if parts_of_one_entry == {False}:
        assert v == entries
    else:
        assert workspace < 5 << 20            # an entry has 5 to 7 MB of planes


def test_presplit_tile_without_room_takes_the_register_tile(program):
    (name, _), = launches(program, 10, 65 * 33, 33, 33, 55, 6, 100)
    assert re.search(r"gemm_bf16x3_big_kernel\w*Li5ELi2E", name)
