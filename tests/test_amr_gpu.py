"""GPU parity of the AMR hierarchy: the HIP path against the CPU oracle,
bit for bit (node sets, x-run/row/plane blocks, every FP32 density, every
per-node particle list in AHF's order)."""
import os
import sys

import numpy as np
import pytest

from ahf_amd import dumps

from helpers import fuzz_snapshot

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import ahf_amd
    c = ahf_amd.Context(0)
    yield c
    c.close()


def _gpu_dump(ctx, snap_path, out_path, mode=0):
    s = dumps.read_snapshot(snap_path)
    ctx.set_gather_mode(mode)
    ctx.set_particles(s.pos, s.mom)
    info = ctx.amr_build(s.L_dom, s.L_max, s.Nth_dom, s.Nth_ref)
    ctx.amr_dump(out_path)
    return info


# every deposit kernel (per-source walk, flat walk, and the per-level choice)
# must give the oracle's bits
# AUTO, SOURCE, FLAT, WAVE (every node folded by a wavefront), FLAT_WIDE (the
# flat walk with the 64-bit record offsets of levels over 4 GiB of records)
MODES = [0, 1, 2, 3, 4]


def _check(oracle, ctx, snap, tmp_path, tag, mode=0):
    o_out = str(tmp_path / f"{tag}_oracle.grid")
    g_out = str(tmp_path / f"{tag}_gpu.grid")
    n = oracle.oracle_amr_dump(snap.encode(), o_out.encode())
    assert n > 0, f"oracle failed ({n})"
    print(f"[amr-gpu] case {tag} gather mode {mode}: {os.path.getsize(snap)} B snapshot", flush=True)
    info = _gpu_dump(ctx, snap, g_out, mode)
    a, b = dumps.read_grids(g_out), dumps.read_grids(o_out)
    diffs = dumps.compare_grids(a, b)
    assert not diffs, f"{tag}: " + "; ".join(diffs[:6])
    assert info.n_levels == len(b)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("cfg,side,seed", [(1, 32, 11), (1, 64, 1001), (0, 64, 1000), (1, 48, 7), (3, 48, 5),
                                          (3, 64, 1003), (4, 64, 1004)])
def test_generated_configs(oracle, snapgen, ctx, tmp_path, cfg, side, seed, mode):
    snap = str(tmp_path / f"cfg{cfg}_{side}.snap")
    assert snapgen.ahf_snapgen_write(cfg, side, seed, snap.encode()) == 0
    _check(oracle, ctx, snap, tmp_path, f"cfg{cfg}_{side}_{seed}", mode)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("seed", list(range(0, 40)))
def test_fuzz(oracle, ctx, tmp_path, seed, mode):
    snap = str(tmp_path / f"fuzz{seed}.snap")
    fuzz_snapshot(snap, seed)
    _check(oracle, ctx, snap, tmp_path, f"fuzz{seed}", mode)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("seed", list(range(40, 52)))
def test_fuzz_non_pow2(oracle, ctx, tmp_path, seed, mode):
    snap = str(tmp_path / f"fuzz{seed}.snap")
    fuzz_snapshot(snap, seed, non_pow2=True)
    _check(oracle, ctx, snap, tmp_path, f"fuzz_np2_{seed}", mode)


@pytest.mark.parametrize("n_bg,clump", [(2000, 2500), (14000, 4000), (40000, 9000)])
def test_staged_plane_overflow(oracle, ctx, tmp_path, n_bg, clump):
    """levels that hold every octet are deposited plane by plane from LDS;
    a tight clump fills a plane's staged slots, so the nodes after it in the
    plane are walked from the position records instead (both slot counts:
    under and over two entries per node)"""
    rng = np.random.default_rng(n_bg + clump)
    bg = rng.random((n_bg, 3))
    c = np.array([0.02, 0.5, 0.97])
    cl = (c + 0.004 * rng.standard_normal((clump, 3))) % 1.0
    pos = np.concatenate([bg, cl]).astype(np.float32)
    pos[pos >= 1.0] = 0.0
    snap = str(tmp_path / f"clump{n_bg}.snap")
    dumps.write_snapshot(snap, pos, L_dom=16, L_max=128, Nth_dom=2.0, Nth_ref=3.0)
    _check(oracle, ctx, snap, tmp_path, f"clump{n_bg}_{clump}", 0)


@pytest.mark.parametrize("L,per_node,clump", [(38, 3, 0), (40, 3, 4000), (42, 1, 900), (48, 3, 4000), (50, 1, 900),
                                              (50, 4, 6000), (62, 1, 900), (64, 2, 4000)])
def test_marched_levels(oracle, ctx, tmp_path, L, per_node, clump):
    """domain grids on both sides of the size from which a level that holds
    every octet marches, with whole and partial tiles, both staging forms,
    and a clump beyond a plane's staged slots at the corner of the box (and
    on the face planes) and one inside"""
    rng = np.random.default_rng(L * 10 + per_node)
    parts = [rng.random((per_node * L ** 3, 3))]
    for c in ([0.0, 0.999, 0.0], [0.31, 0.5, 0.62]):
        parts.append((np.array(c) + 1.5 / L * rng.standard_normal((clump, 3))) % 1.0)
    pos = np.concatenate(parts).astype(np.float32)
    pos[pos >= 1.0] = 0.0
    snap = str(tmp_path / "m.snap")
    dumps.write_snapshot(snap, pos, L_dom=L, L_max=L << 4, Nth_dom=1.5 * per_node, Nth_ref=4.0)
    _check(oracle, ctx, snap, tmp_path, f"march{L}_{per_node}_{clump}", 0)


@pytest.mark.parametrize("seed", [0, 5, 161])
def test_final_lists(oracle, ctx, tmp_path, seed):
    """the final lists with offsets or entries asked for alone; the last
    level of seed 161 got its refinement's particles back"""
    snap = str(tmp_path / "rb.snap")
    fuzz_snapshot(snap, seed)
    _check(oracle, ctx, snap, tmp_path, f"lists{seed}", 0)
    info = _gpu_dump(ctx, snap, str(tmp_path / "again.grid"))
    assert (info.rolled_back == 1) == (seed == 161)
    for lev in range(info.n_levels):
        both = ctx.amr_level(lev)
        list0 = np.zeros_like(both["list0"])
        lst = np.zeros(max(int(both["list0"][-1]), 1), np.uint32)
        ctx._check(ctx.lib.ahfgpu_amr_level_copy(ctx.h, lev, None, None, None, list0.ctypes.data, None))
        ctx._check(ctx.lib.ahfgpu_amr_level_copy(ctx.h, lev, None, None, None, None, lst.ctypes.data))
        assert np.array_equal(list0, both["list0"]) and np.array_equal(lst[:int(list0[-1])], both["list"])


@pytest.mark.parametrize("seed", [0, 5, 161])
def test_final_lists_without_room(oracle, ctx, tmp_path, seed):
    """the final lists made on the host where the device has no room for their
    scratch; the last level of seed 161 got its refinement's particles back"""
    snap = str(tmp_path / "rb.snap")
    fuzz_snapshot(snap, seed)
    assert oracle.oracle_amr_dump(snap.encode(), str(tmp_path / "o.grid").encode()) > 0
    info = _gpu_dump(ctx, snap, str(tmp_path / "g.grid"))
    assert (info.rolled_back == 1) == (seed == 161)
    with_room = [ctx.amr_level(lev) for lev in range(info.n_levels)]
    try:
        ctx.set_memory_limit(1)
        ctx.amr_dump(str(tmp_path / "h.grid"))
        without = [ctx.amr_level(lev) for lev in range(info.n_levels)]
    finally:
        ctx.set_memory_limit(0)
    assert not dumps.compare_grids(dumps.read_grids(str(tmp_path / "h.grid")), dumps.read_grids(str(tmp_path / "o.grid")))
    for a, b in zip(with_room, without):
        assert np.array_equal(a["list0"], b["list0"]) and np.array_equal(a["list"], b["list"])


@pytest.mark.parametrize("n", [32, 33, 1024, 1025, 4096, 4097, 8193, 30000])
def test_fine_buckets(oracle, ctx, tmp_path, n):
    """a node's bucket at the edges of the three ways to split it among the
    children (one thread, one wavefront, one workgroup in steps of 4096)"""
    rng = np.random.default_rng(n)
    lat = (np.stack(np.meshgrid(*[np.arange(16)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) / 16
    lat = lat[np.any(np.floor(lat * 16) != 7, axis=1)]
    cell = (7 + 0.998 * rng.random((n, 3))) / 16
    pos = np.concatenate([np.repeat(lat, 8, 0), cell]).astype(np.float32)
    snap = str(tmp_path / "b.snap")
    dumps.write_snapshot(snap, pos, L_dom=16, L_max=64, Nth_dom=4.0, Nth_ref=2.0)
    _check(oracle, ctx, snap, tmp_path, f"bucket{n}", 0)


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("L,clump,dyadic", [(16, 2047, False), (16, 9000, False), (10, 20000, False), (16, 70000, False),
                                            (16, 20000, True), (10, 4000, True)])
def test_huge_nodes(oracle, ctx, tmp_path, L, clump, dyadic, mode):
    """nodes on both sides of the contribution count from which a workgroup
    folds a node, over position and weight records, blocks of every length;
    positions on a dyadic lattice make steps that are exact halves"""
    rng = np.random.default_rng(clump + L)
    c = np.array([0.5 + 0.3 / L, 0.02, 0.31])
    cl = c + rng.standard_normal((clump, 3)) * np.array([0.05, 0.2, 0.1])[rng.integers(0, 3, (clump, 1))] / L
    if dyadic:
        cl = np.round(cl * 1024.0) / 1024.0
    pos = np.concatenate([rng.random((500, 3)), cl % 1.0]).astype(np.float32)
    pos[pos >= 1.0] = 0.0
    snap = str(tmp_path / "huge.snap")
    dumps.write_snapshot(snap, pos, L_dom=L, L_max=L << 6, Nth_dom=4.0, Nth_ref=4.0)
    _check(oracle, ctx, snap, tmp_path, f"huge{L}_{clump}_{dyadic}", mode)


@pytest.mark.parametrize("sched", [dict(kmax_big=8, kmax_small=8, march_zn=8), dict(kmax_big=1000, kmax_small=300, march_zn=16)])
@pytest.mark.parametrize("cfg,side,seed", [(1, 64, 1001), (3, 64, 1003)])
def test_schedule_variants(oracle, snapgen, ctx, tmp_path, cfg, side, seed, sched):
    """the deposit's fold threshold and the march's planes per workgroup
    change nothing in the hierarchy"""
    snap = str(tmp_path / f"cfg{cfg}_{side}.snap")
    assert snapgen.ahf_snapgen_write(cfg, side, seed, snap.encode()) == 0
    before = ctx.schedule()
    try:
        ctx.set_schedule(**sched)
        _check(oracle, ctx, snap, tmp_path, f"cfg{cfg}_{side}_{seed}_sched", 0)
    finally:
        ctx.set_schedule(**before)
