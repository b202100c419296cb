"""GPU parity of sort + unbinding (and of the rem_outsideRvir cuts around
it) against the CPU oracle: identical membership and order for every halo,
identical M_vir, R_vir, ovdens; Phi0 within the FP64 rounding of a parallel
prefix sum."""
import ctypes

import numpy as np
import pytest

from ahf_amd import dumps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import ahf_amd
    c = ahf_amd.Context(0)
    yield c
    c.close()


def _run_gpu(ctx, s, mode, band=0.0, split=0):
    ctx.set_unbind_split(split)
    ctx.set_particles(s.pos, s.mom)
    ctx.set_halos(s.centre, s.halo_npart, s.ipart)
    info = ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=mode, band=band)
    return info, ctx.unbind_results()


def _compare(ref, npart, props, lists, tag):
    bad = []
    for h in range(len(lists)):
        if int(ref.npart[h]) != int(npart[h]) or not np.array_equal(ref.ipart[h], lists[h]):
            bad.append(h)
    assert not bad, f"{tag}: {len(bad)} haloes differ, first {bad[:5]}"
    assert np.array_equal(ref.M_vir, props[:, 0])
    set_ = (props[:, 5].astype(np.int64) & 2) != 0
    assert np.array_equal(ref.R_vir[set_], props[set_, 1])
    big = ref.npart > 0
    rel = np.abs(ref.Phi0[big] - props[big, 2]) / np.maximum(np.abs(ref.Phi0[big]), 1e-300)
    assert rel.size == 0 or rel.max() < 1e-9, f"{tag}: Phi0 rel err {rel.max():.2e}"


# split: 0 the default threshold, 32 every halo of 32 members or more through
# the split path, -1 none
@pytest.mark.parametrize("split", [0, 32, -1])
@pytest.mark.parametrize("cfg,side,seed,mode", [(1, 64, 1001, 0), (1, 64, 1001, 1), (0, 64, 1000, 0),
                                                (2, 2000, 1002, 0), (2, 300, 7, 1), (4, 96, 1004, 0)])
def test_unbind_matches_oracle(oracle, snapgen, ctx, tmp_path, cfg, side, seed, mode, split):
    snap = str(tmp_path / "h.snap")
    assert snapgen.ahf_snapgen_write(cfg, side, seed, snap.encode()) == 0
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    print(f"[unbind-gpu] cfg{cfg} side {side} mode {mode} split {split}: {s.nhalos} haloes {s.n_ipart} members",
          flush=True)
    info, (npart, props, lists) = _run_gpu(ctx, s, mode, split=split)
    _compare(ref, npart, props, lists, f"cfg{cfg}/{side}/mode{mode}")
    assert info.n_member_out == int(ref.npart.sum())


@pytest.mark.parametrize("mode,split", [(0, 0), (1, 0), (0, 32)])
def test_unbind_replay_band(oracle, snapgen, ctx, tmp_path, mode, split):
    """a wide band sends haloes with members near the threshold to the exact
    sequential replay: the results must still be the oracle's"""
    snap = str(tmp_path / "b.snap")
    assert snapgen.ahf_snapgen_write(2, 2000, 1002, snap.encode()) == 0
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    info, (npart, props, lists) = _run_gpu(ctx, s, mode, band=1e-2, split=split)
    assert info.n_exact_replays > 0
    _compare(ref, npart, props, lists, f"band/mode{mode}")


def test_unbind_repeatable(snapgen, ctx, tmp_path):
    snap = str(tmp_path / "r.snap")
    assert snapgen.ahf_snapgen_write(2, 500, 99, snap.encode()) == 0
    s = dumps.read_snapshot(snap)
    _, r1 = _run_gpu(ctx, s, 0)
    info2 = ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=0)
    r2 = ctx.unbind_results()
    assert np.array_equal(r1[0], r2[0])
    for a, b in zip(r1[2], r2[2]):
        assert np.array_equal(a, b)


WITH_RVIR, RVIR_ONLY = 16, 32


def _construct_gpu(ctx, s, mode, centre=None, npart=None, ipart=None, split=0):
    ctx.set_unbind_split(split)
    ctx.set_particles(s.pos, s.mom)
    ctx.set_halos(s.centre if centre is None else centre, s.halo_npart if npart is None else npart,
                  s.ipart if ipart is None else ipart)
    info = ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=mode,
                      ovlim=s.ovlim, rho_vir=s.rho_vir, rho_fac=s.rho_fac)
    return info, ctx.unbind_results()


@pytest.mark.parametrize("split", [0, 32])
@pytest.mark.parametrize("cfg,side,seed,plain", [(1, 64, 1001, 0), (1, 64, 1001, 1), (0, 64, 1000, 0),
                                                 (4, 96, 1004, 0), (2, 2000, 1002, 0), (2, 300, 7, 1), (3, 48, 5, 0)])
def test_construct_matches_oracle(oracle, snapgen, ctx, tmp_path, cfg, side, seed, plain, split):
    """sort, rem_outsideRvir(0), rem_unbound, rem_outsideRvir(1) in one pass"""
    snap = str(tmp_path / "c.snap")
    assert snapgen.ahf_snapgen_write(cfg, side, seed, snap.encode()) == 0
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_construct_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    print(f"[construct-gpu] cfg{cfg} side {side} plain {plain}: {s.nhalos} haloes {s.n_ipart} members", flush=True)
    info, (npart, props, lists) = _construct_gpu(ctx, s, plain | WITH_RVIR, split=split)
    _compare(ref, npart, props, lists, f"construct cfg{cfg}/{side}/{plain}")
    assert np.array_equal(ref.R_vir, props[:, 1])
    assert np.array_equal(ref.ovdens, props[:, 3])
    small = s.halo_npart < s.minpart
    assert np.all(props[small, 5] == 0) and np.all(props[~small, 5] != 0)
    assert info.n_member_out == int(ref.npart.sum())


class _RvirParams(ctypes.Structure):
    _fields_ = [("minpart", ctypes.c_int32), ("ovlim", ctypes.c_double), ("rho_vir", ctypes.c_double),
                ("rho_fac", ctypes.c_double)]


@pytest.mark.parametrize("plain", [0, 1])
def test_rvir_only_matches_oracle(oracle, snapgen, ctx, tmp_path, plain):
    """one rem_outsideRvir call on radially sorted lists"""
    snap = str(tmp_path / "r.snap")
    assert snapgen.ahf_snapgen_write(2, 1000, 31, snap.encode()) == 0
    s = dumps.read_snapshot(snap)
    off = s.halo_offsets
    ip = s.ipart.copy()
    for h in range(s.nhalos):
        seg = ip[off[h]:off[h + 1]]
        c = np.ascontiguousarray(s.centre[h])
        oracle.oracle_sort_halo(s.pos.ctypes.data, len(seg), seg.ctypes.data, c.ctypes.data, s.minpart, 1)
    info, (npart, props, lists) = _construct_gpu(ctx, s, plain | RVIR_ONLY, ipart=ip, split=32)
    P = _RvirParams(s.minpart, s.ovlim, s.rho_vir, s.rho_fac)
    cut = 0
    for h in range(s.nhalos):
        seg = np.ascontiguousarray(ip[off[h]:off[h + 1]])
        c = np.ascontiguousarray(s.centre[h])
        o = [ctypes.c_double(0.0) for _ in range(3)]
        k = oracle.oracle_rem_outsideRvir(s.pos.ctypes.data, seg.ctypes.data, len(seg), c.ctypes.data,
                                          ctypes.byref(P), *[ctypes.byref(x) for x in o])
        assert int(npart[h]) == k and np.array_equal(lists[h], seg[:k]), f"halo {h}"
        if len(seg) >= s.minpart:
            assert (props[h, 0], props[h, 1], props[h, 3]) == (o[0].value, o[1].value, o[2].value), f"halo {h}"
            assert props[h, 2] == 0.0 and int(props[h, 5]) == 15
        else:
            assert int(props[h, 5]) == 0
        cut += len(seg) - k
    assert cut > 0
    assert info.max_iterations == 0


@pytest.mark.parametrize("seed,big", [(1, False), (2, True), (3, False), (4, True)])
def test_ties_match_oracle(oracle, ctx, tmp_path, seed, big):
    """haloes with members at exactly equal distances (lattices, duplicated
    positions, a halo across the periodic corner, one repeated position,
    with big a lattice over 8192 members): the device sorts them in
    indexx's order of equal keys, so the sort alone, the unbinding (batched,
    per halo, split path) and the construction give the oracle's haloes in
    its reference-pinned indexx mode"""
    from helpers import tie_snapshot
    snap = str(tmp_path / "t.snap")
    nh = tie_snapshot(snap, seed, big=big)
    s = dumps.read_snapshot(snap)
    print(f"[unbind-gpu] ties seed {seed}: {nh} haloes, {s.n_ipart} members", flush=True)
    ctx.set_particles(s.pos, s.mom)
    ctx.set_halos(s.centre, s.halo_npart, s.ipart)
    info = ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=ctx.UNBIND_SORT_ONLY)
    assert info.n_tie_halos == nh
    _, _, lists = ctx.unbind_results()
    off = s.halo_offsets
    for h in range(nh):
        ip = s.ipart[off[h]:off[h + 1]].copy()
        oracle.oracle_sort_halo(s.pos.ctypes.data, len(ip), ip.ctypes.data, s.centre[h].ctypes.data, s.minpart, 0)
        assert np.array_equal(ip, lists[h]), f"sort: halo {h}"
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 4, 0) == 0
    ref = dumps.read_halos(out)
    for mode, split in ((0, 0), (1, 0), (0, 32)):
        info, (npart, props, lists) = _run_gpu(ctx, s, mode, split=split)
        assert info.n_tie_halos == nh
        _compare(ref, npart, props, lists, f"ties {seed} mode {mode} split {split}")
    ctx.set_unbind_split(0)
    assert oracle.oracle_construct_dump(snap.encode(), out.encode(), 4, 0) == 0
    ref = dumps.read_halos(out)
    ctx.set_halos(s.centre, s.halo_npart, s.ipart)
    ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=ctx.UNBIND_WITH_RVIR,
               ovlim=s.ovlim, rho_vir=s.rho_vir, rho_fac=s.rho_fac)
    npart, props, lists = ctx.unbind_results()
    _compare(ref, npart, props, lists, f"ties {seed} construct")
    assert np.array_equal(ref.ovdens, props[:, 3])


@pytest.mark.parametrize("sched", [dict(split_min=4096, big_halo=1024, wave_halo=256, graph_batch=1),
                                   dict(split_min=-1, big_halo=8192, wave_halo=1024),
                                   dict(split_min=64, graph_batch=8),
                                   dict(split_min=64, split_spec=-1), dict(split_min=64, split_spec=1),
                                   dict(split_min=32, split_spec=16)])
def test_schedule_variants(oracle, snapgen, ctx, tmp_path, sched):
    """every schedule (split path threshold, workgroup tiers, graph replays
    between done checks, speculative passes of the split recurrence: none,
    one, sixteen) gives the oracle's haloes"""
    snap = str(tmp_path / "s.snap")
    assert snapgen.ahf_snapgen_write(2, 2000, 1002, snap.encode()) == 0
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_construct_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    before = ctx.schedule()
    try:
        ctx.set_schedule(**sched)
        ctx.set_particles(s.pos, s.mom)
        ctx.set_halos(s.centre, s.halo_npart, s.ipart)
        ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=ctx.UNBIND_WITH_RVIR,
                   ovlim=s.ovlim, rho_vir=s.rho_vir, rho_fac=s.rho_fac)
        npart, props, lists = ctx.unbind_results()
        _compare(ref, npart, props, lists, f"schedule {sched}")
        assert np.array_equal(ref.ovdens, props[:, 3])
    finally:
        ctx.set_schedule(**before)


FORM_SIZES = [19, 20, 21, 63, 64, 65, 127, 128, 129, 255, 511, 512, 513, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8193,
              16383, 16385]


def _form_snapshot(path, seed):
    """one isolated halo of each size around the forms' bounds: radii of a
    cuspy profile, velocities with a tail above the escape speed, one halo
    across the periodic corner, one with members on its centre, one that
    loses every member"""
    rng = np.random.default_rng(seed)
    pos, mom, lists, cen, n0 = [], [], [], [], 0
    for i, n in enumerate(FORM_SIZES):
        c = np.array([0.0, 0.9999, 0.0001]) if i == 5 else rng.uniform(0.05, 0.95, 3)
        r = 0.01 * rng.random(n) ** 1.5
        d = rng.normal(size=(n, 3))
        p = c + r[:, None] * d / np.linalg.norm(d, axis=1)[:, None]
        if i == 8:
            p[:3] = np.float32(c).astype(np.float64)
            c = np.float32(c).astype(np.float64)
        v = rng.normal(0.0, 1.0, (n, 3)) * np.sqrt(n) * 2e-3 + rng.normal(0.0, 3.0, 3)
        v[rng.random(n) < 0.15] *= 3.0
        if i == 12:
            v *= 1e4
        pos.append(p % 1.0)
        mom.append(v)
        lists.append((rng.permutation(n) + n0).astype(np.uint64))
        cen.append(c)
        n0 += n
    pos = np.concatenate(pos).astype(np.float32)
    pos[pos >= 1.0] = 0.0
    dumps.write_snapshot(path, pos, np.concatenate(mom), boxsize=1.0, pmass=1e8, L_dom=16, centres=np.array(cen),
                         halo_lists=lists, r_fac=1.0, v_fac=1.0, phi_fac=2e-7, hubble=10.0, ovlim=200.0, rho_vir=6e13,
                         gather_rad=np.full(len(lists), 0.02))


@pytest.mark.parametrize("cuts", [0, WITH_RVIR])
@pytest.mark.parametrize("plain,split,band,sched", [(0, 0, 0.0, {}), (0, -1, 0.0, {}), (1, 0, 0.0, {}), (0, -1, 3e-2, {}),
                                                    (0, -1, 0.0, dict(big_halo=600, wave_halo=70)), (0, 300, 0.0, {})])
def test_form_sizes(oracle, ctx, tmp_path, cuts, plain, split, band, sched):
    """haloes on both sides of every size at which the unbinding changes its
    form, in the forms that a few haloes take (test_many_short_haloes has the
    others), some sent to the exact replay"""
    snap, out = str(tmp_path / "f.snap"), str(tmp_path / "o.halo")
    _form_snapshot(snap, 5)
    dump = oracle.oracle_construct_dump if cuts else oracle.oracle_unbind_dump
    assert dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    lost = np.array(FORM_SIZES) - ref.npart.astype(int)
    assert lost[12] >= FORM_SIZES[12] - 1 and np.sum(lost > 0) > len(FORM_SIZES) // 2
    s = dumps.read_snapshot(snap)
    before = ctx.schedule()
    try:
        ctx.set_schedule(**sched)
        ctx.set_unbind_split(split)
        ctx.set_particles(s.pos, s.mom)
        ctx.set_halos(s.centre, s.halo_npart, s.ipart)
        info = ctx.unbind(s.minpart, s.vtune, s.r_fac, s.v_fac, s.phi_fac, s.hubble, mode=plain | cuts, band=band,
                          ovlim=s.ovlim, rho_vir=s.rho_vir, rho_fac=s.rho_fac)
        npart, props, lists = ctx.unbind_results()
    finally:
        ctx.set_schedule(**before)
        ctx.set_unbind_split(0)
    assert band == 0.0 or info.n_exact_replays > 5
    _compare(ref, npart, props, lists, f"forms {cuts} {plain} {split} {band} {sched}")
    if cuts:
        assert np.array_equal(ref.ovdens, props[:, 3])


@pytest.mark.parametrize("split", [0, -1])
def test_rvir_only_form_sizes(ctx, tmp_path, split):
    """the cut alone, batched and in the call that allocates nothing, gives the
    records and lists of one halo a launch, on both sides of every form's line"""
    from test_zz_no_alloc import Hip, _noalloc
    snap = str(tmp_path / "f.snap")
    _form_snapshot(snap, 9)
    s = dumps.read_snapshot(snap)
    off, ip = s.halo_offsets, s.ipart.copy()
    for h in range(s.nhalos):
        seg = ip[off[h]:off[h + 1]].astype(np.int64)
        d = np.abs(s.pos[seg].astype(np.float64) - s.centre[h])
        ip[off[h]:off[h + 1]] = seg[np.argsort((np.minimum(d, 1.0 - d) ** 2).sum(1))]
    s.ipart = ip
    _, (np0, pr0, li0) = _construct_gpu(ctx, s, 1 | RVIR_ONLY, ipart=ip)
    assert np.sum(np0 < s.halo_npart) > 5 and pr0[:, 0].max() > 0
    hip = Hip()
    try:
        for got in (_construct_gpu(ctx, s, RVIR_ONLY, ipart=ip, split=split)[1], _noalloc(ctx, hip, s, s.nhalos, RVIR_ONLY)):
            assert np.array_equal(np0, got[0]) and np.array_equal(pr0, got[1])
            assert all(np.array_equal(a, b) for a, b in zip(li0, got[2]))
    finally:
        hip.close()
        ctx.set_unbind_split(0)


ODD = [(n, where, value) for n in (300, 600, 2000, 4000, 5000) for where in ("first", "middle", "last")
       for value in ("nan", "inf", "both")]


def _odd_snapshot(path, seed):
    """isolated haloes whose first, a middle or last wavefront of members holds
    a NaN velocity, one infinite velocity, or a NaN and behind it infinities of
    both signs; none among the members that the first seed is chosen from"""
    rng = np.random.default_rng(seed)
    pos, mom, lists, cen, n0 = [], [], [], [], 0
    for n, where, value in ODD:
        c = np.float32(rng.uniform(0.05, 0.95, 3)).astype(np.float64)
        d = rng.normal(size=(n, 3))
        p = (c + (0.01 * rng.random(n) ** 1.5)[:, None] * d / np.linalg.norm(d, axis=1)[:, None]).astype(np.float32)
        o = np.argsort(((p.astype(np.float64) - c) ** 2).sum(1))
        v = rng.normal(0.0, 1.0, (n, 3)) * np.sqrt(n) * 2e-3 + rng.normal(0.0, 3.0, 3)
        v[rng.random(n) < 0.15] *= 3.0
        at = {"first": min(100, n // 3), "middle": n // 2, "last": n - 15}[where]
        if value != "inf":
            v[o[at], 1] = np.nan
        if value != "nan":
            v[o[at + 3], 0] = np.inf
        if value == "both":
            v[o[at + 5], 0] = -np.inf
        pos.append(p)
        mom.append(v)
        lists.append((rng.permutation(n) + n0).astype(np.uint64))
        cen.append(c)
        n0 += n
    dumps.write_snapshot(path, np.concatenate(pos), np.concatenate(mom), boxsize=1.0, pmass=1e8, L_dom=16,
                         centres=np.array(cen), halo_lists=lists, r_fac=1.0, v_fac=1.0, phi_fac=2e-7, hubble=10.0,
                         ovlim=60.0, rho_vir=6e13, gather_rad=np.full(len(lists), 0.02))


@pytest.mark.parametrize("cuts,plain", [(0, 0), (WITH_RVIR, 0), (0, 1), (WITH_RVIR, 1)])
def test_odd_velocities(oracle, ctx, tmp_path, cuts, plain):
    """a NaN velocity stays bound and an infinite one does not, as in AHF, and
    the rounds of the unbinding end, in every form up to the chunked one"""
    snap, out = str(tmp_path / "n.snap"), str(tmp_path / "o.halo")
    _odd_snapshot(snap, 3)
    dump = oracle.oracle_construct_dump if cuts else oracle.oracle_unbind_dump
    assert dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    nan = np.array([np.isnan(s.mom[m.astype(np.int64)]).any() for m in ref.ipart])
    assert np.array_equal(nan, [value != "inf" for _, _, value in ODD]) and np.all(ref.npart < s.halo_npart)
    print(f"[odd] cuts {cuts} plain {plain}: {s.nhalos} haloes", flush=True)
    _, (npart, props, lists) = _construct_gpu(ctx, s, plain | cuts, split=-1) if cuts else _run_gpu(ctx, s, plain, split=-1)
    _compare(ref, npart, props, lists, f"odd velocities {cuts} {plain}")


FAST = [60, 130, 400, 700, 1800, 3000, 4000, 6000]


def _fast_snapshot(path, seed):
    """isolated haloes with one member of 10^25 times the others' speed, which
    leaves in the first iteration"""
    rng = np.random.default_rng(seed)
    pos, mom, lists, cen, n0 = [], [], [], [], 0
    for n in FAST:
        c = np.float32(rng.uniform(0.05, 0.95, 3)).astype(np.float64)
        d = rng.normal(size=(n, 3))
        p = (c + (0.01 * rng.random(n) ** 1.5)[:, None] * d / np.linalg.norm(d, axis=1)[:, None]).astype(np.float32)
        o = np.argsort(((p.astype(np.float64) - c) ** 2).sum(1))
        v = rng.normal(0.0, 1.0, (n, 3)) * np.sqrt(n) * 2e-3
        v[o[20 + np.flatnonzero(rng.random(n - 20) < 0.15)]] *= 3.0
        v[o[n // 2]] = [1e25, 0.0, -1e25]
        pos.append(p)
        mom.append(v)
        lists.append((rng.permutation(n) + n0).astype(np.uint64))
        cen.append(c)
        n0 += n
    dumps.write_snapshot(path, np.concatenate(pos), np.concatenate(mom), boxsize=1.0, pmass=1e8, L_dom=16,
                         centres=np.array(cen), halo_lists=lists, r_fac=1.0, v_fac=1.0, phi_fac=2e-7, hubble=10.0,
                         ovlim=60.0, rho_vir=6e13, gather_rad=np.full(len(lists), 0.02))


@pytest.mark.parametrize("plain", [0, 1])
def test_fast_member_widens_one_iteration(oracle, ctx, tmp_path, plain):
    """a member too fast for the rounding bound makes the iteration that removes
    it uncertain, in every form, and none of the later ones"""
    snap, out = str(tmp_path / "v.snap"), str(tmp_path / "o.halo")
    _fast_snapshot(snap, 4)
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    info, (npart, props, lists) = _run_gpu(ctx, dumps.read_snapshot(snap), plain, split=-1)
    _compare(ref, npart, props, lists, f"fast member {plain}")
    assert props[:, 4].min() >= 2 and info.n_exact_replays == len(FAST)


def _edge_halo(rng, n, phi_fac, vtune2, minpart):
    """positions (offsets) and velocities of a halo in radial order, one of
    whose members sits within about one unit of rounding of the bound test as
    rem_unbound's sequential sums evaluate it: vx and vy from candidates just
    below the limit, vz (no other member has one) makes up the rest"""
    r = np.sort(rng.uniform(1e-4, 1e-2, n))
    d = rng.normal(size=(n, 3))
    off = np.round(r[:, None] * d / np.linalg.norm(d, axis=1)[:, None] * 2.0 ** 24) / 2.0 ** 24
    dist = np.sqrt(off[:, 0] * off[:, 0] + off[:, 1] * off[:, 1] + off[:, 2] * off[:, 2])
    o = np.argsort(dist)
    off, dist = off[o], dist[o]
    phi, acc, ip, dp = [], 0.0, 0.0, 0.0
    for j, x in enumerate(dist.tolist()):
        cur = float(j + 1) / (x * x)
        acc += (cur + ip) / 2. * (x - dp)
        phi.append(acc)
        ip, dp = cur, x
    phi0 = acc + float(n) / dist[-1]
    lim = vtune2 * (2 * np.abs(np.array(phi) - phi0) * phi_fac)
    v = np.zeros((n, 3), np.float32)
    v[:, :2] = rng.normal(0.0, 0.3, (n, 2)) * np.sqrt(lim)[:, None] + rng.normal(0.0, 0.2, 2) * np.sqrt(lim[-1])
    v2 = v[:minpart // 2, 0] * v[:minpart // 2, 0] + v[:minpart // 2, 1] * v[:minpart // 2, 1]
    js = int(np.argsort(v2)[minpart // 2 // 2 - 1])
    V, M = [float(v[js, 0]), float(v[js, 1])], 1.0
    for j in range(n):
        if j == n // 2:
            ang, k = rng.uniform(0, 2 * np.pi, 4000), np.sqrt(lim[j])
            cx, cy = np.float32(V[0] / M + k * np.cos(ang)), np.float32(V[1] / M + k * np.sin(ang))
            dx, dy = cx.astype(np.float64) - V[0] / M, cy.astype(np.float64) - V[1] / M
            rest = lim[j] - (dx * dx + dy * dy)
            ok = (rest > 0) & (rest < 3e-8 * lim[j])
            cx, cy, dx, dy, cz = cx[ok], cy[ok], dx[ok], dy[ok], np.float32(np.sqrt(rest[ok]))
            gap = np.abs((dx * dx + dy * dy + cz.astype(np.float64) ** 2) - lim[j])
            b = int(np.argmin(gap))
            v[j] = cx[b], cy[b], cz[b]
        x, y, z = (float(c) for c in v[j])
        a, b, c = x - V[0] / M, y - V[1] / M, z
        if not (a * a + b * b + c * c > lim[j]):
            M += 1.0
            V[0] += x
            V[1] += y
    return off, v


@pytest.mark.parametrize("split", [0, -1, 300])
def test_rounding_edge(oracle, ctx, tmp_path, split):
    """members whose bound test AHF's own rounding decides: the parallel
    sums' answer differs for some, the library's must not, in any form"""
    rng = np.random.default_rng(11)
    phi_fac, vtune, minpart = 1e-7, 1.5, 20
    pos, mom, lists, cen, n0 = [], [], [], [], 0
    for i, n in enumerate([60, 400, 1500, 3500, 7000, 12000] * 3):
        off, v = _edge_halo(rng, n, phi_fac, vtune * vtune, minpart)
        c = np.array([0.25 + 0.0625 * (i % 6), 0.5, 0.25 + 0.25 * (i // 6)])
        pos.append(c + off)
        mom.append(v)
        lists.append((rng.permutation(n) + n0).astype(np.uint64))
        cen.append(c)
        n0 += n
    snap, out = str(tmp_path / "e.snap"), str(tmp_path / "o.halo")
    dumps.write_snapshot(snap, np.concatenate(pos), np.concatenate(mom), boxsize=1.0, pmass=1e8, L_dom=16,
                         centres=np.array(cen), halo_lists=lists, r_fac=1.0, v_fac=1.0, phi_fac=phi_fac, hubble=0.0,
                         vtune=vtune, minpart=minpart, gather_rad=np.full(len(lists), 0.02))
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    info, (npart, props, lists) = _run_gpu(ctx, dumps.read_snapshot(snap), 0, split=split)
    assert info.n_exact_replays >= 12
    _compare(ref, npart, props, lists, f"edge split {split}")


@pytest.mark.parametrize("cuts", [0, WITH_RVIR])
def test_many_short_haloes(oracle, ctx, tmp_path, cuts):
    """more short haloes than are resident at once: the one-wavefront forms in
    launches of their own, from the host's order and from the cut's lists"""
    from helpers import short_haloes_snapshot
    snap, out = str(tmp_path / "s.snap"), str(tmp_path / "o.halo")
    left = short_haloes_snapshot(snap, 6, 5000)
    assert all(np.count_nonzero(x) > 20 for x in (left < 128, (left > 128) & (left < 512), left > 512))
    dump = oracle.oracle_construct_dump if cuts else oracle.oracle_unbind_dump
    assert dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    _, (npart, props, lists) = _construct_gpu(ctx, s, cuts) if cuts else _run_gpu(ctx, s, 0)
    _compare(ref, npart, props, lists, f"short haloes {cuts}")


def test_more_haloes_than_a_workgroup_keeps(oracle, ctx, tmp_path):
    """more than 64 short haloes for each workgroup that lists them by form,
    with two larger ones among them"""
    rng = np.random.default_rng(12)
    nh = 140000
    sizes = np.where(rng.random(nh) < 0.9, 20, 24)
    sizes[[5, 90001]] = 700, 3000
    n, off = int(sizes.sum()), np.concatenate([[0], np.cumsum(sizes)])
    cen = np.float32(rng.uniform(0.05, 0.95, (nh, 3))).astype(np.float64)
    d = rng.standard_normal((n, 3))
    r = 0.002 * rng.random(n) ** 1.5
    pos = (np.repeat(cen, sizes, axis=0) + r[:, None] * d / np.linalg.norm(d, axis=1)[:, None]).astype(np.float32)
    mom = rng.standard_normal((n, 3)) * 0.02
    mom[rng.random(n) < 0.1] *= 4.0
    snap, out = str(tmp_path / "k.snap"), str(tmp_path / "o.halo")
    dumps.write_snapshot(snap, pos, mom, boxsize=1.0, pmass=1e8, L_dom=16, centres=cen,
                         halo_lists=[np.arange(off[h], off[h + 1], dtype=np.uint64) for h in range(nh)], r_fac=1.0,
                         v_fac=1.0, phi_fac=2e-7, hubble=10.0, ovlim=200.0, rho_vir=3e14, gather_rad=np.full(nh, 0.004))
    assert oracle.oracle_construct_dump(snap.encode(), out.encode(), 8, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    assert np.any(ref.npart == s.halo_npart) and np.any(ref.npart < s.halo_npart)
    _, (npart, props, lists) = _construct_gpu(ctx, s, WITH_RVIR)
    _compare(ref, npart, props, lists, "140,000 haloes")


def test_schedule_file(tmp_path, monkeypatch):
    """a context applies the schedule file named by AHF_SCHEDULE"""
    import json

    import ahf_amd
    path = tmp_path / "sched.json"
    path.write_text(json.dumps({"split_min": 12345, "kmax_big": 500, "march_zn": 8, "graph_batch": 3,
                                "tuning": {"fields": {"split_min": {"chosen": 1}}}}))
    monkeypatch.setenv("AHF_SCHEDULE", str(path))
    c = ahf_amd.Context(0)
    try:
        sc = c.schedule()
        assert sc["split_min"] == 12345 and sc["kmax_big"] == 500 and sc["march_zn"] == 8 and sc["graph_batch"] == 3
    finally:
        c.close()


def test_timing_off(oracle, snapgen, ctx, tmp_path):
    """with the stage timers off the haloes are the same and the timings
    read 0; on again, they are timed"""
    snap = str(tmp_path / "t.snap")
    assert snapgen.ahf_snapgen_write(1, 64, 1001, snap.encode()) == 0
    out = str(tmp_path / "o.halo")
    assert oracle.oracle_unbind_dump(snap.encode(), out.encode(), 4, 0) == 0
    ref = dumps.read_halos(out)
    s = dumps.read_snapshot(snap)
    try:
        ctx.set_timing(False)
        _, (npart, props, lists) = _run_gpu(ctx, s, 0)
        _compare(ref, npart, props, lists, "timing off")
        assert ctx.last_timing()["unbind_ms"] == 0.0
    finally:
        ctx.set_timing(True)
    _, (npart, props, lists) = _run_gpu(ctx, s, 0)
    _compare(ref, npart, props, lists, "timing on")
    assert ctx.last_timing()["unbind_ms"] > 0.0
