"""Kernel variants and dispatch rules at the sizes where they can go wrong: tile
edges, remainders, the smallest and largest of a range."""
import time

import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

EPS2, DT = 40.0, 0.0035


@pytest.mark.parametrize("n", [1, 33, 1023, 1024, 1025, 3073])
@pytest.mark.parametrize("leaf", [1, 31, 64])
def test_tree_build_at_tile_edges(nb, ora, n, leaf):
    """The build marks bodies in tiles of 1024 with a window of leaf + 1 bodies
    across their edges: topology bit-exact, with runs of equal codes in it."""
    rng = np.random.default_rng(1000 * n + leaf)
    pos = rng.normal(size=(n, 3)) * rng.choice([1.0, 0.01], size=(n, 1))
    pos[n // 2:] = pos[: n - n // 2] if n % 2 else pos[n // 2:]  # coincident bodies
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    with nb.Simulation(n, EPS2, DT, solver=nb.SOLVER_BH, leaf_size=leaf) as sim:
        sim.upload(pos, np.zeros_like(pos), m)
        f = sim.forces()
        codes, perm = sim.debug_morton()
        nodes, _ = sim.debug_tree()
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :3], p4[:, 3] = pos, m
    mn, mx = ora.bbox(p4)
    ccodes = ora.morton(p4, mn, mx, cubic=True)
    cperm, srt = ora.sort_codes(ccodes)
    tree = ora.build_tree(srt, leaf)
    np.testing.assert_array_equal(codes, ccodes)
    np.testing.assert_array_equal(perm, cperm)
    for mine, theirs in (("first_child", "first_child"), ("next", "next"), ("body_start", "start"),
                         ("body_count", "count"), ("level", "level")):
        np.testing.assert_array_equal(nodes[mine], tree[theirs])
    com = ora.tree_com(tree, p4[cperm])
    fc, _ = ora.bh_forces_group(p4[cperm], cperm, mn, mx, tree, com, EPS2, group=nb.BH_WAVE_BODIES,
                                codes_sorted=srt)
    # FP32 sums of at most n terms in another order: n / 2 rounding steps at worst
    scale = np.abs(fc[:, :3]).max() + 1e-30
    assert np.abs(f[:, :3] - fc[:, :3]).max() <= max(n, 64) * 2.0 ** -24 * scale


@pytest.mark.parametrize("n, leaf, eps2", [(3, 8, EPS2), (300, 64, EPS2), (5001, 1, 0.0), (20011, 64, EPS2),
                                           (32767, 8, EPS2), (32768, 16, 0.0), (262143, 8, EPS2),
                                           (262144, 8, EPS2)])
def test_workgroup_walk_equals_pair_walk(nb, n, leaf, eps2):
    """Eight, then four waves per range, against the walk that one wave does for a
    pair of ranges: the same interactions, summed in another order. A level-10
    cell with more bodies than a wave's list holds is among them."""
    pos, _, m = nb.ic_plummer(77 + n, n, 50.0, 1e4)
    pos[: min(n // 2, 700)] = pos[0]
    f = []
    for flags in (0, nb.F_BH_PAIRS):
        with nb.Simulation(n, eps2, DT, solver=nb.SOLVER_BH, leaf_size=leaf, flags=flags) as sim:
            sim.upload(pos, np.zeros_like(pos), m)
            f.append(sim.forces())
            again = sim.forces()
        np.testing.assert_array_equal(f[-1], again)
    # FP32 partial sums of at most 192 terms, folded with compensation
    assert np.percentile(rel_err(f[0], f[1]), 99) < 1e-5
    scale = np.linalg.norm(f[1][:, :3], axis=1).max()
    assert np.abs(f[0] - f[1]).max() <= 192 * 2.0 ** -24 * scale


@pytest.mark.parametrize("n", [1, 63, 2047, 2049, 24576, 24577, 131071, 131073, 264193])
def test_radix_sort_at_tile_and_group_edges(nb, ora, n):
    """Tiles of 2048 keys, in groups of 64 above 24,576: codes and the stable permutation."""
    rng = np.random.default_rng(n)
    pos = np.round(rng.normal(size=(n, 3)) * 8) if n % 4 == 1 else rng.normal(size=(n, 3))
    m = np.ones(n, np.float32)
    with nb.Simulation(n, EPS2, DT, solver=nb.SOLVER_BH) as sim:
        sim.upload(pos, np.zeros_like(pos), m)
        sim.forces()
        codes, perm = sim.debug_morton()
    p4 = np.zeros((n, 4), np.float32)
    p4[:, :3], p4[:, 3] = pos, m
    mn, mx = ora.bbox(p4)
    ccodes = ora.morton(p4, mn, mx, cubic=True)
    np.testing.assert_array_equal(codes, ccodes)
    np.testing.assert_array_equal(perm, np.argsort(ccodes, kind="stable"))


@pytest.mark.parametrize("n, bpl, js", [(1, 0, 0), (511, 0, 0), (1025, 0, 0), (2049, 4, 4), (4097, 0, 0),
                                        (6000, 2, 8), (8193, 1, 1), (16385, 0, 0), (37001, 0, 0)])
def test_direct_sum_in_parts(nb, ora, n, bpl, js):
    """Workgroups that each sum a part of the sources (1 to 8 parts at these sizes):
    forces against FP64, and steps and force passes use the same sum."""
    pos, vel, m = nb.ic_plummer(5 + n, n, 50.0, 1e4)
    tgt = np.random.default_rng(n).choice(n, min(n, 500), replace=False)
    ref = ora.direct_f64(pos.astype(np.float32).astype(np.float64), m.astype(np.float64), EPS2, targets=tgt)
    with nb.Simulation(n, EPS2, DT, bodies_per_lane=bpl, j_split=js) as sim:
        sim.upload(pos, vel, m)
        f = sim.forces_f64()
        sim.step(1)
        _, _, acc = sim.download_f64()
    np.testing.assert_array_equal(acc, f)  # the lagged step's forces are those at its start
    scale = np.linalg.norm(ref, axis=1).max() + 1e-30
    # 256-source FP32 sums, folded with compensation: 256 roundings of the largest force at worst
    assert np.abs(f[tgt] - ref).max() <= 256 * 2.0 ** -24 * scale


@pytest.mark.parametrize("n", [1, 255, 257, 29127, 29128, 43680, 43681, 65521, 131041])
@pytest.mark.parametrize("layout", ["f64", "vec4"])
def test_host_copies_at_stage_edges(nb, n, layout):
    """State in and out through the pinned buffer (whole calls up to 2 MB, halves
    above; uploads directly above), in the caller's order, also after a reorder."""
    rng = np.random.default_rng(n)
    pos, vel, acc = (rng.normal(size=(n, 3)) for _ in range(3))
    m = rng.uniform(1, 2, n).astype(np.float32)
    if layout == "vec4":
        pos, vel, acc = (a.astype(np.float32).astype(np.float64) for a in (pos, vel, acc))
    give = (lambda a: a) if layout == "f64" else nb.to_vec4
    speed = np.sqrt(vel[:, 0] ** 2 + vel[:, 1] ** 2 + vel[:, 2] ** 2)
    with nb.Simulation(n, EPS2, DT) as sim:
        for again in range(2):  # the second upload reuses the buffer that a kernel still reads
            sim.upload(give(np.roll(pos, again, 0)), give(vel), m, give(acc) if again else None)
        pos = np.roll(pos, 1, 0)
        for reordered in (False, True):
            if reordered:
                sim.reorder()
            for got, want in zip(sim.download_f64(), (pos, vel, acc)):
                np.testing.assert_array_equal(got, want)
            for got, want in zip(sim.download(), (pos, vel, acc)):
                np.testing.assert_array_equal(got[:, :3], want.astype(np.float32))
                assert not got[:, 3].any()
            view = sim.render_view()
            np.testing.assert_array_equal(view[:, :3], pos.astype(np.float32))
            np.testing.assert_allclose(view[:, 3], speed, rtol=2.0 ** -22)
        np.testing.assert_array_equal(sim.forces(), sim.forces_f64().astype(np.float32) @ np.eye(3, 4, dtype=np.float32))


@pytest.mark.parametrize("n", [1, 1023, 1025, 2049, 4095, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("integrator", [0, 1])
def test_one_launch_steps(nb, n, integrator):
    """Steps of small systems alternate two views of the bodies: any split of the
    steps into calls, graphs or not, timed or not, gives the same bits."""
    pos, vel, m = nb.ic_plummer(9 + n, n, 50.0, 1e4)
    out = []
    for flags, calls in ((0, [21]), (0, [1, 9, 2, 8, 1]), (nb.F_NO_GRAPH, [21]), (0, [3, -1, 18])):
        with nb.Simulation(n, EPS2 if n % 2 else 0.0, DT, integrator=integrator, flags=flags) as sim:
            sim.upload(pos, vel, m)
            sim.step(1)  # an odd step first
            sim.upload(pos, vel, m)
            for k in calls:
                if k < 0:
                    sim.set_timing(True)
                    f = sim.forces_f64()
                else:
                    sim.step(k)
            sim.set_timing(False)
            out.append(np.concatenate(sim.download_f64() + (sim.forces_f64(),)))
    for o in out[1:]:
        np.testing.assert_array_equal(o, out[0])


@pytest.mark.parametrize("m, radius, eps2, G", [(1.0, 100.0, 40.0, 1.0), (2.4, 50.0, 0.5, 1.0), (1e-9, 1e-3, 1e-9, 1.0),
                                                (2e30, 1e13, 1e20, 6.674e-11), (3e38, 1e15, 1e26, 1e-11),
                                                (7.0, 1e14, 1e20, 1.0), (5.0, 10.0, 1e-19, 1.0)])
@pytest.mark.parametrize("n", [1, 257, 9001])
def test_equal_masses_over_the_range_of_scales(nb, ora, m, radius, eps2, G, n):
    """Equal masses leave the inner loop and the view is scaled by a power of two:
    forces against FP64 at masses and lengths where r^-3 alone would leave FP32's
    range, for a single system and a cluster, before and after a step and a reorder;
    one different mass takes the general form."""
    pos, vel, _ = nb.ic_ball(3 + n, n, radius, 1.0)
    tgt = np.arange(0, n, max(1, n // 200))
    for mass in (np.full(n, m, np.float32), np.concatenate([np.full(n - 1, m), [m / 2]]).astype(np.float32)):
        ref = G * ora.direct_f64(pos.astype(np.float32).astype(np.float64), mass.astype(np.float64), np.float32(eps2),
                                 targets=tgt)
        scale = np.linalg.norm(ref, axis=1).max() + 1e-300
        with nb.Simulation(n, eps2, 0.0, G=G) as sim:  # dt = 0: a step moves nothing
            sim.upload(pos, np.zeros_like(pos), mass)
            got = [sim.forces_f64(), sim.direct_f64(tgt)]
            sim.step(1)
            got.append(sim.download_f64()[2])
            sim.reorder()
            got += [sim.forces_f64(), sim.direct_f64(tgt)]
        with nb.Batch(n + 255, 1) as b:
            c = b.add(pos, np.zeros_like(pos), mass, eps2, 0.0, G)
            got.append(b.forces(c))
            b.step(2)
            got.append(b.download(c)[2])
        for f in got:
            f = f if len(f) == len(tgt) else f[tgt]
            # 256-source FP32 sums, folded: 256 roundings of the largest force at worst
            assert np.abs(f - ref).max() <= 256 * 2.0 ** -24 * scale


@pytest.mark.parametrize("n", [89000, 250001, 700001])
def test_large_host_copies(nb, n):
    """Downloads above 4 MB, where several threads copy, and above 32 MB, through the
    larger stage (which replaces the smaller one on the way)."""
    rng = np.random.default_rng(n)
    pos, vel, acc = (rng.normal(size=(n, 3)) for _ in range(3))
    with nb.Simulation(n, EPS2, DT, solver=nb.SOLVER_BH) as sim:
        sim.upload(pos, vel, np.ones(n, np.float32), acc)
        np.testing.assert_array_equal(sim.render_view()[:, :3], pos.astype(np.float32))
        for _ in range(2):
            for got, want in zip(sim.download_f64(), (pos, vel, acc)):
                np.testing.assert_array_equal(got, want)
            for got, want in zip(sim.download(), (pos, vel, acc)):
                np.testing.assert_array_equal(got[:, :3], want.astype(np.float32))
        sim.energy() if n < 100000 else sim.sync()


@pytest.mark.parametrize("sizes", [(1, 4096, 4097), (8192, 300, 8193), (16384, 16385), (20481, 33000)])
def test_batch_clusters_in_parts(nb, ora, sizes):
    """Large clusters are summed in 1 to 4 parts: forces against FP64, the same bits
    alone and together, and steps use the forces of the force pass."""
    sys_ = [nb.ic_plummer(50 + n, n, 50.0, 1e4) for n in sizes]
    with nb.Batch(sum(n + 256 for n in sizes), len(sizes)) as b:
        ids = [b.add(p, v, m, EPS2, DT) for p, v, m in sys_]
        f = [b.forces(c) for c in ids]
        b.step(1)
        acc = [b.download(c)[2] for c in ids]
    for (pos, vel, m), n, mine, a in zip(sys_, sizes, f, acc):
        np.testing.assert_array_equal(mine, a)
        with nb.Batch(n + 256, 1) as b:
            c = b.add(pos, vel, m, EPS2, DT)
            np.testing.assert_array_equal(b.forces(c), mine)
        tgt = np.arange(0, n, max(1, n // 300))
        ref = ora.direct_f64(pos.astype(np.float32).astype(np.float64), m.astype(np.float64), EPS2, targets=tgt)
        # 256-source FP32 sums, folded: 256 roundings of the largest force at worst
        assert np.abs(mine[tgt] - ref).max() <= 256 * 2.0 ** -24 * (np.linalg.norm(ref, axis=1).max() + 1e-30)


@pytest.mark.parametrize("solver, n, calls", [("direct", 300, (7, 8, 9, 17)), ("direct", 9000, (8, 3)),
                                              ("bh", 700, (31, 32)), ("bh", 5001, (1, 35, 2))])
def test_calls_of_any_length_take_the_same_steps(nb, solver, n, calls):
    """Launched steps, whole graphs and what is left of them, against launched steps only."""
    pos, vel, m = nb.ic_plummer(n, n, 50.0, 1e4)
    out = []
    for flags in (0, nb.F_NO_GRAPH):
        with nb.Simulation(n, EPS2, DT, solver=nb.SOLVER_BH if solver == "bh" else nb.SOLVER_DIRECT,
                           flags=flags) as sim:
            sim.upload(pos, vel, m)
            for k in calls:
                sim.step(k)
            out.append(sim.download_f64())
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("clusters", [1023, 1025, 1040, 3100])
def test_batch_items_beyond_the_first(nb, clusters):
    """More work items than workgroups: every cluster is stepped once per step, and all
    alike ones come out as a cluster does alone."""
    pos, vel, m = nb.ic_plummer(clusters, 64, 50.0, 1e4)
    with nb.Batch(256, 1) as one, nb.Batch(256 * clusters, clusters) as many:
        alone = one.add(pos, vel, m, EPS2, DT)
        ids = [many.add(pos, vel, m, EPS2, DT) for _ in range(clusters)]
        for b in (one, many):
            b.step(3)
        ref = one.download(alone)
        for k in range(0, clusters, 31):
            for a, b in zip(ref, many.download(ids[k])):
                np.testing.assert_array_equal(a, b)
        for a, b in zip(ref, many.download(ids[-1])):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n, bpl, js, eps2", [(8193, 0, 0, 0.0), (12289, 2, 4, 0.0), (16385, 4, 1, EPS2),
                                              (20001, 1, 16, EPS2), (24833, 4, 4, 0.0), (33001, 2, 8, EPS2)])
def test_direct_sum_shares_of_unequal_masses(nb, ora, n, bpl, js, eps2):
    """Shares that end inside a block of targets, with masses of their own and without
    softening: forces against FP64 at the first, last and random targets."""
    rng = np.random.default_rng(n)
    pos = rng.uniform(-100, 100, (n, 3))
    m = rng.uniform(0.5, 2, n).astype(np.float32)
    tgt = np.unique(np.concatenate([[0, 63, 64, n - 1], rng.choice(n, 300, replace=False)]))
    ref = ora.direct_f64(pos.astype(np.float32).astype(np.float64), m.astype(np.float64), eps2, targets=tgt)
    with nb.Simulation(n, eps2, DT, bodies_per_lane=bpl, j_split=js) as sim:
        sim.upload(pos, np.zeros_like(pos), m)
        f = sim.forces_f64()
    scale = np.linalg.norm(ref, axis=1).max()
    # 256-source FP32 sums, folded with compensation: 256 roundings of the largest force at worst
    assert np.abs(f[tgt] - ref).max() <= 256 * 2.0 ** -24 * scale


def test_batch_parts_with_and_without_room(nb):
    """More clusters in parts than there is room for partial sums: those without it, and a
    batch whose removed clusters make room, give the same forces and steps."""
    n, clusters = 16000, 90  # four parts each
    pos, vel, m = nb.ic_plummer(9, n, 50.0, 1e4)
    with nb.Batch(clusters * 16128, clusters) as b:
        ids = [b.add(pos, vel, m, EPS2, DT) for _ in range(clusters)]
        f = [b.forces(c) for c in ids]
        b.step(2)
        for c in ids[: clusters // 2]:
            b.remove(c)
        b.step(1)
        end = [b.download(c) for c in ids[clusters // 2:]]
    with nb.Batch(16128, 1) as b:
        c = b.add(pos, vel, m, EPS2, DT)
        ref = b.forces(c)
        b.step(3)
        last = b.download(c)
    for mine in f:
        np.testing.assert_array_equal(mine, ref)
    for mine in end:
        for x, y in zip(mine, last):
            np.testing.assert_array_equal(x, y)


def test_download_waits_without_spinning(nb):
    """A large download behind queued steps occupies the calling thread at most: the
    threads that will copy sleep until there is something to copy."""
    n = 1 << 18
    pos, vel, m = nb.ic_ball(1, n, 100.0, 1.0)
    with nb.Simulation(n, EPS2, DT) as sim:
        sim.upload(pos, vel, m)
        sim.step(1)
        sim.download_f64()
        sim.step(30)  # some 400 ms
        wall, cpu = time.monotonic(), time.process_time()
        sim.download_f64()
        wall, cpu = time.monotonic() - wall, time.process_time() - cpu
    assert cpu < 2.0 * wall


@pytest.mark.parametrize("n", [1, 1024, 4095, 4097])
def test_timed_small_steps_are_the_steps_that_run(nb, n):
    """One launch per step has one time, with and without timing the same result, and its
    forces are those of the force pass."""
    pos, vel, m = nb.ic_plummer(n + 1, n, 50.0, 1e4)
    with nb.Simulation(n, EPS2, DT) as sim:
        sim.upload(pos, vel, m)
        f = sim.forces_f64()
        sim.set_timing(True)
        sim.step(5)
        t = sim.timing()
        sim.set_timing(False)
        timed = sim.download_f64()
        sim.upload(pos, vel, m)
        sim.step(1)
        p, v, a = sim.download_f64()
        sim.step(4)
        plain = sim.download_f64()
    assert t["step_calls"] == t["force_calls"] == 5 and 0 < t["force_ms"] == t["step_ms"]
    for x, y in zip(timed, plain):
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(a, f)
    # a first lagged step, from no acceleration; three FP64 roundings of each term
    h = 0.5 * float(np.float32(DT))
    np.testing.assert_allclose(v, vel + f * h, rtol=0, atol=4 * 2.0 ** -53 * (np.abs(vel).max() + np.abs(f).max()))
    np.testing.assert_allclose(p, pos + vel * 2 * h, rtol=0, atol=4 * 2.0 ** -53 * (np.abs(pos).max() + np.abs(vel).max()))


@pytest.mark.parametrize("n", [1, 3, 1000, 4097])
def test_padding_of_both_views_adds_nothing(nb, n):
    """Without softening, a body closer to the origin than FP32 has inverse squares for:
    the padding of either view (steps alternate them) must not be there."""
    pos, _, m = nb.ic_ball(5, n, 100.0, 1.0)
    pos[0] = (1e-20, 0, 0)
    zero = np.zeros_like(pos)
    with nb.Simulation(n, 0.0, 0.0) as sim:  # dt = 0: the forces stay
        sim.upload(pos, zero, m)
        f = sim.forces_f64()
        assert np.isfinite(f).all()
        for _ in range(3):
            sim.step(1)
            np.testing.assert_array_equal(sim.download_f64()[2], f)


@pytest.mark.parametrize("n", [3, 40, 5001])
@pytest.mark.parametrize("pairs", [False, True])
def test_padding_of_walk_lists_adds_nothing(nb, ora, n, pairs):
    """As above for the lists of both Barnes-Hut walks; leaves of single bodies, theta so
    small that every body is listed."""
    pos, vel, m = nb.ic_ball(6, n, 100.0, 1.0)
    pos[0] = (1e-20, 0, 0)
    with nb.Simulation(n, 0.0, DT, solver=nb.SOLVER_BH, theta=1e-6, leaf_size=1,
                       flags=nb.F_BH_PAIRS if pairs else 0) as sim:
        sim.upload(pos, vel, m)
        f = sim.forces_f64()
    ref = ora.direct_f64(pos.astype(np.float32).astype(np.float64), m.astype(np.float64), 0.0)
    # FP32 sums of at most 384 terms, folded: as many roundings of the largest force at worst
    assert np.abs(f - ref).max() <= 384 * 2.0 ** -24 * np.linalg.norm(ref, axis=1).max()


@pytest.mark.parametrize("n", [31 * 131072, 31 * 131072 + 1, 64 * 131072 + 1, 9000001])
def test_radix_sort_of_many_groups(nb, n):
    """Below and above the line at which the groups' counts are added up in a launch of
    their own: the permutation is the stable sort of the codes."""
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3)) ** 3
    with nb.Simulation(n, EPS2, DT, solver=nb.SOLVER_BH, theta=2.0) as sim:
        sim.upload(pos, np.zeros_like(pos), np.ones(n, np.float32))
        sim.step(1)
        codes, perm = sim.debug_morton()
    np.testing.assert_array_equal(perm, np.argsort(codes, kind="stable"))


def test_build_time_stays_linear(nb):
    """A body of 2^26 costs what one of 2^23 does: no pass of the build adds up a table
    that grows with the system in each of its blocks."""
    cost = []
    for n in (1 << 23, 1 << 26):
        pos = np.random.default_rng(1).random((n, 3))
        with nb.Simulation(n, 1e-4, 0.0, solver=nb.SOLVER_BH, theta=1.0) as sim:
            sim.upload(pos, np.zeros_like(pos), np.ones(n, np.float32))
            sim.step(1)
            sim.set_timing(True)
            sim.step(3)
            cost.append(sim.timing()["build_ms"] / n)
    assert cost[1] < 1.25 * cost[0]


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 4097, 16384, 16385, 20011])
def test_energy_of_unequal_masses(nb, ora, n):
    """Rows of 64 targets folded two by two against chunks of 64 sources, of 256 above
    16,384 bodies: every pair once, at the edges of rows and chunks."""
    rng = np.random.default_rng(n)
    pos, vel = rng.normal(0, 50, (n, 3)), rng.normal(0, 3, (n, 3))
    m = rng.uniform(0.1, 10, n).astype(np.float32)
    with nb.Simulation(n, EPS2, DT, G=1.5) as sim:
        sim.upload(pos, vel, m)
        ek, ep, p = sim.energy()
    rk, rp, q = ora.energy_f64(pos, vel, m.astype(np.float64), EPS2, 1.5)
    # FP64 sums of one sign: at most 2 n roundings in a row on either side
    tol = (4 * n + 16) * 2.0 ** -53
    assert abs(ek - rk) <= tol * rk and abs(ep - rp) <= tol * abs(rp)
    assert np.abs(p - q).max() <= tol * (m.astype(np.float64)[:, None] * np.abs(vel)).sum(0).max()


@pytest.mark.parametrize("n", [300, 3000, 8000])
def test_small_sizes_use_what_the_tuner_reports(nb, n):
    """Shape 0, 0 is the kernel that takes a step in one launch. Last in the file: a shape
    that wins stays the default of its size class in this process."""
    t = nb.autotune(n, nb.TUNE_DIRECT, 3)
    assert t["direct_ms"] > 0 and (t["bodies_per_lane"] == 0) == (t["j_split"] == 0)
    pos, vel, m = nb.ic_plummer(n, n, 50.0, 1e4)
    m[::3] *= 1.5  # no equal masses: the kernels add in different orders
    out = []
    for shape in ((0, 0), (t["bodies_per_lane"], t["j_split"])):
        with nb.Simulation(n, EPS2, DT, bodies_per_lane=shape[0], j_split=shape[1]) as sim:
            sim.upload(pos, vel, m)
            sim.step(2)
            out.append(sim.download_f64())
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    if t["bodies_per_lane"]:
        got = nb.get_tuning(n)
        assert (got["bodies_per_lane"], got["j_split"]) == (t["bodies_per_lane"], t["j_split"])
