"""Parity of the device-built Barnes-Hut octree with the reference tree.

Topology (node levels, branches, centres, sizes and per-leaf particle) must be
bit-identical to the reference's insertion-built octree (oracle restatement, itself
bit-identical to gravhopper/_jbgrav.c's tree forces).  The FP64 walk must accept the
same nodes as the reference walk (exact interaction counts per target) and give the
same forces up to summation order.

The FP32 walk opens nodes by a group test that accepts a node only where the
reference's test accepts it for every target of the group, so each target's
interactions refine the reference's.  It is checked three ways: (1) its FP32 arithmetic
against the same interaction lists evaluated in FP64 (GH_TUNE_WALK_F64EVAL), at the
direct sum's FP32 tolerance; (2) its accuracy against the FP64 direct sum, which must be
no worse than the reference tree's; (3) at theta = 0 every list is every particle, so
the walk must equal the direct sum.
"""
import numpy as np
import pytest

from conftest import assert_bitwise, rel_err
from gravhopper_amd import Simulation, _native, workloads

pytestmark = pytest.mark.gpu

FP64, FP32 = _native.GH_FP64, _native.GH_FP32

# FP32 walk arithmetic against the same lists in FP64: FP32 monopoles, FP32 sums of at
# most 64 / (64 / G) list entries per lane added into FP64 (the direct sum's tolerance)
FP32_LIST_MEDIAN, FP32_LIST_P99 = 1e-6, 1e-4


def fp32_walk(ctx, pos, mass, eps, theta, fpos=None):
    """FP32 group walk, and the same interaction lists evaluated in FP64."""
    got = ctx.tree(pos, mass, eps, theta, FP32, force_pos=fpos)
    ctx.set_tuning(_native.TUNE_WALK_F64EVAL, 1)
    try:
        ref = ctx.tree(pos, mass, eps, theta, FP32, force_pos=fpos)
    finally:
        ctx.set_tuning(_native.TUNE_WALK_F64EVAL, 0)
    return got, ref


def check_fp32_walk(ctx, oracle, pos, mass, eps, theta, fpos=None, what=""):
    got, lists64 = fp32_walk(ctx, pos, mass, eps, theta, fpos)
    e = rel_err(got, lists64)
    print("%s: fp32 vs same lists in fp64: median %.2e p99 %.2e"
          % (what, np.median(e), np.percentile(e, 99)), flush=True)
    assert np.median(e) <= FP32_LIST_MEDIAN and np.percentile(e, 99) <= FP32_LIST_P99, what
    # accuracy against the FP64 direct sum: no worse than the reference tree's
    if fpos is None:
        direct = oracle.direct(pos, mass, eps)
        reftree = oracle.tree(pos, mass, eps, theta)
    else:
        direct = oracle.direct_position(pos, mass, fpos, eps)
        reftree = oracle.tree(pos, mass, eps, theta, force_pos=fpos)
    eg, er = rel_err(lists64, direct), rel_err(reftree, direct)
    print("%s: vs direct: group walk median %.2e p99 %.2e, reference tree %.2e / %.2e"
          % (what, np.median(eg), np.percentile(eg, 99), np.median(er),
             np.percentile(er, 99)), flush=True)
    assert np.median(eg) <= np.median(er) * 1.001 + 1e-15, what
    assert np.percentile(eg, 99) <= np.percentile(er, 99) * 1.05 + 1e-15, what
    return got


def compare_topology(got, want, name):
    assert len(got) == len(want), "%s: %d vs %d nodes" % (name, len(got), len(want))
    for f in ("level", "branch", "leaf"):
        assert np.array_equal(got[f], want[f]), "%s: %s differs" % (name, f)
    assert_bitwise(got["center"], want["center"], name + " centre")
    assert_bitwise(got["size"], want["size"], name + " size")
    # moments: double-double prefix sums vs the reference's insertion-order sums
    np.testing.assert_allclose(got["mass"], want["mass"], rtol=1e-13)
    scale = np.abs(want["center"]).max() + want["size"][0]
    np.testing.assert_allclose(got["com"], want["com"], rtol=1e-12, atol=1e-13 * scale)


def tree_cases():
    rng = np.random.default_rng(2026)
    cases = []
    cases.append(("one", np.array([[0.5, -0.25, 2.0]]), np.ones(1), 0.1))
    cases.append(("two", np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]]), np.array([1.0, 2.0]), 0.0))
    cases.append(("cauchy_3000", rng.standard_cauchy(size=(3000, 3)), rng.uniform(1, 2, 3000), 1e-3))
    p = workloads.plummer(8192, seed=77)
    cases.append(("plummer_8192", p["pos"], p["mass"], 1e-5))
    g = workloads.galaxy(n_halo=8192, n_disk=8192, seed=78)
    cases.append(("galaxy_16384", g["pos"], g["mass"], 0.05))
    # coordinates exactly on dyadic cell walls of the root box
    w = np.unique(rng.integers(-16, 17, size=(3000, 3)).astype(float) / 16.0, axis=0)
    cases.append(("walls", w, np.ones(len(w)), 0.0))
    # a very close pair needing more than 21 (and 42) levels of octant digits
    deep = rng.normal(size=(500, 3))
    deep[1] = deep[0] + np.array([1e-9, -2e-9, 3e-10])
    deep[2] = deep[0] + np.array([1e-14, 0, 0])
    cases.append(("deep", deep, rng.uniform(1, 2, 500), 1e-3))
    return cases


# edges of a wavefront's list, of the runs and of the range of the two-launch sort
@pytest.mark.parametrize("n", [2, 64, 65, 1023, 1024, 1025, 17000, 100000, 100001])
def test_key_sort_forms_agree(ctx, n):
    # clusters of equal high digits, and (not for the smallest) two particles that only a
    # second key word separates
    sizes = [66, 2] if n > 100 else []
    pos, mass = clustered(n - sum(sizes), sizes, seed=n)
    if n > 64:
        pos[5] = pos[4] * (1.0 + 1e-14)
    fpos = np.random.default_rng(n).normal(size=(max(n, 4096), 3)) * 2.0
    fpos[7:90] = fpos[7]  # equal keys
    out = {}
    for mode in (0, 1, 0, -1):
        ctx.set_tuning(_native.TUNE_TREE_SORT, mode)
        try:
            out[mode] = (ctx.tree(pos, mass, 1e-3, 0.7, FP64),
                         ctx.tree(pos, mass, 1e-3, 0.7, FP32, force_pos=fpos))
        finally:
            ctx.set_tuning(_native.TUNE_TREE_SORT, 0)
    for mode in (1, -1):
        for g, w in zip(out[0], out[mode]):
            assert_bitwise(g, w, "mode %d" % mode)


@pytest.mark.parametrize("case", tree_cases(), ids=lambda c: c[0])
def test_topology_bitwise(ctx, oracle, case):
    name, pos, mass, eps = case
    print("case", name, len(pos), flush=True)
    compare_topology(ctx.tree_dump(pos, mass, eps), oracle.tree_dump(pos, mass, eps), name)


@pytest.mark.parametrize("n", [4096, 4097, 65536, 70000])
def test_topology_bitwise_search_levels(ctx, oracle, n):
    # node ends come from a search over group minima whose number of levels grows with
    # n (3 up to 4096 particles, 4 up to 65536, 5 beyond): sizes on either side of the
    # steps, clustered so that large nodes reach the upper levels
    rng = np.random.default_rng(n)
    pos = np.concatenate([rng.normal(size=(n // 2, 3)) * 1e-3,
                          rng.standard_cauchy(size=(n - n // 2, 3))])
    mass = rng.uniform(1, 2, n)
    print("n", n, flush=True)
    compare_topology(ctx.tree_dump(pos, mass, 1e-3), oracle.tree_dump(pos, mass, 1e-3),
                     "n=%d" % n)


def clustered(n_field, sizes, seed):
    """Field particles plus tight clusters (spread 1e-6 of a root box of about 10), each
    inside one cell of octree level 12, so their keys agree over levels 0-12."""
    rng = np.random.default_rng(seed)
    parts = [rng.normal(size=(n_field, 3)) * 2.0]
    for k in sizes:
        parts.append(rng.normal(size=(1, 3)) + rng.normal(size=(k, 3)) * 1e-6)
    pos = np.concatenate(parts)
    return pos, rng.uniform(1, 2, len(pos))


@pytest.mark.parametrize("mode", [1, -1, 0])
def test_topology_bitwise_key_runs(ctx, oracle, mode):
    # runs of 2..64 keys equal over levels 0-12 are ordered by k_sort_runs after the radix
    # passes over those levels (mode 1); -1 sorts over all levels; each gives the same tree
    pos, mass = clustered(20000, [2, 3, 5, 17, 40, 63, 64], seed=11)
    ctx.set_tuning(_native.TUNE_TREE_SORT, mode)
    try:
        print("mode", mode, len(pos), flush=True)
        compare_topology(ctx.tree_dump(pos, mass, 1e-3), oracle.tree_dump(pos, mass, 1e-3),
                         "runs, mode %d" % mode)
    finally:
        ctx.set_tuning(_native.TUNE_TREE_SORT, 0)


@pytest.mark.parametrize("n", [2, 3, 5])
def test_topology_bitwise_key_runs_small(ctx, oracle, n):
    # n particles 1e-7 apart in a root box of about 10 (set by one far particle): their
    # keys agree over levels 0-12, one run of n
    rng = np.random.default_rng(n)
    pos = np.concatenate([rng.normal(size=(1, 3)) + rng.normal(size=(n, 3)) * 1e-7,
                          [[10.0, -3.0, 2.0]]])
    mass = rng.uniform(1, 2, n + 1)
    ctx.set_tuning(_native.TUNE_TREE_SORT, 1)
    try:
        compare_topology(ctx.tree_dump(pos, mass, 0.0), oracle.tree_dump(pos, mass, 0.0),
                         "one run of %d" % n)
    finally:
        ctx.set_tuning(_native.TUNE_TREE_SORT, 0)


@pytest.mark.parametrize("mode", [1, 0])
def test_topology_bitwise_long_key_run(ctx, oracle, mode):
    # a run of 65 or 300 keys is longer than k_sort_runs takes: the build sorts again over
    # all levels; in the automatic mode the next builds start that way (same results)
    ctx.set_tuning(_native.TUNE_TREE_SORT, mode)
    try:
        for sizes in ([65], [300, 4], [3]):
            pos, mass = clustered(5000, sizes, seed=12)
            print("mode", mode, "clusters", sizes, flush=True)
            compare_topology(ctx.tree_dump(pos, mass, 1e-3),
                             oracle.tree_dump(pos, mass, 1e-3), "clusters %s" % sizes)
            want, wcnt = oracle.tree(pos, mass, 1e-3, 0.7, count=True)
            got, gcnt = ctx.tree_interactions(pos, mass, 1e-3, 0.7)
            assert np.array_equal(gcnt, wcnt), "clusters %s: accepted-node counts" % sizes
            # a cluster member's accepted nodes lie about 1e-6 away, so the reference's
            # centres of mass (running sums, rounding about 1e-15 absolute) move its
            # force by about 1e-8 relative; the device's come from double-double sums
            np.testing.assert_allclose(got, want, rtol=1e-6, atol=1e-10 * np.abs(want).max())
    finally:
        ctx.set_tuning(_native.TUNE_TREE_SORT, 0)


@pytest.mark.parametrize("case", tree_cases(), ids=lambda c: c[0])
def test_fp64_walk_matches_reference(ctx, oracle, case):
    name, pos, mass, eps = case
    print("case", name, len(pos), flush=True)
    for theta in (0.0, 0.7):
        want, wcnt = oracle.tree(pos, mass, eps, theta, count=True)
        got, gcnt = ctx.tree_interactions(pos, mass, eps, theta)
        assert np.array_equal(gcnt, wcnt), "%s theta=%g: accepted-node counts" % (name, theta)
        # same accepted nodes, different summation order and moment rounding
        scale = np.abs(want).max() if len(want) else 1.0
        np.testing.assert_allclose(got, want, rtol=1e-10, atol=1e-12 * scale)


def test_fp64_tree_golden(ctx, golden):
    for name, c in golden.items():
        for theta in (0.3, 0.7):
            want = c["tree_%g" % theta]
            got = ctx.tree(c["pos"], c["mass"], float(c["eps"]), theta, FP64)
            scale = np.abs(want).max()
            np.testing.assert_allclose(got, want, rtol=1e-10, atol=1e-12 * scale, err_msg=name)
            want = c["tree_position_%g" % theta]
            got = ctx.tree(c["pos"], c["mass"], float(c["eps"]), theta, FP64,
                           force_pos=c["force_pos"])
            np.testing.assert_allclose(got, want, rtol=1e-10, atol=1e-12 * np.abs(want).max(),
                                       err_msg=name + " position")


@pytest.mark.parametrize("n_targets", [400, 9000])
def test_position_walk_counts(ctx, oracle, n_targets):
    # 9000 targets are walked in the library's own Morton order of the targets (from
    # 4096 on); results must come back in the caller's order.  Some targets lie
    # outside the particles' root box.
    rng = np.random.default_rng(91)
    pos = rng.normal(size=(5000, 3))
    mass = rng.uniform(size=5000)
    fpos = np.concatenate([pos[:100], rng.normal(size=(n_targets - 100, 3)) * 3])
    want, wcnt = oracle.tree(pos, mass, 0.01, 0.7, force_pos=fpos, count=True)
    got, gcnt = ctx.tree_interactions(pos, mass, 0.01, 0.7, force_pos=fpos)
    assert np.array_equal(gcnt, wcnt)
    np.testing.assert_allclose(got, want, rtol=1e-10, atol=1e-12 * np.abs(want).max())
    got = ctx.tree(pos, mass, 0.01, 0.7, FP64, force_pos=fpos)
    np.testing.assert_allclose(got, want, rtol=1e-10, atol=1e-12 * np.abs(want).max())
    check_fp32_walk(ctx, oracle, pos, mass, 0.01, 0.7, fpos=fpos, what="%d targets" % n_targets)


@pytest.mark.parametrize("theta", [0.3, 0.7, 1.0])
def test_fp32_walk_accuracy(ctx, oracle, theta):
    g = workloads.galaxy(n_halo=16384, n_disk=16384, seed=79)
    check_fp32_walk(ctx, oracle, g["pos"], g["mass"], 0.05, theta,
                    what="galaxy 32768 theta %g" % theta)


def test_fp32_walk_theta0_is_direct_sum(ctx, oracle):
    # theta = 0 opens every internal node: every list is every particle exactly once
    g = workloads.galaxy(n_halo=10000, n_disk=10000, seed=92)
    got = ctx.tree(g["pos"], g["mass"], 0.05, 0.0, FP32)
    e = rel_err(got, oracle.direct(g["pos"], g["mass"], 0.05))
    assert np.median(e) < 1e-6 and np.percentile(e, 99) < 1e-4


def test_tree_edge_cases(ctx):
    with pytest.raises(_native.GravhopError, match="share a position"):
        ctx.tree(np.array([[0.0, 0, 0], [1, 1, 1], [0, 0, 0]]), np.ones(3), 0.1, 0.7)
    out = ctx.tree(np.zeros((0, 3)), np.zeros(0), 0.1, 0.7, FP64, force_pos=np.ones((3, 3)))
    assert np.all(out == 0)
    out = ctx.tree(np.ones((1, 3)), np.ones(1), 0.0, 0.7, FP64)
    assert np.all(out == 0)


def test_tree_deterministic(ctx):
    g = workloads.galaxy(n_halo=30000, n_disk=30000, seed=80)
    a = ctx.tree(g["pos"], g["mass"], 0.05, 0.7, FP32)
    b = ctx.tree(g["pos"], g["mass"], 0.05, 0.7, FP32)
    assert_bitwise(a, b)


def test_simulation_tree_device_vs_host(ctx):
    ic = workloads.plummer(2000, seed=81)
    a = Simulation(dt=0.005, eps=5e-5, algorithm='tree')
    a.add_IC(ic)
    a.run(4)
    b = Simulation(dt=0.005, eps=5e-5, algorithm='tree', device_loop=False)
    b.add_IC(ic)
    b.add_external_force(lambda pos, args: np.zeros_like(pos))
    b.run(4)
    assert_bitwise(a.positions, b.positions)
    assert_bitwise(a.velocities, b.velocities)


@pytest.mark.parametrize("group", [1, 2, 4, 8, 16])
def test_fp32_walk_group_sizes(ctx, oracle, group):
    # any group size: FP32 arithmetic against the same lists in FP64, accuracy no worse
    # than the reference tree, and repeated calls bit-identical
    g = workloads.galaxy(n_halo=12000, n_disk=12000, seed=82)
    ctx.set_tuning(_native.TUNE_WALK_GROUP, group)
    try:
        a = check_fp32_walk(ctx, oracle, g["pos"], g["mass"], 0.05, 0.7,
                            what="group %d" % group)
        b = ctx.tree(g["pos"], g["mass"], 0.05, 0.7, FP32)
    finally:
        ctx.set_tuning(_native.TUNE_WALK_GROUP, 0)
    assert_bitwise(a, b)


def test_fp64_walk_independent_of_target_grouping(ctx):
    # The FP64 walk sums each target's accepted nodes in tree order, whatever the other
    # targets of its wavefront: a target's force is bit-identical among 300 targets
    # (5 per walk), among 20000 (sorted, 5 per walk) or as a particle of the self walk
    # (Morton order, 64 per walk).
    g = workloads.galaxy(n_halo=150000, n_disk=150000, seed=86)
    pos, mass = g["pos"], g["mass"]
    rng = np.random.default_rng(87)
    pick = rng.choice(len(mass), 20000, replace=False)
    fpos = pos[pick]
    self_acc = ctx.tree(pos, mass, 0.05, 0.7, FP64)
    all_pos = ctx.tree(pos, mass, 0.05, 0.7, FP64, force_pos=fpos)
    few_pos = ctx.tree(pos, mass, 0.05, 0.7, FP64, force_pos=fpos[:300])
    assert_bitwise(all_pos[:300], few_pos, "300 vs 20000 targets")
    assert_bitwise(all_pos, self_acc[pick], "position targets vs self walk")


@pytest.mark.parametrize("group", [0, 1, 4, 16, 64])
def test_fp32_walk_prefix_same_lists(ctx, group):
    # the walks of a block of groups start from the nodes k_walk_prefix decided for all of
    # them (accepted into the list, or opened) and the nodes it deferred; every target's
    # list must hold as many nodes as from the root (the same nodes, in another order),
    # and the forces differ only by FP32 summation order
    rng = np.random.default_rng(404)
    g = workloads.galaxy(n_halo=40000, n_disk=40000, seed=405)
    fpos = np.concatenate([g["pos"][:5000], rng.normal(size=(9000, 3)) * 300.0])
    fpos[7000, 1] = np.nan  # its block of groups starts from the root
    cases = [("galaxy", g["pos"], g["mass"], 0.05, None),
             ("cauchy", rng.standard_cauchy(size=(30000, 3)), rng.uniform(1, 2, 30000), 1e-3, None),
             ("positions", g["pos"], g["mass"], 0.05, fpos),
             ("tiny", rng.normal(size=(50, 3)), rng.uniform(1, 2, 50), 1e-2,
              rng.normal(size=(7, 3)))]
    ctx.set_tuning(_native.TUNE_WALK_GROUP, group)
    try:
        for name, pos, mass, eps, fpos in cases:
            for theta in (0.0, 0.4, 0.7, 1.2):
                what = "%s G=%d theta=%g" % (name, group, theta)
                print(what, flush=True)
                got, gcnt = ctx.tree_interactions(pos, mass, eps, theta, force_pos=fpos,
                                                  precision=FP32)
                ctx.set_tuning(_native.TUNE_WALK_PREFIX, -1)
                try:
                    want, wcnt = ctx.tree_interactions(pos, mass, eps, theta, force_pos=fpos,
                                                       precision=FP32)
                finally:
                    ctx.set_tuning(_native.TUNE_WALK_PREFIX, 0)
                assert np.array_equal(gcnt, wcnt), what + ": list lengths"
                fin = np.isfinite(want).all(axis=1)
                assert np.array_equal(fin, np.isfinite(got).all(axis=1)), what
                e = rel_err(got[fin], want[fin])
                assert np.median(e) <= FP32_LIST_MEDIAN and np.percentile(e, 99) <= FP32_LIST_P99, what
    finally:
        ctx.set_tuning(_native.TUNE_WALK_GROUP, 0)


def test_fp32_walk_few_targets(ctx, oracle):
    # few position targets are spread over many short walks (down to one target each)
    rng = np.random.default_rng(88)
    pos = rng.normal(size=(20000, 3))
    mass = rng.uniform(size=20000)
    for nt in (1, 7, 300):
        fpos = rng.normal(size=(nt, 3)) * 2
        check_fp32_walk(ctx, oracle, pos, mass, 0.01, 0.7, fpos=fpos, what="%d targets" % nt)


def test_fp32_walk_zero_softening(ctx, oracle):
    # eps = 0: the walk's guarded form, where a zero separation (a particle's own leaf,
    # or a target on a particle) gives zero force, as in the reference's tree walk
    rng = np.random.default_rng(89)
    pos = rng.normal(size=(6000, 3))
    mass = rng.uniform(1, 2, 6000)
    got = check_fp32_walk(ctx, oracle, pos, mass, 0.0, 0.7, what="eps 0")
    assert np.all(np.isfinite(got))
    fpos = np.concatenate([pos[:50], rng.normal(size=(250, 3))])
    got = check_fp32_walk(ctx, oracle, pos, mass, 0.0, 0.7, fpos=fpos, what="eps 0 targets")
    assert np.all(np.isfinite(got))


@pytest.mark.parametrize("group", [0, 2, 16])
def test_fp32_walk_list_lengths(ctx, group):
    # every target's list refines the reference's accepted nodes, so it is never shorter;
    # and the group test must not open far more than the reference (a loose group, whose
    # sorted targets jump across the system, is walked target by target)
    g = workloads.galaxy(n_halo=32768, n_disk=32768, seed=3)
    _, cref = ctx.tree_interactions(g["pos"], g["mass"], 0.05, 0.7)
    ctx.set_tuning(_native.TUNE_WALK_GROUP, group)
    try:
        _, c32 = ctx.tree_interactions(g["pos"], g["mass"], 0.05, 0.7, precision=FP32)
    finally:
        ctx.set_tuning(_native.TUNE_WALK_GROUP, 0)
    print("group %d: list mean %.0f max %d; reference mean %.0f max %d"
          % (group, c32.mean(), c32.max(), cref.mean(), cref.max()), flush=True)
    assert np.all(c32 >= cref)
    assert c32.mean() < 2.5 * cref.mean()
    assert c32.max() < 8 * cref.max()


# targets per walk change at these counts (walk() in gh_tree.hip), for particles
@pytest.mark.parametrize("n", [2560, 2561, 5121, 10241, 20481, 40961, 200000, 200001])
def test_fp64_walk_shapes_same_bits(ctx, n):
    # a particle's force is the same bits from the self walk and from a walk of its own
    # (few position targets: one per walk)
    rng = np.random.default_rng(n)
    pos = rng.normal(size=(n, 3)) * np.exp(rng.normal(size=(n, 1)))
    mass = rng.uniform(0.5, 2.0, size=n)
    some = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, size=400)]))
    for eps, theta in ((0.01, 0.7), (0.0, 0.7), (0.01, 0.5), (0.01, 0.4)):
        if n > 100000 and theta != 0.7:
            continue
        full = ctx.tree(pos, mass, eps, theta, FP64)
        own = ctx.tree(pos, mass, eps, theta, FP64, force_pos=pos[some])
        assert_bitwise(full[some], own, "eps=%g theta=%g" % (eps, theta))


# ... and for position targets (sorted from 4096 on)
@pytest.mark.parametrize("nf", [1, 4095, 4096, 20001, 40001, 80001, 160001, 400001])
def test_fp64_walk_target_shapes_same_bits(ctx, nf):
    rng = np.random.default_rng(nf)
    pos = rng.normal(size=(5000, 3))
    mass = rng.uniform(0.5, 2.0, size=5000)
    fpos = rng.normal(size=(nf, 3)) * 2
    fpos[::50] = pos[rng.integers(0, 5000, size=len(fpos[::50]))]
    some = np.unique(np.concatenate([[0, nf - 1], rng.integers(0, nf, size=300)]))
    full = ctx.tree(pos, mass, 0.01, 0.7, FP64, force_pos=fpos)
    own = ctx.tree(pos, mass, 0.01, 0.7, FP64, force_pos=fpos[some])
    assert_bitwise(full[some], own)


@pytest.mark.parametrize("n", [3, 70, 600, 6000, 12000])
def test_fp64_walk_full_stack(ctx, oracle, n):
    """Walks that open almost every node (theta 0 to 0.2) of trees of up to 40 levels: the
    stack fills, steps take few nodes, and subtrees are walked one node at a time."""
    rng = np.random.default_rng(n)
    pos = rng.normal(size=(n, 3))
    tight = n // 3
    pos[:tight] = pos[0] + rng.normal(size=(tight, 3)) * 10.0 ** rng.uniform(-10, 0, (tight, 1))
    mass = rng.uniform(0.5, 2.0, size=n)
    some = np.unique(rng.integers(0, n, size=200))
    for theta in (0.0, 0.05, 0.2, 0.7):
        want, cnt = oracle.tree(pos, mass, 0.01, theta, force_pos=pos[some], count=True)
        got = ctx.tree(pos, mass, 0.01, theta, FP64)
        np.testing.assert_allclose(got[some], want, rtol=1e-10,
                                   atol=1e-10 * np.abs(want).max(), err_msg="theta=%g" % theta)
        _, gcnt = ctx.tree_interactions(pos, mass, 0.01, theta, precision=FP64)
        assert np.array_equal(gcnt[some], cnt), theta


def test_fp64_walk_target_not_finite(ctx, oracle):
    # such a target gets what the reference gives it and leaves its neighbours alone
    rng = np.random.default_rng(5)
    n = 6000
    pos = rng.normal(size=(n, 3))
    mass = rng.uniform(0.5, 2.0, size=n)
    fpos = rng.normal(size=(5000, 3))
    fpos[1000] = [np.nan, 0, 0]
    fpos[2000] = [0, np.inf, 0]
    fpos[3000] = [0, 0, 1e300]
    some = np.array([0, 999, 1001, 1999, 2001, 2999, 3001, 4999])
    got = ctx.tree(pos, mass, 0.01, 0.7, FP64, force_pos=fpos)
    assert_bitwise(got[some], ctx.tree(pos, mass, 0.01, 0.7, FP64, force_pos=fpos[some]))
    assert np.all(np.isnan(got[1000]))
    fine = np.delete(np.arange(5000), [1000, 2000, 3000])
    assert np.all(np.isfinite(got[fine]))


@pytest.mark.parametrize("prec", [FP64, FP32])
def test_walk_queued_before_the_node_count(ctx, prec):
    # One context's trees of different kinds in turn: more nodes than the last one left room
    # for, more than 2 per particle, a second key word, equal keys, and trees that are refused.
    # Each equals what a context that has built nothing before gives.
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(5)

    def close_pairs(n, apart):
        pos = rng.normal(size=(n // 2, 3))
        return np.concatenate([pos, pos * (1.0 + apart)])

    trees = [rng.normal(size=(n, 3)) for n in (300, 50, 3000, 2, 3000, 40000)]
    trees += [close_pairs(2000, 1e-5), close_pairs(2000, 1e-14), rng.normal(size=(2000, 3)),
              clustered(101000, [70], seed=3)[0], rng.normal(size=(1, 3)), close_pairs(300, 1e-5)]
    used = _native.Context(0)
    try:
        for k, pos in enumerate(trees):
            mass = rng.uniform(0.5, 1.0, len(pos))
            fresh = _native.Context(0)
            want = fresh.tree(pos, mass, 1e-3, 0.7, prec)
            fresh.close()
            for again in range(2):
                assert_bitwise(used.tree(pos, mass, 1e-3, 0.7, prec), want, "tree %d" % k)
            x = torch.ones((9, 3), dtype=torch.float64, device="cuda")  # all at one place
            m = torch.ones(9, dtype=torch.float64, device="cuda")
            acc = torch.full((9, 3), 7.0, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            with pytest.raises(_native.GravhopError) as e:
                used.tree_dev(x.data_ptr(), m.data_ptr(), 9, 1e-3, 0.7, prec, acc.data_ptr())
            assert e.value.code == _native.GH_ECOINCIDENT
            assert torch.equal(acc, torch.full_like(acc, 7.0))
    finally:
        used.close()


@pytest.mark.parametrize("n", [49152, 49153])  # the most walks of 16 that are resident, and more
def test_fp64_walk_workgroups(ctx, n):
    # one and two walks per workgroup: a target's bits do not depend on its neighbours
    rng = np.random.default_rng(n)
    pos, mass = rng.normal(size=(n, 3)), rng.uniform(0.5, 1.0, size=n)
    whole = ctx.tree(pos, mass, 1e-3, 0.7, FP64)
    for nf in (3072, 3073):
        pick = rng.permutation(n)[:nf]
        assert_bitwise(ctx.tree(pos, mass, 1e-3, 0.7, FP64, force_pos=pos[pick]), whole[pick],
                       "%d targets" % nf)


def massless(case):
    rng = np.random.default_rng(11)
    if case == "pair":
        pos = np.array([[0.0, 0, 0], [1.0, 0.5, 0.2]])
    elif case == "octants":
        pos = rng.uniform(0.5, 1.0, (8, 3)) * (2 * np.indices((2, 2, 2)).reshape(3, 8).T - 1)
    elif case == "close pair":
        pos = np.array([[0.0, 0, 0], [1e-3, 0, 0], [1.0, 0.5, 0.2]])
    else:  # a massless pair among others, whose node few, some or most of them accept
        pos = rng.normal(size=(int(case), 3))
        pos[[1, 4]] = [[4.0, 4.0, 4.0], [4.5, 4.0, 4.0]]
        mass = rng.uniform(0.5, 2.0, len(pos))
        mass[[1, 4]] = 0.0
        return pos, mass
    return pos, np.zeros(len(pos))


# targets per walk: 1 of them up to 2560 particles, 2, 4, 16 and 64
@pytest.mark.parametrize("eps", [0.01, 0.0])
@pytest.mark.parametrize("case", ["pair", "octants", "close pair", "6", "2000", "3000", "6000",
                                  "30000", "200002"])
def test_fp64_walk_massless(ctx, oracle, case, eps):
    """A node without mass has no centre of mass (0/0, as in the reference): who accepts it
    gets NaN, and nobody else does."""
    pos, mass = massless(case)
    some = np.unique(np.concatenate([np.arange(min(len(pos), 9)),
                                     np.random.default_rng(1).integers(0, len(pos), 300)]))
    for theta in (0.7, 0.15, 0.05):
        want = oracle.tree(pos, mass, eps, theta, force_pos=pos[some])
        got = ctx.tree(pos, mass, eps, theta, FP64)[some]
        own = ctx.tree(pos, mass, eps, theta, FP64, force_pos=pos[some])
        assert np.array_equal(np.isnan(got), np.isnan(want)), theta
        np.testing.assert_allclose(got, want, rtol=1e-10, err_msg="theta=%g" % theta,
                                   atol=1e-10 * np.nanmax(np.abs(want), initial=0.0))
        assert np.array_equal(got, own, equal_nan=True), theta


# 2, 16 and 64 targets per walk
@pytest.mark.parametrize("side", [16, 32, 64])
def test_fp64_walk_ties_far_from_the_origin(ctx, oracle, side):
    """A lattice 8 kpc from the origin, and theta where targets lie on the threshold of the
    nodes of eight: what a walk decides for all of its targets at once is what the reference
    decides for each, to the last ulp of their coordinates."""
    h = 1e-6
    pos = np.array([8.1, -8.2, 0.3]) + h * np.indices((side,) * 3).reshape(3, -1).T
    mass = np.random.default_rng(side).uniform(0.5, 2.0, len(pos))
    some = np.random.default_rng(side).permutation(len(pos))[:3000]
    for d2 in (0.5 ** 2 + 0.5 ** 2 + 3.5 ** 2, 0.5 ** 2 + 1.5 ** 2 + 2.5 ** 2, 3 * 2.5 ** 2):
        theta = 2.0 / np.sqrt(d2)
        _, want = oracle.tree(pos, mass, h, theta, force_pos=pos[some], count=True)
        _, count = ctx.tree_interactions(pos, mass, h, theta)
        own, alone = ctx.tree_interactions(pos, mass, h, theta, force_pos=pos[some])
        assert np.array_equal(alone, want), d2
        assert np.array_equal(count[some], want), d2
        assert_bitwise(ctx.tree(pos, mass, h, theta, FP64)[some], own, "d2=%g" % d2)


# the deepest walks (16 and 64 targets, 1536 stack entries) and the sizes before them
@pytest.mark.parametrize("n,nf,theta", [(100000, 0, 0.3), (100001, 0, 0.3), (150000, 0, 0.2),
                                        (150001, 0, 0.2), (150001, 0, 0.349), (150001, 0, 0.35),
                                        (3000, 400001, 0.3), (3000, 400001, 0.4)])
def test_fp64_walk_deep_same_bits(ctx, n, nf, theta):
    rng = np.random.default_rng(n)
    pos = rng.standard_cauchy(size=(n, 3))
    mass = rng.uniform(0.5, 2.0, size=n)
    fpos = rng.standard_cauchy(size=(nf, 3)) if nf else None
    tgt = pos if fpos is None else fpos
    some = rng.permutation(len(tgt))[:400]
    full = ctx.tree(pos, mass, 0.01, theta, FP64, force_pos=fpos)
    assert_bitwise(full[some], ctx.tree(pos, mass, 0.01, theta, FP64, force_pos=tgt[some]))


# fields of few particles: targets per walk and stack entries go by their number
@pytest.mark.parametrize("n,nf", [(2, 200001), (2000, 200000), (2000, 200001), (2001, 200001),
                                  (5000, 30000), (5001, 30000), (20000, 400001), (20001, 400001)])
def test_fp64_walk_few_particles_same_bits(ctx, n, nf):
    rng = np.random.default_rng(n + nf)
    pos = rng.normal(size=(n, 3)) * np.exp(rng.normal(size=(n, 1)))
    mass = rng.uniform(0.5, 2.0, size=n)
    fpos = rng.normal(size=(nf, 3))
    fpos[::40] = pos[rng.integers(0, n, size=len(fpos[::40]))]
    some = rng.permutation(nf)[:400]
    for theta in (0.7, 0.3, 0.0 if n <= 2001 else 0.1):
        full = ctx.tree(pos, mass, 0.01, theta, FP64, force_pos=fpos)
        assert_bitwise(full[some], ctx.tree(pos, mass, 0.01, theta, FP64, force_pos=fpos[some]),
                       "theta=%g" % theta)
