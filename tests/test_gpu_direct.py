"""Parity of the GPU direct sum (libgravhop.so through the C ABI) with the reference.

FP64 mode must be bit-identical to the reference's direct_summation and
direct_summation_position (golden vectors written by the reference's own C code, and
the oracle restatement at other sizes).  FP32 mode is checked against the FP64 result
with a stated tolerance.
"""
import numpy as np
import pytest

from conftest import assert_bitwise, rel_err
from gravhopper_amd import _native, workloads

pytestmark = pytest.mark.gpu

FP64, FP32 = _native.GH_FP64, _native.GH_FP32


def test_fp64_direct_bitwise_golden(ctx, golden):
    for name, c in golden.items():
        print("case", name, flush=True)
        got = ctx.direct(c["pos"], c["mass"], float(c["eps"]), FP64)
        assert_bitwise(got, c["direct"], name)
        got = ctx.direct(c["pos"], c["mass"], float(c["eps"]), FP64, force_pos=c["force_pos"])
        assert_bitwise(got, c["direct_position"], name + " position")


@pytest.mark.parametrize("n", [1, 2, 3, 255, 256, 257, 1000, 2048])
def test_fp64_direct_bitwise_oracle(ctx, oracle, n):
    rng = np.random.default_rng(100 + n)
    pos = rng.standard_cauchy(size=(n, 3))
    mass = rng.uniform(0.1, 3.0, size=n)
    for eps in (0.0, 1e-3, 0.7):
        if n == 1 or eps > 0 or n > 1:
            got = ctx.direct(pos, mass, eps, FP64)
            assert_bitwise(got, oracle.direct(pos, mass, eps), "n=%d eps=%g" % (n, eps))
    fpos = np.concatenate([pos[: min(n, 7)], rng.normal(size=(5, 3))])
    for eps in (0.0, 0.01):
        got = ctx.direct(pos, mass, eps, FP64, force_pos=fpos)
        assert_bitwise(got, oracle.direct_position(pos, mass, fpos, eps), "pos n=%d" % n)


def test_fp64_direct_plummer_n2000(ctx, oracle):
    ic = workloads.plummer(2000, b=1e-3, mass=1e6, seed=20260001)
    got = ctx.direct(ic["pos"], ic["mass"], 5e-5, FP64)
    assert_bitwise(got, oracle.direct(ic["pos"], ic["mass"], 5e-5), "plummer 2000")


def test_empty_and_single(ctx):
    out = ctx.direct(np.zeros((0, 3)), np.zeros(0), 0.1, FP64)
    assert out.shape == (0, 3)
    out = ctx.direct(np.ones((1, 3)), np.ones(1), 0.0, FP64)
    assert np.all(out == 0.0)
    out = ctx.direct(np.ones((1, 3)), np.ones(1), 0.0, FP32)
    assert np.all(out == 0.0)
    out = ctx.direct(np.zeros((0, 3)), np.zeros(0), 0.1, FP32, force_pos=np.ones((4, 3)))
    assert np.all(out == 0.0)


# FP32 tolerance: pair forces in FP32 (v_rsq_f32 is accurate to 1 ulp), FP32 sums of
# 256-source tiles, compensated across tiles.  Median relative error <= 1e-6 and p99
# <= 1e-4 against the FP64 oracle on Plummer spheres.
FP32_MEDIAN = 1e-6
FP32_P99 = 1e-4


@pytest.mark.parametrize("n", [1000, 4096, 16384])
def test_fp32_direct_accuracy(ctx, oracle, n):
    ic = workloads.plummer(n, b=1e-3, mass=1e6, seed=n)
    ref = oracle.direct(ic["pos"], ic["mass"], 1e-5)
    got = ctx.direct(ic["pos"], ic["mass"], 1e-5, FP32)
    e = rel_err(got, ref)
    print("n=%d median %.3g p99 %.3g max %.3g" % (n, np.median(e), np.percentile(e, 99), e.max()))
    assert np.median(e) <= FP32_MEDIAN
    assert np.percentile(e, 99) <= FP32_P99


def test_fp32_position_and_zero_softening(ctx, oracle):
    rng = np.random.default_rng(5)
    pos = rng.normal(size=(3000, 3))
    mass = rng.uniform(size=3000)
    fpos = np.concatenate([pos[:50], rng.normal(size=(200, 3))])
    for eps in (0.0, 0.05):
        ref = oracle.direct_position(pos, mass, fpos, eps)
        got = ctx.direct(pos, mass, eps, FP32, force_pos=fpos)
        assert np.all(np.isfinite(got))
        e = rel_err(got, ref)
        assert np.median(e) < 1e-6, eps
    # self-exclusion with eps = 0 (the self pair is guarded to zero)
    got = ctx.direct(pos, mass, 0.0, FP32)
    e = rel_err(got, oracle.direct(pos, mass, 0.0))
    assert np.all(np.isfinite(got)) and np.median(e) < 1e-6


def test_fp32_split_sources_consistent(ctx, oracle):
    # few targets, many sources: the kernel splits sources over workgroups
    rng = np.random.default_rng(6)
    pos = rng.normal(size=(50000, 3))
    mass = rng.uniform(size=50000)
    fpos = rng.normal(size=(37, 3))
    ref = oracle.direct_position(pos, mass, fpos, 0.01)
    got = ctx.direct(pos, mass, 0.01, FP32, force_pos=fpos)
    assert np.median(rel_err(got, ref)) < 1e-6


def test_energy_matches_oracle(ctx, oracle):
    ic = workloads.plummer(3000, seed=9)
    ke, pe, p = ctx.energy(ic["pos"], ic["vel"], ic["mass"], 5e-5)
    ke0, pe0, p0 = oracle.energy(ic["pos"], ic["vel"], ic["mass"], 5e-5)
    assert abs(ke - ke0) <= 1e-12 * abs(ke0)
    assert abs(pe - pe0) <= 1e-12 * abs(pe0)
    assert np.allclose(p, p0, atol=1e-9 * np.abs(ic["mass"][:, None] * ic["vel"]).sum())


@pytest.mark.parametrize("ipt", [-1, 1, 2, 4])
@pytest.mark.parametrize("n,eps", [(5000, 1e-5), (20001, 1e-5), (3000, 0.0)])
def test_fp32_self_kernels(ctx, oracle, ipt, n, eps):
    """Every FP32 self-field kernel (one-sided, and pair-once with 1/2/4 particles per
    lane) against the FP64 oracle, including padding (n not a block multiple) and
    eps = 0 (zero-separation guard)."""
    ic = workloads.plummer(n, b=1e-3, mass=1e6, seed=n + 7)
    ref = oracle.direct(ic["pos"], ic["mass"], eps)
    ctx.set_tuning(_native.TUNE_DIRECT_SELF, ipt)
    try:
        got = ctx.direct(ic["pos"], ic["mass"], eps, FP32)
    finally:
        ctx.set_tuning(_native.TUNE_DIRECT_SELF, 0)
    assert np.all(np.isfinite(got))
    e = rel_err(got, ref)
    print("ipt=%d n=%d eps=%g median %.3g p99 %.3g" % (ipt, n, eps, np.median(e),
                                                      np.percentile(e, 99)))
    assert np.median(e) <= FP32_MEDIAN
    assert np.percentile(e, 99) <= FP32_P99
    # momentum: the pair-once kernels give exactly opposite pair forces
    if ipt > 0:
        tot = (ic["mass"][:, None] * got).sum(0)
        assert np.all(np.abs(tot) <= 1e-5 * (ic["mass"][:, None] * np.abs(got)).sum(0))


def test_fp32_self_kernels_agree_unequal_masses(ctx):
    rng = np.random.default_rng(55)
    pos = rng.normal(size=(17000, 3))
    mass = rng.lognormal(size=17000)
    out = {}
    for ipt in (-1, 1, 4):
        ctx.set_tuning(_native.TUNE_DIRECT_SELF, ipt)
        out[ipt] = ctx.direct(pos, mass, 0.01, FP32)
    ctx.set_tuning(_native.TUNE_DIRECT_SELF, 0)
    for ipt in (1, 4):
        assert np.median(rel_err(out[ipt], out[-1])) < 1e-6


@pytest.mark.parametrize("tpw", [1, 2, 4, 8, 16, 32, 64, -1, -2, -4, -8, -16])
def test_fp64_direct_targets_per_wave_bitwise(ctx, oracle, tpw):
    # every spread of a target's terms over lanes (positive: the spread kernel, negative:
    # a lane per component sum) adds them in the reference's order
    rng = np.random.default_rng(300 + tpw)
    n = 777
    pos = rng.standard_cauchy(size=(n, 3))
    mass = rng.uniform(0.1, 3.0, size=n)
    fpos = np.concatenate([pos[:9], rng.normal(size=(40, 3))])
    try:
        ctx.set_tuning(_native.TUNE_DIRECT_F64_TPW, tpw)
        for eps in (0.0, 1e-3):
            assert_bitwise(ctx.direct(pos, mass, eps, FP64), oracle.direct(pos, mass, eps),
                           "self eps=%g" % eps)
            assert_bitwise(ctx.direct(pos, mass, eps, FP64, force_pos=fpos),
                           oracle.direct_position(pos, mass, fpos, eps), "position eps=%g" % eps)
            # fewer sources than one chunk, and fewer targets than one wavefront's
            assert_bitwise(ctx.direct(pos[:5], mass[:5], eps, FP64),
                           oracle.direct(pos[:5], mass[:5], eps), "5 particles eps=%g" % eps)
            assert_bitwise(ctx.direct(pos[:70], mass[:70], eps, FP64, force_pos=fpos[:3]),
                           oracle.direct_position(pos[:70], mass[:70], fpos[:3], eps),
                           "3 targets eps=%g" % eps)
    finally:
        ctx.set_tuning(_native.TUNE_DIRECT_F64_TPW, 0)


@pytest.mark.parametrize("n", [1024, 1025, 4096, 4097])
def test_fp64_direct_automatic_shapes_bitwise(ctx, oracle, n):
    # both sides of the automatic shape steps (1, 2 and 4 targets per wavefront of the
    # per-sum-lane kernel) give the reference's bits
    rng = np.random.default_rng(400 + n)
    pos = rng.standard_cauchy(size=(n, 3))
    mass = rng.uniform(0.5, 2.0, size=n)
    assert_bitwise(ctx.direct(pos, mass, 1e-3, FP64), oracle.direct(pos, mass, 1e-3),
                   "self n=%d" % n)
    fpos = rng.normal(size=(n, 3))
    assert_bitwise(ctx.direct(pos, mass, 1e-3, FP64, force_pos=fpos),
                   oracle.direct_position(pos, mass, fpos, 1e-3), "position n=%d" % n)


@pytest.mark.parametrize("n", [2, 3, 255, 2047, 2049, 16384, 65536, 65537])
def test_fp32_sort_forms_agree(ctx, n):
    # the spatial order of up to 32 radix chunks (65536 points) takes one kernel per
    # pass; the classic histogram / scan / scatter passes must give the same order, so
    # the same FP32 forces bit for bit; both within the FP32 tolerance of the FP64 sum
    ic = workloads.plummer(n, b=1e-3, mass=1e6, seed=77 + n)
    pos = ic["pos"] + np.array([3.0, -8.0, 40.0])  # away from the origin
    got = ctx.direct(pos, ic["mass"], 1e-5, FP32)
    ctx.set_tuning(_native.TUNE_SORT_DIRECT, -1)
    try:
        classic = ctx.direct(pos, ic["mass"], 1e-5, FP32)
    finally:
        ctx.set_tuning(_native.TUNE_SORT_DIRECT, 0)
    assert_bitwise(got, classic, "n=%d" % n)
    if n >= 16:
        ref = ctx.direct(pos, ic["mass"], 1e-5, FP64)
        e = rel_err(got, ref)
        assert np.median(e) <= FP32_MEDIAN and np.percentile(e, 99) <= FP32_P99


# edges of the 64-point lists, the runs of 1024 and the part one wavefront searches
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 16385, 92681, 92682])
def test_fp32_run_sort(ctx, n):
    # points on a coarse lattice, so that many keys are equal: ties go by index in both forms
    rng = np.random.default_rng(n)
    pos = rng.integers(0, 6, size=(n, 3)).astype(np.float64)
    mass = rng.uniform(0.5, 1.0, size=n)
    fpos = rng.normal(size=(77, 3))
    got = ctx.direct(pos, mass, 0.1, FP32), ctx.direct(pos, mass, 0.1, FP32, force_pos=fpos)
    ctx.set_tuning(_native.TUNE_SORT_DIRECT, -1)
    try:
        want = ctx.direct(pos, mass, 0.1, FP32), ctx.direct(pos, mass, 0.1, FP32, force_pos=fpos)
    finally:
        ctx.set_tuning(_native.TUNE_SORT_DIRECT, 0)
    for g, w in zip(got, want):
        assert_bitwise(g, w, "n=%d" % n)


@pytest.mark.parametrize("ipt", [1, 2, 4])  # runs of 256, 512 and 1024 places
def test_fp32_run_sort_of_segments(ctx, ipt):
    sims = []
    for k, n in enumerate([1, 255, 256, 257, 513, 1024, 1025, 5000]):
        ic = workloads.plummer(n, seed=k) if n > 1 else {"pos": np.ones((1, 3)),
                                                         "vel": np.zeros((1, 3)),
                                                         "mass": np.ones(1)}
        ic["eps"], ic["dt"] = 1e-5, 1e-4
        sims.append(ic)

    def run(form):
        ctx.set_tuning(_native.TUNE_SORT_DIRECT, form)
        try:
            ens = _native.Ensemble(ctx, sims, ipt=ipt)
            ens.run(3)
            state = [np.concatenate(a) for a in ens.state()]
            ens.close()
            return state
        finally:
            ctx.set_tuning(_native.TUNE_SORT_DIRECT, 0)

    for k, (got, want) in enumerate(zip(run(0), run(-1))):
        assert_bitwise(got, want, "array %d" % k)


# either side of every change of kernel shape (f64_shape in gh_direct.hip)
@pytest.mark.parametrize("nf", [1, 256, 257, 768, 769, 1024, 1025, 2048, 2049, 3072, 3073, 4096,
                                4097, 6500, 6501, 8192, 8193, 16384, 16385, 24576, 24577])
def test_fp64_direct_shape_edges_bitwise(ctx, oracle, nf):
    rng = np.random.default_rng(nf)
    fpos = rng.standard_cauchy(size=(nf, 3))
    # source counts around the chunks of 128 and 256 and the turns of 16 and 32
    for n in (1, 15, 17, 33, 127, 129, 257):
        pos = rng.standard_cauchy(size=(n, 3))
        pos[: min(n, nf) // 2] = fpos[: min(n, nf) // 2]  # coincident pairs
        mass = rng.uniform(0.1, 3.0, size=n)
        for eps in (0.0, 1e-3):
            assert_bitwise(ctx.direct(pos, mass, eps, FP64, force_pos=fpos),
                           oracle.direct_position(pos, mass, fpos, eps), "%d sources" % n)


@pytest.mark.parametrize("n", [2049, 6501, 8193, 16385, 24577, 33000])
def test_fp64_direct_self_shape_edges_bitwise(ctx, oracle, n):
    rng = np.random.default_rng(n)
    pos = rng.standard_cauchy(size=(n, 3))
    mass = rng.uniform(0.1, 3.0, size=n)
    # with eps > 0 a particle's own term is +-0 and leaves its sum as it is
    some = np.unique(np.concatenate([[0, 31, 32, 63, 64, n - 2, n - 1],
                                     rng.integers(0, n, size=300)]))
    assert_bitwise(ctx.direct(pos, mass, 1e-3, FP64)[some],
                   oracle.direct_position(pos, mass, pos[some], 1e-3))


@pytest.mark.parametrize("nf", [5, 900, 7000, 20000])
def test_fp64_direct_operand_range_bitwise(ctx, oracle, nf):
    """Squared separations below, inside and above the pair factor's range (2^-500 to 2^501),
    zero and overflowing ones among them, mixed in the lanes of a wavefront."""
    rng = np.random.default_rng(nf)
    n = 150
    scale = 10.0 ** rng.choice([-170.0, -76.0, -75.0, -3.0, 0.0, 75.0, 76.0, 150.0, 160.0],
                               size=n)
    pos = rng.normal(size=(n, 3)) * scale[:, None]
    mass = rng.uniform(0.1, 3.0, size=n)
    fpos = rng.normal(size=(nf, 3)) * 10.0 ** rng.choice([-170.0, -3.0, 76.0], size=nf)[:, None]
    fpos[::7] = pos[rng.integers(0, n, size=len(fpos[::7]))]
    for eps in (0.0, 1e-3):
        with np.errstate(all="ignore"):
            want = oracle.direct_position(pos, mass, fpos, eps)
        got = ctx.direct(pos, mass, eps, FP64, force_pos=fpos)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        assert_bitwise(got[ok], want[ok], "eps=%g" % eps)


@pytest.mark.parametrize("n", [131071, 131072, 131072 + 300, 140000])
def test_fp32_direct_block_masses(ctx, n):
    """Either side of the size from which blocks of one mass take it out of their pairs'
    factors, with blocks of one mass, of mixed masses and a padded one: as accurate
    against FP64 as the general form (the direct sum's FP32 tolerance)."""
    ic = workloads.plummer(n, seed=n % 1000)
    rng = np.random.default_rng(n)
    mass = ic["mass"].copy()
    mass[ic["pos"][:, 0] > 2e-3] *= 3.0          # a region of another mass
    odd = rng.integers(0, n, size=20)
    mass[odd] *= rng.uniform(0.5, 2.0, size=20)  # and single particles of their own
    got = ctx.direct(ic["pos"], mass, 2e-5, FP32)
    some = np.unique(np.concatenate([odd, rng.integers(0, n, size=2000)]))
    want = ctx.direct(ic["pos"], mass, 2e-5, FP64)[some]
    e = rel_err(got[some], want)
    assert np.median(e) <= 1e-6 and np.percentile(e, 99) <= 1e-4, (np.median(e), e.max())


# a last block with a few particles, a quarter, and all but one; banded too
@pytest.mark.parametrize("ipt,n", [(1, 257), (1, 321), (2, 1025), (2, 1535), (4, 1025), (4, 1281),
                                   (4, 4095)])
def test_fp32_pair_once_leaves_padding_out(ctx, ipt, n):
    ic = workloads.plummer(n, b=1e-3, mass=1e6, seed=n)
    ref = ctx.direct(ic["pos"], ic["mass"], 1e-4, FP64)
    ctx.set_tuning(_native.TUNE_DIRECT_SELF, ipt)
    try:
        got = ctx.direct(ic["pos"], ic["mass"], 1e-4, FP32)
        ctx.set_tuning(_native.TUNE_SYM_BAND, 1)
        band = ctx.direct(ic["pos"], ic["mass"], 1e-4, FP32)
    finally:
        ctx.set_tuning(_native.TUNE_SYM_BAND, 0)
        ctx.set_tuning(_native.TUNE_DIRECT_SELF, 0)
    for e in (rel_err(got, ref), rel_err(band, ref)):
        assert np.median(e) <= FP32_MEDIAN and np.percentile(e, 99) <= FP32_P99


# around one round of 16384 targets, half a round beyond it, two rounds, and the tails' shapes
@pytest.mark.parametrize("n", [16383, 16384, 16385, 16684, 23000, 24576, 24577, 32768, 32769, 34000])
def test_fp64_whole_rounds_apart(ctx, oracle, n):
    """FP64 sums whose last targets have a launch of their own: the bits of one launch for all
    (64 targets per workgroup), and of the oracle at targets away from the sources."""
    ic = workloads.plummer(n, seed=n)
    got = ctx.direct(ic["pos"], ic["mass"], 2e-5, FP64)
    few = workloads.plummer(300, seed=1)
    at = ctx.direct(few["pos"], few["mass"], 2e-5, FP64, force_pos=ic["pos"])
    ctx.set_tuning(_native.TUNE_DIRECT_F64_TPW, 64)
    try:
        want = ctx.direct(ic["pos"], ic["mass"], 2e-5, FP64)
    finally:
        ctx.set_tuning(_native.TUNE_DIRECT_F64_TPW, 0)
    assert_bitwise(got, want, "self field")
    assert_bitwise(at, oracle.direct_position(few["pos"], few["mass"], ic["pos"], 2e-5), "targets")


@pytest.mark.parametrize("n", [2048, 2049, 2304, 2305, 3072, 3073, 4096, 4097, 4608, 4609, 5119,
                               5121, 6500])
def test_fp64_relay_shapes(ctx, oracle, n):
    """Each side of the sizes at which the targets per workgroup change; chunks of 128 sources
    with a remainder of 1."""
    few = workloads.plummer(513, seed=2)
    at = workloads.plummer(n, seed=n)["pos"]
    got = ctx.direct(few["pos"], few["mass"], 2e-5, FP64, force_pos=at)
    assert_bitwise(got, oracle.direct_position(few["pos"], few["mass"], at, 2e-5), "targets")
    ic = workloads.plummer(n, seed=n)
    own = ctx.direct(ic["pos"], ic["mass"], 2e-5, FP64)[-40:]
    assert_bitwise(own, oracle.direct(ic["pos"], ic["mass"], 2e-5)[-40:], "self field")


# the field of few sources: the relay, the ring and one target per lane meet at these counts
@pytest.mark.parametrize("n,nf", [(n, nf) for nf in (2048, 2049, 6500, 16384, 16385)
                                  for n in (1, 3, 16, 17, 64, 65)] +
                         [(n, 70001) for n in (1, 4, 5, 70, 71)] + [(1, 262144), (262, 262145)])
def test_fp64_field_of_few_sources_bitwise(ctx, oracle, n, nf):
    rng = np.random.default_rng(nf + n)
    fpos = rng.standard_cauchy(size=(nf, 3))
    pos = rng.standard_cauchy(size=(n, 3))
    pos[:n // 2] = fpos[nf - n // 2:] if n > 1 else pos[:0]  # coincident pairs
    mass = rng.uniform(0.1, 3.0, size=n)
    for eps in (0.0, 1e-3):
        assert_bitwise(ctx.direct(pos, mass, eps, FP64, force_pos=fpos),
                       oracle.direct_position(pos, mass, fpos, eps), "eps=%g" % eps)


# one run per simulation, and parts of 1024 keys for 1, 4 and 16 wavefronts to search
@pytest.mark.parametrize("ipt", [1, 2, 4])
@pytest.mark.parametrize("most", [2, 256, 257, 1024, 1025, 4096, 4097])
def test_fp32_run_sort_by_largest_segment(ctx, ipt, most):
    rng = np.random.default_rng(most)
    sims = []
    for n in (1, most // 2 + 1, most, min(most, 100)):
        # a coarse lattice, where many keys are equal, far from FP32 overflow when points coincide
        sims.append({"pos": rng.integers(0, 9, size=(n, 3)).astype(np.float64),
                     "vel": rng.normal(size=(n, 3)), "mass": rng.uniform(0.5, 1.0, size=n),
                     "eps": 0.1, "dt": 1e-4})

    def run(form):
        ctx.set_tuning(_native.TUNE_SORT_DIRECT, form)
        try:
            ens = _native.Ensemble(ctx, sims, ipt=ipt)
            ens.run(3)
            state = [np.concatenate(a) for a in ens.state()]
            ens.close()
            return state + [ctx.direct(s["pos"], s["mass"], 0.1, FP32) for s in sims]
        finally:
            ctx.set_tuning(_native.TUNE_SORT_DIRECT, 0)

    for k, (got, want) in enumerate(zip(run(0), run(-1))):
        assert_bitwise(got, want, "array %d" % k)
