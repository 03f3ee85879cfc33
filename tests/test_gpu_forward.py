"""GPU parity of the forward kernels against the oracle (same seeded inputs).

Bars: FP64 paths <= 1e-12 relative (rel_max = max|u-u_ref| / max|u_ref|)
against the C restatement of the reference loop; FP32 path <= 1e-5 relative
(rel_max and rel_rms).  Inputs include the reference's own configurations at
oracle-friendly sizes, large coordinates (phases ~3e5 rad), the guarded
huge-phase path, and ragged / empty sizes.
"""

import copy
import sys

import numpy as np
import pytest
import torch

import oracle
from gstools_amd import (Exponential, Gaussian, IncomprRandMeth, RandMeth, summate, summate_device,
                         summate_grid_device, summate_incompr, summate_incompr_device)
from gstools_amd.geometry import generate_grid

pytestmark = pytest.mark.gpu

FP64_TOL = 1e-12
FP32_TOL = 1e-5


def _case(d, n, p, seed, kscale=1.0, xscale=10.0):
    rs = np.random.RandomState(seed)
    return (rs.normal(size=(d, n)) * kscale, rs.normal(size=n), rs.normal(size=n),
            rs.uniform(-xscale, xscale, size=(d, p)))


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("d,n,p,kscale,xscale", [
    (1, 100, 1000, 1.0, 10.0),
    (2, 1000, 5003, 0.5, 100.0),
    (3, 1024, 4099, 26.0 / 3, 1e4),   # phases up to ~3e5 rad, like the 3D Exponential config
    (3, 257, 1, 1.0, 5.0),            # ragged mode chunk, single point
])
def test_fp64_matches_oracle(d, n, p, kscale, xscale):
    _say(f"fp64 d={d} N={n} P={p}")
    cov, z1, z2, pos = _case(d, n, p, 1000 + d, kscale, xscale)
    ref = oracle.summate_c(cov, z1, z2, pos)
    got = summate(cov, z1, z2, pos)
    assert got.dtype == np.float64 and got.shape == (p,)
    rel_max, rel_rms = oracle.rel_errors(got, ref)
    assert rel_max <= FP64_TOL, (rel_max, rel_rms)


def test_fp64_huge_phase_guarded_path():
    _say("fp64 huge phases")
    cov, z1, z2, pos = _case(2, 300, 2000, 7, 1.0, 1.0)
    pos[:, :1000] *= 3e14  # phases beyond 2^46: the guarded library-sincos path
    ref = oracle.summate_c(cov, z1, z2, pos)
    got = summate(cov, z1, z2, pos)
    assert oracle.rel_errors(got, ref)[0] <= FP64_TOL


def test_empty_and_zero_modes():
    _say("empty sizes")
    cov, z1, z2, pos = _case(2, 0, 777, 3)
    assert np.array_equal(summate(cov, z1, z2, pos), np.zeros(777))
    cov, z1, z2, pos = _case(3, 5, 0, 3)
    assert summate(cov, z1, z2, pos).shape == (0,)
    cov, z1, z2, pos = _case(3, 64, 100, 4)
    cov[:] = 0.0
    assert np.allclose(summate(cov, z1, z2, pos), np.sum(z1), rtol=1e-13, atol=0)


@pytest.mark.parametrize("d", [1, 2, 3])
def test_fp32_within_1e5(d):
    _say(f"fp32 d={d}")
    cov, z1, z2, pos = _case(d, 1024, 20000, 40 + d, 26.0 / 3 if d == 3 else 1.0, 1e4 if d == 3 else 300.0)
    ref = oracle.summate_c(cov, z1, z2, pos)
    got = summate_device(cov, z1, z2, pos, precision="fp32").cpu().numpy()
    rel_max, rel_rms = oracle.rel_errors(got, ref)
    assert rel_max <= FP32_TOL and rel_rms <= FP32_TOL, (rel_max, rel_rms)


@pytest.mark.parametrize("incompr", [False, True])
def test_fp32_phase_reductions_both_regimes(incompr):
    """The FP32 kernels reduce the phase by magic addition for the modes whose
    |k/2pi|_1 times the largest |x|_inf of the point's 2048-point segment stays
    within 2^18 revolutions and by fract-and-convert for the others.  A
    segment of points at |x| ~ 3e6 (phases ~1e6 revolutions) between
    segments at |x| ~ 100 puts both in one launch, over 5 mode chunks; both
    must meet the FP32 bar, and the small segments give the same sums as a
    launch without the far points."""
    _say(f"fp32 magic and fract reductions incompr={incompr}")
    cov, z1, z2, pos = _case(3, 1100, 8192, 91, 1.0, 100.0)
    big = pos.copy()
    big[:, 2048:4096] *= 3e4  # the second 2048-point segment: its large modes take the fract form
    fn = summate_incompr_device if incompr else summate_device
    ref_fn = oracle.summate_incompr_c if incompr else oracle.summate_c
    bound = np.abs(cov).sum(axis=0).max() / (2 * np.pi) * np.abs(big[:, 2048:4096]).max()
    assert bound > 2.0**18 and np.abs(cov).sum(axis=0).max() / (2 * np.pi) * 100.0 < 2.0**18
    got = fn(cov, z1, z2, big, precision="fp32").cpu().numpy()
    ref = ref_fn(cov, z1, z2, big)
    for sl in (np.s_[..., 2048:4096], np.s_[..., :2048]):
        rel_max, rel_rms = oracle.rel_errors(got[sl], ref[sl])
        assert rel_max <= FP32_TOL and rel_rms <= FP32_TOL, (sl, rel_max, rel_rms)
    small = fn(cov, z1, z2, pos, precision="fp32").cpu().numpy()
    assert np.array_equal(small[..., :2048], got[..., :2048])
    assert np.array_equal(small[..., 4096:], got[..., 4096:])


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_non_finite_coordinates_propagate(precision):
    """A NaN or infinite coordinate gives NaN at its point, as the reference's
    loop does (cos of NaN or inf), in both precisions; in FP32 it makes its
    2048-point segment's bound infinite, so the segment's other points take
    the fract-form reduction and still meet the FP32 bar."""
    _say(f"non-finite coordinates {precision}")
    cov, z1, z2, pos = _case(3, 300, 5000, 17, 1.0, 100.0)
    bad = pos.copy()
    bad[1, 100] = np.nan
    bad[2, 2500] = np.inf
    bad[0, 4999] = -np.inf
    got = summate_device(cov, z1, z2, bad, precision=precision).cpu().numpy().astype(np.float64)
    hit = np.zeros(5000, bool)
    hit[[100, 2500, 4999]] = True
    assert np.all(np.isnan(got[hit]))
    assert np.all(np.isfinite(got[~hit]))
    ref = oracle.summate_c(cov, z1, z2, pos)
    rel_max, rel_rms = oracle.rel_errors(got[~hit], ref[~hit])
    assert rel_max <= (FP32_TOL if precision == "fp32" else FP64_TOL), (rel_max, rel_rms)


@pytest.mark.parametrize("incompr,p_big", [(False, 4_500_000), (True, 2_500_000)])
def test_fp32_full_chip_launch_matches_prefix(incompr, p_big):
    """A launch of millions of points (thousands of blocks, every compute unit
    busy) and a small launch of its first 30001 points agree with each other and
    with the oracle.  N = 1000 leaves a ragged last chunk of 232 modes; 30001 is
    ragged against the 2048- (or 1024-) point block.  Bit for bit because every
    mode here takes the magic-addition reduction in both launches (|k/2pi|_1
    |x|_inf stays far below 2^18 revolutions); the test with both reductions
    covers segments that differ."""
    _say(f"fp32 full-chip launch vs prefix incompr={incompr} P={p_big}")
    cov, z1, z2, pos = _case(3, 1000, p_big, 77, 2.0, 500.0)
    fn = summate_incompr_device if incompr else summate_device
    ref_fn = oracle.summate_incompr_c if incompr else oracle.summate_c
    whole = fn(cov, z1, z2, pos, precision="fp32").cpu().numpy()
    k = 30001
    part = fn(cov, z1, z2, np.ascontiguousarray(pos[:, :k]), precision="fp32").cpu().numpy()
    whole_k = whole[..., :k]
    ref = ref_fn(cov, z1, z2, np.ascontiguousarray(pos[:, :k]))
    for got in (whole_k, part):
        rel_max, rel_rms = oracle.rel_errors(got, ref)
        assert rel_max <= FP32_TOL and rel_rms <= FP32_TOL, (rel_max, rel_rms)
    # a point's sum does not depend on the launch it belongs to
    assert np.array_equal(part, whole_k)


@pytest.mark.parametrize("d", [2, 3])
def test_incompr_matches_oracle(d):
    _say(f"incompr d={d}")
    cov, z1, z2, pos = _case(d, 500, 3001, 60 + d, 2.0, 200.0)
    ref = oracle.summate_incompr_c(cov, z1, z2, pos)
    got = summate_incompr(cov, z1, z2, pos)
    assert got.shape == (d, 3001)
    assert oracle.rel_errors(got, ref)[0] <= FP64_TOL
    got32 = summate_incompr_device(cov, z1, z2, pos, precision="fp32").cpu().numpy()
    rel_max, rel_rms = oracle.rel_errors(got32, ref)
    assert rel_max <= FP32_TOL and rel_rms <= FP32_TOL


def test_config1_gaussian_grid():
    """2D Gaussian, var 1, len 10, N 1000, seed 20170519, 100 x 100 grid."""
    _say("config 1")
    model = Gaussian(dim=2, var=1.0, len_scale=10)
    rm = RandMeth(model, mode_no=1000, seed=20170519)
    axes = [np.arange(100.0), np.arange(100.0)]
    pos = generate_grid(axes)
    ref = oracle.summate_c(rm._cov_sample, rm._z_1, rm._z_2, pos)
    unstruct = summate(rm._cov_sample, rm._z_1, rm._z_2, pos)
    assert oracle.rel_errors(unstruct, ref)[0] <= FP64_TOL
    grid = summate_grid_device(rm._cov_sample, rm._z_1, rm._z_2, axes, "fp64").cpu().numpy()
    # same phases and the same accumulation order: bitwise equal
    assert np.array_equal(grid, unstruct)
    grid32 = summate_grid_device(rm._cov_sample, rm._z_1, rm._z_2, axes, "fp32").cpu().numpy()
    assert oracle.rel_errors(grid32, ref)[0] <= FP32_TOL
    field = rm(pos)
    assert np.allclose(field, np.sqrt(1.0 / 1000) * ref, rtol=0, atol=1e-12)


def test_generator_known_values_on_gpu():
    """``tests/test_randmeth.py:33-46`` through the GPU generator."""
    _say("known values")
    m1 = Gaussian(dim=1, var=1.5, len_scale=3.5)
    m3 = copy.deepcopy(m1)
    m3.dim = 3
    x = np.linspace(0.0, 10.0, 10)
    y = np.linspace(-5.0, 5.0, 10)
    z = np.linspace(-6.0, 8.0, 10)
    f1 = RandMeth(m1, mode_no=100, seed=19031977)((x,))
    assert f1[:2] == pytest.approx([3.19799030, 2.44848295], abs=5e-8)
    f3 = RandMeth(m3, mode_no=100, seed=19031977)((x, y, z))
    assert f3[:2] == pytest.approx([1.3240234883187239, 1.6367244277732766], abs=1e-12)
    g2 = Gaussian(dim=2, var=1.5, len_scale=2.5)
    v = IncomprRandMeth(g2, mode_no=100, seed=19031977)((x, y))
    assert [v[0, 0], v[0, 1], v[1, 1]] == pytest.approx([0.50751115, 1.03291018, -0.22003005], abs=5e-8)
    t = RandMeth(m3, mode_no=100, seed=19031977)(torch.tensor(np.array([x, y, z]), device="cuda"))
    assert isinstance(t, torch.Tensor) and t.is_cuda


def test_config2_sample_fp64_fp32():
    """3D Exponential (var 2, len [50,20,5], angles [.5,.2,.1]), N 1024, MCMC modes."""
    _say("config 2 sample")
    model = Exponential(dim=3, var=2.0, len_scale=[50, 20, 5], angles=[0.5, 0.2, 0.1])
    rm = RandMeth(model, mode_no=1024, seed=20170519)
    pos = np.random.RandomState(19970221).uniform(0, 1000, size=(3, 8192))
    iso = model.isometrize(pos)
    ref = oracle.summate_c(rm._cov_sample, rm._z_1, rm._z_2, iso)
    assert oracle.rel_errors(summate(rm._cov_sample, rm._z_1, rm._z_2, iso), ref)[0] <= FP64_TOL
    got32 = summate_device(rm._cov_sample, rm._z_1, rm._z_2, iso, precision="fp32").cpu().numpy()
    rel_max, rel_rms = oracle.rel_errors(got32, ref)
    _say(f"config 2 fp32 rel_max={rel_max:.3e} rel_rms={rel_rms:.3e}")
    assert rel_max <= FP32_TOL and rel_rms <= FP32_TOL


@pytest.mark.parametrize("incompr", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("d,n", [(2, 64), (3, 200), (2, 1500), (3, 1025)])
def test_split_launches_equal_plain_launch(d, n, precision, incompr):
    """Launches of few points share each point's modes out over a block's waves; their values
    equal those of a launch too large for that, bit for bit, at the edges of the block sizes.
    One far point per 2048-point segment keeps the FP32 phase bound of every prefix the same
    and puts some modes of every group on the other phase reduction."""
    big = 600_001  # plain launch for every n here
    rs = np.random.RandomState(n)
    cov = torch.from_numpy(rs.standard_cauchy(size=(d, n))).cuda()
    z1, z2 = torch.from_numpy(rs.normal(size=(2, n))).cuda()
    pos = torch.from_numpy(rs.uniform(-200.0, 200.0, size=(d, big))).cuda()
    pos[:, ::2048] *= 5e3
    fn = summate_incompr_device if incompr else summate_device
    want = fn(cov, z1, z2, pos, precision).reshape(-1, big)
    assert bool(torch.isfinite(want).all())
    for p in (1, 31, 33, 64, 65, 127, 129, 8192, 8193, 16385, 32769, 65537, 131073):
        got = fn(cov, z1, z2, pos[:, :p].contiguous(), precision).reshape(-1, p)
        assert torch.equal(got, want[:, :p]), (p, precision)


@pytest.mark.parametrize("incompr", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("d", [2, 3])
def test_plain_launches_agree_whatever_their_blocks(d, precision, incompr):
    """The points per thread of a plain launch follow its size; a point's value does not:
    launches of 1.4e5 to 1.1e6 points, which take each of the block shapes, give the bits of
    the first.  One far point per 2048-point segment puts some modes of every group on the
    other phase reduction and keeps the segments' bounds the same."""
    n, big = 300, 1_050_001
    rs = np.random.RandomState(d)
    cov = torch.from_numpy(rs.standard_cauchy(size=(d, n))).cuda()
    z1, z2 = torch.from_numpy(rs.normal(size=(2, n))).cuda()
    pos = torch.from_numpy(rs.uniform(-200.0, 200.0, size=(d, big))).cuda()
    pos[:, ::2048] *= 5e3
    fn = summate_incompr_device if incompr else summate_device
    want = fn(cov, z1, z2, pos, precision).reshape(-1, big)
    assert bool(torch.isfinite(want).all())
    for p in (140_003, 262_145, 393_217, 524_289, 600_000, 700_001, 800_000, 1_048_576):
        got = fn(cov, z1, z2, pos[:, :p].contiguous(), precision).reshape(-1, p)
        assert torch.equal(got, want[:, :p]), (p, precision)


@pytest.mark.parametrize("incompr", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("d,n", [(1, 129), (1, 1500), (2, 129), (3, 191)])
def test_split_launches_that_end_inside_a_group(d, n, precision, incompr):
    """As above for mode counts one past a group and for 1D, with points beyond 2^46 rad in FP64."""
    d = max(d, 2) if incompr else d
    _say(f"split launches d={d} N={n} {precision} incompr={incompr}")
    big = 600_001
    rs = np.random.RandomState(n + d)
    cov = torch.from_numpy(rs.standard_cauchy(size=(d, n))).cuda()
    z1, z2 = torch.from_numpy(rs.normal(size=(2, n))).cuda()
    pos = torch.from_numpy(rs.uniform(-200.0, 200.0, size=(d, big))).cuda()
    pos[:, ::2048] *= 5e3 if precision == "fp32" else 1e12
    fn = summate_incompr_device if incompr else summate_device
    want = fn(cov, z1, z2, pos, precision).reshape(-1, big)
    for p in (1, 31, 33, 64, 65, 127, 129, 8192, 8193, 16385, 32768):
        got = fn(cov, z1, z2, pos[:, :p].contiguous(), precision).reshape(-1, p)
        assert torch.equal(got, want[:, :p]), (p, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("d,n,p", [(1, 300, 600_001), (2, 64, 40_000), (3, 300, 600_001)])
def test_plain_launches_with_huge_and_non_finite_coordinates(d, n, p, precision):
    """Launches too large or of too few modes to be split: phases beyond 2^46 rad (FP64) or 2^18
    revolutions (FP32) take the guarded reductions and agree with the oracle; a NaN or infinite
    coordinate gives NaN at its point and changes no other's value beyond the bars."""
    _say(f"plain launches, odd coordinates d={d} N={n} P={p} {precision}")
    cov, z1, z2, pos = _case(d, n, p, 50 + d, 1.0, 100.0)
    pos[:, 1000:1500] *= 3e12 if precision == "fp64" else 3e4
    pos[0, 777], pos[-1, 2500], pos[0, p - 1] = np.nan, np.inf, -np.inf
    got = summate_device(cov, z1, z2, pos, precision).cpu().numpy().astype(np.float64)
    hit = np.zeros(p, bool)
    hit[[777, 2500, p - 1]] = True
    assert np.all(np.isnan(got[hit])) and np.all(np.isfinite(got[~hit]))
    some = np.flatnonzero(~hit)
    some = np.concatenate([some[:6000], some[-3000:]])
    ref = oracle.summate_c(cov, z1, z2, np.ascontiguousarray(pos[:, some]))
    tol = FP64_TOL if precision == "fp64" else FP32_TOL
    rel_max, rel_rms = oracle.rel_errors(got[some], ref)
    assert rel_max <= tol and rel_rms <= tol, (rel_max, rel_rms)
    few = np.ascontiguousarray(pos[:, 996:1600])  # FP64: the same bits from a launch of few points
    if precision == "fp64":
        part = summate_device(cov, z1, z2, few, precision).cpu().numpy()
        assert np.array_equal(part, got[996:1600])
