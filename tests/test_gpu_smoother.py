"""The multigrid smoothers and fused level passes on the GPU: the one-launch 4-colour sweep
(k_mg_gs4) against the per-colour launches (bit for bit) and against the
oracle's multicolour Gauss-Seidel (FP64, within FP32 rounding); the
temporally blocked damped Jacobi against single sweeps (bit for bit)."""
import numpy as np
import pytest

import baorec_hip as bh
import baorec_oracle as orc

pytestmark = pytest.mark.gpu

F32 = np.float32


def recon(shape, los, ctx):
    nz, ny, nx = shape
    return bh.MultigridRecon(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=[4.0 * nx, 4.0 * ny, 4.0 * nz],
                             box_min=[200.0, -300.0, 500.0], los=los, ctx=ctx)


def fields(shape, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(shape).astype(F32), rng.standard_normal(shape).astype(F32)


@pytest.mark.parametrize("shape,los,sweeps", [
    ((8, 16, 64), None, 1),
    ((24, 32, 64), [0.0, 0.0, 1.0], 2),
    ((40, 48, 192), None, 3),
    ((256, 256, 256), None, 2),
    ((512, 512, 512), None, 1),
])
def test_fused_sweep_bitwise_per_colour(ctx, shape, los, sweeps):
    """Shapes: one workgroup column, halos wrapping onto the tile itself
    (64 x 16), non-cubic sides, and the solver's 256^3 and 512^3 levels."""
    v, f = fields(shape, sum(shape))
    rec = recon(shape, los, ctx)
    a = bh.gauss_seidel_(v.copy(), f, rec, sweeps=sweeps, fused=True)
    b = bh.gauss_seidel_(v.copy(), f, rec, sweeps=sweeps, fused=False)
    assert np.all(np.isfinite(a))
    np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("los", [None, [0.3, -0.4, 0.866]])
def test_fused_sweep_matches_oracle(ctx, los):
    shape = (32, 32, 128)
    v, f = fields(shape, 5)
    rec = recon(shape, los, ctx)
    got = bh.gauss_seidel_(v.copy(), f, rec, sweeps=2, fused=True)
    exp = orc.mg_gauss_seidel(v.astype(np.float64), f.astype(np.float64), rec.box_size, rec.box_min, rec.beta,
                              los=los, sweeps=2)
    err = float(np.linalg.norm(got - exp) / np.linalg.norm(exp))
    print(f"los {los}: rel L2 vs FP64 oracle {err:.2e}, max abs {np.max(np.abs(got - exp)):.2e}")
    assert err < 2e-6


def test_fused_sweep_rejects_unsupported_shape(ctx):
    shape = (8, 16, 48)   # x side not a multiple of 64
    v, f = fields(shape, 1)
    with pytest.raises(bh.BaorecError):
        bh.gauss_seidel_(v, f, recon(shape, None, ctx), fused=True)
    bh.gauss_seidel_(v, f, recon(shape, None, ctx), fused=False)


# One sweep per call is a z-marching launch of its own on these grids: this test
# holds the two-sweep launches against the one-sweep ones, which share their
# arithmetic (launches are of two sweeps and one, not of three and two as the
# docstring has it).  The comparison with an independent sweep is
# test_zmarching_jacobi_error_against_fp64's.
@pytest.mark.parametrize("shape,los,sweeps", [
    ((128, 128, 128), None, 5),
    ((128, 128, 128), [0.0, 0.0, 1.0], 3),
    ((32, 256, 256), None, 4),
    ((64, 128, 256), [0.6, 0.0, 0.8], 2),
])
def test_blocked_jacobi_bitwise_single_sweeps(ctx, shape, los, sweeps):
    """jacobi! with 2-5 sweeps on grids of >= 128^3 cells runs 3 or 2 sweeps
    per launch (temporal blocking); one sweep per call runs the plain
    kernel.  Both give the same bits."""
    v, f = fields(shape, 7 + sweeps)
    rec = recon(shape, los, ctx)
    rec.jacobi_niterations = sweeps
    got = bh.jacobi_(v.copy(), f, rec)
    rec.jacobi_niterations = 1
    exp = v.copy()
    for _ in range(sweeps):
        bh.jacobi_(exp, f, rec)
    assert np.all(np.isfinite(got))
    np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("shape,los,sweeps", [
    ((128, 128, 128), None, 1),
    ((8, 16, 16384), None, 2),
    ((2048, 16, 64), [0.3, -0.4, 0.866], 2),
    ((72, 208, 192), None, 5),
])
def test_zmarching_jacobi_matches_oracle(ctx, shape, los, sweeps):
    """The z-marching Jacobi launches (one and two sweeps) on grids whose
    tiles' halos wrap onto themselves in y or z, odd numbers of tiles
    included, against the FP32 oracle's sweeps (jacobi!, src/multigrid.jl:
    193-210): the same sums, their products fused, so at most the rounding
    of one update (a few 1e-7 of the largest value) per sweep apart."""
    v, f = fields(shape, 11 + sweeps)
    rec = recon(shape, los, ctx)
    rec.jacobi_niterations = sweeps
    o = orc.MultigridRecon(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=rec.box_size, box_min=rec.box_min,
                           los=los)
    got = bh.jacobi_(v.copy(), f, rec)
    exp = orc.mg_jacobi(v.copy(), f, o.box_size, o.box_min, o.beta, 0.4, sweeps, los=o.los)
    err = float(np.max(np.abs(got - exp)) / np.abs(exp).max())
    print(f"{shape} los {los} x{sweeps}: max |diff| / max |v| {err:.1e}")
    assert err < 5e-7 * sweeps


@pytest.mark.parametrize("sweeps", [1, 2])
def test_zmarching_jacobi_keeps_infinities(ctx, sweeps):
    """A cell of f at +-infinity or NaN gives the z-marching launches the
    infinities and NaN that the oracle's division gives, at the same cells."""
    shape = (128, 128, 128)
    v, f = fields(shape, 17)
    for i, bad in enumerate((np.inf, -np.inf, np.nan)):
        f.flat[(1 + i) * 500001] = bad
    rec = recon(shape, None, ctx)
    rec.jacobi_niterations = sweeps
    o = orc.MultigridRecon(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=rec.box_size, box_min=rec.box_min,
                           los=None)
    got = bh.jacobi_(v.copy(), f, rec)
    with np.errstate(invalid="ignore"):
        exp = orc.mg_jacobi(v.copy(), f, o.box_size, o.box_min, o.beta, 0.4, sweeps, los=o.los)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(got == np.inf, exp == np.inf)
    np.testing.assert_array_equal(got == -np.inf, exp == -np.inf)


@pytest.mark.parametrize("shape,los", [((128, 128, 128), None), ((64, 64, 512), [0.0, 0.0, 1.0]),
                                       ((32, 256, 256), [0.6, 0.0, 0.8])])
def test_zmarching_residual_and_prolongation_match_oracle(ctx, shape, los):
    """On grids of >= 128^3 cells the FP32 residual runs as a z-marching
    pass and the prolongation two cells per thread; both keep the reference's
    FP32 operation order (residual!, prolong!: src/multigrid.jl:378-395,
    398-518)."""
    v, f = fields(shape, 3)
    rec = recon(shape, los, ctx)
    o = orc.MultigridRecon(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=rec.box_size, box_min=rec.box_min,
                           los=los)
    r = np.zeros_like(v)
    bh.residual_(r, v, f, rec)
    exp = orc.mg_residual(v, f, o.box_size, o.box_min, o.beta, los=o.los)
    print("residual max |diff| / max |r|:", np.max(np.abs(r - exp)) / np.abs(exp).max())
    assert np.max(np.abs(r - exp)) < 1e-6 * np.abs(exp).max()
    c = v[::2, ::2, ::2].copy()
    fine = np.zeros(shape, F32)
    bh.prolong_(fine, c, add=False, ctx=ctx)
    np.testing.assert_array_equal(fine, orc.mg_prolong(c))
    fine2 = v.copy()
    bh.prolong_(fine2, c, add=True, ctx=ctx)
    np.testing.assert_allclose(fine2, v + orc.mg_prolong(c), rtol=0, atol=1e-6)


@pytest.mark.parametrize("shape,los", [
    ((2, 16, 64), None),
    ((24, 32, 64), [0.0, 0.0, 1.0]),
    ((40, 48, 192), None),
    ((128, 128, 128), None),
    ((64, 64, 512), [0.6, 0.0, 0.8]),
    ((512, 512, 512), None),
])
def test_fused_residual_restriction_bitwise(ctx, shape, los):
    """The V-cycle's step down, reduce!(residual!(v, f)), as one pass: the
    same bits as the two kernels, on one-plane-pair grids, halos wrapping
    onto the tile itself, non-cubic sides and the solver's 128^3 and 512^3
    levels."""
    v, f = fields(shape, 11 + shape[0])
    rec = recon(shape, los, ctx)
    half = tuple(s // 2 for s in shape)
    a = bh.residual_restrict_(np.full(half, np.nan, F32), v, f, rec, fused=True)
    b = bh.residual_restrict_(np.full(half, np.nan, F32), v, f, rec, fused=False)
    assert np.all(np.isfinite(a))
    np.testing.assert_array_equal(a, b)
    if shape[0] * shape[1] * shape[2] <= 64 * 64 * 512:
        o = orc.MultigridRecon(bias=2.0, f=0.8, smoothing_radius=15.0, box_size=rec.box_size,
                               box_min=rec.box_min, los=los)
        exp = orc.mg_reduce(orc.mg_residual(v, f, o.box_size, o.box_min, o.beta, los=o.los))
        assert np.max(np.abs(a - exp)) < 1e-6 * np.abs(exp).max()


def test_fused_residual_restriction_rejects_unsupported_shape(ctx):
    shape = (8, 16, 96)   # x side not a multiple of 64
    v, f = fields(shape, 2)
    c = np.zeros((4, 8, 48), F32)
    with pytest.raises(bh.BaorecError):
        bh.residual_restrict_(c, v, f, recon(shape, None, ctx), fused=True)
    bh.residual_restrict_(c, v, f, recon(shape, None, ctx), fused=False)


@pytest.mark.parametrize("shape", [(16, 16, 16), (8, 16, 32), (64, 32, 16), (8, 8, 64), (24, 24, 24), (40, 64, 96)])
@pytest.mark.parametrize("los", [None, [0.3, -0.4, 0.866]])
@pytest.mark.parametrize("fp64_coarse_max", [0, 8, 16])
def test_small_levels_rbgs_solves(ctx, shape, los, fp64_coarse_max):
    """RBGS solves whose levels run in one workgroup's LDS (power-of-two
    sides, at most 4096 cells, either precision), by 8^3 tiles (sides
    multiples of 8) or by the general kernels (24^3 halves to odd sides):
    the solution satisfies the FP64 oracle's operator to the tolerance, up
    to the solve's reported shift of f."""
    f = np.random.default_rng(sum(shape)).standard_normal(shape).astype(F32)
    f -= f.mean()
    rec = recon(shape, los, ctx)
    rec.schedule, rec.tolerance, rec.fp64_coarse_max, rec.rb_sweeps = "rbgs", 1e-5, fp64_coarse_max, 2
    phi = bh.fmg(f, rec)
    assert rec.final_residual <= 1e-5 and rec.vcycles_done <= 30
    r = orc.mg_residual(phi.astype(np.float64), f.astype(np.float64) - rec.rhs_shift, rec.box_size, rec.box_min,
                        rec.beta, los=los)
    rel = float(np.linalg.norm(r) / np.linalg.norm(f))
    print(f"{shape} los {los} fp64 <= {fp64_coarse_max}: {rec.vcycles_done} V-cycles, residual {rel:.1e}")
    assert rel < 3e-5   # the tolerance, and phi's FP32 rounding (|A| |phi| 2^-24 / |f|, about 1e-6)


@pytest.mark.parametrize("shape", [(16, 16, 16), (8, 16, 32), (8, 8, 8), (32, 32, 32)])
@pytest.mark.parametrize("sweeps", [5, 2])
def test_small_levels_fmg_matches_oracle(ctx, shape, sweeps):
    """The reference's schedule on levels in one workgroup's LDS against the
    FP32 oracle (odd and even sweeps per smoothing: the result in either
    buffer): the same operations in the same order, so the schedules stay
    within the growth of single roundings, 2e-5 of the solution's norm."""
    f = np.random.default_rng(7).standard_normal(shape).astype(F32)
    f -= f.mean()
    rec = recon(shape, None, ctx)
    rec.jacobi_niterations, rec.vcycle_niterations = sweeps, 3
    got = bh.fmg(f, rec)
    exp = orc.fmg(f, rec.box_size, rec.box_min, rec.beta, 0.4, sweeps, 3)
    err = float(np.linalg.norm(got - exp) / np.linalg.norm(exp))
    print(f"{shape} x{sweeps}: {err:.1e}")
    assert err < 2e-5
    v = f.copy()
    bh.vcycle_(v, f, rec)
    exp = orc.mg_vcycle(f.copy(), f, rec.box_size, rec.box_min, rec.beta, 0.4, sweeps)
    assert np.linalg.norm(v - exp) < 2e-5 * np.linalg.norm(exp)


@pytest.mark.parametrize("los", [None, [0.3, -0.4, 0.866]])
@pytest.mark.parametrize("sweeps", [1, 2])
def test_zmarching_jacobi_overflows_as_the_oracle(ctx, los, sweeps):
    """Quotients of finite numbers around the largest float: infinite where
    the oracle's division is, finite below (also where the quotient by half
    the diagonal overflows)."""
    shape = (128, 128, 128)
    v, f = fields(shape, 19)
    for i, big in enumerate((3e38, -3e38, 1e38, -1e38, 2e37)):
        f.flat[(1 + i) * 300007] = big
    rec = recon(shape, los, ctx)
    rec.jacobi_niterations = sweeps
    got = bh.jacobi_(v.copy(), f, rec)
    with np.errstate(invalid="ignore", over="ignore"):
        exp = orc.mg_jacobi(v.copy(), f, rec.box_size, rec.box_min, rec.beta, 0.4, sweeps, los=los)
    assert np.isinf(exp).sum() >= 2 and np.isfinite(exp.flat[3 * 300007])
    np.testing.assert_array_equal(np.isnan(got), np.isnan(exp))
    np.testing.assert_array_equal(got == np.inf, exp == np.inf)
    np.testing.assert_array_equal(got == -np.inf, exp == -np.inf)
    on = np.isfinite(exp) & (np.abs(exp) > 1e30)
    assert on.sum() >= 3
    np.testing.assert_allclose(got[on], exp[on], rtol=5e-7 * sweeps)


@pytest.mark.parametrize("sweeps", [1, 2])
@pytest.mark.parametrize("growth,cell", [(0.0, 4.0), (0.8, 3.1 * 2.0 ** -64), (0.8, 2.0 ** 55), (8e6, 4.0)])
def test_large_grid_jacobi_over_coefficients(ctx, growth, cell, sweeps):
    """The sweeps of grids of 128^3 and more without redshift-space distortions
    (beta = 0), with cells so small that the operator's diagonal passes 2^126,
    with very large ones and with a very large beta."""
    shape = (128, 128, 128)
    v, f = (a * F32(0.01) for a in fields(shape, 20))
    f *= F32(1.0 / cell) * F32(1.0 / cell)
    rec = bh.MultigridRecon(bias=2.0, f=growth, smoothing_radius=15.0, box_size=[128 * cell] * 3,
                            box_min=[50 * cell, -75 * cell, 125 * cell], los=None, ctx=ctx)
    rec.jacobi_niterations = sweeps
    got = bh.jacobi_(v.copy(), f, rec)
    exp = orc.mg_jacobi(v.copy(), f, rec.box_size, rec.box_min, rec.beta, 0.4, sweeps, los=None)
    assert np.all(np.isfinite(exp))
    assert np.max(np.abs(got - exp)) < 5e-7 * sweeps * np.abs(exp).max()


def fp64_sweep(v, f, box_size, box_min, beta, omega, los):
    """One damped Jacobi sweep (jacobi!, src/multigrid.jl:14-135) in FP64 from
    the FP32 cell centres, and a bound of an FP32 sweep's rounding per cell in
    units of 2^-24: the summed magnitude of the update's terms times the most
    roundings that one of them passes (6 in a coefficient, 2 in a difference,
    7 in the sum), 8 of the diagonal, 2 of the quotient and its weight, 3 of
    the part that is kept."""
    h = [float(F32(F32(L) / F32(n))) for L, n in zip(box_size, v.shape[::-1])]
    if los is None:
        p = [x / F32(c) for x, c in zip(orc.x_vec(v.shape[::-1], box_size, box_min), h)]
        p = [p[0][None, None, :], p[1][None, :, None], p[2][:, None, None]]
    else:
        p = [F32(w) / F32(c) for w, c in zip(los, h)]
    px, py, pz = (np.asarray(a, np.float64) for a in p)

    def at(dx, dy, dz):
        return np.roll(v, (-dz, -dy, -dx), (0, 1, 2))
    g = beta / ((h[0] * px) ** 2 + (h[1] * py) ** 2 + (h[2] * pz) ** 2)
    total, size, diag = f.copy(), np.abs(f), 0.0
    for a, (e, q) in enumerate(zip(np.eye(3, dtype=int), (px, py, pz))):
        w, up, dn = 1 / h[a] ** 2 + g * q * q, at(*e), at(*-e)
        total += w * (up + dn)
        size += w * (np.abs(up) + np.abs(dn))
        diag = diag + w
        if los is None:
            total += g * q * (up - dn)
            size += np.abs(g * q) * (np.abs(up) + np.abs(dn))
    for i, j, w in ((0, 1, px * py), (0, 2, px * pz), (1, 2, py * pz)):
        e, k = np.eye(3, dtype=int)[i], np.eye(3, dtype=int)[j]
        t = [at(*(e + k)), at(*(-e - k)), at(*(k - e)), at(*(e - k))]
        total += g / 2 * w * (t[0] + t[1] - t[2] - t[3])
        size += np.abs(g / 2 * w) * sum(np.abs(s) for s in t)
    q = total / (2 * diag)
    return (1 - omega) * v + omega * q, omega * 25 * size / (2 * diag) + 3 * np.abs(v)


@pytest.mark.parametrize("shape,los", [((128, 128, 128), None), ((64, 128, 256), None),
                                       ((128, 128, 128), [0.3, -0.4, 0.866])])
@pytest.mark.parametrize("sweeps", [1, 2])
def test_zmarching_jacobi_error_against_fp64(ctx, shape, los, sweeps):
    """What the one- and two-sweep launches' fused sums and corrected quotients
    cost in accuracy: nothing against the reference's order of operations in
    FP32 (the oracle's sweeps on the same fields).  Their rms error against
    FP64 sweeps is no larger (2 % for the scatter of the largest roundings),
    and after one sweep every cell is within its rounding bound."""
    v, f = fields(shape, 23)
    v *= F32(50.0)
    rec = recon(shape, los, ctx)
    rec.jacobi_niterations = sweeps
    beta, omega = float(F32(rec.beta)), float(F32(0.4))
    exact = v.astype(np.float64)
    for _ in range(sweeps):
        exact, bound = fp64_sweep(exact, f.astype(np.float64), rec.box_size, rec.box_min, beta, omega, los)
    got = bh.jacobi_(v.copy(), f, rec) - exact
    ref = orc.mg_jacobi(v.copy(), f, rec.box_size, rec.box_min, rec.beta, 0.4, sweeps, los=los) - exact
    rms = [float(np.sqrt(np.mean(e * e) / np.mean(exact * exact))) for e in (got, ref)]
    worst = float(np.max(np.abs(got) / bound)) * 2.0 ** 24
    print(f"{shape} los {los} x{sweeps}: rms error {rms[0]:.2e}, the reference's order {rms[1]:.2e}, "
          f"largest / bound {worst:.2f}")
    assert rms[0] <= 1.02 * rms[1]
    if sweeps == 1:
        assert worst <= 1.0


@pytest.mark.parametrize("shape,sweeps", [((120, 256, 256), 3), ((128, 256, 256), 2), ((280, 256, 320), 3)])
def test_zmarching_jacobi_over_launch_sizes(ctx, shape, sweeps):
    """Several sweeps in one call (by two or by one per launch, as the grid's
    size has it: just below and at 2^23 cells, and above the size of the
    Infinity Cache) and one call per sweep: the same bits; one against the
    oracle as above."""
    v, f = fields(shape, 29)
    rec = recon(shape, None, ctx)
    rec.jacobi_niterations = sweeps
    got = bh.jacobi_(v.copy(), f, rec)
    rec.jacobi_niterations = 1
    exp = bh.jacobi_(v.copy(), f, rec)
    ref = orc.mg_jacobi(v.copy(), f, rec.box_size, rec.box_min, rec.beta, 0.4, 1)
    assert np.max(np.abs(exp - ref)) < 5e-7 * np.abs(ref).max()
    for _ in range(sweeps - 1):
        bh.jacobi_(exp, f, rec)
    np.testing.assert_array_equal(got, exp)
