"""HMC, the collective variable with its hand-written adjoint, and MetaD-HMC on the
GPU (through the C ABI) against the CPU oracle and the reference's golden vectors."""
import numpy as np
import pytest

from conftest import assert_field_matches, rel_err

pytestmark = pytest.mark.gpu

SMALL = (8, 8, 8, 8)
TINY = (4, 4, 4, 4)
G16 = (16, 16, 16, 16)


def flush(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def la():
    import lettuce_amd
    return lettuce_amd


def smooth(lto, shape, seed=0, n=3):
    return lto.stout(lto.haar(shape, seed), shape, 0.1, n)


def gauge(la, ctx, shape, data=None):
    f = la.GaugeField(ctx, shape)
    if data is not None:
        f.upload(data)
    return f


def matrix(la, ctx, shape, data=None):
    f = la.MatrixField(ctx, shape)
    if data is not None:
        f.upload(data)
    return f


def test_momenta_match_oracle_stream(la, lto, gpu_ctx):
    flush("momenta")
    P = matrix(la, gpu_ctx, SMALL)
    la.RandomMomentum(P, 17, 3)
    ref = lto.random_momentum(SMALL, 17, 3)
    assert rel_err(P.download(), ref) <= 1e-13


def test_force_and_field_updates(la, lto, gpu_ctx):
    flush("force/field update")
    U0 = smooth(lto, SMALL, 1)
    P0 = lto.random_momentum(SMALL, 2, 0)
    U = gauge(la, gpu_ctx, SMALL, U0)
    P = matrix(la, gpu_ctx, SMALL, P0)
    la.UpdateMomenta(U, P, 0.1, 6.0)
    la.UpdateFields(U, P, 0.05)
    Ur, Pr = U0.copy(), P0.copy()
    lto.gauge_force_update(Ur, Pr, SMALL, 0.1, 6.0)
    lto.field_update(Ur, Pr, SMALL, 0.05)
    assert rel_err(P.download(), Pr) <= 1e-13
    assert rel_err(U.download(), Ur) <= 1e-13
    H = la.Hamiltonian(U, P, 6.0)
    assert abs(H - lto.hamiltonian(Ur, Pr, SMALL, 6.0)) <= 1e-12 * abs(H)


@pytest.mark.parametrize("integrator", ["leapfrog", "omf2", "omf4", "leapfrog_slow", "omf2_slow", "omf4_slow"])
def test_integrators_match_oracle(la, lto, gpu_ctx, integrator):
    flush(f"integrate {integrator}")
    U0 = smooth(lto, SMALL, 3)
    P0 = lto.random_momentum(SMALL, 4, 0)
    U = gauge(la, gpu_ctx, SMALL, U0)
    P = matrix(la, gpu_ctx, SMALL, P0)
    la.Integrate(U, P, 6.0, integrator, 0.5, 6)
    Ur, Pr = U0.copy(), P0.copy()
    if integrator == "omf2":
        lto.omf2(Ur, Pr, SMALL, 6.0, 0.5, 6)
    else:   # the schedule-driven oracle with no bias force (schedules pinned to the reference's)
        lto.metad_trajectory(Ur, Pr, SMALL, 6.0, 0.5, 6, 0.12, 1, None, integrator)
    assert rel_err(U.download(), Ur) <= 1e-10
    assert rel_err(P.download(), Pr) <= 1e-10
    # reversibility (hmc_gauge.hpp:585-599): flip momenta, integrate back
    Pm = -P.download()
    P.upload(Pm)
    la.Integrate(U, P, 6.0, integrator, 0.5, 6)
    assert np.max(np.abs(U.download() - U0)) <= 1e-10
    assert np.max(np.abs(-P.download() - P0)) <= 1e-10


def test_omf2_trajectory_golden16(la, lto, golden, gpu_ctx):
    flush("omf2 golden 16^4")
    U0 = lto.stout(lto.haar(G16, 0), G16, 0.1, 3)
    U = gauge(la, gpu_ctx, G16, U0)
    P = matrix(la, gpu_ctx, G16, lto.random_momentum(G16, 5, 0))
    H0 = la.Hamiltonian(U, P, 6.0)
    la.Integrate(U, P, 6.0, "omf2", 1.0, 10)
    H1 = la.Hamiltonian(U, P, 6.0)
    Href = golden["hmc_omf2_smooth_H"]
    assert abs(H0 - Href[0]) <= 1e-12 * abs(Href[0])
    assert abs((H1 - H0) - (Href[1] - Href[0])) <= 1e-7 * max(1.0, abs(Href[1] - Href[0]))
    assert_field_matches(golden, "hmc_omf2_smooth", U.download(), 1e-9)


def test_trajectory_metropolis_and_momentum_stream(la, lto, gpu_ctx):
    flush("hmc trajectory")
    U0 = smooth(lto, SMALL, 5)
    U = gauge(la, gpu_ctx, SMALL, U0)
    Uc = gauge(la, gpu_ctx, SMALL)
    P = matrix(la, gpu_ctx, SMALL)
    U.set_rng(9, 7)
    hmc = la.HMCKernel(U, Uc, P, "omf2", 6.0, 1.0)
    acc = hmc(8, metropolis_step=False)
    assert acc and U.get_rng() == (9, 8)
    # same trajectory on the oracle from the same Philox momenta
    Ur = U0.copy()
    Pr = lto.random_momentum(SMALL, 9, 7)
    H0 = lto.hamiltonian(Ur, Pr, SMALL, 6.0)
    lto.omf2(Ur, Pr, SMALL, 6.0, 1.0, 8)
    dH = lto.hamiltonian(Ur, Pr, SMALL, 6.0) - H0
    assert abs(hmc.delta_H - dH) <= 1e-8 * max(1.0, abs(dH))
    assert rel_err(U.download(), Ur) <= 1e-10
    # rejection restores the field exactly
    before = U.download()
    hmc.trajectory_length = 8.0     # far too long a trajectory: certain rejection
    acc = hmc(4, metropolis_step=True)
    if not acc:
        assert np.array_equal(U.download(), before)


@pytest.mark.parametrize("n_levels", [0, 2, 4])
def test_cv_forward_backward_vs_oracle(la, lto, gpu_ctx, n_levels):
    flush(f"cv levels {n_levels}")
    U0 = smooth(lto, SMALL, 6)
    U = gauge(la, gpu_ctx, SMALL, U0)
    F = matrix(la, gpu_ctx, SMALL)
    cv = la.CollectiveVariable(gpu_ctx, SMALL, n_levels, 0.12)
    Q = cv.forward(U)
    cv.backward(0.7, F)
    Qr, Fr = lto.cv_force(U0, SMALL, 0.12, n_levels, 0.7)
    assert abs(Q - Qr) <= 1e-12 * max(1.0, abs(Qr))
    assert rel_err(F.download(), Fr) <= 1e-11
    cv.close()


# c1 = tr Q^2 / 2 on both sides of the two lines where the exponential changes its evaluation
# (0.02, 1), far from them, and zero
@pytest.mark.parametrize("c1", [0.0, 1e-9, 0.0199999, 0.0200001, 0.3, 0.9999999, 1.0000001, 4.0])
def test_exponential_against_expm(la, gpu_ctx, c1):
    """The field update of unit links is exp(eps P).  Bar 3e-14: about a hundred roundings of
    1.1e-16 on numbers of at most 3 (the exponential's polynomial and the Gram-Schmidt step)."""
    from scipy.linalg import expm
    flush(f"exponential c1 = {c1}")
    rng = np.random.default_rng(int(1e7 * c1) + 1)
    n = 4 * 4**4
    H = rng.normal(size=(n, 3, 3)) + 1j * rng.normal(size=(n, 3, 3))
    H[0] = np.diag([1.0, 1.0, -2.0])      # a double eigenvalue, either sign of det Q
    H[1] = np.diag([-1.0, -1.0, 2.0])
    H[2] = np.diag([1.0, -1.0, 0.0])
    H = H + H.conj().transpose(0, 2, 1)
    H -= np.trace(H, axis1=1, axis2=2)[:, None, None] / 3.0 * np.eye(3)
    H *= np.sqrt(c1 / (0.5 * np.einsum("nij,nji->n", H, H).real))[:, None, None]
    ref = np.array([expm(1j * h) for h in H])
    U, P = gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY)
    U.SetToIdentity()
    shape = U.download().shape
    P.upload(np.ascontiguousarray(2j * H).view(np.float64).reshape(shape))
    la.UpdateFields(U, P, 0.5)
    got = U.download().view(np.complex128).reshape(n, 3, 3)
    assert np.max(np.abs(got - ref)) <= 3e-14, np.max(np.abs(got - ref))
    U.close()
    P.close()


@pytest.mark.parametrize("rho", [0.02, 0.12, 0.4, 0.7])
def test_cv_force_stout_weights(la, lto, gpu_ctx, rho):
    """Exponential and derivative of one stout level on rough links: rho runs the arguments
    through all three evaluations (c1 about 5 rho^2, spread over the links)."""
    flush(f"cv rho {rho}")
    shape = (4, 4, 4, 6)
    U0 = lto.haar(shape, 3)
    U = gauge(la, gpu_ctx, shape, U0)
    F = matrix(la, gpu_ctx, shape)
    cv = la.CollectiveVariable(gpu_ctx, shape, 1, rho)
    Q = cv.forward(U)
    cv.backward(0.7, F)
    Qr, Fr = lto.cv_force(U0, shape, rho, 1, 0.7)
    assert abs(Q - Qr) <= 1e-12 * max(1.0, abs(Qr))
    assert rel_err(F.download(), Fr) <= 1e-11
    cv.close()


# blocks of 64 links: rows of z cut in three, one block that is not full, a partial last block
@pytest.mark.parametrize("shape", [(2, 2, 8, 48), (2, 2, 2, 2), (2, 6, 2, 10)])
def test_cv_force_small_blocks(la, lto, gpu_ctx, shape):
    """The clover derivative and two recursion levels: the bars of one level above."""
    flush(f"cv blocks {shape}")
    U0 = lto.stout(lto.haar(shape, 6), shape, 0.1, 1)
    U = gauge(la, gpu_ctx, shape, U0)
    F = matrix(la, gpu_ctx, shape)
    cv = la.CollectiveVariable(gpu_ctx, shape, 2, 0.12)
    Q = cv.forward(U)
    cv.backward(0.7, F)
    Qr, Fr = lto.cv_force(U0, shape, 0.12, 2, 0.7)
    assert abs(Q - Qr) <= 1e-12 * max(1.0, abs(Qr))
    assert rel_err(F.download(), Fr) <= 1e-11
    cv.close()


def test_cv_force_golden16(la, lto, golden, gpu_ctx):
    flush("cv golden 16^4")
    U0 = lto.stout(lto.haar(G16, 0), G16, 0.1, 3)
    U = gauge(la, gpu_ctx, G16, U0)
    F = matrix(la, gpu_ctx, G16)
    cv = la.CollectiveVariable(gpu_ctx, G16, 4, 0.12)
    Q = cv.forward(U)
    cv.backward(1.0, F)
    assert abs(Q - golden["cv_force_smooth_Q"][0]) <= 1e-12 * max(1.0, abs(Q))
    assert_field_matches(golden, "cv_force_smooth", F.download(), 1e-11)
    cv.close()


def test_clover_derivative_golden16_and_oracle(la, lto, golden, gpu_ctx):
    """lt_clover_derivative: the reference's CloverDerivative on every link at 16^4 (sampled
    links and field sums), the oracle on other extents, linear in the scale."""
    flush("clover derivative 16^4 and 4x6x8x10")
    U0 = lto.stout(lto.haar(G16, 0), G16, 0.1, 3)
    U = gauge(la, gpu_ctx, G16, U0)
    F = matrix(la, gpu_ctx, G16)
    la.CloverDerivative(U, F)
    assert_field_matches(golden, "clover_deriv_smooth", F.download(), 1e-12)
    shape = (4, 6, 8, 10)
    V0 = smooth(lto, shape, 7, 2)
    V, G = gauge(la, gpu_ctx, shape, V0), matrix(la, gpu_ctx, shape)
    la.CloverDerivative(V, G, -2.5)
    assert rel_err(G.download(), -2.5 * lto.clover_derivative(V0, shape)) <= 1e-12
    with pytest.raises(la.LettuceError):
        la.CloverDerivative(V, F)          # extents differ


def test_cv_force_finite_differences_on_gpu(la, lto, gpu_ctx):
    """The adjoint of the smeared clover charge against central differences of the charge,
    at the metadynamics configuration: 16^4, beta = 6.0, 4 stout levels rho = 0.12, the
    start of numerical_derivative.hpp:74-78 (5 x (heatbath + 4 overrelaxation), here from a
    Haar start), 64 distinct links drawn with seed 1, all 8 generators, h = 1e-6.  The
    reference's check (numerical_derivative.hpp:109-138, 214-215): U_l -> exp(+-i h/2
    lambda_a) U_l, (Q_+ - Q_-) / (2h) against Re tr(lambda_a i F_l).

    Q_+ - Q_- is taken as the sum over sites of the difference of the two per-site charge
    densities: only sites within the smearing and clover reach of the perturbed link differ
    (the others are computed from identical inputs by the same kernels, so they cancel
    exactly), and the rounding of a global sum of O(1) (~1e-13, i.e. 5e-8 after dividing by
    2h) never enters.  What remains is the rounding of the smeared field inside the reach
    (the two perturbed fields are smeared independently): about 1e-16 in Q_+ - Q_-, i.e.
    up to ~1e-10 absolute in the difference quotient at h = 1e-6, against gradients of
    1e-3 to 1e-2 per link.  Bars: max |fd - an| <= 1e-7 * max |an| over the whole sample
    (64 x 8 components), and per link max_a |fd_a - an_a| <= 2e-7 * max_a |an_a| (measured
    1.2e-7 at the worst of the 64 links, where the gradient is smallest)."""
    import math
    flush("cv FD 16^4, 64 links x 8 generators, h = 1e-6")
    from test_oracle_golden import gell_mann
    shape = G16
    U = gauge(la, gpu_ctx, shape)
    U.SetToHaar(0)
    U.set_rng(0, 0)
    hb, orx = la.HeatbathKernel(U, 6.0), la.OverrelaxationSubgroupKernel(U)
    for _ in range(5):
        la.Iterator.Checkerboard(hb, 1)
        la.Iterator.Checkerboard(orx, 4)
    U0 = U.download()
    F = matrix(la, gpu_ctx, shape)
    cv = la.CollectiveVariable(gpu_ctx, shape, 4, 0.12)
    cv.forward(U)
    cv.backward(1.0, F)
    cv.close()
    Fm = F.download().reshape(-1, 3, 3, 2)
    Fm = Fm[..., 0] + 1j * Fm[..., 1]
    lam = gell_mann()
    h = 1e-6
    W = U0.copy()
    flat = W.reshape(-1, 18)
    links = np.random.default_rng(1).choice(flat.shape[0], 64, replace=False)
    S = gauge(la, gpu_ctx, shape)
    worst, worst_abs, per_link, an_max = 0.0, 0.0, [], 0.0
    for n, link in enumerate(links):
        keep = flat[link].copy()
        M = keep.reshape(3, 3, 2)
        M = M[..., 0] + 1j * M[..., 1]
        an = np.array([np.real(np.trace(lam[a] @ (1j * Fm[link]))) for a in range(8)])
        fd = np.empty(8)
        for a in range(8):
            q = []
            for sgn in (1, -1):
                X = sgn * 0.5 * h * lam[a]
                E = lto.su3_exp(np.stack([X.real, X.imag], -1)).reshape(3, 3, 2)
                N = (E[..., 0] + 1j * E[..., 1]) @ M
                flat[link] = np.stack([N.real, N.imag], -1).reshape(18)
                U.upload(W)
                la.StoutSmearingN(U, S, 4, 0.12)
                q.append(la.TopChargeCloverDensity(S))
            flat[link] = keep
            d = (q[0] - q[1]).ravel()
            fd[a] = math.fsum(d[d != 0.0]) / (2 * h)
        scale = np.max(np.abs(an))
        err = np.max(np.abs(fd - an))
        per_link.append(err / scale)
        worst = max(worst, err / scale)
        worst_abs = max(worst_abs, err)
        an_max = max(an_max, scale)
        if n % 16 == 15:
            flush(f"  {n + 1} links: worst relative deviation {worst:.2e} (absolute {worst_abs:.2e})")
    flush(f"  per link: median {np.median(per_link):.2e}, worst {worst:.2e}; sample-wide: "
          f"{worst_abs / an_max:.2e} of the largest gradient component {an_max:.2e}")
    assert worst_abs <= 1e-7 * an_max
    assert worst <= 2e-7


def metad_setup(la, lto, golden):
    a = golden["metad_bias_args"]
    bias = la.MetaBiasPotential(a[0], a[1], int(a[2]), a[3], a[4], a[5], a[6], well_tempered=True)
    obias = lto.Bias(a[0], a[1], int(a[2]), a[3], a[4], a[5], a[6], well_tempered=True)
    for d in golden["metad_bias_deposits"]:
        bias.UpdatePotentialSymmetric(d)
        obias.deposit_symmetric(d)
    return bias, obias


def test_metad_trajectory_golden16(la, lto, golden, gpu_ctx):
    """MetaD-HMC OMF2 trajectory with Philox momenta equal to the injected ones of the golden run."""
    flush("metad golden 16^4")
    bias, _ = metad_setup(la, lto, golden)
    U0 = lto.stout(lto.haar(G16, 0), G16, 0.1, 3)
    U = gauge(la, gpu_ctx, G16, U0)
    Uc = gauge(la, gpu_ctx, G16)
    P = matrix(la, gpu_ctx, G16)
    F = matrix(la, gpu_ctx, G16)
    cv = la.CollectiveVariable(gpu_ctx, G16, 4, 0.12)
    U.set_rng(5, 0)     # momenta = lto_random_momentum(seed=5, counter=0), as injected in the reference
    k = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, "omf2", 6.0, 0.5, update_bias=True)
    assert k(5, metropolis_step=False)
    Href = golden["metad_omf2_smooth_H"]
    assert abs(k.delta_H - (Href[1] - Href[0])) <= 1e-7 * max(1.0, abs(Href[1] - Href[0]))
    assert abs(k.cv_value - golden["metad_omf2_smooth_CV"][1]) <= 1e-9
    assert_field_matches(golden, "metad_omf2_smooth", U.download(), 1e-9)
    a = golden["metad_bias_args"]
    x = a[0] + np.arange(int(a[2]) + 1) * (a[1] - a[0]) / int(a[2])
    got = np.array([bias.ReturnPotential(v) for v in x])
    assert rel_err(got, golden["metad_omf2_smooth_grid_after"]) <= 1e-9
    cv.close()


def test_metad_trajectory_vs_oracle_small(la, lto, golden, gpu_ctx):
    flush("metad 4^4 vs oracle")
    bias, obias = metad_setup(la, lto, golden)
    U0 = smooth(lto, TINY, 8, 2)
    U = gauge(la, gpu_ctx, TINY, U0)
    Uc = gauge(la, gpu_ctx, TINY)
    P = matrix(la, gpu_ctx, TINY)
    F = matrix(la, gpu_ctx, TINY)
    cv = la.CollectiveVariable(gpu_ctx, TINY, 2, 0.12)
    U.set_rng(3, 11)
    k = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, "omf2", 6.0, 0.4, update_bias=False)
    k(4, metropolis_step=False)
    Ur = U0.copy()
    Pr = lto.random_momentum(TINY, 3, 11)
    H0, H1, _, cv1, _ = lto.metad_omf2(Ur, Pr, TINY, 6.0, 0.4, 4, 0.12, 2, obias)
    assert abs(k.delta_H - (H1 - H0)) <= 1e-8 * max(1.0, abs(H1 - H0))
    assert abs(k.cv_value - cv1) <= 1e-10
    assert rel_err(U.download(), Ur) <= 1e-10
    cv.close()


@pytest.mark.parametrize("integrator", ["leapfrog_omf4", "omf2_omf4", "omf2_omf4_slow", "omf4", "leapfrog",
                                        "omf4_slow"])
def test_metad_integrators_vs_oracle(la, lto, golden, gpu_ctx, integrator):
    """Every MetaD-HMC schedule (the multiple-timescale ones of hmc_metadynamics.hpp:28-238
    among them) against the oracle's trajectory on the same Philox momenta; the path
    samples too."""
    flush(f"metad {integrator} 4^4 vs oracle")
    bias, obias = metad_setup(la, lto, golden)
    U0 = smooth(lto, TINY, 8, 2)
    U = gauge(la, gpu_ctx, TINY, U0)
    Uc, P, F = gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY)
    cv = la.CollectiveVariable(gpu_ctx, TINY, 2, 0.12)
    U.set_rng(3, 11)
    k = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, integrator, 6.0, 0.4, update_bias=False)
    k(3, metropolis_step=False)
    Ur = U0.copy()
    Pr = lto.random_momentum(TINY, 3, 11)
    H0, H1, _, cv1, samples = lto.metad_trajectory(Ur, Pr, TINY, 6.0, 0.4, 3, 0.12, 2, obias, integrator)
    assert abs(k.delta_H - (H1 - H0)) <= 1e-8 * max(1.0, abs(H1 - H0))
    assert abs(k.cv_value - cv1) <= 1e-10
    assert rel_err(U.download(), Ur) <= 1e-10
    got = k.path_samples()
    assert len(got) == len(samples) == 3
    assert np.max(np.abs(got - np.array(samples))) <= 1e-10
    assert np.array_equal(k.path_samples(deposited=True), got)       # accepted: deposits = visited
    cv.close()


@pytest.mark.parametrize("integrator", ["omf2", "omf4", "leapfrog_omf4", "omf2_omf4", "omf2_omf4_slow"])
def test_reversibility_tests(la, lto, golden, gpu_ctx, integrator):
    """ReversibilityTest (hmc_gauge.hpp:585-599, hmc_metadynamics.hpp:657-674): forward,
    reversed momenta, back to the start -- the field to rounding and H_new = H_old."""
    flush(f"reversibility {integrator}")
    bias, _ = metad_setup(la, lto, golden)
    U0 = smooth(lto, TINY, 12, 2)
    U = gauge(la, gpu_ctx, TINY, U0)
    Uc, P, F = gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY)
    cv = la.CollectiveVariable(gpu_ctx, TINY, 2, 0.12)
    U.set_rng(8, 0)
    h0, h1 = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, integrator, 6.0, 0.5).ReversibilityTest(4)
    assert abs(h1 - h0) <= 1e-9 * abs(h0)
    assert np.max(np.abs(U.download() - U0)) <= 1e-10
    assert U.get_rng() == (8, 1)
    if integrator in ("omf2", "omf4"):
        U.upload(U0)
        g0, g1 = la.HMCKernel(U, Uc, P, integrator, 6.0, 0.5).ReversibilityTest(4)
        assert abs(g1 - g0) <= 1e-9 * abs(g0)
        assert np.max(np.abs(U.download() - U0)) <= 1e-10
    cv.close()


def test_hmc_log_lines(la, lto, golden, gpu_ctx, tmp_path):
    """LogCVData after each trajectory (hmc_metadynamics.hpp:613,642): the visited CVs, then
    with the Metropolis step the deposited ones (CV_old repeated after a rejection), in the
    %g format the reference's stream writes."""
    flush("hmc log lines")
    bias, _ = metad_setup(la, lto, golden)
    U = gauge(la, gpu_ctx, TINY, smooth(lto, TINY, 4, 2))
    Uc, P, F = gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY)
    cv = la.CollectiveVariable(gpu_ctx, TINY, 2, 0.12)
    U.set_rng(2, 0)
    log = tmp_path / "hmc_log.txt"
    k = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, "omf2", 6.0, 0.5, update_bias=True, hmc_log_path=str(log))
    with pytest.raises(la.LettuceError):
        k.LogCVData()                      # no trajectory yet: nothing to log
    assert len(k.path_samples()) == 0
    expect = []
    for step in range(4):
        # coarse steps (n_step = 1) reject now and then; the deposited line then repeats CV_old
        acc = k(1 if step % 2 else 6, metropolis_step=True)
        visited = k.path_samples()
        used = k.path_samples(deposited=True)
        assert len(visited) == len(used) == (1 if step % 2 else 6)
        if acc:
            assert np.array_equal(used, visited)
        else:
            assert np.all(used == k.cv_value)      # CV_old, which the rejected trajectory keeps
        expect.append(" ".join(format(v, "g") for v in visited))
        expect.append(" ".join(format(v, "g") for v in used))
    k(3, metropolis_step=False)
    expect.append(" ".join(format(v, "g") for v in k.path_samples()))
    assert log.read_text().splitlines() == expect
    k.hmc_log_path = str(tmp_path / "missing_dir" / "hmc_log.txt")
    with pytest.raises(la.LettuceError):
        k.LogCVData()                      # unwritable path: an error, not a silent skip
    cv.close()


@pytest.mark.parametrize("n_levels,interval", [(4, 1), (4, 2), (4, 3), (8, 3), (5, 5), (1, 1)])
def test_checkpointed_cv_equals_full_storage(la, lto, gpu_ctx, n_levels, interval):
    """Recomputing stout levels from checkpoints gives the same Q and force bit for bit,
    with less memory."""
    flush(f"checkpointed CV n={n_levels} k={interval}")
    U0 = smooth(lto, SMALL, 12, 1)
    U = gauge(la, gpu_ctx, SMALL, U0)
    F_full, F_ck = matrix(la, gpu_ctx, SMALL), matrix(la, gpu_ctx, SMALL)
    full = la.CollectiveVariable(gpu_ctx, SMALL, n_levels, 0.12)
    ck = la.CollectiveVariable(gpu_ctx, SMALL, n_levels, 0.12, checkpoint=interval)
    q_full, q_ck = full.forward(U), ck.forward(U)
    full.backward(0.7, F_full)
    ck.backward(0.7, F_ck)
    assert q_full == q_ck
    assert np.array_equal(F_full.download(), F_ck.download())
    if (n_levels, interval) == (8, 3):     # about sqrt(n): 7 level and 3 tape buffers instead of 9 and 8
        assert ck.bytes() < 0.75 * full.bytes()
    full.close()
    ck.close()


def test_checkpointed_metad_trajectory_equals_full(la, lto, golden, gpu_ctx):
    flush("checkpointed MetaD trajectory")
    U0 = smooth(lto, SMALL, 13, 2)
    out = []
    for interval in (0, 3):
        bias, _ = metad_setup(la, lto, golden)
        U = gauge(la, gpu_ctx, SMALL, U0)
        Uc, P, F = gauge(la, gpu_ctx, SMALL), matrix(la, gpu_ctx, SMALL), matrix(la, gpu_ctx, SMALL)
        cv = la.CollectiveVariable(gpu_ctx, SMALL, 8, 0.12, checkpoint=interval)
        U.set_rng(21, 0)
        k = la.HMCMetaDKernel(U, Uc, P, F, bias, cv, "omf2", 6.0, 0.3, update_bias=True)
        acc = k(3, metropolis_step=True)
        out.append((k.delta_H, acc, k.cv_value, U.download(), bias.grid()))
        cv.close()
    (d0, a0, q0, u0, g0), (d1, a1, q1, u1, g1) = out
    assert d0 == d1 and a0 == a1 and q0 == q1
    assert np.array_equal(u0, u1) and np.array_equal(g0, g1)


def test_tempering_run_matches_oracle(la, lto, gpu_ctx):
    """TemperingRun (SU3_main.cpp:600-616) against the oracle doing the same iteration:
    tempering_nonmetadynamics_sweeps x (Checkerboard4 HB + OR) on the unbiased stream with
    its Philox counters, a MetaD-HMC OMF2 trajectory with Metropolis (stream 3) and path
    deposits on the biased stream, a swap proposal (stream 4) every second iteration."""
    flush("tempering run vs oracle")
    shape = (4, 4, 4, 8)
    rho, nl, beta, tau, n_hmc = 0.12, 2, 6.0, 0.3, 3
    A, B = smooth(lto, shape, 31, 2), smooth(lto, shape, 32, 2)
    U, Ut = gauge(la, gpu_ctx, shape, A), gauge(la, gpu_ctx, shape, B)
    U.set_rng(5, 0)
    Ut.set_rng(6, 0)
    Uc, P, F = gauge(la, gpu_ctx, shape), matrix(la, gpu_ctx, shape), matrix(la, gpu_ctx, shape)
    bias = la.MetaBiasPotential(-8.0, 8.0, 800, 1.5, 0.3, 10.0, 1000.0, well_tempered=True)
    ob = lto.Bias(-8.0, 8.0, 800, 1.5, 0.3, 10.0, 1000.0, well_tempered=True)
    for d in (0.3, -0.5, 0.05):
        bias.UpdatePotential(d)
        ob.deposit(d)
    cv = la.CollectiveVariable(gpu_ctx, shape, nl, rho)
    hmc = la.HMCMetaDKernel(Ut, Uc, P, F, bias, cv, "omf2", beta, tau, update_bias=True)
    temper = la.MetadynamicsTemperingKernel(U, Ut, bias, cv, seed=77)
    run = la.TemperingRun(la.HeatbathKernel(U, beta), la.OverrelaxationSubgroupKernel(U), hmc, temper,
                          n_heatbath=1, n_orelax=2, tempering_nonmetadynamics_sweeps=2, tempering_swap_period=2)
    host = {"U": A.copy(), "Ut": B.copy()}
    hb_counter, traj, swaps = 0, 0, 0
    for n_count in range(4):
        acc, swapped = run.step(n_count, n_hmc, True)
        for _ in range(2):
            hb_counter = lto.hb_sweep(host["U"], shape, beta, 1, 4, 5, hb_counter)
            lto.or_sweep(host["U"], shape, 2, 4)
        W = host["Ut"].copy()
        H0, H1, q0, q1, samples = lto.metad_trajectory(W, lto.random_momentum(shape, 6, traj), shape, beta, tau,
                                                      n_hmc, rho, nl, ob, "omf2")
        expect_acc = lto.uniform(6, 0xFFFFFFFF, 3, traj) <= np.exp(-(H1 - H0))
        traj += 1
        assert acc == expect_acc, f"iteration {n_count}"
        if acc:
            host["Ut"], cur = W, q1
        else:
            samples, cur = [q0] * len(samples), q0
        for s in samples:
            ob.deposit_symmetric(s)
        if n_count % 2 == 0:
            q_new = lto.cv_charge(host["U"], shape, rho, nl)
            expect_swap = lto.uniform(77, 0, 4, swaps) <= np.exp(-(ob.potential(q_new) - ob.potential(cur)))
            swaps += 1
            assert swapped == expect_swap, f"iteration {n_count}"
            if swapped:
                host["U"], host["Ut"] = host["Ut"], host["U"]
                cur = q_new
        else:
            assert swapped is None
        # rounding of the MetaD trajectory reaches a few 1e-10 per link entry and in the CV; a
        # heatbath, Metropolis or swap decision that went the other way would differ at O(1)
        assert abs(bias.ReturnCV_current() - cur) <= 1e-8
        assert np.max(np.abs(U.download() - host["U"])) <= 1e-8, f"iteration {n_count}: unbiased stream"
        assert np.max(np.abs(Ut.download() - host["Ut"])) <= 1e-8, f"iteration {n_count}: MetaD stream"
        assert rel_err(Ut.download(), host["Ut"]) <= 1e-9
        assert rel_err(bias.grid(), ob.grid) <= 1e-8     # deposits at CVs equal to ~1e-10
        # the next iteration starts the oracle from the device's state: heatbath sweeps
        # amplify rounding differences of the fields (3e-10 -> 1e-6 over two iterations)
        host["U"], host["Ut"] = U.download(), Ut.download()
        ob.grid = bias.grid()
        cur = bias.ReturnCV_current()
    cv.close()


def test_tempering_run_resumes_bit_for_bit(la, lto, gpu_ctx, tmp_path):
    """A two-stream TemperingRun stopped after two iterations and resumed from saved
    state (both fields, the bias grid and current CV, and one PhiloxState holding the
    unbiased field's, the MetaD field's and the swap proposals' streams) continues
    exactly as the uninterrupted run."""
    flush("tempering run resume")
    shape = (4, 4, 4, 8)
    rho, nl, beta, tau, n_hmc = 0.12, 2, 6.0, 0.3, 3

    def make(A, B):
        U, Ut = gauge(la, gpu_ctx, shape, A), gauge(la, gpu_ctx, shape, B)
        Uc, P, F = gauge(la, gpu_ctx, shape), matrix(la, gpu_ctx, shape), matrix(la, gpu_ctx, shape)
        bias = la.MetaBiasPotential(-8.0, 8.0, 800, 1.5, 0.3, 10.0, 1000.0, well_tempered=True)
        cv = la.CollectiveVariable(gpu_ctx, shape, nl, rho)
        hmc = la.HMCMetaDKernel(Ut, Uc, P, F, bias, cv, "omf2", beta, tau, update_bias=True)
        temper = la.MetadynamicsTemperingKernel(U, Ut, bias, cv, seed=77)
        run = la.TemperingRun(la.HeatbathKernel(U, beta), la.OverrelaxationSubgroupKernel(U), hmc, temper,
                              n_heatbath=1, n_orelax=2, tempering_nonmetadynamics_sweeps=1, tempering_swap_period=1)
        return run, U, Ut, bias, temper, cv

    A, B = smooth(lto, shape, 41, 2), smooth(lto, shape, 42, 2)
    run, U, Ut, bias, temper, cv = make(A, B)
    U.set_rng(5, 0)
    Ut.set_rng(6, 0)
    for n in range(2):
        run.step(n, n_hmc, True)
    saved = {"U": U.download(), "Ut": Ut.download(), "grid": bias.grid(), "cv": bias.ReturnCV_current()}
    assert la.PhiloxState(U, Ut, temper).SaveState(str(tmp_path / "prng.txt"), str(tmp_path / "dist.txt"))
    trail = [run.step(n, n_hmc, True) for n in range(2, 5)]
    end = (U.download(), Ut.download(), bias.grid())
    cv.close()
    run2, U2, Ut2, bias2, temper2, cv2 = make(saved["U"], saved["Ut"])
    bias2.set_grid(saved["grid"])
    bias2.SetCV_current(saved["cv"])
    assert la.PhiloxState(U2, Ut2, temper2).LoadState(str(tmp_path / "prng.txt"))
    trail2 = [run2.step(n, n_hmc, True) for n in range(2, 5)]
    assert trail2 == trail
    assert np.array_equal(U2.download(), end[0]) and np.array_equal(Ut2.download(), end[1])
    assert np.array_equal(bias2.grid(), end[2])
    cv2.close()


def test_metad_run_parity_coin(la, lto, golden, gpu_ctx):
    """MetaDRun (SU3_main.cpp:523-531): a trajectory, then ParityUpdate on heads."""
    flush("metad run parity")
    bias, _ = metad_setup(la, lto, golden)
    U = gauge(la, gpu_ctx, TINY, smooth(lto, TINY, 3, 2))
    Uc, P, F = gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY)
    cv = la.CollectiveVariable(gpu_ctx, TINY, 2, 0.12)
    U.set_rng(4, 0)
    run = la.MetaDRun(la.HMCMetaDKernel(U, Uc, P, F, bias, cv, "omf2", 6.0, 0.3, update_bias=False), Uc,
                      np.random.default_rng(3))
    # the same trajectory without the parity step, from the same state each time
    V = gauge(la, gpu_ctx, TINY)
    plain = la.HMCMetaDKernel(V, gauge(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY), matrix(la, gpu_ctx, TINY),
                              bias, cv, "omf2", 6.0, 0.3, update_bias=False)
    coins = np.random.default_rng(3).integers(0, 2, size=6)
    for k in range(6):
        V.upload(U.download())
        V.set_rng(*U.get_rng())
        _, flipped = run.step(2, True)
        plain(2, True)
        assert flipped == bool(coins[k])
        expect = lto.parity_update(V.download(), TINY) if flipped else V.download()
        assert np.max(np.abs(U.download() - expect)) <= 1e-13, f"step {k}"
    assert 0 < coins.sum() < 6
    cv.close()


def test_two_stream_tempering_swap(la, lto, gpu_ctx):
    """MetadynamicsTemperingKernel (tempering.hpp:57-72) against the oracle's rule, call by
    call: CV of the unbiased stream through 4 stout levels, the bias at that CV and at the
    biased stream's current CV, the Philox uniform of stream 4 / site 0; accepted calls
    swap the links and move the bias CV."""
    flush("two-stream tempering")
    shape = (4, 4, 4, 8)
    rho, nl = 0.12, 4
    A = lto.stout(lto.haar(shape, 21), shape, 0.1, 2)
    B = lto.stout(lto.haar(shape, 22), shape, 0.1, 2)
    U = la.GaugeField(gpu_ctx, shape)
    U.upload(A)
    Ut = la.GaugeField(gpu_ctx, shape)
    Ut.upload(B)
    bias = la.MetaBiasPotential(-8.0, 8.0, 800, 1.5, 0.3, 10.0, 1000.0, well_tempered=True)
    ob = lto.Bias(-8.0, 8.0, 800, 1.5, 0.3, 10.0, 1000.0, well_tempered=True)
    for d in (0.3, -0.5, 1.1, 0.05):
        bias.UpdatePotential(d)
        ob.deposit(d)
    cv = la.CollectiveVariable(gpu_ctx, shape, nl, rho)
    cur = lto.cv_charge(B, shape, rho, nl)
    bias.SetCV_current(cur)
    kernel = la.MetadynamicsTemperingKernel(U, Ut, bias, cv, seed=77, counter=0)
    host = {"U": A, "Ut": B}
    seen = set()
    for step in range(12):
        q_new = lto.cv_charge(host["U"], shape, rho, nl)
        dv = ob.potential(q_new) - ob.potential(cur)
        expect = lto.uniform(77, 0, 4, step) <= np.exp(-dv)
        got = kernel()
        assert got == expect and abs(kernel.delta_V - dv) <= 1e-10 * max(1.0, abs(dv))
        seen.add(got)
        if got:
            host["U"], host["Ut"] = host["Ut"], host["U"]
            cur = q_new
        assert abs(bias.ReturnCV_current() - cur) <= 1e-12
        assert np.array_equal(U.download()[..., :12], host["U"][..., :12])
        assert np.array_equal(Ut.download()[..., :12], host["Ut"][..., :12])
    assert seen == {True, False}
    for f in (U, Ut, cv, bias):
        f.close()
