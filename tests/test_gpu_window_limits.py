"""The window kernels at the limits of what a workgroup's LDS holds."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, NoPotential
from pimc.system import chain_desc
from test_gpu_random_configs import run_and_check

pytestmark = pytest.mark.gpu


def gas(N, M, ell, L, nbins, dim=2, beta=1.0, seed=0):
    """A Gaussian-pair chain in a periodic box and rings around uniform centres."""
    rng = np.random.default_rng(1000 * N + M + seed)
    d = chain_desc(NoPotential(), dim=dim, M=M, N=N, L=L, beta=beta, lam=0.5, pair=GaussianPair(1.0, 0.5), ell=ell,
                   r_a=2 * L / nbins, com_step=0.5)
    r = rng.uniform(-L, L, size=(N, dim, 1)) + rng.normal(0, 0.1, size=(N, dim, M))
    return d, (r + L) % (2 * L) - L


@pytest.mark.parametrize("N,M", [(193, 3137), (192, 3137), (168, 3649)])
def test_long_rings_are_measured_fp32(N, M):
    """Long rings: the estimator kernel needs more LDS for one particle's
    partners than the sweep kernels.  One measured sweep gives the energies of
    the paths that it leaves.  Both sides sum the same FP32 terms in FP64, each
    term good to a few roundings of 6e-8: 1e-6 of the sums of absolute values,
    the kinetic constant for E (ctx.energy keeps the pair
    energy apart) and the pair energy itself."""
    d, r = gas(N, M, 2, 8.0, 8)
    opt = A.Options()
    opt.precision, opt.sweeps_per_launch, opt.seed = A.FP32, 1, 5
    ctx = A.Context([d], opt)
    ctx.set_paths(0, r)
    ctx.run(1, measure=True)
    e = ctx.estimates(0)
    E, Ev, Ep, Evp = ctx.energy(0)
    assert abs(e.E - e.Epair - E) < 1e-6 * d.dim * N * M / d.beta
    assert abs(e.Epair - Ep) < 1e-6 * abs(Ep)


@pytest.mark.parametrize("N,M,ell,L,nbins,dim", [(148, 40, 32, 4.0, 4, 2), (504, 9, 8, 8.0, 8, 2), (281, 36, 32, 60.0, 40, 1)])
def test_largest_chains_match_oracle_fp64(N, M, ell, L, nbins, dim):
    """The largest chains of their staging length: the smallest blocks, a pool of
    one particle's partners, and nearly all pairs of a window in memory."""
    d, r = gas(N, M, ell, L, nbins, dim)
    run_and_check([(d, r, "gauss", (1, 1, 1))], 61 + N, 1)
