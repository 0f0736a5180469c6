"""Small Gaussian-pair chains (k_sweep_allpairs) against the oracle, FP64: rings
around a wave's 64 slices and around the sizes where the particles a link is
split over change (2 to 16 groups), a last segment of one link, one and two
particles, more particles than a wave has lanes for one group, paths larger
than LDS (rows in memory), and chains next to them that other kernels run."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, HarmonicTrap, NoPotential
from pimc.system import chain_desc
from test_gpu_random_configs import run_and_check

pytestmark = pytest.mark.gpu


def chain(N, M, ell, dim=2, nbins=3, pot=None, every=(1, 1, 1), seed=0):
    rng = np.random.default_rng(1000 * N + M + seed)
    L = 3.0
    d = chain_desc(pot or HarmonicTrap(0.5), dim=dim, M=M, N=N, L=L, beta=1.5, lam=0.5, pair=GaussianPair(1.0, 0.5), ell=ell,
                   r_a=2 * L / nbins, com_step=0.5, staging_every=every[0], com_every=every[1], swap_every=every[2])
    r = rng.uniform(-L, L, size=(N, dim, 1)).repeat(M, axis=2) + rng.normal(0, 0.1, size=(N, dim, M))
    return d, (r + L) % (2 * L) - L, "gauss", every


@pytest.mark.parametrize("N,M,ell", [(1, 16, 8), (2, 4, 2), (5, 33, 8), (6, 63, 8), (9, 64, 8), (9, 65, 8), (4, 127, 7),
                                     (3, 128, 16), (5, 129, 8), (3, 257, 8), (2, 512, 32), (70, 16, 5), (90, 12, 4),
                                     (12, 700, 8), (30, 400, 9)])
def test_allpairs_chains_match_oracle(N, M, ell):
    run_and_check([chain(N, M, ell)], 21 + N, 2)


def test_allpairs_1d_and_mixed():
    run_and_check([chain(7, 20, 6, dim=1)], 3, 3)
    # rings of several lengths in one launch, move weights, and nbins = 2 (the whole-chain kernel)
    run_and_check([chain(7, 20, 6), chain(11, 70, 8, pot=NoPotential(), every=(2, 1, 1)), chain(5, 40, 9, every=(1, 3, 1)),
                   chain(8, 16, 8, nbins=2)], 4, 3)


@pytest.mark.parametrize("measure_kernel", [1, 2])
def test_allpairs_estimators_agree(measure_kernel):
    """The estimators of the sweep kernel and of the wide kernel are the same
    samples: M = 37 leaves a last window of five slices; sums of the same FP64
    terms in another order agree to 1e-11."""
    d, r, _, _ = chain(9, 37, 8)
    out = []
    for mk in (1, measure_kernel):
        opt = A.Options()
        opt.precision, opt.sweeps_per_launch, opt.seed, opt.measure_kernel = A.FP64, 4, 9, mk
        opt.derivatives, opt.radial_bins, opt.radial_rmax = 1, 16, 4.0
        ctx = A.Context([d], opt)
        ctx.set_paths(0, r)
        ctx.run(8, measure=True)
        e = ctx.estimates(0)
        out.append(([e.E, e.Ev, e.Epair, e.dSdomega, e.dSdg], ctx.radial(0)[0]))
    assert np.allclose(out[0][0], out[1][0], rtol=1e-11, atol=0)
    assert np.array_equal(out[0][1], out[1][1])
