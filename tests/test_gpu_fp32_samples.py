"""One FP32 sweep of the pair and swap kernels against the oracle's FP64 sweep
from the same paths with the same draws, at the sizes where the FP32 kernels
take other blocks, lanes or pools than the FP64 ones.

A new bead is off by the rounding of its normal (hardware log, sine and cosine
of a 24-bit uniform: below 1e-4 but for uniforms within 1e-6 of 1, where it is
below 4e-4) times the bridge's width, below 1, and by 32 steps of 1e-6: 1e-3 in
all, where a move that one side takes and the other does not is a hundred times
that.  A decision differs where log(u) is within the FP32 error of the weight,
some 1e-5, of it: for the at most 3 000 tries of a case three in a hundred cases
have one.  So at most one staging segment and one ring may differ."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, HarmonicTrap
from pimc.system import chain_desc
from test_gpu_random_configs import oracle_of

pytestmark = pytest.mark.gpu


def check(N, M, ell, L, nbins=0, dim=2, swaps=0, swap_m=0, pair_kernel=0, omega=0.5, seed=0):
    rng = np.random.default_rng(100 * N + M + seed)
    pair = GaussianPair(1.0, 0.5) if nbins else None
    d = chain_desc(HarmonicTrap(omega), dim=dim, M=M, N=N, L=L, beta=1.5, lam=0.5, pair=pair, ell=ell,
                   r_a=2 * L / nbins if nbins else 0.0, com_step=0.5, swaps=swaps, swap_m=swap_m)
    r = 0.9 * rng.uniform(-L, L, size=(N, dim, 1)).repeat(M, axis=2) + rng.normal(0, 0.1, size=(N, dim, M))
    r = np.clip(r, -0.99 * L, 0.99 * L).astype(np.float32).astype(np.float64)
    opt = A.Options()
    opt.precision, opt.sweeps_per_launch, opt.seed, opt.pair_kernel = A.FP32, 1, 17 + seed, pair_kernel
    ctx = A.Context([d], opt)
    ctx.set_paths(0, r)
    s = oracle_of(d, r, "gauss" if nbins else "none", None, None)
    ctx.run(1, measure=True)
    s.sweep_every(0, 0, 17 + seed, d.ell, d.com_step, (1, 1, 1), d.swaps, d.swap_m or d.ell, d.swap_rule)
    got = ctx.get_paths(0)
    off = np.abs(got - s.r)
    off = np.minimum(off, 2 * L - off).max(axis=1) > 1e-3
    assert off.sum() <= M + ell, (off.sum(), N * M)
    if swaps:
        assert np.array_equal(ctx.get_next(0), s.next)
        return
    # the estimators of the sweep: those of the paths it leaves, the same FP32 terms summed in FP64
    e, (E, _, Ep, _) = ctx.estimates(0), ctx.energy(0)
    assert abs(e.E - e.Epair - E) < 1e-6 * (dim * N * M / d.beta + abs(E))
    assert abs(e.Epair - Ep) <= 1e-6 * abs(Ep)


@pytest.mark.parametrize("N,M,ell", [(9, 63, 8), (9, 64, 8), (9, 65, 8), (5, 129, 8), (3, 257, 8), (2, 512, 32), (70, 16, 5),
                                     (90, 12, 4), (73, 64, 8)])
def test_small_pair_chains(N, M, ell):
    check(N, M, ell, 3.0, 3)


@pytest.mark.parametrize("N,M,ell,dim", [(12, 16, 8, 2), (13, 16, 8, 2), (13, 17, 8, 2), (30, 48, 8, 1), (30, 49, 8, 1)])
def test_small_pair_chains_at_the_kernels_border(N, M, ell, dim):
    """Short rings run on k_sweep_whole, the next longer ones on k_sweep_allpairs."""
    check(N, M, ell, 3.0, 3, dim=dim)


@pytest.mark.parametrize("N,M,ell,L,nbins,dim", [(65, 12, 5, 6.0, 6, 2), (150, 8, 8, 3.0, 3, 2), (260, 8, 4, 4.0, 4, 2),
                                                 (200, 12, 12, 3.0, 3, 2), (400, 40, 8, 10.0, 10, 2), (110, 16, 8, 20.0, 12, 1),
                                                 (290, 36, 32, 6.0, 6, 2)])
def test_window_chains(N, M, ell, L, nbins, dim):
    """Up to nearly all pairs of a window in memory (the dense chains and the one
    with 32 links a segment)."""
    check(N, M, ell, L, nbins, dim, pair_kernel=2)


@pytest.mark.parametrize("N,M,ell,swaps,swap_m", [(7, 33, 8, 17, 9), (10, 64, 8, 33, 8), (65, 16, 5, 20, 15), (2, 65, 8, 16, 64),
                                                  (3, 513, 32, 2, 40), (64, 100, 8, 4, 8)])
def test_swap_chains(N, M, ell, swaps, swap_m):
    check(N, M, ell, 3.0, swaps=swaps, swap_m=swap_m, omega=1.0)
