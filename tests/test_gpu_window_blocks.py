"""The window kernels at the sizes where their blocks and pools change: particle
counts around the 64-particle words and chunks, dense chains whose pairs do not
fit the staging kernel's LDS (the rest of a window's pairs go through memory)
or one pool (several blocks), one staging window, and few particles
(pair_kernel = 2), against the oracle in FP64."""
import numpy as np
import pytest

from pimc.potentials import GaussianPair, HarmonicTrap
from pimc.system import chain_desc
from test_gpu_random_configs import run_and_check

pytestmark = pytest.mark.gpu


def chain(N, M, ell, L, nbins, omega=0.3, dim=2, spread=1.0, seed=0):
    rng = np.random.default_rng(1000 * N + M + seed)
    d = chain_desc(HarmonicTrap(omega), dim=dim, M=M, N=N, L=L, beta=2.0, lam=0.5, pair=GaussianPair(1.0, 0.5), ell=ell,
                   r_a=2 * L / nbins, com_step=0.5)
    r = spread * rng.uniform(-L, L, size=(N, dim, 1)).repeat(M, axis=2) + rng.normal(0, 0.1, size=(N, dim, M))
    return d, (r + L) % (2 * L) - L, "gauss", (1, 1, 1)


@pytest.mark.parametrize("N", [2, 63, 64, 65, 127, 129, 193])
def test_particle_counts_around_words(N):
    run_and_check([chain(N, 12, 5, 6.0, 6)], 31 + N, 2, pair_kernel=2)


@pytest.mark.parametrize("N,M,ell,L,nbins", [(150, 8, 8, 3.0, 3), (260, 8, 4, 4.0, 4), (200, 12, 12, 3.0, 3)])
def test_dense_chains(N, M, ell, L, nbins):
    """Every particle meets most others: 11 000 to 33 000 pairs a window."""
    run_and_check([chain(N, M, ell, L, nbins, spread=0.8)], 41 + N, 2, pair_kernel=2)


def test_mixed_sizes_and_1d():
    run_and_check([chain(130, 20, 8, 6.0, 6), chain(97, 33, 6, 5.0, 5), chain(70, 270, 9, 8.0, 8), chain(30, 9, 2, 3.0, 2)], 51, 2,
                  pair_kernel=2)
    run_and_check([chain(110, 16, 8, 20.0, 12, dim=1), chain(100, 10, 3, 10.0, 3, dim=1)], 52, 2, pair_kernel=2)
