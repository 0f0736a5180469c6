"""Single moves, energies and adjoints at the sizes where their kernels change
path: move scratch that does not fit LDS, fewer links than lanes, and more beads
than one pass of the grid holds."""
import numpy as np
import pytest

from pimc import _capi as A
from pimc.potentials import GaussianPair, HarmonicTrap, NoPotential
from pimc.system import chain_desc
from test_gpu_parity import make_ctx, oracle_sys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(3, 4), (2, 1365), (3, 1366), (2, 1700)])
def test_moves_of_short_and_long_rings_fp64(N, M):
    """levy_propose and com_propose against the oracle.  A COM try's scratch is
    M (2 x 8 + 4 x 8) bytes: 1365 slices fit 64 KiB, 1366 do not.  The four
    weights are sums of M terms of one sign, each good to a few roundings:
    M 1e-15 of the sum."""
    rng = np.random.default_rng(N * 10000 + M)
    L = 4.0
    d = chain_desc(HarmonicTrap(0.7), dim=2, M=M, N=N, L=L, beta=2.0, lam=0.5, pair=GaussianPair(1.0, 0.5), r_a=2.0)
    r = np.clip(rng.normal(0, 0.5, size=(N, 2, 1)) + rng.normal(0, 0.1, size=(N, 2, M)), -3.9, 3.9)
    ctx = make_ctx([d], A.FP64)
    ctx.set_paths(0, r)
    osys = oracle_sys(d, r)

    def check(got, want):
        (r_gpu, w_gpu), (r_or, w_or) = got, want
        assert np.max(np.abs(r_gpu - r_or)) < 1e-12 * M
        for x, y in zip(w_gpu, (w_or.wV_initial, w_or.wV_updated, w_or.wU_initial, w_or.wU_updated)):
            assert abs(x - y) <= max(1e-13, M * 1e-15 * abs(y)), (x, y)

    for m in sorted({2, 3, M - 1, M}):
        j0 = int(rng.integers(M))
        nrm = rng.standard_normal((m - 1, 2))
        check(ctx.levy_propose(0, N - 1, j0, m, nrm),
              osys.reshape_propose(N - 1, j0, m, nrm))
    disp = rng.uniform(-0.5, 0.5, size=2)
    check(ctx.com_propose(0, 0, disp), osys.com_propose(0, disp))


@pytest.mark.parametrize("N,M", [(1, 4), (5, 7), (64, 513)])
def test_energy_and_adjoint_against_numpy_fp64(N, M):
    """64 x 513 beads of 8 lanes are more than the 1024 x 256 threads of the
    grid; 1 x 4 and 5 x 7 leave most lanes without a bead.  NumPy sums the same
    terms; each output is a sum of at most N M N terms, good to 1e-11 of the
    largest partial sum."""
    rng = np.random.default_rng(M)
    L, beta, g, sigma, w = 8.0, 2.0, 0.7, 0.5, 0.8
    d = chain_desc(HarmonicTrap(w), dim=2, M=M, N=N, L=L, beta=beta, lam=0.5, pair=GaussianPair(g, sigma), r_a=2.0)
    r = np.clip(rng.normal(0, 1.0, size=(N, 2, 1)) + rng.normal(0, 0.2, size=(N, 2, M)), -7.9, 7.9)
    ctx = make_ctx([d], A.FP64)
    ctx.set_paths(0, r)
    tau, h = beta / M, 2.0
    x = r.transpose(2, 0, 1)
    diff = x[:, :, None, :] - x[:, None, :, :]
    diff -= 2 * L * np.rint(diff / (2 * L))
    q = np.sum(diff ** 2, axis=-1)
    near = ((q <= h * h) & ~np.eye(N, dtype=bool)).astype(float)
    e, e1 = np.exp(-q / (2 * sigma ** 2)), np.exp(-np.roll(q, -1, 0) / (2 * sigma ** 2))
    SU = 0.5 * np.sum(near * 0.5 * tau * (e + e1))
    links = near + np.roll(near, 1, 0)
    grad = tau * w * w * x - np.sum((links * 0.5 * tau * g * e / sigma ** 2)[..., None] * diff, axis=2)
    r2 = np.sum(x ** 2)
    S, gr, par = ctx.adjoint(0)
    big = max(1.0, tau * r2, SU)
    assert abs(S - (tau * 0.5 * w * w * r2 + g * SU)) < 1e-11 * big
    assert np.max(np.abs(gr - grad.transpose(1, 2, 0))) < 1e-11 * max(1.0, np.max(np.abs(grad)))
    assert abs(par[0] - tau * w * r2) < 1e-11 * big and abs(par[1] - SU) < 1e-11 * big
    assert ctx.action(0) == S
    E, Ev, Ep, Evp = ctx.energy(0)
    osys = oracle_sys(d, r)
    (Eo, Evo), (Po, Pvo) = osys.energy(), osys.pair_energy()
    scale = d.dim * N / (2 * tau)
    assert abs(E - Eo) < 1e-11 * scale and abs(Ev - Evo) < 1e-11 * max(1.0, abs(Evo))
    assert abs(Ep - Po) < 1e-11 * max(1.0, abs(Po)) and abs(Evp - Pvo) < 1e-11 * max(1.0, abs(Pvo))
    assert abs(Ep - g * SU / beta) < 1e-11 * max(1.0, abs(Ep))
