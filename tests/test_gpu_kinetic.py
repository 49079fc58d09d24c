"""The kinetic passes at the edges of their tiles, against numpy.

One kinetic sub-step of random orbitals is psi_l -> Q_l e^{-i lam dt} Q_l^T psi_l.  Each
pass is a sum of at most N products, so an element of the result is off by at most
about 2 N eps times the norm of its column (|Q rows|, |Q columns| <= 1); the test allows
4 N eps."""
import numpy as np
import pytest

from ggbtddft_amd.system import AtomSystem

pytestmark = pytest.mark.gpu
_systems = {}


def _system(N):
    if N not in _systems:
        _systems[N] = AtomSystem("He", N, 30.0, 4, 0.05)
    return _systems[N]


def _random_columns(S, n):
    rng = np.random.default_rng(n)
    psi = rng.standard_normal((S.n_l, n, S.N)) + 1j * rng.standard_normal((S.n_l, n, S.N))
    return psi / np.linalg.norm(psi, axis=2, keepdims=True)


def _kinetic(S, psi):
    out = np.empty_like(psi)
    for l in range(S.n_l):
        Q, lam = S.Q[l, :, :S.nkeep[l]], S.lam[l, :S.nkeep[l]]
        out[l] = ((psi[l] @ Q) * np.exp(-1j * S.dt * lam)) @ Q.T
    return out


# radial nodes: whole blocks of 8, a remainder, odd, below one 32-row panel; columns:
# one tile (full, partial), a second tile, a last group with one tile left, 64-row panels
@pytest.mark.parametrize("N", [96, 75, 52, 21])
@pytest.mark.parametrize("columns", [1, 8, 9, 17, 33, 41])
def test_fp64_passes_at_tile_edges(N, columns):
    print("case: FP64 kinetic passes, N", N, "columns", columns, flush=True)
    from ggbtddft_amd.engine import Propagator
    S = _system(N)
    psi = _random_columns(S, columns)
    ref = _kinetic(S, psi)
    for variant in ("default", "narrow"):
        with Propagator(S, n_inst=columns) as prop:
            prop.set_field(np.zeros(1))
            prop.set_kinetic_variant(variant)
            prop.upload_orbitals(psi)
            prop.substep(1)
            got = prop.download_orbitals()
        assert np.abs(got - ref).max() < 4 * N * 2.0 ** -53, (variant, np.abs(got - ref).max())
