"""The density and multipole phase in one launch (small contexts) against its two separate
launches (more instances of the same system): the same sums in the same order, so the potential
is the same bit for bit.

Sizes: whole and partial tiles of radial nodes and multipoles, odd and even N_theta, more theta
nodes than one round of 36 per wave, no more orbitals than one round of loads and more."""
import numpy as np
import pytest

from ggbtddft_amd.system import AtomSystem

pytestmark = pytest.mark.gpu


def _run(S, psi, n, precision):
    from ggbtddft_amd.engine import Propagator
    with Propagator(S, n_inst=n, precision=precision) as prop:
        prop.set_field(np.full((n, 3), 0.05))
        prop.upload_orbitals(np.ascontiguousarray(np.tile(psi, (1, n, 1))))
        return prop.download_potential()


# (atom, N, l_max, N_theta): `few` instances take one launch, `many` two (panel form from 8 on)
@pytest.mark.parametrize("atom, N, lmax, n_theta, few, many", [
    ("Ar", 80, 40, 81, 1, 8), ("Ar", 75, 40, 82, 2, 9), ("Ar", 203, 48, 97, 1, 3), ("Ne", 161, 64, 160, 1, 3),
    ("He", 97, 12, 25, 4, 80)])
@pytest.mark.parametrize("precision", [0, 1])
def test_one_launch_equals_two(atom, N, lmax, n_theta, few, many, precision):
    print("case: density and moments,", atom, N, lmax, n_theta, precision, flush=True)
    S = AtomSystem(atom, N, 40.0, lmax, 0.05, n_theta=n_theta, ground_state="device", tables="device")
    psi = S.psi0.copy()
    rng = np.random.default_rng(N)
    psi[1:4] += 0.1 * rng.standard_normal(psi[1:4].shape) * np.exp(-S.grid.r)
    for k in range(S.n_orb):
        psi[:S.m[k], k] = 0.0
    one = _run(S, psi, few, precision)
    two = _run(S, psi, many, precision)
    assert np.abs(one).max() > 1e-3
    assert all(np.array_equal(v, one[0]) for v in one)
    assert all(np.array_equal(v, one[0]) for v in two)
