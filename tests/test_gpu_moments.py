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


@pytest.mark.parametrize("atom, N, lmax, n", [("Ar", 75, 40, 1), ("Ar", 75, 40, 9), ("Ne", 203, 48, 6), ("H", 50, 11, 3)])
def test_channel_dipoles_with_the_density(atom, N, lmax, n):
    """Channel dipoles from the launch of the density (one launch, two, and by itself without
    interaction), against numpy on the orbitals after the step; idle instances hold zero.  A sum of
    4 N products: 8 N eps of the sum of their sizes."""
    from ggbtddft_amd.engine import Propagator
    print("case: channel dipoles,", atom, N, lmax, n, flush=True)
    S = AtomSystem(atom, N, 40.0, lmax, 0.05, ground_state="device", tables="device")
    rng = np.random.default_rng(n)
    E = 0.3 * rng.standard_normal((n, 3))
    active = np.ones(n, dtype=bool)
    active[1:n - 1:3] = False
    with Propagator(S, n_inst=n) as prop:
        prop.set_field(E)
        prop.set_active(active)
        got = prop.run(0, 2, channels=True)["chan"][-1].reshape(n, S.n_orb, S.n_l)
        psi = prop.download_orbitals().reshape(S.n_l, n, S.n_orb, S.N)
    r = S.grid.r
    for k in range(S.n_orb):
        m = S.m[k]
        for l in range(S.n_l):
            if l < m:
                assert not got[:, k, l].any()
                continue

            def c(a):
                return np.sqrt(((a + 1) ** 2 - m * m) / ((2 * a + 1) * (2 * a + 3)))
            z = np.zeros((n, S.N), dtype=complex)
            size = np.zeros((n, S.N))
            for f, b in ((c(l), l + 1), (c(l - 1) if l > m else 0.0, l - 1)):
                if f and m <= b < S.n_l:
                    z += f * r * psi[b, :, k]
                    size += 2 * f * r * np.abs(psi[b, :, k])
            ref = (psi[l, :, k].conj() * z).sum(axis=1)
            tol = 8 * N * 2.0 ** -53 * (np.abs(psi[l, :, k]) * size).sum(axis=1)
            assert (np.abs(got[:, k, l] - ref)[active] <= tol[active]).all(), (k, l)
            assert not got[~active, k, l].any()


# panel and 16 x 16 forms of the two potential products, each against the other: instances below and
# beyond the tile counts at which either product changes (N_theta with 9, 7 and 13 tiles of 16)
@pytest.mark.parametrize("N, lmax, n_theta, counts", [(203, 64, 129, (2, 9, 11, 30)), (203, 48, 97, (5, 14, 30)),
                                                      (100, 96, 193, (1, 9, 30, 60))])
def test_potential_products_by_tiles(N, lmax, n_theta, counts):
    print("case: potential products, N", N, "l_max", lmax, "N_theta", n_theta, flush=True)
    S = AtomSystem("Ne", N, 40.0, lmax, 0.05, n_theta=n_theta, ground_state="device", tables="device")
    psi = S.psi0.copy()
    psi[1:4] += 0.1 * np.random.default_rng(N).standard_normal(psi[1:4].shape) * np.exp(-S.grid.r)
    for k in range(S.n_orb):
        psi[:S.m[k], k] = 0.0
    ref = _run(S, psi, counts[0], 0)[0]
    for n in counts[1:]:
        dv = _run(S, psi, n, 0)
        assert all(np.array_equal(v, ref) for v in dv), n
