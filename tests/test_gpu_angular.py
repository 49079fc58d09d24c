"""The FP64 angular kernel of contexts with many tiles against that of contexts with few.

The same instances run as one batch (a wave per tile of 8 radial nodes) and in three parts (a
work-group per tile, which the other tests compare with the oracle).  An angular phase is two
products with orthonormal tables, sums of at most N_l and N_theta terms, so the two orders of
summation differ by at most about 2 (N_l + N_theta) eps times the norm of the column at each node; two
phases a step, over 3 steps: 12 (N_l + N_theta) eps, and four times that is allowed for the
potential that the differences feed back into.  Observables are sums with weights of at most
r_max (dipole), 1 / r_min^2 (acceleration) and 1 (norm)."""
import numpy as np
import pytest

from ggbtddft_amd.system import AtomSystem

pytestmark = pytest.mark.gpu

STEPS = 3


def _run(S, psi, E, active=None, graph=0):
    from ggbtddft_amd.engine import Propagator
    n = E.shape[0]
    with Propagator(S, n_inst=n) as prop:
        prop.set_field(E)
        prop.upload_orbitals(psi)
        if active is not None:
            prop.set_active(active)
        if graph:
            prop.set_graph(graph)
        obs = prop.run(0, STEPS)
        dv = prop.download_potential()
        prop._check(prop.lib.ggb_rebuild_potential(prop.ctx), "ggb_rebuild_potential")
        again = prop.download_potential()
        return obs, prop.download_orbitals(), dv, again


# N_l and N_theta: one row over the tiles of both (65 / 129, 33 / 65), whole tiles (64 / 128, 32 / 64),
# partial ones (47 / 93: 24 and 23 rows of a parity; 49 / 100; 33 / 67), an even N_theta with a row over (65 / 130)
@pytest.mark.parametrize("n_l, n_theta", [(65, 129), (65, 130), (64, 128), (49, 100), (47, 93), (33, 65), (33, 67),
                                          (32, 64), (24, 47)])
@pytest.mark.parametrize("N", [52, 49])
def test_wave_tiles_against_workgroup_tiles(n_l, n_theta, N):
    print("case: angular kernels, N_l", n_l, "N_theta", n_theta, "N", N, flush=True)
    S = AtomSystem("Ar", N, 30.0, n_l - 1, 0.05, n_theta=n_theta, ground_state="device", tables="device")
    n = 36  # 7 tiles x 7 orbitals each: 1764 tiles, and 588 in a third
    rng = np.random.default_rng(n_l + N)
    psi = rng.standard_normal((n_l, n * S.n_orb, S.N)) + 1j * rng.standard_normal((n_l, n * S.n_orb, S.N))
    for k in range(n * S.n_orb):
        psi[:S.m[k % S.n_orb], k] = 0.0  # l >= m
    psi /= np.sqrt((np.abs(psi) ** 2).sum(axis=(0, 2)))[None, :, None]
    E = 0.3 * rng.standard_normal((n, STEPS + 1))
    E[1] *= 1e7  # arguments of the sines beyond the series' range
    obs, got, dv, again = _run(S, psi, E)
    assert np.array_equal(dv, again)  # a rebuild reproduces the potential bit for bit
    tol = 48 * (n_l + n_theta) * 2.0 ** -53
    scale = {"dip": 30.0, "acc": 1 / S.grid.r.min() ** 2, "norm": 1.0}
    third = n // 3
    for part in range(0, n, third):
        cols = slice(part * S.n_orb, (part + third) * S.n_orb)
        ref_obs, ref, _, _ = _run(S, np.ascontiguousarray(psi[:, cols]), E[part:part + third])
        err = np.sqrt((np.abs(got[:, cols] - ref) ** 2).sum(axis=(0, 2))).max()
        assert err < tol, err
        for key, w in scale.items():
            d = np.abs(obs[key].reshape(STEPS, n, -1)[:, part:part + third] - ref_obs[key].reshape(STEPS, third, -1)).max()
            assert d < tol * w, (key, d)


def test_wave_tiles_idle_slots_and_graph():
    print("case: angular kernel with idle slots and from a graph", flush=True)
    S = AtomSystem("Ar", 52, 30.0, 48, 0.05, ground_state="device", tables="device")
    n = 36
    psi = np.ascontiguousarray(np.tile(S.psi0, (1, n, 1)))
    E = 0.1 * np.random.default_rng(2).standard_normal((n, STEPS + 1))
    obs, got, _, _ = _run(S, psi, E)
    active = np.ones(n, dtype=np.int32)
    active[5:9] = 0
    _, idle, _, _ = _run(S, psi, E, active=active)
    on = np.repeat(active, S.n_orb).astype(bool)
    assert np.array_equal(idle[:, on], got[:, on])
    obs_g, got_g, _, _ = _run(S, psi, E, graph=1)
    assert np.array_equal(got_g, got)
    for key in obs:
        assert np.array_equal(obs_g[key], obs[key]), key


@pytest.mark.parametrize("N, lmax, n_theta", [(75, 40, 81), (72, 40, 82), (77, 64, 129), (50, 12, 25)])
def test_mixed_one_and_two_tiles_per_workgroup(N, lmax, n_theta):
    """Mixed form: a context of few waves takes one angular tile per work-group, a larger one two.  The
    state and potential are the same bit for bit; observables are the same terms added in another
    order: 2 N eps of their weights each way at most."""
    from ggbtddft_amd.engine import Propagator
    print("case: mixed angular tiles, N", N, "l_max", lmax, flush=True)
    S = AtomSystem("Ar", N, 30.0, lmax, 0.05, n_theta=n_theta, ground_state="device", tables="device")
    E = 0.2 * np.random.default_rng(N).standard_normal(STEPS + 1)

    def run(n):
        with Propagator(S, n_inst=n, precision=1) as prop:
            prop.set_kinetic_variant("narrow")
            prop.set_field(np.tile(E, (n, 1)))
            obs = prop.run(0, STEPS)
            return obs, prop.download_orbitals(), prop.download_potential()
    few, many = run(1), run(50)
    assert np.array_equal(few[1], many[1][:, :S.n_orb])
    assert np.array_equal(few[2][0], many[2][0])
    scale = {"dip": 30.0, "acc": 1 / S.grid.r.min() ** 2, "norm": 1.0}
    for key, w in scale.items():
        d = np.abs(few[0][key].reshape(STEPS, 1, -1) - many[0][key].reshape(STEPS, 50, -1)).max()
        assert d <= 4 * N * 2.0 ** -53 * w, (key, d)
