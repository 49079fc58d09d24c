"""A change of the kinetic variant leaves nothing of earlier orbitals behind.

The few-column mixed kernels lay out their intermediate Y differently from the others, which read
its padding as zeros.  Orbitals that hold a NaN pass through one variant; the next one then
advances new orbitals to the same bits as a context that never saw the NaN."""
import numpy as np
import pytest

from ggbtddft_amd.system import AtomSystem

pytestmark = pytest.mark.gpu
_systems = {}


def _system(N):
    if N not in _systems:
        _systems[N] = AtomSystem("He", N, 30.0, 4, 0.05)
        assert (_systems[N].nkeep % 16 != 0).any()  # there is padding
    return _systems[N]


def _advance(prop, psi):
    prop.upload_orbitals(psi)
    prop.substep(1)
    return prop.download_orbitals()


@pytest.mark.parametrize("N", [96, 75])
@pytest.mark.parametrize("columns", [9, 40])
@pytest.mark.parametrize("tuned", [False, True])
def test_nan_does_not_outlive_a_variant_change(N, columns, tuned):
    from ggbtddft_amd.engine import Propagator
    S = _system(N)
    rng = np.random.default_rng(columns)
    psi = rng.standard_normal((S.n_l, columns, N)) + 1j * rng.standard_normal((S.n_l, columns, N))
    psi /= np.linalg.norm(psi, axis=2, keepdims=True)
    for variant in ("narrow", "tiled32", "tiled16"):
        print("case: N", N, "columns", columns, "to", variant, "autotuned" if tuned else "", flush=True)
        got = []
        for spoil in (False, True):
            with Propagator(S, n_inst=columns, precision=1) as prop:
                prop.set_field(np.zeros(1))
                prop.set_kinetic_variant("tiled16")
                if spoil:
                    bad = _advance(prop, np.full_like(psi, np.nan))
                    assert np.isnan(bad).all()
                    if tuned:  # goes through every variant with the NaN in place
                        prop.autotune(1, cache=False)
                prop.set_kinetic_variant(variant)
                got.append(_advance(prop, psi))
        assert np.isfinite(got[0]).all()
        assert np.array_equal(got[0], got[1]), variant
