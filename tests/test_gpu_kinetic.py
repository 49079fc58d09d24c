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


def _mixed(S, psi, columns, variant):
    from ggbtddft_amd.engine import Propagator
    with Propagator(S, n_inst=columns, precision=1) as prop:
        prop.set_field(np.zeros(1))
        prop.set_kinetic_variant(variant)
        prop.upload_orbitals(psi)
        prop.substep(1)
        return prop.download_orbitals()


# The mixed form at the edges of its few-column kernel (9 to 40 columns) and just outside it.  Its
# columns are independent and every shape forms the same sums in the same order, so a column's
# result is the same bit for bit whatever the number of columns.  Against numpy: the ground-state
# component is advanced in FP64, the remainder (norm <= 1) in FP32 with chunk sums of 16, tables
# and columns rounded once: 2 (rounding of both operands) + 16 + N / 16 roundings per pass at most,
# two passes, so 4 (18 + N / 16) eps32.
@pytest.mark.parametrize("N", [96, 75, 52, 21])
def test_mixed_passes_at_tile_edges(N):
    print("case: mixed kinetic passes, N", N, flush=True)
    S = _system(N)
    psi = _random_columns(S, 48)
    ref = _kinetic(S, psi)
    wide = _mixed(S, psi, 48, "tiled16")
    assert np.abs(wide - ref).max() < 4 * (18 + N / 16) * 2.0 ** -24
    for columns in (40, 33, 17, 9):
        got = _mixed(S, psi[:, :columns].copy(), columns, "tiled16")
        assert np.array_equal(got, wide[:, :columns]), (columns, np.abs(got - wide[:, :columns]).max())


def test_mixed_passes_large_shapes():
    """The 2 x 2 and 4 x 1 tile shapes, which a pass with many output tiles takes (N = 330, 128 l, 12 to 40 columns)."""
    print("case: mixed kinetic passes, 2 x 2 and 4 x 1 tiles", flush=True)
    S = AtomSystem("Ne", 330, 60.0, 127, 0.05, ground_state="device", tables="device")
    rng = np.random.default_rng(5)
    psi = rng.standard_normal((S.n_l, 44, S.N)) + 1j * rng.standard_normal((S.n_l, 44, S.N))
    psi /= np.linalg.norm(psi, axis=2, keepdims=True)

    def run(inst):
        return _mixed(S, np.ascontiguousarray(psi[:, :4 * inst]), inst, "tiled16")
    wide = run(11)
    assert np.abs(wide - _kinetic(S, psi)).max() < 4 * (18 + S.N / 16) * 2.0 ** -24
    for inst in (10, 4, 3):
        got = run(inst)
        assert np.array_equal(got, wide[:, :4 * inst]), inst


@pytest.mark.parametrize("N", [80, 75])
def test_mixed_passes_many_columns(N):
    """More than 40 columns: a pass with fewer than 240 tiles of 64 x 128 (448 columns and 33 l
    here, or partly filled tiles) takes the small tiles, one with more full ones (512 columns) the large ones."""
    print("case: mixed kinetic passes, many columns, N", N, flush=True)
    S = AtomSystem("He", N, 30.0, 32, 0.05)
    psi = _random_columns(S, 512)
    wide = _mixed(S, psi, 512, "tiled16")
    assert np.abs(wide - _kinetic(S, psi)).max() < 4 * (18 + N / 16) * 2.0 ** -24
    for columns in (448, 300, 67, 41):
        got = _mixed(S, psi[:, :columns].copy(), columns, "tiled16")
        assert np.array_equal(got, wide[:, :columns]), columns


# The tables that the upload rounds to FP32 and packs for the narrow pass 2, at sizes with partial blocks of
# 64 nodes and of 16 eigenvalues.  A wave sums up to N / 8 products in FP32, eight waves' sums are added
# in FP64: 2 + N / 8 roundings a pass at most.
@pytest.mark.parametrize("N", [130, 96, 75, 21])
def test_mixed_tables_packed_at_upload(N):
    print("case: mixed tables, N", N, flush=True)
    S = _system(N)
    psi = _random_columns(S, 8)
    got = _mixed(S, psi, 8, "narrow")
    assert np.abs(got - _kinetic(S, psi)).max() < 4 * (18 + N / 8) * 2.0 ** -24


# 65 l and 70 to 300 columns: passes of 2000 to 7200 output tiles (64 rows by one column tile) and
# beyond (by two, the last group whole or with one tile left), with rows that end inside a panel
@pytest.mark.parametrize("N", [96, 75])
@pytest.mark.parametrize("columns", [71, 72, 240, 249])
def test_fp64_passes_larger_shapes(N, columns):
    print("case: FP64 kinetic passes, 65 l, N", N, "columns", columns, flush=True)
    from ggbtddft_amd.engine import Propagator
    if ("l", N) not in _systems:
        _systems["l", N] = AtomSystem("He", N, 30.0, 64, 0.05)
    S = _systems["l", N]
    psi = _random_columns(S, columns)
    ref = _kinetic(S, psi)
    got = {}
    for variant in ("default", "narrow"):
        with Propagator(S, n_inst=columns) as prop:
            prop.set_field(np.zeros(1))
            prop.set_kinetic_variant(variant)
            prop.upload_orbitals(psi)
            prop.substep(1)
            got[variant] = prop.download_orbitals()
    assert np.array_equal(got["default"], got["narrow"])
    assert np.abs(got["default"] - ref).max() < 4 * N * 2.0 ** -53


@pytest.mark.parametrize("lmax", [64, 95])
def test_mixed_passes_panel_shapes(lmax):
    """Small-tile passes of more than 4500 output tiles, with 1, 2 or 4 row tiles per wave by how
    full the last panel is (N = 150: 6 row tiles of 16 eigenvalues and 10 of nodes; N = 270: 11 and 17),
    against the large tiles of the same sums (more columns)."""
    print("case: mixed kinetic passes, panel shapes, l_max", lmax, flush=True)
    for N, few, many in ((150, 230, 512), (270, 60, 320)):
        S = AtomSystem("He", N, 60.0, lmax, 0.05, ground_state="device", tables="device")
        psi = _random_columns(S, many)
        wide = _mixed(S, psi, many, "tiled16")
        assert np.abs(wide - _kinetic(S, psi)).max() < 4 * (18 + N / 16) * 2.0 ** -24
        for columns in (few, few - 7, 34):
            got = _mixed(S, psi[:, :columns].copy(), columns, "tiled16")
            assert np.array_equal(got, wide[:, :columns]), (N, columns)


@pytest.mark.parametrize("N", [448, 453])
@pytest.mark.parametrize("columns", [1, 8])
def test_fp64_long_rows(N, columns):
    """One column tile on 448 rows and more: eight waves share the contraction of pass 0."""
    print("case: FP64 kinetic passes, long rows, N", N, "columns", columns, flush=True)
    from ggbtddft_amd.engine import Propagator
    S = AtomSystem("He", N, 100.0, 4, 0.05, ground_state="device", tables="device")
    psi = _random_columns(S, columns)
    with Propagator(S, n_inst=columns) as prop:
        prop.set_field(np.zeros(1))
        prop.upload_orbitals(psi)
        prop.substep(1)
        got = prop.download_orbitals()
    assert np.abs(got - _kinetic(S, psi)).max() < 4 * N * 2.0 ** -53
