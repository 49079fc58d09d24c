"""Every shape that the dispatch rules choose, against another form of the same sums, bit for bit.
`ggb_debug_forms` says which forms run, so a rule that moves makes a test fail instead of
leaving it to compare a kernel with itself."""
import numpy as np
import pytest

from ggbtddft_amd import _lib
from ggbtddft_amd.engine import Propagator
from ggbtddft_amd.system import AtomSystem

pytestmark = pytest.mark.gpu
_systems = {}


def _forms(prop):
    f = np.zeros(5, dtype=np.int32)
    prop._check(prop.lib.ggb_debug_forms(prop.ctx, _lib.iptr(f)), "ggb_debug_forms")
    return f.tolist()


def _columns(S, n, seed):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal((S.n_l, n, S.N)) + 1j * rng.standard_normal((S.n_l, n, S.N))
    return psi / np.linalg.norm(psi, axis=2, keepdims=True)


def _advance(S, psi, precision, variant="default"):
    with Propagator(S, n_inst=psi.shape[1], precision=precision) as prop:
        prop.set_field(np.zeros(1))
        prop.set_kinetic_variant(variant)
        prop.upload_orbitals(np.ascontiguousarray(psi))
        prop.substep(1)
        return prop.download_orbitals(), _forms(prop)[:2]


def _numpy(S, psi):
    out = np.empty_like(psi)
    for l in range(S.n_l):
        Q, lam = S.Q[l, :, :S.nkeep[l]], S.lam[l, :S.nkeep[l]]
        out[l] = ((psi[l] @ Q) * np.exp(-1j * S.dt * lam)) @ Q.T
    return out


# Mixed form: the few-column kernel in each of its shapes against the 64 x 128 tiles (more columns of
# the same system).  Columns are independent and the sums have the same terms in the same order.
# N = 330 and 336 (whole blocks of 16, whose large tiles are copied straight to LDS): 19 row tiles of eigenvalues,
# 21 of nodes, so panels of two row tiles; 250: 13 and 16, panels of four; 75: few tiles, one row tile.  Column counts at the edges of one, two and more column tiles.
SMALL, R22, R21, R41, LARGE = 3411, 3422, 3421, 3441, 2000


@pytest.mark.parametrize("N, r_max, ecut, wide, cases", [
    (330, 60.0, 16.0, 64, [(9, R22), (12, R22), (16, R22), (17, R21), (24, R21), (33, R21), (40, R21)]),
    (336, 60.0, 16.0, 64, [(12, R22), (20, R21), (40, R21)]),
    (250, 60.0, 4.0, 64, [(17, R41), (23, R41), (40, R41)]),
    (75, 30.0, 1.0, 256, [(9, SMALL), (16, SMALL), (17, SMALL), (40, SMALL)])])
def test_mixed_few_column_shapes_against_large_tiles(N, r_max, ecut, wide, cases):
    S = AtomSystem("He", N, r_max, 127, 0.05, ecut_factor=ecut, ground_state="device", tables="device")
    psi = _columns(S, wide, N)
    print("case: mixed passes, N", N, "nk_max", S.nk_max, "columns", wide, flush=True)
    ref, forms = _advance(S, psi, 1, "tiled16")
    assert forms == [LARGE, LARGE]
    # the bound of the other mixed kinetic tests: 4 (18 + N / 16) roundings in FP32
    assert np.abs(ref - _numpy(S, psi)).max() < 4 * (18 + N / 16) * 2.0 ** -24
    for columns, shape in cases:
        print("case: mixed passes, N", N, "columns", columns, flush=True)
        got, forms = _advance(S, psi[:, :columns], 1, "tiled16")
        assert forms == [shape, shape], columns
        assert np.array_equal(got, ref[:, :columns]), columns


# FP64: every shape of four waves forms the same sums in the same order, so a column's result does not
# depend on how many others there are; eight waves (long rows, up to 8 columns) add in another order
@pytest.mark.parametrize("N, cases", [
    (448, [(8, 821, 421), (9, 441, 441), (16, 441, 441), (47, 442, 442)]),
    (330, [(8, 421, 421), (9, 441, 441), (17, 441, 441), (44, 441, 442), (50, 442, 442)])])
def test_fp64_shapes_against_each_other(N, cases):
    S = AtomSystem("He", N, 60.0, 64, 0.05, ecut_factor=8.0, ground_state="device", tables="device")
    psi = _columns(S, cases[-1][0], N)
    ref = None
    exact = _numpy(S, psi)
    for columns, f0, f1 in reversed(cases):
        print("case: FP64 passes, N", N, "nk_max", S.nk_max, "columns", columns, flush=True)
        got, forms = _advance(S, psi[:, :columns], 0)
        assert forms == [f0, f1], columns
        assert np.abs(got - exact[:, :columns]).max() < 4 * N * 2.0 ** -53
        if ref is None:
            ref = got
        elif f0 != 821:
            assert np.array_equal(got, ref[:, :columns]), columns


# The moments in the density's launch, in 16 x 16 tiles and in panels, and the potential in tiles
# and in panels: a context of instances with orbitals of their own against each instance alone.
@pytest.mark.parametrize("atom, N, lmax, n_theta, cases", [
    ("He", 96, 40, 81, [(8, 1, 2), (20, 2, 2), (70, 3, 3)]),
    ("Ar", 75, 40, 82, [(2, 1, 2), (18, 2, 2), (50, 3, 2), (90, 3, 3)])])
@pytest.mark.parametrize("precision", [0, 1])
def test_potential_forms_instance_by_instance(atom, N, lmax, n_theta, cases, precision):
    S = AtomSystem(atom, N, 40.0, lmax, 0.05, n_theta=n_theta, ground_state="device", tables="device")
    rng = np.random.default_rng(N)
    top = cases[-1][0]
    psi = np.concatenate([S.psi0] * top, axis=1)
    psi[:4] += 0.1 * rng.standard_normal((4,) + psi.shape[1:]) * np.exp(-S.grid.r)
    for k in range(psi.shape[1]):
        psi[:S.m[k % S.n_orb], k] = 0.0

    def run(first, n):
        with Propagator(S, n_inst=n, precision=precision) as prop:
            prop.set_field(np.full((n, 1), 0.05))
            prop.upload_orbitals(np.ascontiguousarray(psi[:, first * S.n_orb:(first + n) * S.n_orb]))
            return prop.download_potential(), _forms(prop)[2:4]
    print("case: potential forms,", atom, N, precision, flush=True)
    alone = []
    for k in range(top):
        v, forms = run(k, 1)
        assert forms == [1, 2]
        alone.append(v[0])
    assert np.abs(alone[0] - alone[1]).max() > 1e-6  # the instances differ
    for n, mom, dv in cases:
        print("case: potential forms,", atom, N, precision, "instances", n, flush=True)
        v, forms = run(top - n, n)
        assert forms == [mom, dv], n
        for k in range(n):
            assert np.array_equal(v[k], alone[top - n + k]), (n, k)
