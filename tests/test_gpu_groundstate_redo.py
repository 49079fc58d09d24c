"""Ground-state sweeps whose work-groups give up waiting for each other: the group is done again from
the same start by one work-group, whose sums have the same terms in the same order, so every
result is the same bit for bit, whatever the phase in which the wait ran out.

The host names the phase (`ggb_debug_ground_state`): the wait counts as run out there, and every
kernel ends by itself."""
import ctypes

import numpy as np
import pytest

from ggbtddft_amd import _lib
from ggbtddft_amd.grid import RadialGrid

pytestmark = pytest.mark.gpu
SWEEPS = 2


def _run(N, R, Z, shell_l, max_iter, expire):
    """(u, eps, v_gs, rho_u, iterations, converged) of closed shells of the given l"""
    lib = _lib.load()
    g = RadialGrid(N, R)
    shell_l = np.array(shell_l, dtype=np.int32)
    occ = 2.0 * (2.0 * shell_l + 1.0)
    ls = sorted(set(shell_l.tolist()))
    lam0, Q0 = (np.ascontiguousarray(x) for x in zip(*(np.linalg.eigh(g.hamiltonian(l, Z)) for l in ls)))
    p = _lib.GsProblem(n_r=N, n_shell=len(shell_l), sweeps=SWEEPS, max_iter=max_iter, interacting=1, device=0,
                       Z=Z, mix=0.3, gamma=2.0, tol=1e-9)
    u, eps, v, rho = np.zeros((len(shell_l), N)), np.zeros(len(shell_l)), np.zeros(N), np.zeros(N)
    it, conv = np.zeros(1, dtype=np.int32), np.zeros(1, dtype=np.int32)
    d, i = _lib.dptr, _lib.iptr
    rc = lib.ggb_debug_ground_state(ctypes.byref(p), i(shell_l), d(occ), d(np.ascontiguousarray(g.r)),
                                    d(np.ascontiguousarray(g.wr)), d(np.ascontiguousarray(g.T)), d(Q0), d(lam0), d(u),
                                    d(eps), d(v), d(rho), i(it), i(conv), expire)
    _lib.check(rc, None, "ggb_debug_ground_state")
    return u, eps, v, rho, it[0], conv[0]


# neon-like and krypton-like shells, orbitals in LDS; 8 shells of one l on 960 nodes, where they are
# kept in device memory (13 vectors of 960 do not fit in 96 KB)
@pytest.mark.parametrize("N, R, Z, shell_l, max_iter", [(161, 50.0, 10.0, (0, 0, 1), 300),
                                                        (255, 60.0, 36.0, (0, 0, 1, 0, 1, 2, 0, 1), 300),
                                                        (960, 120.0, 60.0, (0,) * 8, 3)])
def test_a_team_that_gives_up_changes_no_bit(N, R, Z, shell_l, max_iter):
    ref = _run(N, R, Z, shell_l, max_iter, -1)
    k = max(shell_l.count(l) for l in shell_l)
    last = (SWEEPS - 1) * 4 * k  # first phase of the largest group's last sweep
    # the first phase of all; the last sweep's first shell, inside its second and its last one; the last phase
    for expire in (0, last, last + 5, last + 4 * (k - 1) + 2, last + 4 * k - 1):
        print("case: ground state", N, shell_l, "wait of phase", expire, "runs out", flush=True)
        got = _run(N, R, Z, shell_l, max_iter, expire)
        assert got[4] == ref[4] and got[5] == ref[5], expire
        for a, b in zip(got[:4], ref[:4]):
            assert np.array_equal(a, b), expire
