"""The ground-state sweeps at the edges of their teams: one work-group alone, the smallest
team, a last work-group with few rows, odd sizes, and shells kept outside LDS (the largest
grids with many shells).

Without an independent iteration at these sizes the fixed point itself is checked with numpy:
the orbitals are eigenvectors of H[v_gs] and v_gs is the potential of their density.  The
iteration stops at |d eps| < 1e-11 and |v_out - v| < 1e-8, so v_gs is within a few 1e-8 of
the potential it was formed from, and <u|H|u> of eps to second order plus that first-order
change times the density: 1e-7 bounds both; the orbitals themselves converge no slower."""
import numpy as np
import pytest

from ggbtddft_amd.atoms import Atom
from ggbtddft_amd.grid import RadialGrid
from ggbtddft_amd.groundstate import spherical_potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sym,N,R", [("He", 17, 12.0), ("He", 143, 40.0), ("He", 144, 40.0),
                                     ("Ne", 161, 50.0), ("Kr", 255, 60.0), ("Xe", 1300, 200.0)])
def test_fixed_point_at_team_edges(sym, N, R):
    print("case: ground state teams", sym, N, flush=True)
    from ggbtddft_amd.groundstate import DeviceGroundState
    g, atom = RadialGrid(N, R), Atom(sym)
    gs = DeviceGroundState(g, atom)
    assert gs.converged
    u = gs.u.real
    occ = np.array([o for (_, _, o) in atom.shells])
    rho = occ @ (u * u)
    assert np.abs(rho - gs.rho_u).max() < 1e-12 * rho.max()
    v = spherical_potential(g, rho)
    assert np.abs(v - gs.v_gs).max() < 1e-10 * np.abs(v).max()
    for l in sorted(set(l for (_, l, _) in atom.shells)):
        idx = [s for s, (_, ll, _) in enumerate(atom.shells) if ll == l]
        assert np.abs(u[idx] @ u[idx].T - np.eye(len(idx))).max() < 1e-12
        lam = np.linalg.eigvalsh(g.hamiltonian(l, atom.Z, gs.v_gs))
        # eigvalsh is accurate to eps times the largest eigenvalue
        tol = 1e-7 + 4 * np.abs(lam).max() * 2.0 ** -52
        assert np.abs(gs.eps[idx] - lam[:len(idx)]).max() < tol
