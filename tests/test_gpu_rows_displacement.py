"""pgm_rows_displacement, the list test of the Python mirror, against the norm of the differences.

Below 16384 atoms one workgroup takes the maximum, beyond it per-block maxima do; 3 atoms are the smallest
system, 16383 and 16386 lie on both sides of the line, and the atom that moves is the first or the last."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ask(ff, pos):
    from pgm_jax_amd import _lib

    d = C.c_double(-1.0)
    _lib.check(_lib.lib().pgm_rows_displacement(ff._ctx, C.c_void_p(pos.data_ptr()), C.byref(d)), "pgm_rows_displacement")
    return d.value


@pytest.mark.parametrize("nmol,edge", [(1, 2.0), (343, 2.2), (5461, 5.47), (5462, 5.47)])
def test_rows_displacement_is_the_largest_norm(nmol, edge):
    import torch

    import pgm_jax_amd as P

    sys_, x, H = P.models.water_box(nmol, edge, seed=3)
    print(f"displacement {nmol}", flush=True)
    ff = P.PGMForceField(sys_, H, P.MDSettings(cutoff=0.6, skin=0.05, ewald_beta=5.0, pme_grid=(48,) * 3))
    pos = torch.tensor(np.asarray(x), dtype=torch.float64, device="cuda").reshape(-1, 3).contiguous()
    assert _ask(ff, pos) == np.inf
    ff.build_rows(pos)
    assert _ask(ff, pos) == 0.0
    for atom in (0, 3 * nmol - 1):
        moved = pos + 0.001
        moved[atom] += torch.tensor([0.03, -0.04, 0.12], dtype=torch.float64, device="cuda")
        ref = torch.linalg.norm(moved - pos, dim=1).max().item()
        # three roundings of the squares and one of the root, on both sides: 4 eps
        assert abs(_ask(ff, moved) - ref) <= 4 * np.finfo(float).eps * ref


@pytest.mark.parametrize("nmol,edge", [(343, 2.2), (5462, 5.47)])
def test_rows_built_around_a_lost_atom_are_rebuilt(nmol, edge):
    """Rows built while a position was not a number lack that atom: the next proper positions ask for new rows."""
    import torch

    import pgm_jax_amd as P

    sys_, x, H = P.models.water_box(nmol, edge, seed=3)
    print(f"displacement, lost atom, {nmol}", flush=True)
    ff = P.PGMForceField(sys_, H, P.MDSettings(cutoff=0.6, skin=0.05, ewald_beta=5.0, pme_grid=(48,) * 3))
    pos = torch.tensor(np.asarray(x), dtype=torch.float64, device="cuda").reshape(-1, 3).contiguous()
    lost = pos.clone()
    lost[3 * nmol - 1] = float("nan")
    ff.build_rows(lost)
    assert _ask(ff, lost) == 0.0
    assert _ask(ff, pos) == np.inf
    ff.build_rows(pos)
    assert _ask(ff, lost) == 0.0
    assert _ask(ff, pos) == 0.0
