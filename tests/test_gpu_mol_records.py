"""The molecule-block records at the edges of their choices (GPU): their field against the atom rows'.

Sizes either side of the switch from four waves per molecule to one (2,048 molecules), sizes either side
of the row field's lane counts (32 or 16 per molecule; 32 beside the spread in one launch), and a box whose half is hardly more than the
cutoff, where the pairs of a molecule pair can have different lattice shifts; molecules whole and
wrapped into the box atom by atom; cubic boxes and skewed ones, whose minimum image is taken axis by axis
(a molecule pair near half the box along z or y then shifts along x as well).  Same sums in another order, FP64 to 1e-12 and FP32 to 1e-6 relative RMS
(the row layouts' own test).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOXES = [(64, 1.243, 0.55, 0.05, 6.0, 32), (2047, 3.93, 0.7, 0.05, 5.0, 40), (2048, 3.93, 0.7, 0.05, 5.0, 40),
         (4097, 4.97, 0.6, 0.05, 5.0, 48), (8193, 6.26, 0.6, 0.05, 5.0, 64)]


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("n,edge,cutoff,skin,beta,grid", BOXES)
def test_records_against_atom_rows(n, edge, cutoff, skin, beta, grid, precision, tol):
    import pgm_jax_amd as P

    sys_, pos, H = P.models.water_box(n, edge, seed=n)
    print(f"records {n} {precision}", flush=True)
    ff = P.PGMForceField(sys_, H, P.MDSettings(precision=precision, cutoff=cutoff, skin=skin, ewald_beta=beta, pme_grid=(grid,) * 3))
    d = np.random.default_rng(3).normal(scale=0.01, size=pos.shape)
    for x in (pos, pos - np.floor(pos / edge) * edge):
        ff.set_row_layout("molecule", 4)
        f_mol = ff.field(x, d).cpu().numpy()
        ff.set_row_layout("atom")
        f_atom = ff.field(x, d).cpu().numpy()
        assert np.sqrt(np.mean((f_mol - f_atom) ** 2)) <= tol * np.sqrt(np.mean(f_atom**2))


# a reduced lower-triangular box: off-diagonal entries up to half the diagonal of their column
SKEWS = [((1.0, 1.02, 1.05), (0.48, -0.45, 0.49)), ((1.03, 0.99, 0.98), (0.15, -0.11, 0.2))]


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("diag,off", SKEWS)
@pytest.mark.parametrize("n,edge,cutoff,skin,beta,grid", [(64, 1.3, 0.45, 0.04, 6.0, 32), (1331, 3.5, 0.7, 0.05, 5.0, 40),
                                                          (2744, 4.4, 0.7, 0.05, 5.0, 48)])
def test_records_against_atom_rows_in_a_skewed_box(n, edge, cutoff, skin, beta, grid, diag, off, precision, tol):
    """Fractional coordinates of the cubic box in the skewed one, every molecule kept rigid (moved as a whole)."""
    import pgm_jax_amd as P

    sys_, pos, _ = P.models.water_box(n, edge, seed=n)
    H = edge * np.array([[diag[0], 0, 0], [off[0] * diag[0], diag[1], 0], [off[1] * diag[0], off[2] * diag[1], diag[2]]])
    print(f"records skewed {n} {precision}", flush=True)
    mols = np.asarray(pos).reshape(-1, 3, 3)
    centre = mols[:, :1]
    pos = (mols - centre + (centre / edge) @ H).reshape(-1, 3)
    ff = P.PGMForceField(sys_, H, P.MDSettings(precision=precision, cutoff=cutoff, skin=skin, ewald_beta=beta, pme_grid=(grid,) * 3))
    d = np.random.default_rng(3).normal(scale=0.01, size=pos.shape)
    whole, split = pos, pos - np.floor(pos @ np.linalg.inv(H)) @ H
    for x in (whole, split):
        ff.set_row_layout("molecule", 4)
        f_mol = ff.field(x, d).cpu().numpy()
        e_mol, F_mol = ff.energy_forces(x, d)
        ff.set_row_layout("atom")
        f_atom = ff.field(x, d).cpu().numpy()
        e_atom, F_atom = ff.energy_forces(x, d)
        assert np.sqrt(np.mean((f_mol - f_atom) ** 2)) <= tol * np.sqrt(np.mean(f_atom**2))
        F_mol, F_atom = F_mol.cpu().numpy(), F_atom.cpu().numpy()
        assert np.sqrt(np.mean((F_mol - F_atom) ** 2)) <= 10 * tol * np.sqrt(np.mean(F_atom**2))
        assert abs(e_mol["total"] - e_atom["total"]) <= tol * abs(e_atom["total"])
