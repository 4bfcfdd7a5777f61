"""The molecule-block records at the edges of their choices (GPU): their field against the atom rows'.

Sizes either side of the switch from four waves per molecule to one (2,048 molecules), sizes either side
of the row field's lane counts (32 or 16 per molecule; 32 beside the spread in one launch), and a box whose half is hardly more than the
cutoff, where the pairs of a molecule pair can have different lattice shifts; molecules whole and
wrapped into the box atom by atom.  Same sums in another order, FP64 to 1e-12 and FP32 to 1e-6 relative RMS
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
