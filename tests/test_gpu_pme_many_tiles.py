"""More tiles over the beads than one workgroup scans (GPU): the sites are then sorted by the library.

Eight beads of 27 waters on a 200^3 grid of order 6 (8 x 17,576 tiles, nearly all empty): every bead's forces and
energy equal its own single-system context, which scans its own tiles.  FP32 kernels: the same sums in the
same order per bead, so 1e-6 relative covers the two contexts' different launches.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_beads_beyond_the_scan():
    import pgm_jax_amd as P

    sys_, pos, H = P.models.water_box(27, 2.0, seed=4)
    rng = np.random.default_rng(2)
    q = np.stack([pos + rng.normal(scale=0.002, size=pos.shape) for _ in range(8)])
    s = P.MDSettings(precision="mixed", cutoff=0.8, skin=0.05, ewald_beta=4.0, pme_grid=(200, 200, 200), dipole_tol=1e-6)
    beads = P.PGMBeads(sys_, H, s, beads=8)
    f, _, _ = beads.compute(q, H)
    per = beads.bead_results()[0]
    for b in (0, 7):
        r = P.PGMForceField(sys_, H, s).compute(q[b], H)
        F, G = f[b].cpu().numpy(), r.forces.cpu().numpy()
        assert np.sqrt(np.mean((F - G) ** 2)) <= 1e-6 * np.sqrt(np.mean(G**2))
        assert abs(per[b]["total"] - r.energy["total"]) <= 1e-6 * abs(r.energy["total"])
