"""The fused reciprocal transform on grids with factors 3 and 5 against the library plans (GPU).

Axes 2^k times 1, 3, 5 and 15 in every position (radix-3 and radix-5 stages after the powers of two, real
lines of odd half length: 30 = 2 x 15), single systems and beads: the field of 216 waters with the fused
kernels against the library transform, FP64 to 1e-12 and FP32 to 2e-6 relative RMS (the bounds of the
power-of-two grids); other factors stay with the library.  Of two beads the energies and forces after their own
solves, which add the CG tolerance: FP64 to 1e-11 and 1e-9, FP32 to 1e-6 and 1e-4.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(24, 32, 40), (48, 24, 30), (40, 60, 24), (30, 40, 48), (60, 48, 32), (32, 30, 80)]


@pytest.mark.parametrize("precision,tol", [("double", 1e-11), ("mixed", 1e-6)])
@pytest.mark.parametrize("grid", [(60, 48, 30), (24, 40, 32)])
def test_fused_transform_of_beads(grid, precision, tol):
    """Two different beads in one call, fused against library: each bead's planes, columns and energy partials are its own."""
    import pgm_jax_amd as P

    sys_, pos, H = P.models.water_box(216, 1.87, seed=2)
    q = np.stack([pos, P.models.water_box(216, 1.87, seed=5)[1]])
    print(f"fused transform of beads {grid} {precision}", flush=True)
    res = {}
    for transform in ("fused", "library"):
        beads = P.PGMBeads(sys_, H, P.MDSettings(precision=precision, cutoff=0.8, skin=0.05, ewald_beta=4.0, pme_grid=grid,
                                                 dipole_tol=1e-10 if precision == "double" else 1e-7), beads=2)
        beads.set_pme_transform(transform)
        forces, _, _ = beads.compute(q, H)
        res[transform] = forces.cpu().numpy(), beads.bead_results()[0]
    for b in range(2):
        (F, e), (G, g) = ((r[0][b], r[1][b]) for r in (res["fused"], res["library"]))
        assert abs(e["total"] - g["total"]) <= tol * abs(g["total"]), b
        assert np.sqrt(np.mean((F - G) ** 2)) <= 100 * tol * np.sqrt(np.mean(G**2)), b


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("mixed", 2e-6)])
@pytest.mark.parametrize("grid", GRIDS)
def test_fused_transform_with_factors_3_and_5(grid, precision, tol):
    import pgm_jax_amd as P

    sys_, pos, H = P.models.water_box(216, 1.87, seed=2)
    print(f"fused transform {grid} {precision}", flush=True)
    ff = P.PGMForceField(sys_, H, P.MDSettings(precision=precision, cutoff=0.8, skin=0.05, ewald_beta=4.0, pme_grid=grid))
    assert ff.pme_transform() == ("fused", True)
    d = np.random.default_rng(1).normal(scale=0.01, size=pos.shape)
    f = ff.field(pos, d).cpu().numpy()
    e, F = ff.energy_forces(pos, d)
    ff.set_pme_transform("library")
    g = ff.field(pos, d).cpu().numpy()
    el, Fl = ff.energy_forces(pos, d)
    assert np.sqrt(np.mean((f - g) ** 2)) <= tol * np.sqrt(np.mean(g**2))
    assert abs(e["total"] - el["total"]) <= (1e-11 if precision == "double" else 1e-7) * abs(el["total"])
    F, Fl = F.cpu().numpy(), Fl.cpu().numpy()
    assert np.sqrt(np.mean((F - Fl) ** 2)) <= 10 * tol * np.sqrt(np.mean(Fl**2))


def test_other_factors_keep_the_library_transform():
    import pgm_jax_amd as P

    sys_, _, H = P.models.water_box(216, 1.87, seed=2)
    for grid in ((72, 32, 32), (32, 50, 32), (32, 32, 28), (45, 32, 32)):
        ff = P.PGMForceField(sys_, H, P.MDSettings(cutoff=0.8, skin=0.05, pme_grid=grid))
        assert ff.pme_transform() == ("library", False), grid
