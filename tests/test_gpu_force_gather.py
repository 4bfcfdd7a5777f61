"""The tiled force gather at the edges of its tiles (GPU): every spline order, grids with narrow last tiles, odd
numbers of tiles per axis and rows that are not whole 16-byte units.

27 waters in a 2 nm box, FP64: the directional derivative of the energy by a central difference (h = 1e-5 nm: rounding
1e-16 x 1e4 kJ/mol / 1e-5 nm = 1e-7, truncation h^2 = 1e-10 relative) against the forces, to 1e-6 of their
norm along the direction.  FP32 forces against FP64's to 1e-5 relative RMS, as the mixed path's other tests.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = {4: (12, 16, 18), 5: (20, 21, 25), 6: (23, 30, 32), 7: (24, 27, 22), 8: (24, 25, 40)}


@pytest.mark.parametrize("order", [4, 5, 6, 7, 8])
def test_tiled_forces_are_the_energy_gradient(order):
    import pgm_jax_amd as P

    sys_, pos, H = P.models.water_box(27, 2.0, seed=order)
    pos = np.asarray(pos)
    print(f"force gather order {order}", flush=True)

    def ff(precision, tol):
        s = P.MDSettings(precision=precision, cutoff=0.55, skin=0.05, ewald_beta=5.0, pme_order=order, pme_grid=GRIDS[order],
                         dipole_tol=tol)
        return P.PGMForceField(sys_, H, s)

    f64 = ff("double", 1e-11)
    r = f64.compute(pos, H)
    F = r.forces.cpu().numpy()
    d = np.random.default_rng(order).standard_normal(pos.shape)
    d /= np.linalg.norm(d)
    h = 1e-5
    ep, em = (float(f64.compute(pos + k * h * d, H).energy["total"]) for k in (1, -1))
    assert abs((ep - em) / (2 * h) + np.sum(F * d)) <= 1e-6 * np.linalg.norm(F)
    F32 = ff("mixed", 1e-7).compute(pos, H).forces.cpu().numpy()
    assert np.sqrt(np.mean((F32 - F) ** 2)) <= 1e-5 * np.sqrt(np.mean(F**2))
