"""Spread and gather tiles at their edges (GPU): every spline order, grids with narrow last tiles, odd numbers
of tiles per axis and rows that are not whole 16-byte units, and tiles from empty to crowded.

203 sites in a skewed box: 70 within a fraction of one tile (several chunks of the matrix-core spread and
several rounds of the gather's lane pairs), the rest uniform.  Against the oracle's PME: FP64 to 1e-12
(Q) and 1e-10 (dU/dd) of the largest value; FP32 kernels to 1e-6 and 1e-5, as the PME object's own test.
"""

import numpy as np
import pytest

from oracle import pme as opme

pytestmark = pytest.mark.gpu

GRIDS = {4: (12, 13, 18), 5: (16, 21, 25), 6: (23, 30, 32), 7: (24, 27, 22), 8: (23, 24, 40)}


@pytest.mark.parametrize("dtype,tol_q,tol_g", [(np.float64, 1e-12, 1e-10), (np.float32, 1e-6, 1e-5)])
@pytest.mark.parametrize("order", [4, 5, 6, 7, 8])
def test_tiles_against_oracle(order, dtype, tol_q, tol_g):
    import pgm_jax_amd as P

    rng = np.random.default_rng(order)
    H = np.array([[2.0, 0, 0], [0.3, 2.1, 0], [-0.2, 0.4, 1.9]])
    u = rng.random((203, 3))
    u[:70] = 0.97 + 0.06 * u[:70]  # across the box corner
    pos = u @ H
    q = rng.normal(size=203)
    q[:70] *= 0.1
    d = 0.02 * rng.standard_normal((203, 3))
    grid, beta = GRIDS[order], 3.5
    print(f"tiles order {order} grid {grid} {np.dtype(dtype).name}", flush=True)
    ref = opme.PME(grid, order, beta)
    Gr, Sr = ref.influence(H), ref.setup(pos, H)
    pme = P.PME(grid, order, beta, dtype)
    S, G = pme.setup(pos, H), pme.influence(H)
    Q, Qr = pme.spread(S, q, d).cpu().numpy(), ref.spread(Sr, q, d)
    assert np.abs(Q - Qr).max() <= tol_q * np.abs(Qr).max()
    g, gr = pme.grad_dipoles(S, G, q, d).cpu().numpy(), ref.gradients(Sr, Gr, q, d)[0]
    assert np.abs(g - gr).max() <= tol_g * np.abs(gr).max()
