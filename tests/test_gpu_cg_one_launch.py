"""The CG update at the sizes where its launch changes (GPU): one launch with one or two atoms per thread, or two launches.

A bead of up to 1,023 atoms (341 waters) keeps one atom per thread, up to 2,046 (682 waters) two, and from 2,049 on
the two kernels run.  FP64: the solved dipoles are put into the induction equation mu = alpha E(p + mu), with E from the
field evaluation and no part of the CG kernels: the largest component of the difference over the mean of |alpha E(p)| is
what the solve's tolerance bounds, up to what the residual updated along the way loses against the true one (twice the
tolerance, 1e-9).  FP32: the dipoles against those of the FP64 solve, 1e-5 relative RMS (the preconditioners' own test).
Two beads must repeat the single contexts' iterations and dipoles (FP64 1e-10, FP32 1e-6, the bounds of the beads' own
test).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel_rms(a, b):
    return float(np.sqrt(np.mean((a - b) ** 2)) / np.sqrt(np.mean(b**2)))


@pytest.mark.parametrize("precond", ["jacobi", "molecule"])
@pytest.mark.parametrize("n", [341, 342, 682, 683])
def test_solution_and_beads(n, precond):
    import pgm_jax_amd as P

    edge = (n / 33.0) ** (1.0 / 3.0)
    sys_, pos, H = P.models.water_box(n, edge, seed=n)
    q = np.stack([pos, P.models.water_box(n, edge, seed=n + 1)[1]])
    alpha = np.asarray(sys_.alpha)[:, None]
    wide = []
    for precision, tol in (("double", 1e-9), ("mixed", 1e-7)):
        print(f"CG update {n} {precision} {precond}", flush=True)
        s = P.MDSettings(precision=precision, precond=precond, dipole_tol=tol, max_iter=200, cutoff=0.8, skin=0.05, ewald_beta=4.5,
                         pme_grid=(32,) * 3)
        singles = []
        for b, x in enumerate(q):
            ff = P.PGMForceField(sys_, H, s)
            r = ff.compute(x, H)
            assert r.residual <= tol
            mu = r.induction.mu.cpu().numpy()
            if precision == "double":
                p = ff.perm_dipoles(x).cpu().numpy()
                res = alpha * ff.field(x, p + mu).cpu().numpy() - mu
                assert np.abs(res).max() <= 2.0 * tol * np.abs(alpha * ff.field(x, p).cpu().numpy()).mean()
                wide.append(mu)
            else:
                assert _rel_rms(mu, wide[b]) <= 1e-5
            singles.append((r.iterations, mu))
        beads = P.PGMBeads(sys_, H, s, beads=2)
        _, _, e = beads.compute(q, H)
        mu, its = e.induction.mu.cpu().numpy(), beads.bead_results()[1]
        for b in range(2):
            assert its[b] == singles[b][0]
            assert _rel_rms(mu[b], singles[b][1]) <= (1e-10 if precision == "double" else 1e-6)
