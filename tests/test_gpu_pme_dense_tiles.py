"""The lines between the two ways to bin the PME's atoms: counts per tile, or the library's sort.

A tile that may hold more than 256 atoms goes to the library: with 256 atoms in all, no tile can hold more; with 257 and
wide tiles it could.  So do grids of more than 20,000 tiles (here 21,952) with fewer than four atoms a tile.  Both ways sort
the atoms of a tile by index, so an atom more that has neither charge nor dipole changes nothing, bit for bit, though
it takes the call across the line.  Past the first line the cost per atom must not grow with the atoms per tile.
"""

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K, ORDER, BETA = (24, 27, 32), 6, 0.5


@pytest.mark.parametrize("dtype, tol", [(np.float32, 2e-6), (np.float64, 1e-12)])
def test_both_sorts_give_the_same_grid(dtype, tol):
    import torch

    import pgm_jax_amd as P
    from oracle import pme as opme

    rng = np.random.default_rng(4)
    n, H = 257, np.eye(3) * 20.0  # tiles of 6 nm and more
    pos = rng.uniform(0.0, 20.0, (n, 3))
    pos[:200] *= 0.2  # most atoms in a few tiles
    q, d = rng.normal(size=n), rng.normal(size=(n, 3)) * 0.1
    q[-1], d[-1] = 0.0, 0.0
    print(f"dense tiles {np.dtype(dtype).name}", flush=True)
    Q = []
    for m in (n - 1, n):
        pme = P.PME(K, ORDER, BETA, dtype=dtype)
        Q.append(pme.spread(pme.setup(pos[:m], H), q[:m], d[:m]))
    assert torch.equal(Q[0], Q[1])
    ref = opme.PME(K, ORDER, BETA)
    ref = ref.spread(ref.setup(pos, H), q, d)
    got = Q[1].cpu().numpy()
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)


def test_both_sorts_of_a_sparse_grid():
    import torch

    import pgm_jax_amd as P

    rng = np.random.default_rng(6)
    n, L = 4 * 21952, 21.6  # 28^3 tiles, in cubes of eight
    pos, d = rng.uniform(0.0, L, (n, 3)), rng.normal(size=(n, 3)) * 0.1
    d[-1] = 0.0
    print("sparse grid", flush=True)
    Q = []
    for m in (n - 1, n):
        pme = P.PME((224,) * 3, ORDER, 2.0)
        Q.append(pme.spread(pme.setup(pos[:m], np.eye(3) * L), np.zeros(m), d[:m]))
    assert torch.equal(Q[0], Q[1])
    assert torch.count_nonzero(Q[0]).item() > n


def test_cost_per_atom_does_not_grow_with_the_atoms_per_tile():
    import torch

    import pgm_jax_amd as P

    rng = np.random.default_rng(5)
    cost = {}
    for per_tile in (400, 6400):
        n = 216 * per_tile  # 48^3 points in tiles of 8^3
        L = (n / 100.0) ** (1.0 / 3.0)
        pme = P.PME((48, 48, 48), 6, 2.0)
        S = pme.setup(rng.uniform(0.0, L, (n, 3)), np.eye(3) * L)
        q, d = np.zeros(n), torch.tensor(rng.normal(size=(n, 3)) * 0.01, device="cuda")
        print(f"dense tiles, {per_tile} atoms each", flush=True)
        best = np.inf
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            pme.spread(S, q, d)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        cost[per_tile] = best / n
    assert cost[6400] <= 2.0 * cost[400], cost
