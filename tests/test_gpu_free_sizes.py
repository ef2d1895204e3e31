"""PoissonSolverUnbounded over the length classes of its padded transforms (up to 256, 512 and 1024
points; powers of two and not), against the CPU oracle's direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bpd", [(1, 1, 1), (3, 2, 1), (20, 1, 2), (1, 32, 1), (2, 1, 40), (1, 1, 64), (64, 1, 1)])
@pytest.mark.parametrize("precision", [8, 4])
def test_solve(cup, oracle, bpd, precision):
    print(f"bpd={bpd} precision={precision}", flush=True)
    rng = np.random.default_rng(41)
    bc = ("freespace",) * 3
    G = cup.Grid(bpd, maxextent=1.0, precision=precision, decomposition="plain", bc=bc)
    O = oracle.OracleSim(bpd, maxextent=1.0, bc=bc)
    u = [rng.standard_normal(G.shape).astype(np.float32).astype(np.float64) for _ in range(3)]
    G.set_velocity(*u)
    O.set_velocity(*u)
    for _ in range(2):  # the second solve finds the first one's spectrum in its buffers
        G.pressure_rhs(1e-3); G.poisson_unbounded()
    O.pressure_rhs(1e-3); O.poisson_unbounded()
    a, b = G.get("p"), O.get("p")
    # two transforms of up to 2^30 points (30 roundings each way) and the direct sum's own rounding
    tol = 100 * (1.1e-16 if precision == 8 else 6e-8) * 10
    assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)
