"""PoissonSolverMixed's matrix-core transforms at the edges of their tiles, against the CPU
oracle: axes shorter than a tile of 16 and not a multiple of it, each number of lines per
workgroup, and the longest axis (whose tile takes 128 KiB of LDS in FP64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells per axis / 8. Lines per workgroup are chosen by the other axes' blocks: 16 below 256 of
# them, 32 from 256 (where the axis is short enough)
CASES = [
    ((1, 1, 1), ("dirichlet", "wall", "periodic")),
    ((3, 5, 9), ("periodic", "dirichlet", "wall")),
    ((16, 16, 2), ("wall", "periodic", "dirichlet")),
    ((32, 16, 5), ("dirichlet", "dirichlet", "wall")),
    ((128, 1, 1), ("dirichlet", "periodic", "wall")),
    ((1, 128, 1), ("wall", "wall", "periodic")),
    ((1, 2, 128), ("periodic", "wall", "dirichlet")),
]


@pytest.mark.parametrize("bpd,bc", CASES)
@pytest.mark.parametrize("precision", [8, 4])
def test_mixed_solve(cup, oracle, bpd, bc, precision):
    print(f"mixed solve bpd={bpd} bc={bc} precision={precision}", flush=True)
    rng = np.random.default_rng(11)
    G = cup.Grid(bpd, maxextent=1.0, precision=precision, decomposition="plain", bc=bc)
    O = oracle.OracleSim(bpd, maxextent=1.0, bc=bc)
    u = [rng.standard_normal(G.shape).astype(np.float32).astype(np.float64) for _ in range(3)]
    G.set_velocity(*u)
    O.set_velocity(*u)
    G.pressure_rhs(1e-3); G.poisson_mixed()
    O.pressure_rhs(1e-3); O.poisson_mixed()
    a, b = G.get("p"), O.get("p")
    # six contractions of up to 1024 terms: sqrt(6 * 1024) roundings of 1.1e-16 and 6e-8, with a
    # factor 10 for the symbol's amplification of the lowest modes
    tol = 10 * np.sqrt(6 * 1024) * (1.1e-16 if precision == 8 else 6e-8)
    assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)
