"""PoissonSolverUnbounded over the length classes of its padded transforms (up to 256, 512 and 1024
points; powers of two and not), against the CPU oracle's direct sum."""
import hashlib

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


# SHA-256 of p's bytes after the solve below, from the solve that pads the RHS, transforms the whole
# padded grid and multiplies the spectrum in a pass of its own: every length class of its passes along
# y and z (16, 48, 64, 128, 256, 320, 512, 640 and 1024 points).
BITS = {
    ((1, 1, 1), 4): "5b0862b10dbd842b",
    ((1, 1, 1), 8): "79e96ba26c892b70",
    ((3, 3, 2), 4): "1f2a0c725304a8a0",
    ((3, 3, 2), 8): "49c60b3df66a14f6",
    ((2, 4, 4), 4): "d90445e6fb664e99",
    ((2, 4, 4), 8): "0eeade553fe402fb",
    ((4, 8, 8), 4): "a0b857437d7e1e95",
    ((4, 8, 8), 8): "425d92b04e208035",
    ((1, 16, 16), 4): "75e03d036fc80bbe",
    ((1, 16, 16), 8): "09f0c0a3483f4baf",
    ((6, 20, 1), 4): "48599499368ed908",
    ((6, 20, 1), 8): "e3b06985bb37cb21",
    ((1, 32, 1), 4): "2966ec3cb8b00308",
    ((1, 32, 1), 8): "4d2a1766dd95df7c",
    ((1, 1, 32), 4): "4d77eefd1f67d666",
    ((1, 1, 32), 8): "c7567cef656c5fa9",
    ((1, 40, 1), 4): "60a8d6f09a5786fd",
    ((1, 40, 1), 8): "b366840036619458",
    ((1, 1, 40), 4): "ccd86289f1dfb6a5",
    ((1, 1, 40), 8): "9a3cb420af23e06b",
    ((1, 64, 1), 4): "ed7af0150a6d21e7",
    ((1, 64, 1), 8): "1163df74098f50c6",
    ((1, 1, 64), 4): "5f0f20a34f14e2c5",
    ((1, 1, 64), 8): "b0da1a780a766d8f",
    ((20, 1, 4), 4): "f32968f28f4bbd66",
    ((20, 1, 4), 8): "212ad94f2cfd3bc0",
}


@pytest.mark.parametrize("bpd,precision", sorted(BITS))
def test_bits_of_the_whole_grid_solve(cup, bpd, precision):
    print(f"bpd={bpd} precision={precision}", flush=True)
    assert _digest(cup, bpd, precision) == BITS[bpd, precision]


def _digest(cup, bpd, precision):
    rng = np.random.default_rng(43)
    G = cup.Grid(bpd, maxextent=1.0, precision=precision, decomposition="plain", bc=("freespace",) * 3)
    G.set_velocity(*[rng.standard_normal(G.shape) for _ in range(3)])
    for _ in range(2):
        G.pressure_rhs(1e-3); G.poisson_unbounded()
    p = G.get("p").astype(np.float32 if precision == 4 else np.float64) + 0  # one sign of zero
    return hashlib.sha256(p.tobytes()).hexdigest()[:16]


@pytest.mark.parametrize("bpd", [(2, 3, 1), (4, 4, 4), (8, 4, 8), (2, 16, 3), (1, 2, 32), (5, 20, 2), (1, 40, 1), (2, 1, 64)])
def test_error_of_one_fp32_solve(cup, oracle, bpd):
    """The solve alone: velocities of small whole numbers with h and dt powers of two, so that the RHS is
    the oracle's exactly. Up to 60 stages of transforms, each with a relative error of 6e-8 at random,
    leave sqrt(60) 6e-8 = 4.6e-7 in norm; twice that."""
    print(f"bpd={bpd}", flush=True)
    rng = np.random.default_rng(47)
    bc, ext = ("freespace",) * 3, 8 * max(bpd) / 64
    G = cup.Grid(bpd, maxextent=ext, precision=4, decomposition="plain", bc=bc)
    O = oracle.OracleSim(bpd, maxextent=ext, bc=bc)
    u = [rng.integers(-4, 5, G.shape).astype(np.float64) for _ in range(3)]
    G.set_velocity(*u)
    O.set_velocity(*u)
    G.pressure_rhs(2.0 ** -10); G.poisson_unbounded()
    O.pressure_rhs(2.0 ** -10); O.poisson_unbounded()
    a, b = G.get("p"), O.get("p")
    assert np.linalg.norm(a - b) < 9.2e-7 * np.linalg.norm(b)
