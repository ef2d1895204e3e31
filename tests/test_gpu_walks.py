"""The stencil kernels' walks at the block counts where their length changes (1, 2, 4 or 8 blocks
along x in the advection, 1, 2 or 4 along z in the gradient), against the CPU oracle: one fused
step from a random field, FP64 to 1e-12 and FP32 to 2e-6 (the step's rounding, as elsewhere)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bpd", [(8, 8, 8), (8, 16, 8), (8, 16, 16), (16, 16, 16), (3, 16, 32), (6, 12, 10)])
@pytest.mark.parametrize("scheme", [0, 2])
def test_step(cup, oracle, bpd, scheme):
    print(f"bpd={bpd} scheme={scheme}", flush=True)
    rng = np.random.default_rng(17)
    O = oracle.OracleSim(bpd)
    u = [rng.standard_normal(tuple(8 * b for b in reversed(bpd))).astype(np.float32).astype(np.float64)
         for _ in range(3)]
    O.set_velocity(*u)
    dt, nu = 2e-3, 0.01
    O.advect_diffuse(dt, nu, (0, 0, 0), scheme=scheme)
    O.pressure_rhs(dt); O.poisson(); O.grad_p(dt)
    ref = O.velocity()
    for precision, tol in ((8, 1e-12), (4, 2e-6)):
        G = cup.Grid(bpd, precision=precision, decomposition="fused")
        G.set_velocity(*u)
        G.run_steps(1, nu=nu, fixed_dt=dt, scheme=scheme)
        for a, b in zip(G.velocity(), ref):
            assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)
