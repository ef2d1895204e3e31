"""The stencil kernels' walks at the block counts where their length changes (1, 2, 4 or 8 blocks
along x in the advection and the diagnostics, 1, 2 or 4 along z in the gradient), against the CPU
oracle: one fused step from a random field, FP64 to 1e-12 and FP32 to 2e-6 (the step's rounding, as
elsewhere), and the advection and the diagnostics of boxes with faces."""
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


BCS = [("dirichlet", "wall", "periodic"), ("wall", "dirichlet", "dirichlet"), ("dirichlet",) * 3]


@pytest.mark.parametrize("bpd", [(8, 32, 16), (16, 12, 8), (8, 9, 12), (12, 8, 8), (9, 8, 5)])
@pytest.mark.parametrize("bc", BCS)
def test_advection_with_faces(cup, oracle, bpd, bc):
    """The advection's walks of 8, 2 and 1 blocks with open and wall faces, their fades and the inflow
    correction: FP64 to 1e-13 and FP32 to 2e-6, as elsewhere."""
    print(f"bpd={bpd} bc={bc}", flush=True)
    rng = np.random.default_rng(19)
    uinf, nu = (0.3, -0.2, 0.1), 0.01
    O = oracle.OracleSim(bpd, maxextent=1.0, bc=bc)
    u = [rng.standard_normal(tuple(8 * b for b in reversed(bpd))).astype(np.float32).astype(np.float64)
         for _ in range(3)]
    O.set_velocity(*u)
    dt = 4 * O.calc_max_timestep(0.3, nu, uinf)[0]  # a larger step makes the fades of order one
    O.advect_diffuse(dt, nu, uinf)
    ref = O.velocity()
    for precision, tol in ((8, 1e-13), (4, 2e-6)):
        G = cup.Grid(bpd, maxextent=1.0, precision=precision, decomposition="plain", bc=bc)
        G.set_velocity(*u)
        G.calc_max_timestep(0.3, nu, uinf)
        G.advect_diffuse(dt, nu, uinf)
        for a, b in zip(G.velocity(), ref):
            assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)


@pytest.mark.parametrize("bpd,bc", [((16, 16, 8), BCS[0]), ((16, 16, 8), ("periodic",) * 3), ((8, 32, 32), BCS[1]),
                                    ((6, 20, 18), BCS[2])])
def test_diagnostics(cup, oracle, bpd, bc):
    """Walks of 2 and 8 blocks in the diagnostics, periodic and with faces (FP64, 1e-12 as elsewhere)."""
    print(f"bpd={bpd} bc={bc}", flush=True)
    rng = np.random.default_rng(23)
    G = cup.Grid(bpd, maxextent=1.0, precision=8, decomposition="plain", bc=bc)
    O = oracle.OracleSim(bpd, maxextent=1.0, bc=bc)
    for n in ("u", "v", "w", "p"):
        f = rng.standard_normal(G.shape)
        G.set(n, f); O.set(n, f)
    chi = rng.uniform(0, 1, G.shape)
    G.set("chi", chi); O.set("chi", chi)
    a, b = G.diagnostics(0.02), O.dissipation(0.02)
    assert np.all(np.abs(a - b) <= 1e-12 * np.maximum(np.abs(b), 1e-3 * np.abs(b).max()))
