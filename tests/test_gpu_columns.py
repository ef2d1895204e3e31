"""The column transforms (y and z passes) at every length class, against the CPU oracle: lengths of
one stage (8), two (16, 32), the run-time plans of each tile class (up to 256, 512 and 1024 cells),
512 and 1024 themselves; unforced and with the band forcing's modes added in the z pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BPD = [(1, 1, 2), (1, 4, 1), (2, 3, 40), (1, 40, 3), (1, 64, 2), (2, 1, 64), (1, 80, 1), (1, 1, 75), (1, 128, 1),
       (1, 1, 128), (5, 30, 27)]


@pytest.mark.parametrize("bpd", BPD)
@pytest.mark.parametrize("forced", [False, True])
def test_step(cup, oracle, bpd, forced):
    print(f"bpd={bpd} forced={forced}", flush=True)
    rng = np.random.default_rng(23)
    O = oracle.OracleSim(bpd)
    u = [rng.standard_normal(tuple(8 * b for b in reversed(bpd))).astype(np.float32).astype(np.float64)
         for _ in range(3)]
    O.set_velocity(*u)
    dt, nu = 1e-4, 0.01
    tke = 1.05 * 0.5 * sum(float((a * a).mean()) for a in u)
    O.timestep(dt, nu, spectral_forcing=forced, tke_target=tke if forced else 0.0)
    ref, p = O.velocity(), O.get("p")
    # the pressure's lowest modes carry the rounding of h^2/(2 dt) div u over the whole box
    # (forced: in FP64 only, because white noise holds next to nothing in the band, so the factor that
    # brings the energy to its target multiplies the FP32 rounding of the band's modes by hundreds)
    for precision, tol in ((8, 1e-11), (4, 2e-5))[:1 if forced else 2]:
        G = cup.Grid(bpd, precision=precision, decomposition="fused")
        G.set_velocity(*u)
        G.run_steps(1, nu=nu, fixed_dt=dt, spectral_forcing=forced, tke_target=tke)
        for a, b in zip(G.velocity(), ref):
            assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)
        assert np.linalg.norm(G.get("p") - p) < 10 * tol * np.linalg.norm(p)
