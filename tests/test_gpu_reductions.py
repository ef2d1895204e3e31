"""The global reductions over grids whose partial sums take one workgroup, just more than one,
and many, on the GPU: the kinetic energy of the step loop and max |u| against numpy (FP64: sums
of up to 2^20 terms of one sign, 1e-13 of the sum; a maximum is exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# partials of the energy (4 per block): 8192 (the last of the one-workgroup form), 8640 and 9000
# (chunks of unequal length), 65536 (also several chunks of the 16384 maxima)
@pytest.mark.parametrize("bpd", [(16, 16, 8), (27, 4, 20), (15, 15, 10), (32, 32, 16)])
def test_energy_and_max(cup, bpd):
    print(f"bpd={bpd}", flush=True)
    rng = np.random.default_rng(5)
    G = cup.Grid(bpd, precision=8, decomposition="fused")
    u = [rng.standard_normal(G.shape) for _ in range(3)]
    G.set_velocity(*u)
    G.run_steps(0, CFL=0.3, nu=0.01)
    st = G.step_state()
    ke = 0.5 * G.h ** 3 * sum(float((a * a).sum()) for a in u)
    assert abs(st["ke"] - ke) < 1e-13 * ke
    assert st["umax"] == max(float(np.abs(a).max()) for a in u)
    assert G.max_velocity((0.5, -0.25, 0.125)) == max(float(np.abs(a + s).max())
                                                     for a, s in zip(u, (0.5, -0.25, 0.125)))
