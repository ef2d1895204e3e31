"""The HIT analysis where its waves' lines do not come out even, against the oracle: 10240 lines of
(ky, kz) take 3 lines per wave, a last wave of one line and idle waves behind it; 256 cells along x
take two strides of the 64 lanes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("tke", "eps", "uprime", "lambda", "Re_lambda", "l_integral", "tau_integral", "grad_mean", "grad_std")


@pytest.mark.parametrize("bpd", [(2, 10, 16), (32, 2, 2), (1, 1, 1)])
def test_analysis(cup, oracle, bpd):
    print(f"hit analysis bpd={bpd}", flush=True)
    rng = np.random.default_rng(31)
    G = cup.Grid(bpd, precision=8)
    O = oracle.OracleSim(bpd)
    u = tuple(rng.standard_normal(G.shape) for _ in range(3))
    G.set_velocity(*u)
    O.set_velocity(*u)
    rg, ro = G.hit_analysis(0.01), O.hit_analysis(0.01)
    for k in KEYS:
        assert rg[k] == pytest.approx(ro[k], rel=1e-11), k
    np.testing.assert_allclose(rg["E"], ro["E"], rtol=1e-11, atol=1e-14 * ro["E"].max())
