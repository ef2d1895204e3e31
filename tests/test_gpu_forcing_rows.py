"""cup_spectral_forcing's two ways of adding the band: from its modes, row by row (bands of few low
modes), and by filtering the spectra and transforming back (any other band), against the CPU oracle;
boxes of both kinds, with a mean flow (the kx = 0 slot's unpacking) and odd block counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the band 0 < |k|^2 <= 4: 32 modes or fewer with |kx| <= 2 in a 2 pi box, one axis only in flat
# boxes, up to |kx| = 4 in a 4 pi box
CASES = [((4, 4, 4), 2 * np.pi), ((3, 5, 2), 2 * np.pi), ((1, 1, 6), 2 * np.pi), ((5, 1, 2), 2 * np.pi),
         ((2, 9, 8), 2 * np.pi), ((4, 2, 2), 4 * np.pi), ((2, 4, 3), 4 * np.pi)]


@pytest.mark.parametrize("bpd,extent", CASES)
@pytest.mark.parametrize("decomposition", ["plain", "fused"])
def test_forcing(cup, oracle, bpd, extent, decomposition):
    print(f"bpd={bpd} extent={extent} {decomposition}", flush=True)
    rng = np.random.default_rng(31)
    O = oracle.OracleSim(bpd, maxextent=extent)
    G = cup.Grid(bpd, maxextent=extent, precision=8, decomposition=decomposition)
    x, y, z = np.meshgrid(*((np.arange(8 * b) + 0.5) * G.h for b in bpd), indexing="ij")
    low = [np.transpose(np.cos(2 * np.pi * (x / G.extent[0] + 2 * y / G.extent[1] - z / G.extent[2] + q)
                               ) + np.sin(2 * np.pi * (2 * x / G.extent[0] - y / G.extent[1] + q / 3)), (2, 1, 0))
           + np.transpose(np.sin(2 * np.pi * z / G.extent[2]) + np.cos(4 * np.pi * x / G.extent[0]), (2, 1, 0))
           for q in range(3)]
    u = [0.3 * q + a + 0.1 * rng.standard_normal(a.shape) for q, a in enumerate(low)]
    O.set_velocity(*u)
    G.set_velocity(*u)
    tke = 1.1 * 0.5 * sum(float((a * a).mean()) for a in u)
    ref = O.spectral_forcing(1e-3, 0.01, tke_target=tke)
    if decomposition == "fused":  # u* is where the advection left it: the velocity itself here
        G.set("tmpU", u[0]); G.set("tmpV", u[1]); G.set("tmpW", u[2])
    st = G.spectral_forcing(1e-3, 0.01, tke_target=tke)
    for k in ("tke", "eps", "tke_filtered", "l_integral", "fac"):
        assert st[k] == pytest.approx(ref[k], rel=1e-12), k
    got = [G.get(n) for n in (("tmpU", "tmpV", "tmpW") if decomposition == "fused" else "uvw")]
    for a, b in zip(got, O.velocity()):
        assert np.linalg.norm(a - b) < 1e-12 * np.linalg.norm(b)
