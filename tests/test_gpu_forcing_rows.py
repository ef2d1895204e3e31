"""cup_spectral_forcing's two ways of adding the band: from its modes, row by row (32 modes or fewer
with |kx|, |ky| <= 2), and by filtering the spectra and transforming back (any other band), against the
CPU oracle; boxes of both kinds, with a mean flow (the kx = 0 slot's unpacking) and odd block counts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the band 0 < |k|^2 <= 4: 16 canonical modes with every |k_a| <= 2 in a 2 pi cube, one axis only in
# flat boxes, up to |kx| = 4 in a 4 pi box; few modes, but |ky| up to 4 or 3, in boxes long in y, and
# |kz| up to 4 (which the rows take) in boxes long in z
CASES = [((4, 4, 4), 2 * np.pi), ((3, 5, 2), 2 * np.pi), ((1, 1, 6), 2 * np.pi), ((5, 1, 2), 2 * np.pi),
         ((2, 9, 8), 2 * np.pi), ((4, 2, 2), 4 * np.pi), ((2, 4, 3), 4 * np.pi),
         ((2, 4, 2), 4 * np.pi), ((4, 6, 4), 3 * np.pi), ((1, 4, 1), 4 * np.pi), ((2, 2, 4), 4 * np.pi),
         ((4, 4, 8), 4 * np.pi)]


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


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("bpd,extent", [((2, 4, 2), 4 * np.pi), ((4, 6, 4), 3 * np.pi), ((2, 2, 4), 4 * np.pi)])
@pytest.mark.parametrize("decomposition,body", [("plain", False), ("fused", False), ("fused", True)])
def test_forced_step(cup, oracle, bpd, extent, decomposition, body):
    """The forced step where the band reaches |ky| = 4 and 3 (no row synthesis) and |kz| = 4, and with
    the sphere its adjoint, whose oracle central differences of the oracle's step pin."""
    print(f"bpd={bpd} extent={extent} {decomposition} body={body}", flush=True)
    rng = np.random.default_rng(37)
    G = cup.Grid(bpd, maxextent=extent, precision=8, decomposition=decomposition)
    O = oracle.OracleSim(bpd, maxextent=extent)
    U, V, W = (1.0, 0.0, 0.0), (-1.0, 0.1, 0.0), (0.3, -0.4, 0.8)
    sph = None
    if body:
        centre, R = tuple(np.array(G.extent) * [0.45, 0.5, 0.5]), 0.3 * min(G.extent)
        G.chi_from_sphere(centre, R)
        O.sphere_create(R, centre)
        sph = dict(lambda_=1e5, implicit=True, trans_vel=V, ang_vel=W)
    u = [0.3 * rng.standard_normal(G.shape) + m for m in (1.0, 0.8, -0.9)]
    dt, nu, rate = 0.2 * G.h, 1e-3, 0.4
    G.set_velocity(*u); O.set_velocity(*u)
    G.run_steps(1, nu=nu, uinf=U, fixed_dt=dt, sphere=sph, spectral_forcing=True, injection_rate=rate)
    O.timestep(dt, nu, uinf=U, sphere=sph, spectral_forcing=True, injection_rate=rate)
    for a, b in zip(G.velocity(), O.velocity()):
        assert rel(a, b) < 1e-11
    if not body:
        return
    lam = [rng.standard_normal(G.shape) for _ in range(3)]
    G.set_velocity(*u); O.set_velocity(*u)
    for n, f in zip(("adjU", "adjV", "adjW"), lam):
        G.set(n, f)
    dv, dw = G.adjoint_step_body(dt, nu, U, sph, 3.7, rotation=True, injection_rate=rate)
    lam0, dvo, dwo = O.adjoint_step_body(dt, nu, lam, V, 1e5, True, 3.7, U, ang_vel=W, injection_rate=rate)
    for n, b in zip(("adjU", "adjV", "adjW"), lam0):
        assert rel(G.get(n), b) < 1e-11
    np.testing.assert_allclose(dv, dvo, rtol=1e-11, atol=1e-12 * np.abs(dvo).max())
    np.testing.assert_allclose(dw, dwo, rtol=1e-10, atol=1e-11 * np.abs(dwo).max())
