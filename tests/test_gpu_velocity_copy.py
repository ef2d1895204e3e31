"""The block-order velocity copies (cup_get_velocity_device / cup_set_velocity_device) move every byte,
from 16-byte aligned buffers (16-byte accesses) and from buffers that are only aligned to a value."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("bpd", [(1, 1, 1), (3, 5, 2)])
def test_round_trip(cup, precision, offset, bpd):
    import torch
    from cubismup_3d_amd import _lib as L
    print(f"precision={precision} offset={offset} bpd={bpd}", flush=True)
    G, H = (cup.Grid(bpd, precision=precision) for _ in range(2))
    rng = np.random.default_rng(37)
    u = [rng.standard_normal(G.shape).astype("f4" if precision == 4 else "f8") for _ in range(3)]
    G.set_velocity(*u)
    n = 3 * u[0].size
    buf = torch.full((n + 2,), -7.0, dtype=torch.float32 if precision == 4 else torch.float64, device="cuda")
    torch.cuda.synchronize()
    part = buf[offset:offset + n]
    G._c(L.lib().cup_get_velocity_device(G._h, C.c_void_p(part.data_ptr())))
    G.synchronize()
    assert (buf[:offset] == -7).all() and (buf[offset + n:] == -7).all()
    H._c(L.lib().cup_set_velocity_device(H._h, C.c_void_p(part.data_ptr())))
    H.synchronize()
    for a, b in zip(H.velocity(), u):
        assert np.array_equal(a, b)
