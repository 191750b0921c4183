"""The readback's window: positions at the edges and the middle, sensitivities from a
fraction of a cell to wider than the grid and different in x and y, on periodic and open
grids, against a direct numpy sum over every cell in 64 bits.  A sum of n FP64 terms of
mixed sign differs by at most n eps of the sum of their magnitudes, here 1e-12 of it; a
non-finite cell makes every signal non-finite, however far it is."""
import numpy as np
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg
from tests.test_gpu_parity import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("open_", [False, True])
@pytest.mark.parametrize("sx,sy", [(0.3, 0.3), (0.4, 2.0), (1.2, 0.5), (3.0, 3.0), (40.0, 0.5)])
def test_window_matches_direct_sum(open_, sx, sy):
    nx, ny, d = 150, 96, 2e-7
    med = media.make_media(nx, ny, dx=d, dy=d, dz=4e-7, n_lay=2, seed=4)
    x = Llg(nx, ny, 2, d, d, med.dz, demag=False, open=open_)
    x.set_media(med)
    P = np.zeros((ny, nx))
    for k, (m, L) in enumerate(zip(random_state(med, 9, tilt=1.0), med.layers)):
        x.set_state(k, m)
        c = L.grain2grid.reshape(-1, 2) - 1
        P[c[:, 1], c[:, 0]] += np.repeat(L.ms * m[:, 2], np.diff(L.grain2gridindex)) * med.dz[k] * d * d
    x.step(0, diag=False)
    xs = np.array([0.0, 0.5, 1.0, 74.6, 149.5, 150.0, 75.0, 3.2, -20.0, 170.0]) * d
    ys = np.array([0.0, 95.9, 47.0, 0.2, 96.0, 1.0, 48.3, 95.0, 30.0, -5.0]) * d

    def g(n, pos, s):
        u = (np.arange(n) + 0.5) * d - pos[:, None]
        if not open_:
            u -= n * d * np.rint(u / (n * d))
        return np.exp(-u * u / (2.0 * (s * d) ** 2))

    gy, gx = g(ny, ys, sy), g(nx, xs, sx)
    want = np.einsum("pi,pi->p", gy @ P, gx)
    size = np.einsum("pi,pi->p", gy @ np.abs(P), gx)
    got = x.readback(xs, ys, (sx * d, sy * d))
    assert (np.abs(got - want) <= 1e-12 * size + 1e-300).all()
    m, _ = x.get_state(1)
    m[-1] = np.nan
    x.set_state(1, m)
    assert not np.isfinite(x.readback(xs, ys, (sx * d, sy * d))).any()
    x.close()
