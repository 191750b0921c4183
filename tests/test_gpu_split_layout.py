"""Which layout of the columns a long FP64 grid takes, and its demag field in it: the split
columns where the tensor is of z-offset blocks, the unsplit ones where the layers are unequal
or the tensor has nine slots, also where a context's tensor changes from one to the other,
against the convolution in numpy's FFTs (the bar and the oracle of the split transform's own
test, 1e-12 of the largest field)."""
import numpy as np
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg
from tests.test_gpu_parity import random_state

pytestmark = pytest.mark.gpu


def convolution_error(x, med, N, tol_state=None):
    """The cell field of the present state against numpy's."""
    nl, ny, nx = med.n_lay, med.ny, med.nx
    M = np.zeros((3, nl, ny, nx))
    for k, L in enumerate(med.layers):
        m, _ = x.get_state(k)
        c = L.grain2grid.reshape(-1, 2) - 1
        M[:, k, c[:, 1], c[:, 0]] = np.repeat(L.ms[:, None] * m, np.diff(L.grain2gridindex), axis=0).T
    N = N.reshape(nl, nl, 9, x.fy, x.fx)
    Mh = np.fft.rfft2(M, s=(x.fy, x.fx))
    H = np.zeros_like(M)
    for ko in range(nl):
        for a in range(3):
            s = sum(np.fft.rfft2(N[ks, ko, 3 * a + b]) * Mh[b, ks] for ks in range(nl) for b in range(3))
            H[a, ko] = np.fft.irfft2(s, s=(x.fy, x.fx), norm="forward")[:ny, :nx]
    hc, _ = x.demag_field()
    return np.abs(hc - H).max() / np.abs(H).max()


def context(nx, ny, nl, dz, open_=False):
    med = media.make_media(nx, ny, dz=dz, n_lay=nl, seed=3, exchange=False)
    x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, open=open_)
    return x, med


def load(x, med):
    x.set_media(med)
    for k, m in enumerate(random_state(med, 5, tilt=1.0)):
        x.set_state(k, m)


@pytest.mark.parametrize("nx,ny,nl,dz,open_,split", [
    (32, 1024, 3, 2e-7, False, True), (32, 1024, 3, [2e-7, 3e-7, 2e-7], False, False),
    (24, 1024, 4, [2e-7, 2e-7, 2e-7, 3e-7], False, False), (32, 384, 3, [2e-7, 3e-7, 2e-7], True, False),
    (32, 2560, 1, 2e-7, False, True)])
def test_layout_by_tensor(nx, ny, nl, dz, open_, split):
    x, med = context(nx, ny, nl, dz, open_)
    N = x.build_tensor(num_images=0, return_real=True)
    load(x, med)
    x.step(0, diag=False)
    assert (x.get_tune("col_split") > 0) == split
    assert convolution_error(x, med, N) <= 1e-12
    x.close()


def test_layout_follows_the_tensor():
    """z-offset, nine slots, z-offset again, then a copy into a fresh context; tunables set
    before stay."""
    nx, ny, nl = 32, 1024, 3
    x, med = context(nx, ny, nl, 2e-7)
    N = x.build_tensor(num_images=0, return_real=True)
    load(x, med)
    x.tune("row_threads", 64)
    x.tune("col_radix", 8)
    x.tune("row_block", 4)
    x.step(0, diag=False)
    first = x.get_tune("col_split")
    assert first > 1 and convolution_error(x, med, N) <= 1e-12
    N9 = np.array(N).reshape(nl, nl, 9, ny, nx)
    N9[:, :, 1] *= 1.5                      # xy no longer equals yx
    x.set_tensor(N9)
    assert x.get_tune("col_split") == 0 and convolution_error(x, med, N9) <= 1e-12
    assert x.get_tune("row_threads") == 64 and x.get_tune("col_radix") == 8
    y, _ = context(nx, ny, nl, 2e-7)
    y.copy_tensor(x)
    load(y, med)
    y.step(0, diag=False)
    assert y.get_tune("col_split") == 0 and convolution_error(y, med, N9) <= 1e-12
    x.set_tensor(N)
    assert x.get_tune("col_split") == first and convolution_error(x, med, N) <= 1e-12
    y.copy_tensor(x)
    assert y.get_tune("col_split") == first and convolution_error(y, med, N) <= 1e-12
    x.close()
    y.close()
