"""The FP64 column transform split over the row kernels (one column kernel between them):
its demag field against the convolution in numpy's FFTs with the device's own tensor, on
grids too long for the fused column kernel, for each radix that the grid's length and
layers take (8, 4, 2, 1), lengths with factors 3 and 5, 1 to 4 layers, periodic and open
boundaries, a batch against single steps, and the unsplit path beside it (5 layers, an
odd length, FP32).  Two FFT routes of 2 N log2 N FP64 operations differ by a few
log2(N) eps of the largest field, below 1e-12 (the bar of the demag field elsewhere); FP32
2e-6."""
import numpy as np
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg, step_batch
from tests.test_gpu_batch import same, states
from tests.test_gpu_parity import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nl,prec,open_", [
    (40, 4096, 1, abi.MRMG_FP64, False), (40, 2048, 4, abi.MRMG_FP64, False), (36, 2160, 3, abi.MRMG_FP64, False),
    (32, 1028 - 4, 4, abi.MRMG_FP64, False), (45, 540, 4, abi.MRMG_FP64, False), (32, 900, 3, abi.MRMG_FP64, False),
    (32, 1024, 3, abi.MRMG_FP64, True), (30, 540, 2, abi.MRMG_FP64, True), (256, 540, 4, abi.MRMG_FP64, True),
    (512, 1080, 2, abi.MRMG_FP64, False), (32, 729, 3, abi.MRMG_FP64, False), (32, 1024, 5, abi.MRMG_FP64, False),
    (32, 2048, 3, abi.MRMG_FP32, False), (32, 1024, 3, abi.MRMG_FP32, True)])
def test_field_matches_numpy_convolution(nx, ny, nl, prec, open_):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=3, exchange=False)
    x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, precision=prec, open=open_)
    N = x.build_tensor(num_images=0 if open_ else 1, return_real=True).reshape(nl, nl, 9, x.fy, x.fx)
    x.set_media(med)
    for k, m in enumerate(random_state(med, 5, tilt=1.0)):
        x.set_state(k, m)
    x.set_llg(dt=1e-20)      # one step whose field is that of the state it ends in (to dt^2)
    x.step(1)
    st = [x.get_state(k) for k in range(nl)]
    M = np.zeros((3, nl, ny, nx))
    for k, ((m, _), L) in enumerate(zip(st, med.layers)):
        c = L.grain2grid.reshape(-1, 2) - 1
        M[:, k, c[:, 1], c[:, 0]] = np.repeat(L.ms[:, None] * m, np.diff(L.grain2gridindex), axis=0).T
    Mh = np.fft.rfft2(M, s=(x.fy, x.fx))
    H = np.zeros_like(M)
    for ko in range(nl):
        for a in range(3):
            s = sum(np.fft.rfft2(N[ks, ko, 3 * a + b]) * Mh[b, ks] for ks in range(nl) for b in range(3))
            H[a, ko] = np.fft.irfft2(s, s=(x.fy, x.fx), norm="forward")[:ny, :nx]
    hc, hg = x.demag_field()
    assert np.abs(hc - H).max() <= (1e-12 if prec == abi.MRMG_FP64 else 2e-6) * np.abs(H).max()
    # the run sums of the step saw the same field
    off = np.concatenate([[0], np.cumsum(med.ngs)])
    for k, ((m, h), L) in enumerate(zip(st, med.layers)):
        hk = L.hk.reshape(-1, 2)[:, 0] * (m * L.uni_axis.reshape(-1, 3)).sum(1)
        want = hg[off[k]:off[k + 1]] + hk[:, None] * L.uni_axis.reshape(-1, 3)
        assert np.abs(h - want).max() <= (1e-11 if prec == abi.MRMG_FP64 else 2e-6) * np.abs(H).max()
    x.close()


def test_split_batch_matches_solo():
    out = []
    for batch in (False, True):
        xs = []
        for sd in (1, 2):
            med = media.make_media(24, 2048, dz=2e-7, n_lay=4, seed=sd, thermal=True, temperature=300.0)
            x = Llg(24, 2048, 4, med.dx, med.dy, med.dz)
            x.build_tensor(num_images=1)
            x.set_media(med)
            x.set_llg(dt=5e-14)
            xs.append(x)
        if batch:
            step_batch(xs, 4, philox_seeds=[7, 8])
        else:
            for x, p in zip(xs, (7, 8)):
                x.step(4, philox_seed=p)
        out.append([states(x, 4) for x in xs])
        for x in xs:
            x.close()
    assert all(same(a, b) for a, b in zip(*out))
