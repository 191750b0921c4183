"""The grain kernel's splits (lanes per grain 1, 2, 4 and 16) against the oracle where a
split can go wrong: a last wave that is not full, waves whose grains lie in two layers of
which one has a source, grains of more runs than a wave's round of LDS slots holds, and
each kind of moving source (field table, super-Gaussian, temperature table), alone and
together, on fixed and adaptive steps.  The bars are those of the same physics elsewhere:
1e-10 in m (LLG), 1e-9 in m and |m| (LLB)."""
import numpy as np
import pytest

from mrm_amd import abi, media
from tests.test_gpu_llb import compare, llb_media, start
from tests.test_gpu_parity import pair, random_state
from tests.test_gpu_sources import both, head_table, laser

pytestmark = pytest.mark.gpu
LANES = [1, 2, 4, 16]


def temp_table():
    x = np.linspace(-30e-7, 30e-7, 13)
    X, Y = np.meshgrid(x, x)
    return abi.SourceArrays(abi.MRMG_SRC_TEMP_TABLE, x, x, 300.0 * np.exp(-(X ** 2 + Y ** 2) / 2e-12),
                            vel=(-1000.0, 500.0), offset=(60e-7, 40e-7))


@pytest.mark.parametrize("lanes", LANES)
@pytest.mark.parametrize("nx,ny,nl,pitch,head", [(50, 45, 3, 8e-7, False),     # ragged last wave
                                                 (50, 45, 3, 8e-7, True),      # a table on the middle layer only
                                                 (96, 90, 1, 60e-7, True),     # a few grains of some 30 rows
                                                 (16, 8, 1, 40e-7, False)])    # one grain
def test_lanes_llg(oracle_mod, lanes, nx, ny, nl, pitch, head):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, pitch=pitch, seed=7)
    s, gpu = pair(oracle_mod, med)
    gpu.tune("lanes_per_grain", lanes)
    if head:
        both(s, gpu, nl // 2, 0, head_table(med))
    for k, m in enumerate(random_state(med, 3, tilt=0.3)):
        s.set_state(k, m)
        gpu.set_state(k, m)
    gpu.set_llg(dt=5e-14)
    s.step(10, 5e-14)
    gpu.step(10)
    assert max(np.abs(s.get_state(k)[0] - gpu.get_state(k)[0]).max() for k in range(nl)) <= 1e-10


@pytest.mark.parametrize("lanes", LANES)
@pytest.mark.parametrize("second", ["none", "spot", "table"])
@pytest.mark.parametrize("adaptive", [False, True])
def test_lanes_llb_sources(oracle_mod, lanes, second, adaptive):
    """A spot on layer 0; on layer 1 nothing, a spot, or a temperature table with Ms
    following the temperature there (the next evaluation's temperature is needed too)."""
    med = llb_media(nx=50, ny=36, seed=47, use_mag=True)
    for L in med.layers:
        L.temp = np.full(L.ng, 300.0)
    if second == "table":
        med.layers[1].use_mag, med.layers[1].msexp = 0, 1.0
    s, gpu = pair(oracle_mod, med, ufields=[abi.make_ufield((0, 0, -1), scale=8000.0)] * med.n_lay)
    gpu.tune("lanes_per_grain", lanes)
    both(s, gpu, 0, 1, laser(med))
    if second != "none":
        both(s, gpu, 1, 1, laser(med, vel=(1500.0, 0.0)) if second == "spot" else temp_table())
    start(s, gpu, med, seed=8)
    n = 12
    noise = oracle_mod.mt_noise([11, 12], [L.ng for L in med.layers], [True] * med.n_lay, n)
    kw = dict(dt_frac=0.05, dt_max=4e-15, max_dm=2.0) if adaptive else {}
    gpu.set_llg(dt=1e-15, llb=True, **kw)
    s.step(n, 1e-15, noise=noise, llb=True, **kw)
    gpu.step(n, noise=noise)
    compare(s, gpu, med, 1e-9, f"lanes {lanes}, second source {second}, adaptive {adaptive}")
