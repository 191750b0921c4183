"""The fused column kernel's default workgroup: 1024 threads where the product has more than
one item a thread at 512.  The values do not depend on the threads, so the default's steps end
bit for bit where those with 512 asked for end, on both sides of each limit of the rule:
items a workgroup (512, 2048), workgroups (256), both forms, both layouts of the spectra, open
boundaries, layer groups and wave-local transforms (which keep 512)."""
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg
from tests.test_gpu_batch import same, states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.MRMG_FP64, abi.MRMG_FP32])
@pytest.mark.parametrize("nx,ny,nl,open_,tune", [
    (64, 128, 4, False, {}), (64, 135, 4, False, {}), (256, 256, 4, False, {}), (256, 256, 4, False, {"col_path": 2}),
    (40, 1024, 2, False, {}), (40, 1080, 2, False, {}), (500, 180, 3, False, {}), (512, 180, 3, False, {}),
    (64, 64, 8, True, {}), (256, 256, 4, False, {"col_groups": 2}), (256, 256, 4, False, {"col_path": 2, "wave_fft": 1})])
def test_default_matches_512_threads(nx, ny, nl, open_, tune, prec):
    out = []
    for threads in (None, 512):
        med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=3, thermal=True, temperature=300.0)
        x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, precision=prec, open=open_)
        x.build_tensor(num_images=0)
        x.set_media(med)
        if threads:
            x.tune("col_threads", threads)
        for k, v in tune.items():
            x.tune(k, v)
        x.set_llg(dt=5e-14)
        x.step(3, philox_seed=7)
        out.append(states(x, nl))
        x.close()
    assert same(*out)
