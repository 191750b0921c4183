"""get_tune("col_threads") is the number of threads that the fused column kernel is launched
with, on both sides of each limit of the default's rule, and writing the value back changes
nothing: the rule goes on deciding, where other shapes or a batch are asked for later too."""
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg, step_batch
from tests.test_gpu_batch import same, states

pytestmark = pytest.mark.gpu


def context(nx, ny, nl, prec=abi.MRMG_FP64, seed=3):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=seed, thermal=True, temperature=300.0)
    x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, precision=prec)
    x.build_tensor(num_images=0)
    x.set_media(med)
    x.set_llg(dt=5e-14)
    return x


@pytest.mark.parametrize("nx,ny,nl,threads", [(64, 128, 4, 512), (64, 135, 4, 1024), (40, 1024, 2, 1024),
                                              (500, 180, 3, 1024), (512, 180, 3, 512)])
def test_reads_what_is_launched(nx, ny, nl, threads):
    x = context(nx, ny, nl)
    assert x.get_tune("col_threads") == threads
    x.tune("col_threads", threads)
    assert x.get_tune("col_threads") == threads
    x.tune("col_threads", 256 if nl * ny <= 1024 else 512)     # asked for
    assert x.get_tune("col_threads") == (256 if nl * ny <= 1024 else 512)
    x.tune("col_threads", threads)
    assert x.get_tune("col_threads") == threads
    x.close()


def test_writing_it_back_leaves_the_rule():
    x = context(64, 135, 4)
    x.tune("col_threads", x.get_tune("col_threads"))
    x.tune("wave_fft", 1)       # without a 1024-thread kernel
    x.tune("col_path", 2)
    assert x.get_tune("col_threads") == 512
    x.tune("wave_fft", 0)
    x.tune("col_path", 0)
    assert x.get_tune("col_threads") == 1024
    x.close()


def test_written_back_in_a_batch():
    solo, batch = [context(64, 135, 4, seed=s) for s in (1, 2)], [context(64, 135, 4, seed=s) for s in (1, 2)]
    for x in solo + batch:
        x.tune("col_threads", x.get_tune("col_threads"))
    for x, p in zip(solo, (7, 8)):
        x.step(3, philox_seed=p)
    step_batch(batch, 3, philox_seeds=[7, 8])
    assert all(same(states(a, 4), states(b, 4)) for a, b in zip(solo, batch))
    for x in solo + batch:
        x.close()
