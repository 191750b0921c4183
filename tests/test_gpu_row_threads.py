"""The row workgroups' default threads: 128 for rows whose three components have no more than
256 elements, and in batches with more row workgroups than the chip holds (there a member
ends bit for bit where its own steps end, on both sides of the limits)."""
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg, step_batch
from tests.test_gpu_batch import same, states

pytestmark = pytest.mark.gpu


def context(nx, ny, nl, prec, seed=1):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=seed, thermal=True, temperature=300.0)
    x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, precision=prec)
    x.build_tensor(num_images=0)
    x.set_media(med)
    x.set_llg(dt=5e-14)
    return x


@pytest.mark.parametrize("nx,threads", [(64, 128), (81, 128), (90, 256), (128, 256)])
def test_short_rows_take_128_threads(nx, threads):
    x = Llg(nx, 32, 1, 1e-7, 1e-7, [2e-7])
    assert x.get_tune("row_threads") == threads
    x.close()


# row workgroups: members * nl * ny / 2, the chip's at once 7 * 256 (FP32) or 5 * 256 (FP64)
@pytest.mark.parametrize("nx,ny,nl,members,prec", [
    (64, 128, 4, 7, abi.MRMG_FP32), (64, 128, 4, 8, abi.MRMG_FP32), (300, 128, 4, 8, abi.MRMG_FP32),
    (320, 128, 4, 8, abi.MRMG_FP32), (96, 128, 4, 5, abi.MRMG_FP64), (96, 128, 4, 6, abi.MRMG_FP64)])
def test_full_chip_batch_matches_solo(nx, ny, nl, members, prec):
    out = []
    for batch in (False, True):
        xs = [context(nx, ny, nl, prec, seed=1 + i % 2) for i in range(members)]
        if batch:
            step_batch(xs, 3, philox_seeds=list(range(members)))
        else:
            for i, x in enumerate(xs):
                x.step(3, philox_seed=i)
        out.append([states(x, nl) for x in xs])
        for x in xs:
            x.close()
    assert all(same(a, b) for a, b in zip(*out))
