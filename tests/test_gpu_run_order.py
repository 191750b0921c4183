"""The order in which the run sums of the cell field are stored (row by row where a wave
stages 64 grains, grain by grain where several lanes share one): a context whose lanes per
grain are changed while it is live, before its first step or between steps, ends bit for
bit where one ends that had them from the start, on the fused and the split column paths,
the split transform, both forms and open boundaries."""
import pytest

from mrm_amd import abi, media
from mrm_amd.llg import Llg
from tests.test_gpu_batch import same, states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nl,prec,open_,path", [
    (48, 40, 3, abi.MRMG_FP64, False, 0), (48, 45, 3, abi.MRMG_FP32, False, 1), (45, 50, 2, abi.MRMG_FP32, False, 2),
    (32, 1024, 4, abi.MRMG_FP64, False, None), (30, 405, 3, abi.MRMG_FP64, True, None)])
def test_changing_lanes_on_a_live_context(nx, ny, nl, prec, open_, path):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=3, thermal=True, temperature=300.0)

    def run(before, live, then):
        x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, precision=prec, open=open_)
        x.build_tensor(num_images=0)
        if path is not None:
            x.tune("col_path", path)
        if before:
            x.tune("lanes_per_grain", before)
        x.set_media(med)
        x.set_llg(dt=5e-14)
        x.step(0, diag=False)
        for v in live:
            x.tune("lanes_per_grain", v)
        x.step(3, philox_seed=7)
        for v in then:
            x.tune("lanes_per_grain", v)
        x.step(3, philox_seed=7)
        out = states(x, nl)
        x.close()
        return out

    assert same(run(8, [], []), run(1, [8], []))
    assert same(run(8, [], []), run(None, [1, 2, 8], [1, 8]))
    assert same(run(8, [], [1]), run(1, [8], [4, 1]))
    assert same(run(1, [], []), run(16, [1], []))
