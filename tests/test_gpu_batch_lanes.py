"""Batched grain launches: members whose lanes per grain are equal (1, 4 and 8: one launch
for all of them; 2: a launch each) or differ (a launch each) end bit for bit where their
own steps end, with grain counts that differ between the members, for the Heun and the
mid-point pushes."""
import pytest

from mrm_amd import abi
from mrm_amd.llg import step_batch
from tests.test_gpu_batch import member, same, states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [(1, 1, 1), (4, 4, 4), (8, 8, 8), (2, 2, 2), (8, 4, 8)])
@pytest.mark.parametrize("type_", [abi.MRMG_TYPE_HEUN, abi.MRMG_TYPE_BORIS_MID])
@pytest.mark.parametrize("graph", [True, False])
def test_batched_lanes_match_solo(lanes, type_, graph):
    n, seeds = 12, [3, 5, 8]
    solo, batch, meds = [], [], []
    for i, (sd, l) in enumerate(zip(seeds, lanes)):
        for out in (solo, batch):
            x, med = member(48, 40, sd, abi.MRMG_FP32, type_=type_)
            x.tune("lanes_per_grain", l)
            if out is solo:
                x.step(n, philox_seed=100 + i)
            out.append(x)
        meds.append(med)
    assert len({m.G for m in meds}) > 1
    t = [0.0] * 3
    for part in (5, n - 5):     # two calls: the second starts from the first's state
        t = step_batch(batch, part, philox_seeds=[100, 101, 102], t0s=t, graph=graph)
    for a, b, med in zip(solo, batch, meds):
        assert same(states(a, med.n_lay), states(b, med.n_lay))
