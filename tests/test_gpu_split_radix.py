"""The split of the FP64 column transform with radix 2 on open boundaries (one media row a
group: two items exchange their rows between lanes), with odd column lengths, and under the
tunables of the row and column kernels: the demag field against the convolution in numpy's
FFTs (1e-12 of the largest field, as in the split transform's own test), and the launch
shapes that leave the values unchanged bit for bit.  A captured batch whose column or row
kernels ask for more than 64 KB of LDS, with a context of another size beside it."""
import pytest

from mrm_amd import media
from mrm_amd.llg import Llg, step_batch
from tests.test_gpu_batch import same, states
from tests.test_gpu_split_layout import context, convolution_error, load

pytestmark = pytest.mark.gpu


# 768, 720, 810 and 1000 rows of FFT: radix 4 would leave columns under 256
@pytest.mark.parametrize("nx,ny,nl", [(32, 384, 3), (30, 360, 3), (20, 405, 3), (64, 500, 3)])
@pytest.mark.parametrize("tune", [{}, {"row_block": 2}, {"row_block": 4, "row_threads": 64},
                                  {"row_threads": 256, "col_radix": 4}, {"row_radix": 4, "col_radix": 8}])
def test_radix_two_open(nx, ny, nl, tune):
    x, med = context(nx, ny, nl, 2e-7, True)
    N = x.build_tensor(num_images=0, return_real=True)
    load(x, med)
    for k, v in tune.items():
        x.tune(k, v)
    x.step(0, diag=False)
    assert x.get_tune("col_split") == 2
    for k, v in tune.items():
        assert x.get_tune(k) == v
    assert convolution_error(x, med, N) <= 1e-12
    x.close()


@pytest.mark.parametrize("nx,ny,nl,open_,radix", [
    (32, 384, 3, True, 2), (20, 405, 3, True, 2), (30, 540, 2, True, 4), (32, 1024, 3, True, 8), (45, 720, 4, False, 2),
    (32, 1024, 4, False, 4), (40, 2048, 4, False, 8)])
def test_row_shapes_leave_the_values(nx, ny, nl, open_, radix):
    def run(tune):
        med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=3, thermal=True, temperature=300.0)
        x = Llg(nx, ny, nl, med.dx, med.dy, med.dz, open=open_)
        x.build_tensor(num_images=0)
        x.set_media(med)
        x.set_llg(dt=5e-14)
        for k, v in tune.items():
            x.tune(k, v)
        assert x.get_tune("col_split") == radix
        x.step(3, philox_seed=7)
        out = states(x, nl)
        x.close()
        return out

    want = run({})
    for tune in ({"row_block": 2}, {"row_block": 4}, {"row_threads": 64}, {"row_threads": 256}, {"wave_fft": 1}):
        assert same(want, run(tune))


@pytest.mark.parametrize("nx,ny,nl", [(24, 4096, 4), (2000, 1080, 2)])   # 98 KB a column kernel; 68 KB a row kernel
def test_captured_batch_with_wide_lds(nx, ny, nl):
    med = media.make_media(nx, ny, dz=2e-7, n_lay=nl, seed=3, thermal=True, temperature=300.0)

    def member():
        x = Llg(nx, ny, nl, med.dx, med.dy, med.dz)
        x.build_tensor(num_images=0)
        x.set_media(med)
        x.set_llg(dt=5e-14)
        return x

    solo, batch = [member() for _ in range(2)], [member() for _ in range(2)]
    assert solo[0].get_tune("col_split") > 1
    other, m2 = context(24, 3072, 4, 2e-7)      # 74 KB a column kernel
    other.build_tensor(num_images=0)
    load(other, m2)
    other.step(1)
    for x, p in zip(solo, (7, 8)):
        x.step(4, philox_seed=p)
    t = step_batch(batch, 2, philox_seeds=[7, 8], graph=True)
    other.step(1)
    step_batch(batch, 2, philox_seeds=[7, 8], t0s=t, graph=True)
    assert all(same(states(a, nl), states(b, nl)) for a, b in zip(solo, batch))
    for x in solo + batch + [other]:
        x.close()


@pytest.mark.parametrize("nx,ny,nl,open_,rows", [(40, 2048, 4, False, 8), (32, 1024, 4, False, 4), (32, 1024, 3, True, 4),
                                                 (32, 384, 3, True, 1)])
def test_row_block_reads_what_is_launched(nx, ny, nl, open_, rows):
    x, med = context(nx, ny, nl, 2e-7, open_)
    x.build_tensor(num_images=0)
    for v in (2, 4, 8):
        x.tune("row_block", v)
        assert x.get_tune("row_block") == max(v, rows)
        x.tune("row_block", x.get_tune("row_block"))
        assert x.get_tune("row_block") == max(v, rows)
    x.close()


# both sides of each limit of the layout's rule: 256 and 360 to 512 values a column of four
# layers, 256 with open boundaries, other layers from 256 on; rows of 768 points with radix 8,
# longer ones with columns of 512 values or with radix 4 and up to 512; the field is the
# convolution's on each of the small ones
@pytest.mark.parametrize("nx,ny,nl,open_,radix", [
    (16, 1024, 4, False, 4), (16, 540, 4, False, 0), (16, 648, 4, False, 0), (16, 720, 4, False, 2), (16, 1080, 4, False, 0),
    (16, 2160, 4, False, 0), (16, 3072, 4, False, 8), (16, 512, 4, True, 4), (16, 540, 4, True, 0), (16, 384, 4, True, 0),
    (16, 360, 3, True, 2), (16, 720, 3, False, 2), (768, 2160, 1, False, 8), (800, 2160, 1, False, 4),
    (768, 2160, 2, False, 8), (800, 2160, 2, False, 0), (800, 2048, 2, False, 4), (1024, 4096, 1, False, 8),
    (2000, 1080, 2, False, 4), (450, 1080, 2, True, 0), (450, 1024, 2, True, 4), (384, 1080, 2, True, 8),
    (1024, 1350, 2, False, 2), (64, 1080, 3, True, 0), (64, 1024, 3, True, 8)])
def test_layout_rule(nx, ny, nl, open_, radix):
    x, med = context(nx, ny, nl, 2e-7, open_)
    N = x.build_tensor(num_images=0, return_real=nx * ny < 100000)
    assert x.get_tune("col_split") == radix
    if nx * ny < 100000:
        load(x, med)
        x.step(0, diag=False)
        assert convolution_error(x, med, N) <= 1e-12
    x.close()
