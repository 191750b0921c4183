"""bench.py's reading of a profile: the class of each step kernel's name, and the bytes that a
split column transform's row kernels hand over with open boundaries."""
import importlib.util
import os

import pytest

from mrm_amd import media

spec = importlib.util.spec_from_file_location("bench_mod", os.path.join(os.path.dirname(__file__), "..", "bench.py"))
bench = importlib.util.module_from_spec(spec)
spec.loader.exec_module(bench)


@pytest.mark.parametrize("name,cls", [
    ("void k_rowS_fwd<double, 16>(DemagOps<double>, int)", "row_fwd"),
    ("void k_rowS_inv<double, 16, false>(DemagOps<double>, int)", "row_inv"),
    ("void k_colp<double, 16, 4>(DemagOps<double>, int)", "col"),
    ("void k_grain_batch<double, 0, 8, float>(GrainOps<double, float> const*, StepArgs)", "grain1"),
    ("void k_grain_batch<double, 3, 1, float>(GrainOps<double, float> const*, StepArgs)", "grain2"),
    ("void k_colT<double, 16, true>(DemagOps<double>, int)", "col_inv")])
def test_kernel_class(name, cls):
    assert bench.kernel_class(name) == cls


def test_open_split_columns_move_the_padded_length():
    med = media.make_media(16, 24, dz=2e-7, n_lay=2, seed=3)
    whole, split = (bench.kernel_bytes(med, 8, 1, fft=(32, 48), radix=r) for r in (0, 2))
    more = 6 * 2 * 17 * 24 * 8      # the padding half of the spectra
    assert [split[k] - whole[k] for k in ("row_fwd", "row_inv", "col")] == [more, more, 2 * more]
