"""The kernels' size-dependent variants at the sizes where they change over
(edges of slices, groups and rounds, remainders), against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from parm_amd import capi
from tests import systems as S
from tests import test_batch_gpu as B

pytestmark = pytest.mark.gpu


def _device_or_fail():
    if capi.device_count() < 1:
        pytest.fail("no GPU visible: the -m gpu tests need an MI355X")


# build slices of 32 (dense) and 64 (sparse) atoms: one less, equal, one more
@pytest.mark.parametrize("ndim", [2, 3])
@pytest.mark.parametrize("lj", [False, True])
def test_batch_build_slice_edges(ndim, lj):
    _device_or_fail()
    print(f"batch build edges ndim={ndim} lj={lj}", flush=True)
    sizes = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 600]
    systems = B.packings(sizes, 0.4 if lj else 0.64, ndim, seed=11 + ndim)
    b = B.make_batch(systems, ndim, 0.25, lj=lj)
    refs = B.oracle_systems(systems, ndim, 0.25, lj=lj)
    b.initialize()
    for s, r in enumerate(refs):
        r.initialize()
        fd, ld = b.pairs(s)
        fr, lr = r.pairs()
        assert np.array_equal(fd, fr) and np.array_equal(ld, lr), (s, sizes[s])
    b.close()
