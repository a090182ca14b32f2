"""The upwind kernels at the edges of their launch shapes: the compact scheme's
solves with the characteristic projection at the last and first line length of
every chunk count (and with fewer lines than a tile holds), and the y- and
z-faces' runs where the run length or the last run's remainder changes.  The
right-hand side against the oracle with test_gpu_upwind's fields and its
tolerance (1e-12 of the component's maximum: sums of a few hundred rounded
terms of that size)."""
import pytest

from test_gpu_upwind import TOL, make_pair, relmax

pytestmark = pytest.mark.gpu


def check(f, s, dims):
    f.qswap()
    s.qswap()
    got = f.rhscal()
    s.gradcal()
    s.rhscal()
    f.close()
    for m in range(5):
        if m == 3 and dims[2] == 0:
            continue
        assert relmax(got[m], s.qrhs[m]) < TOL, (m, relmax(got[m], s.qrhs[m]))


@pytest.mark.parametrize("dims", [(76, 13, 12), (77, 12, 13), (156, 12, 12), (157, 12, 12), (12, 76, 77), (12, 157, 12),
                                  (12, 12, 156), (316, 12, 12), (317, 12, 0), (12, 316, 0), (12, 12, 317), (569, 12, 0),
                                  (12, 569, 0)])
def test_compact_characteristic_solves_at_shape_edges(dims):
    check(*make_pair(dims, 0, True, conschm="543c"), dims)


@pytest.mark.parametrize("chardec", [False, True])
@pytest.mark.parametrize("dims", [(20, 16, 15), (20, 17, 31), (63, 64, 65), (127, 97, 12), (20, 35, 0)])
def test_faces_at_run_edges(dims, chardec):
    check(*make_pair(dims, 1, chardec), dims)
