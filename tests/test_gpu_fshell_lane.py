"""f classes with La+Lb+Lc+Ld <= 5 have per-lane kernels: they agree with the
wave-per-quartet kernel of the same class, closed and open shell, and a
mixed-precision engine still runs every quartet of an f class in FP64."""
import numpy as np
import pytest

from tests.helpers import announce, molecule, product_basis

pytestmark = pytest.mark.gpu

F_LANE = [(6, 0), (6, 1), (6, 2), (6, 3), (7, 0), (7, 1), (8, 0)]   # (fs|ss) ... (fd|ss)


def engine(kernel, **kw):
    from quick_amd.engine import FockEngine
    e = FockEngine(product_basis(molecule("alkane2"), "def2-TZVP"), cutoff=1e-11, **kw)
    for cb, ck in F_LANE:
        e.set_class_tuning(cb, ck, kernel)
    return e


@pytest.mark.parametrize("kernel", [0, 1])
def test_f_lane_kernels_equal_the_wave_per_quartet_kernel(kernel):
    announce("f lane kernel=%d" % kernel)
    from quick_amd.scf import seeded_density
    a, b = engine(kernel), engine(2)
    S = a.one_electron()[0]
    P, Q = seeded_density(S, 9), seeded_density(S, 8, seed=5)
    for x, y in zip((a.fock2e(P),) + a.fock2e_os(P / 2, Q / 2), (b.fock2e(P),) + b.fock2e_os(P / 2, Q / 2)):
        assert np.abs(x - y).max() <= 1e-11 * max(1.0, np.abs(y).max())   # sums in another order


def test_mixed_precision_leaves_f_classes_in_fp64():
    announce("f lane mixed")
    e = engine(1, precision="mixed")
    e.set_split_classes(0)
    halves = {name for name, fp32, _ in e.launches() if fp32}
    assert halves and not any("f" in name for name in halves)
