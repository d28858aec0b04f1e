"""Several quartet classes in one launch (fock_tile_group and coop_task run by
fused_tile_kernel and fused_coop_kernel) against one launch per class, which
a build with per-launch timing uses, and against the CPU oracle's path through
the general tests.  Both sides add the same terms with atomics in another
order: the difference is bounded by eps times the terms of an element times
their size, 2.2e-16 x 1e4 x 10 at these sizes, and the tolerance is 2e-11."""
import numpy as np
import pytest

from quick_amd import basis as B
from quick_amd import molecules as M
from quick_amd.codegen import gen_eri, gen_grad
from quick_amd.engine import FockEngine

TOL = 2e-11


def test_every_class_has_one_place():
    buckets = gen_eri.fuse_buckets()
    tile = [c for b in buckets if not b["coop"] for c in b["classes"]]
    coop = [c for b in buckets if b["coop"] for c in b["classes"]]
    assert len(set(tile)) == len(tile) and len(set(coop)) == len(coop)
    assert set(coop) == set(gen_eri.COOP_CLASSES)
    assert set(tile) == {c for c in gen_eri.quartet_classes()
                         if gen_eri.has_lane_kernels(*c) and c not in gen_eri.MD_CLASSES}
    for b in buckets:
        for c in b["classes"]:
            if b["coop"]:
                t = gen_eri.coop_tables(*c)
                assert t["glob"] == b["glob"] and t["total"] <= b["stride"]


def _density(n, rng, scale):
    P = rng.standard_normal((n, n)) * scale
    return 0.5 * (P + P.T)


# below and above the sizes at which the shapes change (32, 48, 64, 100, 128,
# 200 functions), bases without d, with d and with f shells
@pytest.mark.gpu
@pytest.mark.parametrize("mol, basis", [
    ("water", "STO-3G"), ("water", "6-31G*"), ("ethane", "6-31G*"), ("alkane4", "3-21G"), ("alkane4", "6-31G*"),
    ("ethane", "def2-TZVP"), ("waters8", "6-31G*"), ("waters8", "cc-pVDZ"), ("waters9", "cc-pVDZ"),
])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_shared_launches(mol, basis, precision):
    m = {"water": M.water, "ethane": lambda: M.alkane(2), "alkane4": lambda: M.alkane(4),
         "waters8": lambda: M.water_cluster(8), "waters9": lambda: M.water_cluster(9)}[mol]()
    bs = B.build_basis(m, basis)
    rng = np.random.default_rng(bs.nbasis)
    P, Q = _density(bs.nbasis, rng, 0.3), _density(bs.nbasis, rng, 0.2)
    eng = FockEngine(bs, cutoff=1e-11, precision=precision)
    shared = [(eng.fock2e(P), eng.fock2e_os(P, Q)) for _ in range(3)]   # eager, replayed, replayed again
    eng.set_timing(True)
    one, two = eng.fock2e(P), eng.fock2e_os(P, Q)
    eng.set_timing(False)
    # mixed precision: the FP32 launches' partial sums are FP32 inside a quartet only
    for G, (Ga, Gb) in shared:
        assert np.abs(G - one).max() < TOL * max(1.0, np.abs(one).max())
        assert np.abs(Ga - two[0]).max() < TOL * max(1.0, np.abs(two[0]).max())
        assert np.abs(Gb - two[1]).max() < TOL * max(1.0, np.abs(two[1]).max())
    eng.close()


def test_every_gradient_class_has_one_place():
    buckets = gen_grad.fuse_buckets()
    cls = [c for b in buckets for c in b["classes"]]
    assert len(set(cls)) == len(cls) and set(cls) == set(gen_grad.grad_classes())
    for b in buckets:
        for c in b["classes"]:
            assert b["coop"] != gen_grad.has_lane_grad(*c)
            t = gen_grad.grad_tables(*c)
            assert not b["coop"] or (t["glob"] == b["glob"] and t["total"] <= b["stride"])


@pytest.mark.gpu
@pytest.mark.parametrize("mol, basis", [("water", "STO-3G"), ("water", "6-31G*"), ("ethane", "6-31G*"),
                                        ("alkane4", "6-31G*"), ("waters8", "6-31G*")])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_shared_gradient_launches(mol, basis, precision):
    m = {"water": M.water, "ethane": lambda: M.alkane(2), "alkane4": lambda: M.alkane(4),
         "waters8": lambda: M.water_cluster(8)}[mol]()
    bs = B.build_basis(m, basis)
    P = _density(bs.nbasis, np.random.default_rng(bs.nbasis), 0.3)
    eng = FockEngine(bs, cutoff=1e-11, precision=precision)
    shared = [eng.eri_grad(P) for _ in range(3)]
    eng.set_timing(True)
    one = eng.eri_grad(P)
    eng.set_timing(False)
    # as above, with the contributions of up to 1e6 quartets to an atom
    for g in shared:
        assert np.abs(g - one).max() < 50 * TOL * max(1.0, np.abs(one).max())
    eng.close()
