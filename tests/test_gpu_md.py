"""The Hermite-Gaussian tile kernels (fock_md_kernel), default above 256
functions, agree with the wave-per-quartet kernels of the same classes in the
Fock build, and the open-shell build and the gradient, which run the
wave-per-quartet tasks beside them, are unchanged.  Both forms are FP64 with
errors of a few ulp per integral and sums in another order: 1e-11 of the
largest element.  On small molecules the kernels are asked for, at the edges
of a wave (one ket, partial and full windows) and with split primitive pairs."""
import numpy as np
import pytest

from tests.helpers import announce, molecule, oracle_for, product_basis, seeded_density_for

pytestmark = pytest.mark.gpu

MD = [(4, 2), (5, 3), (5, 2), (4, 4)]   # (dp|pp), (dd|ds), (dd|pp), (dp|dp)


def close(x, y):
    assert np.abs(x - y).max() <= 1e-11 * max(1.0, np.abs(y).max())


@pytest.mark.parametrize("name,basis", [("water", "6-31G*"), ("LiF", "cc-pVDZ"), ("water3", "cc-pVDZ"),
                                        ("alkane2", "6-31G**"), ("gly1", "6-31G*")])
@pytest.mark.parametrize("shape", [(1, 1, 2, 1, 0), (1, 4, 16, 4, -1), (1, 2, 4, 2, 1)])
def test_md_tile_kernels_match_the_oracle(name, basis, shape):
    announce("md %s %s %s" % (name, basis, shape))
    from quick_amd.engine import FockEngine
    mol = molecule(name)
    orc = oracle_for(mol, basis)
    P, _ = seeded_density_for(orc, mol)
    e = FockEngine(product_basis(mol, basis), cutoff=1e-12)
    for cb, ck in MD:
        e.set_class_tuning(cb, ck, *shape[:4])
        e.set_class_piece(cb, ck, shape[4])
    assert np.abs(e.fock2e(P) - orc.fock2e(P, cutoff=1e-12)[0]).max() <= 1e-10


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_md_defaults_above_256_functions(precision):
    announce("md defaults %s" % precision)
    from quick_amd.engine import FockEngine
    from quick_amd.scf import seeded_density
    bs = product_basis(molecule("water14"), "6-31G*")          # 266 functions
    a, b = (FockEngine(bs, cutoff=1e-10, precision=precision) for _ in range(2))
    for cb, ck in MD[1:]:
        b.set_class_tuning(cb, ck, 2)
    S = a.one_electron()[0]
    P, Q = seeded_density(S, 70), seeded_density(S, 69, seed=3)
    close(a.fock2e(P), b.fock2e(P))
    for x, y in zip(a.fock2e_os(P / 2, Q / 2), b.fock2e_os(P / 2, Q / 2)):
        close(x, y)
    close(a.eri_grad(P), b.eri_grad(P))


@pytest.mark.parametrize("name,basis,copies", [("water", "6-31G*", 14), ("water", "cc-pVDZ", 11), ("LiF", "cc-pVDZ", 9)])
@pytest.mark.parametrize("shape", [(1, 1, 2, 1, 0), (1, 4, 16, 4, -1), (1, 2, 4, 2, 1)])
def test_md_tile_kernels_above_256_functions_match_the_oracle(name, basis, copies, shape):
    """Copies so far apart that the quartets are those of the pairs of single
    molecules: short ket windows in every class."""
    announce("md copies %s %s %s" % (name, basis, shape))
    from quick_amd.basis import Molecule
    from quick_amd.engine import FockEngine
    one = molecule(name)
    mol = Molecule(list(one.symbols) * copies,
                   np.concatenate([one.xyz + np.array([20.0 * k, 3.0 * (k % 2), 0.0]) for k in range(copies)]))
    orc = oracle_for(mol, basis)
    P, _ = seeded_density_for(orc, mol)
    bs = product_basis(mol, basis)
    assert bs.nbasis > 256
    e = FockEngine(bs, cutoff=1e-10)
    for cb, ck in MD:
        e.set_class_tuning(cb, ck, *shape[:4])
        e.set_class_piece(cb, ck, shape[4])
    assert np.abs(e.fock2e(P) - orc.fock2e(P, cutoff=1e-10)[0]).max() <= 1e-10
