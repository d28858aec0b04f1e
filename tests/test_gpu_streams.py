"""The class launches of a build are forked over side streams and joined
again: a caller's stream, a captured graph (its side streams taken by an
earlier eager build, or none of them: a first build under capture runs on the
caller's stream alone) and builds of several engines from several threads
all give the Fock matrix of the timed build, whose launches run one after
another.  Sums in another order differ by rounding only: 1e-12 of the largest
element, as the other same-algorithm comparisons of this suite."""
import threading

import numpy as np
import pytest

from tests.helpers import announce, molecule, product_basis

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def setup(name="water3", basis="6-31G*", cutoff=1e-11):
    from quick_amd.engine import FockEngine
    from quick_amd.scf import seeded_density
    mol = molecule(name)
    eng = FockEngine(product_basis(mol, basis), cutoff=cutoff)
    P = seeded_density(eng.one_electron()[0], mol.nelec() // 2)
    eng.set_timing(True)                # one stream, no fork
    G = eng.fock2e(P)
    eng.set_timing(False)
    return eng, torch.from_numpy(P).cuda(), G


def close(F, G):
    assert np.abs(F.cpu().numpy() - G).max() <= 1e-12 * max(1.0, np.abs(G).max())


@pytest.mark.parametrize("name,basis", [("water", "6-31G*"), ("gly1", "6-31G*"), ("water", "cc-pVTZ")])
def test_forked_build_on_a_caller_stream(name, basis):
    announce("streams %s %s" % (name, basis))
    eng, P, G = setup(name, basis)
    F = torch.empty_like(P)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(3):              # the fill and the copy are ordered by the stream alone
            F.zero_()
            eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
            R = F.clone()
    s.synchronize()
    close(R, G)


@pytest.mark.parametrize("warm", [True, False])
def test_forked_build_in_a_captured_graph(warm):
    announce("streams graph warm=%s" % warm)
    eng, P, G = setup()
    F = torch.zeros_like(P)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        if warm:
            eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            F.zero_()
            eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
    other = torch.zeros_like(P)
    for k in range(4):                  # eager builds of the same engine between the replays
        F.fill_(k)
        g.replay()
        torch.cuda.synchronize()
        close(F, G)
        other.zero_()
        eng.fock2e_device(P.data_ptr(), other.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        close(other, G)


def test_forked_builds_of_several_threads():
    announce("streams threads")
    sets = [setup(n) for n in ("water", "water3", "alkane2")]
    out, errors = [None] * len(sets), []

    def work(k):
        try:
            eng, P, _ = sets[k]
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.default_stream())
            with torch.cuda.stream(s):
                F = torch.zeros_like(P)
                for _ in range(5):
                    F.zero_()
                    eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
            s.synchronize()
            out[k] = F
        except Exception as e:          # reported below: an assertion in a thread is lost
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for F, (_, _, G) in zip(out, sets):
        close(F, G)
