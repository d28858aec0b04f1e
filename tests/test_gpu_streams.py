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


def test_replayed_builds_follow_every_change():
    """From the second build on the class launches are replayed: other buffers,
    a changed cutoff, grid cap or kernel choice and builds of another kind
    between them must all show in the result."""
    announce("streams replay")
    from quick_amd.engine import FockEngine
    eng, P, G = setup("gly1")
    s = torch.cuda.current_stream().cuda_stream

    def closed(density, want):
        F = torch.zeros_like(density)
        eng.fock2e_device(density.data_ptr(), F.data_ptr(), s)
        torch.cuda.synchronize()
        close(F, want)

    Q = P * torch.linspace(0.5, 1.5, P.shape[0], dtype=P.dtype, device="cuda")
    Q = 0.5 * (Q + Q.T).contiguous()
    other = FockEngine(eng.basis, cutoff=eng.cutoff)
    other.set_timing(True)
    GQ = other.fock2e(Q.cpu().numpy())
    g = other.eri_grad(P.cpu().numpy())
    Ga, Gb = other.fock2e_os(P.cpu().numpy() / 2, Q.cpu().numpy() / 2)
    for _ in range(3):
        closed(P, G)
        closed(Q, GQ)
        assert np.abs(eng.eri_grad(P.cpu().numpy()) - g).max() <= 1e-11 * np.abs(g).max()
        a, b = eng.fock2e_os(P.cpu().numpy() / 2, Q.cpu().numpy() / 2)
        close(torch.from_numpy(a), Ga)
        close(torch.from_numpy(b), Gb)
    eng.set_persistent(64)
    eng.set_grad_kernel(lane=False)
    closed(P, G)
    for _ in range(3):
        assert np.abs(eng.eri_grad(P.cpu().numpy()) - g).max() <= 1e-11 * np.abs(g).max()
    eng.set_cutoffs(1e-6)
    other.set_cutoffs(1e-6)
    loose = other.fock2e(P.cpu().numpy())
    assert np.abs(loose - G).max() > 1e-9     # the cutoff shows
    for _ in range(3):
        closed(P, loose)
    eng.close()                               # a replay may still be in flight in a user's program
    other.close()


@pytest.mark.parametrize("name", ["water", "gly1"])
def test_builds_in_flight_keep_their_own_buffers(name):
    """Many builds queued without a wait, each with its own density and Fock
    matrix: a replay's arguments are changed while earlier ones still run."""
    announce("streams in flight %s" % name)
    eng, P, G = setup(name)
    s = torch.cuda.current_stream().cuda_stream
    scale = [1.0 + 0.25 * k for k in range(24)]
    Ps = [P * x for x in scale]
    Fs = [torch.zeros_like(P) for _ in scale]
    gs = [torch.zeros(eng.basis.mol.natom, 3, dtype=P.dtype, device="cuda") for _ in scale]
    torch.cuda.synchronize()
    for k in range(len(scale)):
        eng.fock2e_device(Ps[k].data_ptr(), Fs[k].data_ptr(), s)
        eng.eri_grad_device(Ps[k].data_ptr(), gs[k].data_ptr(), s)
    torch.cuda.synchronize()
    one = gs[0].cpu().numpy()
    for x, F, g in zip(scale, Fs, gs):
        # G is linear in P up to the quartets that the density screen drops or keeps
        assert np.abs(F.cpu().numpy() - x * G).max() <= 1e-8
        assert np.abs(g.cpu().numpy() - x * x * one).max() <= 1e-7


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


@pytest.mark.parametrize("name,basis", [("water16", "6-31G*"), ("water3", "6-31G*")])
def test_first_open_shell_build_and_gradient_under_capture(name, basis):
    """The first calls after a prepare, which has made everything they need, under
    capture and, on another stream, beside it (where an allocation or a synchronous
    copy would end the capture)."""
    announce("streams first call under capture %s" % name)
    eng, P, _ = setup(name, basis, cutoff=1e-10)
    Q = (0.3 * P).contiguous()
    s = torch.cuda.Stream()
    Fa, Fb = torch.zeros_like(P), torch.zeros_like(P)
    g = torch.zeros(eng.basis.mol.natom, 3, dtype=P.dtype, device="cuda")

    def calls():
        for x in (Fa, Fb, g):
            x.zero_()
        eng.fock2e_os_device(P.data_ptr(), Q.data_ptr(), Fa.data_ptr(), Fb.data_ptr(), s.cuda_stream)
        eng.eri_grad_device(P.data_ptr(), g.data_ptr(), s.cuda_stream)

    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(3):              # allocates the buffers of both kinds
            calls()
    s.synchronize()
    want = [x.cpu().numpy() for x in (Fa, Fb, g)]
    eng.set_cutoffs(1e-10)
    eng.prepare()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(graph, stream=s):
            calls()
    for k in range(4):                  # eager calls between the replays
        graph.replay()
        torch.cuda.synchronize()
        for x, w in zip((Fa, Fb, g), want):
            assert np.abs(x.cpu().numpy() - w).max() <= 1e-11 * max(1.0, np.abs(w).max())
        with torch.cuda.stream(s):
            calls()
        s.synchronize()
        for x, w in zip((Fa, Fb, g), want):
            assert np.abs(x.cpu().numpy() - w).max() <= 1e-11 * max(1.0, np.abs(w).max())
    eng.set_cutoffs(1e-10)
    eng.prepare()
    beside = torch.cuda.CUDAGraph()
    t = torch.cuda.Stream()
    for x in (Fa, Fb, g):
        x.zero_()
    F = torch.zeros_like(P)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        with torch.cuda.graph(beside, stream=s):
            eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
            eng.fock2e_os_device(P.data_ptr(), Q.data_ptr(), Fa.data_ptr(), Fb.data_ptr(), t.cuda_stream)
            eng.eri_grad_device(P.data_ptr(), g.data_ptr(), t.cuda_stream)
    torch.cuda.synchronize()
    for x, w in zip((Fa, Fb, g), want):
        assert np.abs(x.cpu().numpy() - w).max() <= 1e-11 * max(1.0, np.abs(w).max())


def test_batch_build_beside_a_capture_of_the_batch():
    """While a capture holds the batch's side streams, a build on another stream
    goes without them and disturbs neither."""
    announce("streams batch beside capture")
    from quick_amd.engine import FockBatch
    sets = [setup(n) for n in ("water", "water3")]
    b = FockBatch([e for e, _, _ in sets])
    for i, (_, P, _) in enumerate(sets):
        b.set_density(i, P.cpu().numpy())
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    b.build(s.cuda_stream)
    torch.cuda.synchronize()
    b.clear_fock(t.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
            b.build(s.cuda_stream)
            b.build(t.cuda_stream)
    torch.cuda.synchronize()
    for k in range(3):                  # the build on t, then each replay
        for i, (_, _, G) in enumerate(sets):
            F = b.get(i, g=False, f=True)[1]
            assert np.abs(F - (k + 1) * G).max() <= 1e-11 * max(1.0, np.abs(G).max())
        g.replay()
        torch.cuda.synchronize()
    b.close()


def test_setters_inside_a_capture():
    """A changed gradient kernel and grid cap inside a capture, after replayed calls."""
    announce("streams setters inside a capture")
    eng, P, G = setup("water3")
    s = torch.cuda.Stream()
    F = torch.zeros_like(P)
    g = torch.zeros(eng.basis.mol.natom, 3, dtype=P.dtype, device="cuda")

    def calls():
        F.zero_()
        g.zero_()
        eng.fock2e_device(P.data_ptr(), F.data_ptr(), s.cuda_stream)
        eng.eri_grad_device(P.data_ptr(), g.data_ptr(), s.cuda_stream)

    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        eng.set_grad_kernel(lane=False)
        calls()                         # the buffers of both kernels
        eng.set_grad_kernel(lane=True)
        for _ in range(3):
            calls()
    s.synchronize()
    want = g.cpu().numpy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(graph, stream=s):
            eng.set_persistent(64)
            eng.set_grad_kernel(lane=False)
            calls()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        close(F, G)
        assert np.abs(g.cpu().numpy() - want).max() <= 1e-11 * np.abs(want).max()
        with torch.cuda.stream(s):
            calls()
        s.synchronize()
        close(F, G)
        assert np.abs(g.cpu().numpy() - want).max() <= 1e-11 * np.abs(want).max()
