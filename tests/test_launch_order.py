"""Order and buffers of a build's launches, on the CPU: the library runs over
mock_hip.cpp, which records every launch with the launches it waits for.

A build is right for every timing if each class kernel starts after the
opening kernel (which clears the accumulators and writes the descriptors), has
ended when the closing kernel sums them, and shares its slice of the global
slot buffer with no kernel that may run at the same time."""
import pytest

from tests import mock_hip


@pytest.fixture(scope="module")
def mock(tmp_path_factory):
    return mock_hip.build(tmp_path_factory.mktemp("mock_hip"))


BUILD = """
import ctypes, numpy as np
from quick_amd import molecules as M
mock = start()

def check(ops, closing=True):
    opens = [i for i, o in enumerate(ops) if "k_open" in o.name]
    assert len(opens) == 1, [o.name for o in ops]
    classes = [i for i, o in enumerate(ops) if any(k in o.name for k in ("fock_", "fused_", "grad_"))]
    assert classes
    for i in classes:
        assert opens[0] in ops[i].before, ("not after the opening kernel", ops[i].name)
    if closing:
        close = [i for i, o in enumerate(ops) if "k_close" in o.name]
        assert len(close) == 1
        for i in classes:
            assert i in ops[close[0]].before, ("not complete at the closing kernel", ops[i].name)
    regions = []
    for i in classes:
        d = slice_doubles(ops[i].name)
        if d:
            a = ops[i].slots
            regions.append((i, a, a + 8 * d * ops[i].grid))
    for x, (i, a, b) in enumerate(regions):
        for j, c, d in regions[:x]:
            if j not in ops[i].before and i not in ops[j].before:
                assert b <= c or d <= a, ("two kernels share slots", ops[i].name[:40], ops[j].name[:40])
    return len(classes), len(regions)

def builds(e, kind, count=3, closing=True):
    n = e.n
    P, Q, F, H = (np.zeros((n, n)) for _ in range(4))
    p = lambda x: x.ctypes.data
    counts = []
    for _ in range(count):
        mock.mock_clear()
        if kind == "fock": e.fock2e_device(p(P), p(F))
        if kind == "os": e.fock2e_os_device(p(P), p(Q), p(F), p(H))
        if kind == "grad": e.eri_grad_device(p(P), p(F))
        ops = launches(mock)
        last = {int(x) for x in mock.mock_stream(None).decode().split()}
        done = last.union(*(ops[i].before for i in last))
        # the accumulator of zeros is filled once per engine, outside the build's graph
        assert done == set(range(len(ops))), "a launch is not ordered before the caller's next one"
        counts.append(check(ops, closing))
    return counts
"""

MOLECULES = [("M.water()", "6-31G*"), ("M.alkane(2)", "6-31G"), ("M.water()", "cc-pVTZ"), ("M.polyglycine(1)", "6-31G**"),
             ("M.alkane(18)", "6-31G*")]     # the last one above 256 functions


@pytest.mark.parametrize("form", [-1, 0, 1, 2])
@pytest.mark.parametrize("mol,basis", MOLECULES)
def test_open_shell_builds(mock, mol, basis, form):
    """Every open-shell form, the first build and the replayed ones: a class in
    the two-pass form issues two kernels, one after the other."""
    out = mock_hip.run(mock, BUILD + f"""
e = engine({mol}, "{basis}", prepare=False)
for cb in range(10):
    for ck in range(cb + 1):
        e.set_class_os(cb, ck, {form})
e.prepare()
c = builds(e, "os")
assert len(set(c)) == 1, c       # a replay issues what the first build issued
print(c)
""")
    print(out)


@pytest.mark.parametrize("two_pass", [[(9, 9)], [(8, 8)], [(9, 5), (9, 7)], [(9, 8), (8, 8), (5, 5)], []])
def test_slot_regions_of_shared_and_own_launches(mock, two_pass):
    """Classes with global slots, some in the two-pass form (a launch of their
    own), the others in a shared launch beside them."""
    mock_hip.run(mock, BUILD + f"""
e = engine(M.alkane(2), "def2-TZVP", prepare=False)
for cb, ck in {two_pass}:
    e.set_class_os(cb, ck, 1)
e.prepare()
c = builds(e, "os")
assert len(set(c)) == 1 and c[0][1] >= 1, c
""")


@pytest.mark.parametrize("mol,basis", MOLECULES)
@pytest.mark.parametrize("kind", ["fock", "os", "grad"])
def test_builds_of_every_kind(mock, mol, basis, kind):
    """Default forms, then a capped grid (one launch per class), then the timed path."""
    if kind == "grad" and "TZ" in basis:
        pytest.skip("no gradient of f shells")
    mock_hip.run(mock, BUILD + f"""
e = engine({mol}, "{basis}")
closing = {kind!r} != "grad"
assert len(set(builds(e, {kind!r}, closing=closing))) == 1
e.set_persistent(64)
assert len(set(builds(e, {kind!r}, closing=closing))) == 1
e.set_persistent(0)
if {kind!r} == "grad":
    e.set_grad_kernel(lane=False)
    assert len(set(builds(e, "grad", closing=False))) == 1
e.set_timing(True)
builds(e, {kind!r}, closing=closing)
""")


@pytest.mark.parametrize("call,fork_calls", [("hipStreamWaitEvent", 3), ("hipEventRecord", 1)])
def test_side_streams_are_joined_after_a_failure(mock, call, fork_calls):
    """A failing event call in the middle of a forked build (here under capture,
    where builds are issued launch by launch) is reported, and every launch that
    was made, except those behind a join that fails itself, is ordered before the
    caller's next one."""
    mock_hip.run(mock, BUILD + f"""
from quick_amd._lib import QuickFockError
e = engine(M.polyglycine(2), "6-31G**")
n = e.n
P, F = np.zeros((n, n)), np.zeros((n, n))
build = lambda: e.fock2e_device(P.ctypes.data, F.ctypes.data)
build()                                   # takes side streams
mock.mock_capture(None, 1)
mock.mock_clear()
build()
assert any(len(o.deps) > 1 for o in launches(mock)), "the captured build is not forked"
check(launches(mock))
for k in range(20):
    mock.mock_clear()
    mock.mock_fail(b"{call}", k)
    try:
        build()
    except QuickFockError as x:
        assert "mock" in str(x) and "{call}" in str(x), x
    else:
        assert k >= 4, k                  # the build makes fewer such calls
        break
    ops = launches(mock)
    last = {{int(x) for x in mock.mock_stream(None).decode().split()}}
    done = last.union(*(ops[i].before for i in last)) if last else set()
    lost = set(range(len(ops))) - done
    heads = [i for i in lost if not any(i in ops[j].before for j in lost)]
    assert len(heads) <= (1 if k >= {fork_calls} else 0), (k, [ops[i].name[:40] for i in heads])
    mock.mock_fail(b"", -1)
    mock.hipGetLastError()
    build()                               # the engine still builds
""")


@pytest.mark.parametrize("call", ["hipStreamCreateWithFlags", "hipEventCreateWithFlags", "hipGraphCreate",
                                  "hipGraphAddKernelNode", "hipGraphInstantiate", "hipHostMalloc"])
@pytest.mark.parametrize("after", [0, 1, 2])
def test_builds_go_on_without_streams_graphs_and_pinned_memory(mock, call, after):
    """What only makes a build faster may fail: the build is issued without it."""
    mock_hip.run(mock, BUILD + f"""
e = engine(M.polyglycine(2), "6-31G**")
mock.mock_fail(b"{call}", {after})
builds(e, "fock", 4)
mock.mock_fail(b"{call}", {after})
builds(e, "os", 4)
mock.mock_fail(b"{call}", {after})
builds(e, "grad", 4, closing=False)
P = np.zeros((e.n, e.n))
mock.mock_fail(b"{call}", 0)
e.fock2e(P), e.fock2e_os(P, P), e.eri_grad(P)
""")


def test_a_reported_error_is_reported_once(mock):
    mock_hip.run(mock, BUILD + """
from quick_amd._lib import QuickFockError
e = engine(M.water(), "6-31G*")
P = np.zeros((e.n, e.n))
for call in (b"hipLaunchKernel", b"hipStreamSynchronize", b"hipMemcpy"):
    mock.mock_fail(call, 0)
    try:
        e.fock2e(P, cutmatrix=np.ones((len(e.basis.shells),) * 2))
    except QuickFockError:
        pass
    else:
        assert 0, call
    e.fock2e(P)
""")


def test_hermite_only_classes_take_the_tile_above_256_functions(mock):
    """(dd|ds), (dd|pp) and (dp|dp) have no other LDS-tile kernel than the Hermite
    one, which is slower up to 256 functions and in batches of such molecules:
    there tile = 1, as in saved tables, keeps them on the wave-per-quartet kernel."""
    mock_hip.run(mock, BUILD + """
from quick_amd.engine import FockBatch
only = ("C2220", "C2211", "C2121")
def setup(n, tile):
    e = engine(M.alkane(n), "6-31G*", prepare=False)
    for cb in range(10):
        for ck in range(cb + 1):
            e.set_class_tuning(cb, ck, tile)
    e.prepare()
    assert (e.n > 256) == (n > 13)
    return e
def hermite():
    names = [o.name for o in launches(mock) if "fock_md_kernel" in o.name]
    return {c for c in only if any(c in x for x in names)}
for n, tile, want in ((1, 1, 0), (4, 1, 0), (13, 1, 0), (13, -1, 0), (14, 1, 3), (14, -1, 3), (14, 2, 0)):
    e = setup(n, tile)
    builds(e, "fock", 2)
    assert len(hermite()) == want, (n, tile, hermite())
    builds(e, "os", 2)
    assert not hermite()
    mock.mock_clear()
    b = FockBatch([e])
    b.build()
    assert len(hermite()) == want, (n, tile, hermite())
    b.close()
    e.close()
""")


@pytest.mark.parametrize("what", ["engine", "batch"])
def test_builds_beside_a_capture_of_the_same_engine(mock, what):
    """The side streams of an engine or batch that took part in a capture belong to
    it until it ends: a build on another stream meanwhile, captured or not, goes
    without them."""
    mock_hip.run(mock, BUILD + f"""
from quick_amd.engine import FockBatch
e = engine(M.polyglycine(2), "6-31G**")
n = e.n
P, F = np.zeros((n, n)), np.zeros((n, n))
if {what!r} == "batch":
    b = FockBatch([e])
    build = lambda s: b.build(s)
else:
    build = lambda s: e.fock2e_device(P.ctypes.data, F.ctypes.data, s)
one, two, three = 1 << 20, 2 << 20, 3 << 20     # three streams of the caller
build(one)
assert mock.mock_streams() == 3
def issue(s, name):
    mock.mock_clear()
    build(s)
    ops = launches(mock)
    assert {{int(x) for x in mock.mock_stream(s).decode().split()}}
    forked = any(len(o.deps) > 1 for o in ops)
    return forked
mock.mock_capture(one, 1)
assert issue(one, "captured")                    # forks
e.set_persistent(0)                              # no graph to replay: issued launch by launch
assert not issue(two, "beside it")
mock.mock_capture(three, 2)
assert not issue(three, "another capture beside it")
mock.mock_capture(one, 0)
mock.mock_capture(three, 0)
e.set_persistent(0)
assert issue(two, "after it")
""")


@pytest.mark.parametrize("mol,basis", [("M.polyglycine(1)", "6-31G**"), ("M.alkane(2)", "def2-TZVP"),
                                       ("M.alkane(14)", "6-31G*")])
def test_builds_need_nothing_but_what_prepare_made(mock, mol, basis):
    """While any stream of the process is captured the runtime refuses allocations
    and synchronous copies (and the capture is lost): a first build of any kind after
    a prepare makes neither, under capture or beside one, and issues the launches
    that later ones do."""
    mock_hip.run(mock, BUILD + f"""
kinds = ["fock", "os"] + ([] if "TZ" in "{basis}" else ["grad"])
e = engine({mol}, "{basis}")
for kind in kinds:
    builds(e, kind, 3, closing=kind != "grad")     # the buffers of its kind are allocated once
want = {{}}
for captured in (0, 1):
    e.set_cutoffs(1e-12)
    e.prepare()
    for kind in kinds:
        mock.mock_capture(None, captured)
        for call in (b"hipMalloc", b"hipMemcpy", b"hipHostMalloc", b"hipStreamSynchronize", b"hipDeviceSynchronize"):
            mock.mock_fail(call, 0)
            builds(e, kind, 1, closing=kind != "grad")
            assert mock.mock_failed() == 0, call
            names = sorted(o.name for o in launches(mock))
            assert want.setdefault(kind, names) == names
        mock.mock_fail(b"", -1)
        mock.mock_capture(None, 0)
""")


def test_setters_between_captured_calls_do_not_wait(mock):
    """Grid cap and gradient kernel may change inside a capture: replays that hold the
    old choice are put aside without a wait (which would end the capture) and
    given back later."""
    mock_hip.run(mock, BUILD + """
e = engine(M.polyglycine(1), "6-31G**")
for kind in ("fock", "os", "grad"):
    builds(e, kind, 3, closing=kind != "grad")
assert mock.mock_execs() == 3
for k in range(40):
    mock.mock_fail(b"hipDeviceSynchronize", 0)
    mock.mock_capture(None, 1)
    if k % 2: e.set_persistent(64 if k % 4 == 1 else 0)
    else: e.set_grad_kernel(k % 4 == 0)
    if k % 5 == 0: e.set_grad_class(1, 0, k % 2)
    for kind in ("fock", "os", "grad"):
        builds(e, kind, 1, closing=kind != "grad")
    mock.mock_capture(None, 0)
    assert mock.mock_failed() == 0
    mock.mock_fail(b"", -1)
    for kind in ("fock", "os", "grad"):
        builds(e, kind, 2, closing=kind != "grad")
    assert mock.mock_execs() <= 3 + 16
e.set_cutoffs(1e-11)
e.prepare()
assert mock.mock_execs() == 0
builds(e, "fock", 2)
e.set_persistent(8)
e.close()
assert mock.mock_execs() == 0
""")


def test_device_bytes_counts_every_task_table(mock):
    """stats()["device_bytes"] follows what is allocated, whether or not classes
    have a second table of wave-per-quartet tasks."""
    mock_hip.run(mock, BUILD + """
held = []
for tile in (-1, 2):
    e = engine(M.water_cluster(16), "6-31G*", prepare=False)
    for c in ((4, 2), (4, 4), (5, 2), (5, 3)):
        e.set_class_tuning(*c, tile)
    before = mock.mock_bytes()
    e.prepare()
    held.append((mock.mock_bytes() - before, e.stats()["device_bytes"]))
    e.close()
(a, x), (b, y) = held
# buffers that the figure leaves out (descriptors, counters, shell maps) differ by
# 43 KB between the two engines; the second table holds 2 MB
assert abs((x - y) - (a - b)) < 200000, held
""")
