"""Calls with host matrices, which pass them through pinned memory up to 80000
doubles and copy them above, against the calls with device matrices: the same
kernels add the same terms in another order (2.2e-16 x 1e4 terms x 10: 2e-11)."""
import numpy as np
import pytest
import torch

from quick_amd import basis as B
from quick_amd import molecules as M
from quick_amd.engine import FockEngine

TOL = 2e-11


# closed shell: up to 200 functions through pinned memory; open shell: up to 141
@pytest.mark.gpu
@pytest.mark.parametrize("mol, basis", [(lambda: M.water(), "STO-3G"), (lambda: M.water_cluster(7), "6-31G*"),
                                        (lambda: M.water_cluster(8), "cc-pVDZ"),
                                        (lambda: M.water_cluster(9), "cc-pVDZ")])
def test_host_calls(mol, basis):
    m = mol()
    bs = B.build_basis(m, basis)
    n = bs.nbasis
    eng = FockEngine(bs, cutoff=1e-11)
    rng = np.random.default_rng(n)
    s = torch.cuda.current_stream().cuda_stream
    dev = lambda a: torch.from_numpy(a).to("cuda:0")
    for k in range(3):                     # eager, replayed, replayed with new matrices
        P, Q = (0.1 * (a + a.T) for a in rng.standard_normal((2, n, n)))
        dP, dQ = dev(P), dev(Q)
        F, Fa, Fb = (torch.zeros_like(dP) for _ in range(3))
        g = torch.zeros(m.natom, 3, dtype=torch.float64, device="cuda:0")
        host = eng.fock2e(P), eng.fock2e_os(P, Q), eng.eri_grad(P)
        eng.fock2e_device(dP.data_ptr(), F.data_ptr(), s)
        eng.fock2e_os_device(dP.data_ptr(), dQ.data_ptr(), Fa.data_ptr(), Fb.data_ptr(), s)
        eng.eri_grad_device(dP.data_ptr(), g.data_ptr(), s)
        torch.cuda.synchronize()
        for a, b, f in ((host[0], F, 1), (host[1][0], Fa, 1), (host[1][1], Fb, 1), (host[2], g, 50)):
            b = b.cpu().numpy()
            assert np.abs(a - b).max() < f * TOL * max(1.0, np.abs(b).max())
    eng.close()
