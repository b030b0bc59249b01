"""mjk_coulomb_noalloc waits for nothing on the device: overlapping calls on one GPU
share its scratch, so a value that a kernel waited for there could be taken away again
and the kernel would never end.  One and two densities therefore run as two launches,
V first, then J, where mjk_coulomb reads the vectors once with workgroups that wait for
each other; the values are the same bits (n = 128: one slice per group at the least
size, 301 and 512: several groups, 1140: two groups, 1260: two passes on either entry).

The launches are counted through the phase times (V pass: one per call)."""
import ctypes

import pytest
import torch

from openmolcas_amd.fock import JKContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,M", [(128, 300), (301, 64), (512, 130), (1140, 4), (1260, 2)])
@pytest.mark.parametrize("nd", [1, 2])
def test_noalloc_in_two_launches(gpu, n, M, nd):
    npair = n * (n + 1) // 2
    g = torch.Generator(device=gpu)
    g.manual_seed(n + M)
    L = torch.randn(M, npair, dtype=torch.float64, device=gpu, generator=g)
    d = torch.randn(nd, npair, dtype=torch.float64, device=gpu, generator=g)
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    want, vwant = jk.coulomb(d, want_v=True)
    j = torch.full((nd, npair), float("nan"), dtype=torch.float64, device=gpu)
    v = torch.full((M, nd), float("nan"), dtype=torch.float64, device=gpu)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    jk.set_profiling(True)
    jk._check(jk.lib.mjk_coulomb_noalloc(jk._h, nd, p(d), npair, p(j), npair, p(v)))
    phases = jk.phase_times()
    jk.set_profiling(False)
    assert torch.equal(j, want) and torch.equal(v, vwant)
    assert phases["coulomb_v"][1] == 1 and phases["coulomb_j"][1] == 1
    jk.close()
