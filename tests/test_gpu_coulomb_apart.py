"""The one-pass Coulomb kernel where the workgroups of a group work apart: the V parts of
a slice in one or several runs of vectors (from 32 vectors a group on), four vectors
a step with one to three left over.  Apart (no looks for the others), together and in the two launches of
mjk_coulomb_noalloc: the same bits, and right.

Reference: torch in float64; V within 2 (np + 16) u |L||D|, J within
2 (np + M + 16) u |L|^T |L||D|, u = 2^-53 (rounding of sums of that length, both sides)."""
import ctypes

import pytest
import torch

from openmolcas_amd.fock import JKContext

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("n,M", [(130, 1025), (301, 1203), (512, 510), (512, 1000), (701, 191), (701, 250), (900, 700),
                                 (1150, 66), (1200, 131)])
@pytest.mark.parametrize("nd", [1, 2])
def test_apart_gives_the_same_bits(gpu, n, M, nd):
    npair = n * (n + 1) // 2
    g = torch.Generator(device=gpu)
    g.manual_seed(n * 1000 + M)
    L = torch.randn(M, npair, dtype=torch.float64, device=gpu, generator=g)
    d = torch.randn(nd, npair, dtype=torch.float64, device=gpu, generator=g)
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    j, v = jk.coulomb(d, want_v=True)
    jk.set_coulomb_looks(0)
    j0, v0 = jk.coulomb(d, want_v=True)
    assert torch.equal(j, j0) and torch.equal(v, v0)
    j1, v1 = torch.empty_like(j), torch.empty_like(v)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    torch.cuda.synchronize()
    jk._check(jk.lib.mjk_coulomb_noalloc(jk._h, nd, p(d), npair, p(j1), npair, p(v1)))
    jk.sync()
    assert torch.equal(j, j1) and torch.equal(v, v1)
    va = L.abs() @ d.abs().T
    assert bool(((v - L @ d.T).abs() <= 2 * (npair + 16) * U * va).all())
    assert bool(((j - (L @ d.T).T @ L).abs() <= 2 * (npair + M + 16) * U * (va.T @ L.abs())).all())
    jk.close()
