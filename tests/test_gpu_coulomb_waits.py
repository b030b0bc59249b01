"""Every wait of the one-pass Coulomb kernel has a limit.  With a limit of zero looks a
value that is not there at once counts as lost: the call still ends, each J and V is the
right one (the same bits) or NaN, and with the default limit all are right again - with
the workgroups of a group together and, with no looks for them to meet, apart."""
import pytest
import torch

from openmolcas_amd.fock import JKContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,M", [(128, 300), (301, 400), (701, 60)])
@pytest.mark.parametrize("nd", [1, 2])
@pytest.mark.parametrize("looks", [64, 0])
def test_lost_values_end_the_wait(gpu, n, M, nd, looks):
    npair = n * (n + 1) // 2
    g = torch.Generator(device=gpu)
    g.manual_seed(n + M)
    L = torch.randn(M, npair, dtype=torch.float64, device=gpu, generator=g)
    d = torch.randn(nd, npair, dtype=torch.float64, device=gpu, generator=g)
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    want = jk.coulomb(d, want_v=True)
    jk.set_coulomb_looks(looks)
    jk.set_coulomb_waits(0)
    for got, w in zip(jk.coulomb(d, want_v=True), want):
        assert bool((got.isnan() | (got == w)).all())
    jk.set_coulomb_waits()
    for got, w in zip(jk.coulomb(d, want_v=True), want):
        assert torch.equal(got, w)
    jk.close()


def test_waits_below_zero_are_refused(gpu):
    jk = JKContext(4, 1, device=gpu)
    with pytest.raises(Exception):
        jk.set_coulomb_waits(-1)
    jk.close()
