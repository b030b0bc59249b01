"""J and V of one and two densities where one read of the vectors serves both: the
ends of its range of sizes (8192 and 786432 pairs), one workgroup a vector
and many, slices that do not divide the pairs, few vectors and more than the groups
take evenly - with the workgroups of a group working together, and apart (the same bits).

Reference: torch in float64.  Tolerance from the rounding of sums of that length, on
both sides: V within 2 (np + 16) u |L||D|, J within 2 (np + M + 16) u |L|^T |L||D|,
u = 2^-53."""
import pytest
import torch

from openmolcas_amd.fock import JKContext

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("n,M", [
    (89, 40), (124, 33), (126, 1), (128, 300), (129, 7), (157, 63), (158, 640), (223, 1100), (301, 64), (350, 257), (512, 130),
    (701, 25), (800, 3), (1140, 4), (1150, 2), (1250, 2), (1260, 1),
])
@pytest.mark.parametrize("nd", [1, 2])
def test_coulomb_one_pass(gpu, n, M, nd):
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
    jk.set_coulomb_looks()
    j1, v1 = jk.coulomb(d, want_v=True)
    assert torch.equal(j, j0) and torch.equal(v, v0) and torch.equal(j, j1) and torch.equal(v, v1)
    va = L.abs() @ d.abs().T
    assert bool(((v - L @ d.T).abs() <= 2 * (npair + 16) * U * va).all())
    assert bool(((j - (L @ d.T).T @ L).abs() <= 2 * (npair + M + 16) * U * (va.T @ L.abs())).all())
    jk.close()


def test_looks_below_zero_are_refused(gpu):
    jk = JKContext(4, 1, device=gpu)
    with pytest.raises(Exception):
        jk.set_coulomb_looks(-1)
    jk.close()


def test_coulomb_one_pass_on_two_streams(gpu):
    """Two contexts at once: each launch asks for the whole GPU."""
    n, M = 301, 900
    npair = n * (n + 1) // 2
    L = torch.randn(M, npair, dtype=torch.float64, device=gpu)
    d = torch.randn(1, npair, dtype=torch.float64, device=gpu)
    ctx = [JKContext(n, M, device=gpu) for _ in range(2)]
    for c in ctx:
        c.upload_packed(L)
    want = ctx[0].coulomb(d)
    torch.cuda.synchronize()
    st = [torch.cuda.Stream() for _ in ctx]
    for c, s in zip(ctx, st):
        c.bind_stream(s)
    out = []
    for _ in range(10):
        for c, s in zip(ctx, st):
            with torch.cuda.stream(s):
                out.append(c.coulomb(d))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in out)
    for c in ctx:
        c.close()
