"""(pw|xy) of the device engine over the edges of its tiles: pairs xy below, at
and past 16 and 64, active orbitals over the bank and Z = X C widths (16, 128),
one slice and many, the vectors in one chunk and in several.

Reference: dense numpy.  Tolerance, element by element, from the rounding of
sums of that length: 2 (3 n + M + 16) u |C|^T |L^J| |C| ... with u = 2^-53 (three
sums over n, one over M, on each side)."""
import numpy as np
import pytest
import torch

from _dense import lfull
from openmolcas_amd.fock import JKContext
from openmolcas_amd.synthetic import chol_vectors_np, orbitals_np

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def pwxy(Lf, c3, cmo):
    h = Lf @ c3                                           # (J, a, w)
    na = c3.shape[1]
    ix = [(x, y) for y in range(na) for x in range(y + 1)]
    z = np.matmul(c3.T, h)[:, [i[0] for i in ix], [i[1] for i in ix]]
    pw = np.matmul(cmo.T, h)                              # (J, p, w)
    return (z.T @ pw.transpose(0, 2, 1).reshape(Lf.shape[0], -1)).reshape(-1)


@pytest.mark.parametrize("n,M,na,nfro,norb,budget", [
    (5, 3, 1, 0, 5, 0), (24, 40, 5, 2, 20, 0), (33, 700, 6, 0, 33, 0), (64, 130, 11, 1, 60, 0), (65, 129, 10, 0, 65, 0),
    (70, 66, 16, 3, 17, 0), (130, 37, 17, 0, 64, 0), (97, 65, 2, 0, 97, 0), (140, 3, 129, 4, 2, 0), (80, 300, 12, 0, 80, 1 << 20),
])
def test_pwxy_at_tile_edges(gpu, n, M, na, nfro, norb, budget):
    L = chol_vectors_np(n, M, seed=n)
    cmo = orbitals_np(n, n, seed=n + 1)
    c3 = np.ascontiguousarray(cmo[:, -na:])
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    if budget:
        jk.set_x_budget(budget)
    w = jk.puvx(torch.from_numpy(c3), torch.from_numpy(cmo), nfro, norb).cpu().numpy()
    jk.close()
    Lf, co = lfull(L, n), cmo[:, nfro:nfro + norb]
    bound = 2.0 * (3 * n + M + 16) * U * pwxy(np.abs(Lf), np.abs(c3), np.abs(co))
    assert np.all(np.abs(w - pwxy(Lf, c3, co)) <= bound)
