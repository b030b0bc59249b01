"""Device memory that an exchange takes beside the vectors: X within its budget, and the
partial tiles of all chunks together within a sixteenth of it (here 4 chunks of 1 GiB;
their slices by time alone would take 268 MB more)."""
import torch
import pytest

from openmolcas_amd.fock import JKContext

pytestmark = pytest.mark.gpu


def test_partial_tiles_stay_within_their_share(gpu):
    n, M, o, budget = 448, 4000, 200, 1 << 30
    npair = n * (n + 1) // 2
    g = torch.Generator(device=gpu)
    g.manual_seed(1)
    jk = JKContext(n, M, device=gpu)
    L = torch.randn(M, npair, dtype=torch.float64, device=gpu, generator=g)
    jk.upload_packed(L)
    C = torch.randn(n, o, dtype=torch.float64, device=gpu, generator=g)
    K = torch.zeros(n, n, dtype=torch.float64, device=gpu)
    i, j = torch.tril_indices(n, n, device=gpu)
    for s in range(0, M, 500):
        F = torch.zeros(len(L[s:s + 500]), n, n, dtype=torch.float64, device=gpu)
        F[:, i, j] = L[s:s + 500]
        F[:, j, i] = L[s:s + 500]
        X = (F.reshape(-1, n) @ C).reshape(-1, n, o).transpose(0, 1).reshape(n, -1)
        K += X @ X.T
    del F, X, L
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    jk.set_x_budget(budget)
    before = torch.cuda.mem_get_info()[0]
    k = jk.exchange([C])
    torch.cuda.synchronize()
    assert before - torch.cuda.mem_get_info()[0] <= budget + budget // 16 + (64 << 20)
    # sums of 2 n and M o terms on both sides, in units of the largest element
    assert float((k[0] - K[i, j]).abs().max()) <= 2 * (2 * n + M * o) * 2.0 ** -53 * float(K.abs().max())
    jk.close()
