"""dE/dL from Z at the sizes where its tiling changes: strips of 32 rows, chunks
of 16 orbitals and their last steps, groups of four vectors, every bank width of
the fused kernel and the first past it, the density given and not, and the FP32
tail.  Z is any matrix (not symmetric), so the order of its indices counts.

Reference: dense numpy.  Tolerance, element by element: each side rounds two
sums over the orbitals and the V P term, 2 (3 o + 8) u S with S = |alpha V| |P| +
|beta| |C||Z||C|^T, u = 2^-53 (2^-24 on the C Z C^T part of an FP32 vector)."""
import numpy as np
import pytest
import torch

from openmolcas_amd.fock import JKContext
from openmolcas_amd.synthetic import chol_vectors_np, npair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,M,o", [
    (1, 1, 1), (5, 3, 2), (31, 4, 3), (32, 5, 4), (33, 9, 5), (63, 2, 15), (64, 6, 16), (65, 3, 17), (96, 7, 33),
    (97, 4, 48), (100, 5, 49), (128, 3, 64), (129, 5, 65), (130, 4, 80), (161, 3, 83), (150, 6, 96), (160, 5, 97),
    (177, 2, 112), (190, 5, 113), (200, 3, 126), (131, 4, 128), (140, 3, 129), (300, 41, 31),
])
@pytest.mark.parametrize("with_p", [False, True])
def test_grad_vectors_at_tile_edges(gpu, n, M, o, with_p):
    rng = np.random.default_rng(n * 1000 + o)
    C = rng.standard_normal((n, o)) / np.sqrt(n)
    Z = rng.standard_normal((M, o, o))
    V = rng.standard_normal(M)
    alpha, beta = 1.25, -2.0
    P = 2.0 * C @ C.T
    if with_p:
        P = P + 0.5 * np.eye(n)
    i, j = np.tril_indices(n)
    s = np.where(i == j, 1.0, 2.0)
    cz = np.matmul(np.matmul(C, Z), C.T)[:, i, j]
    want = s * (alpha * V[:, None] * P[i, j] + beta * cz)
    size_p = (2.0 * np.abs(C) @ np.abs(C).T + (0.5 * np.eye(n) if with_p else 0.0))[i, j]
    size_z = np.matmul(np.matmul(np.abs(C), np.abs(Z)), np.abs(C).T)[:, i, j]
    vp = np.abs(alpha * V)[:, None] * size_p
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(chol_vectors_np(n, M, seed=1))
    t = [torch.tensor(x, device=gpu) for x in (C, V, Z)]
    kw = {"p_lt": torch.tensor(P[i, j], device=gpu)} if with_p else {}
    for f in (None, 0, M // 2):
        got = jk.grad_vectors(t[0], t[1], alpha, beta, z=t[2], fp32_from=f, **kw).cpu().numpy()
        u = np.full((M, 1), 2.0 ** -53)
        if f is not None:
            u[f:] = 2.0 ** -24
        bound = s * 2.0 * (3 * o + 8) * (2.0 ** -53 * vp + u * abs(beta) * size_z)
        assert np.all(np.abs(got - want) <= bound), (f, np.max(np.abs(got - want) / bound))
    assert got.shape == (M, npair(n))
    jk.close()
