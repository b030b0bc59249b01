"""FP64 exchange at the sizes where its tiling changes: below, at and past the
16-, 32- and 64-column tiles of the half-transform and the SYRK, one and many
vectors, orbital counts over every bank width, one and several orbital sets.

Reference: dense numpy products.  Tolerance, element by element, from the
rounding of sums of that length: |K - K_ref| <= 2 (2 n + M o + 16) u S with
S = sum_J (|L^J||C|)(|L^J||C|)^T and u = 2^-53 (each side rounds the
half-transform, n terms twice, and the sum over J and k, M o terms, and its
partial sums); J and V likewise."""
import numpy as np
import pytest
import torch

from _dense import lfull
from openmolcas_amd.fock import JKContext
from openmolcas_amd.synthetic import chol_vectors_np, npair, orbitals_np, pack

pytestmark = pytest.mark.gpu
U = 2.0 ** -53

CASES = [(1, 1, [1]), (2, 3, [2]), (15, 9, [3]), (16, 9, [4]), (17, 5, [16]), (24, 137, [5]), (31, 30, [7]),
         (32, 40, [17]), (33, 41, [5, 3]), (47, 25, [33]), (48, 26, [31]), (63, 20, [9]), (64, 700, [12]), (65, 33, [13]),
         (80, 31, [65]), (95, 12, [50]), (96, 12, [80]), (97, 12, [81]), (111, 9, [96]), (127, 9, [97]), (128, 8, [113]),
         (129, 10, [128]), (144, 7, [129]), (160, 6, [145]), (161, 5, [20, 1, 6]), (177, 4, [160]), (193, 3, [177]),
         (225, 4, [200]), (257, 5, [241]), (258, 2, [256]), (300, 400, [40, 0, 4]), (321, 17, [24])]


@pytest.mark.parametrize("n,M,occ", CASES)
def test_exchange_at_tile_edges(gpu, n, M, occ):
    L = chol_vectors_np(n, M, seed=n + M)
    Cs = [orbitals_np(n, min(o, n), seed=7 * n + d)[:, :o] if o else np.zeros((n, 0)) for d, o in enumerate(occ)]
    rng = np.random.default_rng(n)
    dlt = rng.standard_normal(npair(n))
    Lf = lfull(L, n)
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    Ct = [torch.from_numpy(np.ascontiguousarray(c)) for c in Cs]
    K0 = jk.exchange(Ct).cpu().numpy()
    J, K, V = (t.cpu().numpy() for t in jk.coulomb_exchange(torch.from_numpy(dlt), Ct, want_v=True))
    jk.close()
    assert np.array_equal(K0, K)  # the V pass inside the half-transform does not touch K
    for d, C in enumerate(Cs):
        if C.shape[1] == 0:
            assert np.all(K[d] == 0.0)
            continue
        X = (Lf.reshape(M * n, n) @ C).reshape(M, n, -1).transpose(1, 0, 2).reshape(n, -1)
        A = (np.abs(Lf).reshape(M * n, n) @ np.abs(C)).reshape(M, n, -1).transpose(1, 0, 2).reshape(n, -1)
        bound = 2.0 * (2 * n + M * C.shape[1] + 16) * U * (A @ A.T)
        assert np.all(np.abs(K[d] - pack(X @ X.T)) <= pack(bound)), (n, M, occ, d)
    v = L @ dlt
    vb = 2.0 * (npair(n) + 16) * U * (np.abs(L) @ np.abs(dlt))
    assert np.all(np.abs(V[:, 0] - v) <= vb)
    jb = 2.0 * (npair(n) + M + 16) * U * ((np.abs(L) @ np.abs(dlt)) @ np.abs(L))
    assert np.all(np.abs(J[0] - v @ L) <= jb)


@pytest.mark.parametrize("n,M,occ", [(40, 9, [3]), (41, 9, [21]), (60, 7, [38]), (150, 6, [130]), (170, 6, [70, 5, 66]),
                                     (180, 5, [161]), (210, 5, [120, 9, 14, 4, 6, 13, 11, 5, 10]), (230, 4, [225])])
@pytest.mark.parametrize("n_fp64", [0, 2, 3])
def test_fp64_head_and_fp32_tail_share_one_bank(gpu, n, M, occ, n_fp64):
    """Banks whose FP64 width in quarter tiles is not the reduced precisions' (an even
    number of tiles past eight).  The tail's rounding: the same sums at u = 2^-24, with
    three more for the inputs."""
    L = chol_vectors_np(n, M, seed=n + M)
    Cs = [orbitals_np(n, o, seed=7 * n + d) for d, o in enumerate(occ)]
    Lf = lfull(L, n)
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    K = jk.exchange_mixed([torch.from_numpy(np.ascontiguousarray(c)) for c in Cs], n_fp64, M).cpu().numpy()
    jk.close()
    for d, C in enumerate(Cs):
        X, A = Lf @ C, np.abs(Lf) @ np.abs(C)
        ref = sum(x @ x.T for x in X)
        head, tail = (sum((a @ a.T for a in s), np.zeros((n, n))) for s in (A[:n_fp64], A[n_fp64:]))
        c = 2.0 * (2 * n + M * C.shape[1] + 19)
        assert np.all(np.abs(K[d] - pack(ref)) <= pack(c * (U * head + 2.0 ** -24 * tail))), (n, M, occ, n_fp64, d)
