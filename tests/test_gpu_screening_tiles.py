"""What mjk_exchange_screened leaves out, tile by tile, against a numpy model of the rule:

* half-transform: X^J[:, 64 AOs] = 0 when ||L^J[:, tile]||_F max_d ||C_d||_F < thr_x;
* K: the part of a TM x TM tile that a slice of the vectors gives is left out when
  sum_J ||X^J_A||_F ||X^J_B||_F < tau.  TM is 128 from nbas = 385 on, else 64, or the
  tile of mjk_set_tuning; the slices share out one to eight rounds of two workgroups per
  compute unit, or the split target, over the tiles of nbas rounded up to 128.  (FP32
  tests its own slices, counted over the tiles of nbas, with tau scaled by the ratio.)

So the error at a given tau follows from these numbers alone, not from how a kernel
cuts its work.  Counts are equal to the model's; FP64 K agrees within the rounding of
sums of that length, |K - K_model| <= 2 (2 n + M o + 16) u S, S = sum_J (|L^J||C|)(|L^J||C|)^T,
u = 2^-53 (thresholds lie between values far apart, not at one)."""
import numpy as np
import pytest
import torch

from _dense import lfull
from openmolcas_amd.fock import JKContext
from openmolcas_amd.synthetic import pack
from test_gpu_screening import localized_system

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def tri(t):
    return t * (t + 1) // 2


def model(Lf, Cs, n, tau, thr_x, tile, split, ncu, fp32=False):
    M = Lf.shape[0]
    n_pad = (n + 127) // 128 * 128
    tm = tile if tile else (128 if n_pad >= 512 else 64)
    opad = [(c.shape[1] + 3) // 4 * 4 for c in Cs]
    t, slots = (n + tm - 1) // tm, 2 * ncu

    def slices(op, tiles):
        rounds = 1
        while rounds < 8 and M * sum(opad) * tiles >= 2048 * slots * 2 * rounds:
            rounds *= 2
        return max(1, min((split if split else slots * rounds) * op // (tiles * sum(opad)), M))

    ref = [slices(op, tri(n_pad // tm)) for op in opad]
    if fp32:
        own = [slices(op, tri(t)) for op in opad]
        tau *= min(r / o for r, o in zip(ref, own))
        ref = own
    cmax = max(np.linalg.norm(c) for c in Cs)
    dead = np.zeros((M, (n + 63) // 64), dtype=bool)
    if thr_x > 0.0:
        for st in range(dead.shape[1]):
            dead[:, st] = np.linalg.norm(Lf[:, :, 64 * st:64 * st + 64], axis=(1, 2)) * cmax < thr_x
    items = skipped = 0
    K = []
    for c, ns in zip(Cs, ref):
        X = Lf @ c
        for J, st in zip(*np.nonzero(dead)):
            X[J, 64 * st:64 * st + 64] = 0.0
        per = (M + ns - 1) // ns
        items += ns * tri(t)
        norm = np.stack([np.linalg.norm(X[:, tm * a:tm * a + tm], axis=(1, 2)) for a in range(t)])
        k = np.zeros((n, n))
        for j in range(0, M, per):
            for a in range(t):
                for b in range(a + 1):
                    if norm[a, j:j + per] @ norm[b, j:j + per] < tau:
                        skipped += 1
                        continue
                    xa, xb = (X[j:j + per, tm * i:tm * i + tm].transpose(1, 0, 2) for i in (a, b))
                    k[tm * a:tm * a + tm, tm * b:tm * b + tm] += xa.reshape(len(xa), -1) @ xb.reshape(len(xb), -1).T
        K.append(pack(np.tril(k) + np.tril(k, -1).T))
    return K, {"k_items": items, "k_skipped": skipped, "x_tiles": dead.size if thr_x else 0,
               "x_skipped": int(dead.sum())}


@pytest.mark.parametrize("n,M,occ,tau,thr_x,tile,split", [
    (512, 600, [24], 1e-8, 1e-8, 0, 0), (640, 300, [30, 9], 1e-6, 0.0, 0, 0), (130, 700, [20], 1e-8, 0.0, 0, 0),
    (384, 200, [48], 1e-8, 1e-7, 0, 0), (400, 150, [17], 1e-7, 1e-7, 64, 0), (300, 90, [10], 1e-7, 1e-7, 128, 40),
    (520, 80, [26], 1e-6, 1e-6, 0, 100), (700, 40, [33], 1e-5, 0.0, 0, 1), (192, 260, [29], 1e-7, 1e-7, 0, 0)])
def test_screened_work_follows_the_rule(gpu, n, M, occ, tau, thr_x, tile, split):
    L, C = localized_system(n, M, sum(occ), width=10.0, seed=n + M)
    Cs = [np.ascontiguousarray(c) for c in np.split(C, np.cumsum(occ)[:-1], axis=1)]
    Lf = lfull(L, n)
    ncu = torch.cuda.get_device_properties(gpu).multi_processor_count
    want, stats = model(Lf, Cs, n, tau, thr_x, tile, split, ncu)
    assert stats["k_skipped"] > 0
    jk = JKContext(n, M, device=gpu)
    jk.upload_packed(L)
    jk.set_tuning(tile, split, 0)
    Ct = [torch.from_numpy(c) for c in Cs]
    K = jk.exchange_screened(Ct, tau, thr_x).cpu().numpy()
    assert jk.screening_stats() == stats
    for k, w, c in zip(K, want, Cs):
        A = (np.abs(Lf) @ np.abs(c)).transpose(1, 0, 2).reshape(n, -1)
        bound = 2.0 * (2 * n + M * c.shape[1] + 16) * U * (A @ A.T)
        assert np.all(np.abs(k - w) <= pack(bound))
    jk.exchange_screened(Ct, tau, 0.0, "fp32")
    assert jk.screening_stats() == model(Lf, Cs, n, tau, 0.0, tile, split, ncu, True)[1]
    jk.close()
