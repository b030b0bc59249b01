"""Host arrays of the drop-ins against the same call on device tensors: sizes on
both sides of the 3 MiB line (one staged copy each way below it, one copy per
array above), odd pair counts, an empty orbital set, and calls from several
threads, each on a context of its own.

Both sides run the same J and K kernels on the same numbers.  F = F + J - x K is
then at most three roundings away from the host's own sum, plus the different
grouping of the J pass when it shares the vectors with the half-transform:
2 (M + 2 n + 8) u (|F| + |J| + |x| |K|) bounds it, with u = 2^-53 and the sums'
absolute values from the same vectors' absolute values."""
import threading

import numpy as np
import pytest
import torch

from openmolcas_amd.fock import JKContext
from openmolcas_amd.synthetic import chol_vectors_np, orbitals_np

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def one(gpu, n, M, occ, seed, calls=1):
    g = np.random.default_rng(seed)
    npair, nden = n * (n + 1) // 2, len(occ)
    L = chol_vectors_np(n, M, seed=seed)
    cs = [np.ascontiguousarray(orbitals_np(n, max(o, 1), seed=seed + 1 + d)[:, :o]) for d, o in enumerate(occ)]
    d = g.standard_normal(npair)
    f0 = g.standard_normal((nden, npair))
    out, dev = JKContext(n, M, device=gpu), JKContext(n, M, device=gpu)
    absl = JKContext(n, M, device=gpu)
    try:
        out.upload_packed(L), dev.upload_packed(L), absl.upload_packed(np.abs(L))
        got = []
        for _ in range(calls):
            flt = f0.copy()
            assert out.cho_fscf(nden, flt, [0] * nden, list(occ), cs, d, 0.5) == 0
            got.append(flt)
        dd = torch.from_numpy(d).to(gpu)
        cd = [torch.from_numpy(c).to(gpu) for c in cs]
        j, ja = dev.coulomb(dd).cpu().numpy().reshape(-1), absl.coulomb(dd.abs()).cpu().numpy().reshape(-1)
        for k, o in enumerate(occ):
            kk = dev.exchange([cd[k]]).cpu().numpy()[0] if o else np.zeros(npair)
            ka = absl.exchange([cd[k].abs()]).cpu().numpy()[0] if o else np.zeros(npair)
            want = f0[k] + j - 0.5 * kk
            tol = 2 * (M + 2 * n + 8) * U * (np.abs(f0[k]) + ja + 0.5 * ka)
            for f in got:
                assert np.all(np.abs(f[k] - want) <= tol), (n, M, occ, k, float(np.max(np.abs(f[k] - want) / tol)))
    finally:
        for ctx in (out, dev, absl):
            ctx.close()


@pytest.mark.parametrize("n,M,occ", [
    (1, 1, (1,)), (2, 3, (1, 1)), (5, 7, (2, 0)), (24, 40, (5,)), (57, 33, (9, 8)), (90, 20, (0, 11)),
    (420, 6, (40, 39)), (575, 5, (57,)), (577, 5, (100,)), (480, 4, (47, 50)), (530, 4, (60, 2)),
])
def test_fscf_host_arrays(gpu, n, M, occ):
    one(gpu, n, M, occ, seed=n)


def test_fscf_from_threads(gpu):
    err = []

    def work(k):
        try:
            one(gpu, 40 + 31 * k, 20 + k, (7, 6) if k % 2 else (9,), seed=100 + k, calls=20)
        except BaseException as e:  # noqa: BLE001 - handed to the test's own thread
            err.append(e)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not err, err
