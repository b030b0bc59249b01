"""The screened LK drop-in where its kernels change path: more orbitals than one
64-bit mask word, shells too large for the one-lane-per-pair norms, more batches
than one group, more basis functions than one panel of the half-transform, a
shell with more columns (J, a) than one wave takes.

Against the oracle's screened CHO_LK_SCF: the same counts of listed shells,
half-transformed shell pairs and K blocks, FLT to relative 1e-11 (sums of at
most 1030 x 1700 terms of both signs round to about 1e-13 of the largest)."""
import numpy as np
import pytest

import oracle
from _lk_molecule import local_orbitals, molecule, store
from test_gpu_lk import RTOL, THRCOM, context, fold, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw,nocc,nscreen,dmpk", [
    (dict(natom=15, nvec=60, nred=3), [70], 1, 0.3),
    (dict(natom=15, nvec=60, nred=3), [65, 3], 2, 0.3),
    (dict(natom=6, nvec=40, nred=2, shells_per_atom=(1, 12, 3)), [9], 1, 0.3),
    (dict(natom=4, nvec=1700, nred=2), [5], 10, 0.3),
    (dict(natom=206, nvec=27, nred=2), [3], 10, 0.0),
    (dict(natom=1, nvec=26, nred=1, shells_per_atom=(1,)), [1], 10, 0.3),
    (dict(natom=3, nvec=51, nred=1, shells_per_atom=(40,)), [16], 10, 0.3),
])
def test_lk_shapes_match_oracle(gpu, kw, nocc, nscreen, dmpk):
    mol = molecule(seed=7, **kw)
    n, nden = mol["n"], len(nocc)
    Cs = [local_orbitals(mol["pos"], o, 60 + d) for d, o in enumerate(nocc)]
    plt = fold(sum(C @ C.T for C in Cs))
    flt0 = np.random.default_rng(7).standard_normal((nden, n * (n + 1) // 2))
    want_f, _, want_s = oracle.cho_lk_scf_screened(
        store(mol), flt0, nocc, Cs, plt, 0.5, mol["nbassh"], mol["diag"], THRCOM, nscreen=nscreen,
        dmpk=dmpk, dfmat=1.0, estimate=False, update=True)
    jk = context(mol, gpu)
    flt = [flt0[d].copy() for d in range(nden)]
    jk.cho_lk_scf(nden, flt, None, [0] * nden, nocc, Cs, plt, 0.5, nscreen=nscreen, dmpk=dmpk, dfmat=1.0,
                  nbassh=mol["nbassh"])
    assert list(jk.lk_stats()[:3]) == list(want_s)
    assert rel(np.stack(flt), want_f) < RTOL
    jk.close()
