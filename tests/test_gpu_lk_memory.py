"""The screened LK drop-in takes fewer batches of vectors together where there is little
device memory, with the same bits: on a nearly full device (its group of 14 batches
needs about 600 MB), and under a small X budget."""
import numpy as np
import pytest
import torch

from _lk_molecule import local_orbitals, molecule
from test_gpu_lk import context, fold

pytestmark = pytest.mark.gpu


def build(jk, mol, Cs, plt, flt0):
    flt = [f.copy() for f in flt0]
    klt = [np.zeros_like(f) for f in flt0]
    nocc = [C.shape[1] for C in Cs]
    jk.cho_lk_scf(len(Cs), flt, klt, [0] * len(Cs), nocc, Cs, plt, 0.5, nscreen=10, dmpk=0.3, dfmat=1.0,
                  nbassh=mol["nbassh"])
    return np.stack(flt + klt), list(jk.lk_stats())


def test_lk_with_little_memory(gpu):
    mol = molecule(seed=3, natom=100, nvec=350, nred=1)
    n = mol["n"]
    Cs = [local_orbitals(mol["pos"], o, 60 + d) for d, o in enumerate((200, 190))]
    plt = fold(sum(C @ C.T for C in Cs))
    flt0 = np.random.default_rng(3).standard_normal((2, n * (n + 1) // 2))
    jk = context(mol, gpu)
    want, stats = build(jk, mol, Cs, plt, flt0)
    jk.close()
    small, full = context(mol, gpu), context(mol, gpu)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    small.set_x_budget(100 << 20)
    got, s = build(small, mol, Cs, plt, flt0)
    assert before - torch.cuda.mem_get_info()[0] <= 300 << 20
    assert np.array_equal(got, want) and s == stats
    small.close()
    keep, left = [], 400 << 20
    for _ in range(40):
        free = torch.cuda.mem_get_info()[0]
        if free > left + (32 << 20):
            keep.append(torch.empty(min(free - left, 16 << 30), dtype=torch.uint8, device=gpu))
    try:
        for _ in range(2):
            got, s = build(full, mol, Cs, plt, flt0)
            assert np.array_equal(got, want) and s == stats
    finally:
        del keep
        torch.cuda.empty_cache()
        full.close()
