"""The two inverses of the grouped force's top level, lu_solve_kernel and blocked triangular solves, on both sides of
the line between them: n not a multiple of 32 (always the kernel), few and many matrices of order 64, 224 and 288,
one of order 352 (always blocked); the launch counts say which ran.

Rings with hopping 0.3 per slice and fields N(0, 0.2): cond of all slices below e^5; rounding of n nt 2^-53 times the
condition of 1 + A^-1 (below 1e2): 1e-10."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

SOLVE, TRSM = 9, 24  # launch kinds


@pytest.mark.parametrize("n,batch,blocked", [(64, 8, False), (65, 600, False), (224, 15, False), (224, 16, True),
                                             (288, 7, False), (288, 8, True), (300, 16, False), (352, 1, True)])
def test_inverse_on_both_sides(n, batch, blocked):
    print(f"top level inverse n={n} batch={batch}", flush=True)
    nt = 2
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3
    phis = np.random.RandomState(n + batch).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    a = act.HubbardFermiAction(k, 0.05, -1, act.HFAHopping.EXP)
    got = a.force_batch(dev).cpu().numpy()
    r = ref.HubbardFermiAction(k, 0.05, -1, ref.EXP)
    for b in (0, batch - 1):
        assert rel_l2(got[b], r.force(phis[b])) < 1e-10, b
    out = np.zeros(4 * 38)
    _lib.check(_lib.load().isle_profile_kernels(a.hfm.handle, _lib.ptr(dev), 0, nt, batch, nt, 2, 0, 1, _lib.dptr(out), 38))
    assert (out[4 * SOLVE] > 0) == (not blocked) and (out[4 * TRSM] > 0) == blocked
