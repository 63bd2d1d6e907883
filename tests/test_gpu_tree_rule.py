"""The line between the stable log det's tree of merges and the sequence of eliminations, four matrices of order 288
per group: on it 8 groups take the tree (16 fields: three levels of merges; 17 fields the sequence, six steps and a last
one that leaves no columns to a later launch), 16 groups the sequence (32 fields; 31 the tree); results against the
oracle.

Ring with hopping 1.2 / Nt per slice and fields N(0, 0.2): cond of all slices below e^5; rounding of n nt 2^-53 times
that of 1 + A (below 1e2): 1e-10."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_mod2pi

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

LU_SHAPE_DEFER = 32  # launch kind: one factorisation of every matrix of a level or step


@pytest.mark.parametrize("groups,batch,steps", [(8, 16, 3), (8, 17, 6), (16, 31, 4), (16, 32, 14)])
def test_line_between_tree_and_sequence(groups, batch, steps):
    n, nt = 288, groups
    print(f"stable log det n={n} groups={nt} batch={batch}", flush=True)
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 1.2 / nt
    phis = np.random.RandomState(n + batch).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    a = act.HubbardFermiAction(k, 0.05, -1, act.HFAHopping.EXP, precision="mixed", logdet="stable", logdet_group=1)
    got = a.eval_batch(dev)
    r = ref.HubbardFermiAction(k, 0.05, -1, ref.EXP)
    for b in (0, batch - 1):
        assert rel_mod2pi(got[b], r.eval(phis[b])) < 1e-10, b
    out = np.zeros(4 * 38)
    _lib.check(_lib.load().isle_profile_kernels(a.hfm.handle, _lib.ptr(dev), 5, nt, batch, 1, 2, 0, 1, _lib.dptr(out), 38))
    assert out[4 * LU_SHAPE_DEFER] == steps
