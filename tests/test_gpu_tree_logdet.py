"""The stable log det as a tree of merges against the oracle's log det, at numbers of groups that leave an odd
row out at some level (4, 5, 6, 7, 8, 11, 16 groups; below 4 the sequence of eliminations), orders with one
panel, several, merges of up to 512 and of more candidate rows (256, 288, 384: the panel kernels change
there), the first order of the sequence (416), one and several fields, both hoppings.

Rings with hopping 0.3 per slice and fields N(0, 0.2): the whole product has a condition number below
e^(0.6 nt) <= e^20, within the oracle's reach; rounding of n nt 2^-53 times that of 1 + A (below 1e3): 1e-10."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_mod2pi

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import action as act  # noqa: E402


def _ring(n):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3
    return k


@pytest.mark.parametrize("n,groups,g,batch", [(32, 3, 2, 1), (32, 4, 2, 3), (32, 5, 2, 1), (64, 6, 2, 2), (64, 7, 3, 1),
                                              (96, 8, 2, 1), (128, 11, 2, 2), (32, 16, 2, 1), (256, 4, 2, 1),
                                              (288, 5, 2, 1), (384, 4, 1, 1), (416, 4, 1, 1)])
@pytest.mark.parametrize("hopping", [act.HFAHopping.EXP, act.HFAHopping.DIA])
def test_matches_oracle(n, groups, g, batch, hopping):
    print(f"stable log det n={n} groups={groups} of {g} batch={batch} {hopping.name}", flush=True)
    nt = groups * g
    phis = np.random.RandomState(n + groups).normal(0, 0.2, (batch, n * nt)) + 0j
    a = act.HubbardFermiAction(_ring(n), 0.05, -1, hopping, precision="mixed", logdet="stable", logdet_group=g)
    r = ref.HubbardFermiAction(_ring(n), 0.05, -1, ref.EXP if hopping == act.HFAHopping.EXP else ref.DIA)
    got = a.eval_batch(torch.as_tensor(phis, device="cuda"))
    for x, phi in zip(got, phis):
        assert rel_mod2pi(x, r.eval(phi)) < 1e-10
