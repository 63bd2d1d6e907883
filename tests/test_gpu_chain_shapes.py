"""The strip kernels with two column tiles per strip ({3, 2} of CHAIN_SHAPES), which 17 and 18 tiles (n = 257 to 288)
take from 16 and 15 chains on: with an odd number of tiles half of the last strip lies beyond the matrix, and the
right chains read its rows from the padding behind the suffix products.  One and two groups, first, middle and last
item against the oracle; 15 chains (one species, the hole shortcut) next to 14, which take one column tile.

A ring of n sites with hopping 0.3 per slice (cond of all slices at most e^5) and fields N(0, 0.2): rounding of
Nt n 2^-53 < 2e-13 times the condition of 1 + A^-1 (below 1e2): 1e-10; the mixed force by its FP32 right
chains, 1e-5."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_l2, rel_mod2pi

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import action as act  # noqa: E402


def _ring(n):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3
    return k


@pytest.mark.parametrize("n,nt,batch,group,shortcut", [(257, 4, 8, 4, False), (257, 4, 5, 2, False), (264, 2, 12, 2, False),
                                                       (272, 4, 20, 4, False), (272, 4, 8, 2, False), (273, 4, 8, 4, False),
                                                       (288, 4, 8, 4, False), (288, 3, 70, 3, False),
                                                       (288, 4, 15, 4, True), (288, 4, 14, 4, True)])
def test_two_column_tiles_match_oracle(n, nt, batch, group, shortcut):
    print(f"strips of two column tiles n={n} nt={nt} batch={batch} group={group} shortcut={shortcut}", flush=True)
    kt, sk, mu = _ring(n), 1 if shortcut else -1, 0.0 if shortcut else 0.05
    phis = np.random.RandomState(n + batch).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    want = ref.HubbardFermiAction(kt, mu, sk, ref.EXP)
    plain = act.HubbardFermiAction(kt, mu, sk, act.HFAHopping.EXP, allowShortcut=shortcut)
    mixed = act.HubbardFermiAction(kt, mu, sk, act.HFAHopping.EXP, allowShortcut=shortcut, precision="mixed", group=group)
    assert plain.shortcut == shortcut
    f, s = plain.force_batch(dev).cpu().numpy(), plain.eval_batch(dev)
    fm, sm = mixed.force_batch(dev).cpu().numpy(), mixed.eval_batch(dev)
    for b in sorted({0, batch // 2, batch - 1}):
        f_want, s_want = want.force(phis[b]), want.eval(phis[b])
        assert rel_l2(f[b], f_want) < 1e-10, b
        assert rel_mod2pi(s[b], s_want) < 1e-10, b
        assert rel_l2(fm[b], f_want) < 1e-5, b
        assert rel_mod2pi(sm[b], s_want) < 1e-10, b
