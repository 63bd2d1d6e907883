"""The strip kernels (isle_amd/csrc/chain.hpp) at the edges of their tiles: orders around multiples of
16 (tiles), of 8 (FP64 units of k), the change from registers to streaming (128), the shapes chosen
for few and many chains (288, 384), their largest order (512) and the first of the other path (513);
one slice per group, one group, several groups.

A ring of n sites with hopping 0.3 per slice (cond of a slice e^1.2, of all slices at most e^5) and
fields N(0, 0.2): the products are well conditioned, so FP64 results differ from the oracle's by
rounding only: about Nt n 2^-53 = 5e-13 times the condition of 1 + A^-1 (below 1e2): 1e-10; the mixed
force by its FP32 right chains, 1e-5."""
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
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3 if n > 1 else 0.0
    return k


@pytest.mark.parametrize("n,nt,batch,group", [
    (1, 4, 1, 4), (2, 3, 1, 3), (7, 4, 2, 2), (8, 4, 1, 4), (9, 5, 1, 5), (15, 4, 1, 1), (16, 4, 2, 4), (17, 6, 1, 3),
    (24, 4, 1, 4), (25, 4, 1, 2), (33, 4, 3, 4), (72, 4, 1, 4), (127, 4, 1, 2), (128, 4, 2, 4), (129, 4, 1, 4),
    (161, 4, 1, 2), (208, 3, 1, 3), (257, 4, 1, 4), (288, 4, 2, 2), (288, 4, 16, 2), (303, 3, 1, 3), (384, 4, 1, 2),
    (512, 2, 1, 2), (513, 2, 1, 2)])
@pytest.mark.parametrize("hopping", [act.HFAHopping.EXP, act.HFAHopping.DIA])
def test_strip_chains_match_oracle(n, nt, batch, group, hopping):
    print(f"strip chains n={n} nt={nt} batch={batch} group={group} {hopping.name}", flush=True)
    kt = _ring(n)
    mu = 0.05
    phis = np.random.RandomState(n).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    want = ref.HubbardFermiAction(kt, mu, -1, ref.EXP if hopping == act.HFAHopping.EXP else ref.DIA)
    f_ref, s_ref = want.force(phis[-1]), want.eval(phis[-1])
    plain = act.HubbardFermiAction(kt, mu, -1, hopping)
    assert rel_l2(plain.force_batch(dev)[-1].cpu().numpy(), f_ref) < 1e-10
    assert rel_mod2pi(plain.eval_batch(dev)[-1], s_ref) < 1e-10
    mixed = act.HubbardFermiAction(kt, mu, -1, hopping, precision="mixed", group=group)
    assert rel_l2(mixed.force_batch(dev)[-1].cpu().numpy(), f_ref) < 1e-5
    assert rel_mod2pi(mixed.eval_batch(dev)[-1], s_ref) < 1e-10
