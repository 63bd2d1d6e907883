"""The stable forms of few fields, whose slices are launches of their own where those are split over more of the
GPU than the strips of so few chains (one field in two groups from n = 224 on, and twelve chains at n = 416), and on
strips otherwise, as the FP32 right chains always: which of them runs, and its results against the oracle.

A ring of n sites with hopping 1.2 / Nt per slice (cond of all slices at most e^4.8) and fields N(0, 0.2):
rounding of Nt n 2^-53 < 4e-12 times the condition of 1 + A^-1 (below 1e2): 1e-9 for the force, and 1e-10 relative to
the action of order n; 1e-5 with FP32 right chains."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_l2, rel_mod2pi

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

GEMM64_RC_ROW, SUFFIX64 = 1, 35  # launch kinds: one slice of every chain; whole chains on strips


def _ring(n, hopping):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = hopping
    return k


def _launches(hfm, op, phis, nt, group):
    out = np.zeros(4 * 38)
    _lib.check(_lib.load().isle_profile_kernels(hfm.handle, _lib.ptr(phis), op, nt, phis.shape[0], group, 2, 0, 1,
                                                _lib.dptr(out), 38))
    return out[::4]


@pytest.mark.parametrize("n,nt,group,batch,strips", [(128, 16, 8, 1, True), (192, 16, 8, 1, True), (224, 16, 8, 1, False),
                                                     (288, 16, 8, 1, False), (288, 16, 8, 4, True), (416, 16, 8, 1, False),
                                                     (416, 12, 2, 1, False), (512, 12, 3, 1, True)])
def test_stable_forms_match_oracle(n, nt, group, batch, strips):
    print(f"stable slices n={n} nt={nt} group={group} batch={batch}", flush=True)
    kt = _ring(n, 1.2 / nt)
    phis = np.random.RandomState(n + nt).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    want = ref.HubbardFermiAction(kt, 0.01, -1, ref.EXP)
    f_want = want.force(phis[-1])
    a = act.HubbardFermiAction(kt, 0.01, -1, act.HFAHopping.EXP, precision="stable", group=group)
    b = act.HubbardFermiAction(kt, 0.01, -1, act.HFAHopping.EXP, precision="stable", group=group, right_chains="fp32")
    assert a._group(nt) == b._group(nt) == group
    assert rel_l2(a.force_batch(dev)[-1].cpu().numpy(), f_want) < 1e-9
    assert rel_mod2pi(a.eval_batch(dev)[-1], want.eval(phis[-1])) < 1e-10
    assert rel_l2(b.force_batch(dev)[-1].cpu().numpy(), f_want) < 1e-5
    for op in (4, 5):
        kinds = _launches(a.hfm, op, dev, nt, group)
        assert (kinds[SUFFIX64] > 0) == strips and (kinds[GEMM64_RC_ROW] > 0) == (not strips), (op, kinds)
