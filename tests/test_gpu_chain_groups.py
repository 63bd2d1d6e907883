"""The strip chains of few fields in several groups, where one chain over all slices would leave the GPU idle
(n > 128): time extents without divisors (17, 31, 97: groups of two lengths), orders that are no multiple of 32
(130, 180, 303: the inverse by lu_solve_kernel) and multiples (160, 288), few and more than four (field,
species) items, the mixed form whose group is all slices, the stable form with a single group.

A ring of n sites with hopping 1.2 / Nt per slice (cond of all slices at most e^4.8) and fields N(0, 0.2):
the FP64 results differ from the oracle's by rounding, about Nt n 2^-53 < 5e-12 times the condition of
1 + A^-1 (below 1e2): 1e-9; the mixed force by its FP32 right chains, 1e-5."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

GEMM64_CC = 3  # launch kind: products of group products (one chain over all slices has none)
CASES = [(130, 17, 1), (160, 31, 5), (180, 31, 2), (288, 97, 1), (303, 31, 1)]


def _ring(n, hopping):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = hopping
    return k


def _launches(hfm, op, phis, nt, group):
    """Launches per kind of one force (op 0: FP64, 1: mixed, 4: stable)."""
    out = np.zeros(4 * 38)
    _lib.check(_lib.load().isle_profile_kernels(hfm.handle, _lib.ptr(phis), op, nt, phis.shape[0], group, 2, 0, 1,
                                                _lib.dptr(out), 38))
    return out[::4]


@pytest.mark.parametrize("n,nt,batch", CASES)
@pytest.mark.parametrize("hopping", [act.HFAHopping.EXP, act.HFAHopping.DIA])
def test_forces_match_oracle(n, nt, batch, hopping):
    print(f"chain groups n={n} nt={nt} batch={batch} {hopping.name}", flush=True)
    kt = _ring(n, 1.2 / nt)
    phis = np.random.RandomState(n + nt).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    want = ref.HubbardFermiAction(kt, 0.01, -1, ref.EXP if hopping == act.HFAHopping.EXP else ref.DIA).force(phis[-1])
    forms = [(0, {}, 1e-9), (1, {"precision": "mixed", "group": nt}, 1e-5)]
    if n % 32 == 0:
        forms.append((4, {"precision": "stable", "group": nt}, 1e-9))
    for op, kw, tol in forms:
        a = act.HubbardFermiAction(kt, 0.01, -1, hopping, **kw)
        assert rel_l2(a.force_batch(dev)[-1].cpu().numpy(), want) < tol, kw
        assert a._group(nt) == nt or not kw
        assert _launches(a.hfm, op, dev, nt, nt)[GEMM64_CC] > 0, kw


def test_batches_of_several_time_extents():
    """force_batch_multi's batches share their launches and take their groups together: the same forces as
    each batch alone, to the rounding of another order of products."""
    n, nts = 180, (13, 31, 32)
    kt = _ring(n, 1.2 / 32)
    for kw, tol in (({}, 1e-9), ({"precision": "mixed"}, 1e-5)):
        a = act.HubbardFermiAction(kt, 0.01, -1, act.HFAHopping.EXP, **kw)
        phis = [torch.as_tensor(np.random.RandomState(nt).normal(0, 0.2, (2, n * nt)) + 0j, device="cuda") for nt in nts]
        outs = a.force_batch_multi(phis, [torch.empty_like(p) for p in phis])
        for p, o in zip(phis, outs):
            assert rel_l2(o.cpu().numpy(), a.force_batch(p).cpu().numpy()) < tol, kw
