"""The log det's strip chains of few fields in several groups, multiplied together pairwise (n > 128): numbers of
slices without divisors, orders that are and are not multiples of 32, one and several fields, the reference's
form (particles forward, holes backward with EXP hopping; both backward with DIA), the grouped form with all slices
as its group, the stable form with a single group.

A ring of n sites with hopping 1.2 / Nt per slice (cond of all slices at most e^4.8) and fields N(0, 0.2):
rounding of Nt n 2^-53 < 5e-12 times the condition of 1 + A^-1 (below 1e2), relative to |S| of order n: 1e-10."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_mod2pi

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

GEMM64_CC, GEMM64_CC4 = 3, 33  # launch kinds: products of group products (one chain over all slices has none)


def _ring(n, hopping):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = hopping
    return k


def _launches(hfm, op, phis, nt):
    """Launches per kind of one log det (op 2: FP64, 3: grouped, 5: stable) with all slices as its group."""
    out = np.zeros(4 * 38)
    _lib.check(_lib.load().isle_profile_kernels(hfm.handle, _lib.ptr(phis), op, nt, phis.shape[0], nt, 2, 0, 1,
                                                _lib.dptr(out), 38))
    return out[::4]


@pytest.mark.parametrize("n,nt,batch", [(130, 17, 1), (160, 31, 5), (180, 31, 2), (288, 97, 1), (303, 31, 1), (512, 13, 1)])
@pytest.mark.parametrize("hopping", [act.HFAHopping.EXP, act.HFAHopping.DIA])
def test_actions_match_oracle(n, nt, batch, hopping):
    print(f"log det groups n={n} nt={nt} batch={batch} {hopping.name}", flush=True)
    kt = _ring(n, 1.2 / nt)
    phis = np.random.RandomState(n + nt).normal(0, 0.2, (batch, n * nt)) + 0j
    dev = torch.as_tensor(phis, device="cuda")
    want = ref.HubbardFermiAction(kt, 0.01, -1, ref.EXP if hopping == act.HFAHopping.EXP else ref.DIA).eval(phis[-1])
    forms = [(2, GEMM64_CC4, {}), (3, GEMM64_CC, {"precision": "mixed", "group": nt})]
    if n % 32 == 0:
        forms.append((5, GEMM64_CC, {"precision": "stable", "group": nt}))
    for op, kind, kw in forms:
        a = act.HubbardFermiAction(kt, 0.01, -1, hopping, **kw)
        assert rel_mod2pi(a.eval_batch(dev)[-1], want) < 1e-10, kw
        assert a._group(nt) == nt or not kw
        assert _launches(a.hfm, op, dev, nt)[kind] > 0, kw
