"""The FP32 right-chain product with one launch per slice (launch kind 30) where it runs: the mixed force with the
recompute schedule, and orders above those of the strip kernels (n > 512, multiples of 32).  Every tile of it, pinned,
is the one launched, reproduces the tuned force to 2e-6 (relative L2; the tiles differ only in the order of FP32
sums: 2^-24 times the root of n, 1e-6) and the oracle's to 1e-5.

Tori with fields N(0, U beta / Nt), field 0 from RandomState(1000); the ring of 544 sites has hopping 0.3 per slice
and fields N(0, 0.2)."""
import numpy as np
import pytest
import torch

from oracle import hubbard_ref as ref
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")
from isle_amd import _lib  # noqa: E402
from isle_amd import action as act  # noqa: E402

RCK_KIND, RIGHT32_KIND = 30, 36
RCK_TILES = range(4)


def _ring(n):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3
    return k


@pytest.mark.parametrize("L,nt,batch,recompute", [(12, 128, 8, 8), (8, 64, 12, 8), (4, 32, 6, 4), (0, 4, 2, 0)])
def test_pinned_tiles_run_and_agree(L, nt, batch, recompute):
    kt = isle.honeycomb(L).hopping() * 8.0 / 128 if L else _ring(544)
    n = kt.shape[0]
    print(f"FP32 right-chain launches: Nx={n} Nt={nt} fields={batch} recompute={recompute}", flush=True)
    std = np.sqrt(3.0 * 8.0 / 128) if L else 0.2
    phis = np.random.RandomState(900 + L).normal(0, std, (batch, n * nt)) + 0j
    phis[0] = np.random.RandomState(1000).normal(0, std, n * nt)
    dev = torch.as_tensor(phis, device="cuda")
    a = act.HubbardFermiAction(kt, 0.0, -1, act.HFAHopping.EXP, precision="mixed", group=32, recompute=recompute)
    g = a._group(nt)
    tuned = a.force_batch(dev).cpu().numpy()
    want = ref.HubbardFermiAction(kt, 0.0, -1, ref.EXP).force(phis[0])
    assert rel_l2(tuned[0], want) < 1e-5
    try:
        for tile in RCK_TILES:
            a.hfm.pin_tile(RCK_KIND, tile)
            out = np.zeros(4 * 38)
            _lib.check(_lib.load().isle_profile_kernels(a.hfm.handle, _lib.ptr(dev), 1, nt, batch, g, 2, 0, 1,
                                                        _lib.dptr(out), 38))
            assert out[4 * RCK_KIND] == g and out[4 * RIGHT32_KIND] == 0, tile  # one launch per slice of a group
            got = a.force_batch(dev).cpu().numpy()
            assert max(rel_l2(got[b], tuned[b]) for b in range(batch)) < 2e-6, tile
            assert rel_l2(got[0], want) < 1e-5, tile
    finally:
        a.hfm.pin_tile(RCK_KIND, -1)
