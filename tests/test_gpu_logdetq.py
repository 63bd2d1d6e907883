"""log det Q by block cyclic reduction (isle_logdetq) against the sum of log det d_i of the block LU from
one end (getQLU), for odd and even numbers of blocks at several levels (3, 5, 11, 13: a pair of neighbours
is kept; 4, 12, 24: all halve at first); orders that carry the right-hand sides through the LU (32 divides n)
and that do not, one below a tile, some above the first panel, one beyond the register panels.

Rings with hopping 0.3 per slice and fields N(0, 0.2): cond Q below e^(2 0.6 nt) would be the worst case,
but phases and 1 + A keep the d_i near 2 + O(1); both recursions differ by rounding of nt n^(1/2) 2^-53
times the blocks' condition (below 1e3): 1e-10 relative."""
import numpy as np
import pytest
import torch

from tests.helpers import mod2pi_diff

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")


def _ring(n):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3 if n > 1 else 0.0
    return k


@pytest.mark.parametrize("n,nt", [(1, 3), (7, 4), (18, 5), (18, 11), (18, 12), (32, 3), (32, 13), (33, 24), (64, 12),
                                  (64, 25), (128, 14), (160, 12), (513, 4)])
@pytest.mark.parametrize("hopping", ["exp", "dia"])
def test_matches_the_block_lu(n, nt, hopping):
    print(f"log det Q n={n} nt={nt} {hopping}", flush=True)
    cls = isle.HubbardFermiMatrixExp if hopping == "exp" else isle.HubbardFermiMatrixDia
    m = cls(_ring(n), 0.05, -1)
    phi = torch.as_tensor(np.random.RandomState(n + nt).normal(0, 0.2, n * nt) + 0j, device="cuda")
    want = isle.logdetQ(isle.getQLU(m, phi))
    for _ in range(2):
        assert mod2pi_diff(isle.logdetQ(m, phi), want) < 1e-10 * max(1.0, abs(want))
