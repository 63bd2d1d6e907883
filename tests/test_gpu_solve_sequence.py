"""solveM called in turn with other fields, species, time extents and numbers of right-hand sides on one
matrix (its buffers and launch descriptors are kept between calls), at orders around the tiles of the
prefix chain (16), its largest order (512) and the first of the other path (513), with few and with many
(64: blocked solves where 32 divides n) right-hand sides.

A ring of n sites with hopping 0.3 per slice and fields N(0, 0.2): products of at most 5 slices have
condition numbers below e^6; the residual of a solve by their LUs stays below n cond 2^-53 = 3e-11,
times 10 for the back substitution through the slices: 1e-9."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")


def _ring(n):
    k = np.zeros((n, n))
    for i in range(n):
        k[i, (i + 1) % n] = k[(i + 1) % n, i] = 0.3 if n > 1 else 0.0
    return k


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 64, 97, 98, 128, 129, 160, 288, 512, 513])
@pytest.mark.parametrize("hopping", ["exp", "dia"])
def test_solves_in_turn(n, hopping):
    print(f"solveM sequence n={n} {hopping}", flush=True)
    cls = isle.HubbardFermiMatrixExp if hopping == "exp" else isle.HubbardFermiMatrixDia
    m = cls(_ring(n), 0.05, -1)
    rs = np.random.RandomState(n)
    turns = [(1, 0, 1), (5, 0, 3), (5, 1, 3), (5, 0, 70), (5, 1, 70), (3, 1, 3), (3, 0, 17), (5, 0, 3)]
    for nt, species, nrhs in turns:
        phi = torch.as_tensor(rs.normal(0, 0.2, n * nt) + 0j, device="cuda")
        for reuse in (False, True):
            b = torch.as_tensor(rs.normal(size=(nrhs, n * nt)) + 1j * rs.normal(size=(nrhs, n * nt)), device="cuda")
            x = isle.solveM(m, phi, species, b, reuse_factor=reuse)
            r = b - isle.core.applyM(m, phi, species, x)
            assert (r.abs().max() / b.abs().max()).item() < 1e-9, (nt, species, nrhs, reuse)
