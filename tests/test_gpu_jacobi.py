"""GPU parity of the blocked Jacobi eigensolver (csrc/lowrank.hip) at the
edges of its blocks of 32 and pairs of 64: one pair, a partial last block,
orders just below and above a multiple of 64, several rounds; repeated and
zero eigenvalues.  Against eigh in 64 bits: the solver works in 64 bits on a
T formed in fp32, so eigenvalues are good to fp32's rounding of the largest
(2^-24, with p terms in each sum: 1e-6 covers p <= 200)."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_greedy import _eigs, _planted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2, 34, 62, 64, 66, 126, 130, 192])
def test_jacobi_block_edges(gpu_dev, p):
    evals = torch.logspace(2, -3, p)
    evals[p // 2:] = evals[p // 2]        # a repeated eigenvalue
    if p > 40:
        evals[-8:] = 0.0
    H = _planted(p, evals, p)
    ev, U, sweeps = _eigs(H, p, 0, gpu_dev)
    want = torch.linalg.eigvalsh(H.double()).flip(0)
    lmax = want[0].item()
    assert (ev.double() - want).abs().max().item() <= 1e-6 * lmax
    U = U.double()
    assert (H.double() @ U - U * ev.double()).abs().max().item() <= 4e-6 * lmax
    assert (U.T @ U - torch.eye(p, dtype=torch.float64)).abs().max().item() < 1e-5
    assert 1 <= sweeps < 40   # the solver's limit (converged before it; single rotations take 9-15 sweeps here too)
