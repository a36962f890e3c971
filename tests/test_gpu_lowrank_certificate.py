"""The refusal certificate of ic_lowrank_eigs (csrc/lowrank.hip): tried after
one and after two steps, each on its own."""

from __future__ import annotations

import pytest
import torch

from int_crush_converter_amd import _native as nat
from tests.test_gpu_greedy import _planted

pytestmark = pytest.mark.gpu


def _refused(H, p, iters, dev):
    L, n = nat.lib(), H.shape[0]
    Hg = H.to(dev).contiguous()
    ev, U = torch.empty(p, device=dev), torch.empty(n, p, device=dev)
    ws = nat.workspace(L.ic_lowrank_workspace_bytes(n, p), dev)
    rc = L.ic_lowrank_eigs(Hg, n, p, iters, 7, 0.01, ev, U, None, ws, nat.stream())
    assert rc in (0, 1)
    return rc == 1


def test_second_test_refuses_after_the_first_did_not(gpu_dev):
    # 249 eigenvalues of 0.7 .. 1 and 351 of 0.08 against p = 244: the smallest Ritz value is 0.63 - 0.78 of the
    # bound after one step and 3 - 4.7 times it after two (computed in 64 bits for six starts)
    H = _planted(600, torch.cat([torch.linspace(1.0, 0.7, 249), torch.full((351,), 0.08)]), 3)
    assert not _refused(H, 244, 1, gpu_dev)   # one step, one test
    assert _refused(H, 244, 8, gpu_dev)


def test_tests_that_fail_refuse_nothing(gpu_dev):
    H = _planted(600, torch.cat([torch.linspace(1.0, 0.7, 100), torch.full((500,), 1e-3)]), 4)
    assert not _refused(H, 244, 8, gpu_dev)
