"""Calls whose fast path wants more scratch memory than the GPU has left: the
inverse and the full-rank greedy search then run without their split planes
(csrc/chol.hip, csrc/ldlq.hip), an inverse batch in as many pieces as its room
has planes for.

Bars: a batch in pieces equals each matrix by itself; without planes, those of
the general path (test_gpu_split.py, test_gpu_greedy_split.py)."""

from __future__ import annotations

import pytest
import torch

from int_crush_converter_amd import _native as nat
from oracle import torch_ref as ref
from tests.conftest import lognormal_hessian
from tests.test_gpu_greedy_split import _problem, _search64

pytestmark = pytest.mark.gpu


@pytest.fixture
def full_gpu(monkeypatch):
    """A GPU with room for the least workspace only: `least` to be set by the test."""
    room = {"least": 0, "refused": 0}
    real = nat.workspace

    def workspace(nbytes, dev):
        if nbytes > room["least"]:
            room["refused"] += 1
            raise torch.OutOfMemoryError("no room")
        return real(nbytes, dev)

    monkeypatch.setattr(nat, "workspace", workspace)
    return room


def test_inverse_without_room_for_planes(gpu_dev, full_gpu):
    from int_crush_converter_amd.hessian import inverse_batch
    n = 2049
    H = lognormal_hessian(n, n + 512, n)
    full_gpu["least"] = nat.lib().ic_hessian_inverse_min_workspace_bytes(1, n)
    got = inverse_batch(H.to(gpu_dev), 0.01, "hinv").cpu()
    assert full_gpu["refused"] == 1
    truth = torch.cholesky_inverse(torch.linalg.cholesky(ref.damp(H, 0.01).to(gpu_dev).double())).cpu()
    want = ref.prepare_hinv(H, 0.01)
    s = truth.diagonal().rsqrt()
    e_got, e_ref = (((x.double() - truth) * s[:, None] * s).norm().item() for x in (got, want))
    assert torch.equal(got, got.T) and e_got <= e_ref, (e_got, e_ref)


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("at_once", [0, 1, 2, 3])
def test_inverse_batch_in_pieces(gpu_dev, method, at_once):
    L = nat.lib()
    n, batch = 2178, 3
    Hs = torch.stack([lognormal_hessian(n, n + 512, s) for s in range(batch)]).to(gpu_dev)

    def run(H, nbytes):
        H = H.clone()
        info = torch.zeros(2 * len(H), dtype=torch.int32, device=gpu_dev)
        ws = nat.workspace(nbytes, gpu_dev)
        nat.check(L.ic_hessian_inverse_sized(H, len(H), n, 0.01, method, info, ws, nbytes, nat.stream()), "inverse")
        assert not info.any()
        return H

    least = L.ic_hessian_inverse_min_workspace_bytes
    planes = L.ic_hessian_inverse_workspace_bytes(1, n) - least(1, n)
    room = (planes - 256) * at_once + 256
    got = run(Hs, least(batch, n) + room)
    for b in range(batch):
        assert torch.equal(got[b], run(Hs[b:b + 1], least(1, n) + (planes if at_once else 0))[0]), b


def test_workspace_below_the_least_is_refused(gpu_dev):
    # an argument check: nothing is launched
    L = nat.lib()
    t = torch.zeros(256, device=gpu_dev)
    assert L.ic_hessian_inverse_sized(t, 1, 8, 0.01, 0, t, t, L.ic_hessian_inverse_min_workspace_bytes(1, 8) - 1,
                                      nat.stream()) == -1
    assert L.ic_greedy_sized(t, t, t, 0, t, 8, 8, 1, 4, t, L.ic_greedy_min_workspace_bytes(8, 8) - 1,
                             nat.stream()) == -1


def test_greedy_without_room_for_planes(gpu_dev, full_gpu):
    from int_crush_converter_amd.greedy import greedy_local_search
    rows, cols = 2050, 2048
    W, Q, s, H = _problem(rows, cols, gpu_dev, 3)
    full_gpu["least"] = nat.lib().ic_greedy_min_workspace_bytes(rows, cols)
    got = greedy_local_search(W, Q, s, H, 1, -8, 7)
    assert full_gpu["refused"] == 1
    assert (got != _search64(W, Q, s, H, 1)).any(1).sum().item() <= 0.01 * rows
