"""GPU parity of the split products (csrc/split.hip) through the Hessian
inverse, the sizes at which its paths begin and end: one row past the last
whole 2048-segment, blocks of 128 with and without a remainder, an odd row
pitch, two and three segments (a merge of unequal ones), a batch.

Bar: the error against the 64-bit inverse is at most that of the reference's
own fp32 path (LAPACK) on the same matrix - the exact split adds none, so an
error above it means wrong elements, which would exceed it by orders."""

from __future__ import annotations

import pytest
import torch

from oracle import torch_ref as ref
from tests.conftest import lognormal_hessian

pytestmark = pytest.mark.gpu


# several equal merges in one launch: 8192 (two pairs of 2048-segments, then one of 4096), 8320 (and a short segment)
LARGE = [8192, 8320]


@pytest.mark.parametrize("n", [2049, 2178, 3001, 3200, 4096, 4300])
def test_split_inverse_error_at_most_lapack(gpu_dev, n):
    from int_crush_converter_amd.hessian import inverse_batch
    H = lognormal_hessian(n, n + 512, n)
    truth = ref.damp(H, 0.01).to(gpu_dev).double()
    truth = torch.cholesky_inverse(torch.linalg.cholesky(truth)).cpu()
    got = inverse_batch(H.to(gpu_dev), 0.01, "hinv").cpu()
    want = ref.prepare_hinv(H, 0.01)
    assert torch.equal(got, got.T)
    # scaled by the diagonal, so that every row counts alike
    s = truth.diagonal().rsqrt()
    e_got, e_ref = (((x.double() - truth) * s[:, None] * s).abs() for x in (got, want))
    assert e_got.norm() <= e_ref.norm(), (e_got.norm().item(), e_ref.norm().item())
    assert e_got.max() <= 4 * e_ref.max(), (e_got.max().item(), e_ref.max().item())


def test_split_inverse_batch_equals_single(gpu_dev):
    from int_crush_converter_amd.hessian import inverse_batch
    Hs = torch.stack([lognormal_hessian(4300, 4500, s) for s in range(2)]).to(gpu_dev)
    for method in ("hinv", "cholesky"):
        got = inverse_batch(Hs, 0.01, method)
        for b in range(2):
            assert torch.equal(got[b], inverse_batch(Hs[b], 0.01, method)), (method, b)


def test_split_inverse_failure_is_reported(gpu_dev):
    # a negative pivot in the second 2048-segment: info is set, the fallback inverse returned
    from int_crush_converter_amd.hessian import inverse_batch
    H = torch.eye(3200)
    H[2100, 2100] = -3.0
    fb = []
    got = inverse_batch(H.to(gpu_dev), 0.0, "hinv", fb).cpu()
    assert fb == ["hessian_inv_fallback"]
    assert torch.allclose(got, torch.linalg.inv(H), atol=1e-6)


def _large(n, seed, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    X = torch.randn(n + 512, n, generator=g, device=dev) * torch.exp(torch.randn(n, generator=g, device=dev))
    return X.T @ X / (n + 512)


@pytest.mark.parametrize("n", LARGE)
def test_split_inverse_of_batched_merges(gpu_dev, n):
    # the bars of the smaller sizes, with the fp32 kernels in the place of LAPACK (the same blocks and merges in fp32
    # products, whose error the split ones do not exceed; a misplaced block is of order 1)
    from int_crush_converter_amd import _native as nat
    from int_crush_converter_amd.hessian import _damped, inverse_batch
    L = nat.lib()
    H = _large(n, n, gpu_dev)
    truth = torch.cholesky_inverse(torch.linalg.cholesky(_damped(H, 0.01).double()))
    got = inverse_batch(H, 0.01, "hinv")
    assert torch.equal(got, got.T)
    general = H.clone()
    info = torch.zeros(2, dtype=torch.int32, device=gpu_dev)
    ws = nat.workspace(L.ic_hessian_inverse_min_workspace_bytes(1, n), gpu_dev)
    nat.check(L.ic_hessian_inverse_sized(general, 1, n, 0.01, 0, info, ws, ws.numel(), nat.stream()), "inverse")
    s = truth.diagonal().rsqrt()
    e_got, e_gen = (((x.double() - truth) * s[:, None] * s).abs() for x in (got, general))
    assert e_got.norm() <= e_gen.norm(), (e_got.norm().item(), e_gen.norm().item())
    assert e_got.max() <= 4 * e_gen.max(), (e_got.max().item(), e_gen.max().item())


@pytest.mark.parametrize("n", LARGE)
def test_split_inverse_batch_of_batched_merges(gpu_dev, n):
    from int_crush_converter_amd.hessian import inverse_batch
    Hs = torch.stack([_large(n, s, gpu_dev) for s in range(2)])
    got = inverse_batch(Hs, 0.01, "hinv")
    for b in range(2):
        assert torch.equal(got[b], inverse_batch(Hs[b], 0.01, "hinv")), b
