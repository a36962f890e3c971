"""GPU parity of the Cholesky's diagonal block, panel solve and block inverse
(csrc/chol.hip) at the edges of their 16 x 16 tiles, 128-blocks, 16-row panel
sets and 1024-column super-blocks, odd row pitches included.

Bars: the factor and the inverse are as close to their 64-bit values as the
reference's fp32 path (LAPACK) on the same matrix - the diagonal blocks and
panels are worked in 64 bits here, in 32 there - and four roundings of every
element: of X = L^-1 to fp32 (twice in X^T X), of the product and of the
result, where LAPACK's own error falls by chance."""

from __future__ import annotations

import pytest
import torch

from oracle import torch_ref as ref
from tests.conftest import lognormal_hessian

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 33, 127, 128, 129, 143, 145, 255, 257, 1023, 1025, 1153]


def _cholesky(H, dev):
    from int_crush_converter_amd import _native as nat
    out = H.to(dev).clone()
    n = H.shape[0]
    info = torch.zeros(1, dtype=torch.int32, device=dev)
    ws = nat.workspace(nat.lib().ic_hessian_inverse_workspace_bytes(1, n), out.device)
    nat.check(nat.lib().ic_cholesky(out, 1, n, info, ws, nat.stream()), "ic_cholesky")
    return torch.tril(out).cpu(), int(info.item())


@pytest.mark.parametrize("n", SIZES)
def test_factor_and_inverse_error_at_most_lapack(gpu_dev, n):
    from int_crush_converter_amd.hessian import inverse_batch
    Hd = ref.damp(lognormal_hessian(n, n + 64, n), 0.01)
    L64 = torch.linalg.cholesky(Hd.double())
    L, info = _cholesky(Hd, gpu_dev)
    assert info == 0
    X64 = torch.cholesky_inverse(L64)
    X = inverse_batch(Hd.to(gpu_dev), 0.0, "hinv").cpu()
    assert torch.equal(X, X.T)
    for got, want, lapack in ((L, L64, torch.linalg.cholesky(Hd)),
                              (X, X64, torch.cholesky_inverse(torch.linalg.cholesky(Hd)))):
        e_got, e_ref = ((a.double() - want).norm().item() for a in (got, lapack))
        assert e_got <= e_ref + 4 * 2.0 ** -24 * want.norm().item(), (e_got, e_ref)


@pytest.mark.parametrize("column", [0, 1, 15, 16, 100, 127, 128, 143, 255, 256, 299])
def test_first_bad_pivot_is_reported(gpu_dev, column):
    H = torch.eye(300) + 0.001
    H[column, column] = -1.0
    assert _cholesky(H, gpu_dev)[1] == column + 1
