"""What the inverse asks of its caller (no GPU: the queries are host code)."""

from __future__ import annotations

import pytest

from int_crush_converter_amd import _native as nat


@pytest.mark.parametrize("batch,n", [(1, 1), (1, 128), (3, 1000), (1, 2049), (2, 12288)])
def test_inverse_least_workspace(batch, n):
    # X in fp32, 128 x 128 doubles for every diagonal block, alignment; nothing else is written without planes
    lib = nat.load()
    blocks = -(-n // 128)
    assert lib.ic_hessian_inverse_min_workspace_bytes(batch, n) == 4 * batch * n * n + 8 * batch * blocks * 128 * 128 + 256
