"""GPU parity of the rotation kernels for small launches (csrc/rotate_exact.hip,
narrow): one row, rows and widths around their tiles of 16 and 256, padded
widths, every source type, the outlier count, Hessians 2-D / 3-D / lower
triangle.  Bit for bit the oracle's sequential chains, at sizes on both sides
of the switch to the wide kernels (128 of their work-groups)."""

from __future__ import annotations

import pytest
import torch

from oracle import torch_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rot", [64, 256])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 64), (15, 300), (16, 512), (17, 1000), (64, 256), (129, 1023),
                                       (2048, 1024), (2112, 1024)])
def test_rows_bit_exact(gpu_dev, rot, dtype, rows, cols):
    from int_crush_converter_amd.rotation import rotate_rows_gpu
    g = torch.Generator().manual_seed(rows + cols + rot)
    W = torch.randn(rows, cols, generator=g)
    W[0, cols // 2] = 5000.0
    W[-1, 0] = -2000.0
    W = W.to(dtype)
    nz = torch.zeros(1, dtype=torch.int64, device=gpu_dev)
    got = rotate_rows_gpu(W.to(gpu_dev), rot, 1000.0, nz)
    Wf = W.float()
    want = ref.rotate_weights(Wf.masked_fill(Wf.abs() > 1000.0, 0.0), rot)
    assert torch.equal(got.cpu(), want)
    assert int(nz.item()) == int((Wf.abs() > 1000.0).sum())


@pytest.mark.parametrize("rot", [64, 256])
@pytest.mark.parametrize("shape", [(256, 256), (512, 512), (300, 300), (1280, 1280), (1536, 1536), (3, 256, 256),
                                   (2, 512, 512)])
def test_hessian_bit_exact(gpu_dev, rot, shape):
    from int_crush_converter_amd.rotation import rotate_hessian_gpu
    H = torch.randn(*shape, generator=torch.Generator().manual_seed(sum(shape) + rot))
    want = ref.rotate_hessian(H, rot)
    assert torch.equal(rotate_hessian_gpu(H.to(gpu_dev), rot).cpu(), want)
    if H.dim() == 2 and H.shape[0] % rot == 0:
        work = H.to(gpu_dev)
        low = rotate_hessian_gpu(work, rot, lower_only=True, inplace=True).cpu()
        n = H.shape[0]
        i = torch.arange(n) // rot
        keep = i[:, None] >= i[None, :]
        assert torch.equal(low[keep], want[keep])
