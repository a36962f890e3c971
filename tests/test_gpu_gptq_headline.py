"""Parity at the benchmark's own layer shapes: GPTQ INT4 rot256,
block 128, damping 0.01, on the bench recipe (bf16 W ~ N(0, 0.02^2),
H = X^T X / 8192 with LogNormal(0, 1) channel scales) at [4096, 12288]
(the metric's layer) and C3's [3072, 12288] and [12288, 3072].

Two comparisons per shape, both against the CPU oracle (the reference's
algorithm, converter/rounding.py:37-103 and converter/gptq.py:113-121,
137-417) on the same oracle-rotated W and H:

* same Hinv: the oracle's own damped inverse is handed to the GPU sweep
  (ic_gptq_quantize).  The sweep repeats the reference's fp32 operations,
  and the lazy update subtracts one 128-column block's product at a time
  (each summed in k order from zero, as MKL's sgemm does at K = 128), so
  the codes are expected bit-exact (measured: all equal at every shape); the
  assertion is the stated bar, >= 99.9 % of codes equal and
  tr(dW H dW^T) within 1e-3 relative.
* full path: the GPU computes its own damped inverse.  GPTQ feeds every
  rounding forward, so the bar is relative to the reference's own noise on
  the same inputs: the oracle run again with a half and a quarter of the CPU
  threads (LAPACK's potrf / potri change their fp32 summation order with the
  thread count; the trailing matmul does not) and with the damped inverse
  computed in fp64 and rounded once (the codes of an exact inverse).  The
  GPU's codes must be as close to those exact-inverse codes as the
  reference's are (- 5e-4), agree with the reference within 1.5e-3 of the
  lowest agreement between two of the reference's own thread-count runs, and
  |relative proxy difference| <= max(1e-3, the oracle's own).

The bench path (bf16 W and H rotated on the GPU, then the full layer) is
compared too; its rotation differs from the oracle's matmul by fp32
rounding (within 2e-6 of the row norm), which adds a little noise.  Every
measured number is printed (run with -s to see them).
"""

from __future__ import annotations

import pytest
import torch

from oracle import torch_ref as ref

pytestmark = pytest.mark.gpu

SAMPLES = 8192
SHAPES = [(4096, 12288), (3072, 12288), (12288, 3072)]


def _inputs(M, N, seed):
    """The bench's gptq workload recipe, generated on the GPU, returned on the CPU."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    W = (torch.randn(M, N, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    s = torch.exp(torch.randn(N, generator=g, device=dev))
    H = torch.zeros(N, N, dtype=torch.float32, device=dev)
    for r0 in range(0, SAMPLES, 2048):
        X = torch.randn(min(2048, SAMPLES - r0), N, generator=g, device=dev) * s
        H.addmm_(X.T, X)
        del X
    H /= SAMPLES
    return W.cpu(), H.cpu()


def _sweep_cpu(Wr, s, z, Hinv):
    Q = torch.zeros(Wr.shape, dtype=torch.int8)
    ref.gptq_block(Wr.clone(), Q, s, Hinv, 0, Wr.shape[1], 128, -8, 7, z)
    return Q


@pytest.fixture(scope="module", params=SHAPES, ids=[f"{m}x{n}" for m, n in SHAPES])
def case(gpu_dev, request):
    """The oracle's side of one shape, shared by the three tests of that
    shape (pytest groups the tests by this module-scoped parameter)."""
    return _oracle(*request.param)


def _oracle(M, N, seed=0):
    W, H = _inputs(M, N, seed)
    Wr = ref.rotate_weights(W.float(), 256)
    Hr = ref.rotate_hessian(H, 256)
    s, z = ref.gptq_row_params(Wr, 4, False)
    threads = torch.get_num_threads()
    Hinv_a = ref.prepare_hinv(Hr, 0.01)
    alts = []
    for t in sorted({max(1, threads // 2), max(1, threads // 4)} - {threads}, reverse=True):
        torch.set_num_threads(t)
        try:
            Hinv_t = ref.prepare_hinv(Hr, 0.01)
        finally:
            torch.set_num_threads(threads)
        if not torch.equal(Hinv_a, Hinv_t):
            alts.append(Hinv_t)
    assert alts, "no thread count changes the oracle's inverse"
    # and the inverse computed in fp64 from the same damped fp32 H, rounded
    # once: the reference's own distance from an exact inverse
    Hd64 = ref.damp(Hr, 0.01).double()
    alts.append(torch.cholesky_inverse(torch.linalg.cholesky(Hd64)).float())
    del Hd64
    Qa = _sweep_cpu(Wr, s, z, Hinv_a)
    Qalts = [_sweep_cpu(Wr, s, z, Hi) for Hi in alts]
    # the oracle's own run-to-run noise: its least agreeing variant, and the
    # lowest agreement between any two of its runs (the spread of this
    # statistic between independent fp32 executions)
    Qx = Qalts.pop()
    Qb = min(Qalts, key=lambda q: (q == Qa).float().mean().item())
    runs = [Qa] + Qalts
    pair_min = min((runs[i] == runs[j]).float().mean().item()
                   for i in range(len(runs)) for j in range(i + 1, len(runs)))
    return dict(M=M, N=N, W=W, H=H, Wr=Wr, Hr=Hr, s=s, z=z, Hinv=Hinv_a, Qa=Qa, Qb=Qb, Qx=Qx, pair_min=pair_min)


def _proxy(Wr, Q, s16, z, Hd):
    """tr(dW H dW^T), dW = (Q - z) s - W, in fp64 on the GPU."""
    dev = Hd.device
    d = (Q.to(dev).double() - z.to(dev).double()) * s16.to(dev).double() - Wr.to(dev).double()
    return ((d @ Hd) * d).sum().item()


def _report(tag, **kv):
    print(f"[parity] {tag} " + " ".join(f"{k}={v:.6g}" if isinstance(v, float) else f"{k}={v}"
                                        for k, v in kv.items()), flush=True)


def test_same_hinv_north_star(gpu_dev, case):
    from int_crush_converter_amd.gptq import row_params, sweep
    c = case
    M, N = c["M"], c["N"]
    Wg = c["Wr"].to(gpu_dev)
    s32, z32, s16, z8 = row_params(Wg, 4, False)
    assert torch.equal(s32.cpu(), c["s"].squeeze(1))
    assert torch.equal(z8.cpu(), c["z"].squeeze(1))
    Q = sweep(Wg, c["Hinv"].to(gpu_dev), s32, z32, 4, 128).cpu()
    agree = (Q == c["Qa"]).float().mean().item()
    Hd = c["Hr"].to(gpu_dev).double()
    s16c = c["s"].to(torch.float16).float()
    p_ref = _proxy(c["Wr"], c["Qa"], s16c, c["z"], Hd)
    p_got = _proxy(c["Wr"], Q, s16c, c["z"], Hd)
    rel = p_got / p_ref - 1
    _report(f"same_hinv {M}x{N}", agreement=agree, proxy_rel=rel, mismatches=int((Q != c["Qa"]).sum()))
    assert agree >= 0.999, agree
    assert abs(rel) <= 1e-3, rel
    assert torch.equal(Q, c["Qa"])


def test_full_path_vs_reference_noise(gpu_dev, case):
    from int_crush_converter_amd.gptq import gptq_quantize_layer
    c = case
    M, N = c["M"], c["N"]
    r = gptq_quantize_layer(c["Wr"].to(gpu_dev), c["Hr"].to(gpu_dev), block_size=128, damping=0.01, int_bits=4)
    s16 = c["s"].to(torch.float16)
    assert torch.equal(r.scales.cpu().squeeze(1), s16.squeeze(1))
    assert torch.equal(r.zero_points.cpu(), c["z"])
    Q = r.quantized_W.cpu()
    Hd = c["Hr"].to(gpu_dev).double()
    sf = s16.float()
    p_a = _proxy(c["Wr"], c["Qa"], sf, c["z"], Hd)
    rel = _proxy(c["Wr"], Q, sf, c["z"], Hd) / p_a - 1
    rel_self = _proxy(c["Wr"], c["Qb"], sf, c["z"], Hd) / p_a - 1
    agree = (Q == c["Qa"]).float().mean().item()
    self_agree = (c["Qb"] == c["Qa"]).float().mean().item()
    exact_gpu = (Q == c["Qx"]).float().mean().item()
    exact_ref = (c["Qa"] == c["Qx"]).float().mean().item()
    _report(f"full_path {M}x{N}", agreement=agree, self_agreement=self_agree, self_pair_min=c["pair_min"],
            vs_exact_inverse_gpu=exact_gpu, vs_exact_inverse_oracle=exact_ref, proxy_rel=rel,
            self_proxy_rel=rel_self)
    # as close to the codes of an exact inverse as the reference is
    assert exact_gpu >= exact_ref - 5e-4, (exact_gpu, exact_ref)
    # and as close to the reference as its own runs are to each other, within
    # the spread of that statistic between independent fp32 executions
    assert agree >= c["pair_min"] - 1.5e-3, (agree, c["pair_min"])
    assert abs(rel) <= max(1e-3, abs(rel_self)), (rel, rel_self)


def _fp16_ulps(a, b):
    return (a.to(torch.float16).view(torch.int16).int() - b.to(torch.float16).view(torch.int16).int()).abs().max().item()


def test_bench_path_vs_reference_noise(gpu_dev, case):
    """bf16 W and the raw H rotated on the GPU (the timed step of bench.py),
    then the full layer.  The GPU's butterfly rotation and the reference's
    matmul round differently (within 2e-6 of the row norm), and GPTQ
    amplifies that like any other fp32 difference, so the reference itself
    is the yardstick again: the oracle's layer on the GPU-rotated W and H
    against the oracle's layer on its own rotation.  The GPU path must agree
    with the oracle's own-rotation codes at least as well (- 5e-4), and with
    the oracle on the very same rotated inputs at least as well as the
    oracle agrees with itself across thread counts (- 5e-4).  Measured:
    the end-to-end agreement is within 6e-4 of the oracle's own rotation
    noise (both rounding sources against one), hence the 1e-3 there."""
    from int_crush_converter_amd import layer as L
    from int_crush_converter_amd.rotation import rotate_hessian_gpu
    c = case
    M, N = c["M"], c["N"]
    W_work, _ = L.prepare_weights(c["W"].to(gpu_dev), 256)
    Hg = rotate_hessian_gpu(c["H"].to(gpu_dev), 256).cpu()
    Wg = W_work.cpu()
    codes, s16, z8 = L.gptq_codes(W_work, c["H"].to(gpu_dev), rotate_h=256, block_size=128, damping=0.01,
                                  int_bits=4, asymmetric=False, hessian_method="hinv", fallbacks=[])
    Q = codes.cpu()
    # the oracle on the GPU-rotated inputs
    rg = ref.gptq_quantize_layer(Wg, Hg, 128, 0.01, 4)
    Qr = rg.quantized_W
    Hd = c["Hr"].to(gpu_dev).double()
    sf = c["s"].to(torch.float16).float()
    p_a = _proxy(c["Wr"], c["Qa"], sf, c["z"], Hd)
    # the GPU's codes with the GPU's own stored scales and zero-points
    rel = _proxy(c["Wr"], Q, s16.cpu().float(), z8.cpu(), Hd) / p_a - 1
    rel_rot = _proxy(c["Wr"], Qr, rg.scales.float(), rg.zero_points, Hd) / p_a - 1
    rel_self = _proxy(c["Wr"], c["Qb"], sf, c["z"], Hd) / p_a - 1
    agree = (Q == c["Qa"]).float().mean().item()
    agree_same_inputs = (Q == Qr).float().mean().item()
    rot_agree = (Qr == c["Qa"]).float().mean().item()
    self_agree = (c["Qb"] == c["Qa"]).float().mean().item()
    s_want = c["s"].to(torch.float16).reshape(-1)
    s_got = s16.cpu().reshape(-1)
    ulps = _fp16_ulps(s_got, s_want)
    _report(f"bench_path {M}x{N}", agreement=agree, oracle_rotation_agreement=rot_agree,
            agreement_same_inputs=agree_same_inputs, self_agreement=self_agree, proxy_rel=rel,
            oracle_rotation_proxy_rel=rel_rot, self_proxy_rel=rel_self,
            scale_rows_differing=int((s_got != s_want).sum()), scale_max_ulps=ulps)
    assert ulps <= 1
    assert torch.equal(s16.cpu().reshape(-1), rg.scales.reshape(-1))
    # two rounding sources (rotation and inverse) against one (rotation)
    assert agree >= min(rot_agree, self_agree) - 1e-3, (agree, rot_agree, self_agree)
    assert agree_same_inputs >= self_agree - 5e-4, (agree_same_inputs, self_agree)
    assert abs(rel) <= max(1e-3, 2 * abs(rel_rot), 2 * abs(rel_self)), (rel, rel_rot, rel_self)
