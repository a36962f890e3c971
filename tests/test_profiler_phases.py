"""The launch profiler's phases and the kernels they are graded as."""

from __future__ import annotations

import ctypes
import os
import re

import pytest
import torch

from int_crush_converter_amd import _native as nat

CSRC = os.path.join(os.path.dirname(nat.__file__), "csrc")


def test_profiled_kernels_exist():
    kernels = set()
    for f in os.listdir(CSRC):
        with open(os.path.join(CSRC, f)) as src:
            # the name before the parameter list, attributes and launch bounds skipped
            kernels |= set(re.findall(r"\b(\w+)\s*\(", " ".join(re.findall(r"__global__[^{;]*", src.read()))))
    for table in (nat.PROFILE_KERNELS, {n: (None, b) for n, b in nat.FWHT_KERNELS.values()}):
        for names in table:
            for name in re.split(r" / | \+ ", names):
                assert name in kernels or name + "_kernel" in kernels, name


def test_every_phase_of_a_table_is_read():
    phases = [p for ps, _ in nat.PROFILE_KERNELS.values() for p in ps]
    assert len(phases) == len(set(phases)) and set(phases) <= set(nat.PROFILE_TAGS)


@pytest.mark.gpu
def test_split_products_have_their_own_phases(gpu_dev):
    from int_crush_converter_amd.hessian import inverse_batch
    from tests.conftest import lognormal_hessian
    import bench
    H = lognormal_hessian(4096, 4608, 1).to(gpu_dev)
    inverse_batch(H, 0.01, "hinv")
    torch.cuda.synchronize()
    nat.profile_enable(True)
    try:
        inverse_batch(H, 0.01, "hinv")
        prof = nat.profile_read()
        n = 19   # a caller that knows the phases without split operands
        ms, fl, by = ((ctypes.c_double * n)() for _ in range(3))
        la = (ctypes.c_int64 * n)()
        nat.check(nat.lib().ic_profile_read(ms, fl, by, la, n), "ic_profile_read")
    finally:
        nat.profile_enable(False)
    for split, whole in (("split_cholesky", "gemm_cholesky"), ("split_inverse", "gemm_inverse"),
                         ("split_planes", "other")):
        assert prof[split]["launches"] > 0
        assert la[nat.PROFILE_TAGS.index(whole)] == prof[split]["launches"] + prof[whole]["launches"]
    name, roof = bench.roofline_from(prof, "")
    assert 0 < roof["frac"] < 1, (name, roof)


@pytest.mark.gpu
def test_planes_that_nothing_reads_are_not_formed(gpu_dev):
    # n = 3200: columns 1024 .. 2047 have an update of 1152 rows, which is not split, below them; a merge reads their
    # planes.  chol(H^-1) has no merge: one set of planes, for the split update of 2176 rows
    from int_crush_converter_amd.hessian import inverse_batch
    from tests.conftest import lognormal_hessian
    H = lognormal_hessian(3200, 3712, 1).to(gpu_dev)
    launches = {}
    for method in ("hinv", "cholesky"):
        nat.profile_enable(True)
        try:
            inverse_batch(H, 0.01, method)
            launches[method] = nat.profile_read()["split_planes"]["launches"]
        finally:
            nat.profile_enable(False)
    assert launches["cholesky"] == launches["hinv"] + 1, launches
