"""load_calibration with mmap: the same data as the plain load, files that
cannot be mapped (the pre-zip format) read whole, the same errors."""

from __future__ import annotations

import pytest
import torch

from int_crush_converter_amd.calibration_io import load_calibration

DATA = {"hessians": {"a": torch.arange(9.0).reshape(3, 3)}, "shapes": {"a": [3, 3]}, "layer_types": {"a": "linear"}}


@pytest.mark.parametrize("zipped", [True, False])
def test_mapped_equals_plain(tmp_path, zipped):
    path = str(tmp_path / "c.pt")
    torch.save(DATA, path, _use_new_zipfile_serialization=zipped)
    for mmap in (False, True):
        got = load_calibration(path, mmap=mmap)
        assert torch.equal(got["hessians"]["a"], DATA["hessians"]["a"]) and got["shapes"] == DATA["shapes"]


@pytest.mark.parametrize("mmap", [False, True])
def test_errors(tmp_path, mmap):
    with pytest.raises(ValueError, match="not found"):
        load_calibration(str(tmp_path / "none.pt"), mmap=mmap)
    bad = tmp_path / "bad.pt"
    bad.write_bytes(b"not a checkpoint")
    with pytest.raises(ValueError, match="corrupted"):
        load_calibration(str(bad), mmap=mmap)
    missing = str(tmp_path / "m.pt")
    torch.save({"hessians": {}}, missing)
    with pytest.raises(KeyError):
        load_calibration(missing, mmap=mmap)
