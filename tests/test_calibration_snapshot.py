"""The calibration a run works with is the file as it was when the run began:
the file may be rewritten in place or truncated as soon as it has been loaded
(a mapping of it would show the new bytes, or end the process).  And the
parallel read it is loaded with: the same data as torch's own, tensors below,
at and past a piece of a read, both file formats, the same errors."""

from __future__ import annotations

import io
import os
import pathlib

import pytest
import torch

from int_crush_converter_amd import calibration_io as cio
from int_crush_converter_amd import pipeline
from int_crush_converter_amd.types import QuantizeConfig


class _Loaded(Exception):
    pass


@pytest.mark.parametrize("truncate", [False, True])
def test_run_keeps_the_calibration_it_began_with(tmp_path, monkeypatch, truncate):
    from safetensors.torch import save_file
    model, cal = str(tmp_path / "m.safetensors"), str(tmp_path / "c.pt")
    save_file({"a.weight": torch.ones(8, 512)}, model)
    H = torch.arange(512.0 * 512).reshape(512, 512)
    torch.save({"hessians": {"a": H}, "shapes": {"a": [512, 512]}, "layer_types": {"a": "linear"}}, cal)
    load = pipeline.load_calibration

    def load_then_rewrite(*args, **kwargs):
        data = load(*args, **kwargs)
        size = os.path.getsize(cal)
        with open(cal, "r+b") as f:
            f.write(b"\xff" * size)
        # (first, so that a mapping fails here and not by a signal below)
        assert torch.equal(data["hessians"]["a"], H)
        if truncate:
            os.truncate(cal, 0)
            assert torch.equal(data["hessians"]["a"], H)
        raise _Loaded

    monkeypatch.setattr(pipeline, "load_calibration", load_then_rewrite)
    config = QuantizeConfig(input_path=model, output_dir=str(tmp_path / "out"), rot_size=256, quant_method="gptq",
                            calibration_path=cal, int_bits=4)
    with pytest.raises(_Loaded):
        pipeline.quantize_model(config, streaming=False)


@pytest.mark.parametrize("zipped", [True, False])
def test_parallel_read_equals_torch_load(tmp_path, zipped):
    path = str(tmp_path / "c.pt")
    piece = cio.READ_PIECE
    hess = {str(n): torch.randint(0, 256, (n,), dtype=torch.uint8) for n in (0, 1, piece - 1, piece, piece + 1, 9 * piece + 5)}
    torch.save({"hessians": hess, "shapes": {}, "layer_types": {}}, path, _use_new_zipfile_serialization=zipped)
    with open(path, "rb") as f:
        buffer = io.BytesIO(f.read())
    for source in (path, pathlib.Path(path), buffer):
        got = cio.load_calibration(source)["hessians"]
        assert got.keys() == hess.keys() and all(torch.equal(got[k], hess[k]) for k in hess)


def test_errors(tmp_path):
    with pytest.raises(ValueError, match="not found"):
        cio.load_calibration(str(tmp_path / "none.pt"))
    bad = tmp_path / "bad.pt"
    for content in (b"", b"PK\x03\x04", b"not a checkpoint"):
        bad.write_bytes(content)
        with pytest.raises(ValueError, match="corrupted"):
            cio.load_calibration(str(bad))
    whole = tmp_path / "whole.pt"
    torch.save({"hessians": {"a": torch.zeros(1 << 20)}, "shapes": {}, "layer_types": {}}, whole)
    bad.write_bytes(whole.read_bytes()[:1 << 20])
    with pytest.raises(ValueError, match="corrupted"):
        cio.load_calibration(str(bad))


def test_file_truncated_while_it_is_read(tmp_path, monkeypatch):
    path = str(tmp_path / "c.pt")
    torch.save({"hessians": {"a": torch.zeros(4 << 20)}, "shapes": {}, "layer_types": {}}, path)
    pread = cio._pread_into

    def cut_then_read(fd, mv, *args):
        if len(mv) == cio.READ_PIECE:   # the tensor's data is being read
            os.truncate(path, 4096)
        pread(fd, mv, *args)

    monkeypatch.setattr(cio, "_pread_into", cut_then_read)
    with pytest.raises(ValueError, match="corrupted"):
        cio.load_calibration(path)
