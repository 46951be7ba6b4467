"""The autotuner's table of timed choices (no GPU)."""

import torch

from mr_recon_amd import autotune

CHOICE = {"tile": 32, "samples_per_item": 8192, "ms": {}}


def _lookup(monkeypatch, entries):
    """tune_work's answer from a table, or "timed" where it starts to time candidates."""
    class Timed(Exception):
        pass

    def plan(*a, **k):
        raise Timed

    monkeypatch.setattr(autotune, "_table", entries)
    monkeypatch.setattr(autotune, "SamplePlan", plan)
    try:
        return autotune.tune_work(torch.zeros((1000, 2)), (64, 64), 4.0, 9.0, 2)
    except Timed:
        return "timed"


def test_choices_of_other_kernels_are_not_used(monkeypatch):
    base = autotune.tune_key(2, 4.0, (64, 64), 1000, 2) + "-t8_16_32-s256_512_1024_2048_4096_8192"
    assert _lookup(monkeypatch, {base: CHOICE}) == "timed"  # a table of an older build, without the kernels
    assert _lookup(monkeypatch, {"000000000000-cpu-" + base: CHOICE}) == "timed"
    assert _lookup(monkeypatch, {f"{autotune._kernels()}-gfx90a-{base}": CHOICE}) == "timed"
    assert _lookup(monkeypatch, {f"{autotune._kernels()}-cpu-{base}": CHOICE}) == (32, 8192)
