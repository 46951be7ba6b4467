"""The committed profiles are of kernels that exist: bench.py reports a counter out of one of them."""

import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SOURCES = "".join(p.read_text() for p in (ROOT / "mr_recon_amd" / "csrc").glob("*.h*"))


@pytest.mark.parametrize("path", sorted((ROOT / "profiles").glob("*.md")), ids=lambda p: p.stem)
def test_profiled_kernels_exist(path):
    names = set(re.findall(r"`(?:\w+::)*(\w+_kernel)\b", path.read_text()))
    assert names and not [n for n in names if not re.search(rf"\bvoid {n}\(", SOURCES)]
