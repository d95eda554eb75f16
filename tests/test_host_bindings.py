"""A launch waits while its stream's queue is full, so no call of the host extension may hold the interpreter
meanwhile: other threads would stand still with it."""
import re
from pathlib import Path

import megalodon_amd

HOST = Path(megalodon_amd.__file__).parent / "csrc" / "host"


def test_every_call_releases_the_interpreter():
    calls = [c for f in HOST.glob("*.cpp") for c in re.findall(r"m\.def\((.*?)\);", f.read_text(), flags=re.S)]
    assert len(calls) >= 10
    assert not [c for c in calls if not re.search(r"free\(\)|call_guard<py::gil_scoped_release>\(\)", c)]


def test_no_call_touches_python_objects():
    for f in HOST.glob("*.cpp"):
        text = re.sub(r"//.*", "", f.read_text())
        assert not re.search(r"py::(object|cast|tuple|dict|list|make_tuple|none|getattr|setattr)\b", text), f.name
