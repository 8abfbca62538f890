"""Every device allocation of the library goes through device_malloc, which
gives the spare buffers of destroyed states back and tries again when the
device is full (CPU: the sources are read)."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "latticemodels.jl_amd", "csrc")


def test_one_place_calls_hipMalloc():
    found = {}
    for name in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, name)).read()
        text = re.sub(r"//[^\n]*", "", re.sub(r"/\*.*?\*/", "", text, flags=re.S))
        n = len(re.findall(r"\bhip(?:Ext)?Malloc(?:Async|Managed|WithFlags)?\s*\(", text))
        if n:
            found[name] = n
    assert found == {"api_core.hip": 2}
    body = open(os.path.join(CSRC, "api_core.hip")).read()
    body = body[body.index("hipError_t device_malloc("):]
    assert body[: body.index("\n}\n")].count("hipMalloc(") == 2
