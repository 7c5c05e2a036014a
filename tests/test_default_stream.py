"""The library leaves the default stream alone: any use of it, in any thread, fails beside a
capture and ends it, and engines capture their batches."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_call_uses_the_default_stream():
    found = []
    for path in glob.glob(os.path.join(ROOT, "graph500-bfs_amd", "csrc", "*.h*")):
        with open(path) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        # calls without a stream, and launches on stream 0
        found += [(os.path.basename(path), m.group(0)) for m in re.finditer(
            r"hipMem(cpy|set)(2D|3D|D8|D16|D32|DtoH|HtoD|DtoD|ToSymbol|FromSymbol)?\s*\(|<<<", text)]
        for m in re.finditer(r"hipLaunchKernelGGL\((?:[^;]*?)dim3\([^;]*?dim3\([^;]*?\),\s*[\w()]+,\s*"
                             r"([^,;]+),", text):
            if m.group(1).strip() in ("0", "nullptr", "hipStreamDefault"):
                found.append((os.path.basename(path), m.group(0)[:60]))
    assert not found, found
