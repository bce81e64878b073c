"""Host waits of the library.  With several threads on streams of their own the runtime's
hipStreamSynchronize has returned while the stream's kernels still ran; the host then reads
counts, status words and results that are not there yet, and gives memory on that is in use.
The library waits for events instead (stream_wait)."""
import glob
import os
import re
import subprocess

import dtc_amd._lib as L
from conftest import PKG


def test_no_result_hangs_on_a_wait_by_stream_or_device():
    out = subprocess.run(["nm", "-D", "--undefined-only", L.LIB_PATH], capture_output=True, text=True, check=True).stdout
    names = {line.split()[-1].split("@")[0] for line in out.splitlines()}
    assert "hipEventSynchronize" in names and "hipDeviceSynchronize" not in names
    calls = []
    for f in glob.glob(os.path.join(PKG, "csrc", "*")):
        src = re.sub(r"//.*", "", open(f).read())
        calls += [os.path.basename(f)] * len(re.findall(r"\bhip(?:Stream|Device)Synchronize\s*\(", src))
    # the one before the destruction of a stream or its graph: their work has been waited for, or is given up
    assert calls == ["capi.cpp"]
