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
    for f in sorted(glob.glob(os.path.join(PKG, "csrc", "*"))):
        src = re.sub(r"//.*", "", open(f).read())
        calls += [(os.path.basename(f), src[m.end():m.end() + 80])
                  for m in re.finditer(r"\bhip(?:Stream|Device)Synchronize\s*\(", src)]
    # one ahead of the event's wait, one before the destruction of a stream or its graph
    assert [c[0] for c in calls] == ["capi.cpp", "dtc_internal.hpp"]
    assert "hipEventSynchronize" in calls[1][1]
