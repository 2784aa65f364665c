"""CPU: steps are launched directly.  Replaying a captured graph was taken out
(host segmentation faults without a cause shown), so the library uses none of
the runtime's graph calls."""
import os
import shutil
import subprocess

import pytest


@pytest.mark.skipif(shutil.which("nm") is None, reason="needs nm")
def test_the_library_uses_no_graph_calls():
    import zdx

    if not os.path.exists(zdx.LIB_PATH):
        pytest.skip("libzdx.so not built")
    r = subprocess.run(["nm", "-D", "--undefined-only", zdx.LIB_PATH], capture_output=True, text=True)
    assert r.returncode == 0 and "hipLaunchKernel" in r.stdout
    assert "hipGraph" not in r.stdout and "Capture" not in r.stdout
