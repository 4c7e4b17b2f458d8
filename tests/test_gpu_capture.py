"""HIP graph captures whose eager calls were of other shapes, each in a process
of its own (capture_child.py): the kernel that a call takes does not depend on
what the workspace holds, so a captured call gives the eager call's bits, or
is refused with Q4K_ECAPTURE where no call has set up a workspace at all."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("case", ["prefill", "decode", "first"])
def test_capture_after_other_shapes(case, gpu):
    env = {k: v for k, v in os.environ.items() if not k.startswith(("Q4K_", "Q6K_"))}
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "capture_child.py"), case], env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, f"{case} failed ({r.returncode}):\n{r.stdout[-1000:]}\n{r.stderr[-2000:]}"
