"""mi_conv_up_staged on a conv whose upsampled segment is not what it says ends the process with a message before anything is launched (no GPU: the pointers
are never followed)."""
import os
import signal
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CALL = """
from ufsm_amd import lib, gnp_t, shape5, split_t
xdt, cc, G, staged = %d, %d, %d, %d
sp = split_t(); sp.x2, sp.c_split, sp.up = 4096, cc, 1
sp.gp2.G = -1
gp = gnp_t()
if G: gp.gamma = gp.beta = gp.mean = gp.rstd = 4096; gp.G = G
lib.mi_conv_up_staged(staged)
lib.lp_conv_fwd_f8(4096, xdt, shape5(1, cc + 32, 8, 8, 8), 4096, 4096, 32, 4096, 3, gp, None, 0, sp)
"""


@pytest.mark.parametrize("xdt,cc,G", [(4, 64, 0), (3, 48, 0), (3, 64, 8), (4, 40, 8)])
def test_staged_segment_that_is_no_rows_is_refused(xdt, cc, G):
    r = subprocess.run([sys.executable, "-c", CALL % (xdt, cc, G, 1)], cwd=ROOT, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"), capture_output=True, text=True, timeout=120)
    assert r.returncode == -signal.SIGABRT and "mi_conv_up_staged needs" in r.stderr, (r.returncode, r.stderr)
