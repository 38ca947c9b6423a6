"""Without a device to ask, calls on device operands end with an error status, not with
the process: nothing is launched and no operand is touched."""
import os
import subprocess
import sys

import pytest

from iree_amd import ukernel as uk

CODE = """
from iree_amd import ukernel as uk
lib = uk.load()
assert uk.load().lib.iree_uk_amd_device_count() == 0
lib.set_pointer_mode(uk.POINTER_MODE_DEVICE)
try:
    lib.mmt4d(4096, 0, {k1} * 16 * {k0}, 4096, 0, {k1} * 16 * {k0}, 4096, 0, {n1} * 256, {m1}, {n1}, {k1}, 16, 16, {k0},
              {flags})
except Exception as e:
    print("raised", type(e).__name__)
"""


@pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="for machines without a GPU")
@pytest.mark.parametrize("flags,k0", [(uk.MMT4D_TYPE_F32F32F32, 1), (uk.MMT4D_TYPE_F32F32F32, 4), (uk.MMT4D_TYPE_S8S8S32, 16),
                                      (uk.MMT4D_TYPE_F16F16F32, 8), (uk.MMT4D_TYPE_BF16BF16F32, 2)])
@pytest.mark.parametrize("m1,n1,k1", [(1, 64, 768), (33, 65, 768), (8, 256, 4096), (300, 300, 64)])
def test_a_failing_device_query_is_an_error(flags, k0, m1, n1, k1):
    code = CODE.format(flags=flags, k0=k0, m1=m1, n1=n1, k1=k1)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode == 0 and r.stdout.startswith("raised"), (r.returncode, r.stdout, r.stderr[-500:])
