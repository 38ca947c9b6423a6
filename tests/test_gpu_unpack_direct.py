"""Unpack from registers (unpack_direct_kernel), bit-exact over the whole destination buffer
against the CPU oracle and against the LDS-staged kernel on the same call: pieces of 8 and 16
bytes, tile heights that do not divide the 16 rows of a workgroup, tile rows of one to many
pieces, rows that end at every byte offset an element can have, matrices that end before
their tiles do, rows at any address, both outer orders, one group of 64 pieces and more."""
import numpy as np
import pytest

import uk_testing as T
from golden import make_golden as G
from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tf,t0,t1", [
    (uk.UNPACK_TYPE_F32F32, 16, 16), (uk.UNPACK_TYPE_I32I32, 16, 4), (uk.UNPACK_TYPE_F32F32, 3, 8),
    (uk.UNPACK_TYPE_F32F32, 8, 2), (uk.UNPACK_TYPE_F16F16, 16, 16), (uk.UNPACK_TYPE_BF16BF16, 16, 8),
    (uk.UNPACK_TYPE_F16F16, 20, 4), (uk.UNPACK_TYPE_BF16BF16, 1, 512), (uk.UNPACK_TYPE_F32F32, 1, 1024)])
@pytest.mark.parametrize("flags", [0, uk.UNPACK_TRANSPOSE_OUTER])
def test_unpack_direct(gpu, oracle, tf, t0, t1, flags):
    lib, torch = gpu
    rng = np.random.default_rng(t0 * 1000 + t1)
    es = uk.PACK_TYPE_BYTES[tf]
    sizes = [(1, 320 // es), (15, 100), (16, 101), (17, 102), (33, 103), (50, 257), (5, 4096 // es),
             (31, 4096 // es + 1), (64, 1031), (100, 1024), (257, 259), (3, 5003)]
    for ci, (m, n) in enumerate(sizes):
        # (some with tiles that lie wholly beyond the matrix)
        o0, o1 = -(-m // t0) + (ci % 3 == 2), -(-n // t1) + (ci % 4 == 3)
        s0, s1 = (o1, o0) if flags else (o0, o1)
        c = T.UnpackCase(tf | flags, s0, s1, t0, t1, m, n, s1 * t0 * t1, n + ci % 5, 1, 0, ci % 4)
        inp, out0 = T.make_unpack_buffers(c, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, c, inp, want)
        got = T.gpu_unpack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())
        assert lib.last_kernel_name() == "unpack_direct", c.label()
        lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 1)   # the LDS-staged kernels on the same call
        try:
            staged = T.gpu_unpack(lib, torch, c, inp, out0)
        finally:
            lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        assert np.array_equal(staged, want), (c.label(), "staged")
        assert lib.last_kernel_name() == "unpack_stream", c.label()
