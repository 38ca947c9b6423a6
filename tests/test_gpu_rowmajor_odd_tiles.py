"""Row-major results of mmt4d in tiles whose columns are no multiple of four: a
workgroup's columns then end inside four neighbouring ones, the rest of which
are the next workgroup's. Small integers: equal to the product in 64 bits."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["s8", "f16", "f16f16"])
@pytest.mark.parametrize("variant", [0, 1, 2, 3, 16, 18, 20])
@pytest.mark.parametrize("n0", [7, 9, 10])
def test_blocks_store_their_own_columns_only(gpu, dtype, variant, n0):
    lib, torch = gpu
    flags, tin, tout = {"s8": (uk.MMT4D_TYPE_S8S8S32, torch.int8, torch.int32),
                        "f16": (uk.MMT4D_TYPE_F16F16F32, torch.float16, torch.float32),
                        "f16f16": (uk.MMT4D_TYPE_F16F16F16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, torch.float16,
                                   torch.float16)}[dtype]
    m0, k0, k1, m1 = 16, 16, 24, 20
    n1 = -(-1100 // n0)
    m, n = m1 * m0 - 5, n1 * n0 - 2
    gen = torch.Generator(); gen.manual_seed(n0)
    lhs = torch.randint(-2, 3, (m1, k1, m0, k0), generator=gen)
    rhs = torch.randint(-2, 3, (n1, k1, n0, k0), generator=gen)
    a = lhs.permute(0, 2, 1, 3).reshape(m1 * m0, k1 * k0).double()[:m]
    b = rhs.permute(0, 2, 1, 3).reshape(n1 * n0, k1 * k0).double()[:n]
    d_lhs, d_rhs = lhs.to(tin).cuda(), rhs.to(tin).cuda()
    out = torch.full((m, n), 7, device="cuda", dtype=tout)
    lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + variant if variant else uk.KERNEL_MODE_AUTO)
    try:
        lib.mmt4d_unpack(d_lhs.data_ptr(), 0, k1 * m0 * k0, d_rhs.data_ptr(), 0, k1 * n0 * k0, out.data_ptr(), 0, n, m, n,
                         m1, n1, k1, m0, n0, k0, flags)
        lib.synchronize()
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    assert torch.equal(out.cpu(), (a @ b.T).to(tout)), lib.last_kernel_name()
