"""Blocks of 32x32 to 64x64 of the barrier-free kernel, and those of the LDS pipeline they
are weighed against: each shape with each class of tile rows, at K that ends inside a step
or in whole steps, panels of odd sizes, more block rows than columns and fewer, numbers of
blocks that the eight XCDs do not divide. Small integers, so that every order of the sums
gives the product in 64 bits."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

F16 = (uk.MMT4D_TYPE_F16F16F32, "float16", "float32")
BF16 = (uk.MMT4D_TYPE_BF16BF16F32, "bfloat16", "float32")
BF16BF16 = (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16")
S8 = (uk.MMT4D_TYPE_S8S8S32, "int8", "int32")
F8 = (uk.MMT4D_TYPE_F8E4M3FNF8E4M3FNF32, "float8_e4m3fn", "float32")
F32 = (uk.MMT4D_TYPE_F32F32F32, "float32", "float32")


def _tiles(torch, x, m0, k0):
    rows, k = x.shape
    return (torch.nn.functional.pad(x, (0, -k % k0, 0, -rows % m0)).view(-(-rows // m0), m0, -(-k // k0), k0)
            .permute(0, 2, 1, 3).contiguous())


@pytest.mark.parametrize("kind,tile,m,n,k,name", [
    (F16, (16, 16, 8), 700, 900, 1504, "64x64_ksplit"),
    (F16, (16, 16, 8), 513, 2041, 1020, "32x32_ksplit"),
    (F16, (16, 16, 8), 1000, 1501, 777, "32x64_ksplit"),
    (F8, (16, 16, 16), 1090, 1412, 105, "64x64_rhs_direct"),   # (256 bytes of K and less: not by costs)
    (S8, (16, 16, 16), 716, 2957, 256, "64x64_rhs_direct"),
    (BF16, (16, 16, 1), 131, 521, 2003, "32x32_ksplit"),
    (F16, (16, 16, 16), 300, 4096, 530, "32x32_ksplit"),
    (F16, (48, 16, 8), 1500, 1490, 1504, "128x128_lds_direct"),
    (BF16BF16, (16, 16, 8), 777, 1011, 643, "64x64_ksplit"),
    (BF16, (16, 16, 2), 1000, 1500, 783, "32x64_ksplit"),
    (BF16, (16, 16, 2), 530, 2048, 2047, "64x64_ksplit"),
    (BF16, (16, 32, 4), 1011, 777, 1281, "64x64_ksplit"),
    (S8, (16, 16, 8), 530, 1080, 2047, "32x32_ksplit"),
    (S8, (16, 16, 8), 2000, 300, 4099, "64x64_ksplit"),
    (S8, (32, 16, 16), 600, 800, 3001, "32x64_ksplit"),
    (S8, (16, 16, 2), 700, 1000, 1111, "64x64_lds_direct"),
    (S8, (16, 16, 2), 500, 500, 1111, "32x32_ksplit"),
    (S8, (16, 16, 2), 2000, 700, 2001, "128x128_lds_direct"),
    (S8, (16, 16, 4), 930, 1033, 2111, "64x64_ksplit"),
    (F8, (16, 16, 16), 900, 1100, 1300, "32x32_ksplit"),
    (F8, (16, 16, 16), 512, 2048, 4100, "64x64_ksplit"),
    (F8, (16, 16, 16), 1100, 700, 2051, "64x64_ksplit"),
    (F32, (16, 16, 4), 515, 1027, 770, "48x48_ksplit"),
    (F32, (16, 16, 1), 1027, 515, 771, "48x48_ksplit"),
    (F32, (16, 16, 1), 600, 700, 300, "32x32_ksplit"),
    (F32, (16, 16, 4), 1100, 1300, 2001, "32x48_ksplit"),
    (F32, (16, 16, 4), 1500, 1500, 1000, "32x32_ksplit"),
    (F32, (16, 16, 4), 3140, 237, 2088, "32x48_ksplit"),     # (64x64 blocks by older costs)
    (F32, (16, 16, 1), 958, 810, 690, "32x48_ksplit"),
    (F32, (16, 16, 2), 2988, 3666, 218, "32x32_ksplit"),     # (under 1 KB of K)
    (F32, (16, 16, 2), 2048, 4096, 240, "128x128"),
    (F32, (48, 16, 4), 1030, 1050, 1301, "32x48_ksplit")])
def test_blocks_by_cost(gpu, kind, tile, m, n, k, name):
    lib, torch = gpu
    flags, tin, tout = kind
    (m0, n0, k0), tin, tout = tile, getattr(torch, tin), getattr(torch, tout)
    gen = torch.Generator(device="cuda"); gen.manual_seed(m + n)
    a, b = (torch.randint(-1, 2, (r, k), generator=gen, device="cuda").float() for r in (m, n))
    lhs, rhs = _tiles(torch, a, m0, k0).to(tin), _tiles(torch, b, n0, k0).to(tin)
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    mat = torch.full((m + 1, n), 7, device="cuda", dtype=tout)
    acc = torch.randint(-9, 9, (m1, n1, m0, n0), generator=gen, device="cuda").to(tout)
    out = acc.clone()
    torch.cuda.synchronize()
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    args = (lhs.data_ptr(), 0, k1 * m0 * k0, rhs.data_ptr(), 0, k1 * n0 * k0)
    lib.mmt4d(*args, out.data_ptr(), 0, n1 * m0 * n0, m1, n1, k1, m0, n0, k0, flags | uk.MMT4D_ACCUMULATE)
    tiled_name = lib.last_kernel_name()
    lib.mmt4d_unpack(*args, mat.data_ptr(), 0, n, m, n, m1, n1, k1, m0, n0, k0, flags)
    lib.synchronize()
    want = a @ b.T                                # whole numbers below 2^24: exact
    assert torch.equal(mat[:m], want.to(tout)) and bool((mat[m] == 7).all())
    want = torch.nn.functional.pad(want, (0, n1 * n0 - n, 0, m1 * m0 - m)).view(m1, m0, n1, n0).permute(0, 2, 1, 3)
    assert torch.equal(out, (want + acc.float()).to(tout))
    assert tiled_name == lib.last_kernel_name()
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:   # (which the costs are of)
        assert tiled_name == "mmt4d_mfma_" + name
