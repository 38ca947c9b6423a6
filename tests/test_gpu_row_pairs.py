"""8-byte rows, and 4-byte rows of f32, loaded in twos: the blocks of two column blocks and more
that do so, thin and between thin and large; tiles of an odd number of rows, which are regrouped
to 16-byte rows and give the same; results that end at an odd column, inside a tile and inside
a two; rows and columns swapped; K split over workgroups; K in whole steps and not. Small
integers, so that every order of the sums gives the product in 64 bits."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

S8 = (uk.MMT4D_TYPE_S8S8S32, "int8", "int32", 8)
F16 = (uk.MMT4D_TYPE_F16F16F32, "float16", "float32", 4)
BF16BF16 = (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16", 4)
F32 = (uk.MMT4D_TYPE_F32F32F32, "float32", "float32", 2)
F32_4 = (uk.MMT4D_TYPE_F32F32F32, "float32", "float32", 1)


def _tiles(torch, x, m0, k0):
    rows, k = x.shape
    return (torch.nn.functional.pad(x, (0, -k % k0, 0, -rows % m0)).view(-(-rows // m0), m0, -(-k // k0), k0)
            .permute(0, 2, 1, 3).contiguous())


@pytest.mark.parametrize("kind", [S8, F16, BF16BF16, F32, F32_4], ids=["s8", "f16", "bf16bf16", "f32", "f32k1"])
@pytest.mark.parametrize("m0,n0,m,n,k", [
    (16, 16, 1, 9001, 512), (32, 16, 16, 8211, 1024), (32, 16, 33, 8195, 512), (16, 2, 20, 8205, 256),
    (16, 6, 64, 8193, 512), (16, 7, 16, 8301, 512), (16, 32, 5, 12289, 576), (16, 16, 9001, 17, 512),
    (6, 16, 8201, 33, 512), (16, 16, 64, 200, 8192), (16, 16, 300, 4096, 1000), (16, 16, 513, 2041, 1023),
    (16, 7, 513, 2041, 1023), (48, 48, 96, 4097, 2048), (16, 16, 128, 2049, 2047), (5, 10, 700, 901, 1504),
    (16, 16, 256, 256, 16384), (7, 16, 128, 2049, 2047), (7, 16, 33, 8195, 512)])
def test_row_pairs(gpu, kind, m0, n0, m, n, k):
    lib, torch = gpu
    flags, tin, tout, k0 = kind
    flags |= uk.MMT4D_ALLOW_GENERIC_FALLBACK_TILE_FUNCTION   # (odd tiles are not promised by the info query)
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    if k > 8192 and tout == torch.bfloat16:
        k = 8192
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
    lib.mmt4d_unpack(*args, mat.data_ptr(), 0, n, m, n, m1, n1, k1, m0, n0, k0, flags)
    lib.synchronize()
    want = a @ b.T                                # whole numbers below 2^24: exact
    assert torch.equal(mat[:m], want.to(tout)) and bool((mat[m] == 7).all())
    padded = torch.nn.functional.pad(want, (0, n1 * n0 - n, 0, m1 * m0 - m))
    want4 = padded.view(m1, m0, n1, n0).permute(0, 2, 1, 3)
    assert torch.equal(out, (want4 + acc.float()).to(tout)), lib.last_kernel_name()
    if tin == torch.int8:                         # the scaled store, from the accumulators above
        row = torch.rand(m, generator=gen, device="cuda") + 0.5
        col = torch.rand(n, generator=gen, device="cuda") + 0.5
        scaled = torch.full((m + 1, n), 7.0, device="cuda")
        lib.mmt4d_dequant_unpack(*args, acc.data_ptr(), 0, n1 * m0 * n0, scaled.data_ptr(), 0, n, m, n, row.data_ptr(),
                                 col.data_ptr(), m1, n1, k1, m0, n0, k0, flags | uk.MMT4D_ACCUMULATE)
        lib.synchronize()
        sums = (want4 + acc.float()).permute(0, 2, 1, 3).reshape(m1 * m0, n1 * n0)[:m, :n]
        got, exact = scaled[:m].double(), sums.double() * row.double()[:, None] * col.double()
        # Two roundings to 24 bits.
        assert bool(((got - exact).abs() <= exact.abs() * 2.0 ** -22).all()) and bool((scaled[m] == 7.0).all())


@pytest.mark.parametrize("kind", [S8, F16, F32, F32_4], ids=["s8", "f16", "f32", "f32k1"])
@pytest.mark.parametrize("m,n,k", [(5, 12289, 576), (16, 8211, 1024), (33, 8195, 512), (500, 500, 1000),
                                   (513, 2041, 1023)])
def test_row_pairs_at_odd_addresses(gpu, kind, m, n, k):
    """Rows in twos that begin at an odd byte (8-bit types) or at an odd element."""
    lib, torch = gpu
    flags, tin, tout, k0 = kind
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    gen = torch.Generator(device="cuda"); gen.manual_seed(m + n)
    a, b = (torch.randint(-1, 2, (r, k), generator=gen, device="cuda").float() for r in (m, n))
    lhs, rhs = (_tiles(torch, x, 16, k0).to(tin) for x in (a, b))
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    d_lhs, d_rhs = (torch.cat([x.new_zeros(3), x.reshape(-1)]) for x in (lhs, rhs))
    mat = torch.zeros(m, n, device="cuda", dtype=tout)
    torch.cuda.synchronize()
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.mmt4d_unpack(d_lhs.data_ptr(), 3, k1 * 16 * k0, d_rhs.data_ptr(), 3, k1 * 16 * k0, mat.data_ptr(), 0, n, m, n,
                     m1, n1, k1, 16, 16, k0, flags)
    lib.synchronize()
    assert "thin" in lib.last_kernel_name() or "ksplit" in lib.last_kernel_name(), lib.last_kernel_name()
    assert torch.equal(mat, (a @ b.T).to(tout)), lib.last_kernel_name()
