"""Which blocks f32 products of few rounds take, and K slices whose workgroups do not divide
evenly over the XCDs."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

F16 = (uk.MMT4D_TYPE_F16F16F32, "float16", "float32")

F32 = (uk.MMT4D_TYPE_F32F32F32, "float32", "float32")


def _tiles(torch, x, m0, k0):
    rows, k = x.shape
    return (torch.nn.functional.pad(x, (0, -k % k0, 0, -rows % m0)).view(-(-rows // m0), m0, -(-k // k0), k0)
            .permute(0, 2, 1, 3).contiguous())


def _run(lib, torch, kind, a, b, m0, n0, k0):
    flags, t, tout = kind
    lhs, rhs = (_tiles(torch, x.float(), r0, k0).to(getattr(torch, t)) for x, r0 in ((a, m0), (b, n0)))
    m, n, k1 = a.shape[0], b.shape[0], lhs.shape[1]
    out = torch.zeros(m, n, device="cuda", dtype=getattr(torch, tout))
    torch.cuda.synchronize()
    lib.mmt4d_unpack(lhs.data_ptr(), 0, k1 * m0 * k0, rhs.data_ptr(), 0, k1 * n0 * k0, out.data_ptr(), 0, n, m, n,
                     lhs.shape[0], rhs.shape[0], k1, m0, n0, k0, flags)
    lib.synchronize()
    return out


def _small(torch, rows, k, seed):
    gen = torch.Generator(device="cuda"); gen.manual_seed(seed)
    return torch.randint(-2, 3, (rows, k), generator=gen, device="cuda")


@pytest.mark.parametrize("kind,tile,m,n,k,name", [
    (F32, (16, 16, 4), 41, 12664, 855, "32x32_ksplit"),            # else 32x64 blocks
    (F32, (16, 16, 1), 1879, 1045, 431, "64x64_deep")])
def test_which_blocks(gpu, kind, tile, m, n, k, name):
    lib, torch = gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rules count 256 compute units")
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    a, b = _small(torch, m, k, 1), _small(torch, n, k, 2)
    out = _run(lib, torch, kind, a, b, *tile)
    assert lib.last_kernel_name() == "mmt4d_mfma_" + name
    want = (a.float() @ b.float().T).to(out.dtype)   # whole numbers below 2^24: exact
    assert torch.equal(out, want)


@pytest.mark.parametrize("m,n,slices", [(292, 768, 14), (292, 768, 13), (140, 200, 3), (130, 640, 5), (100, 128, 7)])
def test_slices_that_the_xcds_cannot_share_evenly(gpu, m, n, slices):
    lib, torch = gpu
    k = 32 * 16 * slices + 96
    a, b = _small(torch, m, k, 5), _small(torch, n, k, 6)
    lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 21)
    lib.set_k_slices(slices)
    try:
        out = _run(lib, torch, F16, a, b, 16, 16, 8)
        assert lib.last_k_slices() == slices
    finally:
        lib.set_k_slices(0)
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    assert torch.equal(out, a.float() @ b.float().T)
