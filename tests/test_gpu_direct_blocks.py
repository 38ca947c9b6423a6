"""64x64 blocks with the right-hand side straight to registers in the place of a K split
over waves: which calls take them, K in four parts one after the other (its ends, its
errors), and K slices whose workgroups do not divide evenly over the XCDs."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

F16 = (uk.MMT4D_TYPE_F16F16F32, "float16", "float32")
BF16 = (uk.MMT4D_TYPE_BF16BF16F32, "bfloat16", "float32")
BF16BF16 = (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16")
S8 = (uk.MMT4D_TYPE_S8S8S32, "int8", "int32")
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
    (F16, (16, 16, 16), 2575, 394, 3273, "64x64_rhs_direct"),      # 287 blocks, K ends inside a step
    (F16, (16, 16, 8), 1024, 1024, 3200, "64x64_ksplit"),          # one block a unit
    (F16, (16, 16, 8), 1040, 1024, 3200, "64x64_rhs_direct"),
    (F16, (16, 16, 8), 1040, 2048, 4096, "64x64_ksplit"),          # 8 KB in whole steps
    (BF16BF16, (16, 16, 8), 768, 1024, 3200, "64x64_ksplit"),      # 3/4 of a block a unit
    (BF16BF16, (16, 16, 8), 784, 1024, 3200, "64x64_rhs_direct"),
    (S8, (16, 16, 16), 2898, 418, 7936, "64x64_rhs_direct"),
    (S8, (32, 16, 8), 1083, 950, 16353, "64x64_lds_direct"),
    (F32, (16, 16, 4), 41, 12664, 855, "32x32_ksplit"),            # else 32x64 blocks
    (F32, (16, 16, 1), 1879, 1045, 431, "32x32_ksplit")])
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


@pytest.mark.parametrize("kind", [F16, BF16, BF16BF16])
def test_every_step_of_the_parts_counts(gpu, kind):
    """Numbers of steps around the first that are summed in parts (96) and around a multiple
    of 12, whole steps and a K that ends inside one: equal to the product."""
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 3)
    try:
        a, b = _small(torch, 70, 133 * 32, 3), _small(torch, 130, 133 * 32, 4)
        for steps in (1, 2, 94, 95, 96, 97, 98, 99, 107, 108, 109, 131, 132):
            for more in (0, 8):
                k = steps * 32 + more
                out = _run(lib, torch, kind, a[:, :k], b[:, :k], 16, 16, 8)
                assert lib.last_kernel_name() == "mmt4d_mfma_64x64_rhs_direct"
                assert torch.equal(out, (a[:, :k].float() @ b[:, :k].float().T).to(out.dtype)), (steps, more)
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)


@pytest.mark.parametrize("kind", [F16, BF16])
@pytest.mark.parametrize("k", [3264, 3280, 4008])
def test_error_of_the_parts(gpu, kind, k):
    """No larger than that of four chains of sums over a quarter of K each, which four waves
    that share K have, added in order: the same chains on the CPU, rounded after every eight
    products (16-bit floats are summed in groups), give the bound, 8 % are left for what is
    fitted in that number. One chain over all of K has twice the error."""
    lib, torch = gpu
    gen = torch.Generator(); gen.manual_seed(k)
    a, b = (torch.randn(r, k, generator=gen).to(getattr(torch, kind[1])) for r in (96, 128))
    lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 3)
    try:
        got = _run(lib, torch, kind, a.cuda(), b.cuda(), 16, 16, 8).cpu()
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    a, b = a.double(), b.double()
    want = a @ b.T
    model = torch.zeros(96, 128)
    ends = [k * i // 32 // 8 * 8 for i in (0, 8, 16, 24, 32)]
    for lo, hi in zip(ends, ends[1:]):
        part = torch.zeros(96, 128)
        for i in range(lo, hi, 8):
            part = (part.double() + a[:, i:i + 8] @ b[:, i:i + 8].T).float()
        model += part
    error = lambda x: float(((x.double() - want) ** 2).sum() / (want ** 2).sum()) ** 0.5  # noqa: E731
    assert error(got) <= 1.08 * error(model), (error(got), error(model))


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
