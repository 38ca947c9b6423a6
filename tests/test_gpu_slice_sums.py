"""mmt4d over 128x128 blocks with K in slices whose sums a second launch adds up:
every kind of result (tiled and accumulated, row-major, 16-bit, dequantized), ragged
rows and columns, tiles that do not divide the block, the shortest slices, and where
the choice changes. The inputs are small integers, so every order of the sums gives
the same result: equal to the product in 64 bits."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

TYPES = {"s8": (uk.MMT4D_TYPE_S8S8S32, "int8", "int32", 1), "f16": (uk.MMT4D_TYPE_F16F16F32, "float16", "float32", 2),
         "bf16": (uk.MMT4D_TYPE_BF16BF16F32, "bfloat16", "float32", 2),
         "f16f16": (uk.MMT4D_TYPE_F16F16F16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "float16", "float16", 2),
         "bf16bf16": (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16", 2),
         "f8": (uk.MMT4D_TYPE_F8E4M3FNF8E4M3FNF32, "float8_e4m3fn", "float32", 1)}
KSLICES = "mmt4d_mfma_128x128_kslices"


def _tiled(torch, rows, k, r0, k0, gen):
    """(values as float64 [rows padded][k padded], tiles [r1][k1][r0][k0]); padding zero."""
    r1, k1 = -(-rows // r0), -(-k // k0)
    v = torch.zeros(r1 * r0, k1 * k0)
    v[:rows, :k] = torch.randint(-2, 3, (rows, k), generator=gen).float()
    return v.double(), v.view(r1, r0, k1, k0).permute(0, 2, 1, 3).contiguous()


def _run(gpu, dtype, m, n, k, m0, n0, k0, mode=uk.KERNEL_MODE_AUTO, slices=0):
    """Kernel name and slice count of each call."""
    lib, torch = gpu
    flags, tin, tout, _ = TYPES[dtype]
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    gen = torch.Generator(); gen.manual_seed(m + n)
    a, lhs = _tiled(torch, m, k, m0, k0, gen)
    b, rhs = _tiled(torch, n, k, n0, k0, gen)
    prod = a @ b.T
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    d_lhs, d_rhs = lhs.to(tin).cuda(), rhs.to(tin).cuda()
    acc0 = torch.randint(-50, 50, (m1, n1, m0, n0), generator=gen).to(tout)
    out = acc0.cuda()
    pitch = n + 3   # rows of a 16-bit result that are not 8-byte aligned
    mat = torch.full((m, pitch), 7, dtype=tout, device="cuda")
    args = (d_lhs.data_ptr(), 0, k1 * m0 * k0, d_rhs.data_ptr(), 0, k1 * n0 * k0)
    names = []
    lib.set_kernel_mode(mode)
    lib.set_k_slices(slices)
    try:
        lib.mmt4d(*args, out.data_ptr(), 0, n1 * m0 * n0, m1, n1, k1, m0, n0, k0, flags | uk.MMT4D_ACCUMULATE)
        names.append((lib.last_kernel_name(), lib.last_k_slices()))
        lib.mmt4d_unpack(*args, mat.data_ptr(), 0, pitch, m, n, m1, n1, k1, m0, n0, k0, flags)
        names.append((lib.last_kernel_name(), lib.last_k_slices()))
        deq = None
        if dtype == "s8":
            deq = torch.full((m, n), -1.0, device="cuda")
            rs, cs = torch.rand(m, generator=gen), torch.rand(n, generator=gen)
            d_acc, d_rs, d_cs = acc0.cuda(), rs.cuda(), cs.cuda()
            lib.mmt4d_dequant_unpack(*args, d_acc.data_ptr(), 0, n1 * m0 * n0, deq.data_ptr(), 0, n, m, n,
                                     d_rs.data_ptr(), d_cs.data_ptr(), m1, n1, k1, m0, n0, k0,
                                     flags | uk.MMT4D_ACCUMULATE)
            names.append((lib.last_kernel_name(), lib.last_k_slices()))
        lib.synchronize()
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        lib.set_k_slices(0)
    want = prod.view(m1, m0, n1, n0).permute(0, 2, 1, 3) + acc0.double()
    assert torch.equal(out.cpu(), want.to(tout)), names
    assert torch.equal(mat[:, :n].cpu(), prod[:m, :n].to(tout)), names
    assert (mat[:, n:] == 7).all()
    if deq is not None:
        rows = want.permute(0, 2, 1, 3).reshape(m1 * m0, n1 * n0)[:m, :n].float()
        assert torch.equal(deq.cpu(), rows * rs[:, None] * cs[None, :]), names
    return names


@pytest.mark.parametrize("dtype,m0,n0,k0", [("s8", 16, 16, 16), ("s8", 32, 16, 8), ("f16", 16, 16, 16), ("bf16", 16, 16, 8),
                                            ("bf16", 16, 16, 4), ("f16f16", 16, 16, 8), ("bf16bf16", 16, 16, 8),
                                            ("f8", 16, 16, 32), ("f8", 16, 16, 16), ("f16", 24, 10, 8), ("bf16bf16", 8, 7, 8),
                                            ("s8", 1, 16, 64)])
@pytest.mark.parametrize("m,n,slices,extra", [(65, 129, 2, 0),      # the shortest slices; mostly padding
                                              (200, 300, 3, 5),     # slices of unequal length, odd columns
                                              (128, 256, 16, 16)])  # more workgroups than there are XCDs
def test_slices_against_the_exact_product(gpu, dtype, m0, n0, k0, m, n, slices, extra):
    elem = TYPES[dtype][3]
    step = (128 if dtype == "f8" else 64) // elem
    k = step * (16 * slices + extra)
    for name, got in _run(gpu, dtype, m, n, k, m0, n0, k0, uk.KERNEL_MODE_MFMA_VARIANT + 21, slices):
        assert (name, got) == (KSLICES, slices)


@pytest.mark.parametrize("dtype,k0,m,n,k,slices", [
    ("bf16bf16", 8, 200, 4096, 8192, 4),    # 64 blocks of 128x128
    ("s8", 16, 257, 2048, 14336, 5),        # 48
    ("f16", 16, 384, 4096, 4096, 2),
    ("f16", 16, 200, 4096, 8200, 0),        # K ends inside a step
    ("f16", 16, 130, 1000, 4096, 0),        # shorter in 32x32 blocks
    ("s8", 16, 384, 4096, 4096, 0)])        # K too short
def test_where_slices_are_chosen(gpu, dtype, k0, m, n, k, slices):
    names = _run(gpu, dtype, m, n, k, 16, 16, k0)
    assert all((name == KSLICES) == (slices > 0) for name, _ in names), names
    assert slices == 0 or all(got == slices for _, got in names), names


def test_too_many_slices_run_unsliced(gpu):
    for name, _ in _run(gpu, "f16", 130, 200, 1024, 16, 16, 16, uk.KERNEL_MODE_MFMA_VARIANT + 21, 3):
        assert name != KSLICES


def test_no_workspace_runs_without_slices(gpu):
    """Calls that may not allocate, and calls under capture: the blocks in place."""
    lib, torch = gpu
    m, n, k, k0 = 200, 4096, 8192, 16
    gen = torch.Generator(); gen.manual_seed(3)
    a, lhs = _tiled(torch, m, k, 16, k0, gen)
    b, rhs = _tiled(torch, n, k, 16, k0, gen)
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    d_lhs, d_rhs = lhs.half().cuda(), rhs.half().cuda()
    want = (a @ b.T).float().view(m1, 16, n1, 16).permute(0, 2, 1, 3)
    out = torch.zeros(m1, n1, 16, 16, device="cuda")
    args = (d_lhs.data_ptr(), 0, k1 * 16 * k0, d_rhs.data_ptr(), 0, k1 * 16 * k0, out.data_ptr(), 0, n1 * 256, m1, n1, k1,
            16, 16, k0, uk.MMT4D_TYPE_F16F16F32)
    torch.cuda.synchronize()
    lib.mmt4d_no_alloc(*args)
    assert lib.last_kernel_name() != KSLICES
    lib.synchronize()
    assert torch.equal(out.cpu(), want)
    stream = torch.cuda.Stream()
    lib.set_pointer_mode(uk.POINTER_MODE_DEVICE)
    lib.set_stream(stream.cuda_stream)
    try:
        lib.mmt4d(*args)
        assert lib.last_kernel_name() == KSLICES
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            lib.mmt4d(*args)
            assert lib.last_kernel_name() != KSLICES
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out.cpu(), want)
            out.zero_()
            torch.cuda.synchronize()
            lib.mmt4d(*args)
            stream.synchronize()
            assert torch.equal(out.cpu(), want)
    finally:
        lib.set_stream(None)
        lib.set_pointer_mode(uk.POINTER_MODE_AUTO)


@pytest.mark.parametrize("dtype,m,n,k", [("f16", 128, 1024, 12288), ("bf16", 384, 384, 12288), ("bf16", 512, 256, 13312),
                                         ("f16", 65, 1024, 14336), ("f16", 128, 1024, 16384)])
def test_errors_are_not_above_those_of_the_blocks_in_place(gpu, dtype, m, n, k):
    """Against 64 bits, beside the 64x64 blocks with K over four waves and seven or eight
    workgroups. Fewer parts of K or one chain of 16 slices had 1.03 to 1.14 times their
    error, the slices taken now have 0.95 to 1.00; two estimates from 130000 results
    differ by half a percent."""
    lib, torch = gpu
    flags, tin, _, _ = TYPES[dtype]
    gen = torch.Generator(); gen.manual_seed(k)
    a, b = (torch.randn(-(-r // 16), k // 8, 16, 8, generator=gen).to(getattr(torch, tin)).cuda() for r in (m, n))
    want = (a.double().permute(0, 2, 1, 3).reshape(-1, k) @ b.double().permute(0, 2, 1, 3).reshape(-1, k).T)[:m]
    errors = []
    try:
        for mode in (uk.KERNEL_MODE_AUTO, uk.KERNEL_MODE_MFMA_VARIANT + 6):
            lib.set_kernel_mode(mode)
            out = torch.zeros(m, n, device="cuda")
            torch.cuda.synchronize()
            lib.mmt4d_unpack(a.data_ptr(), 0, k * 16, b.data_ptr(), 0, k * 16, out.data_ptr(), 0, n, m, n, a.shape[0],
                             b.shape[0], k // 8, 16, 16, 8, flags)
            assert lib.last_kernel_name() == ("mmt4d_mfma_64x64_ksplit" if errors else KSLICES)
            lib.synchronize()
            errors.append(float(((out.double() - want) ** 2).sum() / (want ** 2).sum()) ** 0.5)
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    assert errors[0] <= 1.02 * errors[1], errors
