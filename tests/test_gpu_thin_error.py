"""Rounding errors of decode calls with few columns: no larger than with K in the parts
that four waves in up to eight workgroups would sum, each part a chain of roundings,
the waves' sums and then the workgroups' added in order. The same chains on the CPU
give the bound. A matrix instruction rounds after `unit` products (f32: every one;
16-bit floats, whose products it sums in groups first: fitted to calls whose parts are
known, 0.2 to 4 % off). Eight parts where there were 12 to 32 had 1.2 to 1.85 times the
error; the bound leaves 8 %."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

TYPES = {"f16": (uk.MMT4D_TYPE_F16F16F32, "float16", 2, 8), "bf16": (uk.MMT4D_TYPE_BF16BF16F32, "bfloat16", 2, 8),
         "f32": (uk.MMT4D_TYPE_F32F32F32, "float32", 4, 1)}


def _error(got, want):
    return float(((got.double() - want) ** 2).sum() / (want ** 2).sum()) ** 0.5


def _chains(torch, a, b, unit, step, waves, groups):
    parts = waves * groups
    sums = torch.zeros(parts, a.shape[0], b.shape[0])
    for s in range(a.shape[1] // step):
        for k in range(s * step, (s + 1) * step, unit):
            p = a[:, k:k + unit] @ b[:, k:k + unit].T
            sums[s % parts] = (sums[s % parts].double() + p).float()
    out = torch.zeros(a.shape[0], b.shape[0])
    for group in sums.view(groups, waves, *out.shape):
        part = group[0].clone()
        for w in group[1:]:
            part += w
        out += part
    return out


@pytest.mark.parametrize("dtype,rows,cols,k,groups", [
    ("f16", 32, 512, 4096, 8), ("f16", 4, 1024, 2048, 4), ("f16", 64, 1200, 2048, 3), ("bf16", 24, 320, 4096, 8),
    ("f32", 16, 640, 2048, 6), ("f32", 64, 512, 2048, 8)])
@pytest.mark.parametrize("swapped", [False, True])
def test_error_of_few_columns(gpu, dtype, rows, cols, k, groups, swapped):
    lib, torch = gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the parts are for 256 compute units")
    flags, t, elem, unit = TYPES[dtype]
    k0 = 16 // elem
    gen = torch.Generator(); gen.manual_seed(k + cols)
    a, b = (torch.randn(r, k, generator=gen).to(getattr(torch, t)) for r in (rows, cols))
    lhs, rhs = (torch.nn.functional.pad(x.float(), (0, 0, 0, -x.shape[0] % 16)).view(-1, 16, k // k0, k0)
                .permute(0, 2, 1, 3).contiguous().to(x.dtype).cuda() for x in ((b, a) if swapped else (a, b)))
    m, n = (cols, rows) if swapped else (rows, cols)
    out = torch.zeros(m, n, device="cuda")
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.mmt4d_unpack(lhs.data_ptr(), 0, 16 * k, rhs.data_ptr(), 0, 16 * k, out.data_ptr(), 0, n, m, n, -(-m // 16),
                     -(-n // 16), k // k0, 16, 16, k0, flags)
    lib.synchronize()
    assert lib.last_kernel_name().startswith("mmt4d_mfma_thin"), lib.last_kernel_name()
    got = out.cpu().T if swapped else out.cpu()
    a, b = a.double(), b.double()
    want = a @ b.T
    bound = 1.08 * _error(_chains(torch, a, b, unit, 64 // elem, 4, groups), want)
    assert _error(got, want) <= bound, (_error(got, want), bound)


@pytest.mark.parametrize("flags,t,tout,k0", [
    (uk.MMT4D_TYPE_F16F16F32, "float16", "float32", 8), (uk.MMT4D_TYPE_F32F32F32, "float32", "float32", 4),
    (uk.MMT4D_TYPE_F32F32F32, "float32", "float32", 2),
    (uk.MMT4D_TYPE_F16F16F16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "float16", "float16", 8),
    (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16", 4)])
@pytest.mark.parametrize("rows", [16, 48])
def test_the_last_products_of_every_chain_count(gpu, flags, t, tout, k0, rows):
    """Every number of steps a wave's chains end with, on small integers: equal to the
    product. (The matrix instructions' results were read a few cycles early where control
    flow lay in between.)"""
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    cols, t, tout = (512 if rows == 16 else 4000), getattr(torch, t), getattr(torch, tout)
    step = 64 // t.itemsize
    gen = torch.Generator(device="cuda"); gen.manual_seed(rows)
    a, b = (torch.randint(-2, 3, (r, 104 * step), generator=gen, device="cuda") for r in (rows, cols))
    for steps in range(9, 105):
        k = steps * step
        lhs, rhs = (x[:, :k].view(-1, 16, k // k0, k0).permute(0, 2, 1, 3).contiguous().to(t) for x in (a, b))
        out = torch.zeros(rows, cols, device="cuda", dtype=tout)
        torch.cuda.synchronize()
        lib.mmt4d_unpack(lhs.data_ptr(), 0, 16 * k, rhs.data_ptr(), 0, 16 * k, out.data_ptr(), 0, cols, rows, cols,
                         rows // 16, cols // 16, k // k0, 16, 16, k0, flags)
        lib.synchronize()
        want = (a[:, :k].float() @ b[:, :k].float().T).to(tout)
        assert torch.equal(out, want), (steps, lib.last_kernel_name())


# No more than that of 64x64 blocks whose four waves share K: other blocks with four waves have
# the same chains, 48x48 blocks, with eight, 0.56 of it. 8-bit floats, whose matrix instructions round
# to 1.5e-5 however K is divided, also in one chain and in slices: at most 1.000003 of it measured.
@pytest.mark.parametrize("dtype,k0,m,n,k,block", [
    ("f16", 8, 97, 2406, 7048, "32x32_ksplit"), ("f16", 8, 300, 1500, 1504, "32x64_ksplit"),
    ("f16", 8, 200, 4096, 2048, "64x64_ksplit"), ("f16", 4, 300, 1500, 1500, "32x64_ksplit"),
    ("f16", 4, 300, 4096, 1000, "32x64_ksplit"), ("bf16", 8, 700, 900, 1504, "64x64_ksplit"),
    ("f16", 8, 1100, 1200, 112, "32x32_ksplit"), ("bf16", 8, 716, 2957, 128, "32x32_ksplit"),
    ("f32", 4, 515, 1027, 768, "48x48_ksplit"), ("f32", 4, 3140, 237, 2088, "32x48_ksplit"),
    ("f32", 2, 2173, 674, 3168, "32x48_ksplit"), ("f32", 4, 1564, 1150, 2624, "64x64_ksplit"),
    ("f8", 16, 687, 2008, 1280, "32x64_ksplit"), ("f8", 16, 2153, 1308, 3840, "64x64_rhs_direct"),
    ("f8", 16, 508, 1287, 8192, ""), ("f8", 16, 1500, 700, 16384, "")])
def test_error_of_blocks_chosen_by_cost(gpu, dtype, k0, m, n, k, block):
    lib, torch = gpu
    flags, t = (uk.MMT4D_TYPE_F8E4M3FNF8E4M3FNF32, torch.float8_e4m3fn) if dtype == "f8" else \
        (TYPES[dtype][0], getattr(torch, TYPES[dtype][1]))
    gen = torch.Generator(device="cuda"); gen.manual_seed(m + k)
    a, b = ((torch.randn(r, k, generator=gen, device="cuda") * (60 if dtype == "f8" else 1)).clamp(-448, 448).to(t)
            for r in (m, n))
    lhs, rhs = (torch.nn.functional.pad(x.float(), (0, 0, 0, -x.shape[0] % 16)).view(-1, 16, k // k0, k0)
                .permute(0, 2, 1, 3).contiguous().to(t) for x in (a, b))
    want = a.double() @ b.double().T
    errors = []
    try:
        for mode in (uk.KERNEL_MODE_AUTO, uk.KERNEL_MODE_MFMA_VARIANT + 6):
            lib.set_kernel_mode(mode)
            out = torch.zeros(m, n, device="cuda")
            torch.cuda.synchronize()
            lib.mmt4d_unpack(lhs.data_ptr(), 0, 16 * k, rhs.data_ptr(), 0, 16 * k, out.data_ptr(), 0, n, m, n,
                             lhs.shape[0], rhs.shape[0], k // k0, 16, 16, k0, flags)
            lib.synchronize()
            if mode == uk.KERNEL_MODE_AUTO and torch.cuda.get_device_properties(0).multi_processor_count == 256:
                assert lib.last_kernel_name().endswith(block), lib.last_kernel_name()
            if mode != uk.KERNEL_MODE_AUTO:
                assert lib.last_kernel_name() == "mmt4d_mfma_64x64_ksplit"
            errors.append(_error(out, want))
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    assert errors[0] <= (1.0001 if dtype == "f8" else 1.0) * errors[1], errors
