"""mmt4d in 16x16 and 32x32 blocks whose waves share K (problems whose 64x64
blocks would leave compute units idle): where the choice changes, at K that ends
inside a step, for every class of tile rows, into tiled, row-major and
accumulated results. The inputs are small integers, so every order of the sums
gives the same result: equal to the product in 64 bits."""
import numpy as np
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

TYPES = {"s8": (uk.MMT4D_TYPE_S8S8S32, "int8", "int32"), "f16": (uk.MMT4D_TYPE_F16F16F32, "float16", "float32"),
         "bf16": (uk.MMT4D_TYPE_BF16BF16F32, "bfloat16", "float32"),
         "bf16bf16": (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "bfloat16", "bfloat16"),
         "f32": (uk.MMT4D_TYPE_F32F32F32, "float32", "float32"),
         "f8": (uk.MMT4D_TYPE_F8E4M3FNF8E4M3FNF32, "float8_e4m3fn", "float32")}


def _tiled(torch, rows, k, r0, k0, gen):
    """(values as float64 [rows padded][k padded], tiles [r1][k1][r0][k0]); padding zero."""
    r1, k1 = -(-rows // r0), -(-k // k0)
    v = torch.zeros(r1 * r0, k1 * k0)
    v[:rows, :k] = torch.randint(-2, 3, (rows, k), generator=gen).float()
    return v.double(), v.view(r1, r0, k1, k0).permute(0, 2, 1, 3).contiguous()


def _run(gpu, dtype, m, n, k, m0, n0, k0, seed=0):
    lib, torch = gpu
    flags, tin, tout = TYPES[dtype]
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.set_k_slices(0)
    gen = torch.Generator(); gen.manual_seed(seed)
    a, lhs = _tiled(torch, m, k, m0, k0, gen)
    b, rhs = _tiled(torch, n, k, n0, k0, gen)
    prod = a @ b.T
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    d_lhs, d_rhs = lhs.to(tin).cuda(), rhs.to(tin).cuda()
    acc0 = torch.randint(-50, 50, (m1, n1, m0, n0), generator=gen).to(tout)
    out = acc0.cuda()
    mat = torch.full((m, n), 7, dtype=tout, device="cuda")
    args = (d_lhs.data_ptr(), 0, k1 * m0 * k0, d_rhs.data_ptr(), 0, k1 * n0 * k0)
    lib.mmt4d(*args, out.data_ptr(), 0, n1 * m0 * n0, m1, n1, k1, m0, n0, k0, flags | uk.MMT4D_ACCUMULATE)
    names = [lib.last_kernel_name()]
    lib.mmt4d_unpack(*args, mat.data_ptr(), 0, n, m, n, m1, n1, k1, m0, n0, k0, flags)
    names.append(lib.last_kernel_name())
    lib.synchronize()
    want = prod.view(m1, m0, n1, n0).permute(0, 2, 1, 3) + acc0.double()
    assert torch.equal(out.cpu(), want.to(tout)), names
    assert torch.equal(mat.cpu(), prod[:m, :n].to(tout)), names
    return names


@pytest.mark.parametrize("dtype,m0,n0,k0", [("s8", 16, 16, 16), ("s8", 16, 16, 2), ("s8", 32, 16, 8), ("f16", 16, 16, 16),
                                            ("bf16", 16, 16, 2), ("bf16bf16", 16, 16, 8), ("f8", 16, 16, 16),
                                            ("f32", 16, 16, 1), ("f32", 16, 16, 4), ("f32", 8, 32, 2)])
@pytest.mark.parametrize("m,n,k,block", [(80, 70, 701, "16x16"),     # fewer blocks than units
                                         (256, 256, 513, "16x16"),   # one 16x16 block a unit, K one element over
                                         (250, 280, 1100, None),     # just over
                                         (500, 500, 1111, None)])    # 256 blocks of 32x32
def test_small_blocks_against_the_exact_product(gpu, dtype, m0, n0, k0, m, n, k, block):
    names = _run(gpu, dtype, m, n, k, m0, n0, k0, seed=m)
    if block is None:   # (16-bit and 32-bit rows of 1 KB and more)
        block = "16x16" if dtype == "f32" and m == 250 else "32x32" if dtype not in ("s8", "f8") or m == 500 else ""
    assert all(block in x for x in names), names


@pytest.mark.parametrize("k0", [1, 4])
@pytest.mark.parametrize("m,n,k", [(515, 1027, 77),      # 561 blocks of 32x32, four waves each
                                   (1500, 1480, 269),    # three rounds of 64x64: two waves a block
                                   (2900, 2950, 300)])   # three rounds of 128x128
def test_f32_blocks_against_full_rounds(gpu, k0, m, n, k):
    names = _run(gpu, "f32", m, n, k, 16, 16, k0, seed=n)
    if k0 == 1 or k >= 256:
        assert all("32x32_ksplit" in x or "32x48_ksplit" in x for x in names), names


@pytest.mark.parametrize("dtype,k0,m,n", [("f16", 16, 100, 90), ("f32", 1, 100, 90), ("bf16", 2, 100, 90),
                                          ("f32", 4, 500, 500), ("f16", 8, 500, 500),
                                          ("f16", 4, 500, 500), ("f32", 2, 500, 500), ("f32", 1, 500, 500)])  # (rows in twos)
def test_infinities_stay_in_their_row(gpu, dtype, k0, m, n):
    """K ends inside a step: what lies behind it, the first tiles of the next panel or what
    follows the last one, is infinite here and must not reach the sums."""
    lib, torch = gpu
    flags, tin, _ = TYPES[dtype]
    tin = getattr(torch, tin)
    k = 585   # (inside a step of 64 bytes in each of these tiles)
    gen = torch.Generator(); gen.manual_seed(5)
    a, lhs = _tiled(torch, m, k, 16, k0, gen)
    b, rhs = _tiled(torch, n, k, 16, k0, gen)
    want = (a @ b.T)[:m, :n].float()
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    assert k1 * k0 * tin.itemsize % 64 != 0
    whole = [torch.arange(r) // 16 % 2 == 0 for r in (m, n)]   # rows (columns) of the panels left finite
    for x in (lhs, rhs):
        x[1::2, :64] = float("inf")
    after = torch.full((64 * 16 * k0,), float("inf"), dtype=tin)
    d_lhs, d_rhs = (torch.cat([x.to(tin).reshape(-1), after]).cuda() for x in (lhs, rhs))
    mat = torch.zeros(m, n, device="cuda")
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.mmt4d_unpack(d_lhs.data_ptr(), 0, k1 * 16 * k0, d_rhs.data_ptr(), 0, k1 * 16 * k0, mat.data_ptr(), 0, n, m, n,
                     m1, n1, k1, 16, 16, k0, flags)
    lib.synchronize()
    assert "ksplit" in lib.last_kernel_name()
    got = mat.cpu()
    assert torch.equal(got[whole[0]][:, whole[1]], want[whole[0]][:, whole[1]])
    assert not torch.isfinite(got[~whole[0]]).any() and not torch.isfinite(got[:, ~whole[1]]).any()


@pytest.mark.parametrize("dtype,k0", [("s8", 2), ("s8", 4), ("bf16", 1), ("bf16", 2), ("f16", 4), ("f32", 1), ("f32", 2)])
def test_16x16_blocks_with_every_number_of_steps(gpu, dtype, k0):
    """Rows under 16 bytes: every number of steps that four and eight waves can begin and end
    with, three, four or eight in flight, in whole steps and with one tile more."""
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    flags, tin, tout = TYPES[dtype]
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    m, n, step = 100, 130, 64 // tin.itemsize
    many = [320 + s for s in range(70)] if (dtype, k0) == ("f32", 1) else []   # (20 KB and more)
    most = (max(many or [100]) + 1) * step + k0
    gen = torch.Generator(device="cuda"); gen.manual_seed(k0)
    a, b = (torch.randint(-2, 3, (r, most), generator=gen, device="cuda").float() for r in (m, n))
    for steps in list(range(1, 100)) + many:
        k = steps * step + (k0 if steps % 2 else 0)
        lhs, rhs = (torch.nn.functional.pad(x[:, :k], (0, 0, 0, -x.shape[0] % 16)).view(-1, 16, k // k0, k0)
                    .permute(0, 2, 1, 3).contiguous().to(tin) for x in (a, b))
        out = torch.zeros(m, n, device="cuda", dtype=tout)
        torch.cuda.synchronize()
        lib.mmt4d_unpack(lhs.data_ptr(), 0, 16 * k, rhs.data_ptr(), 0, 16 * k, out.data_ptr(), 0, n, m, n, lhs.shape[0],
                         rhs.shape[0], k // k0, 16, 16, k0, flags)
        lib.synchronize()
        assert "16x16_ksplit" in lib.last_kernel_name()
        assert torch.equal(out, (a[:, :k] @ b[:, :k].T).to(tout)), (k, lib.last_kernel_name())


@pytest.mark.parametrize("k0", [1, 2, 4])
@pytest.mark.parametrize("m,n", [(100, 130), (128, 1000)])   # up to one 16x16 block a unit, up to three
def test_f32_sixteen_chains_with_every_number_of_steps(gpu, k0, m, n):
    """A K of 24 KB and more in sixteen chains a wave: every number of steps that the
    chains of four and eight waves can end with, and a K that ends inside a step."""
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    flags, most = TYPES["f32"][0], 24576 // 4 + 161 * 16
    gen = torch.Generator(device="cuda"); gen.manual_seed(k0)
    a, b = (torch.randint(-2, 3, (r, most), generator=gen, device="cuda").float() for r in (m, n))
    for k in [6144 + 16 * s for s in range(0, 161, 1 if k0 == 4 else 3)] + [6148, 6156, 8000 + 4]:
        lhs, rhs = (torch.nn.functional.pad(x[:, :k], (0, 0, 0, -x.shape[0] % 16)).view(-1, 16, k // k0, k0)
                    .permute(0, 2, 1, 3).contiguous() for x in (a, b))
        out = torch.zeros(m, n, device="cuda")
        torch.cuda.synchronize()
        lib.mmt4d_unpack(lhs.data_ptr(), 0, 16 * k, rhs.data_ptr(), 0, 16 * k, out.data_ptr(), 0, n, m, n, lhs.shape[0],
                         rhs.shape[0], k // k0, 16, 16, k0, flags)
        lib.synchronize()
        assert "16x16_ksplit" in lib.last_kernel_name() or k0 == 1, lib.last_kernel_name()
        assert torch.equal(out, a[:, :k] @ b[:, :k].T), (k, lib.last_kernel_name())


@pytest.mark.parametrize("m,n,k", [(128, 128, 6144), (200, 300, 8192), (384, 384, 6144)])
def test_f32_errors_are_not_above_those_of_the_k_split(gpu, m, n, k):
    """Against 64 bits, beside the 64x64 blocks with K over four waves and up to 32
    workgroups: four parts of K instead of those had up to 4.4 times their error, sixteen
    chains in four and eight waves have 0.6 to 0.94."""
    lib, torch = gpu
    gen = torch.Generator(device="cuda"); gen.manual_seed(k)
    a, b = (torch.randn(-(-r // 16), k // 4, 16, 4, generator=gen, device="cuda") for r in (m, n))
    want = (a.double().permute(0, 2, 1, 3).reshape(-1, k) @ b.double().permute(0, 2, 1, 3).reshape(-1, k).T)[:m, :n]
    errors = []
    try:
        for mode, kernel in ((uk.KERNEL_MODE_AUTO, "16x16_ksplit"), (uk.KERNEL_MODE_MFMA_VARIANT + 6, "64x64_ksplit")):
            lib.set_kernel_mode(mode)
            out = torch.zeros(m, n, device="cuda")
            torch.cuda.synchronize()
            lib.mmt4d_unpack(a.data_ptr(), 0, k * 16, b.data_ptr(), 0, k * 16, out.data_ptr(), 0, n, m, n, a.shape[0],
                             b.shape[0], k // 4, 16, 16, 4, TYPES["f32"][0])
            assert lib.last_kernel_name().endswith(kernel)
            lib.synchronize()
            errors.append(float(((out.double() - want) ** 2).sum() / (want ** 2).sum()) ** 0.5)
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    assert errors[0] <= errors[1], errors


@pytest.mark.parametrize("k0", [2, 4, 16])
def test_operands_at_odd_addresses(gpu, k0):
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    m, n, k = 128, 208, 1040
    gen = torch.Generator(device="cuda"); gen.manual_seed(k0)
    a, b = (torch.randint(-128, 128, (r, k), generator=gen, device="cuda") for r in (m, n))
    lhs, rhs = (torch.nn.functional.pad(x.view(-1, 16, k // k0, k0).permute(0, 2, 1, 3).reshape(-1).to(torch.int8), (3, 0))
                for x in (a, b))
    out = torch.zeros(m, n, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()
    lib.mmt4d_unpack(lhs.data_ptr(), 3, 16 * k, rhs.data_ptr(), 3, 16 * k, out.data_ptr(), 0, n, m, n, m // 16, n // 16,
                     k // k0, 16, 16, k0, uk.MMT4D_TYPE_S8S8S32)
    lib.synchronize()
    assert "16x16_ksplit" in lib.last_kernel_name()
    assert torch.equal(out, (a.double() @ b.double().T).int())
