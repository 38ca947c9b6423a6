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
        assert all("32x32_ksplit" in x for x in names), names


@pytest.mark.parametrize("dtype,k0,m,n", [("f16", 16, 100, 90), ("f32", 1, 100, 90), ("bf16", 2, 100, 90),
                                          ("f32", 4, 500, 500), ("f16", 8, 500, 500)])
def test_infinities_stay_in_their_row(gpu, dtype, k0, m, n):
    """K ends inside a step: what the kernel reads in the place of the missing
    elements are the first ones of the first row, which are infinite here."""
    lib, torch = gpu
    flags, tin, _ = TYPES[dtype]
    tin = getattr(torch, tin)
    k = 601
    gen = torch.Generator(); gen.manual_seed(5)
    a, lhs = _tiled(torch, m, k, 16, k0, gen)
    b, rhs = _tiled(torch, n, k, 16, k0, gen)
    want = (a @ b.T)[:m, :n].float()
    lhs[0, 0, 0, 0] = rhs[0, 0, 0, 0] = float("inf")
    m1, n1, k1 = lhs.shape[0], rhs.shape[0], lhs.shape[1]
    d_lhs, d_rhs = lhs.to(tin).cuda(), rhs.to(tin).cuda()
    mat = torch.zeros(m, n, device="cuda")
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.mmt4d_unpack(d_lhs.data_ptr(), 0, k1 * 16 * k0, d_rhs.data_ptr(), 0, k1 * 16 * k0, mat.data_ptr(), 0, n, m, n,
                     m1, n1, k1, 16, 16, k0, flags)
    lib.synchronize()
    assert "ksplit" in lib.last_kernel_name()
    got = mat.cpu()
    assert torch.equal(got[1:, 1:], want[1:, 1:])
    assert not torch.isfinite(got[0]).any() and not torch.isfinite(got[:, 0]).any()
