"""Row-major results of problems that run as 256x256 blocks and two strips, a column
strip on the right and a row strip below what is left of it: with tiles of ten columns
the row strip ends inside a group of four columns, the rest of which are the column
strip's. Small integers: equal to the product in any order."""
import pytest

from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

TYPES = {"s8": (uk.MMT4D_TYPE_S8S8S32, "int8", "int32"), "f16": (uk.MMT4D_TYPE_F16F16F32, "float16", "float32"),
         "f16f16": (uk.MMT4D_TYPE_F16F16F16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, "float16", "float16")}
M0, N0, K0, N1 = 16, 10, 16, 376   # 18 x 16 blocks for 273 to 288 row panels, 17 x 15 without the strips


def _check(gpu, dtype, m1, k1, accumulate):
    lib, torch = gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("sizes are for 256 compute units")
    flags, tin, tout = TYPES[dtype]
    tin, tout = getattr(torch, tin), getattr(torch, tout)
    m, n = m1 * M0, N1 * N0
    gen = torch.Generator(); gen.manual_seed(m1)
    lhs = torch.randint(-2, 3, (m1, k1, M0, K0), generator=gen)
    rhs = torch.randint(-2, 3, (N1, k1, N0, K0), generator=gen)
    a = lhs.permute(0, 2, 1, 3).reshape(m, k1 * K0).float()
    b = rhs.permute(0, 2, 1, 3).reshape(n, k1 * K0).float()
    want = a @ b.T + (7 if accumulate else 0)
    d_lhs, d_rhs = lhs.to(tin).cuda(), rhs.to(tin).cuda()
    out = torch.full((m, n), 7, device="cuda", dtype=tout)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.mmt4d_unpack(d_lhs.data_ptr(), 0, k1 * M0 * K0, d_rhs.data_ptr(), 0, k1 * N0 * K0, out.data_ptr(), 0, n, m, n,
                     m1, N1, k1, M0, N0, K0, flags | (uk.MMT4D_ACCUMULATE if accumulate else 0))
    lib.synchronize()
    name, slices = lib.last_kernel_name(), lib.last_k_slices()
    assert name == "mmt4d_mfma_256x256_lds_direct"
    assert torch.equal(out.cpu(), want.to(tout)), (name, slices)
    return slices


@pytest.mark.parametrize("dtype", list(TYPES))
def test_a_row_strip_with_k_in_slices_keeps_to_its_columns(gpu, dtype):
    """80 rows against a K of 14 KB: the strip's sums meet in rows of its own width."""
    assert _check(gpu, dtype, 277, 448 * (2 if dtype == "s8" else 1), False) == 7


@pytest.mark.parametrize("dtype", list(TYPES))
@pytest.mark.parametrize("m1", [273, 277])
@pytest.mark.parametrize("accumulate", [False, True])
def test_a_row_strip_keeps_to_its_columns(gpu, dtype, m1, accumulate):
    """16 and 80 rows, a short K: the strip runs last, beside the finished column strip."""
    assert _check(gpu, dtype, m1, 5, accumulate) == 1
