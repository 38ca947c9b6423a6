"""conv_nchwc on the GPU against the oracle, through the C-ABI: the reference
test's case grid (tools/conv_nchwc_test.c:187-226; random loose strides and
offsets, ACCUMULATE off/on, degenerate sizes), whole output buffer compared
including the elements between rows, with device and with host buffers."""
import numpy as np
import pytest

import conv_testing as C
import uk_testing as T
from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu


def _run_gpu(lib, torch, c, inp, flt, out0, host):
    a = c.args()
    if host:
        got = out0.copy()
        lib.conv_nchwc(inp.ctypes.data, *a["input"], flt.ctypes.data, *a["filter"],
                       got.ctypes.data, *a["output"], *a["dims"])
        return got
    d = [T.DeviceBytes(torch, x) for x in (inp, flt, out0)]
    lib.conv_nchwc(d[0].ptr, *a["input"], d[1].ptr, *a["filter"], d[2].ptr, *a["output"], *a["dims"])
    lib.synchronize()
    return d[2].numpy().view(np.float32)


def _check(lib, torch, oracle, c, ci, host, exact, mfma, atol=1e-4):
    rng = np.random.default_rng(ci)
    inp, flt, out0 = C.buffers(c, rng, exact=exact)
    want = out0.copy()
    C.run(oracle, c, inp, flt, want)
    got = _run_gpu(lib, torch, c, inp, flt, out0, host)
    if exact or not mfma:
        # Small integers: every partial sum is exact, any order gives the same
        # bits. N(0,1) on the scalar kernel: the reference's own order, with a
        # separate multiply and add.
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), c.label()
    else:
        # MFMA order on N(0,1) data: the same sum to f32 rounding. Bound: K
        # products of magnitude |x||w| summed in f32, error <= K * 2^-24 * sum
        # of magnitudes per output; 1e-4 absolute covers K = 432 here with
        # room, and everything the call must not touch is still bit-equal.
        assert np.allclose(got, want, rtol=1e-5, atol=atol), (c.label(), float(np.abs(got - want).max()))
        mask = np.ones(out0.size, bool)
        for nn in range(c.N):
            for oc in range(c.OC_outer):
                for oh in range(c.OH):
                    b = c.offsets[2] + nn * c.out_strides[0] + oc * c.out_strides[1] + oh * c.out_strides[2]
                    mask[b:b + c.OW * c.k0] = False
        assert np.array_equal(got[mask].view(np.uint32), out0[mask].view(np.uint32)), c.label()


@pytest.mark.parametrize("host", [False, True])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("mode", [uk.KERNEL_MODE_AUTO, uk.KERNEL_MODE_GENERIC])
def test_conv_reference_test_grid(gpu, oracle, host, exact, mode):
    """The reference test's grid. In AUTO mode the 16x16 tile runs on the MFMA
    kernel, everything else (and everything in GENERIC mode) on the scalar one."""
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(mode)
    try:
        for ci, c in enumerate(C.cases(seed=21)):
            mfma = mode == uk.KERNEL_MODE_AUTO and c.k0 == 16 and c.c0 % 16 == 0
            _check(lib, torch, oracle, c, ci, host, exact, mfma)
            early = (c.N == 0 or c.OC_outer == 0 or c.OH == 0 or c.OW == 0 or
                     ((c.IC_outer == 0 or c.FH == 0 or c.FW == 0) and c.flags & C.CONV_ACCUMULATE))
            if not early:
                assert lib.last_kernel_name().startswith("conv_nchwc_mfma_" if mfma else "conv_nchwc_generic")
    finally:
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)


@pytest.mark.parametrize("exact", [True, False])
def test_conv_mfma_wide_shapes(gpu, oracle, exact):
    """Shapes beyond the reference's grid for the MFMA kernel: several panels
    per row (with a partial last one), an odd number of output-channel blocks,
    c0 = 32 and 48, strides 2, loose strides and offsets, ACCUMULATE."""
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    n = 0
    for ci, c in enumerate(C.cases(seed=33, tiles=[(16, 16), (16, 32), (16, 48)],
                                   shapes=C.WIDE_SHAPES)):
        _check(lib, torch, oracle, c, 500 + ci, False, exact, True)
        assert lib.last_kernel_name().startswith("conv_nchwc_mfma_")
        n += 1
    assert n == 24


def test_conv_info_and_fallback_flag(gpu):
    """conv_nchwc.c:139-152,200-218: the info bit names the tile shapes a tuned
    kernel serves; any other shape needs the fallback flag."""
    lib, torch = gpu
    x = torch.zeros(4096, device="cuda")
    info = lib.lib.iree_uk_conv_nchwc_info
    assert info(16, 16, C.CONV_TYPE_F32F32F32, None) == 1
    assert info(16, 32, C.CONV_TYPE_F32F32F32, None) == 1
    assert info(16, 8, C.CONV_TYPE_F32F32F32, None) == 0
    assert info(8, 16, C.CONV_TYPE_F32F32F32, None) == 0
    # 16x16 without the flag: served
    lib.conv_nchwc(x.data_ptr(), 0, 256, 256, 16, x.data_ptr(), 0, 256, 256, 256, x.data_ptr(), 1024,
                   16, 16, 16, 1, 1, 1, 1, 1, 1, 1, 16, 16, 1, 1, C.CONV_TYPE_F32F32F32)
    lib.synchronize()
    with pytest.raises(uk.ContractViolation):
        lib.conv_nchwc(x.data_ptr(), 0, 1, 1, 1, x.data_ptr(), 0, 1, 1, 1, x.data_ptr(), 0, 1, 1, 1,
                       1, 1, 1, 1, 1, 1, 1, 8, 8, 1, 1, C.CONV_TYPE_F32F32F32)


@pytest.mark.parametrize("exact", [True, False])
def test_conv_few_pixels_many_channels_splits_the_input_channels(gpu, oracle, exact):
    """A late layer of an image network at batch 1 (7x7 outputs, 3x3 filter,
    512 -> 512 channels) has fewer output blocks than the device has compute
    units: IC_outer is split over several workgroups per block and a second
    kernel adds the slices up in order. Loose strides, offsets, ACCUMULATE off
    and on; the buffer for the slices shows in iree_uk_amd_workspace_bytes."""
    lib, torch = gpu
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    N, OC, OH, OW, IC, FH, FW, k0, c0 = 1, 32, 7, 7, 32, 3, 3, 16, 16
    H, W = OH + FH - 1, OW + FW - 1
    for ci, acc in enumerate((0, 1)):
        in_sh = W * c0 + 16 * ci
        in_sic = H * in_sh + 32 * ci
        f_sfh = FW * c0 * k0
        f_sic = FH * f_sfh + 256 * ci
        out_soh = OW * k0 + 16 * ci
        out_soc = OH * out_soh + 48 * ci
        c = C.ConvCase(N, OC, OH, OW, IC, FH, FW, 1, 1, k0, c0, C.CONV_TYPE_F32F32F32 | (C.CONV_ACCUMULATE if acc else 0),
                       (IC * in_sic, in_sic, in_sh), (IC * f_sic, f_sic, f_sfh), (OC * out_soc, out_soc, out_soh),
                       (4 * ci, 8 * ci, 12 * ci))
        lib.release_workspaces()
        # K = 4608 products per output here, ten times the grid's: two f32
        # summation orders of that many N(0,1) products (sums of magnitude up to
        # a few hundred) differ by a few 1e-4; the exact-data run pins the
        # indexing bit for bit.
        _check(lib, torch, oracle, c, 40 + ci, host=False, exact=exact, mfma=True, atol=2e-3)
        assert lib.last_kernel_name().startswith("conv_nchwc_mfma_")
        assert lib.workspace_bytes() > 0


# One shape (N, OC_outer, OH, OW, IC_outer, FH, FW, strides, c0) for each kernel
# and tile the MFMA launch chooses from on a device of 256 compute units, with
# ragged pixels and channel blocks; the steps of a sum leave every remainder of
# the direct kernel's register sets.
TILE_SHAPES = [
    ((16, 7, 40, 39, 3, 1, 1, 1, 1, 48), "direct_4x4"),  # 9 steps
    ((3, 7, 57, 55, 4, 2, 1, 1, 1, 16), "direct_2x4"),  # 8 steps
    ((1, 15, 56, 55, 3, 1, 3, 2, 1, 16), "direct_2x2"),  # 9 steps
    ((65, 9, 7, 7, 5, 1, 2, 1, 1, 16), "direct_1x4"),  # 10 steps
    ((65, 5, 1, 1, 7, 1, 1, 1, 2, 16), "direct_1x2"),  # 7 steps
    ((3, 3, 5, 3, 1, 1, 1, 1, 1, 16), "direct_1x1"),  # 1 step
    ((65, 25, 35, 6, 4, 1, 1, 1, 1, 32), "lds_4x4"),  # 8 steps
    ((130, 11, 17, 4, 3, 1, 3, 1, 1, 16), "lds_2x4"),  # 9 steps
    ((16, 31, 31, 33, 1, 1, 1, 1, 1, 16), "lds_1x4"),  # 1 step: sums of fewer than eight choose by costs of their own
    ((300, 7, 13, 17, 1, 1, 2, 1, 1, 16), "lds_1x4"),  # 2 steps
    ((65, 31, 1, 1, 3, 1, 1, 1, 1, 16), "lds_1x4"),
    ((300, 2, 13, 17, 1, 3, 1, 1, 2, 16), "lds_2x2"),
    ((300, 1, 13, 17, 2, 1, 1, 2, 2, 16), "lds_2x1"),
]


@pytest.mark.parametrize("shape,tile", TILE_SHAPES, ids=lambda s: s if isinstance(s, str) else "x".join(map(str, s)))
def test_conv_mfma_tiles(gpu, oracle, shape, tile):
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    for ci, c in enumerate(C.cases(seed=51, tiles=[(16, shape[9])], shapes=[shape[:9]])):
        _check(lib, torch, oracle, c, 900 + ci, host=False, exact=True, mfma=True)
        assert lib.last_kernel_name() == "conv_nchwc_mfma_" + tile


# The same for sums of more than ten steps: tiles of a wave, and tiles whose steps four
# waves, or those of two and four workgroups, divide unevenly.
LONG_SHAPES = [
    ((40, 9, 3, 22, 2, 3, 1, 1, 1, 32), "direct_1x4"),  # 12 steps
    ((40, 1, 15, 27, 3, 2, 2, 1, 1, 16), "direct_2x2"),
    ((40, 3, 29, 14, 2, 3, 1, 1, 1, 32), "direct_2x4"),
    ((1, 1, 1, 2, 5, 3, 1, 1, 1, 16), "split_1x1"),  # 15 steps
    ((5, 13, 1, 1, 5, 7, 7, 1, 1, 16), "split_1x1"),  # 245 steps, two workgroups a tile
    ((3, 1, 1, 1, 5, 5, 5, 2, 1, 16), "split_1x1"),  # 125 steps, four
    ((40, 9, 1, 1, 2, 3, 3, 1, 2, 16), "split_1x4"),
    ((16, 18, 1, 1, 3, 5, 5, 1, 1, 32), "split_1x4"),  # 150 steps, two
    ((40, 1, 8, 13, 2, 1, 3, 1, 1, 32), "split_2x2"),
]


@pytest.mark.parametrize("shape,tile", LONG_SHAPES, ids=lambda s: s if isinstance(s, str) else "x".join(map(str, s)))
def test_conv_long_sums(gpu, oracle, shape, tile):
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    for ci, c in enumerate(C.cases(seed=57, tiles=[(16, shape[9])], shapes=[shape[:9]])):
        for run in range(2):   # the second call finds the counters of the first one's workgroups
            _check(lib, torch, oracle, c, 960 + ci + 10 * run, host=False, exact=True, mfma=True)
            assert lib.last_kernel_name() == "conv_nchwc_mfma_" + tile


@pytest.mark.parametrize("flip", ["h", "ic", "oc", "fh"])
@pytest.mark.parametrize("dims", [(2, 3, 9, 11, 3, 2, 2), (40, 5, 7, 9, 2, 3, 3)])   # a split and a direct kernel
def test_conv_negative_strides(gpu, flip, dims):
    """A dimension stored back to front and walked with a negative stride: the
    result of the layer on the buffer the right way round, bit for bit."""
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    N, OC, OH, OW, IC, FH, FW = dims
    H, W = OH + FH - 1, OW + FW - 1
    g = torch.Generator(device="cuda"); g.manual_seed(9)
    x = torch.randn((N, IC, H, W * 16), generator=g, device="cuda")
    f = torch.randn((OC, IC, FH, FW * 256), generator=g, device="cuda")
    results = []
    for turned in (False, True):
        xs, fs = [IC * H * W * 16, H * W * 16, W * 16], [IC * FH * FW * 256, FH * FW * 256, FW * 256]
        xb, fb, x_off, f_off = x, f, 0, 0
        if turned and flip in ("h", "ic"):
            d = 2 if flip == "h" else 1
            xb = x.flip(d).contiguous()
            x_off, xs[d] = (x.shape[d] - 1) * xs[d], -xs[d]
        if turned and flip in ("oc", "fh"):
            d = 2 if flip == "fh" else 0
            fb = f.flip(d).contiguous()
            f_off, fs[d] = (f.shape[d] - 1) * fs[d], -fs[d]
        y = torch.zeros((N, OC, OH, OW * 16), device="cuda")
        lib.conv_nchwc(xb.data_ptr(), x_off, *xs, fb.data_ptr(), f_off, *fs, y.data_ptr(), 0, OC * OH * OW * 16,
                       OH * OW * 16, OW * 16, N, OC, OH, OW, IC, FH, FW, 16, 16, 1, 1, C.CONV_TYPE_F32F32F32)
        lib.synchronize()
        assert lib.last_kernel_name().startswith("conv_nchwc_mfma_")
        results.append(y)
    assert bool(results[0].any()) and torch.equal(results[0], results[1])


def test_conv_image_beyond_32_bit_offsets(gpu):
    """Planes of input channels 2 GiB apart: more than the direct kernel's 32-bit
    offsets reach, the LDS kernel serves the call."""
    lib, torch = gpu
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    OC, OH, OW, IC, F = 3, 6, 10, 2, 3
    H, W, plane = OH + F - 1, OW + F - 1, 1 << 29
    g = torch.Generator(device="cuda"); g.manual_seed(11)
    x = torch.randint(-3, 4, (IC, H * W * 16), generator=g, device="cuda").float()
    f = torch.randint(-3, 4, (OC * IC * F * F * 256,), generator=g, device="cuda").float()
    far = torch.empty(plane + H * W * 16, device="cuda")
    far[:H * W * 16], far[plane:] = x[0], x[1]
    results, names = [], []
    for buf, sic in ((x, H * W * 16), (far, plane)):
        y = torch.zeros(OC * OH * OW * 16, device="cuda")
        lib.conv_nchwc(buf.data_ptr(), 0, IC * sic, sic, W * 16, f.data_ptr(), 0, IC * F * F * 256, F * F * 256, F * 256,
                       y.data_ptr(), 0, OC * OH * OW * 16, OH * OW * 16, OW * 16, 1, OC, OH, OW, IC, F, F, 16, 16, 1, 1,
                       C.CONV_TYPE_F32F32F32)
        lib.synchronize()
        results.append(y)
        names.append(lib.last_kernel_name())
    assert "lds" not in names[0] and "lds" in names[1], names
    assert bool(results[0].any()) and torch.equal(results[0], results[1])


@pytest.mark.parametrize("dims,kernel", [((1, 3, 6, 10, 3), "split_wide_1x4"),       # 27 steps
                                         ((2, 33, 7, 7, 7), "split_wide_1x4"),       # 147 steps, workgroups meet
                                         ((1, 5, 60, 59, 3), "split_wide_1x4"),      # several rounds
                                         ((4, 16, 28, 28, 3), "direct_wide_2x2"),
                                         ((8, 15, 28, 27, 3), "direct_wide_2x4")])
@pytest.mark.parametrize("back", [False, True])
def test_conv_far_planes_and_few_tiles(gpu, dims, kernel, back):
    """The same with sums long enough for the split and the direct kernel with 64-bit
    addresses, the planes in order and back to front; ACCUMULATE. Equal to the layer with
    its planes side by side."""
    lib, torch = gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the tiles are chosen for 256 compute units")
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    N, OC, OH, OW, F = dims
    IC, H, W, plane = 3, OH + F - 1, OW + F - 1, 1 << 28
    size = H * W * 16
    g = torch.Generator(device="cuda"); g.manual_seed(12)
    x = torch.randint(-3, 4, (IC, N * size), generator=g, device="cuda").float()
    f = torch.randint(-3, 4, (OC * IC * F * F * 256,), generator=g, device="cuda").float()
    y0 = torch.randint(-9, 9, (N * OC * OH * OW * 16,), generator=g, device="cuda").float()
    far = torch.empty((IC - 1) * plane + N * size, device="cuda")
    for i in range(IC):
        at = (IC - 1 - i if back else i) * plane
        far[at:at + N * size] = x[i]
    results, names = [], []
    for buf, off, sic in ((x, 0, N * size), (far, (IC - 1) * plane if back else 0, -plane if back else plane)):
        for run in range(2):   # the second call finds the counters of the first one's workgroups
            y = y0.clone()
            lib.conv_nchwc(buf.data_ptr(), off, size, sic, W * 16, f.data_ptr(), 0, IC * F * F * 256, F * F * 256, F * 256,
                           y.data_ptr(), 0, OC * OH * OW * 16, OH * OW * 16, OW * 16, N, OC, OH, OW, IC, F, F, 16, 16, 1, 1,
                           C.CONV_TYPE_F32F32F32 | C.CONV_ACCUMULATE)
            lib.synchronize()
            results.append(y)
            names.append(lib.last_kernel_name())
    assert "wide" not in names[0] and names[2] == "conv_nchwc_mfma_" + kernel, names
    assert all(torch.equal(results[0], r) for r in results[1:])
