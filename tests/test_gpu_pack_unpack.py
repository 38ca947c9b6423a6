"""GPU parity of iree_uk_pack / iree_uk_unpack against the CPU oracle, through
the C-ABI. Bit-exact over the whole destination buffer (stride gaps must stay
untouched)."""
import numpy as np
import pytest

import uk_testing as T
from golden import make_golden as G
from iree_amd import ukernel as uk

pytestmark = pytest.mark.gpu

MODES = [uk.KERNEL_MODE_AUTO, uk.KERNEL_MODE_GENERIC]


@pytest.fixture(autouse=True)
def _reset_modes(lib):
    yield
    lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
    lib.set_pointer_mode(uk.POINTER_MODE_AUTO)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", range(len(G.PACK_TILES)))
def test_pack_reference_test_grid(gpu, oracle, n, mode):
    """tools/pack_test.c's grid: degenerate and small outer shapes x both
    transposes x padding variants, random strides/offsets/padding value."""
    lib, torch = gpu
    lib.set_kernel_mode(mode)
    tf, t0, t1 = G.PACK_TILES[n]
    for ci, c in enumerate(T.pack_cases(tf, t0, t1, seed=11000 + n)):
        rng = np.random.default_rng(ci)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", range(len(G.UNPACK_TILES)))
def test_unpack_reference_test_grid(gpu, oracle, n, mode):
    lib, torch = gpu
    lib.set_kernel_mode(mode)
    tf, t0, t1 = G.UNPACK_TILES[n]
    for ci, c in enumerate(T.unpack_cases(tf, t0, t1, seed=12000 + n)):
        rng = np.random.default_rng(ci)
        inp, out0 = T.make_unpack_buffers(c, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, c, inp, want)
        got = T.gpu_unpack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())


# Shapes large enough to span several workgroup blocks of the tiled kernels,
# with ragged edges, all-padding tiles, loose strides and shifted bases.
TILED_SHAPES = [
    # (type, tile0, tile1, in0, in1)
    (uk.PACK_TYPE_F16F16, 16, 16, 300, 270),
    (uk.PACK_TYPE_F16F16, 16, 16, 256, 256),
    (uk.PACK_TYPE_I8I8, 16, 32, 130, 515),
    (uk.PACK_TYPE_I8I8, 32, 8, 16, 1024),
    (uk.PACK_TYPE_I8I8, 16, 2, 200, 301),
    (uk.PACK_TYPE_I8I8, 16, 8, 257, 259),
    (uk.PACK_TYPE_F32F32, 16, 1, 259, 263),
    (uk.PACK_TYPE_F32F32, 16, 16, 100, 333),
    (uk.PACK_TYPE_I32I32, 8, 4, 77, 130),
    (uk.PACK_TYPE_BF16BF16, 16, 2, 130, 258),
    (uk.PACK_TYPE_F16F16, 1, 16, 37, 400),
    (uk.PACK_TYPE_F32F32, 3, 5, 200, 200),
    (uk.PACK_TYPE_F16F16, 6, 7, 200, 200),
]


def _tiled_pack_cases():
    g = T.Lcg(77)
    for (tf, t0, t1, in0, in1) in TILED_SHAPES:
        for ti in (0, 1):
            for to in (0, 1):
                for variant in range(3):
                    a0, a1 = (t1, t0) if ti else (t0, t1)  # extent along matrix dims
                    o0 = -(-in0 // a0) + (1 if variant == 2 else 0)
                    o1 = -(-in1 // a1) + (2 if variant == 2 else 0)
                    flags = tf | (0x100 if ti else 0) | (0x200 if to else 0)
                    os0, os1 = (o1, o0) if to else (o0, o1)
                    loose = (0, 4, 1)[variant]
                    yield T.PackCase(flags, in0, in1, os0, os1, t0, t1,
                                     in1 + (0, 8, 3)[variant], 1,
                                     os1 * t0 * t1 + loose,
                                     (0, 16, 5)[variant], (0, 32, 3)[variant], g.u64())


@pytest.mark.parametrize("mode", MODES)
def test_pack_block_spanning_shapes(gpu, oracle, mode):
    lib, torch = gpu
    lib.set_kernel_mode(mode)
    tiled = 0
    for ci, c in enumerate(_tiled_pack_cases()):
        rng = np.random.default_rng(500 + ci)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())
        tiled += lib.last_kernel_name() in ("pack_tiled", "pack_stream", "pack_direct", "pack_transposing")
    if mode == uk.KERNEL_MODE_AUTO:
        assert tiled >= 60, tiled  # the LDS-staged kernel is the one under test
    else:
        assert tiled == 0


# (MFMA_VARIANT + 1 keeps unpack on the LDS-staged kernels.)
@pytest.mark.parametrize("mode", MODES + [uk.KERNEL_MODE_MFMA_VARIANT + 1])
def test_unpack_block_spanning_shapes(gpu, oracle, mode):
    lib, torch = gpu
    lib.set_kernel_mode(mode)
    tiled = 0
    for ci, pc in enumerate(_tiled_pack_cases()):
        if pc.elem_bytes == 1:
            continue  # unpack has no 1-byte type (exported_bits.h:76)
        c = T.UnpackCase(pc.flags, pc.out_size0, pc.out_size1, pc.out_size2,
                         pc.out_size3, pc.in_size0, pc.in_size1, pc.out_stride0,
                         pc.in_stride0, 1, pc.out_offset, pc.in_offset)
        rng = np.random.default_rng(900 + ci)
        inp, out0 = T.make_unpack_buffers(c, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, c, inp, want)
        got = T.gpu_unpack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())
        tiled += lib.last_kernel_name() in ("unpack_tiled", "unpack_stream", "unpack_direct")
    if mode != uk.KERNEL_MODE_GENERIC:
        assert tiled >= 40, tiled


@pytest.mark.parametrize("tf,t0,t1", [
    (uk.PACK_TYPE_I8I8, 16, 16), (uk.PACK_TYPE_I8I8, 16, 32), (uk.PACK_TYPE_I8I8, 32, 64),
    (uk.PACK_TYPE_I8I8, 1, 128), (uk.PACK_TYPE_F16F16, 16, 16), (uk.PACK_TYPE_BF16BF16, 24, 8),
    (uk.PACK_TYPE_F32F32, 8, 4), (uk.PACK_TYPE_I32I32, 5, 16)])
def test_pack_direct_kernel_exact_untransposed_tilings(gpu, oracle, tf, t0, t1):
    """Untransposed packs of a matrix that the tiles cover exactly, tile rows of
    whole 16-byte pieces, 16-byte aligned rows: the register-to-register kernel
    (no LDS staging) serves them up to a few tens of megabytes. Whole output
    buffers against the oracle, loose pitches and offsets included, and the
    LDS-staged kernels on the same call give the same bytes."""
    lib, torch = gpu
    es = uk.PACK_TYPE_BYTES[tf]
    align = 16 // es
    for ci, (o0, o1) in enumerate(((1, 1), (3, 5), (17, 9), (40, 33), (2, 130))):
        in0, in1 = o0 * t0, o1 * t1
        c = T.PackCase(tf, in0, in1, o0, o1, t0, t1, in1 + (ci % 3) * align, 1,
                       o1 * t0 * t1 + (ci % 2) * align, (ci % 2) * align, (ci % 3) * align, 0x1234)
        rng = np.random.default_rng(7000 + ci)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert lib.last_kernel_name() == "pack_direct", (c.label(), lib.last_kernel_name())
        assert np.array_equal(got, want), c.label()
        lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 1)   # keeps pack on the LDS-staged kernels
        try:
            staged = T.gpu_pack(lib, torch, c, inp, out0)
            assert lib.last_kernel_name() in ("pack_stream", "pack_tiled"), lib.last_kernel_name()
        finally:
            lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        assert np.array_equal(staged, want), c.label()


# (type, stored tile shape out_size2 x out_size3, TRANSPOSE_INNER): element-wise
# transpositions, and untransposed tiles whose rows are one, two or four bytes
# (the reference's 16x2 s8 tile,
# arch/x86_64/mmt4d_x86_64_tiles.inl).
TRANSPOSING_TILES = [
    (uk.PACK_TYPE_F16F16, 16, 16, True), (uk.PACK_TYPE_BF16BF16, 16, 8, True), (uk.PACK_TYPE_F16F16, 16, 4, True),
    (uk.PACK_TYPE_F16F16, 64, 32, True), (uk.PACK_TYPE_F16F16, 1, 16, True), (uk.PACK_TYPE_BF16BF16, 128, 16, True),
    (uk.PACK_TYPE_I8I8, 16, 8, True), (uk.PACK_TYPE_I8I8, 16, 16, True), (uk.PACK_TYPE_I8I8, 16, 32, True),
    (uk.PACK_TYPE_I8I8, 8, 32, True), (uk.PACK_TYPE_I8I8, 256, 8, True), (uk.PACK_TYPE_I8I8, 2, 16, True),
    (uk.PACK_TYPE_I8I8, 16, 2, False), (uk.PACK_TYPE_I8I8, 8, 2, False), (uk.PACK_TYPE_I8I8, 32, 2, False),
    (uk.PACK_TYPE_I8I8, 16, 1, False), (uk.PACK_TYPE_I8I8, 8, 1, False),
    (uk.PACK_TYPE_F16F16, 16, 1, False), (uk.PACK_TYPE_BF16BF16, 4, 1, False),
    # transposed tiles less than eight bytes tall (K0 = 2 and 4 from a row-major [K][N] operand)
    (uk.PACK_TYPE_I8I8, 16, 2, True), (uk.PACK_TYPE_I8I8, 16, 4, True), (uk.PACK_TYPE_BF16BF16, 16, 2, True),
    (uk.PACK_TYPE_I8I8, 8, 2, True), (uk.PACK_TYPE_F16F16, 8, 2, True), (uk.PACK_TYPE_I8I8, 4, 4, True),
    (uk.PACK_TYPE_I8I8, 256, 2, True),
    # four-byte elements: f32 / s32 tiles one element wide, 16-bit pairs and s8 quadruples as tile rows
    # (the reference's 16x16x1 f32 and 16x16x2 bf16 tiles on x86, 8x8x4 s8 on arm64), and f32 transposed
    (uk.PACK_TYPE_F32F32, 16, 1, False), (uk.PACK_TYPE_I32I32, 8, 1, False), (uk.PACK_TYPE_F32F32, 4, 1, False),
    (uk.PACK_TYPE_F32F32, 32, 1, False), (uk.PACK_TYPE_BF16BF16, 16, 2, False), (uk.PACK_TYPE_F16F16, 8, 2, False),
    (uk.PACK_TYPE_I8I8, 16, 4, False), (uk.PACK_TYPE_I8I8, 8, 4, False),
    (uk.PACK_TYPE_F32F32, 16, 4, True), (uk.PACK_TYPE_F32F32, 8, 8, True), (uk.PACK_TYPE_I32I32, 64, 16, True), (uk.PACK_TYPE_F16F16, 8, 32, True),
]


def _transposing_cases(tf, s2, s3, ti):
    """Matrix shapes around the kernel's 32-row x 512-byte blocks: one block and
    less, several with ragged edges in both directions, tile grids larger than
    the matrix (tiles of nothing but padding), both outer orders, loose pitches
    and offsets that keep the alignment the kernel asks for (4 bytes on the
    matrix side, 16 on the tiled side)."""
    es = uk.PACK_TYPE_BYTES[tf]
    a0, a1 = (s3, s2) if ti else (s2, s3)    # tile extent along matrix rows / columns
    g = T.Lcg(1234 + s2 * 7 + s3)
    even = 1 if ti else s3                   # (whole tile rows)
    for (in0, in1, extra) in ((5, 6, 0), (32, 512 // es, 0), (67, 2 * (512 // es) + 10, 0), (200, 130, 1),
                              (129, 700, 0), (3 * 32, 3 * (512 // es), 2)):
        in1 = -(-in1 // even) * even
        for to in (0, 1):
            for variant in range(2):
                o0 = -(-in0 // a0) + extra
                o1 = -(-in1 // a1) + (extra + 1) // 2
                os0, os1 = (o1, o0) if to else (o0, o1)
                flags = tf | (0x100 if ti else 0) | (0x200 if to else 0)
                unit = 16 // es
                yield T.PackCase(flags, in0, in1, os0, os1, s2, s3,
                                 -(-in1 // 4) * 4 + (0, 4 * 3)[variant], 1,
                                 os1 * s2 * s3 + (0, unit * 3)[variant],
                                 (0, 4 * 5)[variant], (0, unit * 2)[variant], g.u64())


@pytest.mark.parametrize("tile", TRANSPOSING_TILES, ids=lambda t: f"type{t[0]}_{t[1]}x{t[2]}_{'ti' if t[3] else 'rows'}")
def test_pack_transposing_kernel(gpu, oracle, tile):
    """The kernel built on the LDS transposing reads: whole output buffers
    against the oracle, and the LDS-staged kernels on the same calls."""
    lib, torch = gpu
    tf, s2, s3, ti = tile
    for ci, c in enumerate(_transposing_cases(tf, s2, s3, ti)):
        rng = np.random.default_rng(8000 + ci)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert lib.last_kernel_name() == "pack_transposing", (c.label(), lib.last_kernel_name())
        assert np.array_equal(got, want), c.label()
        lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 1)   # keeps pack on the LDS-staged kernels
        try:
            staged = T.gpu_pack(lib, torch, c, inp, out0)
            assert lib.last_kernel_name() in ("pack_stream", "pack_tiled"), lib.last_kernel_name()
        finally:
            lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        assert np.array_equal(staged, want), c.label()


def test_pack_transposing_kernel_declines_what_it_does_not_serve(gpu, oracle):
    """Rows that are only 2-byte aligned, tile extents that are not powers of
    two, an odd number of columns under two-byte tile rows, four-byte elements
    in tiles less than 16 bytes tall: other kernels, same bytes."""
    lib, torch = gpu
    cases = [T.PackCase(uk.PACK_TYPE_F16F16 | 0x100, 70, 131, 5, 9, 16, 16, 131, 1, 9 * 256, 0, 0, 7),
             T.PackCase(uk.PACK_TYPE_I8I8 | 0x100, 70, 130, 6, 6, 24, 12, 132, 1, 6 * 288, 0, 0, 7),
             T.PackCase(uk.PACK_TYPE_I8I8, 70, 131, 5, 66, 16, 2, 132, 1, 66 * 32, 0, 0, 7),
             T.PackCase(uk.PACK_TYPE_F32F32 | 0x100, 70, 130, 35, 9, 16, 2, 132, 1, 9 * 32, 0, 0, 7),
             T.PackCase(uk.PACK_TYPE_F32F32, 70, 130, 35, 130, 2, 1, 132, 1, 130 * 2, 0, 0, 7)]
    for ci, c in enumerate(cases):
        inp, out0 = T.make_pack_buffers(c, np.random.default_rng(ci))
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert lib.last_kernel_name() != "pack_transposing", c.label()
        assert np.array_equal(got, want), c.label()


@pytest.mark.parametrize("tf,t0,t1,flags", [
    (uk.PACK_TYPE_I8I8, 16, 16, 0), (uk.PACK_TYPE_I8I8, 32, 8, 0), (uk.PACK_TYPE_I8I8, 16, 16, 0x200),
    (uk.PACK_TYPE_I8I8, 16, 2, 0), (uk.PACK_TYPE_I8I8, 16, 4, 0x200), (uk.PACK_TYPE_I8I8, 16, 16, 0x300),
    (uk.PACK_TYPE_I8I8, 16, 2, 0x300), (uk.PACK_TYPE_BF16BF16, 16, 8, 0), (uk.PACK_TYPE_BF16BF16, 24, 4, 0),
    (uk.PACK_TYPE_BF16BF16, 16, 2, 0), (uk.PACK_TYPE_BF16BF16, 16, 8, 0x300), (uk.PACK_TYPE_F32F32, 16, 4, 0),
    (uk.PACK_TYPE_F32F32, 16, 2, 0)])
def test_pack_rows_of_any_length_and_alignment(gpu, oracle, tf, t0, t1, flags):
    """Rows that start at any element and end inside a tile row, a vector of 8
    or 16 bytes, or before the first one: the direct, the transposing and the
    streaming kernel on them, whole buffers against the oracle."""
    lib, torch = gpu
    es = uk.PACK_TYPE_BYTES[tf]
    s0, s1 = (t1, t0) if flags & 0x100 else (t0, t1)
    g = T.Lcg(19)
    rng = np.random.default_rng(tf + t1)
    for ci, in1 in enumerate((1, 3, 7, 8, 9, 15, 16, 17, 31, 33, 65, 129, 257, 517, 1031)):
        in0 = int(rng.integers(1, 70))
        o0, o1 = -(-in0 // s0) + ci % 2, -(-in1 // s1) + ci % 3
        os0, os1 = (o1, o0) if flags & 0x200 else (o0, o1)
        c = T.PackCase(tf | flags, in0, in1, os0, os1, t0, t1, in1 + ci % 4, 1, os1 * t0 * t1, ci % 3,
                       16 // es * (ci % 2), g.u64())
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())
        lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 1)   # the LDS-staged kernels on the same call
        try:
            staged = T.gpu_pack(lib, torch, c, inp, out0)
        finally:
            lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        assert np.array_equal(staged, want), (c.label(), "staged")


@pytest.mark.parametrize("tf,t0,t1,flags", [
    (uk.UNPACK_TYPE_BF16BF16, 16, 16, 0), (uk.UNPACK_TYPE_F16F16, 16, 8, 0x200), (uk.UNPACK_TYPE_F32F32, 16, 16, 0),
    (uk.UNPACK_TYPE_I32I32, 16, 4, 0)])
def test_unpack_rows_of_any_length_and_alignment(gpu, oracle, tf, t0, t1, flags):
    """The same for unpack: what a row ends with is stored in pieces."""
    lib, torch = gpu
    rng = np.random.default_rng(tf)
    for ci, n in enumerate((1, 2, 3, 5, 7, 9, 15, 17, 33, 67, 131, 259, 515, 1033)):
        m = int(rng.integers(1, 70))
        o0, o1 = -(-m // t0) + ci % 2, -(-n // t1) + ci % 3
        s0, s1 = (o1, o0) if flags & 0x200 else (o0, o1)
        c = T.UnpackCase(tf | flags, s0, s1, t0, t1, m, n, s1 * t0 * t1, n + ci % 4, 1, 0, ci % 3)
        inp, out0 = T.make_unpack_buffers(c, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, c, inp, want)
        got = T.gpu_unpack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())


@pytest.mark.parametrize("in0,in1", [(0, 64), (64, 0), (0, 0), (0, 7)])
@pytest.mark.parametrize("tf,s2,s3,flags", [
    (uk.PACK_TYPE_I8I8, 16, 16, 0x100), (uk.PACK_TYPE_I8I8, 16, 2, 0x300), (uk.PACK_TYPE_I8I8, 16, 2, 0),
    (uk.PACK_TYPE_I8I8, 16, 4, 0x200), (uk.PACK_TYPE_F16F16, 16, 16, 0x300), (uk.PACK_TYPE_BF16BF16, 16, 2, 0),
    (uk.PACK_TYPE_F32F32, 16, 4, 0x100), (uk.PACK_TYPE_F32F32, 16, 1, 0x200), (uk.PACK_TYPE_F32F32, 16, 16, 0)])
def test_pack_of_an_empty_matrix_is_all_padding(gpu, oracle, tf, s2, s3, flags, in0, in1):
    """Rows or columns but no element, and no memory behind them (the source is a
    null pointer): every tile is padding, and the kernels that load
    unconditionally stay out of it."""
    lib, torch = gpu
    o0, o1 = 65, 66
    c = T.PackCase(tf | flags, in0, in1, o0, o1, s2, s3, in1, 1, o1 * s2 * s3, 0, 0, 0x1122334455667788)
    inp, out0 = T.make_pack_buffers(c, np.random.default_rng(in0 + in1))
    want = out0.copy()
    G.run_pack_case(oracle, c, inp, want)
    lib.set_pointer_mode(uk.POINTER_MODE_DEVICE)
    d_out = T.DeviceBytes(torch, out0)
    lib.pack(0, 0, c.in_stride0, 1, d_out.ptr, 0, c.out_stride0, c.out_stride1, in0, in1, o0, o1, s2, s3,
             c.padding_value, c.flags)
    lib.synchronize()
    assert np.array_equal(d_out.numpy(), want), (c.label(), lib.last_kernel_name())
    assert lib.last_kernel_name() in ("pack_tiled", "pack_generic"), lib.last_kernel_name()


@pytest.mark.parametrize("n1,kernel", [((1 << 19) + 40, "stream"), ((1 << 20) + 40, "generic")])
def test_pack_and_unpack_of_rows_in_gigabytes_of_padding(gpu, n1, kernel):
    """One row of 16 elements in tiles that pad it to just over 2^31 and 2^32
    bytes: what a piece of a tile lies beyond the row's end is a distance of more
    than 31 bits, and its position a number of more than 32. pack pads all of it,
    unpack stores the 16 elements and nothing else."""
    lib, torch = gpu
    t1, n = 2048, 16
    tiles = torch.empty(n1 * t1, dtype=torch.int16, device="cuda")
    tiles.fill_(1)
    row = torch.arange(100, 100 + n, dtype=torch.int16, device="cuda")
    lib.pack(row.data_ptr(), 0, n, 1, tiles.data_ptr(), 0, t1, t1, 1, n, n1, 1, 1, t1, 0x1234,
             uk.PACK_TYPE_F16F16 | uk.PACK_TRANSPOSE_OUTER)
    lib.synchronize()
    assert lib.last_kernel_name() == "pack_" + kernel
    assert torch.equal(tiles[:n], row)
    assert bool((tiles[n:] == 0x1234).all())
    tiles.fill_(7)
    tiles[:n] = row
    out = torch.full((1 << 20,), 3, dtype=torch.int16, device="cuda")
    lib.unpack(tiles.data_ptr(), 0, t1, t1, out.data_ptr(), 0, n, 1, n1, 1, 1, t1, 1, n,
               uk.UNPACK_TYPE_F16F16 | uk.UNPACK_TRANSPOSE_OUTER)
    lib.synchronize()
    assert lib.last_kernel_name() == "unpack_" + kernel
    assert torch.equal(out[:n], row)
    assert bool((out[n:] == 3).all())


@pytest.mark.parametrize("tf,t0,t1,flags", [
    (uk.PACK_TYPE_F32F32, 16, 4, 0), (uk.PACK_TYPE_F32F32, 8, 8, 0x200), (uk.PACK_TYPE_F32F32, 16, 1, 0x300),
    (uk.PACK_TYPE_BF16BF16, 12, 12, 0), (uk.PACK_TYPE_BF16BF16, 16, 8, 0x200), (uk.PACK_TYPE_I8I8, 12, 12, 0x200),
    (uk.PACK_TYPE_I8I8, 16, 16, 0), (uk.PACK_TYPE_F32F32, 16, 32, 0), (uk.PACK_TYPE_F32F32, 8, 2, 0x200),
    (uk.PACK_TYPE_F32F32, 8, 2, 0x300), (uk.PACK_TYPE_F32F32, 16, 8, 0x300)])
def test_narrow_matrices_take_the_tiled_kernels(gpu, oracle, tf, t0, t1, flags):
    """Rows whose tiles end below 96 bytes (up to 128 under TRANSPOSE_OUTER, there
    up to 192 in tile rows of whole 16-byte granules, 192 or 320 in transposed
    tiles; up to 48 where they are single bytes and not whole words), and the first
    ones beyond: which kernel, and its bytes."""
    lib, torch = gpu
    es = uk.PACK_TYPE_BYTES[tf]
    rng = np.random.default_rng(t0 * 100 + t1)
    tile_row = t1 * es
    for ci, cols in enumerate(sorted({c for b in (16, 33, 64, 80, 95, 96, 97, 112, 128, 129, 144, 192, 320) for c in
                                      (b // es, b // es + 1)})):
        rows = int(rng.integers(100, 300))
        padded = -(-cols // t1) * tile_row
        pitch = cols + ci % 2
        byte_rows = es == 1 and pitch % 4 != 0 and padded % 8 == 0
        if byte_rows:
            limit = 47 if flags & 0x200 else 48
        elif flags & 0x300 == 0x300 and t1 > 1:
            limit = 320 if tile_row >= 16 else 192
        elif flags & 0x200:
            limit = 192 if tile_row % 16 == 0 else 128
        else:
            limit = 95
        narrow = padded <= limit
        o0, o1 = -(-rows // t0), -(-cols // t1)
        so0, so1 = (o1, o0) if flags & 0x200 else (o0, o1)
        s2, s3 = (t1, t0) if flags & 0x100 else (t0, t1)
        c = T.PackCase(tf | flags, rows, cols, so0, so1, s2, s3, pitch, 1, so1 * s2 * s3, 0, 0, 0x0102030405060708)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        lib.set_kernel_mode(uk.KERNEL_MODE_MFMA_VARIANT + 1)   # past the direct and the transposing kernel
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), c.label()
        want_kernel = "pack_tiled" if narrow or cols * es < 16 else "pack_stream"
        assert lib.last_kernel_name() == want_kernel, (c.label(), lib.last_kernel_name())
        if es == 1:
            lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
            continue
        u = T.UnpackCase(tf | flags, so0, so1, s2, s3, rows, cols, so1 * s2 * s3, pitch, 1, 0, 0)
        inp, out0 = T.make_unpack_buffers(u, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, u, inp, want)
        got = T.gpu_unpack(lib, torch, u, inp, out0)
        assert np.array_equal(got, want), u.label()
        want_kernel = "unpack_tiled" if narrow else "unpack_stream"
        assert lib.last_kernel_name() == want_kernel, (u.label(), lib.last_kernel_name())
        lib.set_kernel_mode(uk.KERNEL_MODE_AUTO)
        got = T.gpu_unpack(lib, torch, u, inp, out0)
        assert np.array_equal(got, want), (u.label(), lib.last_kernel_name())


@pytest.mark.parametrize("tf,s2,s3,flags", [
    (uk.PACK_TYPE_BF16BF16, 16, 2, 0), (uk.PACK_TYPE_F32F32, 4, 16, 0x100), (uk.PACK_TYPE_I8I8, 8, 16, 0x300),
    (uk.PACK_TYPE_BF16BF16, 16, 16, 0x300)])
def test_narrow_matrices_stay_off_the_transposing_kernel(gpu, oracle, tf, s2, s3, flags):
    """Rows up to 64 bytes (32 where they are not whole words, 50 of half words in
    tiles that are not transposed) once the blocks of 32 rows are more than 1024, more than 512 for rows under 16 bytes: the
    transposing kernel's blocks are 512 bytes wide. Not tiles of 32 bytes along
    rows of whole words under TRANSPOSE_OUTER."""
    lib, torch = gpu
    es = uk.PACK_TYPE_BYTES[tf]
    t0, t1 = (s3, s2) if flags & 0x100 else (s2, s3)
    rng = np.random.default_rng(s2)
    for rows in (100, 32 * 512, 32 * 512 + 1, 32 * 1024, 32 * 1024 + 1):
        for cols in (15 // es, 16 // es, 32 // es, 32 // es + 1, 50 // es, 54 // es, 64 // es, 64 // es + 4):
            row_bytes = cols * es
            words = row_bytes % 4 == 0
            few = rows <= (32 * 512 if row_bytes < 16 else 32 * 1024)
            wide_tiles = flags & 0x200 and words and t1 * es >= 32
            half_words = not flags & 0x100 and row_bytes % 2 == 0
            transposing = few or wide_tiles or row_bytes > (64 if words else 50 if half_words else 32)
            o0, o1 = -(-rows // t0), -(-cols // t1)
            so0, so1 = (o1, o0) if flags & 0x200 else (o0, o1)
            c = T.PackCase(tf | flags, rows, cols, so0, so1, s2, s3, cols, 1, so1 * s2 * s3, 0, 0, 0x0102030405060708)
            inp, out0 = T.make_pack_buffers(c, rng)
            want = out0.copy()
            G.run_pack_case(oracle, c, inp, want)
            got = T.gpu_pack(lib, torch, c, inp, out0)
            assert np.array_equal(got, want), c.label()
            assert lib.last_kernel_name().startswith("pack_transposing") == transposing, (
                c.label(), lib.last_kernel_name())


@pytest.mark.parametrize("tf,t0,t1,flags,cols,narrow", [
    (uk.PACK_TYPE_BF16BF16, 16, 16, 0, 9, True), (uk.PACK_TYPE_F32F32, 16, 4, 0, 12, True),
    (uk.PACK_TYPE_F32F32, 16, 4, 0, 13, False), (uk.PACK_TYPE_I8I8, 16, 16, 0, 3, True),
    (uk.PACK_TYPE_F32F32, 16, 2, 0x200, 2, True), (uk.PACK_TYPE_BF16BF16, 16, 8, 0x200, 11, True),
    (uk.PACK_TYPE_BF16BF16, 16, 8, 0x200, 17, False), (uk.PACK_TYPE_BF16BF16, 16, 16, 0x200, 4, False),
    (uk.PACK_TYPE_F32F32, 8, 4, 0x200, 5, False)])
def test_narrow_matrices_leave_the_direct_kernel(gpu, oracle, tf, t0, t1, flags, cols, narrow):
    """Up to three pieces of 8 or 16 bytes to a row, beyond 4096 workgroups of 16
    rows; under TRANSPOSE_OUTER pieces of 8 bytes, and up to two longer ones of
    rows that are not whole words."""
    lib, torch = gpu
    for rows in (300, 16 * 4096, 16 * 4096 + 1):
        o0, o1 = -(-rows // t0), -(-cols // t1)
        so0, so1 = (o1, o0) if flags & 0x200 else (o0, o1)
        c = T.PackCase(tf | flags, rows, cols, so0, so1, t0, t1, cols, 1, so1 * t0 * t1, 0, 0, 0x0102030405060708)
        inp, out0 = T.make_pack_buffers(c, np.random.default_rng(cols))
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = T.gpu_pack(lib, torch, c, inp, out0)
        assert np.array_equal(got, want), c.label()
        assert (lib.last_kernel_name() == "pack_tiled") == (narrow and rows > 16 * 4096), (
            c.label(), lib.last_kernel_name())
        assert lib.last_kernel_name() in ("pack_direct", "pack_tiled")


@pytest.mark.parametrize("tf,t0,t1,flags,rows,cols", [
    (uk.PACK_TYPE_F16F16, 16, 16, 0x300, 1031, 8261), (uk.PACK_TYPE_I8I8, 16, 8, 0x100, 2050, 8301),
    (uk.PACK_TYPE_F32F32, 16, 4, 0x300, 2056, 2052), (uk.PACK_TYPE_I8I8, 16, 2, 0, 2050, 8302),
    (uk.PACK_TYPE_I8I8, 16, 1, 0x200, 2050, 8302), (uk.PACK_TYPE_F32F32, 16, 4, 0, 2500, 2622),
    (uk.PACK_TYPE_BF16BF16, 24, 4, 0, 3001, 4300), (uk.PACK_TYPE_I8I8, 16, 16, 0, 4001, 6300)])
def test_pack_of_tiles_that_are_stored_through(gpu, tf, t0, t1, flags, rows, cols):
    """Tiles of 12 MB and more on the transposing kernel (runs of less than 256
    bytes under TRANSPOSE_OUTER are stored as before), of 24 MB and more on the
    streaming one, ragged on both sides; against pad + reshape + transpose."""
    lib, torch = gpu
    es = uk.PACK_TYPE_BYTES[tf]
    rng = np.random.default_rng(cols)
    x = rng.integers(0, 1 << 8 * es, (rows, cols), dtype={1: np.uint8, 2: np.uint16, 4: np.uint32}[es])
    ti, to = bool(flags & 0x100), bool(flags & 0x200)
    s2, s3 = (t1, t0) if ti else (t0, t1)
    want = T.numpy_pack(x, t0, t1, ti, to, 0x5A & 0xFF)
    so0, so1 = want.shape[:2]
    assert want.nbytes >= 16 << 20
    d_in, d_out = T.DeviceBytes(torch, x), T.DeviceBytes(torch, np.zeros(want.nbytes, np.uint8))
    lib.pack(d_in.ptr, 0, cols, 1, d_out.ptr, 0, so1 * s2 * s3, s2 * s3, rows, cols, so0, so1, s2, s3, 0x5A, tf | flags)
    lib.synchronize()
    assert lib.last_kernel_name().startswith(("pack_transposing", "pack_stream")), lib.last_kernel_name()
    assert np.array_equal(d_out.numpy(), np.ascontiguousarray(want).view(np.uint8).reshape(-1))


SINGLE_LINE_TILES = [
    (uk.PACK_TYPE_F32F32, 16, 1), (uk.PACK_TYPE_F32F32, 1, 16), (uk.PACK_TYPE_I32I32, 8, 1),
    (uk.PACK_TYPE_F16F16, 1, 16), (uk.PACK_TYPE_BF16BF16, 16, 1), (uk.PACK_TYPE_I8I8, 1, 16),
    (uk.PACK_TYPE_I8I8, 16, 1), (uk.PACK_TYPE_F32F32, 1, 1), (uk.PACK_TYPE_F32F32, 1, 7),
]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("tile", SINGLE_LINE_TILES, ids=lambda t: f"type{t[0]}_{t[1]}x{t[2]}")
def test_single_row_and_single_column_tiles_under_transpose_inner(gpu, oracle, tile, mode):
    """A tile that is one row or one column holds the same bytes with and without
    TRANSPOSE_INNER, and the library takes it as the untransposed tile of the
    swapped shape (the reference's f32 16x16x1 right-hand side packed from
    [K][N], arch/x86_64/mmt4d_x86_64_tiles.inl). Pack and unpack, both outer
    orders, ragged edges, loose pitches: whole buffers against the oracle."""
    lib, torch = gpu
    lib.set_kernel_mode(mode)
    tf, s2, s3 = tile
    es = uk.PACK_TYPE_BYTES[tf]
    a0, a1 = s3, s2                       # TRANSPOSE_INNER: extents along matrix rows / columns
    g = T.Lcg(77 + 3 * s2 + s3)
    ci = 0
    for (in0, in1) in ((1, 1), (33, 70), (130, 257), (64, 512)):
        for to in (0, 1):
            for variant in range(2):
                o0, o1 = -(-in0 // a0) + variant, -(-in1 // a1)
                os0, os1 = (o1, o0) if to else (o0, o1)
                flags = tf | 0x100 | (0x200 if to else 0)
                c = T.PackCase(flags, in0, in1, os0, os1, s2, s3, in1 + (0, 5)[variant], 1,
                               os1 * s2 * s3 + (0, 3)[variant], (0, 2)[variant], (0, 9)[variant], g.u64())
                inp, out0 = T.make_pack_buffers(c, np.random.default_rng(4100 + ci))
                want = out0.copy()
                G.run_pack_case(oracle, c, inp, want)
                got = T.gpu_pack(lib, torch, c, inp, out0)
                assert np.array_equal(got, want), (c.label(), lib.last_kernel_name())
                if es > 1:                # unpack has no 1-byte type (exported_bits.h:76)
                    u = T.UnpackCase(flags, os0, os1, s2, s3, in0, in1, c.out_stride0, c.in_stride0, 1,
                                     c.out_offset, c.in_offset)
                    uin, uout0 = T.make_unpack_buffers(u, np.random.default_rng(4200 + ci))
                    uwant = uout0.copy()
                    G.run_unpack_case(oracle, u, uin, uwant)
                    ugot = T.gpu_unpack(lib, torch, u, uin, uout0)
                    assert np.array_equal(ugot, uwant), (u.label(), lib.last_kernel_name())
                ci += 1


def test_pack_unpack_round_trip_and_numpy_identity(gpu):
    """Size-independent properties at a size the oracle would be slow on:
    pack == pad+reshape+transpose, unpack(pack(x)) == x."""
    lib, torch = gpu
    rng = np.random.default_rng(1)
    for (dtype, tf, t0, t1, ti, to, shape) in (
            (np.float32, uk.PACK_TYPE_F32F32, 16, 1, False, True, (1537, 1030)),
            (np.float16, uk.PACK_TYPE_F16F16, 16, 16, False, False, (2047, 2049)),
            (np.int32, uk.PACK_TYPE_I32I32, 16, 16, True, True, (1000, 999)),
            # above 192 MB: the 64 KB-block kernels for large element-granular
            # transposes, with rows that are only 4-byte aligned and ragged edges
            (np.float32, uk.PACK_TYPE_F32F32, 16, 1, False, True, (7169, 7171)),
            # above 192 MB with whole tile rows as granules under TRANSPOSE_OUTER:
            # the 16 KB-block kernels with their non-temporal stores
            (np.float32, uk.PACK_TYPE_F32F32, 16, 16, False, True, (8192, 8192 - 16))):
        x = rng.integers(-30000, 30000, shape).astype(dtype)
        pad_val = dtype(-1)
        pad_bits = int(np.array([pad_val]).view({2: np.uint16, 4: np.uint32}[x.itemsize])[0])
        want4 = T.numpy_pack(x, t0, t1, ti, to, pad_val)
        o0, o1, o2, o3 = want4.shape
        d_x = torch.from_numpy(x).cuda()
        d_p = torch.zeros(want4.size * x.itemsize, dtype=torch.uint8, device="cuda")
        flags = tf | (0x100 if ti else 0) | (0x200 if to else 0)
        lib.pack(d_x.data_ptr(), 0, shape[1], 1, d_p.data_ptr(), 0, o1 * o2 * o3,
                 o2 * o3, shape[0], shape[1], o0, o1, o2, o3, pad_bits, flags)
        assert lib.last_kernel_name() in ("pack_stream", "pack_tiled", "pack_direct", "pack_transposing")
        got4 = d_p.cpu().numpy().view(dtype).reshape(want4.shape)
        assert np.array_equal(got4, want4)
        d_y = torch.full((x.size * x.itemsize,), 0x5A, dtype=torch.uint8, device="cuda")
        lib.unpack(d_p.data_ptr(), 0, o1 * o2 * o3, o2 * o3, d_y.data_ptr(), 0,
                   shape[1], 1, o0, o1, o2, o3, shape[0], shape[1], flags)
        assert lib.last_kernel_name() in ("unpack_stream", "unpack_tiled", "unpack_direct")
        assert np.array_equal(d_y.cpu().numpy().view(dtype).reshape(shape), x)


def test_host_pointers_are_staged(gpu, oracle):
    """Ordinary host memory works through the same entry points (staged through
    the GPU) and leaves stride gaps of the destination untouched."""
    lib, torch = gpu
    for ci, c in enumerate(T.pack_cases(uk.PACK_TYPE_F16F16, 6, 7, seed=31,
                                        outer_shapes=((3, 2), (9, 33)), max_offset=64)):
        rng = np.random.default_rng(ci)
        inp, out0 = T.make_pack_buffers(c, rng)
        want = out0.copy()
        G.run_pack_case(oracle, c, inp, want)
        got = out0.copy()
        es = c.elem_bytes
        lib.pack(inp.ctypes.data - c.in_offset * es, c.in_offset, c.in_stride0,
                 c.in_stride1, got.ctypes.data - c.out_offset * es, c.out_offset,
                 c.out_stride0, c.out_stride1, c.in_size0, c.in_size1, c.out_size0,
                 c.out_size1, c.out_size2, c.out_size3, c.padding_value, c.flags)
        assert np.array_equal(got, want), c.label()
    for ci, c in enumerate(T.unpack_cases(uk.UNPACK_TYPE_I32I32, 3, 4, seed=32,
                                          outer_shapes=((3, 2), (9, 33)), max_offset=64)):
        rng = np.random.default_rng(ci)
        inp, out0 = T.make_unpack_buffers(c, rng)
        want = out0.copy()
        G.run_unpack_case(oracle, c, inp, want)
        got = out0.copy()
        es = c.elem_bytes
        lib.unpack(inp.ctypes.data - c.in_offset * es, c.in_offset, c.in_stride0,
                   c.in_stride1, got.ctypes.data - c.out_offset * es, c.out_offset,
                   c.out_stride0, c.out_stride1, c.in_size0, c.in_size1, c.in_size2,
                   c.in_size3, c.out_size0, c.out_size1, c.flags)
        assert np.array_equal(got, want), c.label()
