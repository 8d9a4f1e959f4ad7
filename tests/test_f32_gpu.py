"""GPU parity of the FP32 matrix-core products against numpy.

Inputs are small whole numbers, so that every product and sum is exact in
FP32 (|sum| <= 18 k < 2^24 for k < 2^19): the results must equal numpy's,
whatever the tile, the stages and the splits over k.
"""
import numpy as np
import pytest

from qflex_amd import capi

pytestmark = pytest.mark.gpu

# Edges and remainders of the tiles (128 x 64, 64 x 32, 128 x 16, 32 x 64,
# 32 x 16), of their stages (16, 32, 64 k) and of the splits.
SHAPES = [(2, 2, 17), (9, 17, 64), (33, 15, 65), (31, 65, 100), (32, 64, 1000), (127, 63, 47),
          (129, 130, 33), (65, 2, 4097), (257, 255, 1001), (20, 707, 18), (1000, 1000, 17),
          (40000, 3, 40), (33000, 17, 31), (4097, 515, 50), (3, 5000, 129), (64, 64, 100003)]


def whole(rng, shape):
    return (rng.integers(-3, 4, shape) + 1j * rng.integers(-3, 4, shape)).astype(np.complex64)


def product(a, b):
    return (a.astype(np.complex128) @ b.astype(np.complex128)).astype(np.complex64)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_f32_products_exact_on_whole_numbers(ctx, m, n, k):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a, b = whole(rng, (m, k)), whole(rng, (k, n))
    A = ctx.upload(np.concatenate([[0], a.ravel()]).astype(np.complex64))  # 8-byte operands
    B, C = ctx.upload(b), ctx.alloc((m * n + 1) * 8)
    ctx.zero(C)

    class At8:
        ptr = A.ptr + 8
    ctx.cgemm(capi.FP32, m, n, k, At8, B, C)
    got = ctx.download(C, np.complex64, (m * n + 1,))
    assert np.array_equal(got[:-1].reshape(m, n), product(a, b))
    assert got[-1] == 0  # nothing past the end
    for buf in (A, B, C):
        buf.free()


def test_f32_products_keep_infinities_in_their_rows_and_columns(ctx):
    """k that fills no stage: what pads it must not meet an operand's infinity."""
    m, n, k = 40, 20, 21
    rng = np.random.default_rng(3)
    a, b = whole(rng, (m, k)), whole(rng, (k, n))
    want = product(a, b)
    a[7, 20] = np.inf
    b[20, 11] = np.inf
    A, B, C = ctx.upload(a), ctx.upload(b), ctx.alloc(m * n * 8)
    ctx.cgemm(capi.FP32, m, n, k, A, B, C)
    got = ctx.download(C, np.complex64, (m, n))
    other = np.ones((m, n), bool)
    other[7], other[:, 11] = False, False
    assert np.array_equal(got[other], want[other])
    assert not np.isfinite(got[~other]).any()
    for buf in (A, B, C):
        buf.free()


# (dims of A, its row axes, its k axes): k contiguous, rows contiguous, and
# neither; sizes below a tile and a stage and several stages.
MAPS = [([4, 16, 32], [0, 1], [2]), ([2, 64, 16], [2], [0, 1]), ([16, 2, 32, 8], [1, 3], [0, 2]),
        ([64, 1024], [0], [1]), ([4096, 16], [1], [0]), ([8, 128, 2, 16], [0, 2], [1, 3])]


@pytest.mark.parametrize("n", [2, 16, 32])
@pytest.mark.parametrize("dims,rows,cols", MAPS)
def test_f32_small_mapped_products_exact(ctx, dims, rows, cols, n):
    m, k = (int(np.prod([dims[x] for x in axes])) for axes in (rows, cols))
    rng = np.random.default_rng(m + n + k)
    a, b = whole(rng, dims), whole(rng, (n, k))  # B stored along k
    A, B, C = ctx.upload(a), ctx.upload(b), ctx.alloc(m * n * 8)
    done = ctx.cgemm_mapped(capi.FP32, A, capi.index_map(dims, rows), capi.index_map(dims, cols), B,
                            capi.index_map([n, k], [1]), capi.index_map([n, k], [0]), C)
    assert done
    want = product(a.transpose(rows + cols).reshape(m, k), b.T)
    assert np.array_equal(ctx.download(C, np.complex64, (m, n)), want)
    for buf in (A, B, C):
        buf.free()


def test_f32_rows_beyond_32_bit_offsets(ctx):
    """32 rows of 2^23 elements are 2 GiB: the 64-bit form."""
    m, n, k = 9, 2, (1 << 23) + 5
    rng = np.random.default_rng(1)
    a, b = np.zeros((m, k), np.complex64), np.zeros((k, n), np.complex64)
    pick = np.r_[0:1000, k - 1000:k]
    a[:, pick], b[pick] = whole(rng, (m, 2000)), whole(rng, (2000, n))
    A, B, C = ctx.upload(a), ctx.upload(b), ctx.alloc(m * n * 8)
    ctx.cgemm(capi.FP32, m, n, k, A, B, C)
    assert np.array_equal(ctx.download(C, np.complex64, (m, n)), product(a[:, pick], b[pick]))
    for buf in (A, B, C):
        buf.free()


def test_f32_map_beyond_32_bit_offsets(ctx):
    """A digit of A's rows at stride 2^28 elements (2 GiB)."""
    m, n, k = 16, 8, 64
    rng = np.random.default_rng(2)
    a, b = whole(rng, (m, k)), whole(rng, (k, n))
    A, B, C = ctx.alloc(8 * ((1 << 28) + 8 * k)), ctx.upload(b), ctx.alloc(m * n * 8)

    class At:
        def __init__(self, offset):
            self.ptr = A.ptr + offset
    ctx.upload_async(At(0), a[:8])
    ctx.upload_async(At(8 << 28), a[8:])
    rows = capi.index_map([8, k], [0])
    rows.ndigits, rows.bits[1], rows.shift[1] = 2, 1, 28
    assert ctx.cgemm_mapped(capi.FP32, A, rows, capi.index_map([8, k], [1]), B,
                            capi.index_map([k, n], [0]), capi.index_map([k, n], [1]), C)
    assert np.array_equal(ctx.download(C, np.complex64, (m, n)), product(a, b))
    for buf in (A, B, C):
        buf.free()


@pytest.mark.parametrize("times", [1, 8])
@pytest.mark.parametrize("prec", [capi.FP32, capi.SPLIT_FP16, capi.SPLIT_BF16X3])
def test_grouped_products_off_the_large_tiles_exact(ctx, prec, times):
    """Every route of a grouped call that is FP32 in this precision, several
    products per tile and some alone, operands at 8-byte addresses: k <= 16
    with n above and below 16, and the FP32 kernel's tiles; problem lists as
    kernel arguments and uploaded."""
    shapes = [(5, 3, 1), (300, 16, 16), (70, 17, 5), (64, 64, 16), (129, 200, 11), (1, 40, 9),
              (33, 7, 35), (513, 9, 100), (20, 300, 33), (40, 15, 1025), (63, 90, 49),
              (9, 4, 4097), (32, 64, 17), (1000, 2, 19), (17, 130, 300)]
    if prec == capi.FP32:
        shapes += [(100, 100, 100), (513, 65, 33), (1300, 700, 20), (129, 129, 1000)]
    rng = np.random.default_rng(prec)
    problems, want, bufs = [], [], []
    for m, n, k in shapes * times:
        a, b = whole(rng, (m, k)), whole(rng, (k, n))
        A = ctx.upload(np.concatenate([[0], a.ravel()]).astype(np.complex64))
        B, C = ctx.upload(b), ctx.alloc((m * n + 1) * 8)
        ctx.zero(C)

        class At8:
            ptr = A.ptr + 8
        problems.append((m, n, k, At8, B, C))
        want.append(product(a, b))
        bufs += [A, B, C]
    ctx.cgemm_grouped(prec, problems)
    for (m, n, k, _, _, C), w in zip(problems, want):
        got = ctx.download(C, np.complex64, (m * n + 1,))
        assert np.array_equal(got[:-1].reshape(m, n), w), (m, n, k)
        assert got[-1] == 0, (m, n, k)
    for buf in bufs:
        buf.free()


def test_grouped_products_run_alone_are_profiled(ctx):
    """Products of a grouped call that the FP32 kernel takes one by one (long
    k, or 512 tiles and more) count in the profile as single calls do."""
    rng = np.random.default_rng(8)
    shapes = [(57, 104, 3384), (40, 30, 20000), (8192, 1024, 32)]
    problems = [(m, n, k, ctx.upload(whole(rng, (m, k))), ctx.upload(whole(rng, (k, n))),
                 ctx.alloc(m * n * 8)) for m, n, k in shapes]
    ctx.profile(True)
    ctx.profile_reset()
    ctx.cgemm_grouped(capi.FP32, problems)
    got = ctx.profile_read()["cgemm"]
    ctx.profile(False)
    assert got["flops"] == sum(8.0 * m * n * k for m, n, k in shapes)
    assert got["bytes"] == sum(8.0 * (m * k + k * n + m * n) for m, n, k in shapes)
    for problem in problems:
        for buf in problem[3:]:
            buf.free()


def test_small_outputs_are_one_class_in_the_profile(ctx):
    """The same matrix-core kernel reads them row-major and through index maps."""
    m, n, k = 128, 64, 256
    rng = np.random.default_rng(9)
    A, B, C = ctx.upload(whole(rng, (m, k))), ctx.upload(whole(rng, (k, n))), ctx.alloc(m * n * 8)
    maps = [capi.index_map(dims, [axis]) for dims in ([m, k], [k, n]) for axis in (0, 1)]
    ctx.profile(True)
    ctx.profile_reset()
    ctx.cgemm(capi.FP32, m, n, k, A, B, C)
    assert ctx.cgemm_mapped(capi.FP32, A, maps[0], maps[1], B, maps[2], maps[3], C)
    prof = ctx.profile_read()
    ctx.profile(False)
    assert prof["cgemm"]["launches"] == 2 and prof["cgemm_small"]["launches"] == 0
    for buf in (A, B, C):
        buf.free()


def test_grouped_f32_products_beyond_one_grid():
    """33000 products of 511 tiles each: more blocks than a launch can hold."""
    m, n, k, count = 65408, 2, 17, 33000
    ctx = capi.Context(0)  # 40 GiB that closing it gives back
    rng = np.random.default_rng(11)
    a, b = whole(rng, (m, k)), whole(rng, (k, n))
    A, B, C = ctx.upload(a), ctx.upload(b), ctx.alloc(8 * m * n * count)

    class At:
        def __init__(self, i):
            self.ptr, self.nbytes = C.ptr + 8 * m * n * i, 8 * m * n
    spots = [0, 1, count // 3, count - 200, count - 2, count - 1]
    for i in spots:
        ctx.zero(At(i))
    ctx.cgemm_grouped(capi.FP32, [(m, n, k, A, B, At(i)) for i in range(count)])
    want = product(a, b)
    for i in spots:
        assert np.array_equal(ctx.download(At(i), np.complex64, (m, n)), want), i
    ctx.close()


def test_split_products_beyond_32_bit_offsets_same_bits(ctx):
    """Odd k and an A of more than 2 GiB (rows in equal blocks): the split
    kernels with 64-bit addressing give each block of rows the bits that the
    pipelined ones give it alone."""
    rows, blocks, n, k = 1024, 512, 48, 517
    rng = np.random.default_rng(10)
    rand = lambda *s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    part, B = ctx.upload(rand(rows, k)), ctx.upload(rand(k, n))
    A, C, C1 = ctx.alloc(8 * rows * blocks * k), ctx.alloc(8 * rows * blocks * n), ctx.alloc(8 * rows * n)

    class At:
        def __init__(self, block):
            self.ptr = A.ptr + 8 * rows * k * block
    for block in range(blocks):
        ctx.copy(At(block), part, 8 * rows * k)
    for prec in (capi.SPLIT_FP16, capi.SPLIT_BF16, capi.SPLIT_BF16X3):
        ctx.zero(C)
        ctx.cgemm(prec, rows * blocks, n, k, A, B, C)
        ctx.cgemm(prec, rows, n, k, part, B, C1)
        want = ctx.download(C1, np.uint64, (1, rows, n))
        assert want.any()
        assert (ctx.download(C, np.uint64, (blocks, rows, n)) == want).all(), prec
    for buf in (part, A, B, C, C1):
        buf.free()
