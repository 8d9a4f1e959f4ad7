"""GPU tests of recorded sequences (qfx_graph_*, HIP stream capture): a
sequence of GEMMs, a reorder, a copy, a zero fill and an FP64 accumulation
is recorded once and replayed several times, with other work and
synchronizations between the replays; every replay must give the eager
results bit for bit."""
import numpy as np
import pytest

from qflex_amd import capi

pytestmark = pytest.mark.gpu


def rand_c(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


def test_recorded_sequence_replays_match_eager(ctx):
    rng = np.random.default_rng(31)
    m, n, k = 16384, 256, 256          # large-tile split-FP16 product
    a, b = rand_c(rng, (m, k)), rand_c(rng, (k, n))
    s = rand_c(rng, (16, 16))          # k = 16 product on the vector ALUs
    A, B, S = ctx.upload(a), ctx.upload(b), ctx.upload(s)
    C1, C2, C3, C4 = (ctx.alloc(m * n * 8) for _ in range(4))
    amps = ctx.alloc(64 * 16)
    other_a, other_c = ctx.upload(rand_c(rng, (512, 512))), ctx.alloc(512 * 512 * 8)

    def sequence():
        ctx.cgemm(capi.SPLIT_FP16, m, n, k, A, B, C1)          # C1 = A B
        ctx.reorder(C1, C2, [m // 16, 16, n], [1, 0, 2])       # C2 = C1 with rows permuted
        ctx.cgemm(capi.FP32, m * n // 16, 16, 16, C2, S, C3)   # C3 = C2 (as rows of 16) . S
        ctx.copy(C4, C3, m * n * 8)
        ctx.zero(amps)
        ctx.accumulate(C4, 64, amps)                            # amps = first 64 entries
        ctx.accumulate(C4, 64, amps)                            # twice: 2 x C4[:64]

    def read():
        return (ctx.download(C1, np.complex64, (m, n)), ctx.download(C4, np.complex64, (m, n)),
                ctx.download(amps, np.complex128, (64,)))

    sequence()
    ctx.sync()
    eager = read()
    ref = a.astype(np.complex128) @ b.astype(np.complex128)
    assert np.linalg.norm(eager[0] - ref) / np.linalg.norm(ref) < 1e-5
    assert np.array_equal(eager[2], 2 * eager[1].reshape(-1)[:64].astype(np.complex128))

    ctx.graph_begin(workspace_bytes=64 << 20)
    try:
        sequence()
    finally:
        graph = ctx.graph_end()
    try:
        for rep in range(3):
            for buf in (C1, C2, C3, C4, amps):
                ctx.zero(buf)
            ctx.cgemm(capi.SPLIT_FP16, 512, 512, 512, other_a, other_a, other_c)  # other work
            ctx.sync()
            graph.launch()
            ctx.sync()
            got = read()
            for g, e in zip(got, eager):
                assert np.array_equal(g, e), rep
    finally:
        graph.destroy()
    for buf in (A, B, S, C1, C2, C3, C4, amps, other_a, other_c):
        buf.free()


def test_synchronizing_calls_refused_while_recording(ctx):
    buf = ctx.alloc(1 << 12)
    ctx.graph_begin()
    try:
        with pytest.raises(RuntimeError, match="recorded"):
            ctx.sync()
        with pytest.raises(RuntimeError, match="recorded"):
            ctx.download(buf, np.uint8, (16,))
        ctx.zero(buf)  # a fill kernel is recorded
    finally:
        graph = ctx.graph_end()
    graph.launch()
    ctx.sync()
    assert not ctx.download(buf, np.uint8, (1 << 12,)).any()
    graph.destroy()
    buf.free()


def test_workspace_must_be_reserved_before_recording():
    """A product whose workspace exceeds the reservation fails while
    recording (instead of synchronizing to grow it)."""
    c = capi.Context(0)
    try:
        rng = np.random.default_rng(5)
        m, n, k = 256, 256, 4096      # split-K partials: 16 x 256 x 256 x 8 bytes = 8 MiB
        A, B, C = c.upload(rand_c(rng, (m, k))), c.upload(rand_c(rng, (k, n))), c.alloc(m * n * 8)
        c.graph_begin(workspace_bytes=0)
        try:
            with pytest.raises(RuntimeError, match="workspace"):
                c.cgemm(capi.SPLIT_FP16, m, n, k, A, B, C)
        finally:
            c.graph_end().destroy()
        c.cgemm(capi.SPLIT_FP16, m, n, k, A, B, C)  # eager: the workspace grows
        c.sync()
    finally:
        c.close()


@pytest.mark.parametrize("prec", [capi.FP32, capi.SPLIT_FP16])
@pytest.mark.parametrize("workspace", [0, 64 << 20])
def test_recorded_products_of_few_outputs_match_eager(prec, workspace):
    """Products the FP32 kernel splits over k, at a small and a large
    reservation: the recorded ones give the eager bits."""
    rng = np.random.default_rng(6)
    for m, n, k in [(57, 104, 3384), (200, 14, 1000), (3, 2000, 700)]:
        c = capi.Context(0)  # its workspace has not grown yet
        try:
            A, B = c.upload(rand_c(rng, (m, k))), c.upload(rand_c(rng, (k, n)))
            C = c.alloc(m * n * 8)
            c.graph_begin(workspace_bytes=workspace)
            try:
                c.cgemm(prec, m, n, k, A, B, C)
            finally:
                graph = c.graph_end()
            got = []
            for _ in range(3):
                c.zero(C)
                graph.launch()
                got.append(c.download(C, np.complex64, (m, n)))
            graph.destroy()
            c.zero(C)
            c.cgemm(prec, m, n, k, A, B, C)
            want = c.download(C, np.complex64, (m, n))
            assert all(np.array_equal(g, want) for g in got), (m, n, k)
        finally:
            c.close()


def test_outgrown_workspace_of_a_graph_is_not_handed_out():
    """An eager product grows the workspace that a recorded one uses: the old
    one must not become another buffer's memory while the graph can be
    replayed, and goes back to the arena once the graph is destroyed."""
    rng = np.random.default_rng(12)
    m, n, k = 57, 104, 3384
    reserve = 4 << 20
    c = capi.Context(0)
    try:
        A, B, C = c.upload(rand_c(rng, (m, k))), c.upload(rand_c(rng, (k, n))), c.alloc(m * n * 8)
        c.cgemm(capi.FP32, m, n, k, A, B, C)
        want = c.download(C, np.complex64, (m, n))
        c.graph_begin(workspace_bytes=reserve)
        try:
            c.cgemm(capi.FP32, m, n, k, A, B, C)
        finally:
            graph = c.graph_end()
        # partial sums of 16384 chunks of 8 x 8 outputs, 8 MiB: more than the reservation
        X, Z = c.alloc(8 * 8 * (1 << 25)), c.alloc(8 * 64)
        c.zero(X)
        c.cgemm(capi.FP32, 8, 8, 1 << 25, X, X, Z)
        others = [c.upload(np.full(reserve // 8, i + 1, np.uint64)) for i in range(4)]
        for _ in range(2):
            c.zero(C)
            graph.launch()
            assert np.array_equal(c.download(C, np.complex64, (m, n)), want)
        for i, buf in enumerate(others):
            assert (c.download(buf, np.uint64, (reserve // 8,)) == i + 1).all(), i
        held = c.arena_stats()[1]
        graph.destroy()
        assert held - c.arena_stats()[1] >= reserve
    finally:
        c.close()
