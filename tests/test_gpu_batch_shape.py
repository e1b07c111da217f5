"""The executor shape that a batch chooses for itself: it fits the device memory there is and
the 4 GiB bound, also after programs are added; a shape that the caller chooses is refused or
kept whatever the instances of the moment."""
import numpy as np
import pytest

import qtorch_amd as qa
from qtorch_amd import workloads as wl
from tests.full_device import full_device
from tests.programs import Batch, Program

pytestmark = pytest.mark.gpu

QT_OK, QT_OOM = 0, 2


@pytest.fixture(scope="module")
def ctx():
    c = qa.Context(0)
    yield c
    c.close()


def test_default_shape_without_room_for_its_scratch():
    """1,024 networks with 1.6 MiB of intermediates each: four workgroups a CU need 1.7 GiB,
    one 0.4 GiB; with 1.1 GiB left the batch runs, with the same bits."""
    q = wl.qft_qasm(8)
    strings = [wl.measure_text(format(i % 256, "08b")[::-1]) for i in range(1024)]
    ref_ctx = qa.Context(0)
    b = qa.NetBatch(ref_ctx, [q] * 1024, strings, precision=qa.QT_PLAIN_C128)
    b.launch()
    want = b.results()
    b.close()
    ref_ctx.close()
    ctx = qa.Context(0)
    with full_device(1152):
        b = qa.NetBatch(ctx, [q] * 1024, strings, precision=qa.QT_PLAIN_C128)
        b.launch()
        got = b.results()
        b.close()
    assert np.array_equal(got, want)


def small_program(ctx):
    """Two rank-5 leaves to a rank-10 tensor (16 KiB), summed with itself's transpose."""
    outer = (0, 1, 5, 5, [], [(True, i) for i in range(5)] + [(False, i) for i in range(5)])
    other = (1, 0, 5, 5, [], outer[5])
    return Program(ctx, 1, [5] * 4, [0, 32, 0, 32], [outer, (2, 3, 5, 5, [], other[5]),
                                                     (4, 5, 10, 10, [(i, i) for i in range(10)], [])])


def large_program(ctx):
    """16 outer products of rank-8 leaves u_i v_i, contracted in a balanced tree over v_i and
    u_j: six tensors of 1 MiB (complex128) live at once."""
    free = [(True, i) for i in range(8)] + [(False, 8 + i) for i in range(8)]
    steps, level = [], []
    for i in range(16):
        steps.append((2 * i, 2 * i + 1, 8, 8, [], [(True, k) for k in range(8)] + [(False, k) for k in range(8)]))
        level.append(32 + i)
    while len(level) > 2:
        nxt = []
        for x, y in zip(level[::2], level[1::2]):
            steps.append((x, y, 16, 16, [(8 + i, i) for i in range(8)], free))
            nxt.append(32 + len(steps) - 1)
        level = nxt
    steps.append((level[0], level[1], 16, 16, [(8 + i, i) for i in range(8)] + [(i, 8 + i) for i in range(8)], []))
    return Program(ctx, 1, [8] * 32, [64 + 256 * i for i in range(32)], steps)


def pool():
    rng = np.random.default_rng(12)
    return (rng.standard_normal(64 + 32 * 256) + 1j * rng.standard_normal(64 + 32 * 256)) / 16


def large_value(p):
    """The trace of the product of the 16 dyads."""
    leaf = p[64:].reshape(32, 256)
    return np.prod([leaf[2 * i + 1] @ leaf[(2 * i + 2) % 32] for i in range(16)])


def test_programs_added_to_a_default_shape(ctx):
    small, large = small_program(ctx), large_program(ctx)
    assert large.scratch() * 16 * 256 * 4 > 4 << 30  # four workgroups a CU would pass the bound
    b = Batch(ctx, [small], qa.QT_PLAIN_C128, later=[large])
    p = pool()
    b.set(p, [0] + [1] * 1023)
    assert b.shape() == (256, 2, True)
    got = b.run()
    ref = large_value(p)
    # 16 sums of 2^8 terms, each rounding relative to the terms' norms (about 2 each here)
    assert np.abs(got[1:] - ref).max() <= 1e-12 * max(abs(ref), 1)
    b.close()


def test_chosen_shape_beyond_the_bound_is_refused(ctx):
    """However few the instances; the shape before it stays."""
    b = Batch(ctx, [large_program(ctx)], qa.QT_PLAIN_C128)
    b.set(pool(), [0])
    first = b.run()
    before = b.shape()
    assert b.config(256, 4) == QT_OOM and b.config(256, 16) == QT_OOM
    assert b.shape() == before
    assert np.array_equal(b.run(), first)
    assert b.config(256, 1) == QT_OK
    assert np.array_equal(b.run(), first)
    b.close()
