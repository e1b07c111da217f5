"""Program steps on the matrix cores (executors of 64 and 256 lanes) against the vector
steps of lane groups: the same chain of multiply-adds per output, so the same bits."""
import math
import os

import numpy as np
import pytest

import qtorch_amd as qa
from qtorch_amd import workloads as wl
from tests.programs import Batch, Program

GOLDEN_DIR = os.path.join(os.path.dirname(__file__), "golden")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qa.Context(0)
    yield c
    c.close()


def _same_bits(batch):
    batch.config(16, 1, qa.QT_SCRATCH_GLOBAL)
    batch.launch()
    ref = batch.results()
    for lanes, wgs in ((64, 1), (256, 1), (256, 4)):
        batch.config(lanes, wgs, qa.QT_SCRATCH_GLOBAL)
        batch.launch()
        got = batch.results()
        for x, y in zip(ref, got):
            assert np.array_equal(x, y), (lanes, wgs)


@pytest.mark.parametrize("prec", [qa.QT_PLAIN_C128, qa.QT_C64_4M, qa.QT_C64_3M])
def test_light_cones_of_uneven_size(ctx, prec):
    """Depth 2 on a 3-regular graph: programs of uneven size, taken longest first."""
    rng = np.random.default_rng(3)
    with open(os.path.join(GOLDEN_DIR, "samples", "3regRand30Node50.dgf")) as f:
        b = qa.QaoaBatch(ctx, f.read(), 2, ref_map=False, precision=prec)
    b.set_angles(np.concatenate([rng.uniform(0, math.pi / 2, (3, 2)), rng.uniform(-3, 3, (3, 2))], axis=1))
    _same_bits(b)
    b.close()


@pytest.mark.parametrize("prec", [qa.QT_PLAIN_C128, qa.QT_C64_4M, qa.QT_C64_3M])
@pytest.mark.parametrize("dim_log2,rows,cols,depth", [(1, 3, 4, 8), (2, 2, 3, 6)])
def test_grid_networks(ctx, prec, dim_log2, rows, cols, depth):
    """Dimension 2 (any power of two summed, 8 included) and 4."""
    q = wl.grid_random_circuit(rows, cols, depth, seed=5)
    n = rows * cols
    b = qa.NetBatch(ctx, [q] * 5, [wl.measure_text(wl.bitstring(n, k)) for k in range(5)], precision=prec,
                    dim_log2=dim_log2)
    _same_bits(b)
    b.close()


def _variant(mb, nb, kb):
    """The block of 16 x 16 tiles a wave takes for 2^mb x 2^nb outputs over 2^kb, None for
    vector steps."""
    if mb < 4 or nb < 4 or kb < 2 or mb + nb + kb < 12:
        return None
    blocks = mb + nb - 8
    if kb >= 3 and blocks >= 4 and mb >= 5 and nb >= 5:
        return 2, 2
    if kb >= 3 and blocks >= 3:
        return (1, 2) if nb >= 5 else (2, 1)
    return 1, 1


SHAPES = {
    (1, 1): [(4, 6, 2), (6, 4, 2), (5, 5, 2), (4, 5, 3), (4, 4, 4), (4, 4, 5), (5, 4, 6), (4, 4, 8)],
    (1, 2): [(4, 7, 3), (5, 6, 4), (4, 8, 4), (4, 7, 5), (4, 8, 6)],
    (2, 1): [(7, 4, 3), (8, 4, 4), (7, 4, 5), (8, 4, 6)],
    (2, 2): [(6, 6, 3), (6, 6, 4), (5, 7, 5), (7, 5, 5), (6, 6, 6), (8, 8, 3)],
    None: [(3, 6, 4), (6, 3, 4), (5, 5, 1), (4, 4, 3)],
}


@pytest.mark.parametrize("prec", [qa.QT_PLAIN_C128, qa.QT_C64_4M, qa.QT_C64_3M])
@pytest.mark.parametrize("variant", SHAPES)
def test_every_block_shape(ctx, prec, variant):
    """A step with C's low axes from A and its high ones from B against the same sums with an
    axis of A moved to the top of C, which the matrix cores do not take: operands that are
    leaves, intermediates in LDS and in device memory, tensor results, 64 and 256 lanes."""
    c128 = prec == qa.QT_PLAIN_C128
    dtype = qa.QT_DTYPE_C128 if c128 else qa.QT_DTYPE_C64
    rng = np.random.default_rng(9)
    pool = rng.standard_normal(1 << 18) + 1j * rng.standard_normal(1 << 18)
    placed = set()
    for mb, nb, kb in SHAPES[variant]:
        assert _variant(mb, nb, kb) == variant
        pairs = [(mb + i, nb + kb - 1 - i) for i in range(kb)]
        low, high = [(True, i) for i in range(mb)], [(False, i) for i in range(nb)]
        if variant is None or kb == 2:  # B's summed axes first, too
            pairs, high = [(mb + i, i) for i in range(kb)], [(False, kb + i) for i in range(nb)]
        for a_made, b_made in ((False, False), (True, False), (False, True), (True, True)):
            # an operand that is made: the outer product of two leaves
            ranks, offsets, steps, at = [], [], [], {}
            for name, r, made in (("a", mb + kb, a_made), ("b", nb + kb, b_made)):
                at[name] = len(ranks)
                for part in ((r // 2, r - r // 2) if made else (r,)):
                    offsets.append(offsets[-1] + (1 << ranks[-1]) if ranks else 0)
                    ranks.append(part)
            ids = {}
            for name, r, made in (("a", mb + kb, a_made), ("b", nb + kb, b_made)):
                i = at[name]
                ids[name] = i
                if made:
                    outer = [(True, k) for k in range(ranks[i])] + [(False, k) for k in range(ranks[i + 1])]
                    ids[name] = len(ranks) + len(steps)
                    steps.append((i, i + 1, ranks[i], ranks[i + 1], [], outer))
            last = (ids["a"], ids["b"], mb + kb, nb + kb, pairs)
            split = Program(ctx, 1, ranks, offsets, steps + [last + (low + high,)])
            moved = Program(ctx, 1, ranks, offsets, steps + [last + (low[:-1] + high + low[-1:],)])
            batch = Batch(ctx, [split, moved], prec)
            outs = [qa.Tensor(ctx, mb + nb, 1, dtype) for _ in range(2)]
            batch.set(pool, [0, 1])
            batch.set_outputs(outs)
            for lanes in (64, 256):
                for place in (qa.QT_SCRATCH_LDS, qa.QT_SCRATCH_GLOBAL):
                    if batch.config(lanes, 1, place) != 0:
                        assert place == qa.QT_SCRATCH_LDS
                        continue
                    placed.add(place)
                    batch.launch()
                    got, want = (t.download() for t in outs)
                    # C of `moved`: its highest axis belongs at place mb - 1
                    want = want.reshape(2, 1 << nb, 1 << (mb - 1)).transpose(1, 0, 2).reshape(-1)
                    assert np.array_equal(got, want), (mb, nb, kb, a_made, b_made, lanes, place)
            batch.close()
    assert placed == {qa.QT_SCRATCH_LDS, qa.QT_SCRATCH_GLOBAL}


@pytest.mark.parametrize("prec", [qa.QT_PLAIN_C128, qa.QT_C64_4M, qa.QT_C64_3M, qa.QT_C64_BF16X3])
def test_small_programs_beside_large_ones(ctx, prec):
    """A batch without large steps runs the kernel that has no registers for them; the same
    program in a batch with one, the other kernel: the same bits."""
    small = Program(ctx, 1, [4, 4, 4, 3, 1], [0, 16, 32, 48, 56], [
        (0, 1, 4, 4, [(3, 0), (2, 2)], [(True, 0), (False, 1), (True, 1), (False, 3)]),
        (2, 3, 4, 3, [(0, 1), (3, 0)], [(False, 2), (True, 1), (True, 2)]),
        (5, 6, 4, 3, [(0, 0), (2, 2), (3, 1)], [(True, 1)]),
        (7, 4, 1, 1, [(0, 0)], [])])
    large = Program(ctx, 1, [9, 9, 8], [0, 64, 128], [
        (0, 1, 9, 9, [(4 + i, 4 + i) for i in range(5)], [(True, i) for i in range(4)] + [(False, i) for i in range(4)]),
        (3, 2, 8, 8, [(i, i) for i in range(8)], [])])
    rng = np.random.default_rng(10)
    pool = rng.standard_normal(1024) + 1j * rng.standard_normal(1024)
    alone, beside = Batch(ctx, [small], prec), Batch(ctx, [large, small], prec)
    alone.set(pool, [0, 0])
    beside.set(pool, [1, 0, 1])
    for lanes, place in ((64, qa.QT_SCRATCH_LDS), (64, qa.QT_SCRATCH_GLOBAL), (256, qa.QT_SCRATCH_LDS),
                         (256, qa.QT_SCRATCH_GLOBAL)):
        assert alone.config(lanes, 2, place) == 0 and beside.config(lanes, 2, place) == 0
        x, y = alone.run(), beside.run()
        assert np.array_equal(x, y[[0, 2]]) and x[0] != 0 and y[1] != 0, (lanes, place)
    alone.close()
    beside.close()
