"""Chains of thin steps in one pass (qt_contract_chain) against the same steps through
qt_contract_pair: the same arithmetic in the same order, so the same bits."""
import ctypes

import numpy as np
import pytest

import qtorch_amd as qa
from qtorch_amd import workloads as wl
from qtorch_amd._native import _i32, hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qa.Context(0)
    yield c
    c.close()


# links as (tensor axes summed in the small tensor's order, new axes): counted from the
# tensor so far; -1 is its last axis
CHAINS = [
    (16, 1, [((0, -1), 1), ((-1,), 2)]),                       # the smallest tensor
    (19, 1, [((0, -1), 1), ((-1,), 2), ((5, -1), 1), ((-1,), 2), ((0, -1), 1), ((0,), 2), ((-1,), 1), ((3,), 0)]),
    (21, 1, [((20, 4), 2), ((0,), 2), ((0,), 2), ((1, 0), 0)]),
    (18, 1, [((17,), 2), ((18,), 2), ((19,), 2), ((20, 0), 1)]),  # grows three bits first
    (9, 2, [((0,), 1), ((8,), 1), ((4,), 1)]),                 # dimension 4, two bits a wire
    (22, 1, [((2,), 1), ((9,), 1), ((15,), 1), ((21,), 1), ((20,), 1)]),
]


@pytest.mark.parametrize("prec", [qa.QT_PLAIN_C128, qa.QT_C64_4M, qa.QT_C64_3M, qa.QT_C64_BF16X3])
@pytest.mark.parametrize("rank,d,links", CHAINS)
def test_chain_equals_steps(ctx, rank, d, links, prec):
    rng = np.random.default_rng(rank + 10 * len(links) + d)
    c128 = prec == qa.QT_PLAIN_C128
    dt, dtype = (np.complex128, qa.QT_DTYPE_C128) if c128 else (np.complex64, qa.QT_DTYPE_C64)

    def tensor(r):
        v = (rng.standard_normal(1 << (d * r)) + 1j * rng.standard_normal(1 << (d * r))).astype(dt)
        return qa.Tensor(ctx, r, d, dtype).upload(v)

    x = tensor(rank)
    small, steps, desc, axes = make_links(rng, tensor, rank, links)
    n = hip.qt_chain_links(rank, d, dtype, len(links), _i32(desc), _i32(axes))
    assert n >= 2
    ref = x
    for g, pairs, free in steps[:n]:
        ref, _ = qa.contract_pair(ctx, ref, g, pairs, free, prec)
    assert np.array_equal(run_chain(ctx, x, small[:n], desc, axes, prec).download(), ref.download()), n


def make_links(rng, tensor, rank, links):
    """The small tensors, (tensor, pairs, free) of every step, and the chain's arguments."""
    steps, small, desc, axes, r = [], [], [], [], rank
    for pos, new in links:
        pos = [p % r for p in pos]
        order = [int(i) for i in rng.permutation(len(pos) + new)]  # the small tensor's axes, shuffled
        pairs = list(zip(pos, order))
        free = [(True, i) for i in range(r) if i not in pos] + [(False, a) for a in order[len(pos):]]
        g = tensor(len(order))
        steps.append((g, pairs, free))
        small.append(g)
        r = len(free)
        desc += [len(order), len(pos), r]
        axes += [p for p, _ in pairs] + [q for _, q in pairs]
        axes += [a | qa.QT_FROM_A if from_a else a for from_a, a in free]
    return small, steps, desc, axes


def run_chain(ctx, x, small, desc, axes, prec):
    n = len(small)
    c = qa.Tensor(ctx, desc[3 * n - 1], x.dim_log2, x.dtype)
    gs = (ctypes.c_void_p * n)(*[g.handle for g in small])
    ctx.check(hip.qt_contract_chain(ctx.handle, x.handle, x.rank, n, gs, _i32(desc), _i32(axes), c.handle, prec), "chain")
    return c


EIGHT = [((0, -1), 1), ((-1,), 2), ((5, -1), 1), ((-1,), 2), ((0, -1), 1), ((0,), 2), ((-1,), 1), ((3,), 0)]


@pytest.mark.parametrize("prec", [qa.QT_C64_4M, qa.QT_C64_3M, qa.QT_C64_BF16X3])
@pytest.mark.parametrize("case", ["unit", "1e-6", "1e6", "2^-90", "2^90", "selects", "one tile", "zero", "exponent"])
def test_rescaled_chain_keeps_the_range_of_steps(ctx, case, prec):
    """Eight links whose combined scale leaves FP32: the values that rescaling after every
    step gives.  Scaling by powers of two commutes with every rounding of a step (no value
    here is subnormal either way), so they are equal."""
    rng = np.random.default_rng(17)
    prec |= qa.QT_RESCALE
    scale = {"1e-6": 1e-6, "1e6": 1e6, "2^-90": 2.0 ** -90, "2^90": 2.0 ** 90}.get(case, 1.0)

    def values(r):
        return (rng.standard_normal(1 << r) + 1j * rng.standard_normal(1 << r)).astype(np.complex64)

    def small(r):
        v = values(r) * np.float32(scale)
        if case == "selects":  # large where the tensor is zero, 1e-6 where it is not
            v *= np.where(np.arange(1 << r) & 1, np.float32(1e-6), np.float32(1))
        return qa.Tensor(ctx, r, 1, qa.QT_DTYPE_C64).upload(v)

    v = values(19)
    links = EIGHT
    if case == "selects":
        links = [((0,), 0)] * 8  # the lowest bit summed, nothing added
        v[(np.arange(v.size) & 255) != 255] = 0  # only bit 1 of every summed wire
    if case == "one tile":  # most tiles hold no value at all
        v[: v.size - 1] = 0
    if case == "zero":
        v[:] = 0
    x = qa.Tensor(ctx, 19, 1, qa.QT_DTYPE_C64).upload(v)
    if case == "exponent":  # X carries one already
        x, _ = qa.contract_pair(ctx, x, qa.Tensor(ctx, 1, 1, qa.QT_DTYPE_C64).upload(np.array([1e-30, 2e-30])), [],
                                [(True, i) for i in range(19)] + [(False, 0)], prec)
        assert x.exponent() < -80
    gs, steps, desc, axes = make_links(rng, small, x.rank, links)
    n = hip.qt_chain_links(x.rank, 1, x.dtype, len(links), _i32(desc), _i32(axes))
    assert n >= 6
    ref = x
    for g, pairs, free in steps[:n]:
        ref, _ = qa.contract_pair(ctx, ref, g, pairs, free, prec)
    c = run_chain(ctx, x, gs[:n], desc, axes, prec)
    assert c.exponent() == ref.exponent()
    assert np.array_equal(c.download(), ref.download())
    assert case == "zero" or 0.5 <= max(np.abs(c.download().view(np.float32))) < 1


def test_rescaled_chain_passes_infinities_on(ctx):
    """An infinite element spoils the outputs it reaches, step by step and in one pass; the
    others keep their values."""
    rng = np.random.default_rng(3)

    def tensor(r):
        v = (rng.standard_normal(1 << r) + 1j * rng.standard_normal(1 << r)).astype(np.complex64)
        return qa.Tensor(ctx, r, 1, qa.QT_DTYPE_C64).upload(v * np.float32(1e-3))

    v = (rng.standard_normal(1 << 18) + 1j * rng.standard_normal(1 << 18)).astype(np.complex64)
    v[12345] = np.inf
    x = qa.Tensor(ctx, 18, 1, qa.QT_DTYPE_C64).upload(v)
    gs, steps, desc, axes = make_links(rng, tensor, 18, [((0,), 1), ((16,), 1), ((2,), 1)])
    prec = qa.QT_C64_4M | qa.QT_RESCALE
    assert hip.qt_chain_links(18, 1, x.dtype, 3, _i32(desc), _i32(axes)) == 3
    ref = x
    for g, pairs, free in steps:
        ref, _ = qa.contract_pair(ctx, ref, g, pairs, free, prec)
    c = run_chain(ctx, x, gs, desc, axes, prec)
    got, want = c.download(), ref.download()
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), ok) and not ok.all() and ok.any()
    assert np.array_equal(np.ldexp(got[ok].view(np.float32).astype(np.float64), c.exponent()),
                          np.ldexp(want[ok].view(np.float32).astype(np.float64), ref.exponent()))


def test_what_does_not_chain(ctx):
    """A small tensor, three summed bits, free axes out of order, the small tensor's axes
    first: none of them is taken."""
    def links(rank, per_link):
        desc, axes = [], []
        for pairs, free, rg in per_link:
            desc += [rg, len(pairs), len(free)]
            axes += [p for p, _ in pairs] + [q for _, q in pairs]
            axes += [a | qa.QT_FROM_A if from_a else a for from_a, a in free]
        return hip.qt_chain_links(rank, 1, qa.QT_DTYPE_C64, len(per_link), _i32(desc), _i32(axes))

    def gate(rank, pos, new):
        return ([(p, i) for i, p in enumerate(pos)],
                [(True, i) for i in range(rank) if i not in pos] + [(False, len(pos) + i) for i in range(new)],
                len(pos) + new)

    good = gate(18, (0,), 1)
    assert links(18, [good, good]) == 2
    assert links(18, [good]) == 0
    assert links(15, [gate(15, (0,), 1)] * 2) == 0
    assert links(18, [gate(18, (0, 1, 2), 2)] * 2) == 0
    swapped = (good[0], [good[1][1], good[1][0]] + good[1][2:], good[2])
    assert links(18, [good, swapped]) == 0
    first = (good[0], good[1][-1:] + good[1][:-1], good[2])
    assert links(18, [first, good]) == 0


def test_sweep_with_chains_matches_line_graph(ctx):
    """The sweep order of a 20-qubit circuit (its large steps in chains) against the line-graph
    order of the same circuit, rescaled form included."""
    q, bits = wl.grid_random_circuit(4, 5, 12, seed=3), wl.bitstring(20, 4)
    ref, _ = qa.SlicedNetwork(q, bits, dim_log2=1, order=qa.ORDER_LINEGRAPH, max_bits=26).run(ctx)
    sweep = qa.SlicedNetwork(q, bits, dim_log2=1, order=qa.ORDER_SWEEP, max_bits=28)
    assert sweep.plan()["peak_bits"] >= 16
    for prec, tol in ((qa.QT_PLAIN_C128, 1e-11), (qa.QT_C64_4M, 2e-5), (qa.QT_C64_4M | qa.QT_RESCALE, 2e-5)):
        v, _ = sweep.run(ctx, prec)
        assert abs(v - ref) <= tol * max(abs(ref), 2.0 ** -10)


@pytest.mark.parametrize("order,fusion", [(qa.ORDER_SWEEP, 0), (qa.ORDER_LINEGRAPH, 0), (qa.ORDER_LINEGRAPH, -1)])
def test_runs_take_only_passes_that_fit(order, fusion):
    """Rescaled runs with small tensors that carry exponents (every unfused result does): no
    pass is tried and refused, which would leave its message on the context."""
    ctx = qa.Context(0)
    q, bits = wl.grid_random_circuit(4, 5, 14, seed=3), wl.bitstring(20, 4)
    net = qa.SlicedNetwork(q, bits, dim_log2=1, order=order, max_bits=28)
    ref, _ = net.run(ctx)
    net.set_fusion(fusion)
    v, _ = net.run(ctx, qa.QT_C64_4M | qa.QT_RESCALE)
    assert abs(v - ref) <= 2e-5 * max(abs(ref), 2.0 ** -10)
    assert hip.qt_last_error(ctx.handle) == b""
    net.close()
    ctx.close()
