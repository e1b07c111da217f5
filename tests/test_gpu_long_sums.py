"""Long sums into few outputs (k_reduce_rows) against numpy's tensordot in complex128
(which pins the oracle's loop nest, tests/test_oracle.py): the edges of the rule that chooses it (2^9 and 2^11 summed
indices, 2^11 and 2^16 outputs), one and several row groups and workgroups, free axes of
both sides in any order in C."""
import numpy as np
import pytest

import qtorch_amd as qa
from qtorch_amd._native import _i32, hip
from tests.full_device import full_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = qa.Context(0)
    yield c
    c.close()


def _tensordot(a, ra, b, rb, free, pairs, d):
    """C's flat values; axis i of a tensor is numpy axis -1 - i."""
    a, b = a.astype(np.complex128).reshape([1 << d] * ra), b.astype(np.complex128).reshape([1 << d] * rb)
    c = np.tensordot(a, b, axes=([ra - 1 - x for x, _ in pairs], [rb - 1 - y for _, y in pairs]))
    left = [(True, i) for i in reversed(range(ra)) if i not in [x for x, _ in pairs]]
    left += [(False, i) for i in reversed(range(rb)) if i not in [y for _, y in pairs]]
    return c.transpose([left.index(f) for f in reversed(free)]).reshape(-1)


# (free wires of A, free wires of B, summed wires, dim_log2)
SHAPES = [(0, 0, 9, 1), (0, 3, 10, 1), (11, 0, 9, 1), (5, 6, 9, 1), (2, 3, 5, 2), (0, 1, 13, 1), (3, 2, 14, 1),
          (12, 0, 11, 1), (1, 11, 11, 1), (10, 6, 11, 1), (0, 8, 6, 2), (4, 3, 12, 1)]


@pytest.mark.parametrize("prec,tol", [(qa.QT_PLAIN_C128, 1e-13), (qa.QT_C64_4M, 2e-6), (qa.QT_C64_3M, 4e-6),
                                      (qa.QT_C64_BF16X3, 1e-4)])
@pytest.mark.parametrize("fa,fb,k,d", SHAPES)
def test_long_sums(ctx, fa, fb, k, d, prec, tol):
    rng = np.random.default_rng(1000 * fa + 100 * fb + 10 * k + d)
    c128 = prec == qa.QT_PLAIN_C128
    dt = np.complex128 if c128 else np.complex64
    ra, rb = fa + k, fb + k
    a, b = ((rng.standard_normal(1 << (d * r)) + 1j * rng.standard_normal(1 << (d * r))).astype(dt) for r in (ra, rb))
    ta, tb = (qa.Tensor(ctx, r, d, qa.QT_DTYPE_C128 if c128 else qa.QT_DTYPE_C64).upload(x)
              for r, x in ((ra, a), (rb, b)))
    for interleave in (False, True):
        pa, pb = rng.permutation(ra), rng.permutation(rb)
        pairs = [(int(x), int(y)) for x, y in zip(pa[:k], pb[:k])]
        free = [(True, int(x)) for x in pa[k:]] + [(False, int(y)) for y in pb[k:]]
        if interleave:
            free = [free[i] for i in rng.permutation(len(free))]
        got = qa.contract_pair(ctx, ta, tb, pairs, free, prec)[0].download()
        ref = _tensordot(a, ra, b, rb, free, pairs, d)
        # sums of 2^(d k) products of unit variance: rounding of about sqrt(2^(d k)) terms
        assert np.abs(got - ref).max() <= tol * np.sqrt(1 << (d * k)) * max(np.abs(ref).max(), 1.0)


def test_long_sum_without_room_for_partial_sums():
    """16 MiB of partial sums on a card without them: the sum runs one output a lane."""
    ctx = qa.Context(0)
    rng = np.random.default_rng(8)
    v = (rng.standard_normal(1 << 20) + 1j * rng.standard_normal(1 << 20)).astype(np.complex64)
    k, fa, fb = 20, 6, 7
    a, b = (qa.Tensor(ctx, f + k, 1, qa.QT_DTYPE_C64).upload(np.tile(x, 1 << f)) for f, x in ((fa, v), (fb, v[::-1])))
    pairs = [(i, i) for i in range(k)]  # every row of A equals v, every row of B its reverse
    free = [(i % 2 == 1, k + i // 2) for i in range(2 * fa)] + [(False, k + fa)]  # B and A in turn: no GEMM
    c = qa.Tensor(ctx, fa + fb, 1, qa.QT_DTYPE_C64)
    fs = _i32([(ax | qa.QT_FROM_A) if from_a else ax for from_a, ax in free])
    px = _i32([x for x, _ in pairs])
    ctx.check(hip.qt_ctx_trim(ctx.handle))
    with full_device(0):
        ctx.check(hip.qt_contract_pair(ctx.handle, a.handle, fa + k, b.handle, fb + k, k, px, px, fa + fb, fs, c.handle,
                                       qa.QT_C64_4M, None))
        ctx.sync()
    got = c.download()
    ref = np.dot(v.astype(np.complex128), v[::-1])
    # 2^21 roundings of partial sums of up to about 2^10.5, independent: 2^-24 2^10.5 2^10.5, four times over
    assert np.abs(got - ref).max() <= 0.5
