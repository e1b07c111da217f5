"""bf16x3 products on operands rewritten as bf16 planes (k_gemm_bf16x3): the smallest
shape that takes it, one split over K, uneven sides, and one or both operands already in
GEMM order on either side of the rule, against numpy in complex128 and the path without planes (qt_contract_pair_noalloc)."""
import ctypes

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


@pytest.mark.parametrize("m,n,k,shuffle", [(7, 7, 5, True), (7, 7, 5, False), (8, 7, 6, True), (7, 9, 10, True),
                                           (8, 7, 8, "A"), (11, 7, 8, "A"), (11, 7, 8, "B"), (9, 8, 13, False)])
def test_planes(ctx, m, n, k, shuffle):
    rng = np.random.default_rng(100 * m + 10 * n + k)
    a, b = ((rng.standard_normal((1 << k, 1 << f)) + 1j * rng.standard_normal((1 << k, 1 << f))).astype(np.complex64)
            for f in (m, n))
    ref = (b.astype(np.complex128).T @ a).reshape(-1)  # C[m + M n]
    # wires of A: m free then k summed (axis 0 fastest), moved to the places of a permutation
    tensors, place = [], []
    for name, x, f in (("A", a, m), ("B", b, n)):
        to = rng.permutation(f + k) if shuffle in (True, name) else np.arange(f + k)  # wire i sits on axis to[i]
        r = f + k
        t = x.reshape([2] * r).transpose([r - 1 - int(np.argwhere(to == ax)[0, 0]) for ax in reversed(range(r))])
        tensors.append(qa.Tensor(ctx, r, 1, qa.QT_DTYPE_C64).upload(np.ascontiguousarray(t)))
        place.append([int(v) for v in to])
    pa, pb = place
    # the last pair is the lowest summed digit
    pairs = [(pa[m + i], pb[n + i]) for i in reversed(range(k))]
    free = [(True, pa[i]) for i in range(m)] + [(False, pb[i]) for i in range(n)]
    c, _ = qa.contract_pair(ctx, *tensors, pairs, free, qa.QT_C64_BF16X3)
    got = c.download()
    assert np.abs(got - ref).max() <= 1e-4 * np.sqrt(1 << k) * np.abs(ref).max()
    if (1 << k) < 512:  # no split of the sum: the same products in the same order
        plain = qa.Tensor(ctx, m + n, 1, qa.QT_DTYPE_C64)
        fs = _i32([(ax | qa.QT_FROM_A) if fa else ax for fa, ax in free])
        ctx.check(hip.qt_contract_pair_noalloc(ctx.handle, tensors[0].handle, m + k, tensors[1].handle, n + k, k,
                                               _i32([x for x, _ in pairs]), _i32([y for _, y in pairs]), m + n, fs,
                                               plain.handle, qa.QT_C64_BF16X3, ctypes.byref(ctypes.c_int64())), "noalloc")
        assert np.array_equal(got, plain.download())


@pytest.mark.parametrize("left_mib", [128, 384])
def test_in_place_product_without_room_for_planes(left_mib):
    """Operands of 256 MiB in GEMM order on a full card, with room for neither operand's
    planes or for one's: the product runs on them as they are.  4 output tiles of 64 x 64 or
    one of 128 x 128, 64 parts of the sum either way, so the results are equal."""
    ctx = qa.Context(0)
    m = n = 7
    k = 18
    rng = np.random.default_rng(5)
    v = (rng.standard_normal(1 << 20) + 1j * rng.standard_normal(1 << 20)).astype(np.complex64)
    a, b = (qa.Tensor(ctx, m + k, 1, qa.QT_DTYPE_C64).upload(np.tile(x, 1 << (m + k - 20))) for x in (v, v[::-1]))
    pairs = [(m + i, n + i) for i in reversed(range(k))]
    free = [(True, i) for i in range(m)] + [(False, i) for i in range(n)]
    want = qa.contract_pair(ctx, a, b, pairs, free, qa.QT_C64_BF16X3)[0].download()
    ctx.check(hip.qt_ctx_trim(ctx.handle))
    with full_device(left_mib):
        got = qa.contract_pair(ctx, a, b, pairs, free, qa.QT_C64_BF16X3)[0].download()
    assert np.array_equal(got, want)
