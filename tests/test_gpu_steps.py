"""Queued Krylov steps (rp_arnoldi_steps, rp_lanczos_steps) and the
Gram-Schmidt sweeps at the edges of their launch shapes, against numpy in 64
bits.

Tolerances: a dot product or norm of n terms accumulated in FP64 is off by at
most n eps64 relative to the product of the norms, far below the one rounding
of each stored component, eps(state) / 2; sums over k vectors and the
normalization add a few of those."""
import ctypes

import numpy as np
import pytest

from conftest import random_pauli_sum
from gpu_util import DeviceBuffer, Terms, prec_of

pytestmark = pytest.mark.gpu

_vp = ctypes.c_void_p
EPS = {np.complex64: 6e-8, np.complex128: 1.2e-16}
STEP = 2 * 64 + 2


def _hermitian(rng, length, nterms):
    """Random Pauli strings with phases that make every term Hermitian."""
    bits, _ = random_pauli_sum(rng, length, nterms)
    co = []
    for b in bits:
        y = sum(1 for s in range(length) if (int(b) >> (2 * s)) & 3 == 3)
        co.append(rng.standard_normal() * 1j ** (y % 4))
    return bits, np.array(co)


def _ptrs(bufs):
    return (_vp * len(bufs))(*[b.ptr.value for b in bufs])


def _case(rng, dtype, length):
    """A Hermitian list, the bound sum |c| of its norm and a normalized vector."""
    bits, co = _hermitian(rng, length, 6 * length)
    if dtype == np.complex64:
        co = co.astype(np.complex64).astype(np.complex128)
    v = rng.standard_normal(1 << length) + 1j * rng.standard_normal(1 << length)
    return bits, co, np.abs(co).sum(), (v / np.linalg.norm(v)).astype(dtype)


# Each step is checked from the vectors on the device, by what it leaves of
# H V[j] = sum_i h_i V[i] + norm V[j+1]: the product is rounded once when it
# is stored (EPS ||H||), the coefficients are FP64 sums over the stored
# vector, and the update and the division round once more each.  The bound
# does not grow with j.
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("length,m,j0", [(2, 2, 0), (5, 9, 0), (9, 19, 0), (9, 6, 2), (10, 34, 0),
                                         (14, 10, 0), (17, 4, 0), (18, 9, 0), (20, 4, 1)])
def test_arnoldi_steps(gpu, orc, dtype, length, m, j0):
    rng = np.random.default_rng(100 * length + m)
    n = 1 << length
    bits, co, hnorm, v = _case(rng, dtype, length)
    t = Terms(length, bits, co, prec_of(dtype))
    bufs = [DeviceBuffer.from_array(v if j == 0 else np.zeros(n, dtype)) for j in range(m + 1)]
    out, done = np.zeros((m, STEP)), ctypes.c_int()
    if j0:      # the first steps by a call of their own
        gpu.check(gpu.hip().rp_arnoldi_steps(t.h, _ptrs(bufs[:j0 + 1]), 0, j0, 1e-3,
                                             out.ctypes.data_as(_vp), ctypes.byref(done)))
        assert done.value == j0
    gpu.check(gpu.hip().rp_arnoldi_steps(t.h, _ptrs(bufs), j0, m, 1e-3, out[j0:].ctypes.data_as(_vp),
                                         ctypes.byref(done)))
    assert done.value == m - j0
    V = [b.to_array(dtype, n).astype(np.complex128) for b in bufs]
    tol = 4 * EPS[dtype] * hnorm
    for j in range(m):
        o = out[j]
        got = o[0:2 * j + 2:2] + 1j * o[1:2 * j + 2:2]
        w = orc.apply(length, bits, co, V[j])
        assert np.abs(got - [np.vdot(u, w) for u in V[:j + 1]]).max() <= tol, j
        rest = w - sum(a * u for a, u in zip(got, V))
        assert np.linalg.norm(rest - o[128] * V[j + 1]) <= tol, j
        assert o[129] in (0.0, 1.0)
        # the norm divided by: an FP64 sum of n squares, its terms' roundings
        # adding up as sqrt(n) (beta^2 = ||w||^2 - sum |h|^2 at most doubles
        # them), of a basis that is orthonormal to its own roundings; then one
        # rounding per component
        unit = 4 * EPS[dtype] + 2.2e-16 * np.sqrt(n) + 2 * (j + 1) * EPS[dtype] ** 2 * hnorm ** 2
        if not o[129]:
            assert abs(np.linalg.norm(V[j + 1]) - 1) <= unit, j


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_arnoldi_steps_stop(gpu, dtype):
    """An invariant subspace: Z0 + 2 X1 acts on |00> in a space of dimension
    2, so step 1 leaves nothing; the steps behind it do not run, and the next
    call starts clean."""
    length, m = 2, 6
    bits, co = np.array([2, 1 << 2], np.uint64), np.array([1.0, 2.0 + 0j])
    t = Terms(length, bits, co, prec_of(dtype))
    for _ in range(2):
        v = np.zeros(4, dtype)
        v[0] = 1
        mark = np.full(4, 7, dtype)
        bufs = [DeviceBuffer.from_array(v if j == 0 else mark) for j in range(m + 1)]
        out, done = np.zeros((m, STEP)), ctypes.c_int()
        gpu.check(gpu.hip().rp_arnoldi_steps(t.h, _ptrs(bufs), 0, m, 0.25,
                                             out.ctypes.data_as(_vp), ctypes.byref(done)))
        assert done.value == 2
        assert np.allclose(out[0, :2], [1, 0]) and out[0, 128] == 2.0
        assert abs(out[1, 128]) < 1e-6
        for j in range(3, m + 1):
            assert np.array_equal(bufs[j].to_array(dtype, 4), mark)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("length", [9, 18, 20])
def test_arnoldi_steps_stop_leaves_the_pass_result(gpu, dtype, length):
    """The step that stops leaves its vector unscaled, also where the pass's
    last kernel runs in up to 1024 workgroups and one of them raises the stop
    flag while others start.  H = Z0 + 2 X1 + X2 / 20 on |000> times a random
    state of the other sites: step 1 leaves X1 X2 V0 / (5 b0), b0 = H(1, 0), of
    norm below 0.25."""
    n, m = 1 << length, 4
    rng = np.random.default_rng(length)
    bits = np.array([2, 1 << 2, 1 << 4], np.uint64)
    t = Terms(length, bits, np.array([1.0, 2.0, 0.05]), prec_of(dtype))
    v = np.zeros(n, np.complex128)
    v[::8] = rng.standard_normal(n // 8) + 1j * rng.standard_normal(n // 8)
    v = (v / np.linalg.norm(v)).astype(dtype)
    b0 = np.hypot(2, 0.05)
    want = np.zeros(n, np.complex128)
    want[6::8] = v[::8] * (0.2 / b0)
    mark = np.full(n, 7, dtype)
    for _ in range(4):
        bufs = [DeviceBuffer.from_array(v if j == 0 else mark) for j in range(m + 1)]
        out, done = np.zeros((m, STEP)), ctypes.c_int()
        gpu.check(gpu.hip().rp_arnoldi_steps(t.h, _ptrs(bufs), 0, m, 0.25,
                                             out.ctypes.data_as(_vp), ctypes.byref(done)))
        assert done.value == 2 and out[1, 129] == 0
        # roundings of the stored V0, V1 and V2, of norms 1, 1 and 0.1, carried
        # through H of norm 3.05
        tol = 16 * EPS[dtype]
        assert abs(out[0, 128] - b0) <= tol and abs(out[1, 128] - 0.2 / b0) <= tol
        assert np.linalg.norm(bufs[2].to_array(dtype, n) - want) <= tol
        for j in (3, 4):
            assert np.array_equal(bufs[j].to_array(dtype, n), mark)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("length", [2, 13])
def test_arnoldi_steps_without_terms(gpu, dtype, length):
    """H = 0 stops at its first step: V[1] is zero and the rest untouched."""
    n, m = 1 << length, 4
    t = Terms(length, np.array([2], np.uint64), np.zeros(1), prec_of(dtype))
    mark = np.full(n, 7, dtype)
    v = np.zeros(n, dtype)
    v[1] = 1
    bufs = [DeviceBuffer.from_array(v if j == 0 else mark) for j in range(m + 1)]
    out, done = np.zeros((m, STEP)), ctypes.c_int()
    gpu.check(gpu.hip().rp_arnoldi_steps(t.h, _ptrs(bufs), 0, m, 0.25, out.ctypes.data_as(_vp),
                                         ctypes.byref(done)))
    assert done.value == 1 and out[0, 128] == 0
    assert not bufs[1].to_array(dtype, n).any()
    for j in range(2, m + 1):
        assert np.array_equal(bufs[j].to_array(dtype, n), mark), j
    gpu.check(gpu.hip().rp_apply_ops(t.h, bufs[2].ptr, bufs[0].ptr, 1))
    assert np.array_equal(bufs[2].to_array(dtype, n), mark)
    gpu.check(gpu.hip().rp_apply_ops(t.h, bufs[2].ptr, bufs[0].ptr, 0))
    assert not bufs[2].to_array(dtype, n).any()


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("length,m", [(3, 1), (3, 2), (8, 12), (10, 30), (18, 5)])
def test_lanczos_steps(gpu, orc, dtype, length, m):
    rng = np.random.default_rng(length)
    n = 1 << length
    bits, co, hnorm, v = _case(rng, dtype, length)
    t = Terms(length, bits, co, prec_of(dtype))
    bufs = [DeviceBuffer.from_array(v if j == 0 else np.zeros(n, dtype)) for j in range(m + 1)]
    a, b = np.zeros(m), np.zeros(max(1, m - 1))
    gpu.check(gpu.hip().rp_lanczos_steps(t.h, _ptrs(bufs), m, a.ctypes.data_as(_vp),
                                         b.ctypes.data_as(_vp)))
    V = [b.to_array(dtype, n).astype(np.complex128) for b in bufs]
    tol = 4 * EPS[dtype] * hnorm       # as for the Arnoldi steps
    for j in range(m):
        w = orc.apply(length, bits, co, V[j])
        assert abs(a[j] - np.vdot(V[j], w).real) <= tol, j
        if j == m - 1:
            assert np.linalg.norm(V[m] - w) <= tol
            break
        rest = w - a[j] * V[j] - (b[j - 1] * V[j - 1] if j else 0)
        assert np.linalg.norm(rest - b[j] * V[j + 1]) <= tol, j
        assert b[j] > 0 and abs(np.linalg.norm(V[j + 1]) - 1) <= 4 * EPS[dtype] + 2.2e-16 * np.sqrt(n)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n,k", [(1, 1), (63, 3), (256, 4), (257, 5), (32768, 17), (32769, 9),
                                 (65536, 8), (65537, 16), (262143, 33), (300001, 2), (4096, 64),
                                 (131072, 2), (131073, 1), (131073, 3), (524288, 5), (524289, 3),
                                 (524289, 17), (1048577, 1)])
def test_gs_pass_edges(gpu, dtype, n, k):
    """One pass at the sizes where the launch shape changes (the dots' 256 or
    1024 threads at 2^17 elements for one or two vectors a workgroup, at 2^19
    for more; vectors per workgroup at 2^15; chunks of 16 in the update), twice
    in a row on the same workspace."""
    rng = np.random.default_rng(n + k)
    V = (rng.standard_normal((k, n)) + 1j * rng.standard_normal((k, n))) / np.sqrt(2 * n * k)
    V = V.astype(dtype)
    w = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(dtype)
    V64, w64 = V.astype(np.complex128), w.astype(np.complex128)
    ref = V64.conj() @ w64
    r = w64 - ref @ V64
    vb = [DeviceBuffer.from_array(V[q]) for q in range(k)]
    for _ in range(2):
        wb = DeviceBuffer.from_array(w)
        h, nrm = np.zeros(2 * k), ctypes.c_double()
        gpu.check(gpu.hip().rp_gs_pass(prec_of(dtype), _ptrs(vb), k, wb.ptr, n,
                                       h.ctypes.data_as(_vp), ctypes.byref(nrm)))
        size = np.linalg.norm(V64, axis=1).max() * np.linalg.norm(w64)
        assert np.abs(h.view(np.complex128) - ref).max() <= 4e-16 * np.sqrt(n + 16) * size
        got = wb.to_array(dtype, n).astype(np.complex128)
        assert np.linalg.norm(got - r) <= 4 * EPS[dtype] * np.linalg.norm(w64)
        assert abs(nrm.value - np.linalg.norm(got)) <= 1e-13 * max(nrm.value, 1e-300)
    re, im = ctypes.c_double(), ctypes.c_double()
    wb = DeviceBuffer.from_array(w)
    gpu.check(gpu.hip().rp_vec_prod(prec_of(dtype), vb[0].ptr, wb.ptr, n, ctypes.byref(re),
                                    ctypes.byref(im)))
    assert abs(complex(re.value, im.value) - ref[0]) <= 4e-16 * np.sqrt(n + 16) * size
    gpu.check(gpu.hip().rp_vec_norm(prec_of(dtype), wb.ptr, n, ctypes.byref(nrm)))
    assert abs(nrm.value - np.linalg.norm(w64)) <= 1e-13 * nrm.value
