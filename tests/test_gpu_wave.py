"""The apply without tiles (rp_terms_info kernel RP_APPLY_SMALL) at the edges
of its range: chains below one wavefront, every slice count, one and four
amplitudes per lane, and flip masks with one, two and many terms whose
coefficients are real, imaginary, complex and mixed, with phase bits in the
lane, the row and the remaining index bits.

Tolerance: FP64 sums of the terms (n of them, each off by at most
eps64 |c v|) and one rounding to the state's precision."""
import ctypes

import numpy as np
import pytest

from conftest import random_state
from gpu_util import DeviceBuffer, Terms, prec_of

pytestmark = pytest.mark.gpu

_vp = ctypes.c_void_p


def _terms(rng, L, masks, fp):
    """`masks` flip masks with 1, 2, 3, 1, 2, 9, ... terms of every kind."""
    bits, co = [], []
    xs = {0} | {int(v) for v in rng.integers(0, 1 << L, masks - 1)}
    for i, x in enumerate(sorted(xs)):
        nt = (1, 2, 3, 1, 2, 9)[i % 6]
        kind = (i // 6) % 4
        for q in range(nt):
            z = int(rng.integers(0, 1 << L))
            b = 0
            for s in range(L):
                b |= (x >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)
            c = rng.standard_normal() + 1j * rng.standard_normal()
            c = (c.real, 1j * c.imag, c, c.real if q % 2 else 1j * c.imag)[kind]
            bits.append(b)
            co.append(c)
    co = np.array(co, np.complex128)
    return np.array(bits, np.uint64), co.astype(np.complex64).astype(np.complex128) if fp == 32 else co


@pytest.mark.parametrize("fp,native", [(32, False), (32, True), (64, False)])
@pytest.mark.parametrize("L,masks", [(1, 2), (2, 4), (5, 9), (6, 30), (7, 40), (9, 120), (12, 300),
                                     (15, 70), (16, 3), (17, 12), (18, 40), (20, 16)])
def test_apply_without_tiles(gpu, orc, fp, native, L, masks):
    rng = np.random.default_rng(1000 * L + masks + fp)
    dt = np.complex64 if fp == 32 else np.complex128
    bits, co = _terms(rng, L, masks, fp)
    psi, prior = random_state(rng, L, dt), random_state(rng, L, dt)
    ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
    t = Terms(L, bits, co, prec_of(dt), gpu.RP_TERMS_ACC_NATIVE if native else 0)
    info = t.info()
    assert info.kernel == gpu.RP_APPLY_SMALL and info.tile_bits == 0
    vin = DeviceBuffer.from_array(psi)
    depths = [info.depth] + ([1, 8, 32, 128] if L <= 16 else [])
    # |sum| error: terms times the rounding of the sums, plus the output's
    eps = 1.2e-7 if native else 2.3e-16
    tol = len(bits) * eps * np.abs(co).sum() * np.abs(psi).max() + \
        (6e-8 if fp == 32 else 1.2e-16) * (np.abs(ref).max() + np.abs(prior).max())
    for d in depths:
        if d != info.depth:
            gpu.check(gpu.hip().rp_terms_set_tiling(t.h, 0, 256, d))
        out = DeviceBuffer.from_array(prior)
        for acc in (1, 0, 0):      # twice over the same workspace
            gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, acc))
            got = out.to_array(dt, len(psi)).astype(np.complex128)
            want = ref + prior if acc else ref
            assert np.abs(got - want).max() <= tol, (L, d, acc)
        out.free()
    vin.free()
    t.free()


@pytest.mark.parametrize("fp,native", [(32, False), (32, True), (64, False)])
@pytest.mark.parametrize("L,masks,depth", [(13, 400, 128), (14, 160, 32), (14, 400, 128),
                                           (15, 150, 32), (15, 1250, None), (16, 40, 8),
                                           (16, 400, 32)])
def test_long_lists(gpu, orc, fp, native, L, masks, depth):
    """The slices and four amplitudes a lane that lists of many terms get from
    13 to 16 sites, with phase bits in the row bits (sites 6 and 7)."""
    rng = np.random.default_rng(1000 * L + masks + fp)
    dt = np.complex64 if fp == 32 else np.complex128
    bits, co = _terms(rng, L, masks, fp)
    psi, prior = random_state(rng, L, dt), random_state(rng, L, dt)
    ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
    t = Terms(L, bits, co, prec_of(dt), gpu.RP_TERMS_ACC_NATIVE if native else 0)
    info = t.info()
    assert info.kernel == gpu.RP_APPLY_SMALL and info.depth == (depth or (128 if native else 32))
    vin, out = DeviceBuffer.from_array(psi), DeviceBuffer.from_array(prior)
    eps = 1.2e-7 if native else 2.3e-16
    tol = len(bits) * eps * np.abs(co).sum() * np.abs(psi).max() + \
        (6e-8 if fp == 32 else 1.2e-16) * (np.abs(ref).max() + np.abs(prior).max())
    for acc in (1, 0, 0):
        gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, acc))
        got = out.to_array(dt, len(psi)).astype(np.complex128)
        assert np.abs(got - (ref + prior if acc else ref)).max() <= tol, acc


@pytest.mark.parametrize("fp,native", [(32, False), (32, True), (64, False)])
@pytest.mark.parametrize("L,masks,per,depth", [(9, 1, 33, 1), (12, 2, 100, 8), (14, 1, 300, 8),
                                               (16, 3, 700, 32), (18, 1, 260, 8)])
def test_masks_of_many_terms(gpu, orc, fp, native, L, masks, per, depth):
    """Few flip masks of many terms are cut into pieces that fill the slices
    (the last one of a single term at 33)."""
    rng = np.random.default_rng(1000 * L + per + fp)
    dt = np.complex64 if fp == 32 else np.complex128
    bits, co = [], []
    for x in rng.choice(1 << L, masks, False):
        for q in range(per):
            z = int(rng.integers(0, 1 << L))
            bits.append(sum((int(x) >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)
                            for s in range(L)))
            co.append(rng.standard_normal() * (1j if q % 3 == 1 else 1))
    bits, co = np.array(bits, np.uint64), np.array(co, np.complex128)
    if fp == 32:
        co = co.astype(np.complex64).astype(np.complex128)
    psi = random_state(rng, L, dt)
    ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
    t = Terms(L, bits, co, prec_of(dt), gpu.RP_TERMS_ACC_NATIVE if native else 0)
    info = t.info()
    assert info.kernel == gpu.RP_APPLY_SMALL and info.depth == depth
    assert info.nflips == masks
    vin, out = DeviceBuffer.from_array(psi), DeviceBuffer(psi.nbytes)
    eps = 1.2e-7 if native else 2.3e-16
    tol = len(bits) * eps * np.abs(co).sum() * np.abs(psi).max() + \
        (6e-8 if fp == 32 else 1.2e-16) * np.abs(ref).max()
    for d in [depth] + ([1, 8, 128] if L <= 16 else []):
        if d != info.depth:
            gpu.check(gpu.hip().rp_terms_set_tiling(t.h, 0, 256, d))
        gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, 0))
        assert np.abs(out.to_array(dt, len(psi)).astype(np.complex128) - ref).max() <= tol, d


@pytest.mark.parametrize("L,masks", [(17, 12), (18, 40), (19, 60), (20, 16), (22, 30)])
def test_reported_tiling_can_be_set_again(gpu, L, masks):
    """A program that tries other tilings goes back to the one it was given;
    what no upload chooses is refused."""
    rng = np.random.default_rng(L)
    bits, co = _terms(rng, L, masks, 32)
    dt = np.complex64
    t = Terms(L, bits, co, prec_of(dt))
    i = t.info()
    first = (i.tile_bits, i.threads, i.depth)
    assert first[0] == 0
    psi = random_state(rng, L, dt)
    vin, out = DeviceBuffer.from_array(psi), DeviceBuffer(psi.nbytes)
    gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, 0))
    want = out.to_array(dt, len(psi))
    gpu.check(gpu.hip().rp_terms_set_tiling(t.h, 12, 512, 2))
    gpu.check(gpu.hip().rp_terms_set_tiling(t.h, *first))
    i = t.info()
    assert (i.tile_bits, i.threads, i.depth) == first
    gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, 0))
    assert np.array_equal(out.to_array(dt, len(psi)), want)
    for d in (32, 128) + ((8,) if L > 19 else ()):
        assert gpu.hip().rp_terms_set_tiling(t.h, 0, 256, d) != 0
    many, c = _terms(rng, L, 80, 32)
    u = Terms(L, many, c, prec_of(dt))
    assert (gpu.hip().rp_terms_set_tiling(u.h, 0, 256, 1) == 0) == (L <= 19)


@pytest.mark.parametrize("fp,L", [(32, 28), (32, 29), (64, 27), (64, 28)])
def test_states_around_4_gib(gpu, fp, L):
    """The chain with two- and many-term masks that takes no tiles at any
    length, on both sides of the state size from which the gathers need 64-bit
    offsets: windows of rows at the ends, the middle and at random."""
    rng = np.random.default_rng(L + fp)
    dt, es = (np.complex64, 8) if fp == 32 else (np.complex128, 16)
    pair = [3 << i for i in range(L - 1)]
    x = np.array(pair + pair + [0] * (2 * L - 1))
    z = np.array([0] * (L - 1) + pair + pair + [1 << i for i in range(L)])
    bits = np.zeros(len(x), np.uint64)
    for s in range(L):
        bits |= ((x >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)).astype(np.uint64)
    co = rng.standard_normal(len(x)) + 0j
    if fp == 32:
        co = co.astype(np.complex64).astype(np.complex128)
    t = Terms(L, bits, co, prec_of(dt))
    assert t.info().kernel == gpu.RP_APPLY_SMALL
    hip, n = gpu.hip(), 1 << L
    vin, out = DeviceBuffer(es << L), DeviceBuffer(es << L)
    gpu.check(hip.rp_init_random(prec_of(dt), vin.ptr, n, 3))
    gpu.check(hip.rp_apply_ops(t.h, out.ptr, vin.ptr, 0))

    def window(buf, lo):
        a = np.empty(64, dt)
        gpu.check(hip.rp_memcpy(a.ctypes.data_as(_vp), _vp(buf.ptr.value + lo * es), a.nbytes,
                                gpu.RP_D2H))
        return a.astype(np.complex128)

    for lo in [0, n // 2 - 64, n // 2, n - 64] + [int(v) * 64 for v in rng.integers(0, n // 64, 4)]:
        m = np.arange(lo, lo + 64)
        ref, size = np.zeros(64, np.complex128), 0.0
        for xv in np.unique(x):
            v = window(vin, (lo ^ int(xv)) & ~63)[(m ^ int(xv)) & 63]
            size = max(size, np.abs(v).max())
            for c, zv in zip(co[x == xv], z[x == xv]):
                par = np.array([bin(int(q) & int(zv)).count("1") & 1 for q in m ^ int(xv)])
                ref += c * (1 - 2 * par) * v
        tol = len(co) * 2.3e-16 * np.abs(co).sum() * size + (6e-8 if fp == 32 else 1.2e-16) * \
            np.abs(ref).max()
        assert np.abs(window(out, lo) - ref).max() <= tol, lo
    for b in (vin, out):
        b.free()
