"""The tiled apply with FP64 sums over compact records, and the streamed
apply with group accumulation, at every two-tile tiling: all classes of subs
(real, imaginary and complex single terms with and without phase bits in the
row, lane and tile bits, flip masks with several terms), every row flip, one
and two groups, against the oracle.

Tolerance: FP64 sums of n terms and one rounding of the output; with group
accumulation FP32 sums of the terms of four groups."""
import numpy as np
import pytest

from conftest import random_state
from gpu_util import DeviceBuffer, Terms, prec_of

pytestmark = pytest.mark.gpu

TILINGS = {32: [(8, 128, 2), (10, 128, 2), (12, 512, 2), (12, 1024, 2), (13, 1024, 2)],
           64: [(8, 128, 2), (10, 128, 2), (12, 512, 2)]}


def _list(rng, L, tb, groups):
    """Flip masks in `groups` groups: every combination of bit 0 and the top
    tile bits with a random rest, 1 to 3 terms each."""
    bits, co = [], []
    highs = [0] + [int(h) for h in rng.choice(np.arange(1, 1 << (L - tb)), groups - 1, False)]
    for i in range(64):
        x = highs[i % groups] << tb | int(rng.integers(0, 1 << tb))
        x = x & ~1 | i & 1
        for _ in range((1, 1, 1, 2, 1, 3)[i % 6]):
            z = int(rng.integers(0, 1 << L)) & (~0, 0x3e, -1 << 6, -1 << tb)[(i // 2) % 4]
            b = 0
            for s in range(L):
                b |= (x >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)
            c = rng.standard_normal() + 1j * rng.standard_normal()
            bits.append(b)
            co.append((c.real, 1j * c.imag, c)[(i // 6) % 3])
    return np.array(bits, np.uint64), np.array(co, np.complex128)


@pytest.mark.parametrize("fp,group", [(32, False), (32, True), (64, False)])
@pytest.mark.parametrize("groups", [1, 2, 5])
def test_two_tile_tilings(gpu, orc, fp, group, groups):
    L = 16
    dt = np.complex64 if fp == 32 else np.complex128
    for tb, nt, d in TILINGS[fp]:
        rng = np.random.default_rng(tb * nt + groups)
        bits, co = _list(rng, L, tb, groups)
        if fp == 32:
            co = co.astype(np.complex64).astype(np.complex128)
        psi, prior = random_state(rng, L, dt), random_state(rng, L, dt)
        ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
        t = Terms(L, bits, co, prec_of(dt), gpu.RP_TERMS_ACC_GROUP if group else 0)
        gpu.check(gpu.hip().rp_terms_set_tiling(t.h, tb, nt, d))
        vin = DeviceBuffer.from_array(psi)
        out = DeviceBuffer.from_array(prior)
        eps = 1.2e-7 if group else 2.3e-16
        tol = len(bits) * eps * np.abs(co).sum() * np.abs(psi).max() + \
            (6e-8 if fp == 32 else 1.2e-16) * (np.abs(ref).max() + np.abs(prior).max())
        for acc in (1, 0):
            gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, acc))
            got = out.to_array(dt, len(psi)).astype(np.complex128)
            assert np.abs(got - (ref + prior if acc else ref)).max() <= tol, (tb, nt, acc)
        vin.free()
        out.free()
        t.free()


@pytest.mark.parametrize("fp", [32, 64])
@pytest.mark.parametrize("masks,per", [(109, 1), (110, 1), (60, 3), (75, 2)])
def test_record_formats(gpu, orc, fp, masks, per):
    """Both sides of the list length at which the FP64 sums change from 48-byte
    to 16-byte records (21 sites: 110 masks, or fewer that share terms)."""
    L = 21
    dt = np.complex64 if fp == 32 else np.complex128
    rng = np.random.default_rng(masks + per)
    x = np.repeat(rng.choice(1 << L, masks, False), per)
    z = rng.integers(0, 1 << L, len(x))
    bits = np.zeros(len(x), np.uint64)
    for s in range(L):
        bits |= ((x >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)).astype(np.uint64)
    co = rng.standard_normal(len(x)) * 1j ** (np.arange(len(x)) % 2)
    if fp == 32:
        co = co.astype(np.complex64).astype(np.complex128)
    psi = random_state(rng, L, dt)
    ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
    t = Terms(L, bits, co, prec_of(dt))
    gpu.check(gpu.hip().rp_terms_set_tiling(t.h, 12, 512, 2))
    vin, out = DeviceBuffer.from_array(psi), DeviceBuffer(psi.nbytes)
    gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, 0))
    tol = len(bits) * 2.3e-16 * np.abs(co).sum() * np.abs(psi).max() + \
        (6e-8 if fp == 32 else 1.2e-16) * np.abs(ref).max()
    assert np.abs(out.to_array(dt, len(psi)).astype(np.complex128) - ref).max() <= tol


def _random(rng, L, masks, per, row_bits=True):
    """`masks` distinct flip masks of up to six sites, `per` Hermitian terms each."""
    x = set()
    while len(x) < masks:
        x.add(sum(1 << int(s) for s in rng.choice(L, int(rng.integers(1, 7)), False)))
    bits, co = [], []
    for v in sorted(x):
        for _ in range(per):
            z = int(rng.integers(0, 1 << L)) & (~0 if row_bits else ~(3 << 6))
            bits.append(sum((v >> s & 1) << (2 * s) | (z >> s & 1) << (2 * s + 1)
                            for s in range(L)))
            co.append(rng.standard_normal() * 1j ** bin(v & z).count("1"))
    return np.array(bits, np.uint64), np.array(co, np.complex128)


FREE, S, M, B = (0, 256), (12, 512), (12, 1024), (13, 1024)


@pytest.mark.parametrize("mode,L,masks,per,want", [
    # single terms: the tile by the list's length, the sums and the chain
    ("c64", 20, 60, 1, M), ("c64", 22, 60, 1, S), ("c64", 22, 110, 1, M), ("c64", 23, 110, 1, S),
    ("c64", 24, 240, 1, M), ("c64", 27, 240, 1, M), ("c64", 28, 240, 1, S),
    ("group", 20, 60, 1, M), ("group", 21, 60, 1, S), ("group", 25, 60, 1, S),
    ("group", 26, 60, 1, M), ("group", 26, 70, 1, B), ("group", 28, 60, 1, B),
    ("c128", 20, 60, 1, S), ("native", 26, 60, 1, S),
    # masks that share terms
    ("c64", 26, 60, 3, M), ("c64", 28, 60, 3, M), ("group", 22, 60, 3, M), ("group", 28, 60, 3, M),
    # few of them: without tiles, except where FP32 sums in tiles are cheaper
    ("c64", 24, 20, 4, FREE), ("c128", 26, 40, 4, FREE), ("group", 22, 20, 4, M),
    ("group", 22, 20, -4, FREE), ("native", 24, 20, 4, FREE), ("native", 24, 20, 20, FREE),
    # two terms a mask and as many groups as masks
    ("c64", 25, 10, 2, FREE), ("c64", 26, 10, 2, M), ("c128", 22, 10, 2, FREE),
    ("c128", 23, 10, 2, S), ("group", 23, 10, 2, FREE), ("group", 23, 10, -2, FREE),
    ("group", 25, 10, -2, M), ("group", 25, 10, 2, M),
    ("c64", 26, 10, 1, S),
    # 19 sites: many single-term masks with group accumulation
    ("group", 19, 700, 1, M), ("group", 19, 300, 1, FREE), ("group", 19, 700, 2, FREE),
    ("c64", 19, 700, 1, FREE)])
def test_default_tilings(gpu, orc, mode, L, masks, per, want):
    """The default layout's choice where it changes, and its apply against the
    oracle where that is quick."""
    rng = np.random.default_rng(7)
    bits, co = _random(rng, L, masks, abs(per), per > 0)
    flips = (1 << 2 * L) // 3      # the even bits
    while per == 2 and L > 19 and len({int(b) & flips >> 24 << 24 for b in bits}) < masks:
        bits, co = _random(rng, L, masks, 2)     # until every mask is a group of its own
    dt = np.complex128 if mode == "c128" else np.complex64
    if dt == np.complex64:
        co = co.astype(np.complex64).astype(np.complex128)
    t = Terms(L, bits, co, prec_of(dt), {"group": gpu.RP_TERMS_ACC_GROUP,
                                         "native": gpu.RP_TERMS_ACC_NATIVE}.get(mode, 0))
    i = t.info()
    assert (i.tile_bits, i.threads) == want and (want == FREE or i.depth == 2)
    if len(bits) << L > 1 << 29:
        return
    psi = random_state(rng, L, dt)
    ref = orc.apply(L, bits, co, psi.astype(np.complex128), fp=64)
    vin, out = DeviceBuffer.from_array(psi), DeviceBuffer(psi.nbytes)
    gpu.check(gpu.hip().rp_apply_ops(t.h, out.ptr, vin.ptr, 0))
    eps = 1.2e-7 if mode in ("group", "native") else 2.3e-16
    tol = len(bits) * eps * np.abs(co).sum() * np.abs(psi).max() + \
        (6e-8 if dt == np.complex64 else 1.2e-16) * np.abs(ref).max()
    assert np.abs(out.to_array(dt, len(psi)).astype(np.complex128) - ref).max() <= tol
