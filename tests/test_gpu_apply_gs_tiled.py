"""rp_apply_gs where its fused kernel runs (complex<float>, tiling 12/512 with
two LDS tiles, set by hand because short chains use no tiles by default),
against numpy: h = V^H (H v), the updated vector and its norm, for basis
sizes across the epilogue's chunks of 8 vectors.

Tolerances: FP32 outputs of FP64 sums (group accumulation: FP32 sums of four
groups, the terms' sum within len * 1.2e-7 * sum|c| of an amplitude); the
dots are linear in H v, so their error is at most that of H v in 2-norm."""
import ctypes

import numpy as np
import pytest

from gpu_util import DeviceBuffer, Terms

pytestmark = pytest.mark.gpu

_vp = ctypes.c_void_p


@pytest.mark.parametrize("flags", [0, 4])
@pytest.mark.parametrize("k,fuse_min", [(1, 0.0), (8, 0.0), (9, 0.0), (17, 0.0), (1, 0.25),
                                        (9, 0.25), (9, 1e6)])
def test_apply_gs_on_its_tiling(gpu, orc, flags, k, fuse_min):
    L, n = 14, 1 << 14
    rng = np.random.default_rng(10 * k + flags)
    bits, coeff = orc.syk_terms(2 * L, 8.0, seed=92, fp=32)
    coeff = coeff.astype(np.complex64).astype(np.complex128)
    a = rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k))
    Q = np.linalg.qr(a)[0].astype(np.complex64)
    t = Terms(L, bits, coeff, gpu.RP_C64, flags=flags)
    gpu.check(gpu.hip().rp_terms_set_tiling(t.h, 12, 512, 2))
    V = [DeviceBuffer.from_array(np.ascontiguousarray(Q[:, q])) for q in range(k)]
    out = DeviceBuffer(8 * n)
    h = np.zeros(2 * k)
    norm, nz = ctypes.c_double(), ctypes.c_int()
    gpu.check(gpu.hip().rp_apply_gs(t.h, out.ptr, V[-1].ptr, (_vp * k)(*[b.ptr.value for b in V]), k,
                                    h.ctypes.data_as(_vp), ctypes.byref(norm), fuse_min,
                                    ctypes.byref(nz)))
    h = h.view(np.complex128)
    w = out.to_array(np.complex64, n).astype(np.complex128)
    Q64 = Q.astype(np.complex128)
    hv = orc.apply(L, bits, coeff, Q64[:, -1])
    h_ref = Q64.conj().T @ hv
    r = hv - Q64 @ h_ref
    # |H v - computed| in 2-norm, and one more FP32 rounding of the update
    err = (1.2e-7 * len(bits) ** 0.5 * np.abs(coeff).sum() if flags else 0.0) \
        + 1.2e-7 * np.linalg.norm(hv)
    beta = norm.value
    # normalized where the norm is large enough and free of cancellation
    assert nz.value == (0 < fuse_min <= np.linalg.norm(r) and
                        np.linalg.norm(r) ** 2 >= np.linalg.norm(hv) ** 2 / 2)
    if nz.value:
        w *= beta
    print("flags %d k %d: |dh| %.1e (bound %.1e), |dw| %.1e" % (
        flags, k, np.linalg.norm(h - h_ref), err, np.linalg.norm(w - r)), flush=True)
    assert np.linalg.norm(h - h_ref) <= err
    assert np.linalg.norm(w - r) <= 3 * err
    assert abs(beta - np.linalg.norm(r)) <= 3 * err
    t.free()
