"""Callers whose output array overlaps the iterate.  Residual_iga and Tangent_iga
copy U into U_hist level 0 before anything is written (src/assmcore_iga.c:68, 557),
so R may lie over U at any offset, and U may lie in the value array: the results and
U_hist are those of the call with separate arrays, bit for bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NEL = (9, 4, 5)


@pytest.fixture(scope="module")
def mesh(igap):
    return igap.MeshIGABeam(nelem=NEL, L=(2, 1, 1))


def context(igap, mesh, torder, flags=0):
    ph = igap.PhysGradElastTime() if torder else igap.PhysGradElast()
    return igap.Assm(mesh, ph, igap.BCClampedTip(tip=0.02), flags=flags)


def dev(igap, A, n):
    from igap4_amd import _lib
    p = C.c_void_p()
    _lib.check(_lib.lib().igap_gpu_malloc(A.ctx, C.byref(p), 8 * n))
    return p


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("shift", [-700, -1, 0, 1, 64])
@pytest.mark.parametrize("torder", [0, 2])
def test_residual_over_its_iterate(igap, oracle, mesh, torder, shift, noalloc):
    from igap4_amd import _lib
    with context(igap, mesh, torder) as A:
        n = A.ndof
        H = oracle.glibc_rand_state((torder + 1) * n) * 0.05
        U = oracle.glibc_rand_state(n, seed=7) * 0.05
        call = _lib.lib().igap_gpu_residual_noalloc if noalloc else _lib.lib().igap_gpu_residual
        A.set_uhist(H)
        u = dev(igap, A, n)
        A.htod(u, U)
        _lib.check(call(A.ctx, u, None))
        R_ref = A.dtoh(A.rvec_ptr(), n)
        _lib.check(_lib.lib().igap_gpu_free(A.ctx, u))
        A.set_uhist(H)
        buf = dev(igap, A, n + abs(shift))
        up = C.c_void_p(buf.value + 8 * max(0, -shift))
        rp = C.c_void_p(buf.value + 8 * max(0, shift))
        A.htod(up, U)
        _lib.check(call(A.ctx, up, rp))
        R = A.dtoh(rp, n)
        kept = A.get_uhist()
        _lib.check(_lib.lib().igap_gpu_free(A.ctx, buf))
    assert np.array_equal(R, R_ref)
    assert np.array_equal(kept[:n], U) and np.array_equal(kept[n:], H[n:])


@pytest.mark.parametrize("mode", ["IGAP_TANGENT_ELEMENT_MATRICES", "IGAP_TANGENT_DIRECT"])
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("torder", [0, 2])
def test_tangent_over_its_iterate(igap, oracle, mesh, torder, prec, mode):
    from igap4_amd import _lib
    with context(igap, mesh, torder, getattr(_lib, mode)) as A:
        n, nnz = A.ndof, A.nnz
        es, dt = (8, np.float64) if prec == 0 else (4, np.float32)
        H = oracle.glibc_rand_state((torder + 1) * n) * 0.05
        U = oracle.glibc_rand_state(n, seed=7) * 0.05
        vals = dev(igap, A, nnz + n)
        A.set_uhist(H)
        far = C.c_void_p(vals.value + 8 * nnz)
        A.htod(far, U)
        A.tangent_dev(far, vals, prec)
        K_ref = A.dtoh(vals, nnz, dt)
        for at in (0, 8 * (es * (nnz // 2) // 8), es * nnz - 8):   # the first values, the middle, the last 8 bytes
            A.set_uhist(H)
            up = C.c_void_p(vals.value + at)
            A.htod(up, U)
            A.tangent_dev(up, vals, prec)
            K = A.dtoh(vals, nnz, dt)
            kept = A.get_uhist()
            assert np.array_equal(K, K_ref), at
            assert np.array_equal(kept[:n], U) and np.array_equal(kept[n:], H[n:]), at
        _lib.check(_lib.lib().igap_gpu_free(A.ctx, vals))
