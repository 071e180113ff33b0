"""The tensor-product tangent of patches with equal weights and any geometry
(k_tangent_gen): every entry against the oracle's loop nest
(src/assmcore_iga.c:607-764), on the distorted beam and, through
IGAP_GENERAL_GEOMETRY, on straight patches (periodic ones among them), through
the element matrices and the direct scatter, in both precisions.  One element
fills one workgroup, so the sizes that can go wrong are those of the index
arithmetic: one element in a direction, different counts per direction, the
periodic wrap-around."""
import numpy as np
import pytest

from test_gpu_parity import NTHREADS, TOL32, TOL64, rowfloor_err

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 0, False), ((2, 1, 3), 0, True), ((3, 7, 2), 0, True), ((5, 2, 9), 0, False), ((9, 4, 5), 0, True),
         ((5, 7, 6), 1, False)]


@pytest.mark.parametrize("nelem, per, pert", CASES)
def test_tangent_sizes(igap, oracle, nelem, per, pert):
    from igap4_amd import _lib
    periodic = (per, per, per)
    mo = oracle.Mesh(nelem, L=(2, 1, 1.5), periodic=periodic, perturbed=pert)
    mg = igap.MeshIGABeam(nelem=nelem, L=(2, 1, 1.5), periodic=periodic, perturbed=pert)
    if per:
        pp = [0.01, 0.0, 0.02, 0.0, -0.01, 0.0, 0.005, 0.0, 0.004]
        bc_o, bc_g = oracle.make_bc(par_periodic=pp), igap.BC(par_periodic=pp)
    else:
        bc_o, bc_g = oracle.clamped_tip_bc(tip=0.02), igap.BCClampedTip(tip=0.02)
    ph_o, ph_g = oracle.make_phys(0), igap.PhysGradElast()
    U = oracle.glibc_rand_state(mo.ndof) * 0.05
    rp_o, col_o, K_o = oracle.tangent(mo, ph_o, bc_o, U, nthreads=NTHREADS)
    flags = [_lib.IGAP_TANGENT_ELEMENT_MATRICES] + ([] if per else [_lib.IGAP_TANGENT_DIRECT])
    for fl in flags:
        with igap.Assm(mg, ph_g, bc_g, flags=fl | _lib.IGAP_GENERAL_GEOMETRY) as A:
            for prec, tol in (("f64", TOL64), ("f32", TOL32)):
                rp, col, K = A.tangent(U, prec=prec)
                assert np.array_equal(rp, rp_o) and np.array_equal(col, col_o)
                err = rowfloor_err(K, K_o, rp_o)
                print(f"{nelem} periodic {per} perturbed {pert} flags {fl} {prec}: {err:.2e}")
                assert err < tol
