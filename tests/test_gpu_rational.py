"""Rational patches (unequal control weights): the residual k_residual_gen<*, true>
(quotient rule, its transpose nurbs_param_adj, the factor w_b) and the matrix-core
tangent k_tangent_elem, both scatters and both precisions, entry-wise against the
oracle's loop nests (src/assmcore_iga.c:118-259, 607-764).

Weights: a smooth variation of 25% (the quotient rule's derivative terms are as
large as the others), a different one in every control point, also across the wrap
of a periodic direction.  Tolerances: a basis jet takes about 30 more roundings
through the quotient rule than without (sums over 27 functions, two derivative
orders), of which the weights' spread cancels none: 1e-14 of a row's largest entry
in FP64 and 5e-6 in FP32 at most, so the bounds of the equal-weight parity tests
(1e-12, 2e-5) hold here as well; a missing or misplaced weight is 1e-2 and more."""
import numpy as np
import pytest

from test_gpu_parity import NTHREADS, TOL32, TOL64, rowfloor_err

pytestmark = pytest.mark.gpu

# nelem, periodic, distorted
CASES = [((1, 1, 1), 0, False), ((2, 1, 3), 0, True), ((3, 7, 2), 0, False), ((5, 2, 9), 0, True), ((9, 4, 5), 0, True),
         ((5, 7, 6), 1, False)]


def weights(mesh):
    """1 + 0.25 sin(0.9 i + 0.3) cos(0.7 j) + 0.05 k / (n - 1) at control point (i, j, k)"""
    i, j, k = np.indices(mesh.na)
    mesh.w[:] = (1 + 0.25 * np.sin(0.9 * i + 0.3) * np.cos(0.7 * j) + 0.05 * k / (mesh.na[2] - 1)).reshape(-1)


def build(igap, oracle, nelem, per, pert, torder):
    periodic = (per, per, per)
    mo = oracle.Mesh(nelem, L=(2, 1, 1.5), periodic=periodic, perturbed=pert)
    mg = igap.MeshIGABeam(nelem=nelem, L=(2, 1, 1.5), periodic=periodic, perturbed=pert)
    weights(mo)
    weights(mg)
    if per:
        pp = [0.01, 0.0, 0.02, 0.0, -0.01, 0.0, 0.005, 0.0, 0.004]
        bc_o, bc_g = oracle.make_bc(par_periodic=pp), igap.BC(par_periodic=pp)
    else:
        bc_o, bc_g = oracle.clamped_tip_bc(tip=0.02), igap.BCClampedTip(tip=0.02)
    ph_o, ph_g = oracle.make_phys(torder), igap.PhysGradElastTime() if torder else igap.PhysGradElast()
    U = oracle.glibc_rand_state((torder + 1) * mo.ndof) * 0.05
    return mo, mg, ph_o, ph_g, bc_o, bc_g, U


@pytest.mark.parametrize("torder", [0, 2])
@pytest.mark.parametrize("nelem, per, pert", CASES)
def test_residual(igap, oracle, nelem, per, pert, torder):
    mo, mg, ph_o, ph_g, bc_o, bc_g, U = build(igap, oracle, nelem, per, pert, torder)
    R_o = oracle.residual(mo, ph_o, bc_o, U, nthreads=NTHREADS)
    with igap.Assm(mg, ph_g, bc_g) as A:
        R = A.residual(U)
        free = A.dirichlet()[0] == 0
    # the free rows apart: the Dirichlet rows U - g are the larger ones
    err, err_free = rowfloor_err(R, R_o), rowfloor_err(R[free], R_o[free])
    print(f"{nelem} periodic {per} perturbed {pert} torder {torder}: {err:.2e}, free rows {err_free:.2e}")
    assert err < TOL64 and err_free < TOL64


@pytest.mark.parametrize("torder", [0, 2])
@pytest.mark.parametrize("nelem, per, pert", CASES)
def test_tangent(igap, oracle, nelem, per, pert, torder):
    from igap4_amd import _lib
    mo, mg, ph_o, ph_g, bc_o, bc_g, U = build(igap, oracle, nelem, per, pert, torder)
    rp_o, col_o, K_o = oracle.tangent(mo, ph_o, bc_o, U, nthreads=NTHREADS)
    for fl in [_lib.IGAP_TANGENT_ELEMENT_MATRICES] + ([] if per else [_lib.IGAP_TANGENT_DIRECT]):
        with igap.Assm(mg, ph_g, bc_g, flags=fl) as A:
            for prec, tol in (("f64", TOL64), ("f32", TOL32)):
                rp, col, K = A.tangent(U, prec=prec)
                assert np.array_equal(rp, rp_o) and np.array_equal(col, col_o)
                err = rowfloor_err(K, K_o, rp_o)
                print(f"{nelem} periodic {per} perturbed {pert} torder {torder} flags {fl} {prec}: {err:.2e}")
                assert err < tol
