"""The sum-factorised kernels of equal weights against the kernels of rational
patches on full patches.  For the static physics IGAP_GENERAL_GEOMETRY compares two
users of one contraction (k_tangent_sep and k_tangent_gen run the same z, y and x
stages, write-out and 1-D tables), and a distorted patch with k_tangent_gen either
way; the independent path is the matrix-core kernel k_tangent_elem."""
import numpy as np
import pytest

from test_gpu_parity import TOL32, TOL64, rowfloor_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pert", [False, True])
def test_sum_factorised_vs_matrix_core_full_patch(igap, pert):
    """64x16x16 beam: one control weight an ulp above the others' 1 makes the patch
    rational, so that its tangent is k_tangent_elem's and its residual
    k_residual_gen<1, true>'s, while no entry changes by more than a few roundings
    (the weight's relative change is 2e-16).  Every entry of k_tangent_sep (or, on the
    distorted patch, k_tangent_gen), which share their contraction with each other but
    not with the matrix-core kernel, against it.  The free rows of a smooth field's residual are
    what the elements' contributions leave of each other, about 1e-3 of them: 1e-14 of
    a contribution is 1e-11 of a row."""
    kw = dict(L=(4, 1, 1), nelem=(64, 16, 16), perturbed=pert)
    mesh, ulp = igap.MeshIGABeam(**kw), igap.MeshIGABeam(**kw)
    assert np.all(mesh.w == 1.0)
    ulp.w[ulp.w.size // 2] = np.nextafter(1.0, 2.0)
    U = igap.smooth_state(mesh, amp=0.02)
    ph, bc = igap.PhysGradElast(coef=igap.SVK_COEF), igap.BCClampedTip(tip=0.05)
    out = []
    for m in (mesh, ulp):
        with igap.Assm(m, ph, bc) as A:
            R = A.residual(U)[A.dirichlet()[0] == 0]
            rp, _, k64 = A.tangent(U)
            _, _, k32 = A.tangent(U, prec="f32")
        out.append((R, k64, k32))
    (R, k64, k32), (Rm, m64, m32) = out
    assert not np.array_equal(k64, m64) and not np.array_equal(k32, m32)   # two kernels
    eR, e64, e32, em = rowfloor_err(R, Rm), rowfloor_err(k64, m64, rp), rowfloor_err(k32, m64, rp), rowfloor_err(m32, m64, rp)
    print(f"perturbed {pert}: residual {eR:.2e}, FP64 {e64:.2e}, FP32 {e32:.2e}, matrix-core FP32 {em:.2e}")
    assert eR < 1e-11 and e64 < TOL64 and e32 < TOL32 and em < TOL32
