"""The warm start on time steps (gradelasttime, the 8-mode initial velocity): the
whole driver on a small beam, every arm to the plain path's answer."""
import pytest

pytestmark = pytest.mark.gpu


def test_time_steps_of_every_arm(igap):
    """12 steps, the network trained on the first 8.  Each step of each arm is solved to
    1e-10 of its first residual; the displacements of a step follow from the
    inertia-dominated operator (rho / dt^2 against the stiffness: condition about
    1e3), so the arms agree within 4 x 1e-10 x 1e3 at most."""
    from igap4_amd import warmstart
    s = warmstart.run_transient(nelem=(8, 4, 4), nsteps=12, ntrain=8, epochs=4, prec="f64", verbose=False)
    assert isinstance(s["correction_used"], bool)
    for arm in ("plain", "linear", "quadratic", "learned"):
        print(arm, s[arm])
        assert s[arm]["all_converged"] and s[arm]["steps"] == 4
        assert s[arm]["final_rel_diff_vs_plain"] < 4e-7
