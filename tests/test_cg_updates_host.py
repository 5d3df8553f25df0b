"""What the conjugate-gradient kernels take, and what goes to torch's operators (which refuse it where it is wrong)."""
import pytest

torch = pytest.importorskip("torch")


def test_results_of_apply_that_the_kernels_take():
    from flexspmv_amd.vectors import ConjugateGradientUpdates
    updates = ConjugateGradientUpdates(torch.zeros(6))
    ap, pap = torch.zeros(6), torch.zeros(1)
    assert updates.takes(ap, pap)
    assert updates.takes(ap, torch.zeros(3))                        # pap[0] is the scalar
    assert not updates.takes(ap.view(6, 1), pap)                    # (6, 1) does not broadcast into (6,)
    assert not updates.takes(ap, torch.tensor(0.0))                 # no pap[0]
    assert not updates.takes(ap, torch.zeros(1, 6))                 # pap[0] is no scalar
    assert not updates.takes(torch.zeros(12)[::2], pap)
    assert not updates.takes(ap.double(), pap)
    assert not updates.takes(ap.clone().requires_grad_(), pap)      # autograd records torch's operators only
    assert not updates.takes(ap, pap.clone().requires_grad_())
