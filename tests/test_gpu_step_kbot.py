"""kbot changed in place between the differentiated step's forward and backward
passes: the gradients are those of the forward pass's kbot."""
import pytest
import torch

import test_gpu_adjoint as TA
from conftest import rel_err

pytestmark = pytest.mark.gpu


def test_kbot_changed_before_backward():
    from veros_amd.autodiff import mixing_step
    grads = []
    for change in (False, True):
        ds, p, w = TA._config4()
        vs = ds.variables
        vs.kbot = vs.kbot.to(torch.int32)
        leaf = [TA._t(getattr(p, n), True) for n in ("a", "b", "c", "d")]
        new = mixing_step(ds, *leaf, vs.temp[..., vs.tau].contiguous(), vs.K_iso.clone())
        if change:
            keep = vs.kbot.clone()
            vs.kbot.zero_()
            vs.kbot.copy_(keep)
        torch.sum(TA._t(w) * new).backward()
        grads.append([t.grad for t in leaf])
    for a, b in zip(*grads):
        assert rel_err(b.cpu().numpy(), a.cpu().numpy()) <= 1e-13
