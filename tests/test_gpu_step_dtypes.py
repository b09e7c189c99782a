"""The differentiated step on a state whose temperature is kept in another type:
only its halo is read, as float64, and the gradients are those of the float64
state with the same values."""
import pytest
import torch

import test_gpu_adjoint as TA

pytestmark = pytest.mark.gpu


def test_temperature_in_float32():
    from veros_amd.autodiff import mixing_step
    outs = []
    for dtype in (torch.float64, torch.float32):
        ds, p, w = TA._config4()
        vs = ds.variables
        T_tau = vs.temp[..., vs.tau].contiguous()
        vs.temp = vs.temp.to(torch.float32).to(dtype)
        leaf = [TA._t(getattr(p, n), True) for n in ("a", "b", "c", "d")]
        new = mixing_step(ds, *leaf, T_tau, vs.K_iso.clone())
        torch.sum(TA._t(w) * new).backward()
        outs.append([new.detach()] + [t.grad for t in leaf])
    # the scatter's atomics order the sums into the tracer's gradient, which reaches
    # none of these: every output is the same, bit for bit
    for a, b in zip(*outs):
        assert torch.equal(a, b)
