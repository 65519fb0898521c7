"""Workspaces allocated on first use when the device runs out of memory half way: the call
is refused, and a later call that has the memory is whole."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def test_adjoint_workspace_after_running_out(gpu):
    import torch

    from hyowon_amd import PMSolver
    from hyowon_amd.adjoint import pm_run
    N, L, n = 512, 512.0, 20000
    pos = clumpy_particles(n, L, 3)
    mom = np.random.default_rng(3).normal(0, 1.0, (3, n))

    def grad(s):
        x = [torch.as_tensor(p, device=gpu).requires_grad_() for p in pos]
        p = [torch.as_tensor(m, device=gpu, dtype=torch.float32) for m in mom]
        out = pm_run((*x, *p), s, 1.0, [0.01], [0.02], [0.01])
        sum((o.double() ** 2).sum() for o in out[:3]).backward()
        return [t.grad for t in x]

    ref = grad(PMSolver(L, N, precision="fp32", max_particles=n))
    s = PMSolver(L, N, precision="fp32", max_particles=n)
    # fill the device, then leave two and a half of the four meshes (0.5 GB each) of the workspace
    mesh = 4 * N ** 3
    hold = [torch.empty(torch.cuda.mem_get_info()[0] - 8 * mesh, dtype=torch.uint8, device=gpu)]
    with pytest.raises(torch.cuda.OutOfMemoryError):
        for _ in range(10000):
            hold.append(torch.empty(mesh // 2, dtype=torch.uint8, device=gpu))
    del hold[-5:]
    torch.cuda.empty_cache()
    with pytest.raises(Exception, match="out of memory"):
        grad(s)
    hold.clear()
    torch.cuda.empty_cache()
    for a, b in zip(grad(s), ref):
        assert torch.equal(a, b)
