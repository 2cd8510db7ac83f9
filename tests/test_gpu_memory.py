"""A context's device memory: at most 1500 bytes a ghosted cell for the nine
variables under SST and cavitation, dual time included, so that a grid that
has once fitted the device goes on fitting it."""
import gc

import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("nsteady", [0, 2])
def test_context_memory(pkg, nsteady):
    import torch
    torch.zeros(1, device="cuda")
    block = pkg.cases.bump_channel(128, 64, 64)
    case = pkg.cases.Case("memory", pkg.cases.bump_params(True, True, 4, 2, 8, nsteady=nsteady), [block], 9, 3, 5)
    pkg.Solver(case, metrics="device").close()          # what the runtime keeps from a first context is not the second's
    gc.collect()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    s = pkg.Solver(case, metrics="device")
    used = free - torch.cuda.mem_get_info()[0]
    s.close()
    ghosted = (block.imax + 5) * (block.jmax + 5) * (block.kmax + 5)
    assert 500 * ghosted < used <= 1500 * ghosted
