"""The batch's fused CG launches at their edges: cases that end inside, at and
just past a 2048-row chunk, one-row and one-column cases, and iteration limits
inside, at and past a captured body.  Each case must give the bits of its own
run."""
import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from tests.cases import channel_model, config, same_bits

pytestmark = pytest.mark.gpu

SIZES = [(3, 3), (64, 32), (2, 1025), (60, 69), (64, 64), (1, 130), (130, 1)]


@pytest.mark.parametrize("itmax", [1, 2, 3, 9, 100])
@pytest.mark.parametrize("precision", [L.FP64, L.MIXED])
@pytest.mark.parametrize("precond", [F.DILU, F.Jacobi])
def test_batch_cg_edges(precond, precision, itmax):
    cfg = config(2, precision=precision, p_pre=precond, itmax=itmax)
    make = lambda: [channel_model(F.channel(nx, ny), nu=0.02) for nx, ny in SIZES]
    b = F.BatchSimulation(make(), cfg, [None] * len(SIZES))
    assert b.run(2) == 2
    for k, model in enumerate(make()):
        s = F.Simulation(model, cfg, None)
        assert s.run(2) == 2
        for name in ("Ux", "Uy", "p"):
            assert same_bits(b.get(name, k), s.get(name)), (SIZES[k], name)
        assert b.stats("p", k)["niter"] == s.stats("p")["niter"], SIZES[k]
