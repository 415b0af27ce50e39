"""Contexts next to each other in one process: what one is told, or runs into, does
not change another's results."""

import numpy as np
import pytest

from cc4s_amd import api
from cc4s_amd import synthetic as syn
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("generation", ["1", "2"])
def test_kernel_generation_belongs_to_a_context(generation, monkeypatch):
    """The first context has plans whose last tiles are cut along K, which the kernel
    of the other generation does not know; at these sizes the ring products' are."""
    No, Nv, NG = 18, 60, 90
    print(f"kernel generation {generation}", flush=True)
    inp = syn.generate(No, Nv, NG, "complex", 5)
    T = syn.random_amplitudes(No, Nv, "complex", 6, t1_scale=0.05, t2_scale=0.05)

    def context():
        cc = api.CoupledCluster(No, Nv, NG, field="complex")
        cc.set_inputs(inp.gamma, inp.eps)
        return cc

    monkeypatch.delenv("CC4S_GETT_GENERATION", raising=False)
    with context() as first:
        R = first.residuum(T)
        monkeypatch.setenv("CC4S_GETT_GENERATION", generation)
        with context() as other:
            S = other.residuum(T)
        for r, s, again in zip(R, S, first.residuum(T)):
            assert rel_err(s, r) < 1e-12  # FP64 sums in another order, as for one residuum
            assert np.array_equal(again, r)
        monkeypatch.delenv("CC4S_GETT_GENERATION")
        with context() as last:
            assert all(np.array_equal(x, r) for x, r in zip(last.residuum(T), R))
