"""The two-level step's grouped explosion and its ghost stream (rings 1 and 2;
with three ghost layers ring-3 sources are read as the sentinel, with four
they are streamed), against the oracle: small boxes whose rings overlap, wrap
around the domain and share parents.  The same FP64 operations in the same
order on both sides, so the values are equal."""
import numpy as np
import pytest

from amr_cases import oracle_hierarchy, small_amr, with_sphere_across_fine_edge

pytestmark = pytest.mark.gpu

CASES = {
    "overlapping_rings": lambda: small_amr(n=16, nbox=40, seed=11, fraction=0.25),
    "sphere": lambda: with_sphere_across_fine_edge(small_amr(n=16, nbox=30, seed=7, fraction=0.3)),
}


@pytest.mark.parametrize("ng", [3, 4])
@pytest.mark.parametrize("case", sorted(CASES))
def test_advance_then_coalesce_equals_oracle(oracle, engine, case, ng):
    cfg = CASES[case]()
    C, F = oracle_hierarchy(cfg, ng=ng)
    H = engine.Hierarchy(cfg, ng=ng)
    oracle.amr_evolve(C, F, 3)
    H.advance(3)
    # the coalescence reads the fine ghosts of rings 1 and 2 as the second
    # substep left them
    for lattice in (0, 1):
        oracle.amr_coalesce(F, C, lattice)
    H.coalesce()
    for name in ("f", "g"):
        for E, O in ((H.crse, C), (H.fine, F)):
            assert np.array_equal(E.valid(name), O.valid(name)), (case, ng, name)
    H.close()
