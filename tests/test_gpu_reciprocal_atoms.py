"""Reciprocal-space mode with exchange for motifs of more than ten atoms: the pair sums at Q of 66 and 136
pairs, past the 64 of one wave. Against the oracle's matrix, to the bar of the other reciprocal-mode tests."""
import numpy as np
import pytest

import oracle as O
from cases import gpu_context, oracle_case, rel_err

pytestmark = pytest.mark.gpu

FRACTIONAL = [(i / 4, j / 4) for i in range(4) for j in range(4)]


@pytest.mark.parametrize("natoms", [10, 11, 16])
def test_exchange_pairs(natoms, tmp_path):
    from xatu_amd import synthetic
    print(f"[reciprocal] {natoms} atoms", flush=True)
    path = str(synthetic.write_model(tmp_path / "m.model", natoms=natoms, orb_per_atom=1, fractional=FRACTIONAL[:natoms]))
    ex = oracle_case(path, 3, 1, 0, (1, 1, 10), exchange=True, Q=(0.05, 0.02, 0), cutoff=2)
    H = O.bse_reciprocal(ex, 3)
    no_exchange = oracle_case(path, 3, 1, 0, (1, 1, 10), Q=(0.05, 0.02, 0), cutoff=2)
    assert rel_err(O.bse_reciprocal(no_exchange, 3), H) > 1e-3  # the term is there to be seen
    ctx = gpu_context(ex, n_reciprocal=3)
    Hg = ctx.build(0, copy_out=True)
    ctx.close()
    assert rel_err(Hg, H) < 1e-10
    assert np.array_equal(Hg, Hg.conj().T)
