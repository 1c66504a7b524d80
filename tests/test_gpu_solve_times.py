"""The product time that a solve reports is the products' own time on the device: not above that of the same
product between two events (which wait for each other's kernels and so include a little more), at a dimension
where an iteration's other parts, the host's among them, would show. Both as the least of several runs; 2 us for
the clock's steps (10 ns) and the launches' scatter."""
import numpy as np
import pytest

from cases import MODELS, gpu_context, oracle_case

pytestmark = pytest.mark.gpu


def test_product_time():
    ex = oracle_case(MODELS / "hBN.model", 30, 1, 0, (1, 1, 10), cutoff=20, exchange=True)
    print(f"[solve times] N {ex.N}", flush=True)
    ctx = gpu_context(ex)
    ctx.build(0)
    solve = []
    for _ in range(6):
        _, _, rep = ctx.solve(nstates=8, precision=0, block=16, tol=1e-7, want_vectors=False)
        solve.append(rep.ms_products / (rep.products / 16))
    x = np.random.default_rng(0).normal(size=(ex.N, 16)) + 0j
    alone = []
    for _ in range(12):
        before = ctx.timings().ms_matvec_kernel
        ctx.matvec(x)
        alone.append(ctx.timings().ms_matvec_kernel - before)
    ctx.close()
    print(f"[solve times] in the solve {min(solve) * 1e3:.1f} us, alone {min(alone) * 1e3:.1f} us", flush=True)
    assert 0.25 * min(alone) < min(solve) < min(alone) + 2e-3
