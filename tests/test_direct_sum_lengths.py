"""Collocation runs whose Chebyshev transforms are direct sums (2 (n_r - 1)
with a prime factor above 64) and whose mean flow is not zero, so that the
implicit term of u_phi(m = 0) - two transforms back to the grid - counts:
after the start, in the step (multistep and stages) and in the assembly
stage.  Six steps against the oracle, each field within ten times what one
rounding of the initial state moves the oracle's own result, and at least
1e-11; and the same bits from a second run."""
import numpy as np
import pytest

from helpers import rel
from test_gpu_parity import _fields, _floor, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_r,scheme,solve", [(68, "CNAB2", "direct"), (80, "SBDF3", "influence"), (72, "ARS343", "direct")])
def test_mean_flow_at_direct_sum_lengths(n_r, scheme, solve):
    from pizza_amd import workloads as W
    from pizza_amd.config import default_config
    from pizza_amd.runtime import Run
    cfg = default_config(n_r_max=n_r, n_cheb_max=n_r, m_max=6, time_scheme=scheme, cheb_method="colloc",
                         matrix_solve=solve, dtMax=1.0e-6, ra=1.0e6, ek=1.0e-4, pr=1.0, radratio=0.35, l_ek_pump=True)
    print(f"case: mean flow at n_r {n_r} {scheme} {solve}", flush=True)

    def seed(x):
        W.seed_run(x, cfg, amp_t=1.0e-3, amp_xi=0.0)
        x.init_fields(init_u=-1, amp_u=10.0)

    floors = _floor(cfg, [6], seed)
    g, o = _pair(cfg)
    again = Run(cfg)
    for x in (g, o, again):
        seed(x)
        x.start()
        x.step(6)
    for f in _fields(cfg):
        a, b = g.get_field(f), o.get_field(f)
        assert rel(a, b) < max(1e-11, 10 * floors[0][f]), f
        if f in ("up", "om"):  # the mean flow by itself
            assert np.abs(b[0]).max() > 1.0
            assert rel(a[0], b[0]) < max(1e-11, 10 * floors[0][f]), f
        assert np.array_equal(a, again.get_field(f)), f
