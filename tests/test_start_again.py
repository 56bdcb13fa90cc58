"""A run started again with other fields goes on as a new run does, bit for
bit: the captured step is kept from the first start, with another history
behind it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method,scheme", [("integ", "BPR353"), ("colloc", "SBDF4"), ("fd", "CNAB2"), ("fd", "ARS343")])
def test_start_again(method, scheme):
    from pizza_amd import workloads as W
    from pizza_amd.config import default_config
    from pizza_amd.runtime import Run
    kw = dict(radial_scheme="FD") if method == "fd" else dict(cheb_method=method, matrix_solve="direct")
    cfg = default_config(n_r_max=33, n_cheb_max=33, m_max=8, time_scheme=scheme, dtMax=1.0e-6, ra=1.0e6, raxi=1.0e6,
                         sc=3.0, ek=1.0e-4, pr=1.0, radratio=0.35, **kw)
    print(f"case: second start {method} {scheme}", flush=True)

    def go(r, amp, steps):
        for f in ("us", "up", "om", "psi"):
            r.set_field(f, np.zeros((r.n_m, 33), complex))
        W.seed_run(r, cfg, amp_t=amp, amp_xi=amp)
        r.start()
        r.step(1)
        r.step(steps - 1)
        return [r.get_field(f).copy() for f in ("temp", "xi", "us", "up", "om")]

    again, new = Run(cfg), Run(cfg)
    go(again, 1.0e-1, 7)
    a, b = go(again, 1.0e-3, 5), go(new, 1.0e-3, 5)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
