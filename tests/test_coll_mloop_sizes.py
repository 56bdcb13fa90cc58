"""The collocation method's m-loop at the sizes and options where its loads
ahead, its thread groups and its tables take another form: fewer rows than
columns loaded ahead (8 to 13 and 16, 17), one and several rows a thread,
register and Stockham FFTs, tables in LDS and in L2 (n_r 97 and 256); T alone,
xi alone and both; every slot of SBDF4 and the stage sums of ARS443; the
coupled and the influence-matrix solve.  One and six steps against the oracle,
each field within ten times what one rounding of the initial state moves the
oracle's own result (its conditioning), and at least 1e-11; above n_r 97 that
grows as n_r^4 in the first step, as the condition of the second-derivative
collocation matrices does, whose inverses two implementations round
differently (n_r 256: 4.9e-10).  In each further step the residual of an
explicit inverse, which an LU solve does not leave, comes in once more, so the
difference grows in proportion to the steps: at n_r 256 the elimination with
row swaps that this one replaced was 2.3e-9, 1.0e-8 and 1.8e-8 away after two,
four and six steps (u_phi; 2.0e-9, 6.0e-9 and 1.1e-8 with this one), and the
bound for six steps is four times its 1.8e-8."""
import pytest

from helpers import rel
from test_gpu_parity import _fields, _floor, _pair

pytestmark = pytest.mark.gpu

CASES = [  # n_r, scheme, ra, raxi, buoyancy, pumping, solve
    (8, "CNAB2", 1e5, 1e5, "IMP", True, "direct"),
    (9, "SBDF2", 1e5, 0.0, "IMP", True, "direct"),
    (9, "CNAB2", 1e5, 1e5, "EXP", True, "direct"),
    (10, "SBDF2", 1e5, 0.0, "IMP", True, "direct"),
    (11, "SBDF3", 1e5, 0.0, "IMP", True, "direct"),
    (12, "SBDF4", 1e5, 0.0, "IMP", False, "direct"),
    (13, "ARS443", 0.0, 1e5, "EXP", True, "direct"),
    (16, "CNLF", 1e5, 1e5, "EXP", True, "influence"),
    (17, "SBDF3", 1e6, 0.0, "EXP", True, "direct"),
    (33, "SBDF4", 1e6, 1e6, "IMP", True, "direct"),
    (33, "ARS443", 1e6, 1e6, "IMP", False, "direct"),
    (48, "ARS222", 0.0, 1e6, "IMP", True, "influence"),
    (65, "SBDF2", 1e6, 0.0, "IMP", True, "direct"),
    (97, "BPR353", 1e6, 1e6, "EXP", True, "direct"),
    (256, "CNAB2", 1e6, 1e6, "IMP", True, "direct"),
]


@pytest.mark.parametrize("n_r,scheme,ra,raxi,buo,pump,solve", CASES)
def test_coll_mloop_sizes(n_r, scheme, ra, raxi, buo, pump, solve):
    from pizza_amd import workloads as W
    from pizza_amd.config import default_config
    cfg = default_config(n_r_max=n_r, n_cheb_max=n_r, m_max=6, time_scheme=scheme, cheb_method="colloc",
                         matrix_solve=solve, buo_term=buo, dtMax=1.0e-6, ra=ra, raxi=raxi, sc=3.0, ek=1.0e-4, pr=1.0,
                         radratio=0.35, l_ek_pump=pump)
    print(f"case: collocation m-loop n_r {n_r} {scheme} {solve}", flush=True)
    seed = lambda x: W.seed_run(x, cfg, amp_t=1.0e-3, amp_xi=1.0e-3)  # noqa: E731
    floors = _floor(cfg, [1, 6], seed)
    g, o = _pair(cfg)
    for x in (g, o):
        seed(x)
        x.start()
    least = (1e-11, 1e-11) if n_r <= 97 else (1e-11 * (n_r / 97) ** 4, 7.2e-8)
    for i, n in enumerate((1, 5)):
        g.step(n)
        o.step(n)
        for f in _fields(cfg):
            err = rel(g.get_field(f), o.get_field(f))
            assert err < max(least[i], 10 * floors[i][f]), (f, i, err, floors[i][f])
