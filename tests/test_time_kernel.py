"""pz_time_kernel(0) of a finite-difference run times the m-loop alone: a
rebuild that the last step needed is not part of the repetitions, and the
state behind the call is the one before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_timed_m_loop_does_not_rebuild():
    from pizza_amd import workloads as W
    from pizza_amd.runtime import Run
    print("case: m-loop timing after a rebuild, n_r 257", flush=True)
    cfg = W.c5_fd(n_r=257, m_max=66)
    timed, plain = Run(cfg), Run(cfg)
    for r in (timed, plain):
        W.seed_run(r, cfg)
        r.start()
        r.step(1)  # the first step builds the matrices
    after_rebuild = min(timed.time_kernel(0, 50) for _ in range(3))
    for r in (timed, plain):
        r.step(5)  # the last ones do not
    without = min(timed.time_kernel(0, 50) for _ in range(3))
    for f in ("temp", "us", "up", "om"):
        assert np.array_equal(timed.get_field(f), plain.get_field(f)), f
    # a rebuild makes a launch about three times as long
    assert after_rebuild < 1.5 * without, (after_rebuild, without)
