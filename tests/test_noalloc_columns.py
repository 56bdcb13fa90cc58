"""pz_get_ddr_noalloc against pz_get_ddr, bit for bit, over the numbers of
columns that a workgroup takes (one, two, four, with a short last group and
with tiles that do not divide by the eight chiplets), register, Stockham and
direct-sum transform lengths; written over its own input; and two handles of
one process at once, whose results must not depend on each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(n_r):
    from pizza_amd.config import default_config
    from pizza_amd.runtime import Run
    return Run(default_config(n_r_max=n_r, n_cheb_max=n_r, m_max=6, radratio=0.35, cheb_method="colloc",
                              matrix_solve="direct"))


def _field(rng, n_m, n_r):
    return rng.standard_normal((n_m, n_r)) + 1j * rng.standard_normal((n_m, n_r))


def _call(run, d_f, d_1, d_2, n_m, dct):
    from pizza_amd.runtime import lib
    rc = lib().pz_get_ddr_noalloc(run.h, d_f.data_ptr(), d_1.data_ptr(), d_2.data_ptr() if d_2 is not None else None, n_m, dct)
    assert rc == 0, lib().pz_last_error(run.h)


@pytest.mark.parametrize("n_r,n_m,dct,second", [
    (33, 1, 1, True), (33, 1025, 1, True), (33, 1030, 0, False), (65, 513, 1, True), (80, 515, 1, True), (97, 1027, 1, False),
    (193, 1358, 1, True), (193, 511, 0, True), (257, 520, 1, True)])
def test_noalloc_columns(n_r, n_m, dct, second):
    import torch
    print(f"case: noalloc derivative n_r {n_r}, {n_m} columns", flush=True)
    run, f = _run(min(n_r, 256)) if n_r < 257 else None, _field(np.random.default_rng(5), n_m, n_r)
    if run is None:  # the longest grid belongs to finite differences
        from pizza_amd import workloads as W
        from pizza_amd.runtime import Run
        run = Run(W.c5_fd(n_r=257, m_max=6))
    want = run.get_ddr(f, bool(dct)) if second else (run.get_dr(f, bool(dct)),)
    x = torch.from_numpy(np.ascontiguousarray(f.T)).cuda()
    out = [torch.zeros_like(x) for _ in want]
    torch.cuda.synchronize()
    _call(run, x, out[0], out[1] if second else None, n_m, dct)
    torch.cuda.synchronize()
    for o, w in zip(out, want):
        assert np.array_equal(o.cpu().numpy().T, w)
    _call(run, x, x, out[1] if second else None, n_m, dct)  # in place
    torch.cuda.synchronize()
    assert np.array_equal(x.cpu().numpy().T, want[0])


def test_noalloc_two_handles_at_once():
    import torch
    print("case: noalloc derivative, two handles", flush=True)
    rng = np.random.default_rng(6)
    runs, fs = [_run(97), _run(193)], [_field(rng, 2000, 97), _field(rng, 1300, 193)]
    want = [r.get_ddr(f, True) for r, f in zip(runs, fs)]
    xs = [torch.from_numpy(np.ascontiguousarray(f.T)).cuda() for f in fs]
    outs = [(torch.zeros_like(x), torch.zeros_like(x)) for x in xs]
    torch.cuda.synchronize()
    for _ in range(20):
        for r, f, x, o in zip(runs, fs, xs, outs):
            _call(r, x, o[0], o[1], f.shape[0], 1)
    torch.cuda.synchronize()
    for o, w in zip(outs, want):
        assert np.array_equal(o[0].cpu().numpy().T, w[0]) and np.array_equal(o[1].cpu().numpy().T, w[1])
