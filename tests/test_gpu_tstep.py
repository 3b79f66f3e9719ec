"""GPU parity of the Scarborough time-step statistics
(src/tstepper/mod_tstepper_scarborough.f90) against the oracle, which the
CPU tests pin to the compiled reference: bit for bit, host and device
arrays."""
import numpy as np
import pytest

from test_oracle_golden import _scarb_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 3), (70, 33), (258, 130), (1026, 514)])
def test_mean_cc_and_dt_match_oracle(gpu, orc, nx, ny):
    import torch

    from mach2d import tstep
    au, av, at, ap = _scarb_inputs(nx, ny, nx + ny)
    for a in (au, av, at, ap):
        want = orc.mean_cc(a, nx, ny)
        assert tstep.mean_cc(a, nx, ny) == want
        assert tstep.mean_cc(torch.tensor(a.reshape(-1), device="cuda"), nx, ny) == want
    rng = np.random.default_rng(2)
    J, u, v = (rng.uniform(0.5, 2.0, nx * ny), rng.uniform(-5, 5, nx * ny),
               rng.uniform(-5, 5, nx * ny))
    assert tstep.dt0(J, u, v, nx, ny) == orc.dt0_scarborough(J, u, v, nx, ny)
    c = max(orc.mean_cc(a, nx, ny) for a in (au, av, at, ap))
    dev = [torch.tensor(a.reshape(-1), device="cuda") for a in (au, av, at, ap)]
    for mincc, maxcc in ((2 * c, 4 * c), (0.5 * c, 2 * c), (0.1 * c, 0.5 * c)):
        want = orc.dt_scarborough(1.5e-3, au, av, at, ap, nx, ny, 0.25, mincc, maxcc)
        assert tstep.dt(1.5e-3, au, av, at, ap, nx, ny, 0.25, mincc, maxcc) == want
        assert tstep.dt(1.5e-3, *dev, nx, ny, 0.25, mincc, maxcc) == want


def _sum_patterns(n, rng):
    """Arrays of n terms at which a sum in parallel can part from the
    left-to-right loop: exact ties, zeros, numbers that leave the running
    sum's binade at every size, subnormals, negative and non-finite terms."""
    wide = 10.0 ** rng.uniform(-300, 300, n)
    grow = np.minimum(1.5 ** np.minimum(np.arange(n), 1500), 1e250)
    some = rng.uniform(0, 1, n)
    neg, late = rng.normal(size=n), rng.uniform(0, 1, n)
    late[n // 2:] *= -1.0
    nan, inf = some.copy(), some.copy()
    nan[n - 1], inf[n // 3] = np.nan, np.inf
    lead = some.copy()
    lead[: (3 * n) // 4] = 0.0
    lead[::7] = -0.0
    return {
        "uniform": some, "constant": np.full(n, 0.1), "integers": np.floor(some * 9.0),
        "halves": np.floor(some * 9.0) / 2.0 + 2.0 ** 52, "ties": rng.integers(0, 64, n) * 2.0 ** -10 + 2.0 ** -53,
        "few bits": some.astype(np.float32).astype(np.float64) * 2.0 ** rng.integers(-20, 20, n),
        "wide": wide, "grow": grow, "zeros": np.zeros(n), "leading zeros": lead,
        "subnormal": some * 1e-310, "overflow": np.full(n, 1e307), "signed": neg,
        "signed late": late, "nan": nan, "inf": inf,
    }


def _average(nx, ny, t):
    """get_average on the GPU of the terms t as the real volumes."""
    import torch

    from mach2d import assembly as A
    F = np.zeros((ny, nx))
    F[1:-1, 1:-1] = t.reshape(ny - 2, nx - 2)
    return F.reshape(-1), A.get_average(nx, ny, torch.tensor(F.reshape(-1), device="cuda"))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1535,
                               2047, 2048, 2049, 2560, 2561, 4095, 4096, 4097, 4608, 32768, 33291,
                               66049])
def test_in_order_sums_are_the_left_to_right_loop(gpu, orc, n):
    """get_average of n real volumes (nx = n + 2, ny = 3): the oracle's loop
    bit for bit, for sizes at the edges of the segments of 512 terms, on both
    sides of the one-launch range (2048), and for a last segment of one."""
    for name, t in _sum_patterns(n, np.random.default_rng(n)).items():
        F, got = _average(n + 2, 3, t)
        with np.errstate(over="ignore", invalid="ignore"):
            want = orc.get_average(n + 2, 3, F)
        assert np.array_equal(got, want, equal_nan=True), (name, got, want)


@pytest.mark.parametrize("nx,ny", [(1026, 514), (1027, 515), (2051, 515)])
def test_in_order_sums_beyond_the_staged_maps(gpu, orc, nx, ny):
    """524288 terms (1024 segments: all that the last kernel stages at once)
    and more: sums that leave their binade, stop at a bad term or meet ties in
    the first round of staged segments, at its end, and in a later round."""
    n = (nx - 2) * (ny - 2)
    rng = np.random.default_rng(n)
    base = rng.uniform(0, 1, n)
    edge = 1024 * 512                      # first term of the second round
    cases = {"uniform": base, "ties": rng.integers(0, 64, n) * 2.0 ** -10 + 2.0 ** -34,
             "zeros, then one": np.r_[np.zeros(n - 1), 1.0], "constant": np.full(n, 0.1)}
    for at in (700, edge - 1, edge, edge + 513, n - 1):
        if at < n:
            for name, v in (("negative", -0.25), ("nan", np.nan), ("inf", np.inf),
                            ("next binade", 3e6), ("far binade", 1e300)):
                cases["%s at %d" % (name, at)] = base.copy()
                cases["%s at %d" % (name, at)][at] = v
    for name, t in cases.items():
        F, got = _average(nx, ny, t)
        with np.errstate(over="ignore", invalid="ignore"):
            want = orc.get_average(nx, ny, F)
        assert np.array_equal(got, want, equal_nan=True), (name, got, want)
