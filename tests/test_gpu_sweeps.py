"""The single-system sweeps at the edges of their bands (64 rows), chunks (8
and 16 steps), LDS rings (5 chunks, 256 columns) and placements: fed sweeps
where four times the bands have CUs of their own (64 bands on consecutive
XCDs, 8 on one XCD, of 256 CUs), register sweeps above.  FP64 iterates equal
the oracle's bit for bit; FP32 solves equal those of the LDS-staged sweeps,
whose arithmetic is the same."""
import numpy as np
import pytest

from mach2d import problems as P

pytestmark = pytest.mark.gpu


def _system(nx, ny, nd):
    s = P.random_f3_system(nx, ny, seed=nx + 3 * ny)
    if nd == 5:
        s.a = np.ascontiguousarray(s.a[[1, 3, 4, 5, 7]])
    return s


def _solve(gpu, s, nd, prec, nitm, stride=None, staged=False):
    import torch
    dev = gpu.DeviceMSI(s.nx, s.ny, prec, ndiag=nd)
    if stride:
        dev.set_tuning(32, stride)
    dev.set_staging(staged)
    a = torch.tensor(s.a.reshape(-1), device="cuda")
    b = torch.tensor(s.rhs, device="cuda")
    x = torch.zeros(s.N, dtype=torch.float64, device="cuda")
    dev.factor(a)
    st = dev.solve(a, b, x, 0.0, nitm)
    assert st.status == 0
    dev.close()
    return x.cpu().numpy()


@pytest.mark.parametrize("nd", [9, 5])
@pytest.mark.parametrize("nx,ny", [(3, 3), (5, 64), (4, 65), (8, 66), (9, 127), (129, 128),
                                   (600, 63), (131, 193), (40, 577)])
def test_fp64_bitwise(gpu, orc, nx, ny, nd):
    s = _system(nx, ny, nd)
    lu, fb = (orc.lu2d9, orc.fb2d9) if nd == 9 else (orc.lu2d5, orc.fb2d5)
    dl, du = lu(s.a, nx, ny)
    ox = fb(s.a, dl, du, nx, ny, np.zeros(s.N), 0.0, 5, s.rhs)[0]
    for stride in (1, 8):
        assert np.array_equal(_solve(gpu, s, nd, "fp64", 5, stride), ox), stride


@pytest.mark.parametrize("ny", [4096, 4097, 4163])
def test_many_bands(gpu, orc, ny):
    """64 bands, the most that take the fed sweeps, and 65 and 66 (one and
    three rows into the last band), which take the register sweeps."""
    nx = 6
    s = _system(nx, ny, 9)
    dl, du = orc.lu2d9(s.a, nx, ny)
    ox = orc.fb2d9(s.a, dl, du, nx, ny, np.zeros(s.N), 0.0, 3, s.rhs)[0]
    assert np.array_equal(_solve(gpu, s, 9, "fp64", 3), ox)


@pytest.mark.parametrize("nd", [9, 5])
@pytest.mark.parametrize("nx,ny", [(3, 3), (17, 65), (33, 129), (300, 130), (40, 577)])
def test_fp32_equals_staged(gpu, nx, ny, nd):
    s = _system(nx, ny, nd)
    ref = _solve(gpu, s, nd, "fp32_ir", 2, staged=True)
    for stride in (1, 8):
        assert np.array_equal(_solve(gpu, s, nd, "fp32_ir", 2, stride), ref), stride
