"""The TDMA line chains at the edges of their operand chunks (512 / R steps,
R = 64 .. 4 lines a workgroup, chosen by the line's length): lines one step
shorter, equal and one longer than whole chunks and groups of four steps, in
both passes, equal to the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 5, 7, 8, 9, 12, 13, 16, 17, 255, 256, 257, 272, 273, 575, 577,
                               1023, 1025, 2048])
@pytest.mark.parametrize("x_lines", [True, False])
def test_chunk_edges(gpu, orc, n, x_lines):
    nx, ny = (n, 5) if x_lines else (5, n)
    rng = np.random.default_rng(n)
    a = -rng.uniform(0.05, 1.0, size=(9, nx * ny))
    a[4] = 1.5 * np.sum(np.abs(a[[0, 1, 2, 3, 5, 6, 7, 8]]), axis=0) + 0.1
    b = rng.normal(size=nx * ny)
    x = rng.normal(size=nx * ny)
    ref = orc.tdma2d9(a, b, x, nx, ny, 2)
    got = x.copy()
    gpu.tdma2d9(nx, ny, 2, a, b, got)
    assert np.array_equal(got, ref)
