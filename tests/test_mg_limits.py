"""Limits of the multigrid set-up: the workspace of the power iterations over all shapes of levels (host arithmetic, no
GPU), and boxes that cannot be coarsened far enough, which are refused."""
import ctypes
import random

import pytest

torch = pytest.importorskip("torch")  # (before the library: one HIP runtime in the process)
C = pytest.importorskip("dohp_amd.capi")


def _sums(box):
    places, single, pair = ctypes.c_long(), ctypes.c_long(), ctypes.c_long()
    assert C.lib().dohpMGPowerSums_Private(*box, ctypes.byref(places), ctypes.byref(single), ctypes.byref(pair)) == 0
    return places.value, single.value, pair.value


def _boxes():
    rng = random.Random(17)
    yield from ((2, 800, 800), (2, 1441, 1383), (2, 4000, 4000), (191, 191, 191), (95, 95, 95), (3, 700, 700))
    for _ in range(100000):
        nx = rng.choice((1, 2, 3, 4, 7, 8, 9, 16, 33, 100, 400))
        ny = int(2 ** rng.uniform(0, 12.5))
        nz = int(2 ** rng.uniform(0, 12.5))
        if nx * ny * nz < 2 ** 31:
            yield rng.choice(((nx, ny, nz), (ny, nx, nz), (ny, nz, nx)))


def test_power_iteration_sums_fit_their_workspace():
    more = 0
    for box in _boxes():
        places, single, pair = _sums(box)
        assert places >= 256 and places >= single and places >= pair, box
        more += pair > max(256, single)
    assert more > 0  # (boxes on which the pairs' sums are the larger ones are among them)


@pytest.mark.gpu
def test_plate_is_refused():
    """2 x 800 x 800 rows: one coarsening leaves 160,000 rows, too many for the direct solve."""
    from dohp_amd.mesh import block_vertices
    M = (1, 267, 267)
    fs = C.FS(M, 3, block_vertices(M))
    assert fs.nowned == 2 * 800 * 800
    op = C.Ellip(fs, p=2.0)
    q1 = op.assemble_q1()
    for _ in range(2):
        with pytest.raises(C.DohpError) as ei:
            C.MG(q1)
        assert ei.value.code == C.ERR_ARG and "too large for a direct solve" in str(ei.value)
    x = torch.ones(fs.nowned, dtype=torch.float64, device="cuda")
    y = torch.zeros_like(x)
    q1.mult(x, y)
    assert torch.isfinite(y).all()
