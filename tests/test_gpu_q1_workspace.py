"""The workspace of the embedded-Q1 assembly: one per operator, whatever the number of its matrices, and taken in turn by
assemblies on different streams."""
import gc

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


def test_matrices_of_one_operator_share_it(C):
    M, p = (48, 64, 64), 2  # 288 bytes per sub-cell: three passes of up to 192 MiB
    fs = C.FS(M, p, block_vertices(M))
    op = C.Ellip(fs, p=2.0)

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    gc.collect()
    torch.cuda.empty_cache()
    at = [used()]
    mats = []
    for _ in range(3):
        mats.append(op.assemble_q1())
        at.append(used())
    first, second, third = (b - a for a, b in zip(at, at[1:]))
    layer = 288 * (2 * 64) ** 2 * 2
    assert first - second >= 20 * layer  # (21 layers of elements fit in 192 MiB)
    assert abs(third - second) <= layer


def test_two_streams_take_it_in_turn(C):
    """Two matrices of one operator on two streams, the first behind other work; both are those of assemblies by turns."""
    M, p = (4, 5, 3), 4
    fs = C.FS(M, p, block_vertices(M, perturb=0.05, seed=2))
    op = C.Ellip(fs, p=2.0)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    mats, ref = [], []
    for mode in (0, 1):
        op.set_q1_mode(mode)
        mats.append(op.assemble_q1())
        torch.cuda.synchronize()
        ref.append(mats[-1].to_scipy())
    w = torch.randn(4096, 4096, device="cuda")
    for _ in range(3):
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            for _ in range(20):
                w = torch.tanh(w @ w)
        for mode, s in ((0, a), (1, b)):
            op.set_q1_mode(mode)
            op.assemble_q1(mat=mats[mode], stream=s)
        torch.cuda.synchronize()
        for mode in (0, 1):
            assert abs(mats[mode].to_scipy() - ref[mode]).max() == 0, mode
