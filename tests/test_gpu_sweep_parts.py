"""The sweeps' split of a box into eight parts along J, and the FP16 sweeps against FP64 sweeps on the rounded operators
themselves: boxes below the split, at its first sizes (where the last parts are empty), and with parts that end inside a
tile."""
import numpy as np
import pytest
import torch

from test_gpu_sweeps import C, setup, vcycle  # noqa: F401

pytestmark = pytest.mark.gpu


def shifted(x, t, value=0.0):
    """x at the neighbour in direction t of every row."""
    i, j, k = t // 9, t // 3 % 3, t % 3
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1), value=value)
    return xp[i:i + x.shape[0], j:j + x.shape[1], k:k + x.shape[2]]


def half(x):
    """x rounded to halves at once (torch rounds to single precision in between, which moves near-ties)."""
    return torch.as_tensor(x.cpu().numpy().astype(np.float16).astype(np.float64), device=x.device)


def rounded(st):
    """The FP16 operator of a level as a 27-point stencil: scaled off-diagonals rounded, row sums kept.  A lower entry is
    the upper one of the lower neighbour's row (the two differ in the last bits, which can round to different halves)."""
    s = torch.sqrt(st[13]).float().double()
    a = torch.stack([st[t] if t >= 13 else shifted(st[26 - t], t) for t in range(27)])
    out = a.clone()
    for t in range(27):
        if t != 13:
            ss = s * shifted(s, t, 1.0)
            out[t] = ss * half(a[t] / ss)
            out[13] += a[t] - out[t]
    return out


def check(C, M, p, degree):  # noqa: F811
    print(f"FP16 V-cycle M={M} p={p} degree={degree}", flush=True)
    op, q1, mg, L = setup(C, M, p, 7, degree)
    assert abs(mg.lmax - L[0][1]) <= 1e-12 * L[0][1]
    g = torch.Generator(device="cuda").manual_seed(5)
    r = (torch.rand(q1.nrows, dtype=torch.float64, device="cuda", generator=g) * 2 - 1).float()
    shape = L[0][0].shape[1:]
    z = torch.full_like(r, float("nan"))
    z64 = torch.full_like(r, float("nan"), dtype=torch.float64)
    mg.apply(r.double(), z64)
    ref = vcycle(L, 0, degree, r.double().reshape(shape)).reshape(-1)
    assert float(torch.linalg.norm(z64 - ref)) <= 1e-12 * float(torch.linalg.norm(ref))
    R = [(rounded(st) if l + 1 < len(L) else st, lmax) for l, (st, lmax) in enumerate(L)]
    ref = vcycle(R, 0, degree, r.double().reshape(shape)).reshape(-1)
    mg.set_coefficients(True)
    for _ in range(3):  # eager, captured, replayed
        z.fill_(float("nan"))
        mg.apply_f32(r, z)
    err = z.double() - ref
    assert float(torch.linalg.norm(err)) <= 5e-5 * float(torch.linalg.norm(ref))
    assert float(err.abs().max()) <= 5e-5 * float(ref.abs().max())  # (no single row off, edges of the box included)


# Owned boxes (M p - 1 rows a side): lines along J 47 (one part), 49 and 51 (64 x 4 tiles split, the last part empty or
# nearly), 113 and 119 lines (64 x 8 tiles split), the last two from 1024 tiles on.  What separates the two sides is FP32
# rounding: about 30 roundings of 6e-8 per row and sweep, a dozen sweeps on each of up to five levels: 5e-5.
@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("M", [(3, 12, 5), (2, 25, 9), (5, 26, 3), (48, 57, 34), (27, 60, 65)])
def test_fp16_vcycle_on_the_rounded_operators(C, M, degree):  # noqa: F811
    check(C, M, 4 if M[1] == 12 else 2, degree)


# Two sweeps in one pass (FP64 from 600 k rows, FP16 from 800 k, degree 2; power iterations), or one FP16 sweep at degree 1
# (from 1.2 M): faces that end inside a workgroup's, one workgroup's face larger than the box's, few planes, columns from
# 49 to 68 and 129 rows; 67 x 95 x 95 = 604,675 rows takes FP64 pairs only.  Tolerances as above, lmax as the power
# iteration's in FP64.
@pytest.mark.parametrize("M,degree", [((8, 120, 120), 2), ((120, 8, 120), 2), ((120, 120, 8), 2), ((34, 48, 48), 2),
                                      ((25, 65, 65), 2), ((128, 65, 13), 2), ((54, 54, 54), 1), ((8, 150, 150), 1),
                                      ((150, 150, 8), 1)])
def test_paired_sweeps(C, M, degree):  # noqa: F811
    check(C, M, 2, degree)
