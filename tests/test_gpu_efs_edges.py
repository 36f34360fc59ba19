"""dEFSApply's kernel at the edges of its layout: every contracted length 1..12 in both directions, odd and even pitches,
components that fit at once and in several rounds, partly filled and single-element workgroups, results in place."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


def _reference(C, P, rc, jinv, D, x, amode):
    """Plain numpy (einsum over the 1-D tables of the oracle)."""
    B, Dm = O.tensor_basis(P, rc)[:2]
    Q, ne = len(rc), len(x)
    if amode == C.APPLY_INTERP:
        return np.einsum("ai,bj,ck,nijkd->nabcd", B, B, B, x.reshape(ne, P, P, P, D), optimize=True).reshape(ne, -1)
    if amode == C.APPLY_INTERP_TRANSPOSE:
        return np.einsum("ai,bj,ck,nabcd->nijkd", B, B, B, x.reshape(ne, Q, Q, Q, D), optimize=True).reshape(ne, -1)
    T = [(Dm, B, B), (B, Dm, B), (B, B, Dm)]
    J = None if jinv is None else jinv.reshape(ne, Q, Q, Q, 3, 3)
    if amode == C.APPLY_GRAD:
        f = np.stack([np.einsum("ai,bj,ck,nijkd->nabcd", *t, x.reshape(ne, P, P, P, D), optimize=True) for t in T], -1)
        return (f if J is None else np.einsum("nabcdm,nabcme->nabcde", f, J)).reshape(ne, -1)
    f = np.einsum("nabcde,nabcme->nabcdm", x.reshape(ne, Q, Q, Q, D, 3), J)
    return sum(np.einsum("ai,bj,ck,nabcd->nijkd", *t, f[..., m], optimize=True) for m, t in enumerate(T)).reshape(ne, -1)


CASES = [(2, 1, 1, 3), (2, 2, 1, 700), (3, 2, 2, 17), (4, 4, 1, 130), (5, 6, 3, 9), (6, 5, 1, 41), (7, 8, 2, 5), (8, 7, 1, 7),
         (9, 9, 5, 2), (10, 3, 4, 3), (11, 12, 1, 2), (12, 11, 2, 1), (12, 12, 3, 1), (3, 3, 70, 2), (2, 3, 130, 1)]


# Up to 3 * 12 products a pass, three passes: some 30 roundings of 1.1e-16 on values of order one: 1e-13 of the norm.
@pytest.mark.parametrize("P,Q,D,ne", CASES)
def test_apply_edges(C, P, Q, D, ne):
    rng = np.random.default_rng(100 * P + Q + D)
    rc = O.gauss_legendre(Q)[0]
    jn = rng.uniform(-1, 1, (ne, Q ** 3, 9))
    n, q = P ** 3 * D, Q ** 3 * D
    for amode, nin, nout in ((C.APPLY_INTERP, n, q), (C.APPLY_INTERP_TRANSPOSE, q, n), (C.APPLY_GRAD, n, 3 * q),
                             (C.APPLY_GRAD_TRANSPOSE, 3 * q, n)):
        for jinv in ((jn, None) if amode == C.APPLY_GRAD else (jn,)):
            print(f"efs P={P} Q={Q} D={D} ne={ne} amode={amode} jinv={jinv is not None}", flush=True)
            x, y0 = rng.uniform(-1, 1, (ne, nin)), rng.uniform(-1, 1, (ne, nout))
            ref = _reference(C, P, rc, jinv, D, x, amode)
            J = None if jinv is None else dev(jinv)
            for imode, want in ((C.INSERT_VALUES, ref), (C.ADD_VALUES, y0 + ref)):
                y = torch.cat([dev(y0).reshape(-1), torch.full((8,), 7.0, dtype=torch.float64, device="cuda")])
                C.efs_apply_hex_batched(P, rc, ne, J, D, dev(x), y, amode, imode)
                got = y[:-8].cpu().numpy().reshape(ne, nout)
                assert np.linalg.norm(got - want) <= 1e-13 * np.linalg.norm(want)
                assert bool((y[-8:] == 7.0).all())


@pytest.mark.parametrize("P,D,ne", [(4, 1, 33), (7, 2, 5)])
def test_interpolation_in_place(C, P, D, ne):
    rng = np.random.default_rng(P)
    rc = O.gauss_legendre(P)[0]
    x = dev(rng.uniform(-1, 1, (ne, P ** 3 * D)))
    y = torch.empty_like(x)
    C.efs_apply_hex_batched(P, rc, ne, None, D, x, y, C.APPLY_INTERP)
    C.efs_apply_hex_batched(P, rc, ne, None, D, x, x, C.APPLY_INTERP)
    assert torch.equal(x, y)


def test_captured_and_concurrent_calls(C):
    """Calls on several streams with different rules do not share tables; a captured call replays with its own."""
    rng = np.random.default_rng(3)
    jobs = []
    for P, Q in ((3, 4), (5, 5), (7, 6), (4, 8)):
        rc = O.gauss_legendre(Q)[0]
        x = dev(rng.uniform(-1, 1, (64, P ** 3)))
        ref = torch.empty(64, Q ** 3, dtype=torch.float64, device="cuda")
        C.efs_apply_hex_batched(P, rc, 64, None, 1, x, ref, C.APPLY_INTERP)
        jobs.append((P, rc, x, torch.zeros_like(ref), ref, torch.cuda.Stream()))
    torch.cuda.synchronize()
    for _ in range(20):
        for P, rc, x, y, ref, st in jobs:
            C.efs_apply_hex_batched_noalloc(P, rc, 64, None, 1, x, y, C.APPLY_INTERP, stream=st)
    torch.cuda.synchronize()
    for P, rc, x, y, ref, st in jobs:
        assert torch.equal(y, ref)
    P, rc, x, y, ref, st = jobs[0]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        C.efs_apply_hex_batched_noalloc(P, rc, 64, None, 1, x, y, C.APPLY_INTERP, stream=torch.cuda.current_stream())
    for k in range(3):
        y.zero_()
        C.efs_apply_hex_batched(5, jobs[1][1], 64, None, 1, jobs[1][2], jobs[1][3], C.APPLY_INTERP)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref), k


def test_physical_flags_do_not_outlive_their_call(C):
    """A negative or non-finite determinant is that call's error alone, from several threads and streams at once."""
    import threading

    w = np.array([5 / 9, 8 / 9, 5 / 9])
    out = []

    def calls(kind):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            jac = (torch.eye(3, dtype=torch.float64, device="cuda") * 0.5).expand(700, 3, 3, 3, 3, 3).contiguous()
            if kind == 1:
                jac[699, 2, 2, 2, 0, 0] = -0.5
            elif kind == 2:
                jac[0, 0, 0, 0, 0, 0] = float("nan")
            jinv, jw = torch.zeros_like(jac), torch.zeros(jac.shape[:4], dtype=torch.float64, device="cuda")
            st.synchronize()
            for _ in range(20):
                try:
                    C.rule_compute_physical_batched(w, 700, jac, jinv, jw)
                    out.append((kind, "ok"))
                except C.DohpError as e:
                    out.append((kind, "negative" if "egative" in str(e) else "finite" if "finite" in str(e) else str(e)))

    threads = [threading.Thread(target=calls, args=(k % 3,)) for k in range(12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(out) == 240 and set(out) == {(0, "ok"), (1, "negative"), (2, "finite")}
