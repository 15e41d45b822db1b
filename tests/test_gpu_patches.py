"""One step per launch: the 8 x 8 patches that the layout cuts out of uniform
parts of a mesh, at sizes where their number and their rings change, against
the CPU oracle (the parity gates) and, bit for bit, against launches of
several steps."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {0: 1e-12, 1: 1e-5}   # FP64 against the oracle, FP32C likewise


def layer(cases, nx, nz, het):
    """nx x nz cells of 5 m; het: (lambda, mu) of its own in every element."""
    w, h = 5.0 * nx, 5.0 * nz
    text = cases.problem_text(w, h, 0.4, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                              [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.2, 0.2, 1.0, 5.0])
    case = cases.S.case_from_problem_text(text, sheet=(-3.3, w - 10.0, 4.1), name="layer")
    return cases.perturbed(case, seed=nx + nz) if het else case


# no patch (8 x 8 nodes are never all interior below 10 cells), one, several in
# a row, cells cut by the sides, more patches than a workgroup holds
@pytest.mark.parametrize("nx,nz", [(12, 7), (17, 17), (24, 16), (40, 33), (70, 50)])
@pytest.mark.parametrize("het", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
def test_patches(nx, nz, het, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    case = layer(cases, nx, nz, het)
    n = 120   # the pulse is inside the layer
    u_o, up_o, _, rec_o = O.run(case, nsteps=n, recv_interval=1)
    ref = None
    for tuning in ((128, 1, 0, 3), (64, 0, 0, 1), (64, 1, 12, 1), (256, 1, 0, 1)):
        print(f"nx={nx} nz={nz} het={het} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        s.set_tuning(*tuning)
        rec = s.run(n)
        u, up, _ = s.state()
        s.close()
        if ref is None:
            ref = (rec, u, up)
            assert np.abs(u_o).max() > 1e-3, "case must carry signal"
            for got, want in ((rec, rec_o), (u, u_o), (up, up_o)):
                assert rel_l2(got, want) <= TOL[prec]
        for got, want in zip((rec, u, up), ref):
            assert np.array_equal(got, want)


@pytest.mark.parametrize("prec", [0, 1])
def test_state_across_layouts(prec):
    """Layouts of one and of several steps per launch keep the state levels in
    rings of different length: changing the shape between calls, at every
    residue of the step, keeps the trajectory."""
    from damian_hip import cases, lib
    case = cases.f2()
    ref = lib.Solver(case, precision=prec)
    r0 = ref.run(120)
    u0, up0, _ = ref.state()
    ref.close()
    s = lib.Solver(case, precision=prec)
    parts, n, k = [], 0, 0
    while n < 120:
        s.set_tuning(*((64, 0, 0, 1), (128, 1, 0, 3), (256, 1, 12, 1), (64, 1, 0, 2))[k % 4])
        m = min(120 - n, 1 + k % 7)
        parts.append(s.run(m))
        n, k = n + m, k + 1
    u, up, _ = s.state()
    t = s.autotune(5)   # leaves the state where it was
    assert len(t) == 4
    u1, up1, _ = s.state()
    s.close()
    assert np.array_equal(np.concatenate(parts), r0)
    for a, b in ((u, u0), (up, up0), (u1, u0), (up1, up0)):
        assert np.array_equal(a, b)
