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


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name", ["f1", "f2het_buried", "pointd", "layer_1023"])
def test_whole_mesh_in_one_tile(name, prec):
    """Meshes of one tile, up to the largest (1023 nodes), take as many steps
    per launch as the LDS holds source terms for: calls shorter, as long and
    longer than a launch, sampled every step and every third, give the bits of
    launches of few steps in several tiles."""
    from damian_hip import cases, lib
    if name == "layer_1023":
        case = layer(cases, 32, 30, True)
    elif name.endswith("_buried"):
        case = cases.with_buried_receivers(cases.BUILDERS[name[:-len("_buried")]]())
    else:
        case = cases.BUILDERS[name]()
    n = case.mesh.nnodes - len(case.hanging)
    assert n <= 1023
    for io in (1, 3):
        ref = lib.Solver(case, precision=prec, io_interval=io)
        ref.set_tuning(64, 0, 0, 2)
        want = ref.run(200), ref.state()
        ref.close()
        assert np.abs(want[0]).max() > 0
        for tuning in (None, (max(n, 32), 0, 12, 2)):
            print(f"name={name} nodes={n} prec={prec} io={io} tuning={tuning}", flush=True)
            s = lib.Solver(case, precision=prec, io_interval=io)
            if tuning:
                s.set_tuning(*tuning)
            parts = [s.run(k) for k in (1, 1, 8, 31, 32, 33)] + [s.run(17, noalloc=True), s.run(77)]
            got = s.state()
            s.close()
            assert np.array_equal(np.concatenate(parts), want[0])
            for a, b in zip(got, want[1]):
                assert np.array_equal(a, b)


# more tiles than compute units (32 nodes each): 16 x 16 patches with 2 to 8
# rings, uniform and with moduli per element, and in a mesh with hanging nodes
@pytest.mark.parametrize("name", ["layer", "layer_het", "basin"])
@pytest.mark.parametrize("prec", [0, 1])
def test_block_patches(name, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    case = cases.c4_valley(62.0, "SV", 10.0) if name == "basin" else layer(cases, 143, 77, name == "layer_het")
    n = 61
    ref = lib.Solver(case, precision=prec)
    ref.set_tuning(128, 1, 0, 3)   # fewer tiles than compute units: no patches
    ref.run(400 if name == "basin" else 60)
    want = (ref.run(n),) + ref.state()[:2]
    ref.close()
    assert np.abs(want[1]).max() > 1e-3
    if name == "layer_het":
        u_o, _, _, rec_o = O.run(case, nsteps=60 + n, recv_interval=1)
        assert rel_l2(want[0], rec_o[61:]) <= TOL[prec]
    for tuning in ((32, 0, 0, 2), (32, 1, 12, 3), (33, 1, 0, 4), (40, 1, 0, 5), (32, 1, 0, 8)):
        print(f"name={name} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        try:
            s.set_tuning(*tuning)
        except lib.DmpError as e:   # hanging nodes widen the rings of deep launches
            assert name == "basin" and tuning[3] > 4 and e.code == -4
            continue
        s.run(400 if name == "basin" else 60)
        got = (s.run(n),) + s.state()[:2]
        s.close()
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name", ["valley", "canyon"])
def test_halved_tiles(name, prec):
    """Layouts with more workgroups than compute units halve the few tiles
    that need more than 512 lanes (those that hanging nodes widen)."""
    from damian_hip import cases, lib
    case = cases.c4_valley(200.0, "SV", 10.0) if name == "valley" else cases.BUILDERS["c2"]()
    n = 41
    ref = lib.Solver(case, precision=prec)
    ref.set_tuning(256, 1, 0, 1)
    ref.run(300)
    want = (ref.run(n),) + ref.state()[:2]
    ref.close()
    assert np.abs(want[0]).max() > 0
    for tuning in ((256, 1, 0, 3), (200, 1, 0, 4), (170, 0, 12, 4), (140, 1, 0, 4)):
        print(f"name={name} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        try:
            s.set_tuning(*tuning)
        except lib.DmpError as e:   # hanging nodes widen the rings of deep launches
            assert e.code == -4
            continue
        s.run(300)
        got = (s.run(n),) + s.state()[:2]
        s.close()
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
