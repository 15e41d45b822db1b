"""Layouts and kernels chosen by a rule, on both sides of its line: the samples
and states of every layout are the same bits, and those of the plain ones are
held to the CPU oracle by the other tests."""
import copy

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {0: 1e-12, 1: 1e-5}   # against the oracle (FP32C against its FP64), as for every parity case


def layer(cases, nx, nz, sheet=None):
    w, h = 5.0 * nx, 5.0 * nz
    text = cases.problem_text(w, h, 0.4, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                              [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.2, 0.2, 1.0, 5.0])
    return cases.S.case_from_problem_text(text, sheet=sheet or (-3.3, w - 10.0, 4.1), name="layer")


def scattered(cases, case, n, seed):
    """n receivers at seeded points of the mesh, some in no element."""
    rng = np.random.default_rng(seed)
    out = copy.copy(case)
    e = rng.integers(0, case.nelems, n)
    c = case.mesh.corners()[e] - 1
    x0 = case.mesh.nodes[c[:, 0]]
    h = case.mesh.nodes[c[:, 2], 1] - x0[:, 1]
    out.recv_elem = np.where(rng.random(n) < 0.05, 0, e + 1).astype(np.int32)
    out.recv_xy = x0 + h[:, None] * rng.uniform(0.03, 0.97, (n, 2))
    out.recv_ff = cases.S.inside_soil(case.model, *out.recv_xy.T).astype(np.uint8)   # as the oracle does
    return out


# one workgroup up to 896 receivers, whole and partial groups of 256 above
@pytest.mark.parametrize("nrecv", [896, 897, 1024, 1025, 2500])
@pytest.mark.parametrize("prec", [0, 1])
def test_receivers_only_kernel(nrecv, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    case = scattered(cases, layer(cases, 60, 40), nrecv, nrecv)
    n = 90
    _, _, _, rec_o = O.run(case, nsteps=n, recv_interval=1)
    assert np.abs(rec_o).max() > 1e-3
    for tuning in ((128, 1, 0, 3), (256, 1, 0, 1)):
        print(f"nrecv={nrecv} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        s.set_tuning(*tuning)
        # calls that end in the receivers-only kernel: whole launches
        rec = np.concatenate([s.run(k, noalloc=k == 6) for k in (30, 3, 3, 6, 48)])
        s.close()
        assert rel_l2(rec, rec_o) <= TOL[prec]
        assert not rec[:, case.recv_elem == 0].any()


def fronts(cases, nx, nz, part, seed=7):
    """10 m cells, halved everywhere but in the first `part` of the width, there at random."""
    w, h = 10.0 * nx, 10.0 * nz
    text = cases.problem_text(w, h, 1.0, 0.002, 0.2, 10, 5.0, [("p", 1000, "s", 500, 2000)], "WAVESV",
                              [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.1, 0.0, 1.0, 5.0])
    mdl = cases.S.build_model(cases.S.parse_problem(text))
    rng = np.random.default_rng(seed)
    m = cases.S.quadtree_mesh(mdl.totcols - 1, mdl.totrows - 1, mdl.blength, 2,
                              lambda x, z, s: (x >= part * w) | (rng.random(len(x)) < 0.5))
    return cases.S.finish_case(mdl, m, sheet=(-3.3, w - 10.0, 19.1), name="fronts")


def same_bits(cases, lib, case, prec, tunings, n, first=(256, 1, 0, 2)):
    """Samples and states of n steps (calls of several lengths) are those of `first`."""
    want = None
    for tuning in (first,) + tunings:
        print(f"{case.name} nodes={case.mesh.nnodes} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        s.set_tuning(*tuning)
        got = [np.concatenate([s.run(k) for k in (1, 2, n // 2 - 3, n - n // 2)])] + list(s.state())
        s.close()
        want = want or got
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
    return want


# below and above the line (196,608 nodes), with per-element moduli; hanging
# nodes in half of the mesh (tiles of 128) and in a twentieth of it (of 64)
@pytest.mark.parametrize("name", ["layer_195804", "layer_198891", "layer_het", "fronts_half", "fronts_twentieth"])
@pytest.mark.parametrize("prec", [0, 1])
def test_one_step_layouts(name, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    if name.startswith("layer"):
        case = layer(cases, 443 if name == "layer_195804" else 450, 440, sheet=(-3.3, 2200.0, 19.1))
        case = cases.perturbed(case, seed=3) if name == "layer_het" else case
    else:
        case = fronts(cases, 400, 200, 0.5 if name == "fronts_half" else 0.05)
    n = 80
    want = same_bits(cases, lib, case, prec, ((256, 1, 0, 1), (64, 0, 12, 1), (32, 1, 0, 1)), n)
    assert np.abs(want[1]).max() > 1e-3
    if name in ("layer_het", "fronts_half"):
        u_o, up_o, _, rec_o = O.run(case, nsteps=n, recv_interval=1, threads=8)
        for a, b in ((want[0], rec_o), (want[1], u_o), (want[2], up_o)):
            assert rel_l2(a, b) <= TOL[prec]


@pytest.mark.parametrize("prec", [0, 1])
def test_one_step_tiles_that_do_not_fit(prec):
    """Cut into patches and small tiles (of 64 and of 128 nodes) instead."""
    from damian_hip import cases, lib
    for case in (cases.c2(), fronts(cases, 60, 40, 1.0)):
        want = same_bits(cases, lib, case, prec, ((1024, 1, 0, 1), (1024, 0, 12, 1)), 80)
        assert np.abs(want[1]).max() > 0


@pytest.mark.parametrize("prec", [0, 1])
def test_patches_of_small_instances(prec):
    """A batch with patches (above the line as a whole) of meshes at whose sizes
    the patches' number and rings change: none, one, several in a row, cells cut
    by the sides, uniform and with moduli per element."""
    from damian_hip import cases, lib
    sizes = [(12, 7), (17, 17), (24, 16), (40, 33), (70, 50), (31, 24)]
    small = [layer(cases, nx, nz) for nx, nz in sizes]
    small += [cases.perturbed(m, seed=k) for k, m in enumerate(small)] + [cases.BUILDERS["f2"]()]
    n = 90
    want = []
    for m in small:
        s = lib.Solver(m, precision=prec)
        s.set_tuning(64, 1, 0, 2)
        want.append((s.run(n),) + s.state()[:2])
        s.close()
        assert np.abs(want[-1][1]).max() > 1e-3
    large = layer(cases, 450, 440, sheet=(-3.3, 2200.0, 19.1))
    for tuning in ((256, 1, 0, 1), (32, 0, 30, 1)):
        print(f"prec={prec} tuning={tuning}", flush=True)
        b = lib.Batch([lib.Solver(m, precision=prec, init=False) for m in small + [large]])
        b.set_tuning(*tuning)
        rec = np.concatenate([b.run(k) for k in (1, 29, 60)])
        at = 0
        for q, (m, w) in enumerate(zip(small, want)):
            k = len(m.recv_elem)
            assert np.array_equal(rec[:, at:at + k], w[0])
            at += k
            for a, x in zip(b.state(q), w[1:]):
                assert np.array_equal(a, x)
        b.close()


# block patches with 2 to 8 rings (test_host_runtime.py holds that they are there)
BLOCK_SHAPES = ((128, 0, 0, 2), (192, 1, 12, 3), (128, 1, 0, 4), (96, 1, 0, 5), (64, 1, 0, 6), (48, 1, 0, 8))


@pytest.mark.parametrize("name", ["layer", "layer_het", "basin"])
@pytest.mark.parametrize("prec", [0, 1])
def test_block_patch_layouts(name, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    if name == "basin":
        case = cases.c4_valley(200.0, "SV", 10.0)
    else:
        case = layer(cases, 300, 200, sheet=(-3.3, 1490.0, 19.1))
        case = cases.perturbed(case, seed=5) if name == "layer_het" else case
    shapes = []
    probe = lib.Solver(case, precision=prec)
    for t in BLOCK_SHAPES:
        try:
            probe.set_tuning(*t)
            shapes.append(t)
        except lib.DmpError as e:   # hanging nodes widen the rings of deep launches
            assert name == "basin" and t[3] > 4 and e.code == -4
    probe.close()
    assert len(shapes) >= 3
    n = 300 if name == "basin" else 60   # the pulse is in the box
    want = same_bits(cases, lib, case, prec, tuple(shapes), n, first=(256, 1, 0, 1))
    assert np.abs(want[1]).max() > 1e-3
    if name != "layer":
        u_o, up_o, _, _ = O.run(case, nsteps=n, recv_interval=1, threads=8)
        for a, b in ((want[1], u_o), (want[2], up_o)):
            assert rel_l2(a, b) <= TOL[prec]
